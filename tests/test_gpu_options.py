"""What the engine's options read back."""
import pytest

from tests import test_gpu_parity as el

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    import fwi2d_amd
    fwi2d_amd.load()
    return fwi2d_amd


def test_shots_per_block_reads_back(lib):
    """A number of shots per workgroup that was set reads back as it was set, also one above the number
    of shots; while none is set the statistic is the number in effect."""
    case = el.engine_case(ns=2, nt=40)
    for key in ("shots_per_block", "shots_per_block_edge"):
        e, _ = el.run_engine(lib, *case)
        assert e.stat(key) == 1
        e.set_option(key, 16)
        assert e.stat(key) == 16
        e.close()


@pytest.mark.parametrize("mb", [16, 17, 21])
def test_checkpoint_budget_holds_the_rows_below_a_free_surface(lib, mb):
    """Checkpoints (two levels and the 16 rows' carry for each segment after the first) and snapshot
    slots (two more than a segment has) stay within the budget wherever it allows longer segments than
    the default ones."""
    nx, ns, nt = 300, 2, 301
    e, _ = el.run_engine(lib, *el.engine_case(nx=nx, nz=60, nt=nt, ns=ns), sub=1, keep=True,
                         options=(("checkpoint_budget", mb),))
    row = ns * 2 * nx * 4
    level, carry = row * 64, row * 16
    k, n = e.stat("segment"), e.stat("nseg")
    e.close()
    assert k > 25
    assert (n - 1) * (2 * level + carry) + (k + 2) * level <= mb << 20

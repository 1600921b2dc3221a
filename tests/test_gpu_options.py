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

"""The speed of the waves on the grid: a stencil whose FP32 coefficients are no longer consistent
(D2 weights that do not sum to zero, a D1 that does not return a straight line's slope) carries
the same error at every cell and step, which delays every wave by an amount that grows with time.

1500 steps of waves with about 15 cells per wavelength, against the FP64 oracle: the delay is the
least-squares factor of the traces' error on their change per step.  Tolerance 1e-4 steps: of
the factors that FP32 has to round, 1 / (24 h^2) and the pair of D1, each moves the squared speed
by at most 6e-8, which is 4.5e-5 steps after 1500; the random rounding of the levels, 5e-6 of the
traces against a change of about 0.04 of them a step, adds 1e-4 over the root of the 50 and more
independent samples that the traces hold, and the random rounding of the weights, of the same
size per cell, averages over the thousands of cells on the way.  (Rounded one by one, 5/6,
1/24 and 1/6 leave D2 a sum of 6.7e-8 c / h^2: 3e-4 steps here.)
"""
import numpy as np
import pytest

from fwi2d_amd import workloads as W
from tests import test_gpu_acoustic as ac
from tests import test_gpu_parity as el

pytestmark = pytest.mark.gpu

NX, NZ, H, DT, NT = 240, 90, 0.01, 0.001, 1500


def delay(out, ref):
    d, du = out.astype(np.float64) - ref, np.gradient(ref, axis=-1)
    return float((d * du).sum() / (du * du).sum()), float(np.linalg.norm(d) / np.linalg.norm(ref))


def traces(orc64, physics):
    """the engine's traces and the oracle's"""
    import fwi2d_amd as lib

    x, z = np.arange(NX)[:, None] * H, np.arange(NZ)[None, :] * H
    vp = 1.6 + 0.7 * z + 0.08 * np.sin(5 * x + 1) * np.cos(7 * z) + 0 * x
    rho = 2.0 + 0.15 * np.sin(4 * x) * np.cos(6 * z)
    sxz = np.array([[0.4, 0.03]])
    rxz = [np.stack([np.linspace(0.3, 2.1, 40), np.full(40, 0.02)], 1)]
    if physics == "acoustic":
        grid = ac.case(nt=NT, bc=(1, 2, 2, 2), taper=20)[0]
        grid.update(nx=NX, nz=NZ, sub=0)
        model = np.stack([rho * vp ** 2, 1 / rho]).astype(np.float32).astype(np.float64)
        src = W.ricker(NT, DT, 9.0)[None]
        assert grid["dt"] == DT
        sxz[0, 1] = rxz[0][0, 1] = 0.1  # away from the free surface, where the pressure is zero
        ref = ac.oracle_run(orc64, grid, model, sxz, rxz, src)[0]
        e = ac.engine(lib, grid, model, sxz, rxz)
        out = e.forward(src)
    else:
        prob = el.engine_case(nx=NX, nz=NZ, nt=NT, vti=physics == "vti", ns=1)[0]
        vs = vp / 1.9
        mu = rho * vs ** 2
        lam = rho * vp ** 2 - 2 * mu
        fields = [lam, mu, rho]
        if physics == "vti":
            del_, eps = 0.06 + 0.03 * np.sin(3 * x) + 0 * z, 0.1 + 0.04 * np.cos(4 * z) + 0 * x
            fields += [np.sqrt(2 * (lam + 2 * mu) * (lam + mu) * del_ + (lam + mu) ** 2) - mu, eps]
        model = np.stack(fields).astype(np.float32).astype(np.float64)  # the values that both sides take
        wav = W.ricker(NT, DT, 5.0)
        src = np.stack([0.3 * wav[None], wav[None]])
        ref = el.oracle_forward(orc64, prob, model, sxz, rxz, src, NT, DT)
        _, out = el.run_engine(lib, prob, model, sxz, rxz, src, NT, DT)
    return out, ref


@pytest.mark.parametrize("physics", ["iso", "vti", "acoustic"])
def test_no_delay(orc64, physics):
    a, err = delay(*traces(orc64, physics))
    print("%s: delay %.2e steps, relative error %.2e" % (physics, a, err))
    assert abs(a) <= 1e-4


@pytest.mark.parametrize("physics", ["iso", "vti"])
def test_surface_waves_below_the_rounding_of_the_levels(orc64, physics):
    """The traces of a free surface are nearer to FP64 than levels rounded to FP32 at every step leave
    them, since the rows below it carry their rounding over.  Tolerance 2.5e-6, two thirds of the
    3.7e-6 that exact arithmetic on rounded levels leaves here (rounding errors of rms 0.3 ulp,
    integrated twice over 1500 steps): the right-hand side's own rounding, of terms a tenth of
    the levels' size, and the waves' share below the 16 rows remain."""
    out, ref = traces(orc64, physics)
    err = delay(out, ref)[1]
    print("%s: relative error %.2e" % (physics, err))
    assert err <= 2.5e-6

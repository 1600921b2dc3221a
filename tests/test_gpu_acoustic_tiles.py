"""The acoustic step's 32 x 32 tiles where their frame arithmetic can go wrong: the smallest grid
(both sides' closure rows in one tile), grids that end just before, at and just after a tile
boundary along either axis, every boundary kind on every side; the gradient by parts in time
(sub 1) and per snapshot (sub 2), with a time window that weights the snapshots unequally.
Against the FP64 oracle with the engine's tolerances: traces within twice the FP32 gap of the
oracle itself (at least 1e-5), gradients within 1e-4."""
import numpy as np
import pytest

from fwi2d_amd import workloads as W
from tests.test_gpu_acoustic import case, engine, lib, oracle_run, rel  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sub", [1, 2])
@pytest.mark.parametrize("nx,nz,bc", [(12, 12, (1, 2, 3, 1)), (13, 33, (3, 1, 2, 2)), (37, 38, (2, 1, 1, 3)),
                                      (64, 32, (1, 3, 2, 1)), (70, 101, (2, 3, 1, 2))])
def test_acoustic_tile_edges(lib, orc64, orc32, nx, nz, bc, sub):  # noqa: F811
    nt, h = 160, 0.01
    grid = case(nt=nt, bc=bc, taper=3, sub=sub)[0]
    grid.update(nx=nx, nz=nz, gdamp_tmin=0.0, gdamp_tmax=0.2, gdamp_power=0.5)
    x, z = np.arange(nx)[:, None] * h, np.arange(nz)[None, :] * h
    vp = 1.8 + 0.8 * z + 0.4 * x
    rho = 2.0 + 0.2 * np.sin(40 * x) * np.cos(50 * z)
    model = np.stack([rho * vp ** 2, 1 / rho])
    lx, lz = (nx - 1) * h, (nz - 1) * h
    sxz = np.array([[0.3 * lx, 0.4 * lz], [0.62 * lx, 0.13 * lz]])
    rxz = [np.stack([np.linspace(0.05 * lx, 0.95 * lx, 7), np.linspace(0.9 * lz, 0.1 * lz, 7)], 1) for _ in range(2)]
    src = np.stack([W.ricker(nt, grid["dt"], f) for f in (25.0, 30.0)])
    adj = np.random.default_rng(nx).standard_normal((14, nt)) * np.hanning(nt)
    ref, gref = oracle_run(orc64, grid, model, sxz, rxz, src, adj=adj)
    gap = rel(oracle_run(orc32, grid, model, sxz, rxz, src)[0], ref)
    e = engine(lib, grid, model, sxz, rxz)
    err = rel(e.forward(src, keep_snapshots=True), ref)
    gk = e.adjoint(adj)
    e.close()
    errs = [rel(gk[c], gref[c]) for c in range(2)]
    print("%dx%d bc=%s sub=%d: traces %.3e (FP32 gap %.3e), gradients %.3e %.3e" % (nx, nz, bc, sub, err, gap, *errs))
    assert err <= max(1e-5, 2 * gap)
    assert max(errs) <= 1e-4

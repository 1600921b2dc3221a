"""Grids whose level or closure weights lie past 32-bit offsets: an acoustic level of 1.6e9 cells
(6 GiB: byte offsets past 2^32) and 22.4 million columns (2 nx 48 closure weights: indices past 2^31),
on both engines.  Ten steps next to the far side equal those of a small grid with the same
cells there; 22.4 million and 96 columns are whole tiles, so the same cells fall into the same kinds
of tiles and the values are the same bit for bit.  (All positions are binary fractions, so that the
points' weights are the same too.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NX, SMALL, H, DT, NT = 22_400_000, 96, 1 / 64, 1 / 1024, 10


@pytest.fixture(scope="module")
def lib():
    import fwi2d_amd
    fwi2d_amd.load()
    return fwi2d_amd


def grid(lib, nx, nz, sub, bc):
    prob = dict(nx=nx, nz=nz, dx=H, dz=H, bc_top=bc[0], bc_bottom=bc[1], bc_left=2, bc_right=bc[2], taper_top=0,
                taper_bottom=4, taper_left=4, taper_right=4, taper_strength=0.05, vti=0)
    return lib.grid_from(prob, NT, DT, sub)


def fields(base, nz, nx):
    """smooth fields in the last SMALL columns, constant before them"""
    x, z = np.arange(SMALL)[:, None], np.arange(nz)[None, :]
    out = np.empty((len(base), nx, nz), np.float32)
    for k, v in enumerate(base):
        out[k, :-SMALL] = v
        out[k, -SMALL:] = v * (1 + 0.1 * np.sin(0.2 * x + k) * np.cos(0.15 * z))
    return out


def points(nx, nz, ns):
    x0 = (nx - SMALL) * H
    sxz = np.array([[x0 + 80.25 * H, (nz - 4) * H], [x0 + 71.5 * H, 5.75 * H]])
    rxz = [np.array([[x0 + (94 - 6 * s - 2 * k) * H, (nz - 3.5 + 2 * s - k / 2) * H] for k in range(7)]) for s in range(2)]
    return sxz[:ns], rxz[:ns]


def test_acoustic_level_past_4_gib(lib):
    nz = 70  # rows 32-63 hold an interior tile
    src = np.random.default_rng(0).standard_normal((1, NT)).astype(np.float32)
    adj = np.random.default_rng(1).standard_normal((7, NT)).astype(np.float32)
    out = []
    for nx in (SMALL, NX):
        e = lib.AcousticEngine(grid(lib, nx, nz, 1, (1, 2, 3)), 1.0)
        e.set_model(fields((6.0, 0.5), nz, nx))
        e.set_shots(*points(nx, nz, 1))
        d = e.forward(src, keep_snapshots=True)
        g = e.adjoint(adj)
        out.append((d, g[:, -48:].copy()))
        print("nx %d: done" % nx, flush=True)
        e.close()
        del g
    assert np.abs(out[0][0]).max() > 0 and np.abs(out[0][1]).max() > 0
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])


def test_elastic_closure_weights_past_2_31(lib):
    nz = 12
    src = np.random.default_rng(2).standard_normal((2, 2, NT)).astype(np.float32)
    out = []
    for nx in (SMALL, NX):
        e = lib.Engine(grid(lib, nx, nz, 0, (1, 1, 2)))
        e.set_model(fields((2.5, 1.7, 2.0), nz, nx))
        e.set_shots(*points(nx, nz, 2))
        out.append(e.forward(src))
        print("nx %d: done" % nx, flush=True)
        e.close()
    assert np.abs(out[0]).max() > 0
    assert np.array_equal(out[0], out[1])

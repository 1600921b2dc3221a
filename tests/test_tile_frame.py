"""CPU emulation of the index arithmetic of the frame tiles of k_step and k_img
(fwi2d_amd/csrc/kernels.hip): tiles with closure rows or SAT terms.

For every tile of many grid shapes and each axis (the stencils are separable):
  * the tiles' cells partition the grid;
  * closure rows of the cells and of the products lie only in tiles that run their passes;
  * every read of a used value lands inside the LDS window on a loaded grid cell, and every
    other read inside the window's arrays;
  * the closure terms are kept in window cells that lie outside the grid.
"""
import pytest

TZ, HX, HZ = 64, 4, 8


def tile_range(k, ntile, T, n, last):
    if ntile == 1:
        return 0, n
    if k == ntile - 1:
        return last, n
    return k * T, min(k * T + T, last)


def window_start(s, H):
    return 0 if H <= s < H + 2 else s - H


def product_range(s, e, n):
    lo, hi = max(0, s - 2), min(n, e + 2)
    if s < 4:
        lo, hi = 0, max(hi, 6)
    if e > n - 4:
        lo, hi = min(lo, n - 6), n
    return lo, hi


def rows(g, n, depth, points):
    """points of a closure row (depth rows from a side), or the interior stencil's"""
    if g < depth:
        return list(range(points))
    if g >= n - depth:
        return [n - 1 - j for j in range(points)]
    return [g - 2, g - 1, g, g + 1, g + 2]


def nonzero(g, n):
    """points of the D1 rows with a coefficient"""
    if g < 4:
        return list(range(6))
    if g >= n - 4:
        return [n - 1 - j for j in range(6)]
    return [g - 2, g - 1, g + 1, g + 2]


def check_x(nx, TX):
    WX, IX = TX + 2 * HX, TX + 4
    ntx = -(-nx // TX)
    seen = []
    for k in range(ntx):
        s, e = tile_range(k, ntx, TX, nx, nx - TX)
        seen += range(s, e)
        ws, (lo, hi) = window_start(s, HX), product_range(s, e, nx)
        left, right = s == 0, k == ntx - 1
        assert e - s <= TX and hi - lo <= IX
        if left:  # the SAT terms' column
            assert 0 <= -1 - ws
        if right:
            assert nx - ws < WX
        for g in range(lo, hi):
            for c in nonzero(g, nx):
                assert 0 <= c < nx and 0 <= c - ws < WX, (nx, s, g, c)
        for g in range(s, e):
            assert hi - 1 - lo < IX
            if g < 4 or g >= nx - 4:  # imaging D1 on the snapshot window: 6 points
                assert all(0 <= c - lo < IX for c in rows(g, nx, 4, 6))
            assert (g != 0 or left) and (g != nx - 1 or right)
            for c in rows(g, nx, 6, 8) + nonzero(g, nx):  # state: D2, imaging D1
                assert 0 <= c < nx and 0 <= c - ws < WX
            for c in nonzero(g, nx):  # products with a coefficient: formed; snapshot window: loaded
                assert lo <= c < hi
        # k_img: halo 2
        ws = window_start(s, 2)
        for g in range(s, e):
            for c in nonzero(g, nx):
                assert 0 <= c < nx and 0 <= c - ws < TX + 4
    assert sorted(seen) == list(range(nx))


def check_z(nz):
    ldz = (nz + 31) // 32 * 32
    ntz = -(-ldz // TZ)
    WZ, PZ = TZ + 2 * HZ, TZ + 8
    seen = []
    for k in range(ntz):
        s, e = tile_range(k, ntz, TZ, nz, ldz - TZ)
        seen += range(s, e)
        ws, p0, (lo, hi) = s - HZ, s - 4, product_range(s, e, nz)
        top, bot = s == 0, k == ntz - 1
        if top:  # the closure terms' rows, 8 above; the imaging derivatives', 4 above
            assert ws == -8 and p0 == -4
        if bot:  # 8 below; the 4 rows past the tile
            assert nz - 6 + 8 >= nz and nz - 1 + 8 - ws < WZ
            assert s + TZ >= ldz and s + TZ + 3 - ws < WZ and s + TZ + 3 - p0 < PZ
        for z0 in range(p0, p0 + PZ, 4):  # product quads
            if z0 + 3 < lo or z0 >= hi:
                continue
            assert 0 <= z0 - 4 - ws and z0 + 7 - ws < WZ and 0 <= z0 and z0 + 3 < ldz
        for g in range(lo, hi):
            closure = g < 4 or g >= nz - 4
            assert not closure or (top if g < 4 else bot)
            assert 0 <= g - p0 < PZ
            for c in nonzero(g, nz):
                assert 0 <= c < nz and 0 <= c - ws < WZ
        for z0 in range(s, e, 4):  # new-level quads: whole-quad reads
            assert 0 <= z0 - 4 - ws and z0 + 7 - ws < WZ and 0 <= z0 - 4 - p0 and z0 + 7 - p0 < PZ
        for g in range(s, e):
            closure = g < 6 or g >= nz - 6
            assert not closure or (top if g < 6 else bot)
            for c in rows(g, nz, 6, 8) + nonzero(g, nz):
                assert 0 <= c < nz and 0 <= c - ws < WZ and 0 <= c - p0 < PZ
            for c in nonzero(g, nz):
                assert lo <= c < hi
    assert sorted(seen) == list(range(nz))


@pytest.mark.parametrize("TX", [16, 32])
def test_frame_tiles_x(TX):
    for nx in list(range(12, 140)) + [601, 801, 1000, 1700, 3001]:
        check_x(nx, TX)


def test_frame_tiles_z():
    for nz in list(range(12, 300)) + [500, 501, 1000, 1003]:
        check_z(nz)

// Device kernels of the elastic SBP-SAT propagation engine, written for gfx950.
//
// Layout: every field is [x][ldz] with z contiguous (index ix*ldz + iz), the reference's
// [x][z] order with z padded to a multiple of 32 cells (128-byte columns).  Workgroups
// of 256 threads own a tile of cells and a group of shots; a thread moves 4 consecutive
// z cells (a quad) with 128-bit accesses.  The time step and the imaging kernel run over
// the tile grid below.
//
// Tile grid: tiles start at multiples of the tile size except the last one in each
// direction, which is anchored to end at the grid edge (start = n - T).  Each tile
// writes the cells in [start, next tile start) (the last tile writes to the edge), so
// writes never overlap and the SBP closure rows near the far edge are always written by
// the anchored tile.
#include "kernels.h"
#include "sbp_tables.h"
#include <hip/hip_fp16.h>

namespace fwi2d {

// Interior rows and the SAT's boundary derivative, as literals in the kernels (the frame tiles are
// short of scalar registers).  Elastic rows: see kD2Interior24; the acoustic ones are rounded one
// by one.
template <int N>
struct Row {
    float c[N];
};
template <int N>
constexpr Row<N> rounded(const double (&v)[N])
{
    Row<N> r{};
    for (int i = 0; i < N; i++) r.c[i] = (float)v[i];
    return r;
}
constexpr Row<2> kD1A = rounded(kD1Interior);
constexpr Row<10> kD2A = rounded(kD2Interior);
constexpr Row<4> kSC = rounded(kBoundaryDeriv);

// ---------------------------------------------------------------------------
// Tile geometry.  x: tiles of TX columns; z: tiles of 64 cells aligned on quads.  The
// last tile of each axis is anchored at the far edge so that the SBP closure rows there
// are always written by one tile; write ranges partition the grid.
// ---------------------------------------------------------------------------
__host__ __device__ __forceinline__ void tile_range_x_hd(int k, int ntile, int T, int n, int& s, int& e)
{
    if (ntile == 1) { s = 0; e = n; return; }
    if (k == ntile - 1) { s = n - T; e = n; return; }
    s = k * T;
    e = (s + T < n - T) ? s + T : n - T;
}

__host__ __device__ __forceinline__ void tile_range_z_hd(int k, int ntile, int nz, int ldz, int& s, int& e)
{
    const int last = ldz - kTileZ;  // quad-aligned start of the anchored tile
    if (ntile == 1) { s = 0; e = nz; return; }
    if (k == ntile - 1) { s = last; e = nz; return; }
    s = k * kTileZ;
    e = (s + kTileZ < last) ? s + kTileZ : last;
}

int tiles_x(int nx, int tile_x) { return (nx + tile_x - 1) / tile_x; }
int tiles_z(int ldz) { return (ldz + kTileZ - 1) / kTileZ; }
void tile_range_x(int k, int ntile, int T, int n, int& s, int& e) { tile_range_x_hd(k, ntile, T, n, s, e); }
void tile_range_z(int k, int ntile, int nz, int ldz, int& s, int& e) { tile_range_z_hd(k, ntile, nz, ldz, s, e); }

// first cell of a tile's window with halo H such that SBP closures at the near edge
// (rows < 6 for D2, < 4 for D1) always see the edge itself
__device__ __forceinline__ int window_start(int s, int H)
{
    return (s >= H && s < H + 2) ? 0 : s - H;
}

// Range [lo, hi) of first-derivative products a tile writing [s, e) of n cells reads:
// its cells +/- 2, widened to the 6 closure inputs of D1 rows at either grid edge.
__host__ __device__ __forceinline__ void product_range(int s, int e, int n, int& lo, int& hi)
{
    lo = s - 2 > 0 ? s - 2 : 0;
    hi = e + 2 < n ? e + 2 : n;
    if (s < 4) { lo = 0; hi = hi > 6 ? hi : 6; }
    if (e > n - 4) { lo = lo < n - 6 ? lo : n - 6; hi = n; }
}

// Workgroups are dispatched round-robin over the 8 XCDs; give each XCD a contiguous run
// of (shot, tile) work items so that neighbouring tiles share that XCD's L2.
__device__ __forceinline__ int xcd_remap(int bid, int nb)
{
    const int q = nb >> 3, r = nb & 7;
    const int xcd = bid & 7, local = bid >> 3;
    return (xcd < r) ? xcd * (q + 1) + local : r * (q + 1) + (xcd - r) * q + local;
}

// every quad access is 16-byte aligned (quads start at multiples of 4 cells of 16-byte
// aligned arrays); saying so lets LDS quads load with one 128-bit read
__device__ __forceinline__ float4 ld4(const float* p)
{
    return *reinterpret_cast<const float4*>(__builtin_assume_aligned(p, 16));
}
__device__ __forceinline__ void st4(float* p, float4 v) { *reinterpret_cast<float4*>(__builtin_assume_aligned(p, 16)) = v; }
typedef float v4f __attribute__((ext_vector_type(4)));
// the same with a uniform choice of the streaming form (data that no cache will hold until it is
// used again leaves the room to data that is)
__device__ __forceinline__ float4 ld4(const float* p, bool stream)
{
    if (!stream) return ld4(p);
    const v4f v = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(__builtin_assume_aligned(p, 16)));
    return make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void st4(float* p, float4 v, bool stream)
{
    const v4f x = {v.x, v.y, v.z, v.w};
    if (stream) __builtin_nontemporal_store(x, reinterpret_cast<v4f*>(__builtin_assume_aligned(p, 16)));
    else st4(p, v);
}
__device__ __forceinline__ void unpack(float4 v, float* d)
{
    d[0] = v.x;
    d[1] = v.y;
    d[2] = v.z;
    d[3] = v.w;
}

// ---------------------------------------------------------------------------
// SBP stencils on LDS lines.  p points at the element of global index g (0 <= g < n);
// s is the LDS stride along the differentiated axis.  Results are not divided by h.
// Closure rows are evaluated out of line so that the interior path stays small.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float d1_int(const float* p, int s)
{
    return kD1InteriorF[0] * (p[s] - p[-s]) + kD1InteriorF[1] * (p[2 * s] - p[-2 * s]);
}

// Closure row R of D1 from the edge point q along stride st, with the coefficients as
// immediates (zero ones skipped).
template <int R>
__device__ __forceinline__ float d1_closure_row(const float* q, int st)
{
    float v = 0.f;
#pragma unroll
    for (int j = 0; j < 6; j++)
        if (kD1Closure[R][j] != 0.0) v += (float)kD1Closure[R][j] * q[j * st];
    return v;
}

// D1 closure row of point g of n: rows 0..3 at the near edge, mirrored with opposite sign
// at the far edge.  The row is dispatched to a compile-time instance (a uniform branch
// where the row is the same for a whole wavefront).
__device__ __forceinline__ float d1_closure(const float* p, int s, int g, int n)
{
    const bool near = g < 4;
    const int r = near ? g : n - 1 - g;
    const float* q = near ? p - g * s : p + r * s;
    const int st = near ? s : -s;
    float v;
    switch (r) {
    case 0: v = d1_closure_row<0>(q, st); break;
    case 1: v = d1_closure_row<1>(q, st); break;
    case 2: v = d1_closure_row<2>(q, st); break;
    default: v = d1_closure_row<3>(q, st); break;
    }
    return near ? v : -v;
}

template <bool IN>
__device__ __forceinline__ float d1(const float* p, int s, int g, int n)
{
    if (IN || (g >= 4 && g < n - 4)) return d1_int(p, s);
    return d1_closure(p, s, g, n);
}

// interior weights of D2(c) at one point, times 24 h^2: u[-2..2] coefficients (Dzz_var/Dxx_var interior)
struct W5 {
    float m2, m1, c, p1, p2;
};

__device__ __forceinline__ W5 d2_weights(const float* pc, int s)
{
    const float fm2 = pc[-2 * s], fm1 = pc[-s], f0 = pc[0], fp1 = pc[s], fp2 = pc[2 * s];
    W5 w;
    w.c = kD2Interior24[0] * f0 + kD2Interior24[1] * (fm1 + fp1) + kD2Interior24[2] * (fm2 + fp2);
    w.m1 = kD2Interior24[3] * fm2 + kD2Interior24[4] * fm1 + kD2Interior24[5] * f0 + kD2Interior24[6] * fp1;
    w.p1 = kD2Interior24[3] * fp2 + kD2Interior24[4] * fp1 + kD2Interior24[5] * f0 + kD2Interior24[6] * fm1;
    w.m2 = kD2Interior24[7] * fm2 + kD2Interior24[8] * fm1 + kD2Interior24[9] * f0;
    w.p2 = kD2Interior24[7] * fp2 + kD2Interior24[8] * fp1 + kD2Interior24[9] * f0;
    return w;
}

// D2 weights of the 4 cells of a quad along x and z (coefficient mu); they depend on the
// model only, so a workgroup forms them once and reuses them for all its shots
struct QuadW {
    W5 x[4], z[4];
};

__device__ __forceinline__ W5 d2_scaled(W5 w, float f)
{
    w.m2 *= f;
    w.m1 *= f;
    w.c *= f;
    w.p1 *= f;
    w.p2 *= f;
    return w;
}

__device__ __forceinline__ float d2_apply(const W5& w, const float* pu, int s)
{
    return w.c * pu[0] + w.m1 * pu[-s] + w.p1 * pu[s] + w.m2 * pu[-2 * s] + w.p2 * pu[2 * s];
}

// ---------------------------------------------------------------------------
// Fused time step
//
// A workgroup owns a 64 (z) x TX (x) tile of the tile grid and advances a group of shots
// through it one after the other, so that the coefficient window and the per-cell factors
// are read once per tile, not once per shot.  Per shot: the state window (halo 4 in x, 8 in
// z) goes straight from global memory into LDS, the products of first derivatives are
// formed on the tile +/- 2 (x) and +/- 4 (z), then each thread computes the new level of its
// quads (4 consecutive z cells; column-major, so that a wavefront covers 4 whole columns).
//
// Tiles whose cells are all interior run without closure code.  The frame of tiles around
// them runs the same phases plus the SBP closures and SAT terms, arranged so that the code
// stays small: closure rows are table-driven loops, not one instance per row.
//   * Along x the closure columns are whole quads: the D2(mu) weights of a closure column's
//     8 points come from a model array (formed once per model), D1 coefficients from an LDS
//     table.
//   * Along z a closure row is part of a quad.  Every quad forms the interior rows, and the
//     closure rows are dealt one cell per thread in passes of their own: the products of
//     rows 0-3 from either side, then the z terms of rows 0-5, and the impedance terms of
//     absorbing left and right sides, which go to the quads' owners through the out-of-grid
//     cells of the state windows.
//   * The SAT terms of a side are part of its boundary row: its D2 weights and its first D1
//     coefficient (see z_cell).
//   * In the rows below a free surface at the top the leapfrog carries, per cell, what the
//     rounding of the new level leaves of its increment to the next step (StepArgs::carry).  Every
//     rounding of a level is a kick that the scheme integrates twice; surface waves meet them all
//     the way and do not spread, and they were nearly the whole error: 14 rows in FP64 bring a
//     one-shot gradient of 1500 steps from 4.8e-6 to 2.3e-7 off FP64.  With the carry such
//     gradients are 1.0 to 1.3e-6 off, 3.0 to 7.0e-6 without.  16 rows are 3% of 500: a step of
//     64 shots takes 391.5 instead of 389.6 us, of one on 201 x 601 11.1 us with or without.
// The instance-per-row form this replaced (34-60 KB of code per kernel, edge bands beside a
// core launch) was bound by instruction fetch: one band workgroup took 30 us alone, and a
// step of one shot on 201 x 601 cells 105 us; it takes 11 us in this form (one launch), and
// 64 shots of 500 x 1700 392 us instead of 407.  A frame tile costs more than an interior one
// in VALU work (at first 1209 against 527 vector instructions per wavefront and shot, most of
// the surplus addresses), so it loads per shot what its passes need and keeps no D2 weights:
// spills cost it more than both.
// ---------------------------------------------------------------------------
template <int TX_>
struct StepShape {
    static constexpr int TX = TX_, TZ = kTileZ;
    static constexpr int HX = 4, HZ = 8;
    static constexpr int WX = TX + 2 * HX;       // state window columns
    static constexpr int WQ = (TZ + 2 * HZ) / 4; // state window quads per column
    static constexpr int WZ = 4 * WQ;            // LDS column stride of the window
    static constexpr int IX = TX + 4;            // product columns
    static constexpr int PQ = (TZ + 8) / 4;      // product quads: rows [sz-4, sz+TZ+4)
    static constexpr int PZ = 4 * PQ;            // LDS column stride of the products
    static constexpr int QC = TZ / 4;            // new-level quads per column
    static constexpr int NQ1 = (WX * WQ + kThreads - 1) / kThreads;  // window quads per thread
    static constexpr int NQ2 = (IX * PQ + kThreads - 1) / kThreads;  // product quads per thread
    static constexpr int NQ3 = TX * QC / kThreads;                   // new-level quads per thread
    static_assert((TX * QC) % kThreads == 0, "tile must give every thread whole quads");
};

struct TileInfo {
    int sx, ex, sz, ez, wsx, wsz, plx, phx, plz, phz, pz0;
};

// new-level quad i of a tile
template <class S>
__device__ __forceinline__ void out_quad(const TileInfo& t, int i, int& gx, int& z0)
{
    gx = t.sx + i / S::QC;
    z0 = t.sz + 4 * (i % S::QC);
}

// D1 rows 0-5 on points 0-7 in LDS (rows 4 and 5 are interior rows), row stride rs; the step's
// table holds as row kSatRow the row 0 of the products, with the SAT terms' share (see z_cell)
constexpr int kSatRow = 6;
struct EdgeTable {
    float* c;
    int rs;
};

struct StepSmem {
    float *ux, *uz, *mu, *mux, *px, *pz, *qx, *qz;
    EdgeTable tb;
};

// D1 of a 12-cell column (cells z0-4 .. z0+7) at the 4 quad cells
__device__ __forceinline__ void d1_quad_z(const float* c, float* out, float c1, float c2)
{
#pragma unroll
    for (int k = 0; k < 4; k++) out[k] = c1 * (c[5 + k] - c[3 + k]) + c2 * (c[6 + k] - c[2 + k]);
}

// D2(c) of a 12-cell column at the 4 quad cells (2 fields sharing the coefficient)
__device__ __forceinline__ void d2_quad_z(const float* m, const float* u1, const float* u2, float* o1, float* o2)
{
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const W5 w = d2_weights(&m[4 + k], 1);
        o1[k] = d2_apply(w, &u1[4 + k], 1);
        o2[k] = d2_apply(w, &u2[4 + k], 1);
    }
}

// i is a multiple of 4: the reads are indexed in quads, so that the compiler knows their
// 16-byte alignment and emits 128-bit LDS reads (not pairs of 64-bit ones, which conflict
// on banks for lanes 16 bytes apart)

__device__ __forceinline__ void load_col12(const float* base, int i, float* c)
{
    const v4f* q = reinterpret_cast<const v4f*>(base) + (i >> 2);
    v4f a = q[-1], b = q[0], d = q[1];
    // whole quads: the compiler would otherwise read only the 8 rows a first derivative
    // uses, as 64-bit LDS reads 8 bytes off the 16-byte grid (2-way bank conflicts)
    __asm__ volatile("" : "+v"(a), "+v"(d));
#pragma unroll
    for (int k = 0; k < 4; k++) {
        c[k] = a[k];
        c[4 + k] = b[k];
        c[8 + k] = d[k];
    }
}

// D1 rows 0-5 from a side on the 8 points next to it: four closure rows and the first two
// interior ones; then the products' row 0, whose first coefficient -24/17 the SAT terms turn into
// 24/17 (+ 1 / H0)
struct EdgeD1 {
    float c[56];
};
constexpr EdgeD1 edge_d1_table()
{
    EdgeD1 t{};
    for (int r = 0; r < 4; r++)
        for (int j = 0; j < 6; j++) t.c[8 * r + j] = (float)kD1Closure[r][j];
    for (int r = 4; r < 6; r++) {
        t.c[8 * r + r - 2] = -kD1InteriorF[1];
        t.c[8 * r + r - 1] = -kD1InteriorF[0];
        t.c[8 * r + r + 1] = kD1InteriorF[0];
        t.c[8 * r + r + 2] = kD1InteriorF[1];
    }
    for (int j = 0; j < 8; j++) t.c[8 * kSatRow + j] = j ? t.c[j] : -t.c[0];
    return t;
}
__constant__ EdgeD1 cEdgeD1 = edge_d1_table();

// ---- table-driven closure rows -------------------------------------------------------
// A closure row of point g of n: the edge point's offset o from g and the inward step st
// along a line of stride s, the row r from the edge, and the sign of D1 there.
struct EdgeRow {
    int o, st, r;
    float sg;
};
__device__ __forceinline__ EdgeRow edge_row(int g, int n, int s)
{
    const bool far = 2 * g >= n;
    const int r = far ? n - 1 - g : g;
    return {(far ? r : -r) * s, far ? -s : s, r, far ? -1.f : 1.f};
}

// D1 (times h) of two fields at point g of n along stride s: interior or closure row
__device__ __forceinline__ void d1_pair(const float* u, const float* v, int s, int g, int n, EdgeTable tb,
                                        float& du, float& dv)
{
    if (g >= 4 && g < n - 4) {
        du = d1_int(u, s);
        dv = d1_int(v, s);
        return;
    }
    const EdgeRow e = edge_row(g, n, s);
    float a = 0.f, b = 0.f;
#pragma unroll
    for (int j = 0; j < 6; j++) {
        const float c = tb.c[tb.rs * e.r + j];
        a += c * u[e.o + j * e.st];
        b += c * v[e.o + j * e.st];
    }
    du = e.sg * a;
    dv = e.sg * b;
}

// The N cells of a column next to its top or bottom cell p, from the side inwards.  They are
// read in memory order (immediate offsets from one address, all in flight at once; a loop
// with the side's step as its stride waits for each) and reversed in registers.
template <int N>
__device__ __forceinline__ void edge_cells(const float* p, bool far, float* e)
{
    const float* b = far ? p - (N - 1) : p;
    float v[N];
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = b[i];
#pragma unroll
    for (int j = 0; j < N; j++) e[j] = far ? v[N - 1 - j] : v[j];
}
__device__ __forceinline__ void edge_coefficients(EdgeTable tb, int r, float* c)
{
    unpack(ld4(tb.c + tb.rs * r), c);
    unpack(ld4(tb.c + tb.rs * r + 4), c + 4);
}
// D1 along z (times h) of closure row r from the top or bottom, whose boundary cell is p;
// c: the row's coefficients
__device__ __forceinline__ float d1z_closure(const float* p, bool far, const float* c)
{
    float e[6], v = 0.f;
    edge_cells<6>(p, far, e);
#pragma unroll
    for (int j = 0; j < 6; j++) v += c[j] * e[j];
    return far ? -v : v;
}

// D1 along x (times h) of two fields at the 4 cells of a quad of a closure column (rows 0-3
// from a side), column stride CS
template <int CS>
__device__ __forceinline__ void d1_quad_closure(const float* u, const float* v, int gx, int nx, EdgeTable tb,
                                                float* du, float* dv)
{
    const EdgeRow e = edge_row(gx, nx, CS);
#pragma unroll
    for (int k = 0; k < 4; k++) du[k] = dv[k] = 0.f;
#pragma unroll 2
    for (int j = 0; j < 6; j++) {
        const float c = e.sg * tb.c[tb.rs * e.r + j];
        float U[4], V[4];
        unpack(ld4(u + e.o + j * e.st), U);
        unpack(ld4(v + e.o + j * e.st), V);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            du[k] += c * U[k];
            dv[k] += c * V[k];
        }
    }
}

// ---- products of first derivatives on one quad --------------------------------------
template <bool VTI>
__device__ __forceinline__ void products(const float* lam, const float* lamx, const float* c13, const float* mu,
                                         const float* dxux, const float* dxuz, const float* dzux, const float* dzuz,
                                         int k, float* p, float* pz, float* qx, float* qz)
{
    if (!VTI) {
        p[k] = lam[k] * (dxux[k] + dzuz[k]);
        pz[k] = 0.f;
    } else {
        p[k] = lamx[k] * dxux[k] + c13[k] * dzuz[k];
        pz[k] = lam[k] * dzuz[k] + c13[k] * dxux[k];
    }
    qx[k] = mu[k] * dxuz[k];
    qz[k] = mu[k] * dzux[k];
}

// z rows by the interior stencil whatever the row: in frame tiles product_pass replaces the
// closure rows
template <bool VTI, class S, bool EDGE>
__device__ __forceinline__ void product_quad(const StepArgs& a, const StepSmem& sm, const TileInfo& t, int gx, int z0,
                                             float4 lam4, float4 lamx4, float4 c134, float* p, float* pz, float* qx,
                                             float* qz)
{
    const int w = (gx - t.wsx) * S::WZ + (z0 - t.wsz);
    float dxux[4], dxuz[4], dzux[4], dzuz[4];
    if (!EDGE || (gx >= 4 && gx < a.nx - 4)) {
        float X[4][4], Z[4][4];
        const int off[4] = {-2, -1, 1, 2};
#pragma unroll
        for (int c = 0; c < 4; c++) {
            unpack(ld4(&sm.ux[w + off[c] * S::WZ]), X[c]);
            unpack(ld4(&sm.uz[w + off[c] * S::WZ]), Z[c]);
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            dxux[k] = a.c1x * (X[2][k] - X[1][k]) + a.c2x * (X[3][k] - X[0][k]);
            dxuz[k] = a.c1x * (Z[2][k] - Z[1][k]) + a.c2x * (Z[3][k] - Z[0][k]);
        }
    } else if constexpr (EDGE) {
        d1_quad_closure<S::WZ>(&sm.ux[w], &sm.uz[w], gx, a.nx, sm.tb, dxux, dxuz);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            dxux[k] *= a.rdx;
            dxuz[k] *= a.rdx;
        }
    }
    {
        float Uc[12], Zc[12];
        load_col12(sm.ux, w, Uc);
        load_col12(sm.uz, w, Zc);
        d1_quad_z(Uc, dzux, a.c1z, a.c2z);
        d1_quad_z(Zc, dzuz, a.c1z, a.c2z);
    }
    float mu[4], lam[4], lamx[4], c13[4];
    unpack(ld4(&sm.mu[w]), mu);
    unpack(lam4, lam);
    unpack(lamx4, lamx);
    unpack(c134, c13);
#pragma unroll
    for (int k = 0; k < 4; k++)
        products<VTI>(lam, lamx, c13, mu, dxux, dxuz, dzux, dzuz, k, p, pz, qx, qz);
}

// Frame tiles at the top or bottom: the products of the closure rows (0-3 from the side)
// over the tile's product columns, one cell per thread: cell c of the pass, whose model
// values are loaded ahead of the shot's window.
struct PCell {
    int gx, gz;
    float lam, lamx, c13;
};
template <bool VTI, class S>
__device__ __forceinline__ bool p_cell(const StepArgs& a, const TileInfo& t, int c, bool top, bool bot, PCell& e)
{
    constexpr int per = 4 * S::IX;
    if (c >= (top + bot) * per) return false;
    const bool far = !top || c >= per;
    const int i = c - (top && far ? per : 0);
    e.gx = t.plx + (i >> 2);
    e.gz = far ? a.nz - 1 - (i & 3) : i & 3;
    if (e.gx >= t.phx) return false;
    const int g = e.gx * a.ldz + e.gz;
    e.lam = a.lam[g];
    if (VTI) {
        e.lamx = a.lamx[g];
        e.c13 = a.c13[g];
    }
    return true;
}
template <bool VTI, class S>
__device__ __forceinline__ void p_cell_run(const StepArgs& a, const StepSmem& sm, const TileInfo& t, const PCell& e)
{
    const int w = (e.gx - t.wsx) * S::WZ + (e.gz - t.wsz);
    float dxux, dxuz, dzux, dzuz;
    d1_pair(&sm.ux[w], &sm.uz[w], S::WZ, e.gx, a.nx, sm.tb, dxux, dxuz);
    const bool far = e.gz >= 4;
    const int r = far ? a.nz - 1 - e.gz : e.gz, wb = w + (far ? r : -r);
    float c[8];
    edge_coefficients(sm.tb, r, c);
    dzux = d1z_closure(&sm.ux[wb], far, c);
    dzuz = d1z_closure(&sm.uz[wb], far, c);
    dxux *= a.rdx;
    dxuz *= a.rdx;
    dzux *= a.rdz;
    dzuz *= a.rdz;
    const float mu = sm.mu[w];
    float p, pz, qx, qz;
    products<VTI>(&e.lam, &e.lamx, &e.c13, &mu, &dxux, &dxuz, &dzux, &dzuz, 0, &p, &pz, &qx, &qz);
    const int o = (e.gx - t.plx) * S::PZ + (e.gz - t.pz0);
    sm.px[o] = p;
    if (VTI) sm.pz[o] = pz;
    sm.qx[o] = qx;
    sm.qz[o] = qz;
}

// The passes hand their terms to the quads' owners through cells of the state window outside
// the grid, which no result that is used reads: the term of a top row 8 window rows above
// its cell, of a bottom row 8 below, of a left or right boundary cell one column outside; x
// component in the ux window, z component in the uz window.
constexpr int kTermRows = 8;

// previous level at one cell, tapered as the step takes it
__device__ __forceinline__ void prev_at(const StepArgs& a, const float* prev, long long nxz, int gx, int gz, float& px,
                                        float& pz)
{
    const int g = gx * a.ldz + gz;
    px = prev[g];
    pz = prev[nxz + g];
    if (a.taper_prev) {
        px = (px * a.taper_z[gz]) * a.taper_x[gx];
        pz = (pz * a.taper_z[gz]) * a.taper_x[gx];
    }
}

// The z part of the right-hand side (D2z[mu] ux, 2 D2z[mu] uz, Dz of the products) of the
// closure rows 0-5 from the top or bottom, one cell per thread, with the SAT terms of that side
// on the boundary row (we_op.cpp:726-774, 1705-1752).  Those are minus the boundary derivative,
// which the row's D2 weights hold, and, for the traction's derivatives along the side and the
// scheme's complement term together, plus the products there over H0 h: that turns the row's
// first D1 coefficient -24/17 into 24/17.  Absorbing sides add the impedance term of the
// previous level.  Cell c of the pass, whose D2 weights and boundary values are loaded ahead
// of the shot's window.
struct ZCell {
    int gx, r;
    bool bot;
    float w[8], lam, rho, prx, prz;
};
template <class S>
__device__ __forceinline__ bool z_cell(const StepArgs& a, const TileInfo& t, int c, bool top, bool bot,
                                       const float* prev, long long nxz, ZCell& e)
{
    constexpr int per = 6 * S::TX;
    if (c >= (top + bot) * per) return false;
    e.bot = !top || c >= per;
    const int i = c - (top && e.bot ? per : 0);
    e.r = i / S::TX;
    e.gx = t.sx + i % S::TX;
    if (e.gx >= t.ex) return false;
    // weights [side][nx][6 rows][8 points], divided by dz^2
    const float* W = a.wz + ((size_t)((e.bot ? a.nx : 0) + e.gx) * 6 + e.r) * 8;
    unpack(ld4(W), e.w);
    unpack(ld4(W + 4), e.w + 4);
    if (e.r == 0 && (e.bot ? a.bc_bottom : a.bc_top) == 2) {
        const int gz = e.bot ? a.nz - 1 : 0, g = e.gx * a.ldz + gz;
        e.lam = a.lam[g];
        e.rho = a.rho[g];
        prev_at(a, prev, nxz, e.gx, gz, e.prx, e.prz);
    }
    return true;
}
template <bool VTI, class S>
__device__ __forceinline__ void z_cell_run(const StepArgs& a, const StepSmem& sm, const TileInfo& t, const ZCell& e)
{
    const int st = e.bot ? -1 : 1, edge = e.bot ? a.nz - 1 : 0;
    const int w = (e.gx - t.wsx) * S::WZ + (edge - t.wsz);  // the boundary cell
    const int q = (e.gx - t.plx) * S::PZ + (edge - t.pz0);
    float c[8], ux[8], uz[8], v[8];
    edge_coefficients(sm.tb, e.r ? e.r : kSatRow, c);
    edge_cells<8>(&sm.ux[w], e.bot, ux);
    edge_cells<8>(&sm.uz[w], e.bot, uz);
    float d2x = 0.f, d2z = 0.f, dp = 0.f, dq = 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        d2x += e.w[j] * ux[j];
        d2z += e.w[j] * uz[j];
    }
    edge_cells<8>((VTI ? sm.pz : sm.px) + q, e.bot, v);
#pragma unroll
    for (int j = 0; j < 8; j++) dp += c[j] * v[j];
    edge_cells<8>(sm.qx + q, e.bot, v);
#pragma unroll
    for (int j = 0; j < 8; j++) dq += c[j] * v[j];
    const float sg = e.bot ? -a.rdz : a.rdz;
    float rx = d2x + sg * dq, rz = 2.f * d2z + sg * dp;
    if (e.r == 0 && (e.bot ? a.bc_bottom : a.bc_top) == 2) {
        const float mu0 = sm.mu[w];
        rx += a.sat_z * ((0.5f * sqrtf(mu0 * e.rho)) * e.prx / a.dt);
        rz += a.sat_z * ((0.5f * sqrtf((e.lam + 2.f * mu0) * e.rho)) * e.prz / a.dt);
    }
    const int o = w + st * (e.r - kTermRows);
    sm.ux[o] = rx;
    sm.uz[o] = rz;
}

// The impedance terms of absorbing left and right boundary columns of a tile (we_op.cpp:776-822,
// 1754-1800; the SAT's other terms are in the columns' D2 weights and D1 coefficients, as along
// z), one cell per thread.
template <bool VTI, class S>
__device__ __forceinline__ void x_sat_pass(const StepArgs& a, const StepSmem& sm, const TileInfo& t, int tid,
                                           bool left, bool right, const float* prev, long long nxz)
{
    for (int c = tid; c < 2 * S::TZ; c += kThreads) {
        const bool rt = c >= S::TZ;
        const int gz = t.sz + (rt ? c - S::TZ : c);
        if (!(rt ? right : left) || gz >= t.ez) continue;
        const int gx = rt ? a.nx - 1 : 0, sn = rt ? -S::WZ : S::WZ;
        const int w = (gx - t.wsx) * S::WZ + (gz - t.wsz), g = gx * a.ldz + gz;
        const float mu0 = sm.mu[w], lam0 = a.lam[g], rho0 = a.rho[g];
        const float epsf = VTI ? 1.f + 2.f * a.eps[g] : 1.f;
        float prx, prz;
        prev_at(a, prev, nxz, gx, gz, prx, prz);
        sm.ux[w - sn] = a.sat_x * ((0.5f * sqrtf(epsf * (lam0 + 2.f * mu0) * rho0)) * prx / a.dt);
        sm.uz[w - sn] = a.sat_x * ((0.5f * sqrtf(mu0 * rho0)) * prz / a.dt);
    }
}

// ---- right-hand side of one quad before sources: volume terms (we_op.cpp:690-720,
// 1665-1700).  Frame tiles (EDGE): the x part in rx, rz and the z part by the interior rows
// in zx, zz, for frame_terms to complete ------------------------------------------------
template <bool VTI, class S, bool EDGE, bool CW>
__device__ __forceinline__ void rhs_quad(const StepArgs& a, const StepSmem& sm, const TileInfo& t, int gx, int z0,
                                         float* rx, float* rz, float* zx, float* zz, const QuadW& qw)
{
    const int nx = a.nx, nz = a.nz;
    const int w = (gx - t.wsx) * S::WZ + (z0 - t.wsz);
    const int q = (gx - t.plx) * S::PZ + (z0 - t.pz0);
    // x part: D2x[2mu or 2(1+2eps)mu] ux, D2x[mu] uz, Dx of the products
    if (!EDGE || (gx >= 6 && gx < nx - 6)) {
        float U[5][4], Z[5][4], M[CW ? 1 : 5][4], MX[VTI ? 5 : 1][4];
#pragma unroll
        for (int c = 0; c < 5; c++) {
            unpack(ld4(&sm.ux[w + (c - 2) * S::WZ]), U[c]);
            unpack(ld4(&sm.uz[w + (c - 2) * S::WZ]), Z[c]);
            if (!CW) unpack(ld4(&sm.mu[w + (c - 2) * S::WZ]), M[c]);
            if (VTI) unpack(ld4(&sm.mux[w + (c - 2) * S::WZ]), MX[c]);
        }
        float P[4][4], Q[4][4];
        const int off[4] = {-2, -1, 1, 2};
#pragma unroll
        for (int c = 0; c < 4; c++) {
            unpack(ld4(&sm.px[q + off[c] * S::PZ]), P[c]);
            unpack(ld4(&sm.qz[q + off[c] * S::PZ]), Q[c]);
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float uk[5] = {U[0][k], U[1][k], U[2][k], U[3][k], U[4][k]};
            const float zk[5] = {Z[0][k], Z[1][k], Z[2][k], Z[3][k], Z[4][k]};
            W5 wx;
            if constexpr (CW) {
                wx = qw.x[k];
            } else {
                const float mk[5] = {M[CW ? 0 : 0][k], M[CW ? 0 : 1][k], M[CW ? 0 : 2][k], M[CW ? 0 : 3][k],
                                     M[CW ? 0 : 4][k]};
                wx = d2_weights(&mk[2], 1);
            }
            float d2u;
            if (VTI) {
                const float xk[5] = {MX[0][k], MX[1][k], MX[2][k], MX[3][k], MX[4][k]};
                d2u = d2_apply(d2_weights(&xk[2], 1), &uk[2], 1);
            } else {
                d2u = d2_apply(wx, &uk[2], 1);
            }
            if constexpr (CW) {  // cached weights already carry 1/dx^2
                rx[k] = 2.f * d2u;
                rz[k] = d2_apply(wx, &zk[2], 1);
            } else {
                rx[k] = 2.f * d2u * a.rdx2;
                rz[k] = d2_apply(wx, &zk[2], 1) * a.rdx2;
            }
            rx[k] += a.c1x * (P[2][k] - P[1][k]) + a.c2x * (P[3][k] - P[0][k]);
            rz[k] += a.c1x * (Q[2][k] - Q[1][k]) + a.c2x * (Q[3][k] - Q[0][k]);
        }
    } else if constexpr (EDGE) {
        // closure column r from a side: weights [side][column][point][ldz], divided by dx^2
        const EdgeRow e = edge_row(gx, nx, 1);
        const size_t wo = (size_t)((gx >= 6 ? 6 : 0) + e.r) * 8 * a.ldz + z0;
        const float *W = a.wx + wo, *WX = VTI ? a.wxx + wo : W;
        const float* crow = sm.tb.c + sm.tb.rs * (e.r ? e.r : kSatRow);
        float d2u[4], d2z[4], dp[4], dq[4];
#pragma unroll
        for (int k = 0; k < 4; k++) d2u[k] = d2z[k] = dp[k] = dq[k] = 0.f;
#pragma unroll 2
        for (int j = 0; j < 8; j++) {
            const int o = e.o + j * e.st;
            const float c = crow[j];
            float wj[4], xj[4], U[4], Z[4];
            unpack(ld4(W + (size_t)j * a.ldz), wj);
            if (VTI) unpack(ld4(WX + (size_t)j * a.ldz), xj);
            unpack(ld4(&sm.ux[w + o * S::WZ]), U);
            unpack(ld4(&sm.uz[w + o * S::WZ]), Z);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                d2u[k] += (VTI ? xj[k] : wj[k]) * U[k];
                d2z[k] += wj[k] * Z[k];
            }
            if (c != 0.f) {  // the other points may lie before the product columns
                float P[4], Q[4];
                unpack(ld4(&sm.px[q + o * S::PZ]), P);
                unpack(ld4(&sm.qz[q + o * S::PZ]), Q);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    dp[k] += c * P[k];
                    dq[k] += c * Q[k];
                }
            }
        }
        const float sg = e.sg * a.rdx;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            rx[k] = 2.f * d2u[k] + sg * dp[k];
            rz[k] = d2z[k] + sg * dq[k];
        }
    }
    // z part: D2z[2mu] uz, D2z[mu] ux, Dz of the products
    if (EDGE) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < 4; k++) zx[k] = zz[k] = 0.f;
    }
    {
        float Uc[12], Zc[12], d2zx[4], d2zz[4];
        load_col12(sm.ux, w, Uc);
        load_col12(sm.uz, w, Zc);
        if constexpr (CW) {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                d2zz[k] = d2_apply(qw.z[k], &Zc[4 + k], 1);
                d2zx[k] = d2_apply(qw.z[k], &Uc[4 + k], 1);
            }
        } else {
            float Mc[12];
            load_col12(sm.mu, w, Mc);
            d2_quad_z(Mc, Zc, Uc, d2zz, d2zx);
        }
        float Pc[12], Qc[12], dpz[4], dqz[4];
        load_col12(VTI ? sm.pz : sm.px, q, Pc);
        load_col12(sm.qx, q, Qc);
        d1_quad_z(Pc, dpz, a.c1z, a.c2z);
        d1_quad_z(Qc, dqz, a.c1z, a.c2z);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if constexpr (CW) {  // cached weights already carry 1/dz^2
                zz[k] += 2.f * d2zz[k];
                zx[k] += d2zx[k];
            } else {
                zz[k] += 2.f * d2zz[k] * a.rdz2;
                zx[k] += d2zx[k] * a.rdz2;
            }
            zz[k] += dpz[k];
            zx[k] += dqz[k];
        }
    }
}

// Frame tiles: the z part of one quad with its closure rows, and the left and right SAT terms
template <class S>
__device__ __forceinline__ void frame_terms(const StepArgs& a, const StepSmem& sm, const TileInfo& t, int gx, int z0,
                                            float* rx, float* rz, float* zx, float* zz)
{
    const int nx = a.nx, nz = a.nz;
    const int w = (gx - t.wsx) * S::WZ + (z0 - t.wsz);
    float tx[4], tz[4];
    if (z0 < 6) {  // quads 0 and 4: rows 0-5
        unpack(ld4(&sm.ux[w - kTermRows]), tx);
        unpack(ld4(&sm.uz[w - kTermRows]), tz);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            zx[k] = k < 2 || z0 == 0 ? tx[k] : zx[k];
            zz[k] = k < 2 || z0 == 0 ? tz[k] : zz[k];
        }
    }
    if (z0 + 3 >= nz - 6) {  // (nz 12 and 13: a quad holds rows of both sides)
        unpack(ld4(&sm.ux[w + kTermRows]), tx);
        unpack(ld4(&sm.uz[w + kTermRows]), tz);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            zx[k] = z0 + k >= nz - 6 ? tx[k] : zx[k];
            zz[k] = z0 + k >= nz - 6 ? tz[k] : zz[k];
        }
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
        rx[k] += zx[k];
        rz[k] += zz[k];
    }
    if ((gx == 0 && a.bc_left == 2) || (gx == nx - 1 && a.bc_right == 2)) {
        const int o = gx == 0 ? w - S::WZ : w + S::WZ;
        unpack(ld4(&sm.ux[o]), tx);
        unpack(ld4(&sm.uz[o]), tz);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            rx[k] += tx[k];
            rz[k] += tz[k];
        }
    }
}

// First derivatives of a pair of fields (u, v) at the 4 cells of a quad from an LDS
// array with column stride CS: (dx u, dz u, dx v, dz v), scaled by 1/h.  In frame tiles
// (EDGE) the z derivatives of the closure rows come from d1z_pass: u and v are arrays whose
// rows start H above the tile, row0 their index of the quad's column at the tile's row 0.
template <bool EDGE, int CS>
__device__ __forceinline__ void quad_derivs(const StepArgs& a, const float* u, const float* v, int w, int row0, int gx,
                                            int z0, EdgeTable tb, float* xu, float* zu, float* xv, float* zv)
{
    const int nx = a.nx, nz = a.nz;
    if (!EDGE || (gx >= 4 && gx < nx - 4)) {
        float U[4][4], V[4][4];
        const int off[4] = {-2, -1, 1, 2};
#pragma unroll
        for (int c = 0; c < 4; c++) {
            unpack(ld4(&u[w + off[c] * CS]), U[c]);
            unpack(ld4(&v[w + off[c] * CS]), V[c]);
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            xu[k] = a.c1x * (U[2][k] - U[1][k]) + a.c2x * (U[3][k] - U[0][k]);
            xv[k] = a.c1x * (V[2][k] - V[1][k]) + a.c2x * (V[3][k] - V[0][k]);
        }
    } else if constexpr (EDGE) {
        d1_quad_closure<CS>(u + w, v + w, gx, nx, tb, xu, xv);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            xu[k] *= a.rdx;
            xv[k] *= a.rdx;
        }
    }
    {
        float Uc[12], Vc[12];
        load_col12(u, w, Uc);
        load_col12(v, w, Vc);
        d1_quad_z(Uc, zu, a.c1z, a.c2z);
        d1_quad_z(Vc, zv, a.c1z, a.c2z);
    }
    if constexpr (EDGE) {
        if (z0 < 4 || z0 + 3 >= nz - 4) {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int gz = z0 + k;
                const bool bot = gz >= 4;
                if ((bot && gz < nz - 4) || gz >= nz) continue;
                const int i = row0 + (bot ? kTileZ + nz - 1 - gz : gz - 4);
                zu[k] = u[i];
                zv[k] = v[i];
            }
        }
    }
}

// Frame tiles at the top or bottom: the z derivatives (times 1/h) of two fields on the
// closure rows 0-3 from the side, one cell per thread, into the arrays' rows outside the
// grid: row r of the top at r - 4, of the bottom at r below the tile.  u and v have column
// stride CS and first column wx; row0 is their index of the first tile column's row 0.
template <int TX, int CS>
__device__ __forceinline__ void d1z_pass(const StepArgs& a, float* u, float* v, int row0, int sx, int ex, int sz,
                                         int tid, bool near, bool far, EdgeTable tb)
{
    constexpr int per = 4 * TX;
    for (int c = tid; c < (near + far) * per; c += kThreads) {
        const bool bot = !near || c >= per;
        const int i = c - (near && bot ? per : 0);
        const int col = i >> 2, r = i & 3;
        if (sx + col >= ex) continue;
        const int w = row0 + col * CS, wb = w + (bot ? a.nz - 1 : 0) - sz;
        float cf[8];
        edge_coefficients(tb, r, cf);
        const float du = d1z_closure(&u[wb], bot, cf), dv = d1z_closure(&v[wb], bot, cf);
        u[w + (bot ? kTileZ + r : r - 4)] = du * a.rdz;
        v[w + (bot ? kTileZ + r : r - 4)] = dv * a.rdz;
    }
}

// Imaging condition of one quad (compute_gradients, we_op.cpp:519-561): a* are the
// derivatives of the lagged adjoint level (x_x, x_z, z_x, z_z), t* those of forward
// snapshot idx (x_x, z_z, z_x, x_z), f0/fm/fp the snapshots idx, idx-1, idx+1 at the
// cells, o the adjoint level of the density term.  Adds to the accumulators of the
// lambda, mu, rho gradients (VTI stiffness mode: c11, c13, c33, c55, rho).
//
// Density term of the imaging condition of one quad: o is the adjoint level after the
// step, f0/fm/fp the snapshots idx, idx-1, idx+1 at the cells (second time difference;
// one-sided at the first and last snapshot, mode 1 and 2).  It goes to gr, or to g4 in
// the VTI stiffness mode.  (The accumulators are updated unconditionally with selected
// values: a branch on the mode that picks the array would put the arrays in scratch.)
template <bool VTI>
__device__ __forceinline__ void image_rho(const StepArgs& a, int z0, const float* f0x, const float* f0z,
                                          const float* fmx, const float* fmz, const float* fpx, const float* fpz,
                                          const float* ox, const float* oz, float* gr, float* g4)
{
    const bool st = VTI && a.stiff;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        if (z0 + k >= a.nz) continue;
        float d2x, d2z;
        if (a.img_mode == 0) {
            d2x = fpx[k] - 2.f * f0x[k] + fmx[k];
            d2z = fpz[k] - 2.f * f0z[k] + fmz[k];
        } else if (a.img_mode == 1) {
            d2x = fpx[k] - f0x[k];
            d2z = fpz[k] - f0z[k];
        } else {
            d2x = -f0x[k] + fmx[k];
            d2z = -f0z[k] + fmz[k];
        }
        const float r = a.wrho * (ox[k] * d2x + oz[k] * d2z);
        if (VTI) {
            gr[k] += st ? 0.f : r;
            g4[k] += st ? r : 0.f;
        } else {
            gr[k] += r;
        }
    }
}

// Stiffness terms of the imaging condition of one quad: a* are the derivatives of the
// lagged adjoint level (x_x, x_z, z_x, z_z), t* those of forward snapshot idx (x_x,
// z_z, z_x, x_z).  Adds to the lambda and mu accumulators gl, gm; in the VTI stiffness
// mode to the c11, c13, c33, c55 accumulators gl, gm, gr, g3.
template <bool VTI>
__device__ __forceinline__ void image_stiff(const StepArgs& a, long long g, int z0, const float* axx, const float* azx,
                                            const float* axz, const float* azz, const float* t0x, const float* t1z,
                                            const float* t2x, const float* t3z, float* gl, float* gm, float* gr,
                                            float* g3)
{
    const bool st = VTI && a.stiff;
    float e[4], v2[4], v3[4];
    if (VTI && !st) {
        unpack(ld4(a.ge + g), e);
        unpack(ld4(a.gv2 + g), v2);
        unpack(ld4(a.gv3 + g), v3);
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
        if (z0 + k >= a.nz) continue;
        const float shear = (azx[k] + axz[k]) * (t2x[k] + t3z[k]);
        if (!VTI) {
            gl[k] += a.wlm * (axx[k] + azz[k]) * (t0x[k] + t1z[k]);
            gm[k] += a.wlm * (shear + 2.f * axx[k] * t0x[k] + 2.f * azz[k] * t1z[k]);
        } else {
            const float xx = axx[k] * t0x[k], zz = azz[k] * t1z[k];
            const float cr = axx[k] * t1z[k] + azz[k] * t0x[k];
            // stiffness mode: d/dc11, d/dc13, d/dc33, d/dc55 of the same bilinear form
            const float dl = st ? xx : e[k] * xx + zz + v2[k] * cr;
            const float dm = st ? cr : shear + 2.f * e[k] * xx + 2.f * zz + v3[k] * cr;
            gl[k] += a.wlm * dl;
            gm[k] += a.wlm * dm;
            gr[k] += st ? a.wlm * zz : 0.f;
            g3[k] += st ? a.wlm * shear : 0.f;
        }
    }
}

// Imaging condition of one quad (compute_gradients, we_op.cpp:519-561) into the
// accumulators of the lambda, mu, rho gradients (VTI stiffness mode: c11, c13, c33, c55,
// rho in gl, gm, gr, g3, g4).
template <bool VTI>
__device__ __forceinline__ void image_accumulate(const StepArgs& a, long long g, int z0, const float* axx,
                                                 const float* azx, const float* axz, const float* azz,
                                                 const float* t0x, const float* t1z, const float* t2x,
                                                 const float* t3z, const float* f0x, const float* f0z,
                                                 const float* fmx, const float* fmz, const float* fpx,
                                                 const float* fpz, const float* ox, const float* oz, float* gl,
                                                 float* gm, float* gr, float* g3, float* g4)
{
    image_stiff<VTI>(a, g, z0, axx, azx, axz, azz, t0x, t1z, t2x, t3z, gl, gm, gr, g3);
    image_rho<VTI>(a, z0, f0x, f0z, fmx, fmz, fpx, fpz, ox, oz, gr, g4);
}

// Hides a value from the optimiser so that address arithmetic derived from it is
// recomputed inside the shot loop instead of being hoisted out and kept live in
// registers across it (which multiplies the register footprint of the loop body).
__device__ __forceinline__ void opaque(int& v) { __asm__ volatile("" : "+s"(v)); }
template <class I>
__device__ __forceinline__ void opaque_v(I& v) { __asm__ volatile("" : "+v"(v)); }
__device__ __forceinline__ void opaque(TileInfo& t)
{
    opaque(t.sx);
    opaque(t.ex);
    opaque(t.sz);
    opaque(t.ez);
    opaque(t.wsx);
    opaque(t.wsz);
    opaque(t.plx);
    opaque(t.phx);
    opaque(t.plz);
    opaque(t.phz);
    opaque(t.pz0);
}

// 16 zero bytes: the source of direct-to-LDS window loads at positions outside the grid
__device__ __attribute__((aligned(16))) float kZeroQuad[4] = {0.f, 0.f, 0.f, 0.f};

// One quad of a window straight from global memory into LDS (global_load_lds_dwordx4):
// lane l of the wavefront writes the 16 bytes at lds_wave + 16 l, lds_wave being the
// same for all lanes of the wavefront.
__device__ __forceinline__ void quad_to_lds(const float* src, float* lds_wave)
{
    __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)lds_wave, 16, 0, 0);
}

// receiver component k of 2 nrec (receiver k / 2): its footprints of one level into its trace
__device__ __forceinline__ void extract_component(int k, const float* state, long long shot_stride, long long nxz,
                                                  int ldz, const PointEntry* ents, const int* rptr, float* trace,
                                                  int it)
{
    const int r = k >> 1, comp = k & 1;
    float v = 0.f;
    long long out = 0;
    for (int f = rptr[r]; f < rptr[r + 1]; f++) {
        const PointEntry en = ents[f];
        const float* u = state + en.shot * shot_stride + comp * nxz;
        for (int ix = 0; ix < 3; ix++)
            for (int iz = 0; iz < 3; iz++) v += en.wx[ix] * en.wz[iz] * u[(long long)(en.xi0 + ix) * ldz + en.zi0 + iz];
        out = comp ? en.tz : en.trace;
    }
    if (rptr[r + 1] > rptr[r]) trace[out + it] = v;
}

// Point sources (we_op.cpp:722-724), added to the new level once it is stored: cells c0, c0 +
// 256, ... before c1, one thread per touched cell summing its contributions in injector order.  The step
// forms next = (dt^2/rho (r + s) + 2 curr - prev) / d * taper, which is linear in the
// source term s, so the sources add dt^2/rho * s / d * taper (d: the absorbing divisor on
// the perimeter, 1 elsewhere).  img: the imaging fused into the step took the new level before this increment;
// its share of the density term by parts, wn f0 . (increment), goes to the shot's own slab.
__device__ __forceinline__ void inject_cells(const StepArgs& a, int c0, int c1, bool img, long long nxz)
{
    const PointTable& pt = *a.points;
    const int nx = a.nx, nz = a.nz, ldz = a.ldz;
    for (int c = c0; c < c1; c += kThreads) {
        const InjCell cell = pt.cells[c];
        float fx = 0.f, fz = 0.f;
        for (int k = pt.ptr[c]; k < pt.ptr[c + 1]; k++) {
            fx += pt.w[k] * a.inj_trace[pt.ctx[k] + a.it];
            fz += pt.w[k] * a.inj_trace[pt.ctz[k] + a.it];
        }
        const int gx = cell.gx, gz = cell.gz;
        const long long g = (long long)gx * ldz + gz;
        float dx = 1.f, dz = 1.f;
        if (gz == 0) { dx = a.div_tb[gx]; dz = a.div_tb[nx + gx]; }
        else if (gz == nz - 1) { dx = a.div_tb[2 * nx + gx]; dz = a.div_tb[3 * nx + gx]; }
        else if (gx == 0) { dx = a.div_lr[gz]; dz = a.div_lr[ldz + gz]; }
        else if (gx == nx - 1) { dx = a.div_lr[2 * ldz + gz]; dz = a.div_lr[3 * ldz + gz]; }
        const float f = a.irho[g] * a.taper_z[gz] * a.taper_x[gx];
        const float ix = f * fx / dx, iz = f * fz / dz;
        float* u = a.next + cell.shot * a.shot_stride + g;
        const float ux = u[0], uz = u[nxz], nx1 = ux + ix, nz1 = uz + iz;
        u[0] = nx1;
        u[nxz] = nz1;
        if (a.carry && gz < kCarryRows) {
            float* e = a.carry + ((cell.shot * 2LL) * nx + gx) * kCarryRows + gz;
            e[0] += ix - (nx1 - ux);
            e[(long long)nx * kCarryRows] += iz - (nz1 - uz);
        }
        if (img) {
            const long long fo = cell.shot * a.fshot_stride + g;
            a.grad[cell.shot * a.gslab_stride + (a.stiff ? 4 : 2) * nxz + g] +=
                a.wn * (ix * a.f0[fo] + iz * a.f0[fo + nxz]);
        }
    }
}

// The point sources and receivers of a step in a launch of their own (the sources go into
// the new level, the receivers read the current one): blocks [0, nsrc) the sources' cells,
// the others the receivers' components.
__global__ void __launch_bounds__(kThreads) k_points(const StepArgs a, int ncell, int nsrc, int img)
{
    const long long nxz = (long long)a.nx * a.ldz;
    if ((int)blockIdx.x < nsrc) {
        const int c = blockIdx.x * kThreads + threadIdx.x;
        inject_cells(a, c, min(c + 1, ncell), img != 0, nxz);
    } else {
        const int k = (blockIdx.x - nsrc) * kThreads + threadIdx.x;
        if (k < 2 * a.nrec)
            extract_component(k, a.curr, a.shot_stride, nxz, a.ldz, a.points->rec, a.points->rec_ptr, a.rec_trace, a.it);
    }
}

// One tile and shot group of a time step (see above).  EDGE: a frame tile.
// IMG (the image_fused option; by default the imaging runs in k_img): adjoint step it with
// the imaging by parts in time fused in (see k_img with SBP): the density term of
// snapshot j = f0 against wn next + wc curr + wp prev at the cells (prev as stored, before
// the step's taper; next before the step's point sources, whose share inject_cells
// adds), and the stiffness terms of snapshot j-1 = fm, whose derivatives meet those of the
// step's current level (the reference's lag).  fm's window goes through the LDS of the
// products once the new level is done.  The gradient contributions of the workgroup's
// shots are summed in registers and added once per launch to the gradient slab of the
// group's first shot.
template <bool VTI, class S, bool EDGE, bool IMG, bool PTS>
__device__ __forceinline__ void step_tile(const StepArgs& a, const StepSmem& sm, int tix, int tiz, int s0, int s1)
{
    const int* const tile_ptr = PTS ? a.points->tile_ptr + (tix * a.ntz + tiz) * a.nshots : nullptr;
    // IMG: snapshot fm's window in the product layout, over the products (dead by then)
    float* const sFx = sm.px;
    float* const sFz = sm.qx;
    TileInfo t;
    const int nx = a.nx, nz = a.nz, ldz = a.ldz;
    tile_range_x_hd(tix, a.ntx, S::TX, nx, t.sx, t.ex);
    tile_range_z_hd(tiz, a.ntz, nz, ldz, t.sz, t.ez);
    t.wsx = window_start(t.sx, S::HX);
    t.wsz = t.sz - S::HZ;
    t.pz0 = t.sz - 4;
    product_range(t.sx, t.ex, nx, t.plx, t.phx);
    product_range(t.sz, t.ez, nz, t.plz, t.phz);
    // closure rows in the tile
    const bool top = EDGE && t.sz == 0, bot = EDGE && tiz == a.ntz - 1;
    const bool left = EDGE && t.sx == 0 && a.bc_left == 2, right = EDGE && tix == a.ntx - 1 && a.bc_right == 2;
    const long long nxz = (long long)nx * ldz;
    const int tid = threadIdx.x;

    // ---- per tile: coefficient window, product coefficients, new-level factors ----
#pragma unroll
    for (int m = 0; m < S::NQ1; m++) {
        const int i = tid + m * kThreads;
        if (i < S::WX * S::WQ) {
            const int lx = i / S::WQ, lq = i - lx * S::WQ;
            const int gx = t.wsx + lx, gz = t.wsz + 4 * lq;
            const bool ok = gx >= 0 && gx < nx && gz >= 0 && gz < ldz;
            const int g = ok ? gx * ldz + gz : 0;
            const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
            const int o = lx * S::WZ + 4 * lq;
            st4(&sm.mu[o], ok ? ld4(a.mu + g) : z4);
            if (VTI) st4(&sm.mux[o], ok ? ld4(a.mux + g) : z4);
        }
    }
    // interior tiles hold the product coefficients and the new level's factors across the
    // shots; frame tiles, whose passes need the registers, load them per shot
    float4 plam[S::NQ2], plamx[VTI ? S::NQ2 : 1], pc13[VTI ? S::NQ2 : 1];
    auto load_coefficients = [&](const TileInfo& t, int tid) {
#pragma unroll
        for (int m = 0; m < S::NQ2; m++) {
            const int i = tid + m * kThreads;
            const int lc = i / S::PQ, lq = i - lc * S::PQ;
            const int gx = t.plx + lc, z0 = t.pz0 + 4 * lq;
            const bool ok = i < S::IX * S::PQ && gx < t.phx && z0 + 3 >= t.plz && z0 < t.phz;
            const int g = ok ? gx * ldz + z0 : 0;
            const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
            plam[m] = ok ? ld4(a.lam + g) : z4;
            if (VTI) {
                plamx[m] = ok ? ld4(a.lamx + g) : z4;
                pc13[m] = ok ? ld4(a.c13 + g) : z4;
            }
        }
    };
    float4 qir[S::NQ3], qtz[S::NQ3];
    float qtx[S::NQ3];
    auto load_factors = [&](const TileInfo& t, int tid) {
#pragma unroll
        for (int m = 0; m < S::NQ3; m++) {
            const int i = tid + m * kThreads;
            int gx, gz;
            out_quad<S>(t, i, gx, gz);
            const bool ok = gx < t.ex && gz < t.ez;
            const int g = ok ? gx * ldz + gz : 0;
            const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
            qir[m] = ok ? ld4(a.irho + g) : z4;
            qtz[m] = ok ? ld4(a.taper_z + gz) : z4;
            qtx[m] = ok ? a.taper_x[gx] : 0.f;
        }
    };
    if (!EDGE) {
        load_coefficients(t, tid);
        load_factors(t, tid);
    }

    // ---- D2 weights of the new-level quads (interior tiles, isotropic): once per workgroup ----
    // (not with IMG: the imaging's accumulators and second phase need the registers)
    constexpr bool CW = !EDGE && !VTI && S::NQ3 == 1 && !IMG;
    QuadW qw[CW ? S::NQ3 : 1];
    if constexpr (CW) {
        __syncthreads();  // the coefficient window is in LDS
#pragma unroll
        for (int m = 0; m < S::NQ3; m++) {
            const int i = tid + m * kThreads;
            int gx, z0;
            out_quad<S>(t, i, gx, z0);
            if (gx >= t.ex || z0 >= t.ez) continue;
            const int w = (gx - t.wsx) * S::WZ + (z0 - t.wsz);
            float M[5][4], Mc[12];
#pragma unroll
            for (int c = 0; c < 5; c++) unpack(ld4(&sm.mu[w + (c - 2) * S::WZ]), M[c]);
            load_col12(sm.mu, w, Mc);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float mk[5] = {M[0][k], M[1][k], M[2][k], M[3][k], M[4][k]};
                qw[m].x[k] = d2_scaled(d2_weights(&mk[2], 1), a.rdx2);
                qw[m].z[k] = d2_scaled(d2_weights(&Mc[4 + k], 1), a.rdz2);
            }
        }
    }

    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    float gl[IMG ? S::NQ3 : 1][4], gm[IMG ? S::NQ3 : 1][4], gr[IMG ? S::NQ3 : 1][4];
    float g3[IMG && VTI ? S::NQ3 : 1][4], g4[IMG && VTI ? S::NQ3 : 1][4];  // VTI stiffness mode
    if constexpr (IMG) {
#pragma unroll
        for (int m = 0; m < S::NQ3; m++)
#pragma unroll
            for (int k = 0; k < 4; k++) {
                gl[m][k] = gm[m][k] = gr[m][k] = 0.f;
                if (VTI) g3[m][k] = g4[m][k] = 0.f;
            }
    }

    const TileInfo t0 = t;
    const int tid0 = tid;
    for (int shot = s0; shot < s1; shot++) {
        TileInfo t = t0;
        int tid = tid0;
        opaque(t);
        opaque_v(tid);
        // previous level of this shot's new-level quads; frame tiles: what their last step carries over
        float4 qprx[S::NQ3], qprz[S::NQ3], qex[EDGE ? S::NQ3 : 1], qez[EDGE ? S::NQ3 : 1];
        const float* pux = a.prev + shot * a.shot_stride;
        const int inj0 = PTS ? tile_ptr[shot] : 0, inj1 = PTS ? tile_ptr[shot + 1] : 0;  // the sources' cells
        auto load_prev = [&] {
#pragma unroll
        for (int m = 0; m < S::NQ3; m++) {
            const int i = tid + m * kThreads;
            int gx, gz;
            out_quad<S>(t, i, gx, gz);
            const bool ok = gx < t.ex && gz < t.ez;
            const int g = ok ? gx * ldz + gz : 0;
            const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
            qprx[m] = ok ? ld4(pux + g) : z4;
            qprz[m] = ok ? ld4(pux + nxz + g) : z4;
            if constexpr (EDGE) {
                const bool c = ok && a.carry && gz < kCarryRows;
                const float* e = a.carry + ((shot * 2LL) * nx + gx) * kCarryRows + gz;
                qex[m] = c ? ld4(e) : z4;
                qez[m] = c ? ld4(e + (long long)nx * kCarryRows) : z4;
            }
        }
        };
        if (!EDGE) load_prev();
        if (EDGE) load_coefficients(t, tid);
        // frame tiles: this thread's cells of the closure passes, with what they read of the
        // model and the previous level
        // (the z pass takes two of the four wavefronts, alternating with the shot and the
        // workgroup, so that it does not fall on the same SIMDs in every workgroup of a CU)
        PCell pc;
        ZCell zc;
        const int ztid = tid ^ (((shot ^ tix) & 1) << 7);
        bool has_p = false, has_z = false;
        if (EDGE && (top || bot)) {
            has_p = p_cell<VTI, S>(a, t, kThreads - 1 - tid, top, bot, pc);
            has_z = z_cell<S>(a, t, ztid, top, bot, pux, nxz, zc);
        }
        __syncthreads();  // the previous shot is done with the LDS state and products
        if (EDGE && VTI && shot == s0 && tid < 56)
            sm.tb.c[sm.tb.rs * (tid >> 3) + (tid & 7)] = cEdgeD1.c[tid];
        const float* cux = a.curr + shot * a.shot_stride;
#pragma unroll
        for (int m = 0; m < S::NQ1; m++) {
            const int i = tid + m * kThreads;
            if (i < S::WX * S::WQ) {
                const int lx = i / S::WQ, lq = i - lx * S::WQ;
                const int gx = t.wsx + lx, gz = t.wsz + 4 * lq;
                const bool ok = gx >= 0 && gx < nx && gz >= 0 && gz < ldz;
                const int g = gx * ldz + gz;
                const int o = 4 * (m * kThreads + wave * 64);  // window quad i at 4 i
                quad_to_lds(ok ? cux + g : kZeroQuad, &sm.ux[o]);
                quad_to_lds(ok ? cux + nxz + g : kZeroQuad, &sm.uz[o]);
            }
        }
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();

        // products of first derivatives
#pragma unroll
        for (int m = 0; m < S::NQ2; m++) {
            const int i = tid + m * kThreads;
            if (i >= S::IX * S::PQ) continue;
            const int lc = i / S::PQ, lq = i - lc * S::PQ;
            const int gx = t.plx + lc, z0 = t.pz0 + 4 * lq;
            float p[4] = {0.f, 0.f, 0.f, 0.f}, pz[4] = {0.f, 0.f, 0.f, 0.f}, qx[4] = {0.f, 0.f, 0.f, 0.f},
                  qz[4] = {0.f, 0.f, 0.f, 0.f};
            if (gx < t.phx && z0 + 3 >= t.plz && z0 < t.phz)
                product_quad<VTI, S, EDGE>(a, sm, t, gx, z0, plam[m], VTI ? plamx[m] : plam[m], VTI ? pc13[m] : plam[m],
                                           p, pz, qx, qz);
            const int o = lc * S::PZ + 4 * lq;
            if (EDGE && ((top && z0 >= 0 && z0 < 4) || z0 + 3 >= nz - 4)) {
                // the closure rows are the pass's
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (z0 >= 4 && z0 + k < nz - 4) {
                        sm.px[o + k] = p[k];
                        if (VTI) sm.pz[o + k] = pz[k];
                        sm.qx[o + k] = qx[k];
                        sm.qz[o + k] = qz[k];
                    }
                continue;
            }
            st4(&sm.px[o], make_float4(p[0], p[1], p[2], p[3]));
            if (VTI) st4(&sm.pz[o], make_float4(pz[0], pz[1], pz[2], pz[3]));
            st4(&sm.qx[o], make_float4(qx[0], qx[1], qx[2], qx[3]));
            st4(&sm.qz[o], make_float4(qz[0], qz[1], qz[2], qz[3]));
        }
        if (EDGE && (top || bot)) {
            if (has_p) p_cell_run<VTI, S>(a, sm, t, pc);
            if (8 * S::IX > kThreads && p_cell<VTI, S>(a, t, 2 * kThreads - 1 - tid, top, bot, pc))
                p_cell_run<VTI, S>(a, sm, t, pc);
        }
        __syncthreads();

        // new level; frame tiles: the closure and SAT terms and the quads' own parts, then
        // (after a barrier) the rest of the step
        float* nux = a.next + shot * a.shot_stride;
        float* nuz = nux + nxz;
        float erx[EDGE ? S::NQ3 : 1][4], erz[EDGE ? S::NQ3 : 1][4], ezx[EDGE ? S::NQ3 : 1][4], ezz[EDGE ? S::NQ3 : 1][4];
        if constexpr (EDGE) {
            if (top || bot) {
                if (has_z) z_cell_run<VTI, S>(a, sm, t, zc);
                if (12 * S::TX > kThreads && z_cell<S>(a, t, kThreads + ztid, top, bot, pux, nxz, zc))
                    z_cell_run<VTI, S>(a, sm, t, zc);
            }
            if (left || right) x_sat_pass<VTI, S>(a, sm, t, tid, left, right, pux, nxz);
#pragma unroll
            for (int m = 0; m < S::NQ3; m++) {
                const int i = tid + m * kThreads;
                int gx, z0;
                out_quad<S>(t, i, gx, z0);
                if (gx >= t.ex || z0 >= t.ez) continue;
                rhs_quad<VTI, S, EDGE, CW>(a, sm, t, gx, z0, erx[m], erz[m], ezx[m], ezz[m], qw[0]);
#pragma unroll
                for (int k = 0; k < 4; k++)  // formed here, not sunk past the barrier with their inputs kept
                    __asm__ volatile("" : "+v"(erx[m][k]), "+v"(erz[m][k]), "+v"(ezx[m][k]), "+v"(ezz[m][k]));
            }
            load_factors(t, tid);
            load_prev();
            __syncthreads();
        }
#pragma unroll
        for (int m = 0; m < S::NQ3; m++) {
            const int i = tid + m * kThreads;
            int gx, z0;
            out_quad<S>(t, i, gx, z0);
            if (gx >= t.ex || z0 >= t.ez) continue;
            float rx[4], rz[4];
            if constexpr (EDGE) {
                frame_terms<S>(a, sm, t, gx, z0, erx[m], erz[m], ezx[m], ezz[m]);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    rx[k] = erx[m][k];
                    rz[k] = erz[m][k];
                }
            } else {
                rhs_quad<VTI, S, EDGE, CW>(a, sm, t, gx, z0, rx, rz, rx, rz, qw[CW ? m : 0]);
            }
            float prx[4], prz[4], ir[4], tz[4];
            unpack(qprx[m], prx);
            unpack(qprz[m], prz);
            unpack(qir[m], ir);
            unpack(qtz[m], tz);
            const float txf = qtx[m];
            // factors of 1 instead of a branch, which would keep the right-hand side's inputs
            // live across it
            const float txp = a.taper_prev ? txf : 1.f;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float tzp = a.taper_prev ? tz[k] : 1.f;
                prx[k] = (prx[k] * tzp) * txp;
                prz[k] = (prz[k] * tzp) * txp;
            }
            const int wq = (gx - t.wsx) * S::WZ + (z0 - t.wsz);
            float cx[4], cz[4], vx[4], vz[4];
            unpack(ld4(&sm.ux[wq]), cx);
            unpack(ld4(&sm.uz[wq]), cz);
            // leapfrog (we_op.cpp:824-830) with ir = dt^2 / rho
            if constexpr (EDGE) {
                float ex[4], ez[4];
                unpack(qex[m], ex);
                unpack(qez[m], ez);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const float wx = (ir[k] * rx[k] + (cx[k] - prx[k])) + ex[k];
                    const float wz = (ir[k] * rz[k] + (cz[k] - prz[k])) + ez[k];
                    vx[k] = cx[k] + wx;
                    vz[k] = cz[k] + wz;
                    ex[k] = wx - (vx[k] - cx[k]);
                    ez[k] = wz - (vz[k] - cz[k]);
                }
                if (a.carry && z0 < kCarryRows) {
                    float* e = a.carry + ((shot * 2LL) * nx + gx) * kCarryRows + z0;
                    st4(e, make_float4(ex[0], ex[1], ex[2], ex[3]));
                    st4(e + (long long)nx * kCarryRows, make_float4(ez[0], ez[1], ez[2], ez[3]));
                }
            } else {
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    vx[k] = ir[k] * rx[k] + (2.f * cx[k] - prx[k]);
                    vz[k] = ir[k] * rz[k] + (2.f * cz[k] - prz[k]);
                }
            }
            if constexpr (EDGE) {
                // implicit part of the absorbing SAT on the perimeter (spatial_operators.cpp:307-521)
                if (gx == 0 || gx == nx - 1) {  // the corners' divisors are in both arrays
                    const float* d = a.div_lr + (gx ? 2 * ldz : 0) + z0;
                    float dx[4], dz[4];
                    unpack(ld4(d), dx);
                    unpack(ld4(d + ldz), dz);
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        vx[k] = vx[k] / dx[k];
                        vz[k] = vz[k] / dz[k];
                    }
                } else {
                    if (z0 == 0) {
                        vx[0] = vx[0] / a.div_tb[gx];
                        vz[0] = vz[0] / a.div_tb[nx + gx];
                    }
                    if (z0 == ((nz - 1) & ~3)) {
                        const float dx = a.div_tb[2 * nx + gx], dz = a.div_tb[3 * nx + gx];
#pragma unroll
                        for (int k = 0; k < 4; k++)
                            if (k == ((nz - 1) & 3)) {  // the same for all lanes
                                vx[k] = vx[k] / dx;
                                vz[k] = vz[k] / dz;
                            }
                    }
                }
            }
            // cos^2 taper of the new level (we_op.cpp:846-861); cells past nz stay zero
            float ox[4], oz[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const bool in = !EDGE || z0 + k < nz;
                ox[k] = in ? (vx[k] * tz[k]) * txf : 0.f;
                oz[k] = in ? (vz[k] * tz[k]) * txf : 0.f;
            }
            const int g = gx * ldz + z0;
            st4(nux + g, make_float4(ox[0], ox[1], ox[2], ox[3]));
            st4(nuz + g, make_float4(oz[0], oz[1], oz[2], oz[3]));
            if constexpr (IMG) {
                // density term of snapshot j: f0 against the weighted adjoint levels
                __builtin_amdgcn_sched_barrier(0);
                const long long fo = shot * a.fshot_stride + g;
                float f0x[4], f0z[4], pvx[4], pvz[4];
                unpack(ld4(a.f0 + fo), f0x);
                unpack(ld4(a.f0 + fo + nxz), f0z);
                unpack(qprx[m], pvx);
                unpack(qprz[m], pvz);
                const bool st = VTI && a.stiff;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const float ax = a.wn * ox[k] + a.wc * cx[k] + a.wp * pvx[k];
                    const float az = a.wn * oz[k] + a.wc * cz[k] + a.wp * pvz[k];
                    const float r = !EDGE || z0 + k < nz ? f0x[k] * ax + f0z[k] * az : 0.f;
                    if (VTI) {
                        gr[m][k] += st ? 0.f : r;
                        g4[VTI ? m : 0][k] += st ? r : 0.f;
                    } else {
                        gr[m][k] += r;
                    }
                }
            }
        }
        if constexpr (IMG) {
            // stiffness terms of snapshot j-1: its window replaces the products
            __syncthreads();  // every wavefront is done with the products
            const float* Fm = a.fm + shot * a.fshot_stride;
#pragma unroll
            for (int m = 0; m < S::NQ2; m++) {
                const int i = tid + m * kThreads;
                if (i < S::IX * S::PQ) {
                    const int lc = i / S::PQ, lq = i - lc * S::PQ;
                    const int gx = t.plx + lc, z0 = t.pz0 + 4 * lq;
                    const bool ok = gx < nx && z0 >= 0 && z0 < ldz;
                    const int g = ok ? gx * ldz + z0 : 0;
                    const int o = 4 * (m * kThreads + wave * 64);  // quad i at float 4 i, as the state window
                    quad_to_lds(ok ? Fm + g : kZeroQuad, &sFx[o]);
                    quad_to_lds(ok ? Fm + nxz + g : kZeroQuad, &sFz[o]);
                }
            }
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            const int wrow = (t.sx - t.wsx) * S::WZ + S::HZ, frow = (t.sx - t.plx) * S::PZ + 4;
            if (EDGE && (top || bot)) {
                d1z_pass<S::TX, S::WZ>(a, sm.ux, sm.uz, wrow, t.sx, t.ex, t.sz, tid, top, bot, sm.tb);
                d1z_pass<S::TX, S::PZ>(a, sFx, sFz, frow, t.sx, t.ex, t.sz, tid, top, bot, sm.tb);
                __syncthreads();
            }
#pragma unroll
            for (int m = 0; m < S::NQ3; m++) {
                const int i = tid + m * kThreads;
                int gx, z0;
                out_quad<S>(t, i, gx, z0);
                if (gx >= t.ex || z0 >= t.ez) continue;
                const int col = gx - t.sx;
                const int wq = wrow + col * S::WZ + (z0 - t.sz), q = frow + col * S::PZ + (z0 - t.sz);
                // adjoint derivatives of the step's current level, forward derivatives of
                // snapshot j-1 (we_op.cpp:519-541)
                float axx[4], azx[4], axz[4], azz[4], t0x[4], t1z[4], t2x[4], t3z[4];
                quad_derivs<EDGE, S::WZ>(a, sm.ux, sm.uz, wq, wrow + col * S::WZ, gx, z0, sm.tb, axx, azx, axz, azz);
                quad_derivs<EDGE, S::PZ>(a, sFx, sFz, q, frow + col * S::PZ, gx, z0, sm.tb, t0x, t3z, t2x, t1z);
                image_stiff<VTI>(a, (long long)gx * ldz + z0, z0, axx, azx, axz, azz, t0x, t1z, t2x, t3z, gl[m],
                                 gm[m], gr[m], g3[VTI ? m : 0]);
            }
        }
        if (PTS && inj1 > inj0) {
            __syncthreads();  // the tile's new level is stored
            inject_cells(a, inj0 + tid, inj1, IMG, nxz);
        }
    }
    if constexpr (IMG) {
        if (PTS) __syncthreads();  // the point sources' shares of the first shot are in its slab
        float* G = a.grad + s0 * a.gslab_stride;
#pragma unroll
        for (int m = 0; m < S::NQ3; m++) {
            const int i = tid + m * kThreads;
            int gx, z0;
            out_quad<S>(t, i, gx, z0);
            if (gx >= t.ex || z0 >= t.ez || s0 >= s1) continue;
            const long long g = (long long)gx * ldz + z0;
            float4 v = ld4(G + g);
            st4(G + g, make_float4(v.x + gl[m][0], v.y + gl[m][1], v.z + gl[m][2], v.w + gl[m][3]));
            v = ld4(G + nxz + g);
            st4(G + nxz + g, make_float4(v.x + gm[m][0], v.y + gm[m][1], v.z + gm[m][2], v.w + gm[m][3]));
            v = ld4(G + 2 * nxz + g);
            st4(G + 2 * nxz + g, make_float4(v.x + gr[m][0], v.y + gr[m][1], v.z + gr[m][2], v.w + gr[m][3]));
            if (VTI && a.stiff) {
                v = ld4(G + 3 * nxz + g);
                st4(G + 3 * nxz + g, make_float4(v.x + g3[m][0], v.y + g3[m][1], v.z + g3[m][2], v.w + g3[m][3]));
                v = ld4(G + 4 * nxz + g);
                st4(G + 4 * nxz + g, make_float4(v.x + g4[m][0], v.y + g4[m][1], v.z + g4[m][2], v.w + g4[m][3]));
            }
        }
    }
}

// wavefronts per SIMD the registers must leave room for: the LDS's share
constexpr int step_waves(bool vti, int tx, bool img) { return tx == 32 ? 2 : (vti || img ? (vti && img ? 2 : 3) : 4); }

// One launch for all tiles: the frame's workgroups first (their extra passes make them the
// slowest), then the interior rectangle's, each class spread over all XCDs (the frame's
// block count rounded up to a multiple of 8, the extra blocks idle) and remapped within its
// class so that an XCD runs neighbouring tiles.  PTS: the launch also takes the point sources
// and receivers (see step_launch).
template <bool VTI, int TX, bool IMG, bool PTS>
__global__ void __launch_bounds__(kThreads, step_waves(VTI, TX, IMG)) k_step(const StepArgs a)
{
    using S = StepShape<TX>;
    __shared__ __attribute__((aligned(16))) float sUx[S::WX * S::WZ];
    __shared__ __attribute__((aligned(16))) float sUz[S::WX * S::WZ];
    __shared__ __attribute__((aligned(16))) float sMu[S::WX * S::WZ];
    __shared__ __attribute__((aligned(16))) float sMuX[VTI ? S::WX * S::WZ : 4];  // (1+2eps) mu
    __shared__ __attribute__((aligned(16))) float sPx[S::IX * S::PZ];
    __shared__ __attribute__((aligned(16))) float sPz[VTI ? S::IX * S::PZ : 4];
    __shared__ __attribute__((aligned(16))) float sQx[S::IX * S::PZ];
    __shared__ __attribute__((aligned(16))) float sQz[S::IX * S::PZ];
    // frame tiles' D1 table; VTI: in the (1 + 2 eps) mu window, for the 42 LDS granules that
    // leave 3 workgroups per CU
    __shared__ __attribute__((aligned(16))) float sT[VTI ? 4 : 56];
    StepSmem sm{sUx, sUz, sMu, sMuX, sPx, sPz, sQx, sQz, {sT, 8}};

    const int nin_x = a.itx1 - a.itx0, nin_z = a.itz1 - a.itz0;
    const int nin = nin_x * nin_z, nedge = a.ntx * a.ntz - nin;
    const int ne = nedge * a.ngroups_e, ne8 = (ne + 7) & ~7;
    const int b = blockIdx.x;
    if (b < ne8) {
        if (b >= ne) return;  // padding: the whole workgroup leaves before any barrier
        if (!VTI && threadIdx.x < 56) sT[threadIdx.x] = cEdgeD1.c[threadIdx.x];  // read after the first barrier
        // frame: the rows of tiles above and below the rectangle, then its side columns
        const int lin = xcd_remap(b, ne);
        const int tile = lin / a.ngroups_e, grp = lin - tile * a.ngroups_e;
        const int top = a.itz0 * a.ntx, bot = (a.ntz - a.itz1) * a.ntx;
        int tix, tiz;
        if (tile < top + bot) {
            const int r = tile < top ? tile : tile - top;
            tix = r % a.ntx;
            tiz = (tile < top ? 0 : a.itz1) + r / a.ntx;
        } else {
            const int r = tile - top - bot, w = a.ntx - nin_x;
            const int c = r % w;
            tiz = a.itz0 + r / w;
            tix = c < a.itx0 ? c : a.itx1 + (c - a.itx0);
        }
        if (VTI) {
            // out-of-grid cells of the (1 + 2 eps) mu window: 8 rows above or below the grid, or
            // the first or last window column
            const bool t = tiz == 0, b = tiz == a.ntz - 1;
            sm.tb = {sMuX + (t ? 0 : b ? S::TZ + S::HZ : tix == 0 ? S::HZ : (S::WX - 1) * S::WZ + S::HZ),
                     t || b ? S::WZ : 8};
        }
        const int s0 = grp * a.spb_e;
        step_tile<VTI, S, true, IMG, PTS>(a, sm, tix, tiz, s0, min(a.nshots, s0 + a.spb_e));
    } else if (PTS && b >= ne8 + nin * a.ngroups) {
        // receivers of the current level
        const PointTable& pt = *a.points;
        const int k = (b - ne8 - nin * a.ngroups) * kThreads + threadIdx.x;
        if (k < 2 * pt.nrec)
            extract_component(k, a.curr, a.shot_stride, (long long)a.nx * a.ldz, a.ldz, pt.rec, pt.rec_ptr, a.rec_trace,
                              a.it);
    } else {
        const int lin = xcd_remap(b - ne8, nin * a.ngroups);
        const int tile = lin / a.ngroups, grp = lin - tile * a.ngroups;
        const int s0 = grp * a.spb;
        step_tile<VTI, S, false, IMG, PTS>(a, sm, a.itx0 + tile / nin_z, a.itz0 + tile % nin_z, s0,
                                      min(a.nshots, s0 + a.spb));
    }
}

// ---------------------------------------------------------------------------
// Imaging condition after an adjoint step (compute_gradients, we_op.cpp:505-562).
// a.curr is the lagged adjoint level (its first derivatives are imaged), a.next the
// level after the step and its point sources (the density term), a.f0/fm/fp forward
// snapshots idx, idx-1, idx+1.  A workgroup owns a TX x 64 tile of the tile grid and a
// group of a.spb shots; per shot the adjoint and snapshot windows (halo 2 in x, 4 in z)
// go through LDS, the next shot's windows are loaded into registers meanwhile, and the
// contributions are summed in registers and added once to the gradient slab of the
// group's first shot.  Tiles with every cell at least 4 from the edges take the interior
// stencils only; the others the closure columns per quad and the closure rows from a pass
// with one cell per thread (d1z_pass).
// ---------------------------------------------------------------------------
// SBP = true: the density term by parts in time (a.aprev is the derivative level, the
// cell values are the adjoint levels it and it+1, see StepArgs).
template <bool VTI, int TX, int NBUF, bool SBP>
__global__ void __launch_bounds__(kThreads) k_img(const StepArgs a)
{
    constexpr int TZ = kTileZ, HX = 2, HZ = 4;
    constexpr int WX = TX + 2 * HX, WZ = TZ + 2 * HZ, WQ = WZ / 4;
    constexpr int NQ1 = (WX * WQ + kThreads - 1) / kThreads;
    constexpr int QC = TZ / 4, NQ3 = TX * QC / kThreads;
    constexpr int WS = WX * WZ;  // floats per window array
    static_assert((TX * QC) % kThreads == 0, "tile must give every thread whole quads");
    // [buffer][Ax, Az, Fx, Fz][window]: window quad i of an array at float offset 4 i, so
    // that the quads a wavefront loads are consecutive in LDS
    __shared__ __attribute__((aligned(16))) float sW[NBUF * 4 * WS];
    __shared__ __attribute__((aligned(16))) float sT[48];
    if (threadIdx.x < 48) sT[threadIdx.x] = cEdgeD1.c[threadIdx.x];  // read after the first barrier
    const EdgeTable tb{sT, 8};

    // group-major order: the tiles of one shot group follow each other (z first), so that
    // the window halos a tile shares with its neighbours are still in the XCD's L2
    const int lin = xcd_remap(blockIdx.x, gridDim.x);
    const int ntiles = a.ntx * a.ntz;
    const int group = lin / ntiles;
    const int tile = lin - group * ntiles;
    const int tix = tile / a.ntz, tiz = tile - tix * a.ntz;
    const int nx = a.nx, nz = a.nz, ldz = a.ldz;
    int sx, ex, sz, ez;
    tile_range_x_hd(tix, a.ntx, TX, nx, sx, ex);
    tile_range_z_hd(tiz, a.ntz, nz, ldz, sz, ez);
    const int wsx = window_start(sx, HX), wsz = sz - HZ;
    const bool inner = sx >= 4 && ex <= nx - 4 && sz >= 4 && ez <= nz - 4;
    const bool top = sz == 0, bot = tiz == a.ntz - 1;
    const long long nxz = (long long)nx * ldz;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int s0 = group * a.spb;
    const int s1 = min(a.nshots, s0 + a.spb);

    // windows of one shot into buffer b: window quads tid + m * 256
    auto issue_windows = [&](int shot, int b) {
        const float* A = (SBP ? a.aprev : a.curr) + shot * a.shot_stride;
        const float* F = a.f0 + shot * a.fshot_stride;
        float* base = sW + b * 4 * WS;
#pragma unroll
        for (int m = 0; m < NQ1; m++) {
            const int i = tid + m * kThreads;
            if (i < WX * WQ) {
                const int lx = i / WQ, lq = i - lx * WQ;
                const int gx = wsx + lx, gz = wsz + 4 * lq;
                const bool ok = gx >= 0 && gx < nx && gz >= 0 && gz < ldz;
                const long long g = (long long)gx * ldz + gz;
                float* dst = base + 4 * (m * kThreads + wave * 64);
                quad_to_lds(ok ? A + g : kZeroQuad, dst);
                quad_to_lds(ok ? A + nxz + g : kZeroQuad, dst + WS);
                quad_to_lds(ok ? F + g : kZeroQuad, dst + 2 * WS);
                quad_to_lds(ok ? F + nxz + g : kZeroQuad, dst + 3 * WS);
            }
        }
    };

    float gl[NQ3][4], gm[NQ3][4], gr[NQ3][4], g3[VTI ? NQ3 : 1][4], g4[VTI ? NQ3 : 1][4];
#pragma unroll
    for (int m = 0; m < NQ3; m++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
            gl[m][k] = gm[m][k] = gr[m][k] = 0.f;
            if (VTI) g3[m][k] = g4[m][k] = 0.f;
        }

    if (NBUF == 2 && s0 < s1) issue_windows(s0, 0);
    for (int shot = s0; shot < s1; shot++) {
        const int b = NBUF == 2 ? (shot - s0) & 1 : 0;
        if (NBUF == 1) {
            if (shot > s0) __syncthreads();  // every wavefront is done with the windows
            issue_windows(shot, 0);
        }
        // cell values of this shot: the adjoint density level and snapshots idx-1, idx+1
        // (by parts: the adjoint levels it+1 and it)
        float4 qnx[NQ3], qnz[NQ3], qmx[NQ3], qmz[NQ3], qpx[NQ3], qpz[SBP ? 1 : NQ3];
#pragma unroll
        for (int m = 0; m < NQ3; m++) {
            const int i = tid + m * kThreads;
            const int gx = sx + i / QC, z0 = sz + 4 * (i % QC);
            const bool ok = gx < ex && z0 < ez;
            const long long g = ok ? (long long)gx * ldz + z0 : 0;
            const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
            const float* N = a.next + shot * a.shot_stride;
            qnx[m] = ok ? ld4(N + g) : z4;
            qnz[m] = ok ? ld4(N + nxz + g) : z4;
            if constexpr (SBP) {
                const float* C = a.curr + shot * a.shot_stride;
                qmx[m] = ok ? ld4(C + g) : z4;
                qmz[m] = ok ? ld4(C + nxz + g) : z4;
            } else {
                const long long fo = shot * a.fshot_stride + g;
                qmx[m] = ok && a.img_mode != 1 ? ld4(a.fm + fo) : z4;
                qmz[m] = ok && a.img_mode != 1 ? ld4(a.fm + fo + nxz) : z4;
                qpx[m] = ok && a.img_mode != 2 ? ld4(a.fp + fo) : z4;
                qpz[m] = ok && a.img_mode != 2 ? ld4(a.fp + fo + nxz) : z4;
            }
        }
        __builtin_amdgcn_s_waitcnt(0);  // the windows (and cell values) have landed
        __syncthreads();
        // the next shot's windows go into the other buffer while this one is imaged
        if (NBUF == 2 && shot + 1 < s1) issue_windows(shot + 1, b ^ 1);
        float* const sAx = sW + b * 4 * WS;
        float* const sAz = sAx + WS;
        float* const sFx = sAx + 2 * WS;
        float* const sFz = sAx + 3 * WS;
        const int wrow = (sx - wsx) * WZ + HZ;
        if ((top || bot) && !(SBP && !a.img_deriv)) {
            // z derivatives of the closure rows, into the windows' rows outside the grid
            d1z_pass<TX, WZ>(a, sAx, sAz, wrow, sx, ex, sz, tid, top, bot, tb);
            d1z_pass<TX, WZ>(a, sFx, sFz, wrow, sx, ex, sz, tid, top, bot, tb);
            __syncthreads();
        }
#pragma unroll
        for (int m = 0; m < NQ3; m++) {
            const int i = tid + m * kThreads;
            const int gx = sx + i / QC, z0 = sz + 4 * (i % QC);
            if (gx >= ex || z0 >= ez) continue;
            const int w = (gx - wsx) * WZ + (z0 - wsz);
            if constexpr (SBP) {
                // density term by parts: snapshot j against the weighted adjoint levels
                float f0x[4], f0z[4], px[4], pz[4], cx[4], cz[4], nx4[4], nz4[4];
                unpack(ld4(&sFx[w]), f0x);
                unpack(ld4(&sFz[w]), f0z);
                unpack(ld4(&sAx[w]), px);
                unpack(ld4(&sAz[w]), pz);
                unpack(qmx[m], cx);
                unpack(qmz[m], cz);
                unpack(qnx[m], nx4);
                unpack(qnz[m], nz4);
                const bool st = VTI && a.stiff;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    if (z0 + k >= nz) continue;
                    const float ax = a.wn * nx4[k] + a.wc * cx[k] + a.wp * px[k];
                    const float az = a.wn * nz4[k] + a.wc * cz[k] + a.wp * pz[k];
                    const float r = f0x[k] * ax + f0z[k] * az;
                    if (VTI) {
                        gr[m][k] += st ? 0.f : r;
                        g4[VTI ? m : 0][k] += st ? r : 0.f;
                    } else {
                        gr[m][k] += r;
                    }
                }
            } else {
                // density term first, so that the cell values are dead before the
                // derivative reads
                float f0x[4], f0z[4], fmx[4], fmz[4], fpx[4], fpz[4], ox[4], oz[4];
                unpack(ld4(&sFx[w]), f0x);
                unpack(ld4(&sFz[w]), f0z);
                unpack(qmx[m], fmx);
                unpack(qmz[m], fmz);
                unpack(qpx[m], fpx);
                unpack(qpz[m], fpz);
                unpack(qnx[m], ox);
                unpack(qnz[m], oz);
                image_rho<VTI>(a, z0, f0x, f0z, fmx, fmz, fpx, fpz, ox, oz, gr[m], g4[VTI ? m : 0]);
            }
            if (SBP && !a.img_deriv) continue;
            __builtin_amdgcn_sched_barrier(0);
            float axx[4], azx[4], axz[4], azz[4], t0x[4], t1z[4], t2x[4], t3z[4];
            const int row0 = w - (z0 - sz);
            if (inner) {
                quad_derivs<false, WZ>(a, sAx, sAz, w, row0, gx, z0, tb, axx, azx, axz, azz);
                quad_derivs<false, WZ>(a, sFx, sFz, w, row0, gx, z0, tb, t0x, t3z, t2x, t1z);
            } else {
                quad_derivs<true, WZ>(a, sAx, sAz, w, row0, gx, z0, tb, axx, azx, axz, azz);
                quad_derivs<true, WZ>(a, sFx, sFz, w, row0, gx, z0, tb, t0x, t3z, t2x, t1z);
            }
            const long long g = (long long)gx * ldz + z0;
            image_stiff<VTI>(a, g, z0, axx, azx, axz, azz, t0x, t1z, t2x, t3z, gl[m], gm[m], gr[m],
                             g3[VTI ? m : 0]);
        }
        if (NBUF == 2) __syncthreads();  // every wavefront is done with buffer b
    }
    if (s0 >= s1) return;
    float* G = a.grad + s0 * a.gslab_stride;
#pragma unroll
    for (int m = 0; m < NQ3; m++) {
        const int i = tid + m * kThreads;
        const int gx = sx + i / QC, z0 = sz + 4 * (i % QC);
        if (gx >= ex || z0 >= ez) continue;
        const long long g = (long long)gx * ldz + z0;
        float4 v = ld4(G + g);
        st4(G + g, make_float4(v.x + gl[m][0], v.y + gl[m][1], v.z + gl[m][2], v.w + gl[m][3]));
        v = ld4(G + nxz + g);
        st4(G + nxz + g, make_float4(v.x + gm[m][0], v.y + gm[m][1], v.z + gm[m][2], v.w + gm[m][3]));
        v = ld4(G + 2 * nxz + g);
        st4(G + 2 * nxz + g, make_float4(v.x + gr[m][0], v.y + gr[m][1], v.z + gr[m][2], v.w + gr[m][3]));
        if (VTI && a.stiff) {
            v = ld4(G + 3 * nxz + g);
            st4(G + 3 * nxz + g, make_float4(v.x + g3[m][0], v.y + g3[m][1], v.z + g3[m][2], v.w + g3[m][3]));
            v = ld4(G + 4 * nxz + g);
            st4(G + 4 * nxz + g, make_float4(v.x + g4[m][0], v.y + g4[m][1], v.z + g4[m][2], v.w + g4[m][3]));
        }
    }
}

// ---------------------------------------------------------------------------
// Initial condition: prev = 1/2 dt^2/rho * inject(trace[0])  (we_op.cpp:655-663) on a zero
// level, one thread per touched cell summing its contributions in injector order
// ---------------------------------------------------------------------------
__global__ void k_init_cells(const InjCell* cells, int ncell, const int* ptr, const long long* ctx,
                             const long long* ctz, const float* cw, const float* trace, float* prev,
                             long long shot_stride, long long nxz, int ldz, const float* rho, float half_dt2)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncell) return;
    const InjCell cell = cells[c];
    float fx = 0.f, fz = 0.f;
    for (int k = ptr[c]; k < ptr[c + 1]; k++) {
        fx += cw[k] * trace[ctx[k]];
        fz += cw[k] * trace[ctz[k]];
    }
    const long long g = (long long)cell.gx * ldz + cell.gz;
    const float f = half_dt2 / rho[g];
    float* u = prev + cell.shot * shot_stride + g;
    u[0] = fx * f;
    u[nxz] = fz * f;
}

// extraction of one level (the last one; the others are read by the step that follows them)
__global__ void k_extract(const float* state, long long shot_stride, long long nxz, int ldz, const PointEntry* ents,
                          const int* rptr, int nrec, float* trace, int it)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < 2 * nrec) extract_component(k, state, shot_stride, nxz, ldz, ents, rptr, trace, it);
}

// ---------------------------------------------------------------------------
// Imaging condition (we_op.cpp:505-562 iso, 1478-1557 vti), one adjoint step
// ---------------------------------------------------------------------------
template <bool VTI, int TX>
__global__ void __launch_bounds__(kThreads) k_image(const ImageArgs a)
{
    constexpr int TZ = kTileZ, H = 2;
    constexpr int WZ = TZ + 2 * H, WX = TX + 2 * H;
    __shared__ float sAx[WX * WZ], sAz[WX * WZ], sFx[WX * WZ], sFz[WX * WZ];
    const int ntiles = a.ntx * a.ntz;
    const int lin = xcd_remap(blockIdx.x, gridDim.x);
    const int shot = lin / ntiles;
    const int tile = lin - shot * ntiles;
    const int tix = tile / a.ntz, tiz = tile - (tile / a.ntz) * a.ntz;
    const int nx = a.nx, nz = a.nz, ldz = a.ldz;
    int sx, ex, sz, ez;
    tile_range_x_hd(tix, a.ntx, TX, nx, sx, ex);
    tile_range_z_hd(tiz, a.ntz, nz, ldz, sz, ez);
    const int wsx = window_start(sx, H), wsz = window_start(sz, H);
    const long long nxz = (long long)nx * ldz;
    const float* dA = (a.lag ? a.adj_prev : a.adj) + shot * a.shot_stride;
    const float* F0 = a.f0 + shot * a.fshot_stride;
    for (int i = threadIdx.x; i < WX * WZ; i += kThreads) {
        const int lx = i / WZ, lz = i - lx * WZ;
        const int gx = wsx + lx, gz = wsz + lz;
        float ax = 0.f, az = 0.f, fx = 0.f, fz = 0.f;
        if (gx >= 0 && gx < nx && gz >= 0 && gz < nz) {
            const long long g = (long long)gx * ldz + gz;
            ax = dA[g];
            az = dA[nxz + g];
            fx = F0[g];
            fz = F0[nxz + g];
        }
        sAx[i] = ax;
        sAz[i] = az;
        sFx[i] = fx;
        sFz[i] = fz;
    }
    __syncthreads();
    const float* A = a.adj + shot * a.shot_stride;
    const float* Fm = a.fm ? a.fm + shot * a.fshot_stride : nullptr;
    const float* Fp = a.fp ? a.fp + shot * a.fshot_stride : nullptr;
    float* G = a.grad + shot * a.gshot_stride;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int gz = sz + lane; gz < ez; gz += 64) {
        for (int j = 0; j < TX / 4; j++) {
            const int gx = sx + wave * (TX / 4) + j;
            if (gx >= ex) break;
            const int w = (gx - wsx) * WZ + (gz - wsz);
            const long long g = (long long)gx * ldz + gz;
            const float axx = d1<false>(&sAx[w], WZ, gx, nx) * a.rdx;  // adjoint x_x
            const float azx = d1<false>(&sAx[w], 1, gz, nz) * a.rdz;   // adjoint x_z
            const float axz = d1<false>(&sAz[w], WZ, gx, nx) * a.rdx;  // adjoint z_x
            const float azz = d1<false>(&sAz[w], 1, gz, nz) * a.rdz;   // adjoint z_z
            const float t0 = d1<false>(&sFx[w], WZ, gx, nx) * a.rdx;   // forward x_x
            const float t1 = d1<false>(&sFz[w], 1, gz, nz) * a.rdz;    // forward z_z
            const float t2 = d1<false>(&sFz[w], WZ, gx, nx) * a.rdx;   // forward z_x
            const float t3 = d1<false>(&sFx[w], 1, gz, nz) * a.rdz;    // forward x_z
            const float f0x = F0[g], f0z = F0[nxz + g];
            float d2x, d2z;
            if (a.mode == 0) {
                d2x = Fp[g] - 2.f * f0x + Fm[g];
                d2z = Fp[nxz + g] - 2.f * f0z + Fm[nxz + g];
            } else if (a.mode == 1) {
                d2x = Fp[g] - f0x;
                d2z = Fp[nxz + g] - f0z;
            } else {
                d2x = -f0x + Fm[g];
                d2z = -f0z + Fm[nxz + g];
            }
            if (!VTI) {
                G[g] += a.wlm * (axx + azz) * (t0 + t1);
                G[nxz + g] += a.wlm * ((azx + axz) * (t2 + t3) + 2.f * axx * t0 + 2.f * azz * t1);
            } else {
                const float l = a.lam[g], m = a.mu[g], c = a.c13[g];
                const float del = ((c + m) * (c + m) - (l + m) * (l + m)) / (2.f * (l + m) * (l + 2.f * m));
                const float v1 = sqrtf(2.f * (l + 2.f * m) * (l + m) * del + (l + m) * (l + m));
                const float v2 = ((1.f + 2.f * del) * l + (1.f + 3.f * del) * m) / v1;
                const float v3 = ((1.f + 3.f * del) * l + (1.f + 4.f * del) * m) / v1 - 1.f;
                const float e = 1.f + 2.f * a.eps[g];
                G[g] += a.wlm * (e * axx * t0 + azz * t1 + v2 * (axx * t1 + azz * t0));
                G[nxz + g] += a.wlm * ((azx + axz) * (t2 + t3) + 2.f * e * axx * t0 + 2.f * azz * t1 +
                                       v3 * (axx * t1 + azz * t0));
            }
            G[2 * nxz + g] += a.wrho * (A[g] * d2x + A[nxz + g] * d2z);
        }
    }
}

// ---------------------------------------------------------------------------
// Utilities
// ---------------------------------------------------------------------------
// sum of the gradient slabs in slab order; columns of ldz cells in, of nz out
__global__ void k_sum_slabs(const float* slabs, long long stride, int nslab, long long ncol, int nz, int ldz,
                            float* out)
{
    const long long n = ncol * nz;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const long long c = i / nz, p = c * ldz + (i - c * nz);
        float v = 0.f;
        for (int s = 0; s < nslab; s++) v += slabs[s * stride + p];
        out[i] = v;
    }
}

// The elastic model's device fields from the model [np][nx][nz]: the padded fields (padding
// cells hold lambda = mu = c13 = eps = 0, rho = 1), and the per-cell factors of the step,
// formed in double and rounded once: dt^2 / rho and, VTI, (1 + 2 eps) mu, (1 + 2 eps) lambda
// and the imaging factors 1 + 2 eps, d c13 / d lambda, d c13 / d mu (we_op.cpp:1510-1519, delta
// recovered from c13); zero in the padding.
__global__ void k_model(const float* m, int np, int nx, int nz, int ldz, double dt2, float* model, float* deriv)
{
    const long long nc = (long long)nx * nz, nxz = (long long)nx * ldz;
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < nxz;
         p += (long long)gridDim.x * blockDim.x) {
        const long long ix = p / ldz;
        const int iz = (int)(p - ix * ldz);
        const bool in = iz < nz;
        const long long i = ix * nz + iz;
        for (int c = 0; c < np; c++) model[c * nxz + p] = in ? m[c * nc + i] : (c == 2 ? 1.f : 0.f);
        deriv[p] = in ? (float)(dt2 / (double)m[2 * nc + i]) : 0.f;
        if (np == 5) {
            float d[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
            if (in) {
                const double l = m[i], u = m[nc + i], c = m[3 * nc + i], e = 1.0 + 2.0 * (double)m[4 * nc + i];
                const double del = ((c + u) * (c + u) - (l + u) * (l + u)) / (2.0 * (l + u) * (l + 2.0 * u));
                const double v1 = sqrt(2.0 * (l + 2.0 * u) * (l + u) * del + (l + u) * (l + u));
                d[0] = (float)(e * u);
                d[1] = (float)(e * l);
                d[2] = (float)e;
                d[3] = (float)(((1.0 + 2.0 * del) * l + (1.0 + 3.0 * del) * u) / v1);
                d[4] = (float)(((1.0 + 3.0 * del) * l + (1.0 + 4.0 * del) * u) / v1 - 1.0);
            }
            for (int k = 0; k < 5; k++) deriv[(k + 1) * nxz + p] = d[k];
        }
    }
}

// The acoustic model's device fields from (K, 1/rho) [2][nx][nz]: both padded with zeros, the
// leapfrog factor dt^2 K, and the divisors of the absorbing sides (asat_scale_boundaries,
// spatial_operators.cpp:779-860: a boundary cell takes v dt / (2 h H0) from each absorbing side
// it lies on; ab: top, bottom, left, right), formed in double.
__global__ void k_amodel(const float* m, int nx, int nz, int ldz, double dt, double fx, double fz, int4 ab, float* K,
                         float* ri, float* kd, float* dv)
{
    const long long nc = (long long)nx * nz, nxz = (long long)nx * ldz;
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < nxz;
         p += (long long)gridDim.x * blockDim.x) {
        const int ix = (int)(p / ldz), iz = (int)(p - (long long)ix * ldz);
        const bool in = iz < nz;
        const long long i = (long long)ix * nz + iz;
        const double k = in ? (double)m[i] : 0.0, r = in ? (double)m[nc + i] : 0.0, v = sqrt(k * r) * dt;
        double s = 0;
        if (ab.x && iz == 0) s += v * fz;
        if (ab.y && iz == nz - 1) s += v * fz;
        if (ab.z && ix == 0) s += v * fx;
        if (ab.w && ix == nx - 1) s += v * fx;
        K[p] = (float)k;
        ri[p] = (float)r;
        kd[p] = (float)(dt * dt * k);
        dv[p] = (float)(1 + s);
    }
}

// D2 closure rows as a dense table [row][field point][coefficient point]
struct ClosureD2 {
    float c[6 * 8 * 8];
};
constexpr ClosureD2 closure_d2_table()
{
    ClosureD2 t{};
    for (const D2Entry& e : kD2ClosureNZ) t.c[(e.row * 8 + e.point) * 8 + e.coef] = (float)(e.num / e.den);
    return t;
}
__constant__ ClosureD2 cClosureD2 = closure_d2_table();

// D2(c) closure rows of a model (see launch_closures): the weight of field point j in row r is
// sum_k table(r, j, k) c_k over the coefficients k cells in from the side.  One thread per x
// weight (consecutive threads down z) or z weight; runs once per model.
__global__ void k_closures(const float* c, int nx, int nz, int ldz, float* wx, float* wz)
{
    const long long nwx = 2LL * 6 * 8 * ldz, nwz = 2LL * nx * 6 * 8;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < nwx + nwz;
         i += (long long)gridDim.x * blockDim.x) {
        const bool x = i < nwx;
        const long long line = x ? i / ldz : (i - nwx) / 48;  // (side 6 + row) 8 + point, or side nx + column
        const int z = (int)(x ? i - line * ldz : 0);
        const int rj = (int)(x ? line % 48 : (i - nwx) - line * 48);
        const bool far = line >= (x ? 48 : nx);
        long long p = x ? (far ? (long long)(nx - 1) * ldz : 0) + z : (line - (far ? nx : 0)) * ldz + (far ? nz - 1 : 0);
        const long long st = (x ? ldz : 1) * (far ? -1 : 1);
        float v = 0.f;
        for (int k = 0; k < 8; k++, p += st) v += cClosureD2.c[rj * 8 + k] * c[p];
        if (x) wx[i] = v;
        else wz[i - nwx] = v;
    }
}

__global__ void k_fill(float* p, long long n, float v)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) p[i] = v;
}

// dipole_to_strain (misc.cpp:18-43) of DAS channels, in place on traces [2][nr][nt]:
// forward x = (c x + s z) / gl, z = 0; adjoint z = s x / gl, x = c x / gl, with cs = (cos,
// sin) of each channel's dip; in double precision, one sample per thread.
__global__ void k_das_strain(float* tr, const double* cs, int nr, int nt, double gl, int adjoint)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)nr * nt) return;
    const int r = (int)(i / nt);
    const double c = cs[2 * r], sn = cs[2 * r + 1];
    float* px = tr + i;
    float* pz = tr + (long long)nr * nt + i;
    const double x = *px;
    if (!adjoint) {
        *px = (float)((c * x + sn * (double)*pz) / gl);
        *pz = 0.f;
    } else {
        *pz = (float)(sn * x / gl);
        *px = (float)(c * x / gl);
    }
}

// The per-trace time map of the operator level (resampling, time derivative, quadrature
// weights, reversal, composed on the host): out[x][i] = sum_k w[k] in[x][col[k]] over the
// row-compressed entries k of row i, accumulated in double precision; one output sample
// per thread, consecutive threads on consecutive samples of one trace.
__global__ void k_trace_matvec(const int* __restrict__ ptr, const int* __restrict__ col, const double* __restrict__ w,
                               int nrow, int ncol, const float* __restrict__ in, float* __restrict__ out, long long n)
{
    for (long long gid = blockIdx.x * (long long)blockDim.x + threadIdx.x; gid < n;
         gid += (long long)gridDim.x * blockDim.x) {
        const long long x = gid / nrow;
        const int i = (int)(gid - x * nrow);
        const float* a = in + x * ncol;
        double acc = 0.0;
        for (int k = ptr[i]; k < ptr[i + 1]; k++) acc += w[k] * (double)a[col[k]];
        out[gid] = (float)acc;
    }
}

// 16-bit checkpoint levels (BF16 or FP16) with a max-abs scale per (level, shot):
// x = round16(u / s), u = s x.
// Scales are kept as the bit patterns of non-negative floats, whose integer order is the
// float order, so the per-shot maximum is an integer atomic max.
__global__ void k_absmax_shots(const float* u, long long per_shot, int nshots, unsigned* amax)
{
    const int shot = blockIdx.y;
    const float* p = u + shot * per_shot;
    float m = 0.f;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < per_shot;
         i += (long long)gridDim.x * blockDim.x)
        m = fmaxf(m, fabsf(p[i]));
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0) atomicMax(&amax[shot], __float_as_uint(m));
}

__device__ __forceinline__ unsigned short to_bf16(float x)
{
    const unsigned b = __float_as_uint(x);
    return (unsigned short)((b + 0x7FFFu + ((b >> 16) & 1u)) >> 16);  // round to nearest even
}

template <bool F16>
__global__ void k_pack16(const float* u, unsigned short* q, const unsigned* amax, float* scale, long long per_shot)
{
    const int shot = blockIdx.y;
    const float s = __uint_as_float(amax[shot]);
    const float inv = s > 0.f ? 1.f / s : 0.f;
    if (blockIdx.x == 0 && threadIdx.x == 0) scale[shot] = s;
    const float* p = u + shot * per_shot;
    unsigned short* d = q + shot * per_shot;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < per_shot;
         i += (long long)gridDim.x * blockDim.x)
        d[i] = F16 ? __half_as_ushort(__float2half_rn(p[i] * inv)) : to_bf16(p[i] * inv);
}

template <bool F16>
__global__ void k_unpack16(const unsigned short* q, const float* scale, float* u, long long per_shot)
{
    const int shot = blockIdx.y;
    const float s = scale[shot];
    const unsigned short* p = q + shot * per_shot;
    float* d = u + shot * per_shot;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < per_shot;
         i += (long long)gridDim.x * blockDim.x)
        d[i] = (F16 ? __half2float(__ushort_as_half(p[i])) : __uint_as_float((unsigned)p[i] << 16)) * s;
}

__global__ void k_copy(float* dst, const float* src, long long n)
{
    const long long n4 = n >> 2;
    const float4* s4 = reinterpret_cast<const float4*>(src);
    float4* d4 = reinterpret_cast<float4*>(dst);
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n4; i += (long long)gridDim.x * blockDim.x) d4[i] = s4[i];
    for (long long i = (n4 << 2) + blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) dst[i] = src[i];
}

// partial[b] = sum over this block's elements of a*b*w (b, w optional) in FP64
__global__ void k_dot_f64(const float* x, const float* y, const float* w, long long n, double* partial)
{
    __shared__ double red[kThreads];
    double acc = 0.0;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        double v = (double)x[i] * (y ? (double)y[i] : (double)x[i]);
        if (w) v *= (double)w[i];
        acc += v;
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = kThreads / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ void k_reduce_f64(const double* partial, int n, double* out)
{
    __shared__ double red[kThreads];
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += kThreads) acc += partial[i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = kThreads / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0];
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
static inline int grid_for(long long n, int cap = 4096)
{
    long long b = (n + kThreads - 1) / kThreads;
    return (int)(b < 1 ? 1 : (b > cap ? cap : b));
}

template <bool VTI, int TX>
static void step_launch(const StepArgs& a, bool image, int ncell, hipStream_t s)
{
    const int nin = (a.itx1 - a.itx0) * (a.itz1 - a.itz0), ne = (a.ntx * a.ntz - nin) * a.ngroups_e;
    const int nstep = ((ne + 7) & ~7) + nin * a.ngroups;
    const int nrec = a.rec_trace ? (2 * a.nrec + kThreads - 1) / kThreads : 0;
    // Point sources and receivers: in the step's launch below 6144 tiles x shots (24 a CU), which saves
    // a launch of 3 us: us a step with them in the launch and in one of their own,
    //   201 x 601, 1 shot (152 tiles x shots)   11.1  14.8     500 x 1700, 2 (1712)    20.1  22.3
    //   200 x 800, 10 shots (2000)              23.6  26.6     the same, VTI (2000)    31.6  34.8
    //   100 x 1200, 30 (4500)                   56.5  66.1     the same, VTI (4500)    68.5  78.1
    //   500 x 1700, 6 (5136)                    42.2  42.7     the same, VTI (5136)    55.7  58.1
    // Above, the step kernel without their code gains more from its registers, most where tiles
    // are interior ones: 500 x 1700, 12 shots (10272) 89.7 and 78.3 us, VTI 113.7 and 113.2, 64
    // shots 446 and 391 us; a gradient of 200 steps on 200 x 800, 48 shots (9600), 71.6 and
    // 69.6 ms, of 100 x 1200, 60 (9000), 94.1 and 93.0 ms.
    if constexpr (TX == 16) {
        if ((long long)a.ntx * a.ntz * a.nshots < 6144) {
            const dim3 grid(nstep + nrec);
            if (image) hipLaunchKernelGGL((k_step<VTI, TX, true, true>), grid, dim3(kThreads), 0, s, a);
            else hipLaunchKernelGGL((k_step<VTI, TX, false, true>), grid, dim3(kThreads), 0, s, a);
            return;
        }
    }
    if (image) hipLaunchKernelGGL((k_step<VTI, TX, true, false>), dim3(nstep), dim3(kThreads), 0, s, a);
    else hipLaunchKernelGGL((k_step<VTI, TX, false, false>), dim3(nstep), dim3(kThreads), 0, s, a);
    const int nsrc = (ncell + kThreads - 1) / kThreads;
    if (nsrc + nrec > 0)
        hipLaunchKernelGGL(k_points, dim3(nsrc + nrec), dim3(kThreads), 0, s, a, ncell, nsrc, image ? 1 : 0);
}

void launch_step(const StepArgs& a, bool vti, int tile_x, bool image, int ncell, hipStream_t s)
{
    if (vti && tile_x == 32) step_launch<true, 32>(a, image, ncell, s);
    else if (vti) step_launch<true, 16>(a, image, ncell, s);
    else if (tile_x == 32) step_launch<false, 32>(a, image, ncell, s);
    else step_launch<false, 16>(a, image, ncell, s);
}

template <bool VTI, int NBUF, bool SBP>
static void img_dispatch(const StepArgs& a, int tile_x, int n, hipStream_t s)
{
    if (tile_x == 32) k_img<VTI, 32, NBUF, SBP><<<n, kThreads, 0, s>>>(a);
    else k_img<VTI, 16, NBUF, SBP><<<n, kThreads, 0, s>>>(a);
}

template <bool VTI, bool SBP>
static void img_bufs(const StepArgs& a, int tile_x, int nbuf, int n, hipStream_t s)
{
    if (nbuf == 2) img_dispatch<VTI, 2, SBP>(a, tile_x, n, s);
    else img_dispatch<VTI, 1, SBP>(a, tile_x, n, s);
}

void launch_img(const StepArgs& a, bool vti, int tile_x, int nbuf, bool sbp, hipStream_t s)
{
    const int n = a.ntx * a.ntz * a.ngroups;
    if (n <= 0) return;
    if (vti) {
        if (sbp) img_bufs<true, true>(a, tile_x, nbuf, n, s);
        else img_bufs<true, false>(a, tile_x, nbuf, n, s);
    } else {
        if (sbp) img_bufs<false, true>(a, tile_x, nbuf, n, s);
        else img_bufs<false, false>(a, tile_x, nbuf, n, s);
    }
}

template <bool VTI>
static void image_dispatch(const ImageArgs& a, int tile_x, hipStream_t s)
{
    const int nb = a.ntx * a.ntz * a.nshots;
    if (tile_x == 32) hipLaunchKernelGGL((k_image<VTI, 32>), dim3(nb), dim3(kThreads), 0, s, a);
    else hipLaunchKernelGGL((k_image<VTI, 16>), dim3(nb), dim3(kThreads), 0, s, a);
}

void launch_image(const ImageArgs& a, bool vti, int tile_x, hipStream_t s)
{
    if (vti) image_dispatch<true>(a, tile_x, s);
    else image_dispatch<false>(a, tile_x, s);
}

void launch_init_cells(const InjCell* cells, int ncell, const int* ptr, const long long* ctx, const long long* ctz,
                       const float* cw, const float* trace, float* prev, long long shot_stride, long long nxz, int ldz,
                       const float* rho, float half_dt2, hipStream_t s)
{
    if (ncell <= 0) return;
    hipLaunchKernelGGL(k_init_cells, dim3((ncell + kThreads - 1) / kThreads), dim3(kThreads), 0, s, cells, ncell, ptr,
                       ctx, ctz, cw, trace, prev, shot_stride, nxz, ldz, rho, half_dt2);
}

void launch_extract(const float* state, long long shot_stride, long long nxz, int ldz, const PointEntry* ents,
                    const int* rptr, int nrec, float* trace, int it, hipStream_t s)
{
    if (nrec <= 0) return;
    hipLaunchKernelGGL(k_extract, dim3((2 * nrec + kThreads - 1) / kThreads), dim3(kThreads), 0, s, state,
                       shot_stride, nxz, ldz, ents, rptr, nrec, trace, it);
}

void launch_sum_slabs(const float* slabs, long long stride, int nslab, long long ncol, int nz, int ldz, float* out,
                      hipStream_t s)
{
    hipLaunchKernelGGL(k_sum_slabs, dim3(grid_for(ncol * nz)), dim3(kThreads), 0, s, slabs, stride, nslab, ncol, nz,
                       ldz, out);
}

void launch_model(const float* m, int np, int nx, int nz, int ldz, double dt2, float* model, float* deriv,
                  hipStream_t s)
{
    hipLaunchKernelGGL(k_model, dim3(grid_for((long long)nx * ldz)), dim3(kThreads), 0, s, m, np, nx, nz, ldz, dt2,
                       model, deriv);
}

void launch_amodel(const float* m, int nx, int nz, int ldz, double dt, double fx, double fz, int4 ab, float* K,
                   float* ri, float* kd, float* dv, hipStream_t s)
{
    hipLaunchKernelGGL(k_amodel, dim3(grid_for((long long)nx * ldz)), dim3(kThreads), 0, s, m, nx, nz, ldz, dt, fx, fz,
                       ab, K, ri, kd, dv);
}

void launch_closures(const float* c, int nx, int nz, int ldz, float* wx, float* wz, hipStream_t s)
{
    hipLaunchKernelGGL(k_closures, dim3(grid_for(2LL * 48 * (ldz + nx))), dim3(kThreads), 0, s, c, nx, nz, ldz, wx, wz);
}

void launch_fill(float* p, long long n, float v, hipStream_t s)
{
    hipLaunchKernelGGL(k_fill, dim3(grid_for(n)), dim3(kThreads), 0, s, p, n, v);
}

void launch_trace_matvec(const int* ptr, const int* col, const double* w, int nrow, int ncol, const float* in,
                         float* out, long long ntr, hipStream_t s)
{
    const long long n = ntr * nrow;
    if (n <= 0) return;
    hipLaunchKernelGGL(k_trace_matvec, dim3(grid_for(n)), dim3(kThreads), 0, s, ptr, col, w, nrow, ncol, in, out, n);
}

void launch_das_strain(float* tr, const double* cs, int nr, int nt, double gl, bool adjoint, hipStream_t s)
{
    const long long n = (long long)nr * nt;
    if (n <= 0) return;
    hipLaunchKernelGGL(k_das_strain, dim3(grid_for(n)), dim3(kThreads), 0, s, tr, cs, nr, nt, gl, adjoint ? 1 : 0);
}

void launch_pack16(bool f16, const float* u, unsigned short* q, float* scale, unsigned* amax, long long per_shot,
                   int nshots, hipStream_t s)
{
    const int gx = (int)std::min<long long>((per_shot + kThreads - 1) / kThreads, 512);
    hipLaunchKernelGGL(k_fill, dim3(1), dim3(kThreads), 0, s, (float*)amax, (long long)nshots, 0.f);
    hipLaunchKernelGGL(k_absmax_shots, dim3(gx, nshots), dim3(kThreads), 0, s, u, per_shot, nshots, amax);
    if (f16) hipLaunchKernelGGL(k_pack16<true>, dim3(gx, nshots), dim3(kThreads), 0, s, u, q, amax, scale, per_shot);
    else hipLaunchKernelGGL(k_pack16<false>, dim3(gx, nshots), dim3(kThreads), 0, s, u, q, amax, scale, per_shot);
}

void launch_unpack16(bool f16, const unsigned short* q, const float* scale, float* u, long long per_shot, int nshots,
                     hipStream_t s)
{
    const int gx = (int)std::min<long long>((per_shot + kThreads - 1) / kThreads, 512);
    if (f16) hipLaunchKernelGGL(k_unpack16<true>, dim3(gx, nshots), dim3(kThreads), 0, s, q, scale, u, per_shot);
    else hipLaunchKernelGGL(k_unpack16<false>, dim3(gx, nshots), dim3(kThreads), 0, s, q, scale, u, per_shot);
}

void launch_copy(float* dst, const float* src, long long n, hipStream_t s)
{
    hipLaunchKernelGGL(k_copy, dim3(grid_for((n + 3) / 4)), dim3(kThreads), 0, s, dst, src, n);
}

void launch_dot_f64(const float* x, const float* y, const float* w, long long n, double* partial, int nblocks,
                    hipStream_t s)
{
    hipLaunchKernelGGL(k_dot_f64, dim3(nblocks), dim3(kThreads), 0, s, x, y, w, n, partial);
}

void launch_reduce_f64(const double* partial, int n, double* out, hipStream_t s)
{
    hipLaunchKernelGGL(k_reduce_f64, dim3(1), dim3(kThreads), 0, s, partial, n, out);
}

// ---------------------------------------------------------------------------
// Acoustic operator (nl_we_op_a::propagate, we_op.cpp:1937-2135; the SAT terms and their
// scaling, spatial_operators.cpp:551-860).  A workgroup owns a 32 (x) x 32 (z) tile of
// a group of shots; the level windows go straight from global memory into LDS, one shot ahead
// (two buffers), and each thread forms the new level of one quad (column-major, so a
// wavefront covers 8 whole columns) from 128-bit LDS reads: D2x + D2z of the 1/rho-weighted
// Laplacian, the SAT terms of the boundary cells, the leapfrog with dt^2 K, the absorbing
// boundary divisor and the cos^2 taper.  The reference tapers the current level in place after
// each step; here the previous level is tapered on load instead (taper_prev), which gives the
// same values.  Frame tiles take their closures as the elastic step's do: columns along x from
// model weight arrays, rows along z one cell per thread, handed to the quads' owners through
// window cells outside the grid.
// ---------------------------------------------------------------------------
static_assert(kAcTX * (kAcTZ / 4) == kThreads, "one quad per thread");

// one-sided outward boundary derivative sum_k SC[k] u_k (times h), the order of its roundings
// written out
__device__ __forceinline__ float ac_bnd(float u0, float u1, float u2, float u3)
{
    return __builtin_fmaf(kSC.c[3], u3, __builtin_fmaf(kSC.c[2], u2, __builtin_fmaf(kSC.c[0], u0, kSC.c[1] * u1)));
}
// d2_apply and d2_weights with the order of their roundings written out, so that the results do
// not depend on how the compiler contracts the expressions around them.  The orders, and where each
// holds, are those of the first kernel of this operator, kept so that its results stay the same bit
// for bit; no order is more accurate than another.  On a free surface the 1/rho gradient is a sum
// of large cancelling terms: with one order for all cells, or with the elastic step's consistent
// rows, single values move by 5 to 9e-4 of the gradient's rms, and stay 1.4 to 2.4e-3 of it off
// FP64 (1.6 to 2.8e-3 as it is), which is the rounding of the stored levels.
// CF: the centre's product is rounded, not the lower neighbour's; MN, PN: on the lower and the upper
// side the nearer coefficient's product is; sf: the nearest pair's product is, not the centre's.
template <bool CF>
__device__ __forceinline__ float ac_d2(const W5& w, float m2, float m1, float u0, float p1, float p2)
{
    auto fma = [](float a, float b, float c) { return __builtin_fmaf(a, b, c); };
    const float v = CF ? fma(w.m1, m1, w.c * u0) : fma(w.c, u0, w.m1 * m1);
    return fma(w.p2, p2, fma(w.m2, m2, fma(w.p1, p1, v)));
}
template <bool MN, bool PN>
__device__ __forceinline__ W5 ac_weights(float m2, float m1, float f0, float p1, float p2, bool sf = false)
{
    auto fma = [](float a, float b, float c) { return __builtin_fmaf(a, b, c); };
    auto two = [&](bool near, float cf, float f, float cn, float n) {
        return near ? fma(cf, f, cn * n) : fma(cn, n, cf * f);
    };
    W5 w;
    const float s = m1 + p1;
    w.c = fma(kD2A.c[2], m2 + p2, sf ? fma(kD2A.c[0], f0, kD2A.c[1] * s) : fma(kD2A.c[1], s, kD2A.c[0] * f0));
    w.m1 = fma(kD2A.c[6], p1, fma(kD2A.c[5], f0, two(MN, kD2A.c[3], m2, kD2A.c[4], m1)));
    w.p1 = fma(kD2A.c[6], m1, fma(kD2A.c[5], f0, two(PN, kD2A.c[3], p2, kD2A.c[4], p1)));
    w.m2 = fma(kD2A.c[9], f0, two(MN, kD2A.c[7], m2, kD2A.c[8], m1));
    w.p2 = fma(kD2A.c[9], f0, two(PN, kD2A.c[7], p2, kD2A.c[8], p1));
    return w;
}

// The level windows.  An interior tile reads 2 columns and (whole quads) 4 rows around it.  A
// frame tile's window holds 2 columns before the tile and 6 after it, moved left to start at
// column nx - 8 at the far side, and 8 rows each side.  That holds every point its cells read:
// interior D2 rows +-2, the closure rows of columns 0-5 read columns 0-7 (first tile) and those of
// columns nx-6..nx-1 columns nx-8..nx-1 (a tile holding such a column ends at most 5 columns
// before its window does), and the SAT terms the boundary column and its 3 neighbours.
template <bool EDGE>
struct AcShape {
    static constexpr int HL = 2, HZ = EDGE ? 8 : 4;
    static constexpr int WX = kAcTX + HL + (EDGE ? 6 : 2);
    static constexpr int WZ = kAcTZ + 2 * HZ, WQ = WZ / 4;  // LDS column stride, quads of a column
    static constexpr int NQ = (WX * WQ + kThreads - 1) / kThreads;
};
constexpr int kAcWin = AcShape<true>::WX * AcShape<true>::WZ;  // floats of the largest window

struct AcTile {
    int sx, ex, sz, ez, wsx, wsz;
};
template <bool EDGE>
__device__ __forceinline__ AcTile ac_tile(const AcousticArgs& a, int tix, int tiz)
{
    AcTile t;
    t.sx = tix * kAcTX;
    t.sz = tiz * kAcTZ;
    t.ex = min(t.sx + kAcTX, a.nx);
    t.ez = min(t.sz + kAcTZ, a.ldz);
    t.wsx = t.sx - AcShape<EDGE>::HL;
    if (EDGE) t.wsx = min(t.wsx, a.nx - 8);
    t.wsz = t.sz - AcShape<EDGE>::HZ;
    return t;
}

__device__ __forceinline__ float sel4(const float (&v)[4], int k)
{
    return k == 0 ? v[0] : (k == 1 ? v[1] : (k == 2 ? v[2] : v[3]));
}

// Cell i of a level at a uniform address.  I = int: a level below 4 GiB, whose byte offsets fit 32
// bits (an address in scalar registers and one vector register); I = long long: any level.
__device__ __forceinline__ const float* at(const float* base, int i)
{
    return reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + 4 * (unsigned)i);
}
__device__ __forceinline__ float* at(float* base, int i)
{
    return reinterpret_cast<float*>(reinterpret_cast<char*>(base) + 4 * (unsigned)i);
}
__device__ __forceinline__ const float* at(const float* base, long long i) { return base + i; }
__device__ __forceinline__ float* at(float* base, long long i) { return base + i; }

// The thread's quads of a window: window quad i goes to float 4 i of the LDS window and comes
// from float off of the level (kOutside: outside the grid, zeros).  Interior tiles' windows lie
// inside the grid: such a tile starts at a multiple of 32 rows, ends before row nz - 6, and
// before column nx - 6.
constexpr int kOutside = -1;
template <bool EDGE, class I>
struct AcQuads {
    using S = AcShape<EDGE>;
    I off[S::NQ];
    __device__ __forceinline__ AcQuads(const AcousticArgs& a, const AcTile& t)
    {
#pragma unroll
        for (int m = 0; m < S::NQ; m++) {
            const int i = threadIdx.x + m * kThreads, lx = i / S::WQ;
            const int gx = t.wsx + lx, gz = t.wsz + 4 * (i - lx * S::WQ);
            off[m] = !EDGE || (gx >= 0 && gx < a.nx && gz >= 0 && gz < a.ldz) ? (I)gx * a.ldz + gz : kOutside;
        }
    }
    __device__ __forceinline__ void load(const float* u, float* w) const
    {
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
        for (int m = 0; m < S::NQ; m++)
            if (threadIdx.x + m * kThreads < S::WX * S::WQ)
                quad_to_lds(!EDGE || off[m] != kOutside ? at(u, off[m]) : kZeroQuad, w + 4 * (m * kThreads + wave * 64));
    }
};

// A closure row of a frame tile's cell along z: column gx, row r from the top or bottom, its D2
// weights, and on the boundary row the bulk modulus and the tapered previous level
struct AcCell {
    int gx, r;
    bool bot;
    float w[8], K, p;
};
// cell c of the tile's pass: rows 0-5 of the top (where the tile holds it), then of the bottom
template <class I>
__device__ __forceinline__ bool ac_cell(const AcousticArgs& a, const AcTile& t, int c, int ntop, int nbot,
                                        const float* prev, AcCell& e)
{
    const int row = c / kAcTX;
    e.gx = t.sx + (c - row * kAcTX);
    if (row >= ntop + nbot || e.gx >= t.ex) return false;
    e.bot = row >= ntop;
    const int gz = e.bot ? max(a.nz - 6, t.sz) + (row - ntop) : row;
    e.r = e.bot ? a.nz - 1 - gz : gz;
    const float* W = a.wz + ((I)((e.bot ? a.nx : 0) + e.gx) * 6 + e.r) * 8;
    unpack(ld4(W), e.w);
    unpack(ld4(W + 4), e.w + 4);
    if (e.r == 0) {
        const I g = (I)e.gx * a.ldz + gz;
        e.K = a.K[g];
        e.p = prev[g];
        if (a.taper_prev) e.p = (e.p * a.taper_z[gz]) * a.taper_x[e.gx];
    }
    return true;
}
// D2z[1/rho] (times h^2) of the cell into the level window's cell 8 rows outside, on rows 0-3 its
// side's SAT terms into the 1/rho window's; IMG: the z derivatives of the level and of the snapshot F on rows 0-3, into F's cells 4 and 8
// rows outside
template <bool IMG>
__device__ __forceinline__ void ac_cell_run(const AcousticArgs& a, const AcTile& t, const AcCell& e, float* U,
                                            float* R, float* F, EdgeTable tb)
{
    const int st = e.bot ? -1 : 1;
    const int w = (e.gx - t.wsx) * AcShape<true>::WZ + (e.bot ? a.nz - 1 : 0) - t.wsz;  // the boundary cell
    float u[8], v = 0.f, sat = 0.f;
    edge_cells<8>(&U[w], e.bot, u);
#pragma unroll
    for (int j = 0; j < 8; j++) v += e.w[j] * u[j];
    const int bc = e.bot ? a.bc[1] : a.bc[0];
    const float ri = R[w];
    if (bc == 1) {
        // Dirichlet (free surface): + H^-1 S^T (ri u)_0 on the first 4 cells, - penalty at 0
        if (e.r < 4) sat = sel4(a.dir_z, e.r) * ri * u[0];
        if (e.r == 0) sat -= ri * u[0] * a.pen_z;
    } else if (e.r == 0) {
        // Neumann: - H^-1 (ri S u)_0; absorbing: + the impedance term of the previous level
        sat = -a.neu_z * ri * ac_bnd(u[0], u[1], u[2], u[3]);
        if (bc == 2) sat += a.abs_z * e.p / sqrtf(e.K / ri);
    }
    const int o = w + st * e.r;
    U[o - st * 8] = v;
    if (e.r < 4) R[o - st * 8] = sat;
    if (IMG && e.r < 4) {
        float c[8];
        edge_coefficients(tb, e.r, c);
        float du = 0.f;
#pragma unroll
        for (int j = 0; j < 6; j++) du += c[j] * u[j];
        F[o - st * 4] = (e.bot ? -du : du) * a.rdz;
        F[o - st * 8] = d1z_closure(&F[w], e.bot, c) * a.rdz;
    }
}

// x part of the Laplacian (times h^2) of a closure column's quad (columns 0-5 from a side), and
// its SAT terms into sat;
// w: the quad's window index, g its model index, p the tapered previous level
template <class I>
__device__ __forceinline__ void ac_closure_column(const AcousticArgs& a, const float* U, const float* R, int w, int gx,
                                                  int z0, I g, const float* p, float* rhs, float* sat)
{
    const EdgeRow e = edge_row(gx, a.nx, 1);
    const float* W = a.wx + ((size_t)((e.sg < 0 ? 6 : 0) + e.r) * 8) * a.ldz + z0;
    const int w0 = w + e.o * AcShape<true>::WZ, st = e.st * AcShape<true>::WZ;
    float ub[4][4], ri[4];  // the 4 cells next to the side
#pragma unroll
    for (int k = 0; k < 4; k++) rhs[k] = 0.f;
    unpack(ld4(&R[w0]), ri);
#pragma unroll
    for (int j = 0; j < 8; j++) {
        float wj[4], u[4];
        unpack(ld4(W + (size_t)j * a.ldz), wj);
        unpack(ld4(&U[w0 + j * st]), u);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            rhs[k] += wj[k] * u[k];
            if (j < 4) ub[j][k] = u[k];
        }
    }
    const int bc = e.sg < 0 ? a.bc[3] : a.bc[2];
    if (bc == 1) {
        if (e.r < 4) {
            const float d = sel4(a.dir_x, e.r);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                sat[k] = d * ri[k] * ub[0][k];
                if (e.r == 0) sat[k] -= ri[k] * ub[0][k] * a.pen_x;
            }
        }
    } else if (e.r == 0) {
        float K[4];
        unpack(ld4(a.K + g), K);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            sat[k] = -a.neu_x * ri[k] * ac_bnd(ub[0][k], ub[1][k], ub[2][k], ub[3][k]);
            if (bc == 2) sat[k] += a.abs_x * p[k] / sqrtf(K[k] / ri[k]);
        }
    }
}

// D1 along x of a quad of two windows: interior or closure column
template <bool EDGE>
__device__ __forceinline__ void ac_d1x(const AcousticArgs& a, const float* u, const float* v, int w, int gx,
                                       EdgeTable tb, float* du, float* dv)
{
    if (!EDGE || (gx >= 4 && gx < a.nx - 4)) {
        auto d1x = [&](const float* f, float* d) {
            float X[4][4];
#pragma unroll
            for (int c = 0; c < 4; c++) unpack(ld4(&f[w + (c < 2 ? c - 2 : c - 1) * AcShape<EDGE>::WZ]), X[c]);
#pragma unroll
            for (int k = 0; k < 4; k++) d[k] = kD1A.c[0] * (X[2][k] - X[1][k]) + kD1A.c[1] * (X[3][k] - X[0][k]);
        };
        d1x(u, du);
        d1x(v, dv);
    } else if constexpr (EDGE) {
        d1_quad_closure<AcShape<true>::WZ>(u + w, v + w, gx, a.nx, tb, du, dv);
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
        du[k] *= a.rdx;
        dv[k] *= a.rdx;
    }
}

// Point sources of a tile's shot (we_op.cpp injects them into the right-hand side): the new
// level's cells c0, c0 + 256, ... before c1 get dt^2 K f over the divisor, tapered; sums in
// injector order.  IMG: the increment's share of the K gradient by parts, which the imaging did
// not see, goes to the group's slab.
template <bool IMG, class I>
__device__ __forceinline__ void ac_inject(const AcousticArgs& a, int c0, int c1, float* G)
{
    const PointTable& pt = *a.points;
    for (int c = c0; c < c1; c += kThreads) {
        const InjCell cell = pt.cells[c];
        float f = 0.f;
        for (int k = pt.ptr[c]; k < pt.ptr[c + 1]; k++) f += pt.w[k] * a.inj_trace[pt.ctx[k] + a.it];
        const I g = (I)cell.gx * a.ldz + cell.gz;
        const float inc = ((a.kdt2[g] * f / a.div[g]) * a.taper_z[cell.gz]) * a.taper_x[cell.gx];
        a.next[cell.shot * a.shot_stride + g] += inc;
        if (IMG) G[g] -= (a.wk + a.dwn) * inc * a.f0[cell.shot * a.fshot_stride + g] / (a.K[g] * a.K[g]);
    }
}

// One tile of a.spb consecutive shots.  EDGE = false: a tile of the rectangle of interior tiles,
// whose D2 weights, dt^2 K and tapers stay in registers across the shots; EDGE =
// true: a frame tile, which forms the weights of its interior cells per shot.
// IMG (an adjoint step): the imaging of snapshot j = f0 by parts in time, as in the elastic step.
// The K gradient -sum_j (w_j / dtg) / K^2 a_j (F_j+1 - 2 F_j + F_j-1) collected per snapshot is
// -F_j / K^2 times the second difference of w a / dtg, formed as wk (next - 2 curr + prev) +
// dwn next + dwp prev (prev as stored; the point sources' share of next is ac_inject's), so a
// step reads one snapshot, and its 1/rho term meets the step's own level (img_deriv): 16 B per
// shot-cell instead of the 12 B of a step and 16 B of a separate k_agrad.
template <bool EDGE, bool IMG, class I>
__device__ __forceinline__ void astep_tile(const AcousticArgs& a, int tix, int tiz, int grp, float* sR, float* sU,
                                           float* sF, EdgeTable tb)
{
    constexpr int WZ = AcShape<EDGE>::WZ;
    const AcTile t = ac_tile<EDGE>(a, tix, tiz);
    const int nx = a.nx, nz = a.nz, ldz = a.ldz, tid = threadIdx.x;
    const int s0 = grp * a.spb, s1 = min(s0 + a.spb, a.nshots);
    const int* const tile_ptr = a.points->tile_ptr + (tix * a.ntz + tiz) * a.nshots;
    AcQuads<EDGE, I> q(a, t);
    q.load(a.ri, sR);
    q.load(a.curr + s0 * a.shot_stride, sU);
    if (IMG) q.load(a.f0 + s0 * a.fshot_stride, sF);
    // threads past the last column compute the tile's first one and store nothing
    const bool active = t.sx + tid / (kAcTZ / 4) < t.ex;
    int gx = active ? t.sx + tid / (kAcTZ / 4) : t.sx, z0 = t.sz + 4 * (tid % (kAcTZ / 4));
    I g = (I)gx * ldz + z0;
    int w = (gx - t.wsx) * WZ + (z0 - t.wsz);
    float kd[4], tz[4], pn[4];  // pn: the previous level of the next shot, in flight with its windows
    unpack(ld4(at(a.prev + s0 * a.shot_stride, g), a.stream), pn);
    unpack(ld4(a.kdt2 + g), kd);
    unpack(ld4(a.taper_z + z0), tz);
    const float tx = a.taper_x[gx];
    // closure rows of the tile: rows 0 .. ntop - 1 and the nbot last rows of the grid it holds
    const int zr = min(t.ez, nz);
    const int ntop = EDGE && t.sz == 0 ? min(6, zr) : 0;
    const int nbot = EDGE ? max(0, zr - max(nz - 6, t.sz)) : 0;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    W5 wx[EDGE ? 1 : 4], wz[EDGE ? 1 : 4];
    if constexpr (!EDGE) {
        float M[5][4], Mc[12];
#pragma unroll
        for (int c = 0; c < 5; c++) unpack(ld4(&sR[w + (c - 2) * WZ]), M[c]);
        load_col12(sR, w, Mc);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float* z = &Mc[4 + k];
            wx[k] = ac_weights<true, false>(M[0][k], M[1][k], M[2][k], M[3][k], M[4][k]);
            wz[k] = k == 0   ? ac_weights<true, true>(z[-2], z[-1], z[0], z[1], z[2])
                    : k == 1 ? ac_weights<false, true>(z[-2], z[-1], z[0], z[1], z[2])
                             : ac_weights<true, false>(z[-2], z[-1], z[0], z[1], z[2]);
        }
    }
    float gk[4] = {0.f, 0.f, 0.f, 0.f}, gr[4] = {0.f, 0.f, 0.f, 0.f};
    float* const G = IMG ? a.grad + grp * a.gslab_stride : nullptr;
    if (IMG) unpack(ld4(G + a.shot_stride + g), gr);
    for (int sh = s0; sh < s1; sh++) {
        const int b = (sh - s0) & 1;
        float* const U = sU + b * kAcWin;
        float* const F = IMG ? sF + b * kAcWin : nullptr;
        const float* prev = a.prev + sh * a.shot_stride;
        const int inj0 = tile_ptr[sh], inj1 = tile_ptr[sh + 1];  // the sources' cells
        int cell = tid;
        // addresses are formed per shot: held (or advanced) across the shots, they spill
        opaque_v(g);
        opaque_v(w);
#pragma unroll
        for (int m = 0; m < AcShape<EDGE>::NQ; m++) opaque_v(q.off[m]);
        if constexpr (EDGE) {
            opaque_v(gx);
            opaque_v(z0);
            opaque_v(cell);
        }
        float pv[4], p[4];
#pragma unroll
        for (int k = 0; k < 4; k++) pv[k] = pn[k];
        AcCell e;
        if (sh + 1 < s1) {  // the next shot's windows, while this one is computed
            unpack(ld4(at(prev + a.shot_stride, g), a.stream), pn);
            q.load(a.curr + (sh + 1) * a.shot_stride, sU + (b ^ 1) * kAcWin);
            if (IMG) q.load(a.f0 + (sh + 1) * a.fshot_stride, sF + (b ^ 1) * kAcWin);
        }
        const float txp = a.taper_prev ? tx : 1.f;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            p[k] = (pv[k] * (a.taper_prev ? tz[k] : 1.f)) * txp;
            __asm__("" : "+v"(p[k]));  // rounded as the stored level would be, not fused into 2 u - p
        }
        float rhs[4], zt[4], Uc[12], sat[EDGE ? 4 : 1] = {};  // D2 along x and z times h^2, SAT terms
        if constexpr (EDGE) {
            // x, then z, the reads of one not held beside the other's
            const bool closure_x = gx < 6 || gx >= nx - 6;
            if (!closure_x) {
                float X[5][4], M[5][4];
#pragma unroll
                for (int c = 0; c < 5; c++) {
                    unpack(ld4(&U[w + (c - 2) * WZ]), X[c]);
                    unpack(ld4(&sR[w + (c - 2) * WZ]), M[c]);
                }
#pragma unroll
                for (int k = 0; k < 4; k++)
                    rhs[k] = ac_d2<true>(ac_weights<true, false>(M[0][k], M[1][k], M[2][k], M[3][k], M[4][k],
                                                                 z0 + k < 6 || z0 + k >= nz - 6),
                                         X[0][k], X[1][k], X[2][k], X[3][k], X[4][k]);
            } else {
                ac_closure_column(a, U, sR, w, gx, z0, g, p, rhs, sat);
            }
#pragma unroll
            for (int k = 0; k < 4; k++) __asm__ volatile("" : "+v"(rhs[k]), "+v"(sat[k]));
            __builtin_amdgcn_sched_barrier(0);
            float Mc[12];
            load_col12(sR, w, Mc);
            load_col12(U, w, Uc);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float *c = &Mc[4 + k], *u = &Uc[4 + k];
                zt[k] = ac_d2<true>(ac_weights<true, false>(c[-2], c[-1], c[0], c[1], c[2], closure_x), u[-2], u[-1], u[0],
                                    u[1], u[2]);
            }
        } else {
            float X[5][4];
#pragma unroll
            for (int c = 0; c < 5; c++) unpack(ld4(&U[w + (c - 2) * WZ]), X[c]);
            load_col12(U, w, Uc);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float* u = &Uc[4 + k];
                rhs[k] = ac_d2<false>(wx[k], X[0][k], X[1][k], X[2][k], X[3][k], X[4][k]);
                zt[k] = k == 0 ? ac_d2<false>(wz[k], u[-2], u[-1], u[0], u[1], u[2])
                               : ac_d2<true>(wz[k], u[-2], u[-1], u[0], u[1], u[2]);
            }
        }
        if (EDGE && ntop + nbot > 0) {
#pragma unroll
            for (int k = 0; k < 4; k++) __asm__ volatile("" : "+v"(zt[k]));
            bool has = ac_cell<I>(a, t, cell, ntop, nbot, prev, e);
#pragma unroll 1
            while (has) {
                ac_cell_run<IMG>(a, t, e, U, sR, F, tb);
                cell += kThreads;
                has = ac_cell<I>(a, t, cell, ntop, nbot, prev, e);
            }
            __syncthreads();  // the closure rows' terms are in the windows
            float c[4];
            if (z0 < 6) {
                unpack(ld4(&U[w - 8]), c);
#pragma unroll
                for (int k = 0; k < 4; k++) zt[k] = z0 + k < 6 ? c[k] : zt[k];
            }
            if (z0 + 3 >= nz - 6) {
                unpack(ld4(&U[w + 8]), c);
#pragma unroll
                for (int k = 0; k < 4; k++) zt[k] = z0 + k >= nz - 6 ? c[k] : zt[k];
            }
        }
#pragma unroll
        for (int k = 0; k < 4; k++) rhs[k] = __builtin_fmaf(rhs[k], a.rdx2, zt[k] * a.rdz2);
        if constexpr (EDGE) {  // SAT terms: top, bottom, then the column's
            float c[4];
            if (z0 < 4) {
                unpack(ld4(&sR[w - 8]), c);
#pragma unroll
                for (int k = 0; k < 4; k++) rhs[k] += c[k];
            }
            if (z0 + 3 >= nz - 4) {
                unpack(ld4(&sR[w + 8]), c);
#pragma unroll
                for (int k = 0; k < 4; k++) rhs[k] += z0 + k >= nz - 4 ? c[k] : 0.f;
            }
#pragma unroll
            for (int k = 0; k < 4; k++) rhs[k] += sat[k];
        }
        float out[4];
#pragma unroll
        for (int k = 0; k < 4; k++) out[k] = kd[k] * rhs[k] + (2.f * Uc[4 + k] - p[k]);  // leapfrog (we_op.cpp:2093-2098)
        if (EDGE && (gx == 0 || gx == nx - 1 || z0 == 0 || z0 + 3 >= nz - 1)) {
            float dv[4];  // boundary divisor (asat_scale_boundaries)
            unpack(ld4(a.div + g), dv);
#pragma unroll
            for (int k = 0; k < 4; k++) out[k] = out[k] / dv[k];
        }
#pragma unroll
        for (int k = 0; k < 4; k++) out[k] = !EDGE || z0 + k < nz ? (out[k] * tz[k]) * tx : 0.f;
        if (active) st4(at(a.next + sh * a.shot_stride, g), make_float4(out[0], out[1], out[2], out[3]), a.stream);
        if constexpr (IMG) {
            __builtin_amdgcn_sched_barrier(0);  // no reads for the imaging while the step's are held
            float Fc[12], ax[4], az[4], fx[4], fz[4];
            load_col12(F, w, Fc);
            // K term by parts (1 / K^2 at the end)
#pragma unroll
            for (int k = 0; k < 4; k++)
                gk[k] += Fc[4 + k] * (a.wk * ((out[k] - Uc[4 + k]) + (pv[k] - Uc[4 + k])) + (a.dwn * out[k] + a.dwp * pv[k]));
            ac_d1x<EDGE>(a, U, F, w, gx, tb, ax, fx);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                az[k] = (kD1A.c[0] * (Uc[5 + k] - Uc[3 + k]) + kD1A.c[1] * (Uc[6 + k] - Uc[2 + k])) * a.rdz;
                fz[k] = (kD1A.c[0] * (Fc[5 + k] - Fc[3 + k]) + kD1A.c[1] * (Fc[6 + k] - Fc[2 + k])) * a.rdz;
            }
            if (EDGE && ntop + nbot > 0) {
                float c[4], d[4];
                if (z0 < 4) {
                    unpack(ld4(&F[w - 4]), az);
                    unpack(ld4(&F[w - 8]), fz);
                }
                if (z0 + 3 >= nz - 4) {
                    unpack(ld4(&F[w + 4]), c);
                    unpack(ld4(&F[w + 8]), d);
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        az[k] = z0 + k >= nz - 4 ? c[k] : az[k];
                        fz[k] = z0 + k >= nz - 4 ? d[k] : fz[k];
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (!EDGE || z0 + k < nz) gr[k] += a.wr * (ax[k] * fx[k] + az[k] * fz[k]);
        }
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();  // the next shot's windows are in, this one's are read, the new level is stored
        if (inj1 > inj0) ac_inject<IMG, I>(a, inj0 + tid, inj1, G);
    }
    if (IMG) __syncthreads();  // the point sources' shares are in the slab
    if (IMG && active) {
        float K[4], v[4];
        unpack(ld4(a.K + g), K);
        unpack(ld4(G + g), v);
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (z0 + k < nz) v[k] -= gk[k] / (K[k] * K[k]);
        st4(G + g, make_float4(v[0], v[1], v[2], v[3]));
        if (a.img_deriv) st4(G + a.shot_stride + g, make_float4(gr[0], gr[1], gr[2], gr[3]));
    }
}

// One launch for all tiles: the frame tiles' workgroups first (their closure rows make
// them the slowest), then the interior rectangle's, each class spread over all XCDs (the
// frame's block count rounded up to a multiple of 8, the extra blocks idle) and remapped
// within its class so that an XCD runs neighbouring tiles; then the receivers of the current
// level.
// Bound by HBM: 64 shots of 500 x 1700 move 0.89 GB in 158 us a step (5.6 TB/s; 0.66 GB without
// the windows' halos) and 1.30 GB in 269 us an imaged one (4.8 TB/s); a large copy reaches 4.9 TB/s.
// The form before (loads through registers, the frame's cells dealt one per thread with one code
// instance per closure row, a launch of its own for the imaging, the points and each kept level)
// took 208 us a step, 299 us an imaging launch and 78 us a copy.  Waves per SIMD: scratch reloads in the shot loop wait for
// the windows in flight, so the bounds are the tightest ones that do not spill there (5 and 4
// instead: 246 and 650 us); what the frame spills costs 1%.  Streamed levels (stream): 151
// instead of 168 us above the memory-side cache's size, 2 to 12% slower below it.
template <bool IMG, class I>
__global__ void __launch_bounds__(kThreads, IMG ? 3 : 4) k_astep(const AcousticArgs a)
{
    __shared__ __attribute__((aligned(16))) float sR[kAcWin];
    __shared__ __attribute__((aligned(16))) float sU[2 * kAcWin];
    __shared__ __attribute__((aligned(16))) float sF[IMG ? 2 * kAcWin : 4];  // snapshot windows
    __shared__ __attribute__((aligned(16))) float sT[IMG ? 48 : 4];
    const EdgeTable tb{sT, 8};
    const int nin_x = a.itx1 - a.itx0, nin_z = a.itz1 - a.itz0;
    const int nin = nin_x * nin_z, nedge = a.ntx * a.ntz - nin;
    const int groups = (a.nshots + a.spb - 1) / a.spb;
    const int ne = nedge * groups, ne8 = (ne + 7) & ~7;
    const int b = blockIdx.x;
    if (b < ne8) {
        if (b >= ne) return;  // padding: the whole workgroup leaves before any barrier
        if (IMG && threadIdx.x < 48) sT[threadIdx.x] = cEdgeD1.c[threadIdx.x];  // read after the first barrier
        // frame: the rows of tiles above and below the rectangle, then its side columns
        const int lin = xcd_remap(b, ne);
        const int grp = lin / nedge, tile = lin - grp * nedge;
        const int top = a.itz0 * a.ntx, bot = (a.ntz - a.itz1) * a.ntx;
        int tix, tiz;
        if (tile < top + bot) {
            const int r = tile < top ? tile : tile - top;
            tix = r % a.ntx;
            tiz = (tile < top ? 0 : a.itz1) + r / a.ntx;
        } else {
            const int r = tile - top - bot, w = a.ntx - nin_x;
            const int c = r % w;
            tiz = a.itz0 + r / w;
            tix = c < a.itx0 ? c : a.itx1 + (c - a.itx0);
        }
        astep_tile<true, IMG, I>(a, tix, tiz, grp, sR, sU, sF, tb);
    } else if (b < ne8 + nin * groups) {
        const int lin = xcd_remap(b - ne8, nin * groups);
        const int grp = lin / nin, tile = lin - grp * nin;
        astep_tile<false, IMG, I>(a, a.itx0 + tile / nin_z, a.itz0 + tile % nin_z, grp, sR, sU, sF, tb);
    } else {
        const int r = (b - ne8 - nin * groups) * kThreads + threadIdx.x;
        if (r < a.nrec) {
            const PointEntry e = a.points->rec[r];
            const float* p = a.curr + e.shot * a.shot_stride;
            float v = 0.f;
            for (int ix = 0; ix < 3; ix++)
                for (int iz = 0; iz < 3; iz++)
                    v += e.wx[ix] * e.wz[iz] * p[(long long)(e.xi0 + ix) * a.ldz + e.zi0 + iz];
            a.rec_trace[e.trace + a.it] = v;
        }
    }
}

// nl_we_op_a::compute_gradients (we_op.cpp:1883-1935) for every shot: the K term from the
// second time difference of the snapshots against the adjoint level, the 1/rho term
// from first derivatives of both.  A workgroup images one tile of a.spb consecutive
// shots (the step kernel's groups and windows, adjoint level and snapshot windows one shot
// ahead), sums their terms in shot order in registers and adds the sum to the group's
// gradient slab once.
template <class I>
__global__ void __launch_bounds__(kThreads, 5) k_agrad(const AcousticArgs a)
{
    __shared__ __attribute__((aligned(16))) float sA[2 * kAcWin];
    __shared__ __attribute__((aligned(16))) float sF[2 * kAcWin];
    __shared__ __attribute__((aligned(16))) float sT[48];
    const EdgeTable tb{sT, 8};
    const int ntile = a.ntx * a.ntz, tid = threadIdx.x;
    if (tid < 48) sT[tid] = cEdgeD1.c[tid];  // read after the first barrier
    const int lin = xcd_remap(blockIdx.x, gridDim.x);
    const int grp = lin / ntile, tile = lin - grp * ntile;
    const int tix = tile / a.ntz, tiz = tile - tix * a.ntz;
    constexpr int WZ = AcShape<true>::WZ;
    const AcTile t = ac_tile<true>(a, tix, tiz);
    const int nz = a.nz, ldz = a.ldz;
    const int s0 = grp * a.spb, s1 = min(s0 + a.spb, a.nshots);
    const AcQuads<true, I> q(a, t);
    q.load(a.curr + s0 * a.shot_stride, sA);
    q.load(a.f0 + s0 * a.fshot_stride, sF);
    // threads past the last column compute the tile's first one and store nothing
    const bool active = t.sx + tid / (kAcTZ / 4) < t.ex;
    const int gx = active ? t.sx + tid / (kAcTZ / 4) : t.sx, z0 = t.sz + 4 * (tid % (kAcTZ / 4));
    const I g = (I)gx * ldz + z0;
    const int w = (gx - t.wsx) * WZ + (z0 - t.wsz);
    const int zr = min(t.ez, nz);
    const int ntop = t.sz == 0 ? min(4, zr) : 0, nbot = max(0, zr - max(nz - 4, t.sz));
    float K[4], kw[4], gk[4], gr[4];  // kw: the K term's weight w / (dtg K^2)
    float* const G = a.grad + grp * a.gslab_stride + g;
    unpack(ld4(a.K + g), K);
    unpack(ld4(G), gk);
    unpack(ld4(G + a.shot_stride), gr);
#pragma unroll
    for (int k = 0; k < 4; k++) kw[k] = z0 + k < nz ? a.wk / (K[k] * K[k]) : 0.f;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    for (int sh = s0; sh < s1; sh++) {
        const int b = (sh - s0) & 1;
        float *const A = sA + b * kAcWin, *const F = sF + b * kAcWin;
        const long long fo = sh * a.fshot_stride + g;
        float fm[4] = {0.f, 0.f, 0.f, 0.f}, fp[4] = {0.f, 0.f, 0.f, 0.f};
        if (a.mode != 1) unpack(ld4(a.fm + fo), fm);
        if (a.mode != 2) unpack(ld4(a.fp + fo), fp);
        if (sh + 1 < s1) {
            q.load(a.curr + (sh + 1) * a.shot_stride, sA + (b ^ 1) * kAcWin);
            q.load(a.f0 + (sh + 1) * a.fshot_stride, sF + (b ^ 1) * kAcWin);
        }
        if (ntop + nbot > 0) {
            // z derivatives of rows 0-3 from the top and bottom, one cell per thread, into the
            // windows' cells 8 rows outside
            for (int c = tid; c < (ntop + nbot) * kAcTX; c += kThreads) {
                const int row = c / kAcTX, col = c - row * kAcTX;
                const bool bot = row >= ntop;
                const int gz = bot ? max(nz - 4, t.sz) + (row - ntop) : row, r = bot ? nz - 1 - gz : gz;
                if (t.sx + col >= t.ex) continue;
                const int wb = (t.sx + col - t.wsx) * WZ + (bot ? nz - 1 : 0) - t.wsz, o = wb + (bot ? 8 - r : r - 8);
                float cf[8];
                edge_coefficients(tb, r, cf);
                A[o] = d1z_closure(&A[wb], bot, cf) * a.rdz;
                F[o] = d1z_closure(&F[wb], bot, cf) * a.rdz;
            }
            __syncthreads();
        }
        float Ac[12], Fc[12], ax[4], az[4], fx[4], fz[4];
        load_col12(A, w, Ac);
        load_col12(F, w, Fc);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float f = Fc[4 + k];
            const float d2 = a.mode == 0 ? fp[k] - 2.f * f + fm[k] : (a.mode == 1 ? fp[k] - f : -f + fm[k]);
            gk[k] -= kw[k] * Ac[4 + k] * d2;
            az[k] = (kD1A.c[0] * (Ac[5 + k] - Ac[3 + k]) + kD1A.c[1] * (Ac[6 + k] - Ac[2 + k])) * a.rdz;
            fz[k] = (kD1A.c[0] * (Fc[5 + k] - Fc[3 + k]) + kD1A.c[1] * (Fc[6 + k] - Fc[2 + k])) * a.rdz;
        }
        ac_d1x<true>(a, A, F, w, gx, tb, ax, fx);
        if (ntop + nbot > 0) {
            float c[4], d[4];
            if (z0 < 4) {
                unpack(ld4(&A[w - 8]), az);
                unpack(ld4(&F[w - 8]), fz);
            }
            if (z0 + 3 >= nz - 4) {
                unpack(ld4(&A[w + 8]), c);
                unpack(ld4(&F[w + 8]), d);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    az[k] = z0 + k >= nz - 4 ? c[k] : az[k];
                    fz[k] = z0 + k >= nz - 4 ? d[k] : fz[k];
                }
            }
        }
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (z0 + k < nz) gr[k] += a.wr * (ax[k] * fx[k] + az[k] * fz[k]);
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();  // the next shot's windows are in; this shot's are read
    }
    if (active) {
        st4(G, make_float4(gk[0], gk[1], gk[2], gk[3]));
        st4(G + a.shot_stride, make_float4(gr[0], gr[1], gr[2], gr[3]));
    }
}

// Initial condition prev = 1/2 dt^2 K inject(trace sample 0) on a zero level, one thread per
// touched cell summing its contributions in injector order
__global__ void k_ainit(const InjCell* cells, int ncell, const int* ptr, const long long* off, const float* w,
                        const float* trace, float* u, long long shot_stride, int ldz, const float* kdt2)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncell) return;
    const InjCell cell = cells[c];
    float f = 0.f;
    for (int k = ptr[c]; k < ptr[c + 1]; k++) f += w[k] * trace[off[k]];
    const long long g = (long long)cell.gx * ldz + cell.gz;
    u[cell.shot * shot_stride + g] = 0.5f * kdt2[g] * f;
}

__global__ void k_aextract(const float* u, long long shot_stride, int ldz, const PointEntry* ents, int nrec,
                           float* trace, int it)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nrec) return;
    const PointEntry e = ents[r];
    const float* p = u + e.shot * shot_stride;
    float v = 0.f;
    for (int ix = 0; ix < 3; ix++)
        for (int iz = 0; iz < 3; iz++) v += e.wx[ix] * e.wz[iz] * p[(long long)(e.xi0 + ix) * ldz + e.zi0 + iz];
    trace[e.trace + it] = v;
}

// Whether 32-bit offsets reach every cell of a level (in bytes, see at) and every closure weight
// (2 nx 48 of wz).  64-bit ones everywhere, also in the closure and point cells alone, cost 3 to 5%.
static bool small_level(const AcousticArgs& a) { return (long long)a.nx * std::max(a.ldz, 48) < (1LL << 30); }

void launch_astep(const AcousticArgs& a, hipStream_t s)
{
    const int groups = (a.nshots + a.spb - 1) / a.spb;
    const int nin = (a.itx1 - a.itx0) * (a.itz1 - a.itz0), ne = (a.ntx * a.ntz - nin) * groups;
    const int nrec = a.rec_trace ? (a.nrec + kThreads - 1) / kThreads : 0;
    const dim3 grid(((ne + 7) & ~7) + nin * groups + nrec);
    if (a.img && small_level(a)) hipLaunchKernelGGL((k_astep<true, int>), grid, dim3(kThreads), 0, s, a);
    else if (a.img) hipLaunchKernelGGL((k_astep<true, long long>), grid, dim3(kThreads), 0, s, a);
    else if (small_level(a)) hipLaunchKernelGGL((k_astep<false, int>), grid, dim3(kThreads), 0, s, a);
    else hipLaunchKernelGGL((k_astep<false, long long>), grid, dim3(kThreads), 0, s, a);
}

void launch_agrad(const AcousticArgs& a, hipStream_t s)
{
    const int groups = (a.nshots + a.spb - 1) / a.spb;
    const dim3 grid(a.ntx * a.ntz * groups);
    if (small_level(a)) hipLaunchKernelGGL(k_agrad<int>, grid, dim3(kThreads), 0, s, a);
    else hipLaunchKernelGGL(k_agrad<long long>, grid, dim3(kThreads), 0, s, a);
}

void launch_ainit(const InjCell* cells, int ncell, const int* ptr, const long long* off, const float* w,
                  const float* trace, float* u, long long shot_stride, int ldz, const float* kdt2, hipStream_t s)
{
    if (ncell <= 0) return;
    hipLaunchKernelGGL(k_ainit, dim3((ncell + 127) / 128), dim3(128), 0, s, cells, ncell, ptr, off, w, trace, u,
                       shot_stride, ldz, kdt2);
}

void launch_aextract(const float* u, long long shot_stride, int ldz, const PointEntry* ents, int nrec, float* trace,
                     int it, hipStream_t s)
{
    if (nrec <= 0) return;
    hipLaunchKernelGGL(k_aextract, dim3((nrec + 127) / 128), dim3(128), 0, s, u, shot_stride, ldz, ents, nrec, trace,
                       it);
}

}  // namespace fwi2d

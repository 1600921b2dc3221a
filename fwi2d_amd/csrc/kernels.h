// Kernel argument blocks and launchers of the elastic propagation engine (gfx950).
//
// Device layout: every field is [x][ldz] with z contiguous and ldz = nz rounded up to a
// multiple of 32 (128-byte columns, so that a 64-cell column segment of a tile is two
// whole cache lines); each thread moves 4 consecutive z cells (a "quad") with one
// 128-bit access; the padding cells are zero and never read as stencil data.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace fwi2d {

constexpr int kTileZ = 64;     // z extent of a tile: 16 quads
constexpr int kThreads = 256;  // 4 wavefronts per workgroup

// One 3x3 footprint of a point injector or extractor, starting at (xi0, zi0), with
// separable weights wx[i] wz[j]; it feeds (or is read into) trace sample offset `trace`
// for the x field component and `tz` for the z component.  A delta_m3 point is one
// footprint (trace and tz the two components of one trace), a ddelta_m3 moment tensor
// two (the x- and z-derivative parts, reading the mxx/mxz and mxz/mzz traces), a
// dipole_m3 DAS channel two (the gauge ends, with opposite signs).
struct PointEntry {
    int xi0, zi0;
    float wx[3], wz[3];
    long long trace, tz;
    int shot;
    int pad;
};

// A cell touched by point injectors: shot and grid position; its contributions are
// listed in a CSR (trace offsets of the x and z field components, weight) in injector
// order.
struct InjCell {
    int shot, gx, gz, pad;
};

// Point sources and receivers of a propagation, in device memory: the touched cells ordered
// by (tile, shot), so that a step's workgroup adds the sources of its own tile, and the
// receivers' footprints.
struct PointTable {
    const InjCell* cells;
    const int* tile_ptr;  // [tiles x shots + 1]: cells of a tile's shot
    const int* ptr;       // [cells + 1]: contributions of a cell
    const long long *ctx, *ctz;
    const float* w;
    const PointEntry* rec;  // receiver r: footprints rec_ptr[r] .. rec_ptr[r + 1]
    const int* rec_ptr;
    int nrec;
};

// Rows below a free surface at the top whose leapfrog carries what the rounding of the new level
// leaves of its increment to the next step (kernels.hip, frame tiles): whole quads, and no more
// than the first row of tiles holds.  8 and 32 rows leave 3% more and 5% less of the error.
constexpr int kCarryRows = 16;

struct StepArgs {
    int nx, nz, ldz, ntx, ntz, nshots, nt, it, taper_prev;
    int spb, ngroups;      // shots per workgroup, shot groups (ceil(nshots / spb))
    int spb_e, ngroups_e;  // the same for frame tiles
    int itx0, itx1, itz0, itz1;  // the tiles [itx0, itx1) x [itz0, itz1) hold interior cells only
    float rdx, rdz, rdx2, rdz2, dt, dt2, sat_x, sat_z;  // rdx2, rdz2: 1 / (24 dx^2), 1 / (24 dz^2)
    float c1x, c2x, c1z, c2z;  // interior first-derivative coefficients divided by dx, dz
    int bc_top, bc_bottom, bc_left, bc_right;
    const float *lam, *mu, *rho, *c13, *eps;
    const float* irho;     // dt^2 / rho
    const float *mux, *lamx;  // VTI: (1 + 2 eps) mu, (1 + 2 eps) lambda
    // D2 closure rows of the model, times 1 / h^2: x columns 0-5 from the left and right
    // [2 sides][6 columns][8 points][ldz] for mu (wx) and, VTI, (1 + 2 eps) mu (wxx); z rows
    // 0-5 from the top and bottom [2 sides][nx][6 rows][8 points] for mu.  Row 0 includes the
    // SAT's boundary derivative
    const float *wx, *wxx, *wz;
    const float *div_tb;   // [2 sides][2 comps][nx] absorbing divisors, top then bottom
    const float *div_lr;   // [2 sides][2 comps][ldz]
    const float *taper_x;  // [nx]
    const float *taper_z;  // [ldz]
    const float* prev;     // shot 0 base of [2][nx][ldz]; shot stride below
    const float* curr;
    float* next;
    long long shot_stride;
    // imaging (k_img after an adjoint step, or fused into it): the derivatives of the
    // step's current level and its new level image forward snapshot idx
    // (compute_gradients, we_op.cpp:505-562)
    int img_mode;              // 0 interior idx, 1 first (idx 0), 2 last
    float wlm, wrho;           // lambda/mu and rho weights of this snapshot
    const float *f0, *fm, *fp; // forward snapshots idx, idx-1, idx+1 (shot 0 base)
    long long fshot_stride;
    float* grad;               // raw gradient slabs [shot][np][nx][ldz]; a workgroup adds its
    long long gslab_stride;    // shots' sum to the slab of its first shot
    const float *ge, *gv2, *gv3;  // VTI: 1 + 2 eps, d c13 / d lambda, d c13 / d mu
    int stiff;                 // VTI: image c11, c13, c33, c55, rho instead of lambda, mu, rho
    // density term by parts in time (k_img, one snapshot per step): f0 is snapshot j, its
    // derivatives meet those of aprev; the density term is f0 . (wn next + wc curr + wp
    // aprev) with the second-difference weights of the neighbouring snapshots
    const float* aprev;
    float wn, wc, wp;
    int img_deriv;             // 0: snapshot j has no stiffness terms (only density terms)
    // point sources added to the new level, receivers read from the current one
    const PointTable* points;
    const float* inj_trace;
    float* rec_trace;          // null: no receivers
    int nrec;
    float* carry;              // [shot][2][nx][kCarryRows] of a free surface at the top, or null
};

struct ImageArgs {
    int nx, nz, ldz, ntx, ntz, nshots, mode;  // mode 0 interior, 1 first (idx 0), 2 last
    float rdx, rdz, wlm, wrho;                // weights: lambda/mu (w*dtg or w*dtg/2), rho (w/dtg)
    const float *lam, *mu, *c13, *eps;
    const float* adj;        // current adjoint level, shot 0 base
    const float* adj_prev;   // previous adjoint level (its derivatives are imaged)
    long long shot_stride;
    const float* f0;         // forward snapshot idx   [shot][2][nx][ldz], shot stride fshot_stride
    const float* fm;         // forward snapshot idx-1 (mode 0, 2)
    const float* fp;         // forward snapshot idx+1 (mode 0, 1)
    long long fshot_stride;
    float* grad;             // per-shot raw gradients [shot][ncomp][nx][ldz]
    int ncomp;
    long long gshot_stride;
    int lag;                 // 1: derivatives of adj_prev (reference), 0: of adj
};

int tiles_x(int nx, int tile_x);
int tiles_z(int ldz);
void tile_range_x(int k, int ntile, int T, int n, int& s, int& e);
void tile_range_z(int k, int ntile, int nz, int ldz, int& s, int& e);

// one time step of every shot over the tile grid, with its ncell point source cells and
// receivers (a.points)
void launch_step(const StepArgs& a, bool vti, int tile_x, bool image, int ncell, hipStream_t s);
// initial condition: prev = 1/2 dt^2 / rho * sum of the cell's contributions at sample 0
void launch_init_cells(const InjCell* cells, int ncell, const int* ptr, const long long* ctx, const long long* ctz,
                       const float* cw, const float* trace, float* prev, long long shot_stride, long long nxz, int ldz,
                       const float* rho, float half_dt2, hipStream_t s);
// receiver r sums the footprints ents[rptr[r]] .. ents[rptr[r+1]-1] into its traces
void launch_extract(const float* state, long long shot_stride, long long nxz, int ldz, const PointEntry* ents,
                    const int* rptr, int nrec, float* trace, int it, hipStream_t s);
void launch_image(const ImageArgs& a, bool vti, int tile_x, hipStream_t s);
// imaging condition after an adjoint step over the tile_x x 64 tile grid (a.ntx x a.ntz
// tiles, a.ngroups groups of a.spb shots); a.curr lagged adjoint level, a.next the new
// one (sbp: the density term by parts, a.aprev the lagged level, see StepArgs); nbuf 2:
// the next shot's windows load into a second LDS buffer during this shot
void launch_img(const StepArgs& a, bool vti, int tile_x, int nbuf, bool sbp, hipStream_t s);
// sum of nslab gradient slabs of ncol columns into out, columns unpadded from ldz to nz
void launch_sum_slabs(const float* slabs, long long stride, int nslab, long long ncol, int nz, int ldz, float* out,
                      hipStream_t s);
// device fields of a model on the device: elastic [np][nx][nz] into the padded fields and the
// step's factors; acoustic (K, 1/rho) into K, 1/rho, dt^2 K and the boundary divisors (fx, fz:
// 1 / (2 h H0))
void launch_model(const float* m, int np, int nx, int nz, int ldz, double dt2, float* model, float* deriv,
                  hipStream_t s);
void launch_amodel(const float* m, int nx, int nz, int ldz, double dt, double fx, double fz, int4 ab, float* K,
                   float* ri, float* kd, float* dv, hipStream_t s);
// D2(c) closure rows (times h^2) of a coefficient c [nx][ldz]: wx [2 sides][6 rows][8 points][ldz],
// wz [2 sides][nx][6 rows][8 points]
void launch_closures(const float* c, int nx, int nz, int ldz, float* wx, float* wz, hipStream_t s);
void launch_fill(float* p, long long n, float v, hipStream_t s);
// out [ntr][nrow] = per-trace row-compressed matrix (ptr [nrow + 1], col, w) times in [ntr][ncol]
void launch_trace_matvec(const int* ptr, const int* col, const double* w, int nrow, int ncol, const float* in,
                         float* out, long long ntr, hipStream_t s);
void launch_copy(float* dst, const float* src, long long n, hipStream_t s);
// dipole_to_strain of nr DAS channels in place on traces [2][nr][nt] (cs: cos, sin of
// each channel's dip; forward or adjoint)
void launch_das_strain(float* tr, const double* cs, int nr, int nt, double gl, bool adjoint, hipStream_t s);
// per-shot max-abs scaled 16-bit packing of a time level, FP16 (f16) or BF16 (amax:
// nshots words of scratch)
void launch_pack16(bool f16, const float* u, unsigned short* q, float* scale, unsigned* amax, long long per_shot,
                   int nshots, hipStream_t s);
void launch_unpack16(bool f16, const unsigned short* q, const float* scale, float* u, long long per_shot, int nshots,
                     hipStream_t s);
void launch_dot_f64(const float* a, const float* b, const float* w, long long n, double* partial,
                    int nblocks, hipStream_t s);
void launch_reduce_f64(const double* partial, int n, double* out, hipStream_t s);

// ---------------------------------------------------------------------------
// Acoustic operator (nl_we_op_a, we_op.cpp:1863-2135): one field per shot, [nshots][nx][ldz]
// ---------------------------------------------------------------------------
constexpr int kAcTX = 32, kAcTZ = 32;  // step and imaging tiles (x, z)

struct AcousticArgs {
    int nx, nz, ldz, nshots, ntx, ntz, taper_prev, it;
    int spb;                     // shots per workgroup (consecutive shots of one tile)
    int stream;                  // k_astep: prev and next are read and written past the caches
    int itx0, itx1, itz0, itz1;  // k_astep: the tiles [itx0, itx1) x [itz0, itz1) hold interior cells only
    int bc[4];                   // top, bottom, left, right: 1 Dirichlet, 2 absorbing, 3 Neumann
    float rdx, rdz, rdx2, rdz2;  // 1 / dx, 1 / dz and their squares
    float dir_x[4], dir_z[4];    // Dirichlet SAT S^T terms SC[k] / (H[k] h^2)
    float pen_x, pen_z;          // Dirichlet penalty 1 / (a H0 h^2)
    float neu_x, neu_z;          // Neumann / absorbing 1 / (H0 h^2)
    float abs_x, abs_z;          // absorbing 1 / (2 dt H0 h)
    const float *K, *ri, *kdt2, *div, *taper_x, *taper_z;  // [nx][ldz] (tapers per axis)
    const float *wx, *wz;        // D2[1/rho] closure rows (launch_closures)
    const float* prev;
    const float* curr;
    float* next;
    long long shot_stride;       // nx * ldz
    // point sources added to the new level, receivers read from the current one (null: none)
    const PointTable* points;
    const float* inj_trace;
    float* rec_trace;
    int nrec;
    // imaging: adjoint level curr against snapshot f0 (k_agrad: and its neighbours fm, fp)
    const float *f0, *fm, *fp;
    long long fshot_stride;
    float* grad;                 // per shot-group slabs [groups][2][nx][ldz] (groups of spb shots)
    long long gslab_stride;
    int mode;                    // k_agrad: 0 interior snapshot, 1 the first, 2 the last
    int img;                     // k_astep: image snapshot f0 by parts in time as well
    int img_deriv;               // k_astep: 0: snapshot f0 has no 1/rho term
    float wk, dwn, dwp;          // K term weight w / dtg; k_astep: those of the neighbours less it
    float wr;                    // 1/rho term weight w dtg (halved for the first snapshot)
};
// one time step of every shot: next from prev and curr, with the point sources
void launch_astep(const AcousticArgs& a, hipStream_t s);
// imaging condition of one snapshot for every shot, into the shot groups' slabs
void launch_agrad(const AcousticArgs& a, hipStream_t s);
// initial condition: u[cell] = 1/2 scale[cell] * sum_k w[k] trace[off[k]] (scale = dt^2 K)
void launch_ainit(const InjCell* cells, int ncell, const int* ptr, const long long* off, const float* w,
                  const float* trace, float* u, long long shot_stride, int ldz, const float* kdt2, hipStream_t s);
// receivers: trace[r][it] = sum over the 9 footprint cells of w * u (shot of the receiver)
void launch_aextract(const float* u, long long shot_stride, int ldz, const PointEntry* ents, int nrec, float* trace,
                     int it, hipStream_t s);

}  // namespace fwi2d

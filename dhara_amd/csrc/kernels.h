// kernels.h -- argument blocks and host launchers of the gfx950 kernels (kernels.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.h"

namespace dh {

enum Face { FW = 0, FE = 1, FS = 2, FN = 3, FT = 4, FB = 5 };

// Row flags of the subsurface operator (only built when a Dirichlet face exists):
// identity row, or an off-diagonal coupling removed (src/subsurface.cu:144-352).
enum RowFlag : uint8_t {
    RF_IDENTITY = 1, RF_CUT_W = 2, RF_CUT_E = 4, RF_CUT_S = 8, RF_CUT_N = 16,
    RF_CUT_D = 32,   // coupling to k-1 (toward the top)
    RF_CUT_U = 64,   // coupling to k+1 (toward the bottom)
};

struct Geo {
    int nx, ny, nz, nxy, n;
    double dx, dy, dz;
    double wx, wy, wz;    // 1/dx^2, 1/dy^2, 1/dz^2
};

struct Geo2 {
    int nx, ny, n;
    double dx, dy;
    double cx, cy;        // dt/dx^2, dt/dy^2
};

struct Soil {
    const double* Ks;
    const double* alpha_f;   // nullptr: scalar alpha
    const double* n_f;       // nullptr: scalar n
    double alpha, n, ts, tr;
};

// Control block of one Krylov launch.  `it` is the iteration index within the solve (the
// host counts launches; kernels after the end of a solve return at once).  Partials of the
// previous kernel are read from part_in (nparts blocks) and this kernel's go to part_out.
struct SolveCtl {
    int it;
    int maxit;
    int mixed_inner;      // inner FP32 solve of the mixed path
    int first_sweep;      // ||b||^2 is taken from part_in (first solve of a Picard iteration)
    int segment_start;    // part_in holds a fresh residual (assembly or FP64 reliable update):
                          // read all four partials, re-check the outer residual, restart the
                          // inner target, keep the search direction
    int after_init;       // one-kernel PCG: part_in comes from the segment start-up kernel
    double lin_tol, inner_tol;
    const double* part_in;
    int nparts;
    double* part_out;
    PcgState* st;
};

// Start of a PCG update kernel (x += alpha p, r -= alpha q): alpha = (r, z) / (p, A p) from the
// SpMV kernel's (p, A p) partials and the state's (r, z); false when the solve is over (or, with
// a zero or non-finite step, marks it over).  Every block takes the same decision.
__device__ __forceinline__ bool update_begin(const SolveCtl& sc, double& alpha, int bid)
{
    PcgState* st = sc.st;
    if (st->done) return false;
    double pq[1];
    sum_partials<1>(sc.part_in, sc.nparts, 1, pq);
    const double a = st->rz[sc.it & 1] / pq[0];
    if (!(pq[0] != 0.0) || !isfinite(a)) {
        if (bid == 0 && lin_tid() == 0) {
            st->iter = sc.it;
            st->conv = 0;
            st->nan = 1;
            st->done = 1;
        }
        return false;
    }
    alpha = a;
    return true;
}

struct VgArgs {
    Geo g;
    Soil soil;
    const double* psi;       // evaluated head (x for the Picard pass)
    double* psi_m;           // Picard pass: read for the increment, then psi^m <- am psi^m + (1-am) x
    const double* theta_m;   // REL_THETA rule
    double* theta;           // out
    double* K;               // out
    double* C;               // out
    float* K32;              // out (mixed precision), may be null
    int rule;
    double am;
    int relax;               // Picard pass: 1 = write the relaxed update into psi_m (0: an
                             // Anderson pass follows and needs psi_m as it is)
    double* part_out;        // Picard pass: [max increment, NaN flag] per block
};

// Anderson-accelerated Picard update (k_picard_next).  The increment f = x - psi^m and relaxed
// update y = psi^m + beta f of this pass and of the last ncols passes, whose differences are the
// columns of dF and dY; per column of cells, the least-squares coefficients over them; then
// psi^m <- y - dY gamma and theta, K, C at it.
constexpr int kAaMaxDepth = 5;  // = DHARA_PICARD_ACCEL_MAX
constexpr double kAaDrop = 1e-3;   // a ring column is left out when its part orthogonal to the
                                   // newer ones is below this fraction of its norm
struct AaArgs {
    Geo g;
    Soil soil;
    const double* x;         // G(psi^m): the linear solve's result
    double* psi_m;           // in: psi^m, out: the next iterate
    double* theta_m;         // out: theta, K, C (K32) of the next iterate
    double* K;
    double* C;
    float* K32;
    double* f[kAaMaxDepth + 1];   // f of this pass (written) and of the previous ncols passes, newest first
    double* y[kAaMaxDepth + 1];   // y likewise
    int ncols;               // previous passes of this step in the ring, at most the depth
    double beta;             // 1 - am
    int active;              // the pass may update (not the one at the iteration limit)
};

// Whether work queued behind a solve's launches, before the host has seen how the solve ended, may run.
enum GateKind {
    GATE_OPEN,       // the host has decided
    GATE_UPDATE,     // gate == 2: the reliable update's outer test has passed (k_refine_conv)
    GATE_SOLVED,     // the solve ended, converged or at its limit, without NaN
    GATE_OUTER,      // mixed precision: the solve ended with its FP64 residual passing the outer test
};
struct Gate {
    const PcgState* st;
    int kind;
    __device__ __forceinline__ bool open() const
    {
        if (kind == GATE_OPEN) return true;
        if (kind == GATE_UPDATE) return st->gate == 2;
        return st->done && !st->nan && (kind == GATE_SOLVED || st->outer_conv);
    }
};

// What the last kernel of a queue leaves for the host, in pinned host memory (read after a stream
// synchronisation): the solver state and, if the Picard pass ran, its [increment, NaN flag].  Written
// by the kernel itself, which a copy queued behind it would make the host wait a launch longer for.
struct HostReport {
    PcgState st;
    double red[2];
    double sums[kMaxSums];   // launch_report_sums
};

// What follows a Picard increment (k_picard_next): the maxima of the increment's block partials
// [increment, NaN flag]; then, unless a NaN was seen, the Anderson update when the increment is
// not below tol (and aa.active), else theta, K, C of the converged x (fin set).  The state and the
// maxima go to rep.
struct NextArgs {
    AaArgs aa;
    VgArgs vg;
    const double* part;
    int nparts;
    int fin;
    double tol;
    Gate gate;
    HostReport* rep;
};

struct AsmArgs {
    Geo g;
    double dt, Ss, poros;
    const double *K, *C, *theta_m, *theta_n, *psi_n, *psi_m, *x;
    const double *transp, *root;
    const int* procmap;
    int has_transp;
    const int* bctype[6];
    const double* bcpsi[6];
    double* bcq[6];          // bcq[FB] is written (free drainage flux = K of the cell)
    const uint8_t* flags;
    int quirk;
    double* D;
    double* b;
    double* r;               // FP64 residual (FP64 path)
    float* D32;              // mixed path
    float* r32;
    float* d32;
    double* part_out;        // [rz, rr, bb, rr64] per block
    PcgState* st;
};

struct RefineArgs {
    Geo g;
    const double* K;
    const double* D;
    const double* b;
    double* x;
    const uint8_t* flags;
    float* r32;
    const float* D32;
    float* d32;
    double* part_out;        // [rz32, rr32, 0, rr64] per block
    PcgState* st;
};

struct SurfArgs {
    int nxy;
    double dt, dz, ts;
    const double *K, *psi_n, *theta_n, *Ks;   // top layer = first nxy cells
    double *h, *hpoten, *qcapa;
    const double *rain, *evap;
    double* qtop;                              // bcq[FT]
    int* toptype;                              // bctype[FT]
};

struct EndArgs {
    Geo g;
    double dt, Ss, poros;
    const double *x, *theta_new, *theta_m;
    double *psi_n, *theta_n;
    const double *transp, *root;
    const int* procmap;
    int has_transp;
    int carry_reference;
    const int* bctype[6];
    const double* bcq[6];
    double* part_out;        // 9 sums per block
};

struct OlfArgs {
    Geo2 g;
    double hmin, delta, K0;
    double* h;
    const double *z, *mann;
    double* H;
    double *ke, *kn;
    double *D, *b, *r;
    double* part_out;
    PcgState* st;
};

// Overland operator after elimination of the Dirichlet ring: ring rows are identity,
// interior rows couple only to interior neighbours through face conductances
// ke (east face of a cell) and kn (north face) scaled by dt/dx^2, dt/dy^2
// (src/overland.cu:65-189).
template <class PF>
__device__ __forceinline__ double op2_row(const Geo2& g, int c, double Dc, double pc, PF pf,
                                          const double* __restrict__ ke,
                                          const double* __restrict__ kn)
{
    const int j = c / g.nx, i = c - j * g.nx;
    if (i == 0 || j == 0 || i == g.nx - 1 || j == g.ny - 1) return pc;
    double acc = Dc * pc;
    if (i > 1) acc -= g.cx * ke[c - 1] * pf(c - 1);
    if (i < g.nx - 2) acc -= g.cx * ke[c] * pf(c + 1);
    if (j > 1) acc -= g.cy * kn[c - g.nx] * pf(c - g.nx);
    if (j < g.ny - 2) acc -= g.cy * kn[c] * pf(c + g.nx);
    return acc;
}

// Totals of three per-thread values, returned to every thread of the block.
__device__ __forceinline__ void block_sum3(double (&v)[3], double* lds)
{
    block_reduce<3, false>(v, lds);
}

// The overland Jacobi-PCG of a whole surface in one workgroup (surfaces of at most
// kOlfBlockCells cells; r = b - A x, D and b from k_olf_assemble; x is H).  p and q are work
// arrays of the surface's size; the solve's end is recorded in st as by the grid-wide form.
constexpr int kOlfBlockCells = 128 * 128;
constexpr int kOlfBlockThreads = 1024;
struct OlfCgArgs {
    Geo2 g;
    const double *ke, *kn, *D, *b;
    double *x, *r, *p, *q;
    double tol;
    int maxit;
    PcgState* st;
};
void launch_olf_cg_block(hipStream_t s, const OlfCgArgs& a);
// One workgroup per model of args[0 .. nmodels-1]; active[m] == 0 skips model m (active may be NULL).
void launch_batched_olf_cg_block(hipStream_t s, const OlfCgArgs* args, int nmodels, const int* active);

// Number of blocks (= partials) of the grid-stride kernels over n cells.
int grid_for(int n);

// ---- launchers (all asynchronous on `s`) ----------------------------------------------
// Optional kernel timestamps: with `start` set, a Krylov launch goes through
// hipExtLaunchKernelGGL, which stamps the two events with the kernel's own begin and end
// (what a kernel trace reports), rather than with markers queued around the launch.
struct LaunchEv {
    hipEvent_t start = nullptr, stop = nullptr;
};

void launch_vg(hipStream_t s, const VgArgs& a);                 // theta, K, C of psi
void launch_vg_picard(hipStream_t s, const VgArgs& a, const Gate& gate);   // + increment + relax
// the Picard pass's second kernel without the Anderson update: the maxima of rows 0 and 1 of part
// and the state to rep
void launch_picard_report(hipStream_t s, const double* part, int nparts, const Gate& gate, HostReport* rep);
// the state alone; the sums of the first nv rows of part (nparts partials each)
void launch_report(hipStream_t s, const PcgState* st, HostReport* rep);
void launch_report_sums(hipStream_t s, const double* part, int nparts, int nv, HostReport* rep);
// after a gated check-only update (launch_refine_line, kRefineCheck): the outer test on the
// device (st->gate = 2 when the sum of part's slot-3 partials passes lin_tol^2 ||b||^2, the sum
// in st->rr_update)
void launch_refine_conv(hipStream_t s, const double* part, int nparts, double lin_tol, PcgState* st);
// The Picard pass's second kernel with the Anderson update of depth `depth` (1..kAaMaxDepth)
void launch_picard_next(hipStream_t s, const NextArgs& a, int depth, const LaunchEv* ev = nullptr);
// Its first kernel for the rules on psi (ABS_PSI / REL_PSI): the increment of a.psi against a.psi_m
// into a.part_out
void launch_picard_inc(hipStream_t s, const VgArgs& a, const Gate& gate);
// Initial state: psi_n (read, or written from theta_n first), theta_n and the copies theta_m,
// theta_new, psi_m, x, and K, C (and K32) at psi_n.
struct InitArgs {
    Geo g;
    Soil soil;
    double *psi_n, *psi_m, *x, *theta_n, *theta_m, *theta_new, *K, *C;
    float* K32;
};
void launch_init_state(hipStream_t s, const InitArgs& a, bool from_theta);
void launch_vg_inverse(hipStream_t s, const Geo& g, const Soil& soil, const double* theta,
                       double* psi);
void launch_row_flags(hipStream_t s, const Geo& g, const int* const bctype[6], uint8_t* flags);
void launch_group_scatter(hipStream_t s, int nxy, const int* procmap, const double* groups, double* out);
void launch_surface_pre(hipStream_t s, const SurfArgs& a);
void launch_surface_post(hipStream_t s, const SurfArgs& a);
void launch_assemble(hipStream_t s, const AsmArgs& a, bool mixed);
// the same on an SpMV tile (LDS-staged K and x; untiled with Dirichlet rows or tx = 0);
// returns the number of partials written
struct TileCfg;
int launch_assemble_tiled(hipStream_t s, const AsmArgs& a, bool mixed, const TileCfg& t);
void launch_refine(hipStream_t s, const RefineArgs& a);
// the same on an SpMV tile (LDS-tiled FP64 residual; untiled with Dirichlet rows or tx = 0);
// returns the number of partials written
struct TileCfg;
int launch_refine_tiled(hipStream_t s, const RefineArgs& a, const TileCfg& t);
// reliable update of the mixed column-preconditioned PCG (flux faces, nz <= 64): x += d, then
// r32 = b - A x, d = 0 and z32 = T32^-1 r32 in one launch; partials [rz, rr, 0, rr64] to
// a.part_out; returns their number, or 0 without launching anything when the surface has more
// column tiles than partial slots.  kRefineCheck: x += d and the FP64 residual's norm only
// (partials [0, 0, 0, rr64]), both gated on the end of the segment (a.st->gate, set by a gate
// launch first: nothing runs if the segment has not ended, or ended converged or with NaN), so
// that it may be queued behind a batch; kRefineRest: r32, d, z32 and all partials of an x
// already updated.
enum RefineLineMode { kRefineFull, kRefineCheck, kRefineRest };
int launch_refine_line(hipStream_t s, const RefineArgs& a, float* z32, RefineLineMode mode = kRefineFull);
void launch_end_step(hipStream_t s, const EndArgs& a);

// Jacobi-PCG iteration `sc.it` on the 3D operator, split in its two kernels:
//   spmv:   p = M^-1 r + beta p (p[it&1] -> p[(it+1)&1]), q = A p, partial (p, q)
//   update: x += alpha p, r -= alpha q, partials (r, M^-1 r), (r, r)
void launch_pcg3_spmv_f64(hipStream_t s, const Geo& g, const uint8_t* flags, const double* K,
                          const double* D, const double* r, double* const p[2], double* q,
                          const SolveCtl& sc, const LaunchEv& ev = LaunchEv{});
void launch_pcg3_spmv_f32(hipStream_t s, const Geo& g, const uint8_t* flags, const float* K,
                          const float* D, const float* r, float* const p[2], float* q,
                          const SolveCtl& sc, const LaunchEv& ev = LaunchEv{});
void launch_pcg_update_f64(hipStream_t s, int n, double* x, double* r, const double* D,
                           const double* p, const double* q, const SolveCtl& sc, const LaunchEv& ev = LaunchEv{});
void launch_pcg_update_f32(hipStream_t s, int n, float* x, float* r, const float* D,
                           const float* p, const float* q, const SolveCtl& sc, const LaunchEv& ev = LaunchEv{});
// LDS-tiled 2.5D variant of the SpMV kernel: a TX x TY tile of columns marches through a
// chunk of kc planes; the p/K planes are staged in LDS with a one-cell halo, the vertical
// neighbours stay in registers.  Returns the number of blocks (= partials for the update).
struct TileCfg {
    int tx, ty, kc;
    int grid = 0;   // one-kernel PCG: at most this many blocks (multiple of 8), 0 = one per tile
};
bool tile_supported(const TileCfg& t);
int tile_blocks(const Geo& g, const TileCfg& t);
void launch_pcg3_spmv_tiled_f64(hipStream_t s, const Geo& g, const TileCfg& t, const uint8_t* flags,
                                const double* K, const double* D, const double* r, double* const p[2],
                                double* q, const SolveCtl& sc, const LaunchEv& ev = LaunchEv{});
void launch_pcg3_spmv_tiled_f32(hipStream_t s, const Geo& g, const TileCfg& t, const uint8_t* flags,
                                const float* K, const float* D, const float* r, float* const p[2],
                                float* q, const SolveCtl& sc, const LaunchEv& ev = LaunchEv{});
// One kernel per Jacobi-PCG iteration (single-reduction recurrences, no Dirichlet rows):
// iteration sc.it reads r_in and p_in (= p_{it-1}), writes r_out, p_out and x in place, and
// the partials [gamma, rho, delta, eps, pi]; k_cg1_init starts a segment from a fresh residual
// (partials [rz, rr, bb, rr64] of the assembly or of a reliable update).
bool cg1_tile_supported(const TileCfg& t);
int cg1_blocks(const Geo& g, const TileCfg& t);
constexpr int kCg1FillTiles = 400;   // blocks up to which a small surface's columns are split
int cg1_default_planes(const Geo& g);   // planes per block of the 32 x 8 tile when none is set or tuned
void launch_cg1_f64(hipStream_t s, const Geo& g, const TileCfg& t, const double* K, const double* D,
                    const double* r_in, double* r_out, const double* p_in, double* p_out, double* x,
                    const SolveCtl& sc, const LaunchEv& ev = LaunchEv{});
void launch_cg1_f32(hipStream_t s, const Geo& g, const TileCfg& t, const float* K, const float* D,
                    const float* r_in, float* r_out, const float* p_in, float* p_out, float* x,
                    const SolveCtl& sc, const LaunchEv& ev = LaunchEv{});
// start-up kernel on the SpMV tile t (tx = 0: untiled); cg1_init_blocks = its partial count
int cg1_init_blocks(const Geo& g, const TileCfg& t);
void launch_cg1_init_f64(hipStream_t s, const Geo& g, const TileCfg& t, const double* K, const double* D,
                         const double* r, const double* p_old, const SolveCtl& sc, const LaunchEv& ev = LaunchEv{});
void launch_cg1_init_f32(hipStream_t s, const Geo& g, const TileCfg& t, const float* K, const float* D,
                         const float* r, const float* p_old, const SolveCtl& sc, const LaunchEv& ev = LaunchEv{});
// Column-preconditioned PCG (z = T^-1 r, T the vertical tridiagonal part of A; no Dirichlet rows,
// nz <= kLineMaxNz), two kernels per iteration:
//   spmv_z: p = z + beta p (p[it&1] -> p[(it+1)&1]), q = A p, partial (p, q) -- tiled on t
//           (t.tx = 0: untiled); its partial count is tile_blocks / grid_for(n) as for Jacobi
//   line update: x += alpha p, r -= alpha q, z = T^-1 r, partials [(r, z), (r, r)]
//   line init (segment start): z = T^-1 r, partials [(r, z), (r, r)] + slots 2, 3 of the
//           assembly / reliable-update partials
// The line kernels write line_blocks(g) partials.
constexpr int kLineMaxNz = 64;
bool line_supported(const Geo& g);
int line_blocks(const Geo& g);
void launch_pcg3_spmv_z_f64(hipStream_t s, const Geo& g, const TileCfg& t, const double* K, const double* D,
                            const double* z, double* const p[2], double* q, const SolveCtl& sc,
                            const LaunchEv& ev = LaunchEv{});
void launch_pcg3_spmv_z_f32(hipStream_t s, const Geo& g, const TileCfg& t, const float* K, const float* D,
                            const float* z, float* const p[2], float* q, const SolveCtl& sc,
                            const LaunchEv& ev = LaunchEv{});
void launch_line_init_f64(hipStream_t s, const Geo& g, const double* K, const double* D, const double* r, double* z,
                          const SolveCtl& sc, const LaunchEv& ev = LaunchEv{});
void launch_line_init_f32(hipStream_t s, const Geo& g, const float* K, const float* D, const float* r, float* z,
                          const SolveCtl& sc, const LaunchEv& ev = LaunchEv{});
void launch_line_update_f64(hipStream_t s, const Geo& g, const double* K, const double* D, double* x, double* r,
                            const double* p, const double* q, double* z, const SolveCtl& sc,
                            const LaunchEv& ev = LaunchEv{});
void launch_line_update_f32(hipStream_t s, const Geo& g, const float* K, const float* D, float* x, float* r,
                            const float* p, const float* q, float* z, const SolveCtl& sc,
                            const LaunchEv& ev = LaunchEv{});
// y = A x (tests)
void launch_apply3_f64(hipStream_t s, const Geo& g, const uint8_t* flags, const double* K,
                       const double* D, const double* x, double* y);
void launch_apply3_f32(hipStream_t s, const Geo& g, const uint8_t* flags, const float* K,
                       const float* D, const float* x, float* y);
void launch_cast_f32(hipStream_t s, int n, const double* in, float* out);
void launch_cast_f64(hipStream_t s, int n, const float* in, double* out);

// Overland
void launch_olf_faces(hipStream_t s, const OlfArgs& a);   // H = h + z and the face conductances
void launch_olf_assemble(hipStream_t s, const OlfArgs& a);
void launch_pcg2_spmv(hipStream_t s, const Geo2& g, const double* ke, const double* kn,
                      const double* D, const double* r, double* const p[2], double* q, const SolveCtl& sc);
void launch_olf_post(hipStream_t s, const OlfArgs& a);

// ---- batched launches over an ensemble of models (kernels.hip) ----------------------------
// A batched launch runs one kernel body for many models at once: physical block b works as
// block map[b].id of map[b].n blocks of model map[b].m, with that model's argument struct.
// Models whose active flag is 0 return at once.
struct BlkMap {
    int m, id, n;
};
// Krylov arguments of one model for batched solves (the iteration index comes from *it_base
// plus the launch's position k in the batch, so a captured batch can be replayed unchanged).
template <typename T>
struct KrylovArgs {
    Geo g;
    Geo2 g2;
    const T *K, *D, *r;
    T *x, *res, *p[2], *q;
    const double *ke, *kn;       // overland operator (2D solves)
    SolveCtl spmv, upd;          // part_in/part_out/st of the two kernels; `it` is ignored
    // column-preconditioned form: z = T^-1 r, the start-up kernel's control (reads the assembly /
    // refinement partials, writes part_first) and the partials the first SpMV reads
    T* z;
    SolveCtl init;
    const double* part_first;
    // batched solves: the iteration index of the model's current segment is *it_base + k - seg0
    // (a model whose segment restarts while others keep iterating starts again at 0)
    int seg0;
};
// One-kernel PCG of one model in a batched launch: tiles of kCg1BatchTx x kCg1BatchTy columns
// and kc planes, one block per tile.  Iteration it reads r[it & 1], p[(it + 1) & 1] and the
// partials part[(it + 1) & 1], writes r[(it + 1) & 1], p[it & 1], x and part[it & 1]; the
// start-up reads the assembly / reliable-update partials part_asm and writes part[1].  Every
// solve (and every refinement round) restarts at it = 0.
template <typename T>
struct Cg1Args {
    Geo g;
    const T *K, *D;
    T *r[2], *p[2], *x;
    double *part_asm, *part[2];
    int nparts_asm, ntiles;
    int kc, ntx, nty, nkz;
    SolveCtl ctl;                // maxit, tolerances, mixed_inner, first_sweep, st
};
constexpr int kCg1BatchTx = 32, kCg1BatchTy = 8;
// start-up on the map of the grid-stride kernels (grid_for(N) blocks per model)
void launch_batched_cg1_init(hipStream_t s, bool fp32, const void* args, const BlkMap* map, int nblocks,
                             const int* active);
// iteration *it_base + k on the tile map
void launch_batched_cg1(hipStream_t s, bool fp32, const void* args, const BlkMap* map, int nblocks,
                        const int* active, const int* it_base, int k);
enum BatchKind { BK_VG = 0, BK_VG_PICARD, BK_SURF_PRE, BK_SURF_POST, BK_ASM_F64, BK_ASM_MIXED,
                 BK_REFINE_ADD, BK_REFINE_RES, BK_END, BK_OLF_FACES, BK_OLF_ASM, BK_OLF_POST,
                 BK_PICARD_INC };   // BK_PICARD_INC: VgArgs, the increment of psi (x) over psi_m alone
// args points to an array of the argument struct of the kind (VgArgs, SurfArgs, AsmArgs,
// RefineArgs, EndArgs or OlfArgs), one per model.
void launch_batched(hipStream_t s, BatchKind kind, const void* args, const BlkMap* map, int nblocks,
                    const int* active);
// Column-preconditioned form (untiled SpMV with z as input over map3; the column kernel over a map
// of line_blocks(g) blocks per member, nz_max the planes of the tallest member; init: the start-up
// z = T^-1 r of a fresh residual).
void launch_batched_spmv_z(hipStream_t s, bool fp32, const void* kargs, const BlkMap* map, int nblocks,
                           const int* active, const int* it_base, int k);
// Anderson pass of the active members (the host has decided), over a map of aa_blocks(g) blocks
// per member; every member has the same depth.
void launch_batched_aa(hipStream_t s, int depth, const AaArgs* args, const BlkMap* map, int nblocks,
                       const int* active);
int aa_blocks(const Geo& g);
void launch_batched_line(hipStream_t s, bool fp32, bool init, int nz_max, const void* kargs, const BlkMap* map,
                         int nblocks, const int* active, const int* it_base, int k);
void launch_batched_spmv3(hipStream_t s, bool fp32, const void* kargs, const BlkMap* map, int nblocks,
                          const int* active, const int* it_base, int k);
void launch_batched_update3(hipStream_t s, bool fp32, const void* kargs, const BlkMap* map, int nblocks,
                            const int* active, const int* it_base, int k);
void launch_batched_spmv2(hipStream_t s, const void* kargs, const BlkMap* map, int nblocks, const int* active,
                          const int* it_base, int k);
void launch_batched_update2(hipStream_t s, const void* kargs, const BlkMap* map, int nblocks, const int* active,
                            const int* it_base, int k);
// *it_base += by, and the nst solver states to out (pinned host memory).
void launch_advance(hipStream_t s, int* it_base, int by, const PcgState* st, int nst, PcgState* out);
// active[m] = flags[m] (pinned host memory) of M models, and for each of n block maps cur = the blocks
// full[start[m] .. start[m] + count[m]) of the models whose flag is set, in the models' order.
struct ActMap {
    const BlkMap* full;
    const int *start, *count;
    BlkMap* cur;
};
struct ActMaps {
    ActMap m[4];
    int n;
};
void launch_activate(hipStream_t s, const int* flags, int M, int* active, const ActMaps& maps);
// out[m*nv + v] = sum (or max) of row v of model m's partials part[m] (nparts[m] entries),
// in block order; one block per model.
void launch_reduce_models(hipStream_t s, int nmodels, const double* const* part, const int* nparts, int nv,
                          bool take_max, double* out);

// ---- overland multigrid preconditioner (olf_mg.hip) ---------------------------------------
// One level of the 2 x 2 aggregation hierarchy: operator A = d - weights (we: cell to its east
// neighbour, wn: to its north neighbour), right-hand side b, pre-smoothed x, V-cycle result y.
struct MgLevel {
    int nx, ny;
    double *d, *we, *wn, *b, *x, *y;
};
constexpr int kMgMaxLevels = 24;
struct MgHier {
    int nlev;
    MgLevel lv[kMgMaxLevels];
    int le;          // coarsest level used: solved exactly with the dense inverse inv
    double* inv;     // kMgExactCells^2 doubles: (level le's operator)^-1, row-major
};
constexpr int kMgExactCells = 64;   // the V-cycle bottoms out on the first coarse level this small
int mg_exact_level(const MgHier& h);   // that level
int mg_levels(int nx, int ny, int dims[][2]);   // level sizes down to 1 x 1; returns the count
int mg_coarse_level(const MgHier& h);           // first level handled by the single-block kernel
int mg_partials(const MgHier& h);               // blocks of the V-cycle's last kernel (single-reduction form)
// Level-0 weights from the face conductances and the Galerkin operators of all coarse levels.
void launch_mg_setup(hipStream_t s, const Geo2& g, const double* ke, const double* kn, const MgHier& h);
void launch_mg_vcycle(hipStream_t s, const MgHier& h);   // y_0 = V-cycle(b_0)

// Single-reduction (Chronopoulos-Gear) form of the multigrid-preconditioned overland CG, for
// surfaces whose V-cycle has tiled levels (mg_coarse_level(h) > 0).  The V-cycle's last kernel
// also forms w = A z and the partial sums [(r, z), (r, r), (w, z), (bb_src, bb_src)]; iteration
// i is then the V-cycle alone, its first kernel starting with the CG update:
//   beta = gamma_i / gamma_{i-1}, pi_i = delta_i - beta^2 pi_{i-1}, alpha = gamma_i / pi_i,
//   s = w + beta s_old, r_new = r_old - alpha s (tile and halo), p = z + beta p, x += alpha p,
// so an iteration needs no SpMV kernel.  r and s are read across the tile halo and must
// alternate between two buffers each; p, z and x are read only inside the tile.
struct MgCg1 {
    SolveCtl sc;
    double* x;
    double* p;
    const double* z;
    double* w;
    const double* s_old;
    double* s_new;
    const double* r_old;
    double* r_new;
};
// The multigrid-preconditioned overland CG of a whole surface of at most kOlfBlockCells cells
// in one workgroup (the one-workgroup Jacobi-PCG's iteration with z = V-cycle(r)): the level-0
// weights, the Galerkin coarse operators and the exact level's inverse are formed in the same
// launch; h's level arrays are its work space (level 0: d = the assembled D, y = z).
struct OlfMgArgs {
    OlfCgArgs cg;
    MgHier h;
};
void launch_olf_mgcg_block(hipStream_t s, const OlfMgArgs& a);
// One workgroup per model of args[0 .. nmodels-1]; active[m] == 0 skips model m.
void launch_batched_olf_mgcg_block(hipStream_t s, const OlfMgArgs* args, int nmodels, const int* active);

// The same for surfaces that fit one workgroup's registers and LDS (mg_small: up to 64 x 64 cells and
// shapes like it); of h only the levels' sizes are used.
bool mg_small(const MgHier& h);
void launch_olf_mgcg_small(hipStream_t s, const OlfMgArgs& a);

// z_0 = V-cycle(r_0), w_0 = A z_0, partials of the above (bb_src: the right-hand side).
void launch_mg_vcycle_cg1_start(hipStream_t s, const MgHier& h, const PcgState* st, double* part,
                                const double* bb_src, double* w);
void launch_mg_vcycle_cg1(hipStream_t s, const MgHier& h, const PcgState* st, double* part, const MgCg1& v);

}  // namespace dh

// olf_mg.hip -- multigrid preconditioner of the overland solve (gfx950).
//
// The overland system of one step (src/overland.cu:65-189, Dirichlet ring eliminated) is a
// symmetric 5-point operator A = d - (east/north face weights) whose coefficients jump by six
// orders of magnitude between dry faces (K0) and ponded ones; Jacobi-preconditioned CG needs
// ~1500 iterations per step on a 400 x 400 surface.  This preconditioner is one V-cycle of
// unsmoothed-aggregation multigrid:
//   * levels: 2 x 2 aggregates, Galerkin coarse operators P^T A P with P piecewise constant --
//     on a structured grid these stay 5-point (d, we, wn), so every level uses the same kernels
//     -- down to the first level of at most 64 cells, which is solved exactly with its dense
//     inverse (formed once per overland step);
//   * smoothing: two red-black Gauss-Seidel sweeps before (red first) and after (black first)
//     the coarse correction, which keeps the V-cycle symmetric, so CG stays valid; the cell
//     update multiplies by the reciprocal of the diagonal (held in LDS);
//   * coarse correction scaled by 1.2 (over-correction for piecewise-constant interpolation;
//     1.5 took 17 % more iterations on the 400 x 400 coupled run, 1.1 to 1.25 about the same);
//   * a thread owns a 2 x 2 aggregate (two red and two black cells): its operator, right-hand
//     side and iterate stay in registers and only the iterate is exchanged, through four LDS
//     planes (one per cell of the aggregate, so every access is stride 1);
//   * the first red half-sweep from x = 0 needs no neighbours, the residual of the cells smoothed
//     last is zero, so the restriction sums the red residuals alone, and the post-smoothing starts
//     by overwriting the black cells, so only red x and y are carried between the kernels;
//   * large levels: one tiled kernel down (smooth, residual, restrict) and one up (prolong,
//     smooth) per level; a tile of 32 x 32 cells works with a halo of 4 cells (6 where A z is
//     formed too) recomputed redundantly, so the half-sweeps need no grid-wide synchronisation
//     and the tile interior equals a global sweep exactly;
//   * the coarsest levels (as many as give one aggregate to each of 1024 threads: 50 x 50 down to
//     7 x 7 on a 400 x 400 surface): the rest of the V-cycle in one single-block kernel, every
//     level's aggregates on threads of their own.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.h"

namespace dh {

constexpr double kMgOver = 1.2;   // coarse-correction scaling
constexpr int kMgT = 32;          // tile edge of the large-level kernels (even)
constexpr int kMgHalo = 2;        // halo in aggregates: the three half-sweeps after the first and the residual
constexpr int kMgHaloA = 3;       // the four half-sweeps after the prolongation, and A z
constexpr int kMgThreads = 1024;   // threads of the single-block kernels

// The first level handled by the single-block kernel: the finest whose aggregates and those of
// every coarser level (an aggregate of a level is a cell of the next) fit its threads (50 x 50 ...
// 7 x 7 on a 400 x 400 surface).  Host and device use the same rule.
__host__ __device__ inline int mg_first_single_block(const MgHier& h)
{
    int l = h.le, aggs = 0;
    while (l > 0 && aggs + h.lv[l].nx * h.lv[l].ny <= kMgThreads) {
        aggs += h.lv[l].nx * h.lv[l].ny;
        --l;
    }
    return l;
}

namespace {

__device__ __forceinline__ int mg_coarse_first(const MgHier& h) { return mg_first_single_block(h); }

// Level-0 operator: the eliminated overland matrix.  Diagonal = the assembled D (ring rows 1);
// weights only between two interior cells (couplings to the ring moved to the right-hand side).
__device__ __forceinline__ void mg_fine_cell(const Geo2& g, const double* ke, const double* kn, double* we, double* wn,
                                             int i, int j)
{
    const int c = j * g.nx + i;
    const bool in = i > 0 && j > 0 && i < g.nx - 1 && j < g.ny - 1;
    we[c] = (in && i + 1 < g.nx - 1) ? g.cx * ke[c] : 0.0;
    wn[c] = (in && j + 1 < g.ny - 1) ? g.cy * kn[c] : 0.0;
}

__device__ __forceinline__ void mg_fine_cells(const Geo2& g, const double* ke, const double* kn, double* we,
                                              double* wn, int first, int stride)
{
    for (int c = first; c < g.n; c += stride) mg_fine_cell(g, ke, kn, we, wn, c % g.nx, c / g.nx);
}

// Galerkin coarse operator of 2 x 2 aggregates: d_C = sum d_f - 2 (couplings inside C),
// weight between C and its east/north neighbour = sum of the fine couplings that cross.
__device__ __forceinline__ void mg_coarsen_cells(const MgLevel& F, const MgLevel& C, int first, int stride)
{
    for (int cc = first; cc < C.nx * C.ny; cc += stride) {
        const int J = cc / C.nx, I = cc - J * C.nx;
        const int i0 = 2 * I, j0 = 2 * J;
        const bool i1 = i0 + 1 < F.nx, j1 = j0 + 1 < F.ny;
        double d = 0.0, e = 0.0, n = 0.0;
        for (int dj = 0; dj < (j1 ? 2 : 1); ++dj)
            for (int di = 0; di < (i1 ? 2 : 1); ++di) {
                const int f = (j0 + dj) * F.nx + i0 + di;
                d += F.d[f];
                if (di == 0 && i1) d -= 2.0 * F.we[f];        // (i0, i0+1) inside C
                if (di == 1 || !i1) e += F.we[f];             // crosses to the east aggregate
                if (dj == 0 && j1) d -= 2.0 * F.wn[f];
                if (dj == 1 || !j1) n += F.wn[f];
            }
        C.d[cc] = d;
        C.we[cc] = e;
        C.wn[cc] = n;
    }
}

__global__ __launch_bounds__(kBlock) void k_mg_coarsen(MgLevel F, MgLevel C)
{
    mg_coarsen_cells(F, C, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}

// The level-0 weights and the operator of level 1 (whose cells need only their own children's).
__global__ __launch_bounds__(kBlock) void k_mg_fine_coarsen(Geo2 g, const double* __restrict__ ke,
                                                            const double* __restrict__ kn, MgLevel F, MgLevel C)
{
    for (int cc = blockIdx.x * blockDim.x + threadIdx.x; cc < C.nx * C.ny; cc += gridDim.x * blockDim.x) {
        const int J = cc / C.nx, I = cc - J * C.nx;
        for (int dj = 0; dj < 2; ++dj)
            for (int di = 0; di < 2; ++di)
                if (2 * I + di < F.nx && 2 * J + dj < F.ny) mg_fine_cell(g, ke, kn, F.we, F.wn, 2 * I + di, 2 * J + dj);
        mg_coarsen_cells(F, C, cc, C.nx * C.ny);   // this cell alone
    }
}

// A thread's 2 x 2 aggregate of a level: cells 0 (i, j), 1 (i + 1, j), 2 (i, j + 1), 3 (i + 1, j + 1)
// with i and j even, so 0 and 3 are red and 1 and 2 black.  Cells outside the level have d = 1,
// b = 0 and no couplings.
struct MgAgg {
    double b[4], d[4], di[4], x[4];
    double h0, h1, v0, v1;                   // couplings inside: 0-1, 2-3, 0-2, 1-3
    double w0, w2, e1, e3, s0, s1, n2, n3;   // and out: west, east, south (j - 1), north
};

struct MgIn {
    bool c[4];   // cell inside the level
};

__device__ __forceinline__ MgIn agg_in(const MgLevel& L, int gi, int gj)
{
    MgIn in;
    in.c[0] = gi >= 0 && gj >= 0 && gi < L.nx && gj < L.ny;
    in.c[1] = in.c[0] && gi + 1 < L.nx;
    in.c[2] = in.c[0] && gj + 1 < L.ny;
    in.c[3] = in.c[1] && in.c[2];
    return in;
}

__device__ __forceinline__ double ld_if(bool in, const double* __restrict__ p, int g, double other)
{
    return in ? p[g] : other;
}

// The operator of the aggregate at (gi, gj).
__device__ __forceinline__ void agg_load(const MgLevel& L, int gi, int gj, const MgIn& in, MgAgg& a)
{
    const int nx = L.nx, g = gj * nx + gi;
    a.d[0] = ld_if(in.c[0], L.d, g, 1.0);
    a.d[1] = ld_if(in.c[1], L.d, g + 1, 1.0);
    a.d[2] = ld_if(in.c[2], L.d, g + nx, 1.0);
    a.d[3] = ld_if(in.c[3], L.d, g + nx + 1, 1.0);
    const bool we = gi > 0, ea = gi + 2 < nx, so = gj > 0, no = gj + 2 < L.ny;
    a.h0 = ld_if(in.c[1], L.we, g, 0.0);
    a.h1 = ld_if(in.c[3], L.we, g + nx, 0.0);
    a.w0 = ld_if(in.c[0] && we, L.we, g - 1, 0.0);
    a.w2 = ld_if(in.c[2] && we, L.we, g + nx - 1, 0.0);
    a.e1 = ld_if(in.c[1] && ea, L.we, g + 1, 0.0);
    a.e3 = ld_if(in.c[3] && ea, L.we, g + nx + 1, 0.0);
    a.v0 = ld_if(in.c[2], L.wn, g, 0.0);
    a.v1 = ld_if(in.c[3], L.wn, g + 1, 0.0);
    a.s0 = ld_if(in.c[0] && so, L.wn, g - nx, 0.0);
    a.s1 = ld_if(in.c[1] && so, L.wn, g - nx + 1, 0.0);
    a.n2 = ld_if(in.c[2] && no, L.wn, g + nx, 0.0);
    a.n3 = ld_if(in.c[3] && no, L.wn, g + nx + 1, 0.0);
}

__device__ __forceinline__ void agg_invert(MgAgg& a)
{
#pragma unroll
    for (int c = 0; c < 4; ++c) a.di[c] = 1.0 / a.d[c];
}

// The LDS planes of a grid of aggregates: plane c holds cell c of every aggregate, with a border of
// zeros; `q` is this thread's slot of plane 0, `pitch` the slots of a row, `plane` of a plane.
struct MgPlanes {
    double* q;
    int pitch, plane;
    __device__ __forceinline__ double at(int c, int off) const { return q[c * plane + off]; }
    __device__ __forceinline__ void put(int c, double v) const { q[c * plane] = v; }
};

// Zeros around the planes (the border slots that a neighbour read can reach), by the edge threads.
__device__ __forceinline__ void planes_border(const MgPlanes& s, bool west, bool east, bool south, bool north)
{
    if (west) { s.q[s.plane - 1] = 0.0; s.q[3 * s.plane - 1] = 0.0; }
    if (east) { s.q[1] = 0.0; s.q[2 * s.plane + 1] = 0.0; }
    if (south) { s.q[2 * s.plane - s.pitch] = 0.0; s.q[3 * s.plane - s.pitch] = 0.0; }
    if (north) { s.q[s.pitch] = 0.0; s.q[s.plane + s.pitch] = 0.0; }
}

// Sums of the couplings times the neighbours' values of the red cells (0, 3) and of the black ones (1, 2).
__device__ __forceinline__ void red_sums(const MgAgg& a, const MgPlanes& s, double& t0, double& t3)
{
    t0 = a.h0 * a.x[1] + a.w0 * s.at(1, -1) + a.v0 * a.x[2] + a.s0 * s.at(2, -s.pitch);
    t3 = a.e3 * s.at(2, 1) + a.h1 * a.x[2] + a.n3 * s.at(1, s.pitch) + a.v1 * a.x[1];
}
__device__ __forceinline__ void black_sums(const MgAgg& a, const MgPlanes& s, double& t1, double& t2)
{
    t1 = a.e1 * s.at(0, 1) + a.h0 * a.x[0] + a.v1 * a.x[3] + a.s1 * s.at(3, -s.pitch);
    t2 = a.h1 * a.x[3] + a.w2 * s.at(3, -1) + a.n2 * s.at(0, s.pitch) + a.v0 * a.x[0];
}
__device__ __forceinline__ void put_red(const MgAgg& a, const MgPlanes& s)
{
    s.put(0, a.x[0]);
    s.put(3, a.x[3]);
}
__device__ __forceinline__ void red_sweep(MgAgg& a, const MgPlanes& s)
{
    double t0, t3;
    red_sums(a, s, t0, t3);
    a.x[0] = (a.b[0] + t0) * a.di[0];
    a.x[3] = (a.b[3] + t3) * a.di[3];
    put_red(a, s);
}
__device__ __forceinline__ void black_sweep(MgAgg& a, const MgPlanes& s)
{
    double t1, t2;
    black_sums(a, s, t1, t2);
    a.x[1] = (a.b[1] + t1) * a.di[1];
    a.x[2] = (a.b[2] + t2) * a.di[2];
    s.put(1, a.x[1]);
    s.put(2, a.x[2]);
}

// Two forward sweeps from x = 0 and the restricted residual of the aggregate (returned).  Every
// thread of the block calls it; `on`: this thread has an aggregate.
__device__ __forceinline__ double agg_down(MgAgg& a, const MgPlanes& s, bool on)
{
    double u0 = 0.0, u3 = 0.0, t0 = 0.0, t3 = 0.0;
    if (on) {
        a.x[0] = a.b[0] * a.di[0];
        a.x[3] = a.b[3] * a.di[3];
        put_red(a, s);
    }
    __syncthreads();
    if (on) black_sweep(a, s);
    __syncthreads();
    if (on) {
        red_sums(a, s, u0, u3);
        a.x[0] = (a.b[0] + u0) * a.di[0];
        a.x[3] = (a.b[3] + u3) * a.di[3];
        put_red(a, s);
    }
    __syncthreads();
    if (on) black_sweep(a, s);
    __syncthreads();
    if (on) red_sums(a, s, t0, t3);   // d x + couplings changed by t - u since the red cells were set
    return (t0 - u0) + (t3 - u3);
}

// Two backward sweeps on the prolonged iterate (its red cells, in a.x[0] and a.x[3]); the last
// red values are in the registers and, if put, in the planes (no barrier after them).
__device__ __forceinline__ void agg_up(MgAgg& a, const MgPlanes& s, bool on, bool put)
{
    if (on) put_red(a, s);
    __syncthreads();
    if (on) black_sweep(a, s);
    __syncthreads();
    if (on) red_sweep(a, s);
    __syncthreads();
    if (on) black_sweep(a, s);
    __syncthreads();
    if (on) {
        double t0, t3;
        red_sums(a, s, t0, t3);
        a.x[0] = (a.b[0] + t0) * a.di[0];
        a.x[3] = (a.b[3] + t3) * a.di[3];
        if (put) put_red(a, s);
    }
}

// Start of iteration sc.it of the single-reduction CG (MgCg1): the stopping test on (r, r)
// (||b||^2 from the first iteration's partials), then beta, pi and alpha; false when the solve
// is over.  Every block takes the same decision from the same fixed-order sums.
__device__ __forceinline__ bool olf_cg1_begin(const SolveCtl& sc, double& alpha, double& beta, int bid)
{
    PcgState* st = sc.st;
    if (st->done) return false;
    const bool fresh = sc.it == 0;
    double in[4];
    sum_partials<4>(sc.part_in, sc.nparts, fresh ? 4 : 3, in);
    const double gam = in[0], rr = in[1], del = in[2];
    const bool lead = bid == 0 && lin_tid() == 0;
    double tol2;
    int nan = !isfinite(rr);
    if (fresh) {
        tol2 = sc.lin_tol * sc.lin_tol * in[3];
        nan |= !isfinite(in[3]);
        if (lead) {
            st->bb = in[3];
            st->tol2 = tol2;
        }
    } else {
        tol2 = st->tol2;
    }
    const int conv = (rr <= tol2) ? 1 : 0;
    if (conv || nan || sc.it >= sc.maxit) {
        if (lead) {
            st->iter = sc.it;
            st->conv = conv;
            st->rr = rr;
            st->nan = st->nan | nan;
            st->outer_conv = conv;
            st->done = 1;
        }
        return false;
    }
    const double b = fresh ? 0.0 : gam / st->rz[(sc.it - 1) & 1];
    const double pi = fresh ? del : del - b * b * st->pi[(sc.it - 1) & 1];
    const double a = gam / pi;
    if (!(pi > 0.0) || !isfinite(a) || !isfinite(b)) {
        if (lead) {
            st->iter = sc.it;
            st->conv = 0;
            st->nan = 1;
            st->done = 1;
        }
        return false;
    }
    if (lead) {
        st->rz[sc.it & 1] = gam;
        st->pi[sc.it & 1] = pi;
    }
    alpha = a;
    beta = b;
    return true;
}

// Threads of a tile of kMgT x kMgT cells with a halo of H aggregates.
constexpr int mg_tile_threads(int H)
{
    const int n = (kMgT / 2 + 2 * H) * (kMgT / 2 + 2 * H);
    return (n + kWave - 1) / kWave * kWave;
}

// The aggregate of this thread in the tile of this block.
template <int H>
struct MgTile {
    static constexpr int NB = kMgT / 2 + 2 * H, P = NB + 2;
    int I, J, gi, gj;
    bool on, interior;
    __device__ __forceinline__ explicit MgTile(const MgLevel& L)
    {
        const int ntx = (L.nx + kMgT - 1) / kMgT;
        const int t = threadIdx.x;
        J = t / NB;
        I = t - J * NB;
        on = t < NB * NB;
        gi = (int)(blockIdx.x % ntx) * kMgT + 2 * (I - H);
        gj = (int)(blockIdx.x / ntx) * kMgT + 2 * (J - H);
        interior = on && I >= H && J >= H && I < NB - H && J < NB - H;
    }
    __device__ __forceinline__ MgPlanes planes(double* sx) const
    {
        return MgPlanes{sx + (on ? (J + 1) * P + I + 1 : P + 1), P, P * P};
    }
    __device__ __forceinline__ void border(const MgPlanes& s) const
    {
        if (on) planes_border(s, I == 0, I == NB - 1, J == 0, J == NB - 1);
    }
};

// Down: x = 2 forward RBGS sweeps from 0 on b, b_coarse = P^T (b - A x).  CG1 (level 0 of the
// single-reduction CG): b is the CG residual after this iteration's update, done here (see MgCg1).
// Every load is issued before the partial sums are reduced, so that their latency overlaps it.
// Bound by latency (one tile is ~8 us of dependent steps, a surface of 400 x 400 169 tiles on 256
// CUs).  With the operator in LDS (ten LDS reads per cell and half-sweep, 80 KB a tile) these
// kernels took 12.9 us (CG1) and 5.7 us.
template <bool CG1>
__global__ __launch_bounds__(mg_tile_threads(kMgHalo)) void k_mg_down(MgLevel L, MgLevel C, const PcgState* st, MgCg1 v)
{
    using Tile = MgTile<kMgHalo>;
    __shared__ double sx[4 * Tile::P * Tile::P];
    const Tile t(L);
    const MgPlanes s = t.planes(sx);
    const MgIn in = agg_in(L, t.gi, t.gj);
    const bool on = t.on;
    const int nx = L.nx, g = t.gj * nx + t.gi;
    const int off[4] = {0, 1, nx, nx + 1};
    MgAgg a;
    if constexpr (CG1) {
        const bool first = v.sc.it == 0;
        double w[4], so[4], ro[4], z[4], p[4], x[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const bool i = on && in.c[c], ii = t.interior && in.c[c];
            w[c] = ld_if(i, v.w, g + off[c], 0.0);
            so[c] = ld_if(i && !first, v.s_old, g + off[c], 0.0);
            ro[c] = ld_if(i, v.r_old, g + off[c], 0.0);
            z[c] = ld_if(ii, v.z, g + off[c], 0.0);
            p[c] = ld_if(ii && !first, v.p, g + off[c], 0.0);
            x[c] = ld_if(ii, v.x, g + off[c], 0.0);
        }
        if (on) agg_load(L, t.gi, t.gj, in, a);
        double alpha, beta;
        if (!olf_cg1_begin(v.sc, alpha, beta, blockIdx.x)) return;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const double sn = w[c] + beta * so[c];
            a.b[c] = ro[c] - alpha * sn;
            if (t.interior && in.c[c]) {
                v.s_new[g + off[c]] = sn;
                v.r_new[g + off[c]] = a.b[c];
                const double pn = z[c] + beta * p[c];
                v.p[g + off[c]] = pn;
                v.x[g + off[c]] = x[c] + alpha * pn;
            }
        }
    } else {
        const int done = st ? st->done : 0;
        if (on) {
            agg_load(L, t.gi, t.gj, in, a);
#pragma unroll
            for (int c = 0; c < 4; ++c) a.b[c] = ld_if(in.c[c], L.b, g + off[c], 0.0);
        }
        if (done) return;
    }
    if (on) agg_invert(a);
    t.border(s);
    const double rc = agg_down(a, s, on);
    if (t.interior && in.c[0]) {
        C.b[(t.gj >> 1) * C.nx + (t.gi >> 1)] = rc;
        L.x[g] = a.x[0];
        if (in.c[3]) L.x[g + nx + 1] = a.x[3];
    }
}

// Up: x = x_l + 1.2 P y_{l+1}, 2 backward RBGS sweeps, written to out.  CG1 (level 0 of the
// single-reduction CG): also w = A x on the tile, written to w_out, and the partial sums
// (b, x), (b, b), (w, x), (bb_src, bb_src).  (With the operator in LDS: 9.9 us (CG1) and 5.4 us.)
template <bool CG1>
__global__ __launch_bounds__(mg_tile_threads(CG1 ? kMgHaloA : kMgHalo)) void k_mg_up(MgLevel L, MgLevel C, double* out,
                                                                                  const PcgState* st, double* part,
                                                                                  const double* bb_src, double* w_out)
{
    using Tile = MgTile<CG1 ? kMgHaloA : kMgHalo>;
    __shared__ double sx[4 * Tile::P * Tile::P];
    const int done = st ? st->done : 0;
    const Tile t(L);
    const MgPlanes s = t.planes(sx);
    const MgIn in = agg_in(L, t.gi, t.gj);
    const bool on = t.on;
    const int nx = L.nx, g = t.gj * nx + t.gi;
    const int off[4] = {0, 1, nx, nx + 1};
    MgAgg a;
    double bs[4] = {0.0, 0.0, 0.0, 0.0};
    if (on) {
        const double yc = kMgOver * ld_if(in.c[0], C.y, (t.gj >> 1) * C.nx + (t.gi >> 1), 0.0);
        a.x[0] = ld_if(in.c[0], L.x, g, 0.0);
        a.x[3] = ld_if(in.c[3], L.x, g + nx + 1, 0.0);
        agg_load(L, t.gi, t.gj, in, a);
#pragma unroll
        for (int c = 0; c < 4; ++c) a.b[c] = ld_if(in.c[c], L.b, g + off[c], 0.0);
        if (CG1 && bb_src) {
#pragma unroll
            for (int c = 0; c < 4; ++c) bs[c] = ld_if(t.interior && in.c[c], bb_src, g + off[c], 0.0);
        }
        if (in.c[0]) a.x[0] += yc;
        if (in.c[3]) a.x[3] += yc;
    }
    if (done) return;
    if (on) agg_invert(a);
    t.border(s);
    agg_up(a, s, on, CG1);
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    if constexpr (CG1) __syncthreads();
    if (t.interior) {
        double w[4] = {0.0, 0.0, 0.0, 0.0};
        if constexpr (CG1) {
            red_sums(a, s, w[0], w[3]);
            black_sums(a, s, w[1], w[2]);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (!in.c[c]) continue;
            out[g + off[c]] = a.x[c];
            if constexpr (CG1) {
                const double wq = a.d[c] * a.x[c] - w[c];
                w_out[g + off[c]] = wq;
                acc[0] += a.b[c] * a.x[c];
                acc[1] += a.b[c] * a.b[c];
                acc[2] += wq * a.x[c];
                acc[3] += bs[c] * bs[c];
            }
        }
    }
    if constexpr (CG1) block_partials<4, false>(acc, part);
}

// Dense inverse of level le's operator (at most 64 cells) by Gauss-Jordan elimination; the operator
// is symmetric positive definite and diagonally dominant, so no pivoting.  A lane holds column
// `lane` of the rows w, w + 16, w + 32, w + 48 of its wave w in registers: a row's own pivot-column
// entry is a lane read, and only the pivot row goes through LDS (two buffers, one barrier a
// step).  With the matrix in LDS and two barriers a step the 49 steps of a 7 x 7 level took 48 us.
// m[c] receives the inverse's entry (w + 16 c, lane); every thread of a block of kMgThreads calls it.
constexpr int kMgInvRows = kMgExactCells / (kMgThreads / kWave);   // rows of the inverse per wave
__device__ __forceinline__ void mg_gauss_jordan(const MgLevel& L, double (&m)[kMgInvRows])
{
    constexpr int NE = kMgExactCells, NW = kMgThreads / kWave, PER = kMgInvRows;
    static_assert(NE == kWave && NE % NW == 0, "a lane is a column, a wave whole rows");
    __shared__ double row[2][NE];
    const int nx = L.nx, n = L.nx * L.ny;
    const int j = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
#pragma unroll
    for (int c = 0; c < PER; ++c) {
        const int i = w + c * NW;
        double v = 0.0;
        if (i < n && j < n) {
            if (i == j) v = L.d[i];
            else if (j == i + 1 && i % nx != nx - 1) v = -L.we[i];
            else if (i == j + 1 && j % nx != nx - 1) v = -L.we[j];
            else if (j == i + nx) v = -L.wn[i];
            else if (i == j + nx) v = -L.wn[j];
        }
        m[c] = v;
    }
#pragma unroll
    for (int ck = 0; ck < PER; ++ck)
        for (int kk = 0; kk < NW; ++kk) {
            const int k = ck * NW + kk;
            if (k >= n) break;
            if (w == kk) row[k & 1][j] = m[ck];
            __syncthreads();
            const double pr = row[k & 1][j];
            const double ip = 1.0 / lane_value(pr, k);
            const double rk = (j == k ? 1.0 : pr) * ip;   // row k, scaled (its own column holds the inverse)
#pragma unroll
            for (int c = 0; c < PER; ++c) {
                const double f = lane_value(m[c], k);
                const double v = fma(-f, rk, j == k ? 0.0 : m[c]);
                m[c] = (c == ck && w == kk) ? rk : v;
            }
        }
}

// Entries (w + 16 c, lane) of an n x n matrix, from or to memory (row pitch n; zeros outside).
__device__ __forceinline__ void mg_store_inverse(const double (&m)[kMgInvRows], double* out, int n, int pitch)
{
    const int j = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
#pragma unroll
    for (int c = 0; c < kMgInvRows; ++c) {
        const int i = w + c * (kMgThreads / kWave);
        if (i < n && j < n) out[i * pitch + j] = m[c];
    }
}
__device__ __forceinline__ void mg_load_inverse(double (&m)[kMgInvRows], const double* inv, int n)
{
    const int j = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
#pragma unroll
    for (int c = 0; c < kMgInvRows; ++c) {
        const int i = w + c * (kMgThreads / kWave);
        m[c] = (i < n && j < n) ? inv[i * n + j] : 0.0;
    }
}

// ye = inverse * rhs (n entries in LDS), the inverse symmetric and held as above: each wave sums
// its rows' share of every entry, then one wave the shares.  A barrier before and inside; one must
// follow before ye is read.
struct MgExactLds {
    double pp[kMgThreads / kWave][kMgExactCells], ye[kMgExactCells];
};
__device__ __forceinline__ void mg_exact_solve(const double (&m)[kMgInvRows], const double* rhs, int n, MgExactLds& e)
{
    const int j = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    constexpr int NW = kMgThreads / kWave;
    double v = 0.0;
#pragma unroll
    for (int c = 0; c < kMgInvRows; ++c) {
        const int i = w + c * NW;
        v += m[c] * (i < n ? rhs[i] : 0.0);
    }
    e.pp[w][j] = v;
    __syncthreads();
    if (w == 0) {
        double y = 0.0;
#pragma unroll
        for (int c = 0; c < NW; ++c) y += e.pp[c][j];
        e.ye[j] = y;
    }
}

// The V-cycle from level lc down to le and back, in one block: reads b of level lc, writes y of
// level lc.  A thread owns one aggregate of one of the levels
// lc .. le - 1 (all operators are loaded at once at the start), so a phase is a barrier and at most
// one aggregate's update; the residual sum of thread t's aggregate is cell t of the array of the
// coarser levels' right-hand sides.  A chain of ~36 dependent phases of ~100 ns; with the operators in
// LDS and the levels' cells dealt anew to the threads in every phase it took 26 us (50 x 50 down to
// 7 x 7).
__global__ __launch_bounds__(kMgThreads) void k_mg_coarse(MgHier h, const PcgState* st)
{
    // a level of bx x by aggregates takes 4 (bx + 2) (by + 2) slots; a row of n aggregates is the worst
    __shared__ double sx[12 * kMgThreads + 24 * kMgMaxLevels];
    __shared__ double sb[kMgThreads];
    __shared__ MgExactLds ex;
    const int done = st ? st->done : 0;
    const int le = h.le, lc = mg_coarse_first(h);
    const int tid = threadIdx.x;
    int lv = -1, base = 0, xo = 0;        // this thread's level, its first thread and first slot
    int own_b = 0;                        // where this level's right-hand side starts in sb
    for (int l = lc, b0 = 0, x0 = 0, prev = 0; l < le; ++l) {
        const int n = h.lv[l + 1].nx * h.lv[l + 1].ny;
        if (tid >= b0 && tid < b0 + n) {
            lv = l;
            base = b0;
            xo = x0;
            own_b = prev;
        }
        prev = b0;
        b0 += n;
        x0 += 4 * (h.lv[l + 1].nx + 2) * (h.lv[l + 1].ny + 2);
    }
    const bool has = lv >= 0;
    const int ll = has ? lv : le;
    const MgLevel L = h.lv[ll];
    const int bx = has ? h.lv[ll + 1].nx : 1, by = has ? h.lv[ll + 1].ny : 1;
    const int J = has ? (tid - base) / bx : 0, I = has ? (tid - base) - J * bx : 0;
    const MgPlanes s{sx + xo + (J + 1) * (bx + 2) + I + 1, bx + 2, (bx + 2) * (by + 2)};
    const MgIn in = agg_in(L, 2 * I, 2 * J);
    const int nx = L.nx, g = 2 * J * nx + 2 * I;
    const int off[4] = {0, 1, nx, nx + 1};
    MgAgg a;
    if (has) {
        agg_load(L, 2 * I, 2 * J, in, a);
        if (lv == lc) {
#pragma unroll
            for (int c = 0; c < 4; ++c) a.b[c] = ld_if(in.c[c], L.b, g + off[c], 0.0);
        }
    }
    const int ne = h.lv[le].nx * h.lv[le].ny;
    double inv[kMgInvRows];
    mg_load_inverse(inv, h.inv, ne);
    if (lc == le && tid < ne) sb[tid] = L.b[tid];
    if (done) return;
    if (has) {
        agg_invert(a);
        planes_border(s, I == 0, I == bx - 1, J == 0, J == by - 1);
    }
    int eb = 0;   // the exact level's right-hand side in sb
    for (int l = lc; l < le; ++l) {
        const bool on = lv == l;
        if (on && l > lc) {
#pragma unroll
            for (int c = 0; c < 4; ++c) a.b[c] = in.c[c] ? sb[own_b + g + off[c]] : 0.0;
        }
        const double rc = agg_down(a, s, on);
        if (on) sb[tid] = rc;
        if (l > lc) eb += h.lv[l].nx * h.lv[l].ny;
        __syncthreads();
    }
    if (lc == le) __syncthreads();
    mg_exact_solve(inv, sb + eb, ne, ex);
    __syncthreads();
    for (int l = le - 1; l >= lc; --l) {
        const bool on = lv == l;
        if (on) {
            double yc;
            if (l + 1 == le) {
                yc = ex.ye[tid - base];
            } else {   // cell (I, J) of the next level, in that level's planes
                const int cbx = h.lv[l + 2].nx, cby = h.lv[l + 2].ny;
                const double* cx = sx + xo + 4 * s.plane;
                yc = cx[((J & 1) * 2 + (I & 1)) * (cbx + 2) * (cby + 2) + ((J >> 1) + 1) * (cbx + 2) + (I >> 1) + 1];
            }
            if (in.c[0]) a.x[0] += kMgOver * yc;
            if (in.c[3]) a.x[3] += kMgOver * yc;
        }
        agg_up(a, s, on, true);
        __syncthreads();
    }
    if (lc == le) {
        if (tid < ne) L.y[tid] = ex.ye[tid];
    } else if (lv == lc) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (in.c[c]) L.y[g + off[c]] = a.x[c];
    }
}

// The operators of the levels below the first one the single-block kernel handles (and level 0's
// weights when that is level 0), and the exact level's inverse, by one block: a launch per level
// took longer than their few cells.
__global__ __launch_bounds__(kMgThreads) void k_mg_setup_coarse(Geo2 g, const double* ke, const double* kn, MgHier h)
{
    const int lc = mg_coarse_first(h);
    if (lc == 0) {
        mg_fine_cells(g, ke, kn, h.lv[0].we, h.lv[0].wn, threadIdx.x, blockDim.x);
        __syncthreads();
    }
    for (int l = lc; l < h.le; ++l) {
        mg_coarsen_cells(h.lv[l], h.lv[l + 1], threadIdx.x, blockDim.x);
        __syncthreads();
    }
    const int n = h.lv[h.le].nx * h.lv[h.le].ny;
    double m[kMgInvRows];
    mg_gauss_jordan(h.lv[h.le], m);
    mg_store_inverse(m, h.inv, n, n);
}

// ---- the whole multigrid-preconditioned CG of a small surface in one workgroup, on chip ------
// Surfaces whose level 0 has at most one aggregate per thread (64 x 64 cells).  A thread keeps its
// level-0 aggregate -- operator, residual, search direction, solution -- in registers for the whole
// solve; the coarser levels' operators and right-hand sides and every level's planes are in LDS, so
// after the first loads an iteration moves nothing but register spills.  The iteration is the
// Hestenes-Stiefel one of the other one-workgroup forms, with (p, A p) summed directly: on flat deep
// pools (face conductances from 1e-2 to 1e12 side by side) the single-reduction form's recurrence for
// it loses every digit and comes out negative, and in one workgroup a second block reduction costs
// one barrier, which that form spends on A z.  A chain of ~40 barriers an iteration bound by LDS
// latency: 226 us a solve of 11 iterations on 64 x 48 cells (single-reduction form: 277), 261 on
// 64 x 64 (327); the grid-wide kernels take three launches an iteration and three for the set-up.
constexpr int kMgDeepAggs = 384;       // aggregates of levels 1 .. le - 1 together
constexpr int kMgSmallPlanes = 10240;  // plane slots of all levels together (a strip of 3 x 712 cells: 9,544)
constexpr int kMgOps = 16;             // operator values of a coarser aggregate
struct MgSmallLevel {
    int bx, by, x, op, b;   // aggregates; first plane slot, operator column, right-hand side entry
};

__device__ __forceinline__ double olf_we(const Geo2& g, const double* __restrict__ ke, int i, int j)
{
    return (i > 0 && j > 0 && i < g.nx - 2 && j < g.ny - 1) ? g.cx * ke[j * g.nx + i] : 0.0;
}
__device__ __forceinline__ double olf_wn(const Geo2& g, const double* __restrict__ kn, int i, int j)
{
    return (i > 0 && j > 0 && i < g.nx - 1 && j < g.ny - 2) ? g.cy * kn[j * g.nx + i] : 0.0;
}

__device__ __forceinline__ void b_olf_mgcg_small(const OlfCgArgs& a, const MgHier& h)
{
    __shared__ double sx[kMgSmallPlanes], sop[kMgOps * kMgDeepAggs], sb[kMgThreads + kMgDeepAggs];
    __shared__ MgExactLds ex;
    __shared__ MgSmallLevel lev[kMgMaxLevels];
    __shared__ double red[3 * 16], red_pq[16];   // one reduction's barrier frees the other's words
    const Geo2 g2 = a.g;
    const int le = h.le, tid = threadIdx.x;
    if (tid == 0) {
        int x = 0, op = 0, b = 0;
        for (int l = 0; l <= le; ++l) {
            const int bx = (h.lv[l].nx + 1) / 2, by = (h.lv[l].ny + 1) / 2;
            lev[l] = MgSmallLevel{bx, by, x, op, b};
            x += 4 * (bx + 2) * (by + 2);
            if (l > 0) op += bx * by;
            if (l > 0) b += h.lv[l].nx * h.lv[l].ny;
        }
    }
    // level 0: the aggregate of this thread
    const int nx = g2.nx, ny = g2.ny, bx0 = (nx + 1) / 2, by0 = (ny + 1) / 2;
    const bool on0 = tid < bx0 * by0;
    const int J0 = on0 ? tid / bx0 : 0, I0 = on0 ? tid - J0 * bx0 : 0;
    const int gi = 2 * I0, gj = 2 * J0, g = gj * nx + gi;
    const int off[4] = {0, 1, nx, nx + 1};
    const MgLevel dims{nx, ny, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    MgIn in = agg_in(dims, gi, gj);
#pragma unroll
    for (int c = 0; c < 4; ++c) in.c[c] = in.c[c] && on0;
    const MgPlanes s0{sx + (J0 + 1) * (bx0 + 2) + I0 + 1, bx0 + 2, (bx0 + 2) * (by0 + 2)};
    MgAgg A;
    double p[4] = {}, x[4], bb = 0.0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        A.d[c] = ld_if(in.c[c], a.D, g + off[c], 1.0);
        A.b[c] = ld_if(in.c[c], a.r, g + off[c], 0.0);
        A.x[c] = 0.0;
        x[c] = ld_if(in.c[c], a.x, g + off[c], 0.0);
        const double bc = ld_if(in.c[c], a.b, g + off[c], 0.0);
        bb += bc * bc;
    }
    A.h0 = olf_we(g2, a.ke, gi, gj);
    A.h1 = olf_we(g2, a.ke, gi, gj + 1);
    A.w0 = olf_we(g2, a.ke, gi - 1, gj);
    A.w2 = olf_we(g2, a.ke, gi - 1, gj + 1);
    A.e1 = olf_we(g2, a.ke, gi + 1, gj);
    A.e3 = olf_we(g2, a.ke, gi + 1, gj + 1);
    A.v0 = olf_wn(g2, a.kn, gi, gj);
    A.v1 = olf_wn(g2, a.kn, gi + 1, gj);
    A.s0 = olf_wn(g2, a.kn, gi, gj - 1);
    A.s1 = olf_wn(g2, a.kn, gi + 1, gj - 1);
    A.n2 = olf_wn(g2, a.kn, gi, gj + 1);
    A.n3 = olf_wn(g2, a.kn, gi + 1, gj + 1);
    agg_invert(A);
    // the coarser operators: each aggregate's cell of the next level (d, east, north couplings)
    // goes to LDS, the next level's aggregates collect theirs from there
    double inv[kMgInvRows];
    {
        constexpr int CS = kMgThreads;
        double *cd = sx, *ce = sx + CS, *cn = sx + 2 * CS;   // the planes are not in use yet
        if (le == 0) {
            if (on0) {
                const double we[4] = {A.h0, A.e1, A.h1, A.e3}, wn[4] = {A.v0, A.v1, A.n2, A.n3};
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (in.c[c]) {
                        cd[g + off[c]] = A.d[c];
                        ce[g + off[c]] = we[c];
                        cn[g + off[c]] = wn[c];
                    }
            }
        } else if (on0) {
            cd[tid] = (in.c[0] ? A.d[0] : 0.0) + (in.c[1] ? A.d[1] : 0.0) + (in.c[2] ? A.d[2] : 0.0) +
                      (in.c[3] ? A.d[3] : 0.0) - 2.0 * (A.h0 + A.h1 + A.v0 + A.v1);
            ce[tid] = A.e1 + A.e3;
            cn[tid] = A.n2 + A.n3;
        }
        __syncthreads();
        for (int l = 1; l < le; ++l) {
            const MgSmallLevel v = lev[l];
            const MgLevel C{h.lv[l].nx, h.lv[l].ny, cd, ce, cn, nullptr, nullptr, nullptr};
            double cdn = 0.0, cen = 0.0, cnn = 0.0;
            const bool on = tid < v.bx * v.by;
            if (on) {
                MgAgg t;
                const int J = tid / v.bx, I = tid - J * v.bx;
                const MgIn ti = agg_in(C, 2 * I, 2 * J);
                agg_load(C, 2 * I, 2 * J, ti, t);
                agg_invert(t);
                const double o[kMgOps] = {t.di[0], t.di[1], t.di[2], t.di[3], t.h0, t.h1, t.v0, t.v1,
                                          t.w0, t.w2, t.e1, t.e3, t.s0, t.s1, t.n2, t.n3};
#pragma unroll
                for (int q = 0; q < kMgOps; ++q) sop[q * kMgDeepAggs + v.op + tid] = o[q];
                cdn = (ti.c[0] ? t.d[0] : 0.0) + (ti.c[1] ? t.d[1] : 0.0) + (ti.c[2] ? t.d[2] : 0.0) +
                      (ti.c[3] ? t.d[3] : 0.0) - 2.0 * (t.h0 + t.h1 + t.v0 + t.v1);
                cen = t.e1 + t.e3;
                cnn = t.n2 + t.n3;
            }
            __syncthreads();
            if (on) {
                cd[tid] = cdn;
                ce[tid] = cen;
                cn[tid] = cnn;
            }
            __syncthreads();
        }
        const MgLevel E{h.lv[le].nx, h.lv[le].ny, cd, ce, cn, nullptr, nullptr, nullptr};
        mg_gauss_jordan(E, inv);
        __syncthreads();   // the planes are used from here on
    }
    const int ne = h.lv[le].nx * h.lv[le].ny;
    if (on0) planes_border(s0, I0 == 0, I0 == bx0 - 1, J0 == 0, J0 == by0 - 1);
    for (int l = 1; l < le; ++l) {
        const MgSmallLevel v = lev[l];
        if (tid < v.bx * v.by) {
            const int J = tid / v.bx, I = tid - J * v.bx;
            planes_border(MgPlanes{sx + v.x + (J + 1) * (v.bx + 2) + I + 1, v.bx + 2, (v.bx + 2) * (v.by + 2)}, I == 0,
                          I == v.bx - 1, J == 0, J == v.by - 1);
        }
    }
    // a coarser level's aggregate of this thread, from LDS (only what the caller uses is read)
    struct Deep {
        bool on;
        int I, J;
        MgIn in;
        MgPlanes s;
        const double *o, *b;
        int nx;
        __device__ __forceinline__ MgAgg get() const
        {
            MgAgg t;
            auto q = [&](int i) { return o[i * kMgDeepAggs]; };
            t.di[0] = q(0); t.di[1] = q(1); t.di[2] = q(2); t.di[3] = q(3);
            t.h0 = q(4); t.h1 = q(5); t.v0 = q(6); t.v1 = q(7);
            t.w0 = q(8); t.w2 = q(9); t.e1 = q(10); t.e3 = q(11);
            t.s0 = q(12); t.s1 = q(13); t.n2 = q(14); t.n3 = q(15);
            t.b[0] = in.c[0] ? b[0] : 0.0;
            t.b[1] = in.c[1] ? b[1] : 0.0;
            t.b[2] = in.c[2] ? b[nx] : 0.0;
            t.b[3] = in.c[3] ? b[nx + 1] : 0.0;
#pragma unroll
            for (int c = 0; c < 4; ++c) t.x[c] = s.at(c, 0);
            return t;
        }
    };
    auto deep = [&](int l) {
        const MgSmallLevel v = lev[l];
        Deep t;
        t.on = tid < v.bx * v.by;
        t.J = t.on ? tid / v.bx : 0;
        t.I = t.on ? tid - t.J * v.bx : 0;
        const MgLevel d{h.lv[l].nx, h.lv[l].ny, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
        t.in = agg_in(d, 2 * t.I, 2 * t.J);
        t.s = MgPlanes{sx + v.x + (t.J + 1) * (v.bx + 2) + t.I + 1, v.bx + 2, (v.bx + 2) * (v.by + 2)};
        t.o = sop + v.op + (t.on ? tid : 0);
        t.nx = d.nx;
        t.b = sb + v.b + 2 * t.J * d.nx + 2 * t.I;
        return t;
    };
    auto sweep = [&](const Deep& t, bool red_cells) {   // one half-sweep and its barrier
        if (t.on) {
            MgAgg v = t.get();
            if (red_cells) red_sweep(v, t.s);
            else black_sweep(v, t.s);
        }
        __syncthreads();
    };
    auto vcycle = [&]() {   // A.x = V-cycle(A.b)
        if (le == 0) {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (in.c[c]) sb[g + off[c]] = A.b[c];
            __syncthreads();
            mg_exact_solve(inv, sb, ne, ex);
            __syncthreads();
#pragma unroll
            for (int c = 0; c < 4; ++c) A.x[c] = in.c[c] ? ex.ye[g + off[c]] : 0.0;
            return;
        }
        {
            const double rc = agg_down(A, s0, on0);
            if (on0) sb[tid] = rc;
            __syncthreads();
        }
        for (int l = 1; l < le; ++l) {
            const Deep t = deep(l);
            if (t.on) {
                MgAgg v = t.get();
                v.x[0] = v.b[0] * v.di[0];
                v.x[3] = v.b[3] * v.di[3];
                put_red(v, t.s);
            }
            __syncthreads();
            sweep(t, false);
            double u0 = 0.0, u3 = 0.0;
            if (t.on) {
                MgAgg v = t.get();
                red_sums(v, t.s, u0, u3);
                v.x[0] = (v.b[0] + u0) * v.di[0];
                v.x[3] = (v.b[3] + u3) * v.di[3];
                put_red(v, t.s);
            }
            __syncthreads();
            sweep(t, false);
            if (t.on) {
                MgAgg v = t.get();
                double t0, t3;
                red_sums(v, t.s, t0, t3);
                sb[lev[l + 1].b + tid] = (t0 - u0) + (t3 - u3);
            }
            __syncthreads();
        }
        mg_exact_solve(inv, sb + lev[le].b, ne, ex);
        __syncthreads();
        // the correction of aggregate (I, J) of level l: that cell of level l + 1
        auto correction = [&](int l, int I, int J, int t) {
            if (l + 1 == le) return ex.ye[t];
            const MgSmallLevel v = lev[l + 1];
            return sx[v.x + ((J & 1) * 2 + (I & 1)) * (v.bx + 2) * (v.by + 2) + ((J >> 1) + 1) * (v.bx + 2) + (I >> 1) + 1];
        };
        for (int l = le - 1; l >= 1; --l) {
            const Deep t = deep(l);
            if (t.on) {
                const double yc = kMgOver * correction(l, t.I, t.J, tid);
                if (t.in.c[0]) t.s.put(0, t.s.at(0, 0) + yc);
                if (t.in.c[3]) t.s.put(3, t.s.at(3, 0) + yc);
            }
            __syncthreads();
            sweep(t, false);
            sweep(t, true);
            sweep(t, false);
            sweep(t, true);
        }
        if (on0) {
            const double yc = kMgOver * correction(0, I0, J0, tid);
            if (in.c[0]) A.x[0] += yc;
            if (in.c[3]) A.x[3] += yc;
        }
        agg_up(A, s0, on0, false);
    };
    // z = A.x = V-cycle(r); (r, z), (r, r) and, at the start, (b, b)
    double sums[3];
    auto cycle = [&](double bb_c) {
        vcycle();
        sums[0] = sums[1] = 0.0;
        sums[2] = bb_c;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (!in.c[c]) continue;
            sums[0] += A.b[c] * A.x[c];
            sums[1] += A.b[c] * A.b[c];
        }
        block_reduce<3, false, false>(sums, red);
    };
    cycle(bb);
    bb = sums[2];
    const double tol2 = a.tol * a.tol * bb;
    double rz = sums[0], rr = sums[1], beta = 0.0;
    int it = 0, conv = 0, nan = !isfinite(bb);
    for (;;) {
        nan |= !(isfinite(rr) && isfinite(rz));
        conv = (rr <= tol2) ? 1 : 0;
        if (conv || nan || it >= a.maxit) break;
        // p, and A p through the planes (no wave still reads them: the reduction's barrier)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            p[c] = A.x[c] + beta * p[c];
            A.x[c] = p[c];
        }
        if (on0) {
            put_red(A, s0);
            s0.put(1, p[1]);
            s0.put(2, p[2]);
        }
        __syncthreads();
        double t[4] = {0.0, 0.0, 0.0, 0.0}, q[4], pq[1] = {0.0};
        if (on0) {
            red_sums(A, s0, t[0], t[3]);
            black_sums(A, s0, t[1], t[2]);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            q[c] = in.c[c] ? A.d[c] * p[c] - t[c] : 0.0;
            pq[0] += p[c] * q[c];
        }
        block_reduce<1, false, false>(pq, red_pq);
        const double alpha = rz / pq[0];
        if (!(pq[0] != 0.0) || !isfinite(alpha)) {
            nan = 1;
            break;
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            x[c] += alpha * p[c];
            A.b[c] -= alpha * q[c];
        }
        cycle(0.0);
        ++it;
        beta = sums[0] / rz;
        rz = sums[0];
        rr = sums[1];
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (in.c[c]) a.x[g + off[c]] = x[c];
    if (tid == 0) {
        PcgState* st = a.st;
        st->bb = bb;
        st->tol2 = tol2;
        st->iter = it;
        st->conv = conv && !nan;
        st->rr = rr;
        st->nan = nan;
        st->outer_conv = conv && !nan;
        st->done = 1;
    }
}

__global__ __launch_bounds__(kMgThreads) void k_olf_mgcg_small(OlfMgArgs a)
{
    b_olf_mgcg_small(a.cg, a.h);
}

// ---- the multigrid-preconditioned CG of a small surface in one workgroup -----------------
// The V-cycle of the grid kernels (same smoother, restriction, coarse correction and exact
// level), each phase a pass of the block over a level held in global memory, a barrier between
// phases; the exact level's inverse stays in LDS.
__device__ __forceinline__ void mgb_half(const MgLevel& L, const double* __restrict__ b, double* __restrict__ x,
                                         int color)
{
    const int nx = L.nx, ny = L.ny, hw = (nx + 1) / 2;
    for (int u = threadIdx.x; u < ny * hw; u += blockDim.x) {
        const int j = u / hw;
        const int i = ((color - j) & 1) + 2 * (u - j * hw);
        if (i >= nx) continue;
        const int f = j * nx + i;
        double s = b[f];
        if (i + 1 < nx) s += L.we[f] * x[f + 1];
        if (i > 0) s += L.we[f - 1] * x[f - 1];
        if (j + 1 < ny) s += L.wn[f] * x[f + nx];
        if (j > 0) s += L.wn[f - nx] * x[f - nx];
        x[f] = s * (1.0 / L.d[f]);
    }
    __syncthreads();
}

// b_coarse = P^T (b - A x): each coarse cell sums the residuals of its (up to) 2 x 2 children.
__device__ __forceinline__ void mgb_restrict(const MgLevel& L, const double* __restrict__ b,
                                             const double* __restrict__ x, const MgLevel& C)
{
    const int nx = L.nx, ny = L.ny;
    for (int t = threadIdx.x; t < C.nx * C.ny; t += blockDim.x) {
        const int J = t / C.nx, I = t - J * C.nx;
        double s = 0.0;
        for (int dj = 0; dj < 2; ++dj)
            for (int di = 0; di < 2; ++di) {
                const int i = 2 * I + di, j = 2 * J + dj;
                if (i >= nx || j >= ny) continue;
                const int f = j * nx + i;
                double ax = L.d[f] * x[f];
                if (i + 1 < nx) ax -= L.we[f] * x[f + 1];
                if (i > 0) ax -= L.we[f - 1] * x[f - 1];
                if (j + 1 < ny) ax -= L.wn[f] * x[f + nx];
                if (j > 0) ax -= L.wn[f - nx] * x[f - nx];
                s += b[f] - ax;
            }
        C.b[t] = s;
    }
    __syncthreads();
}

// z = V-cycle(r) (levels 0 .. le; Minv: level le's inverse, row pitch kMgExactCells).
__device__ __forceinline__ void mgb_vcycle(const MgHier& h, const double* Minv, const double* r, double* z)
{
    const int le = h.le;
    for (int l = 0; l < le; ++l) {
        const MgLevel& L = h.lv[l];
        const double* b = l ? L.b : r;
        for (int f = threadIdx.x; f < L.nx * L.ny; f += blockDim.x) L.x[f] = 0.0;
        __syncthreads();
        mgb_half(L, b, L.x, 0);
        mgb_half(L, b, L.x, 1);
        mgb_half(L, b, L.x, 0);
        mgb_half(L, b, L.x, 1);
        mgb_restrict(L, b, L.x, h.lv[l + 1]);
    }
    {   // the exact level (level 0 itself on a surface of at most kMgExactCells cells)
        const MgLevel& E = h.lv[le];
        const int n = E.nx * E.ny;
        const double* eb = le ? E.b : r;
        double* ex = le ? E.x : z;
        for (int t = threadIdx.x; t < n; t += blockDim.x) {
            double v = 0.0;
            for (int j = 0; j < n; ++j) v += Minv[t * kMgExactCells + j] * eb[j];
            ex[t] = v;
        }
        __syncthreads();
    }
    for (int l = le - 1; l >= 0; --l) {
        const MgLevel& L = h.lv[l];
        const MgLevel& C = h.lv[l + 1];
        const double* b = l ? L.b : r;
        double* x = l ? L.x : z;
        for (int f = threadIdx.x; f < L.nx * L.ny; f += blockDim.x) {
            const int j = f / L.nx, i = f - j * L.nx;
            x[f] = L.x[f] + kMgOver * C.x[(j >> 1) * C.nx + (i >> 1)];
        }
        __syncthreads();
        mgb_half(L, b, x, 1);
        mgb_half(L, b, x, 0);
        mgb_half(L, b, x, 1);
        mgb_half(L, b, x, 0);
    }
}

__device__ __forceinline__ void b_olf_mgcg_block(const OlfCgArgs& a, const MgHier& h)
{
    __shared__ double Minv[kMgExactCells * kMgExactCells];
    __shared__ double lds[3 * 16];
    const Geo2 g = a.g;
    const int n = g.n, tid = threadIdx.x, nt = blockDim.x;
    // the operators of this step's system: level-0 weights, Galerkin coarse levels, exact inverse
    mg_fine_cells(g, a.ke, a.kn, h.lv[0].we, h.lv[0].wn, tid, nt);
    __syncthreads();
    for (int l = 0; l < h.le; ++l) {
        mg_coarsen_cells(h.lv[l], h.lv[l + 1], tid, nt);
        __syncthreads();
    }
    {
        double m[kMgInvRows];
        mg_gauss_jordan(h.lv[h.le], m);
        mg_store_inverse(m, Minv, h.lv[h.le].nx * h.lv[h.le].ny, kMgExactCells);
    }
    __syncthreads();
    const double* __restrict__ b = a.b;
    double* __restrict__ x = a.x;
    double* __restrict__ r = a.r;
    double* __restrict__ p = a.p;
    double* __restrict__ q = a.q;
    double* __restrict__ z = h.lv[0].y;
    mgb_vcycle(h, Minv, r, z);
    double v[3] = {0.0, 0.0, 0.0};   // (r, z), (r, r), (b, b)
    for (int c = tid; c < n; c += nt) {
        const double rc = r[c];
        p[c] = z[c];
        v[0] += rc * z[c];
        v[1] += rc * rc;
        v[2] += b[c] * b[c];
    }
    block_sum3(v, lds);
    double rz = v[0], rr = v[1], beta = 0.0;
    const double bb = v[2], tol2 = a.tol * a.tol * bb;
    int it = 0, conv = 0, nan = !isfinite(bb);
    for (;;) {
        nan |= !(isfinite(rr) && isfinite(rz));
        conv = (rr <= tol2) ? 1 : 0;
        if (conv || nan || it >= a.maxit) break;
        if (it > 0)
            for (int c = tid; c < n; c += nt) p[c] = z[c] + beta * p[c];
        __syncthreads();   // p of the neighbours
        double w[3] = {0.0, 0.0, 0.0};
        for (int c = tid; c < n; c += nt) {
            const double pc = p[c];
            const double qc = op2_row(g, c, a.D[c], pc, [&](int k) { return p[k]; }, a.ke, a.kn);
            q[c] = qc;
            w[0] += pc * qc;
        }
        block_sum3(w, lds);
        const double alpha = rz / w[0];
        if (!(w[0] != 0.0) || !isfinite(alpha)) {
            nan = 1;
            break;
        }
        double u[3] = {0.0, 0.0, 0.0};
        for (int c = tid; c < n; c += nt) {
            x[c] = x[c] + alpha * p[c];
            const double rc = r[c] - alpha * q[c];
            r[c] = rc;
            u[1] += rc * rc;
        }
        mgb_vcycle(h, Minv, r, z);   // its first barrier orders the r writes before its reads
        for (int c = tid; c < n; c += nt) u[0] += r[c] * z[c];
        block_sum3(u, lds);
        ++it;
        beta = u[0] / rz;
        rz = u[0];
        rr = u[1];
    }
    if (tid == 0) {
        PcgState* st = a.st;
        st->bb = bb;
        st->tol2 = tol2;
        st->iter = it;
        st->conv = conv && !nan;
        st->rr = rr;
        st->nan = nan;
        st->outer_conv = conv && !nan;
        st->done = 1;
    }
}

__global__ __launch_bounds__(kMgThreads) void k_olf_mgcg_block(OlfMgArgs a)
{
    b_olf_mgcg_block(a.cg, a.h);
}

// One workgroup per model; the model's hierarchy descriptor is copied to LDS first.
__global__ __launch_bounds__(kMgThreads) void kb_olf_mgcg_block(const OlfMgArgs* __restrict__ args,
                                                               const int* __restrict__ active)
{
    if (active && !active[blockIdx.x]) return;
    __shared__ MgHier hs;
    __shared__ OlfCgArgs cs;
    if (threadIdx.x == 0) {
        hs = args[blockIdx.x].h;
        cs = args[blockIdx.x].cg;
    }
    __syncthreads();
    b_olf_mgcg_block(cs, hs);
}

inline int mg_tiles(const MgLevel& L) { return ((L.nx + kMgT - 1) / kMgT) * ((L.ny + kMgT - 1) / kMgT); }

}  // namespace

int mg_levels(int nx, int ny, int dims[][2])
{
    int n = 0;
    for (;;) {
        dims[n][0] = nx;
        dims[n][1] = ny;
        ++n;
        if (nx == 1 && ny == 1) break;
        nx = (nx + 1) / 2;
        ny = (ny + 1) / 2;
    }
    return n;
}

int mg_exact_level(const MgHier& h)
{
    int l = 0;
    while (l < h.nlev - 1 && h.lv[l].nx * h.lv[l].ny > kMgExactCells) ++l;
    return l;
}

int mg_coarse_level(const MgHier& h) { return mg_first_single_block(h); }

int mg_partials(const MgHier& h) { return mg_tiles(h.lv[0]); }

void launch_mg_setup(hipStream_t s, const Geo2& g, const double* ke, const double* kn, const MgHier& h)
{
    // levels 0 and 1 together, the other levels above the single-block kernel's first one a launch each
    const int lc = mg_coarse_level(h);
    if (lc > 0)
        hipLaunchKernelGGL(k_mg_fine_coarsen, dim3(grid_for(h.lv[1].nx * h.lv[1].ny)), dim3(kBlock), 0, s, g, ke, kn,
                           h.lv[0], h.lv[1]);
    for (int l = 1; l < lc; ++l) {
        const int nc = h.lv[l + 1].nx * h.lv[l + 1].ny;
        hipLaunchKernelGGL(k_mg_coarsen, dim3(grid_for(nc)), dim3(kBlock), 0, s, h.lv[l], h.lv[l + 1]);
    }
    hipLaunchKernelGGL(k_mg_setup_coarse, dim3(1), dim3(kMgThreads), 0, s, g, ke, kn, h);
}

static void mg_down0(hipStream_t s, const MgHier& h, int l, const PcgState* st)
{
    hipLaunchKernelGGL(k_mg_down<false>, dim3(mg_tiles(h.lv[l])), dim3(mg_tile_threads(kMgHalo)), 0, s, h.lv[l],
                       h.lv[l + 1], st, MgCg1{});
}

static void mg_up0(hipStream_t s, const MgHier& h, int l, const PcgState* st)
{
    hipLaunchKernelGGL(k_mg_up<false>, dim3(mg_tiles(h.lv[l])), dim3(mg_tile_threads(kMgHalo)), 0, s, h.lv[l],
                       h.lv[l + 1], h.lv[l].y, st, nullptr, nullptr, nullptr);
}

void launch_mg_vcycle(hipStream_t s, const MgHier& h)
{
    const int lc = mg_coarse_level(h);
    for (int l = 0; l < lc; ++l) mg_down0(s, h, l, nullptr);
    hipLaunchKernelGGL(k_mg_coarse, dim3(1), dim3(kMgThreads), 0, s, h, (const PcgState*)nullptr);
    for (int l = lc - 1; l >= 0; --l) mg_up0(s, h, l, nullptr);
}

// The V-cycle below level 0 (down kernels of levels 1 .. lc-1, the single-block kernel, up
// kernels of levels lc-1 .. 1) and level 0's up kernel in its single-reduction form.
static void mg_vcycle_cg1_rest(hipStream_t s, const MgHier& h, const PcgState* st, double* part,
                               const double* bb_src, double* w)
{
    const int lc = mg_coarse_level(h);
    for (int l = 1; l < lc; ++l) mg_down0(s, h, l, st);
    hipLaunchKernelGGL(k_mg_coarse, dim3(1), dim3(kMgThreads), 0, s, h, st);
    for (int l = lc - 1; l >= 1; --l) mg_up0(s, h, l, st);
    hipLaunchKernelGGL(k_mg_up<true>, dim3(mg_tiles(h.lv[0])), dim3(mg_tile_threads(kMgHaloA)), 0, s, h.lv[0], h.lv[1],
                       h.lv[0].y, st, part, bb_src, w);
}

void launch_mg_vcycle_cg1_start(hipStream_t s, const MgHier& h, const PcgState* st, double* part,
                                const double* bb_src, double* w)
{
    mg_down0(s, h, 0, st);
    mg_vcycle_cg1_rest(s, h, st, part, bb_src, w);
}

bool mg_small(const MgHier& h)
{
    int deep = 0, planes = 0;
    for (int l = 0; l < std::max(h.le, 1); ++l) {
        const int bx = (h.lv[l].nx + 1) / 2, by = (h.lv[l].ny + 1) / 2;
        if (l == 0 && bx * by > kMgThreads) return false;
        if (l > 0) deep += bx * by;
        planes += 4 * (bx + 2) * (by + 2);
    }
    return deep <= kMgDeepAggs && planes <= kMgSmallPlanes;
}

void launch_olf_mgcg_small(hipStream_t s, const OlfMgArgs& a)
{
    hipLaunchKernelGGL(k_olf_mgcg_small, dim3(1), dim3(kMgThreads), 0, s, a);
}

void launch_olf_mgcg_block(hipStream_t s, const OlfMgArgs& a)
{
    hipLaunchKernelGGL(k_olf_mgcg_block, dim3(1), dim3(kMgThreads), 0, s, a);
}

void launch_batched_olf_mgcg_block(hipStream_t s, const OlfMgArgs* args, int nmodels, const int* active)
{
    if (nmodels > 0)
        hipLaunchKernelGGL(kb_olf_mgcg_block, dim3(nmodels), dim3(kMgThreads), 0, s, args, active);
}

void launch_mg_vcycle_cg1(hipStream_t s, const MgHier& h, const PcgState* st, double* part, const MgCg1& v)
{
    MgHier hh = h;
    hh.lv[0].b = v.r_new;   // level 0 of this V-cycle: the updated residual
    hipLaunchKernelGGL(k_mg_down<true>, dim3(mg_tiles(hh.lv[0])), dim3(mg_tile_threads(kMgHalo)), 0, s, hh.lv[0],
                       hh.lv[1], st, v);
    mg_vcycle_cg1_rest(s, hh, st, part, nullptr, v.w);
}

}  // namespace dh

// kernels.hip -- gfx950 kernels of the subsurface (3D Richards) and overland (2D diffusive
// wave) solvers.  Every kernel is grid-stride over cells in the reference layout
// (k*nx*ny + j*nx + i, k = 0 top) and keeps per-cell state in HBM as SoA arrays.
//
// Reductions: every kernel writes one partial per block; the next kernel sums them in a fixed order
// (device_common.h).  The Krylov kernels read PcgState::done at entry and
// return at once when the solve has finished, so the host can queue iterations in batches
// without a round trip per iteration.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <type_traits>

#include "kernels.h"

namespace dh {

// 1024 blocks of 256 threads = 4 blocks (16 wavefronts) per CU on 256 CUs; larger grids
// only add partials for the consumer to sum.
int grid_for(int n)
{
    constexpr int cap = 1024;
    static_assert(cap <= kMaxBlocks, "partial buffers too small");
    int g = (n + kBlock - 1) / kBlock;
    if (g < 1) g = 1;
    return g < cap ? g : cap;
}

namespace {

__device__ __forceinline__ void decompose(const Geo& g, int c, int& i, int& j, int& k)
{
    k = c / g.nxy;
    const int rem = c - k * g.nxy;
    j = rem / g.nx;
    i = rem - j * g.nx;
}

__device__ __forceinline__ double cell_alpha(const Soil& s, int c) { return s.alpha_f ? s.alpha_f[c] : s.alpha; }
__device__ __forceinline__ double cell_n(const Soil& s, int c) { return s.n_f ? s.n_f[c] : s.n; }

// y_c = (A p)_c of the subsurface operator: diagonal D plus the 7-point couplings
// -K_f/h^2 with arithmetic-mean faces K_f = (K_c + K_nb)/2 (src/subsurface.cu:26-102);
// domain faces carry no coupling; Dirichlet rows/cuts come from the row flags.
template <typename T, bool DIR, class PF>
__device__ __forceinline__ T op3_row(const Geo& g, int c, int i, int j, int k, T Dc, T pc, PF pf,
                                     const T* __restrict__ K, unsigned fl)
{
    if (DIR && (fl & RF_IDENTITY)) return pc;
    const T Kc = K[c];
    const T h = T(0.5);
    const T wx = (T)g.wx, wy = (T)g.wy, wz = (T)g.wz;
    T acc = Dc * pc;
    if (k > 0 && !(DIR && (fl & RF_CUT_D))) acc -= wz * (h * (Kc + K[c - g.nxy])) * pf(c - g.nxy);
    if (j > 0 && !(DIR && (fl & RF_CUT_S))) acc -= wy * (h * (Kc + K[c - g.nx])) * pf(c - g.nx);
    if (i > 0 && !(DIR && (fl & RF_CUT_W))) acc -= wx * (h * (Kc + K[c - 1])) * pf(c - 1);
    if (i < g.nx - 1 && !(DIR && (fl & RF_CUT_E))) acc -= wx * (h * (Kc + K[c + 1])) * pf(c + 1);
    if (j < g.ny - 1 && !(DIR && (fl & RF_CUT_N))) acc -= wy * (h * (Kc + K[c + g.nx])) * pf(c + g.nx);
    if (k < g.nz - 1 && !(DIR && (fl & RF_CUT_U))) acc -= wz * (h * (Kc + K[c + g.nxy])) * pf(c + g.nxy);
    return acc;
}


// ---------------------------------------------------------------------------------------
// Constitutive kernels
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ void b_vg(VgArgs a, Blk bk)
{
    for (int c = bk.id * blockDim.x + threadIdx.x; c < a.g.n; c += bk.n * blockDim.x) {
        double th, K, C;
        vg_eval(a.psi[c], a.soil.Ks[c], cell_alpha(a.soil, c), cell_n(a.soil, c), a.soil.ts,
                a.soil.tr, th, K, C);
        a.theta[c] = th;
        a.K[c] = K;
        a.C[c] = C;
        if (a.K32) a.K32[c] = (float)K;
    }
}

__global__ __launch_bounds__(kBlock) void k_vg(VgArgs a)
{
    b_vg(a, hw_blk());
}

// A model's initial state in one launch: psi from theta (FROM_THETA) or as given, theta, K, C at it,
// and the iteration's copies of both.  12 arrays at most, against an inverse pass, a vG pass and four
// copies: 231 -> 168 us at 400 x 400 x 30 (bound by the FP64 operations of the two evaluations).
template <bool FROM_THETA>
__global__ __launch_bounds__(kBlock) void k_init_state(InitArgs a)
{
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < a.g.n; c += gridDim.x * blockDim.x) {
        const double al = cell_alpha(a.soil, c), nv = cell_n(a.soil, c);
        double psi;
        if constexpr (FROM_THETA) {
            psi = vg_inverse(a.theta_n[c], al, nv, a.soil.ts, a.soil.tr);
            a.psi_n[c] = psi;
        } else {
            psi = a.psi_n[c];
        }
        double th, K, C;
        vg_eval(psi, a.soil.Ks[c], al, nv, a.soil.ts, a.soil.tr, th, K, C);
        a.theta_n[c] = th;
        a.theta_m[c] = th;
        a.theta_new[c] = th;
        a.psi_m[c] = psi;
        a.x[c] = psi;
        a.K[c] = K;
        a.C[c] = C;
        if (a.K32) a.K32[c] = (float)K;
    }
}

// vanGenuchten on psi^{m+1} (src/subsurface.cu:754) fused with GetIterationDifference
// (432-446), the max reduction (777) and ModifiedPicardUpdate (450-461).
__device__ __forceinline__ void b_vg_picard(VgArgs a, Blk bk)
{
    double mx[2] = {0.0, 0.0};   // increment, NaN flag
    for (int c = bk.id * blockDim.x + threadIdx.x; c < a.g.n; c += bk.n * blockDim.x) {
        const double xc = a.psi[c];
        const double pm = a.psi_m[c];
        double th, K, C;
        vg_eval(xc, a.soil.Ks[c], cell_alpha(a.soil, c), cell_n(a.soil, c), a.soil.ts, a.soil.tr,
                th, K, C);
        double d;
        if (a.rule == 1) d = fabs((xc - pm) / xc);
        else if (a.rule == 2) d = fabs((th - a.theta_m[c]) / th);
        else d = fabs(xc - pm);
        if (!(d == d) || !isfinite(xc)) mx[1] = 1.0;
        else mx[0] = fmax(mx[0], d);
        a.theta[c] = th;
        a.K[c] = K;
        a.C[c] = C;
        if (a.K32) a.K32[c] = (float)K;
        if (a.relax) a.psi_m[c] = a.am * pm + (1.0 - a.am) * xc;
    }
    block_partials<2, true>(mx, a.part_out, bk.id);
}

__global__ __launch_bounds__(kBlock) void k_vg_picard(VgArgs a, Gate gate)
{
    if (!gate.open()) return;
    b_vg_picard(a, hw_blk());
}

// Anderson acceleration of the Picard map (Walker & Ni 2011, SIAM J. Numer. Anal. 49:1715-1735;
// for Richards' equation Lott, Walker, Woodward & Yang 2012, Adv. Water Resour. 38:92-101), with
// one set of coefficients per column of cells: the vertical couplings of the operator exceed the
// horizontal ones by (dx/dz)^2, and a column's iterates oscillate on their own.  Not in the
// reference, whose ModifiedPicardUpdate (src/subsurface.cu:450-461) is the depth-0 case.
// Per column: gamma = argmin || f - dF gamma ||_2 over the ring's columns, from the normal
// equations G gamma = dF^T f by a Cholesky factorisation taken newest column first that leaves
// out a column whose pivot is below kAaDrop^2 of its diagonal (the pivot is the squared norm of
// the column's part orthogonal to the newer ones); then psi^m <- y - dY gamma, and theta, K, C
// at the new iterate (what the next assembly reads).
// A block owns kAaCols columns of cells; each column is split into kAaChunks runs of planes, one per wave
// (the 64 lanes of a wave: 64 neighbouring columns, so every plane access is one coalesced
// row).  Pass 1 streams a thread's planes once (f and y kept for the next passes, the differences of
// the ring's f formed as they are read, its share of G and dF^T f), the shares of a column are
// summed through LDS in chunk order (every thread of the column gets the same sums and the same
// gamma), pass 2 streams the planes once more (the update and vG); this pass's y waits in LDS.
// The ring holds f and y themselves and not their differences: with a full ring of 3 a pass moves
// 5 + 2 + 4 + 4 arrays (124 B per cell with K32) instead of 160 B, with the same differences.
// Bytes bound it on large surfaces: 118 us a launch at 400 x 400 x 30 (672 MB / 130 us with the
// differences stored), 775 us at 1024 x 1024 x 30 (909 us).  A surface of few columns is bound by the
// chain of van Genuchten evaluations of a thread (about 1.7 us each, 515 dependent FP64 operations)
// on the few CUs that its blocks reach: COLS = 16 columns per block spread it over four times the CUs
// and four times the threads in pass 2; pass 1 keeps the four chunks, so the sums are the same
// (32 x 32 x 20: 12.7 -> 8.8 us a launch).
constexpr int kAaCols = 64, kAaChunks = kBlock / kAaCols;
constexpr int kAaColsSmall = 16;
constexpr int kAaLds = 32;   // planes whose y is kept in LDS

// Block `bid` (kAaCols columns of cells) of the pass; every thread of the block calls it.
template <int M, int COLS>
__device__ __forceinline__ void b_aa_column(const AaArgs& a, int bid)
{
    constexpr int CH = kAaChunks, NV = M * (M + 1) / 2 + M;   // lower triangle of G, then dF^T f
    constexpr int CH2 = kBlock / COLS;                        // chunks of pass 2
    __shared__ double share[CH][NV][COLS];
    __shared__ double ysh[kAaLds][COLS];
    const Geo g = a.g;
    const int lane = threadIdx.x % COLS, chunk = threadIdx.x / COLS;
    const int col = bid * COLS + lane;
    const bool in = col < g.nxy, ylds = g.nz <= kAaLds;
    const int per = (g.nz + CH - 1) / CH;
    const int k0 = min(g.nz, chunk * per), k1 = min(g.nz, k0 + per);   // (chunk >= CH: none)
    const int nc = a.ncols;
    double G[M][M], rhs[M];
#pragma unroll
    for (int i = 0; i < M; ++i) {
        rhs[i] = 0.0;
#pragma unroll
        for (int j = 0; j < M; ++j) G[i][j] = 0.0;
    }
    // Both passes load plane k + 1 before plane k's stores: the arrays may alias as far as the
    // compiler knows, so it would not hoist those loads itself, and a plane's loads would wait
    // for the previous plane's arithmetic (in pass 2 the van Genuchten evaluation).
    if (in && k0 < k1) {
        int c = k0 * g.nxy + col;
        double pm = a.psi_m[c], xv = a.x[c], fo[M];
#pragma unroll
        for (int i = 0; i < M; ++i) fo[i] = (i < nc) ? a.f[i + 1][c] : 0.0;
        for (int k = k0; k < k1; ++k) {
            const int cn = c + g.nxy;
            double pm1 = 0.0, x1 = 0.0, fo1[M];
#pragma unroll
            for (int i = 0; i < M; ++i) fo1[i] = 0.0;
            if (k + 1 < k1) {
                pm1 = a.psi_m[cn];
                x1 = a.x[cn];
#pragma unroll
                for (int i = 0; i < M; ++i) fo1[i] = (i < nc) ? a.f[i + 1][cn] : 0.0;
            }
            const double f = xv - pm;
            const double y = pm + a.beta * f;
            a.f[0][c] = f;
            a.y[0][c] = y;
            if (ylds) ysh[k][lane] = y;
            double v[M];
#pragma unroll
            for (int i = 0; i < M; ++i) v[i] = (i == 0 ? f : fo[i - 1]) - fo[i];
#pragma unroll
            for (int i = 0; i < M; ++i) {
                if (i < nc) {
                    rhs[i] += v[i] * f;
#pragma unroll
                    for (int j = 0; j <= i; ++j) G[i][j] += v[i] * v[j];
                }
            }
            pm = pm1;
            xv = x1;
#pragma unroll
            for (int i = 0; i < M; ++i) fo[i] = fo1[i];
            c = cn;
        }
    }
    if (chunk < CH) {
        int q = 0;
#pragma unroll
        for (int i = 0; i < M; ++i)
#pragma unroll
            for (int j = 0; j <= i; ++j) share[chunk][q++][lane] = G[i][j];
#pragma unroll
        for (int i = 0; i < M; ++i) share[chunk][q++][lane] = rhs[i];
    }
    __syncthreads();
    {
        int q = 0;
#pragma unroll
        for (int i = 0; i < M; ++i)
#pragma unroll
            for (int j = 0; j <= i; ++j) {
                double v = 0.0;
#pragma unroll
                for (int h = 0; h < CH; ++h) v += share[h][q][lane];
                G[i][j] = v;
                ++q;
            }
#pragma unroll
        for (int i = 0; i < M; ++i) {
            double v = 0.0;
#pragma unroll
            for (int h = 0; h < CH; ++h) v += share[h][q][lane];
            rhs[i] = v;
            ++q;
        }
    }
    if (!in) return;   // no barrier below
    // L L^T = G restricted to the kept columns (dropped rows and columns of L are 0, with a unit
    // diagonal, so the substitutions below give them gamma = 0)
    double L[M][M];
    bool keep[M];
#pragma unroll
    for (int t = 0; t < M; ++t) {
#pragma unroll
        for (int b = 0; b < M; ++b) L[t][b] = 0.0;
        keep[t] = false;
        double s = 0.0;   // the pivot: G[t][t] less the squares of row t of L
        if (t < nc) {
            s = G[t][t];
#pragma unroll
            for (int b = 0; b < t; ++b) {
                if (keep[b]) {
                    double v = G[t][b];
#pragma unroll
                    for (int e = 0; e < b; ++e) v -= L[t][e] * L[b][e];
                    v /= L[b][b];
                    L[t][b] = v;
                    s -= v * v;
                }
            }
            keep[t] = G[t][t] > 0.0 && s >= kAaDrop * kAaDrop * G[t][t];
        }
        if (keep[t]) {
            L[t][t] = sqrt(s);
        } else {
#pragma unroll
            for (int b = 0; b < t; ++b) L[t][b] = 0.0;
            L[t][t] = 1.0;
        }
    }
    double z[M], gam[M];
#pragma unroll
    for (int t = 0; t < M; ++t) {
        double v = keep[t] ? rhs[t] : 0.0;
#pragma unroll
        for (int e = 0; e < t; ++e) v -= L[t][e] * z[e];
        z[t] = v / L[t][t];
    }
#pragma unroll
    for (int t = M - 1; t >= 0; --t) {
        double v = z[t];
#pragma unroll
        for (int e = t + 1; e < M; ++e) v -= L[e][t] * gam[e];
        gam[t] = keep[t] ? v / L[t][t] : 0.0;
    }
    const Soil& sl = a.soil;
    const int per2 = (g.nz + CH2 - 1) / CH2;
    const int m0 = min(g.nz, chunk * per2), m1 = min(g.nz, m0 + per2);
    if (m0 >= m1) return;
    int c = m0 * g.nxy + col;
    double yv = ylds ? ysh[m0][lane] : a.y[0][c], ks = sl.Ks[c], al = cell_alpha(sl, c), nv = cell_n(sl, c), yo[M];
#pragma unroll
    for (int t = 0; t < M; ++t) yo[t] = (t < nc) ? a.y[t + 1][c] : 0.0;
    for (int k = m0; k < m1; ++k) {
        const int cn = c + g.nxy;
        double y1 = 0.0, ks1 = 0.0, al1 = 0.0, nv1 = 0.0, yo1[M];
#pragma unroll
        for (int t = 0; t < M; ++t) yo1[t] = 0.0;
        if (k + 1 < m1) {
            y1 = ylds ? ysh[k + 1][lane] : a.y[0][cn];
            ks1 = sl.Ks[cn];
            al1 = cell_alpha(sl, cn);
            nv1 = cell_n(sl, cn);
#pragma unroll
            for (int t = 0; t < M; ++t) yo1[t] = (t < nc) ? a.y[t + 1][cn] : 0.0;
        }
        double v = yv;
#pragma unroll
        for (int t = 0; t < M; ++t)
            if (t < nc) v -= gam[t] * ((t == 0 ? yv : yo[t - 1]) - yo[t]);
        a.psi_m[c] = v;
        double th, K, C;
        vg_eval(v, ks, al, nv, sl.ts, sl.tr, th, K, C);
        a.theta_m[c] = th;
        a.K[c] = K;
        a.C[c] = C;
        if (a.K32) a.K32[c] = (float)K;
        yv = y1;
        ks = ks1;
        al = al1;
        nv = nv1;
#pragma unroll
        for (int t = 0; t < M; ++t) yo[t] = yo1[t];
        c = cn;
    }
}

// The Picard increment of the Anderson path (rules DHARA_PICARD_ABS_PSI / _REL_PSI): the block
// maxima of |x - psi^m| and the NaN flag only.  theta, K, C of x are needed only after the last
// pass; the other passes evaluate them at the next iterate (both in k_picard_next).
__device__ __forceinline__ void b_picard_inc(const double* __restrict__ x, const double* __restrict__ pm, int n,
                                             int rule, double* part_out, Blk bk)
{
    double mx[2] = {0.0, 0.0};
    for (int c = bk.id * blockDim.x + threadIdx.x; c < n; c += bk.n * blockDim.x) {
        const double xc = x[c];
        const double d = (rule == 1) ? fabs((xc - pm[c]) / xc) : fabs(xc - pm[c]);
        if (!(d == d) || !isfinite(xc)) mx[1] = 1.0;
        else mx[0] = fmax(mx[0], d);
    }
    block_partials<2, true>(mx, part_out, bk.id);
}

__global__ __launch_bounds__(kBlock) void k_picard_inc(const double* x, const double* pm, int n, int rule,
                                                         double* part_out, Gate gate)
{
    if (!gate.open()) return;
    b_picard_inc(x, pm, n, rule, part_out, hw_blk());
}

// The solver state to the host's report, by the first threads of a block (one word each).
__device__ __forceinline__ void report_state(const PcgState* st, HostReport* rep)
{
    constexpr int NW = sizeof(PcgState) / sizeof(int);
    static_assert(NW <= kWave && sizeof(PcgState) % sizeof(int) == 0, "one word per lane of a wave");
    if (threadIdx.x < NW) reinterpret_cast<int*>(&rep->st)[threadIdx.x] = reinterpret_cast<const int*>(st)[threadIdx.x];
}

__global__ void k_report(const PcgState* st, HostReport* rep) { report_state(st, rep); }

// One wave per row.
__global__ __launch_bounds__(1024) void k_report_sums(const double* __restrict__ part, int nparts, int nv,
                                                      HostReport* rep)
{
    const int w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    if (w >= nv) return;
    double v = 0.0;
    for (int b = lane; b < nparts; b += kWave) v += part[w * kMaxBlocks + b];
    v = wave_sum(v);
    if (lane == 0) rep->sums[w] = v;
}

__device__ __forceinline__ void picard_maxima(const double* __restrict__ part, int nparts, double (&mx)[2])
{
    __shared__ double lds[2 * 16];
    mx[0] = mx[1] = -INFINITY;
    for (int b = threadIdx.x; b < nparts; b += blockDim.x) {
        mx[0] = fmax(mx[0], part[b]);
        mx[1] = fmax(mx[1], part[kMaxBlocks + b]);
    }
    block_reduce<2, true, false>(mx, lds);
}

__global__ __launch_bounds__(kBlock) void k_picard_report(const double* part, int nparts, Gate gate, HostReport* rep)
{
    report_state(gate.st, rep);
    if (!gate.open()) return;
    double mx[2];
    picard_maxima(part, nparts, mx);
    if (threadIdx.x < 2) rep->red[threadIdx.x] = mx[threadIdx.x ? 1 : 0];
}

// After the increment: every block takes its maxima from the block partials (a maximum does not
// depend on the order), and the launch is the Anderson update or theta, K, C of the converged x, or
// (a NaN, or rule on theta and converged) neither.  One launch where the maxima, the update and the
// final evaluation each took one of 2 to 4 us, two of them idle.
template <int M, int COLS>
__global__ __launch_bounds__(kBlock) void k_picard_next(NextArgs a)
{
    if (blockIdx.x == 0) report_state(a.gate.st, a.rep);
    if (!a.gate.open()) return;
    double mx[2];
    picard_maxima(a.part, a.nparts, mx);
    if (blockIdx.x == 0 && threadIdx.x < 2) a.rep->red[threadIdx.x] = mx[threadIdx.x ? 1 : 0];
    if (mx[1] > 0.0) return;
    if (a.aa.active && mx[0] >= a.tol) b_aa_column<M, COLS>(a.aa, blockIdx.x);
    else if (a.fin) b_vg(a.vg, hw_blk());
}

__global__ __launch_bounds__(kBlock) void k_vg_inverse(Geo g, Soil s, const double* theta, double* psi)
{
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < g.n; c += gridDim.x * blockDim.x)
        psi[c] = vg_inverse(theta[c], cell_alpha(s, c), cell_n(s, c), s.ts, s.tr);
}

// ---------------------------------------------------------------------------------------
// Boundary handling
// ---------------------------------------------------------------------------------------
struct BcTypes { const int* t[6]; };

__global__ __launch_bounds__(kBlock) void k_row_flags(Geo g, BcTypes bt, uint8_t* flags)
{
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < g.n; c += gridDim.x * blockDim.x) {
        int i, j, k;
        decompose(g, c, i, j, k);
        const int bi = k * g.ny + j, bj = k * g.nx + i, bk = j * g.nx + i;
        unsigned f = 0;
        if (bt.t[FT][bk] == 0) { if (k == 1) f |= RF_CUT_D; if (k == 0) f |= RF_IDENTITY; }
        if (bt.t[FB][bk] == 0) { if (k == g.nz - 2) f |= RF_CUT_U; if (k == g.nz - 1) f |= RF_IDENTITY; }
        if (bt.t[FS][bj] == 0) { if (j == 1) f |= RF_CUT_S; if (j == 0) f |= RF_IDENTITY; }
        if (bt.t[FN][bj] == 0) { if (j == g.ny - 2) f |= RF_CUT_N; if (j == g.ny - 1) f |= RF_IDENTITY; }
        if (bt.t[FW][bi] == 0) { if (i == 1) f |= RF_CUT_W; if (i == 0) f |= RF_IDENTITY; }
        if (bt.t[FE][bi] == 0) { if (i == g.nx - 2) f |= RF_CUT_E; if (i == g.nx - 1) f |= RF_IDENTITY; }
        flags[c] = (uint8_t)f;
    }
}

// SendFluxDataToGrids (src/subsurface.cu:364-378): group value -> surface cells.
__global__ __launch_bounds__(kBlock) void k_group_scatter(int nxy, const int* procmap, const double* groups,
                                                          double* out)
{
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < nxy; t += gridDim.x * blockDim.x)
        out[t] = groups[procmap[t]];
}

// EstimateFluxes (src/global.cu:172-191) + IdentifyTopBoundary (206-257).  Both only use
// quantities fixed within a step, so the top flux is computed once per step.
__device__ __forceinline__ void b_surface_pre(SurfArgs a, Blk bk)
{
    for (int t = bk.id * blockDim.x + threadIdx.x; t < a.nxy; t += bk.n * blockDim.x) {
        const double ph = a.h[t];
        const double hp = ph + a.rain[t] * a.dt - a.evap[t] * a.dt;
        double qc = -a.K[t] * ((a.psi_n[t] - hp - 0.5 * a.dz) / (0.5 * a.dz));
        if (ph / a.dt > a.Ks[t]) qc = fmax(qc, a.Ks[t]);
        double q;
        if (hp > 0.0) {
            q = (hp / a.dt > qc) ? qc : hp / a.dt;
            q = fmin(q, (a.ts - a.theta_n[t]) * a.dz / a.dt);
            q = fmin(q, a.Ks[t]);
        } else {
            q = hp / a.dt;
        }
        a.hpoten[t] = hp;
        a.qcapa[t] = qc;
        a.qtop[t] = q;
        a.toptype[t] = 1;
    }
}

__global__ __launch_bounds__(kBlock) void k_surface_pre(SurfArgs a)
{
    b_surface_pre(a, hw_blk());
}

// SubsurfaceEstimateInfiltrationPonding, flux branch (src/subsurface.cu:474-481).
__device__ __forceinline__ void b_surface_post(SurfArgs a, Blk bk)
{
    for (int t = bk.id * blockDim.x + threadIdx.x; t < a.nxy; t += bk.n * blockDim.x)
        a.h[t] = fmax(a.hpoten[t] - a.qtop[t] * a.dt, 0.0);
}

__global__ __launch_bounds__(kBlock) void k_surface_post(SurfArgs a)
{
    b_surface_post(a, hw_blk());
}

constexpr int kXcd = 8;

__device__ __forceinline__ int xcd_tile(int w, int nb)
{
    // workgroup w runs on XCD w % 8; give XCD x the tiles [x*q + min(x, rem), ...)
    const int x = w % kXcd, slot = w / kXcd;
    const int q = nb / kXcd, rem = nb % kXcd;
    return x * q + (x < rem ? x : rem) + slot;
}

// ---------------------------------------------------------------------------------------
// Matrix-free assembly: diagonal D and right-hand side b of the mixed-form modified Picard
// system (src/subsurface.cu:381-429 with 26-353), fused with the initial residual of the
// warm-started solve r0 = b - A x0 and its dot products.
// ---------------------------------------------------------------------------------------
template <bool DIR, bool MIXED>
__device__ __forceinline__ void b_assemble(AsmArgs a, Blk bk)
{
    const Geo g = a.g;
    const double dx = g.dx, dy = g.dy, dz = g.dz, dt = a.dt;
    const double dx2inv = -1.0 / (dx * dx), dy2inv = -1.0 / (dy * dy), dz2inv = -1.0 / (dz * dz);
    // reciprocals of the step constants: one product per use instead of a division per cell
    const double idt = 1.0 / dt, idz = 1.0 / dz, sst = a.Ss * idt / a.poros;
    const double* __restrict__ K = a.K;
    const double* __restrict__ x = a.x;
    double acc[4] = {0.0, 0.0, 0.0, 0.0};   // rz, rr (solver precision), bb, rr (FP64)
    if (bk.id == 0 && threadIdx.x == 0) a.st->done = 0;   // a new solve starts
    for (int c = bk.id * blockDim.x + threadIdx.x; c < g.n; c += bk.n * blockDim.x) {
        int i, j, k;
        decompose(g, c, i, j, k);
        const double Kc = K[c];
        const double kd = (k == 0) ? 0.0 : 0.5 * (Kc + K[c - g.nxy]);
        const double ku = (k == g.nz - 1) ? 0.0 : 0.5 * (Kc + K[c + g.nxy]);
        const double ks = (j == 0) ? 0.0 : 0.5 * (Kc + K[c - g.nx]);
        const double kn = (j == g.ny - 1) ? 0.0 : 0.5 * (Kc + K[c + g.nx]);
        const double kw = (i == 0) ? 0.0 : 0.5 * (Kc + K[c - 1]);
        const double ke = (i == g.nx - 1) ? 0.0 : 0.5 * (Kc + K[c + 1]);
        const double thm = a.theta_m[c];
        const double Cc = a.C[c];
        double D = sst * thm + Cc * idt - (ke + kw) * dx2inv - (kn + ks) * dy2inv -
                   (ku + kd) * dz2inv;
        const int id2d = j * g.nx + i;
        double sink = 0.0;
        if (a.has_transp) {
            const double tr = a.transp[id2d];
            if (tr > 0.0) sink = -tr * a.root[a.procmap[id2d] * g.nz + k] * idz;
        }
        double b = sst * thm * a.psi_n[c] + Cc * idt * a.psi_m[c] - (ku - kd) * idz + (a.theta_n[c] - thm) * idt +
                   sink;
        const int bi = k * g.ny + j, bj = k * g.nx + i, bk = j * g.nx + i;
        bool ident = false;
        // top
        if (DIR && a.bctype[FT][bk] == 0) {
            if (k == 1) b -= dz2inv * kd * a.bcpsi[FT][bk];
            if (k == 0) { ident = true; b = a.bcpsi[FT][bk]; }
        } else if (k == 0) {
            b += (-a.bcq[FT][bk] * dz) * dz2inv;
        }
        // bottom: flux type means free drainage, qb = K of the cell
        if (DIR && a.bctype[FB][bk] == 0) {
            if (k == g.nz - 2) b -= dz2inv * ku * a.bcpsi[FB][bk];
            if (k == g.nz - 1) { ident = true; b = a.bcpsi[FB][bk]; }
        } else if (k == g.nz - 1) {
            a.bcq[FB][bk] = Kc;
            b += (Kc * dz) * dz2inv;
        }
        // south
        if (DIR && a.bctype[FS][bj] == 0) {
            if (j == 1) b -= dy2inv * (a.quirk ? kn : ks) * a.bcpsi[FS][bj];
            if (j == 0) { ident = true; b = a.bcpsi[FS][bj]; }
        } else if (j == 0) {
            b += (-a.bcq[FS][bj] * dy) * dy2inv;
        }
        // north
        if (DIR && a.bctype[FN][bj] == 0) {
            if (j == g.ny - 2) b -= dy2inv * (a.quirk ? ks : kn) * a.bcpsi[FN][bj];
            if (j == g.ny - 1) { ident = true; b = a.bcpsi[FN][bj]; }
        } else if (j == g.ny - 1) {
            b += (a.bcq[FN][bj] * dy) * dy2inv;
        }
        // west
        if (DIR && a.bctype[FW][bi] == 0) {
            if (i == 1) b -= dx2inv * (a.quirk ? ke : kw) * a.bcpsi[FW][bi];
            if (i == 0) { ident = true; b = a.bcpsi[FW][bi]; }
        } else if (i == 0) {
            b += (-a.bcq[FW][bi] * dx) * dx2inv;
        }
        // east
        if (DIR && a.bctype[FE][bi] == 0) {
            if (i == g.nx - 2) b -= dx2inv * (a.quirk ? kw : ke) * a.bcpsi[FE][bi];
            if (i == g.nx - 1) { ident = true; b = a.bcpsi[FE][bi]; }
        } else if (i == g.nx - 1) {
            b += (a.bcq[FE][bi] * dx) * dx2inv;
        }
        if (ident) D = 1.0;
        a.D[c] = D;
        a.b[c] = b;
        // r0 = b - A x0
        const unsigned fl = DIR ? a.flags[c] : 0u;
        double Ax;
        if (DIR && (fl & RF_IDENTITY)) {
            Ax = x[c];
        } else {
            Ax = D * x[c];
            if (k > 0 && !(DIR && (fl & RF_CUT_D))) Ax += dz2inv * kd * x[c - g.nxy];
            if (j > 0 && !(DIR && (fl & RF_CUT_S))) Ax += dy2inv * ks * x[c - g.nx];
            if (i > 0 && !(DIR && (fl & RF_CUT_W))) Ax += dx2inv * kw * x[c - 1];
            if (i < g.nx - 1 && !(DIR && (fl & RF_CUT_E))) Ax += dx2inv * ke * x[c + 1];
            if (j < g.ny - 1 && !(DIR && (fl & RF_CUT_N))) Ax += dy2inv * kn * x[c + g.nx];
            if (k < g.nz - 1 && !(DIR && (fl & RF_CUT_U))) Ax += dz2inv * ku * x[c + g.nxy];
        }
        const double r = b - Ax;
        acc[2] += b * b;
        acc[3] += r * r;
        if (MIXED) {
            const float r32 = (float)r, D32 = (float)D;
            a.D32[c] = D32;
            a.r32[c] = r32;
            a.d32[c] = 0.0f;
            const float z32 = r32 / D32;
            acc[0] += (double)r32 * (double)z32;
            acc[1] += (double)r32 * (double)r32;
        } else {
            a.r[c] = r;
            acc[0] += r * (r / D);
            acc[1] += r * r;
        }
    }
    block_partials<4, false>(acc, a.part_out, bk.id);
}

template <bool DIR, bool MIXED>
__global__ __launch_bounds__(kBlock) void k_assemble(AsmArgs a)
{
    b_assemble<DIR, MIXED>(a, hw_blk());
}

// The assembly of b_assemble (flux faces only) on an SpMV tile: a TX x TY block of columns
// marches through kc planes with the K and x planes staged in LDS (one-cell halo, double
// buffered, one barrier per plane) and the vertical neighbours in registers, so every array
// is read once per launch instead of through the caches for each of the six neighbours.  The
// arithmetic of a cell is that of b_assemble, term for term, so D, b and r are the same.
template <bool MIXED, int TX, int TY>
__global__ __launch_bounds__(TX * TY) void k_assemble_tiled(AsmArgs a, int kc, int ntx, int nty, int nkz)
{
    const Geo g = a.g;
    if (lin_bid() == 0 && lin_tid() == 0) a.st->done = 0;   // a new solve starts
    __shared__ double sx[2][TY + 2][TX + 2];
    __shared__ double sk[2][TY + 2][TX + 2];
    const int nb = ntx * nty * nkz;
    const int t = xcd_tile(blockIdx.x, nb);
    const int bz = t % nkz, bxy = t / nkz;
    const int bx = bxy % ntx, by = bxy / ntx;
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int i = bx * TX + tx, j = by * TY + ty;
    const int k0 = bz * kc, k1 = min(k0 + kc, g.nz);
    const bool in = (i < g.nx) && (j < g.ny);
    const int col = j * g.nx + i;
    const int lid = ty * TX + tx;
    int hx = -2, hy = -2;
    if (lid < TX) { hx = lid; hy = -1; }
    else if (lid < 2 * TX) { hx = lid - TX; hy = TY; }
    else if (lid < 2 * TX + TY) { hx = -1; hy = lid - 2 * TX; }
    else if (lid < 2 * TX + 2 * TY) { hx = TX; hy = lid - 2 * TX - TY; }
    const int hi = bx * TX + hx, hj = by * TY + hy;
    const bool has_halo = hx > -2 && hi >= 0 && hi < g.nx && hj >= 0 && hj < g.ny;
    const int hcol = hj * g.nx + hi;
    const double* __restrict__ x = a.x;
    const double* __restrict__ K = a.K;
    const double dx = g.dx, dy = g.dy, dz = g.dz, dt = a.dt;
    const double dx2inv = -1.0 / (dx * dx), dy2inv = -1.0 / (dy * dy), dz2inv = -1.0 / (dz * dz);
    const double idt = 1.0 / dt, idz = 1.0 / dz, sst = a.Ss * idt / a.poros;

    double xm = 0.0, km = 0.0, xc = 0.0, kcur = 0.0;
    if (in) {
        if (k0 > 0) { xm = x[(k0 - 1) * g.nxy + col]; km = K[(k0 - 1) * g.nxy + col]; }
        if (k0 < k1) { xc = x[k0 * g.nxy + col]; kcur = K[k0 * g.nxy + col]; }
    }
    double tr = 0.0;
    int rgrp = 0;
    if (in && a.has_transp) {
        tr = a.transp[col];
        rgrp = a.procmap[col];
    }
    // the plane's cell fields and halo values are loaded one plane ahead, with the next plane's
    // x and K, so that a plane does not wait a memory latency after its barrier
    struct Cell { double thm, C, psi_n, psi_m, theta_n; };
    auto load_cell = [&](int c) { return Cell{a.theta_m[c], a.C[c], a.psi_n[c], a.psi_m[c], a.theta_n[c]}; };
    Cell cc{0.0, 0.0, 0.0, 0.0, 0.0};
    double hxc = 0.0, hkc = 0.0;
    if (in && k0 < k1) cc = load_cell(k0 * g.nxy + col);
    if (has_halo && k0 < k1) { hxc = x[k0 * g.nxy + hcol]; hkc = K[k0 * g.nxy + hcol]; }
    double acc[4] = {0.0, 0.0, 0.0, 0.0};   // rz, rr (solver precision), bb, rr (FP64)
    for (int k = k0; k < k1; ++k) {
        double xn = 0.0, kn = 0.0, hxn = 0.0, hkn = 0.0;
        Cell cn{0.0, 0.0, 0.0, 0.0, 0.0};
        if (in && k + 1 < g.nz) { xn = x[(k + 1) * g.nxy + col]; kn = K[(k + 1) * g.nxy + col]; }
        if (in && k + 1 < k1) cn = load_cell((k + 1) * g.nxy + col);
        if (has_halo && k + 1 < k1) { hxn = x[(k + 1) * g.nxy + hcol]; hkn = K[(k + 1) * g.nxy + hcol]; }
        const int buf = k & 1;
        sx[buf][ty + 1][tx + 1] = xc;
        sk[buf][ty + 1][tx + 1] = kcur;
        if (has_halo) {
            sx[buf][hy + 1][hx + 1] = hxc;
            sk[buf][hy + 1][hx + 1] = hkc;
        }
        __syncthreads();
        if (in) {
            const int c = k * g.nxy + col;
            const double Kc = kcur;
            const double kd = (k == 0) ? 0.0 : 0.5 * (Kc + km);
            const double ku = (k == g.nz - 1) ? 0.0 : 0.5 * (Kc + kn);
            const double ks = (j == 0) ? 0.0 : 0.5 * (Kc + sk[buf][ty][tx + 1]);
            const double kno = (j == g.ny - 1) ? 0.0 : 0.5 * (Kc + sk[buf][ty + 2][tx + 1]);
            const double kw = (i == 0) ? 0.0 : 0.5 * (Kc + sk[buf][ty + 1][tx]);
            const double ke = (i == g.nx - 1) ? 0.0 : 0.5 * (Kc + sk[buf][ty + 1][tx + 2]);
            const double thm = cc.thm;
            const double Cc = cc.C;
            const double D = sst * thm + Cc * idt - (ke + kw) * dx2inv - (kno + ks) * dy2inv -
                             (ku + kd) * dz2inv;
            double sink = 0.0;
            if (tr > 0.0) sink = -tr * a.root[rgrp * g.nz + k] * idz;
            double b = sst * thm * cc.psi_n + Cc * idt * cc.psi_m - (ku - kd) * idz + (cc.theta_n - thm) * idt + sink;
            const int bi = k * g.ny + j, bj = k * g.nx + i;
            if (k == 0) b += (-a.bcq[FT][col] * dz) * dz2inv;
            if (k == g.nz - 1) {
                a.bcq[FB][col] = Kc;
                b += (Kc * dz) * dz2inv;
            }
            if (j == 0) b += (-a.bcq[FS][bj] * dy) * dy2inv;
            if (j == g.ny - 1) b += (a.bcq[FN][bj] * dy) * dy2inv;
            if (i == 0) b += (-a.bcq[FW][bi] * dx) * dx2inv;
            if (i == g.nx - 1) b += (a.bcq[FE][bi] * dx) * dx2inv;
            a.D[c] = D;
            a.b[c] = b;
            double Ax = D * xc;
            if (k > 0) Ax += dz2inv * kd * xm;
            if (j > 0) Ax += dy2inv * ks * sx[buf][ty][tx + 1];
            if (i > 0) Ax += dx2inv * kw * sx[buf][ty + 1][tx];
            if (i < g.nx - 1) Ax += dx2inv * ke * sx[buf][ty + 1][tx + 2];
            if (j < g.ny - 1) Ax += dy2inv * kno * sx[buf][ty + 2][tx + 1];
            if (k < g.nz - 1) Ax += dz2inv * ku * xn;
            const double r = b - Ax;
            acc[2] += b * b;
            acc[3] += r * r;
            if (MIXED) {
                const float r32 = (float)r, D32 = (float)D;
                a.D32[c] = D32;
                a.r32[c] = r32;
                a.d32[c] = 0.0f;
                const float z32 = r32 / D32;
                acc[0] += (double)r32 * (double)z32;
                acc[1] += (double)r32 * (double)r32;
            } else {
                a.r[c] = r;
                acc[0] += r * (r / D);
                acc[1] += r * r;
            }
        }
        xm = xc; km = kcur; xc = xn; kcur = kn;
        cc = cn; hxc = hxn; hkc = hkn;
    }
    block_partials<4, false>(acc, a.part_out);
}

// FP64 iterative refinement: x <- x + d (pointwise), then r = b - A x in FP64 with the
// FP32 copy of r as the next inner right-hand side.
__device__ __forceinline__ void b_refine_add(int n, double* x, const float* d, Blk bk)
{
    for (int c = bk.id * blockDim.x + threadIdx.x; c < n; c += bk.n * blockDim.x)
        x[c] += (double)d[c];
}

__global__ __launch_bounds__(kBlock) void k_refine_add(int n, double* x, const float* d)
{
    b_refine_add(n, x, d, hw_blk());
}

// The gate of a reliable update queued behind a batch of Krylov launches before the host has
// seen whether the segment ended: open (1) when the segment ended without outer convergence or
// NaN.  The gated kernels read it; the kernel that starts the next segment (k_refine_line,
// block 0) resets `done` only after every gated kernel before it has read the gate.
__global__ void k_refine_gate(PcgState* st)
{
    if (threadIdx.x == 0) st->gate = (st->done && !st->outer_conv && !st->nan) ? 1 : 0;
}

__global__ __launch_bounds__(kBlock) void k_refine_add_gated(int n, double* x, const float* d, const PcgState* st)
{
    if (!st->gate) return;
    b_refine_add(n, x, d, hw_blk());
}

// Outer test of a gated check-only update, on the device: the sum of the update's FP64 residual
// partials (slot 3, summed in a fixed order) into rr_update and, when it passes
// lin_tol^2 ||b||^2, gate = 2 (the solve has converged).  The host adopts this decision.
__global__ __launch_bounds__(kBlock) void k_refine_conv(const double* __restrict__ part, int nparts, double lin_tol,
                                                        PcgState* st)
{
    if (st->gate != 1) return;
    __shared__ double lds[16];
    double v[1] = {0.0};
    for (int b = threadIdx.x; b < nparts; b += blockDim.x) v[0] += part[3 * kMaxBlocks + b];
    block_reduce<1, false>(v, lds);
    if (threadIdx.x == 0) {
        st->rr_update = v[0];
        if (v[0] <= lin_tol * lin_tol * st->bb) st->gate = 2;
    }
}

template <bool DIR>
__device__ __forceinline__ void b_refine_residual(RefineArgs a, Blk bk)
{
    const Geo g = a.g;
    const double* __restrict__ x = a.x;
    double acc[4] = {0.0, 0.0, 0.0, 0.0};   // rz32, rr32, (unused), rr64
    if (bk.id == 0 && threadIdx.x == 0) a.st->done = 0;   // next inner solve starts
    for (int c = bk.id * blockDim.x + threadIdx.x; c < g.n; c += bk.n * blockDim.x) {
        int i, j, k;
        decompose(g, c, i, j, k);
        const unsigned fl = DIR ? a.flags[c] : 0u;
        const double Dc = a.D[c];
        auto pf = [&](int cc) { return x[cc]; };
        const double Ax = op3_row<double, DIR>(g, c, i, j, k, Dc, x[c], pf, a.K, fl);
        const double r = a.b[c] - Ax;
        const float r32 = (float)r;
        a.r32[c] = r32;
        a.d32[c] = 0.0f;
        const float z32 = r32 / a.D32[c];
        acc[3] += r * r;
        acc[0] += (double)r32 * (double)z32;
        acc[1] += (double)r32 * (double)r32;
    }
    block_partials<4, false>(acc, a.part_out, bk.id);
}

template <bool DIR>
__global__ __launch_bounds__(kBlock) void k_refine_residual(RefineArgs a)
{
    b_refine_residual<DIR>(a, hw_blk());
}

// ---------------------------------------------------------------------------------------
// Jacobi-PCG.  Iteration i:
//   (1) p = M^-1 r + beta p (beta = 0 on the first iteration), q = A p, pq = (p, q)
//   (2) alpha = rz / pq, x += alpha p, r -= alpha q, rz' = (r, M^-1 r), rr = (r, r)
// Stopping: ||r||_2 <= tol ||b||_2, checked before the first and after every iteration
// (the order of cusp::monitor, cusp/detail/monitor.inl:178-200).
// ---------------------------------------------------------------------------------------
// Start of the SpMV kernel of iteration sc.it: sum the residual partials of the previous
// kernel, decide whether the solve is over, and return beta.  Every block takes the same
// decision from the same fixed-order sums; block 0 records it.
__device__ __forceinline__ bool pcg_begin(const SolveCtl& sc, double& beta, int bid)
{
    PcgState* st = sc.st;
    if (st->done) return false;
    const bool fresh = sc.it == 0 || sc.segment_start;
    double in[4];
    sum_partials<4>(sc.part_in, sc.nparts, fresh ? 4 : 2, in);
    const double rz = in[0], rr = in[1];
    const bool lead = bid == 0 && lin_tid() == 0;
    double tol2;
    int outer = 0, nan;
    if (fresh) {
        const double bb = sc.first_sweep ? in[2] : st->bb;
        if (sc.mixed_inner) {
            outer = (in[3] <= sc.lin_tol * sc.lin_tol * bb) ? 1 : 0;
            // reduce by inner_tol, but not below half the outer target: the FP64 residual
            // after the next reliable update then meets the outer test without a further
            // FP32 segment that over-solves
            tol2 = fmax(sc.inner_tol * sc.inner_tol * rr, 0.25 * sc.lin_tol * sc.lin_tol * bb);
        } else {
            tol2 = sc.lin_tol * sc.lin_tol * bb;
            outer = (rr <= tol2) ? 1 : 0;
        }
        nan = !(isfinite(rr) && isfinite(bb) && isfinite(in[3]));
        if (lead) {
            if (sc.first_sweep) st->bb = bb;
            st->tol2 = tol2;
            st->rr_outer = in[3];
            st->outer_conv = outer;
            st->nan = nan;
        }
    } else {
        tol2 = st->tol2;
        nan = !isfinite(rr);
    }
    const int conv = (rr <= tol2) ? 1 : 0;
    if (outer || conv || nan || sc.it >= sc.maxit) {
        if (lead) {
            st->iter = sc.it;
            st->conv = conv;
            st->rr = rr;
            st->nan = st->nan | nan;
            if (!sc.mixed_inner) st->outer_conv = conv;
            st->done = 1;
        }
        return false;
    }
    if (lead) st->rz[sc.it & 1] = rz;
    beta = (sc.it == 0) ? 0.0 : rz / st->rz[(sc.it - 1) & 1];
    return true;
}


// ZIN: r holds the preconditioned residual z (column preconditioner) instead of r.
template <typename T, bool DIR, bool ZIN = false>
__device__ __forceinline__ void b_pcg3_spmv(Geo g, const uint8_t* __restrict__ flags,
                                                      const T* __restrict__ K, const T* __restrict__ D,
                                                      const T* __restrict__ r, const T* __restrict__ pold,
                                                      T* __restrict__ pnew, T* __restrict__ q, SolveCtl sc, Blk bk)
{
    double beta_d;
    if (!pcg_begin(sc, beta_d, bk.id)) return;
    const bool first = (sc.it == 0);
    const T beta = (T)beta_d;
    auto pf = [&](int c) -> T {
        const T z = ZIN ? r[c] : r[c] / D[c];
        return first ? z : z + beta * pold[c];
    };
    double acc[1] = {0.0};
    for (int c = bk.id * blockDim.x + threadIdx.x; c < g.n; c += bk.n * blockDim.x) {
        int i, j, k;
        decompose(g, c, i, j, k);
        const T pc = pf(c);
        pnew[c] = pc;
        const unsigned fl = DIR ? flags[c] : 0u;
        const T qc = op3_row<T, DIR>(g, c, i, j, k, D[c], pc, pf, K, fl);
        q[c] = qc;
        acc[0] += (double)pc * (double)qc;
    }
    block_partials<1, false>(acc, sc.part_out, bk.id);
}

template <typename T, bool DIR, bool ZIN = false>
__global__ __launch_bounds__(kBlock) void k_pcg3_spmv(Geo g, const uint8_t* __restrict__ flags,
                                                      const T* __restrict__ K, const T* __restrict__ D,
                                                      const T* __restrict__ r, const T* __restrict__ pold,
                                                      T* __restrict__ pnew, T* __restrict__ q, SolveCtl sc)
{
    b_pcg3_spmv<T, DIR, ZIN>(g, flags, K, D, r, pold, pnew, q, sc, hw_blk());
}

template <typename T>
__device__ __forceinline__ void b_pcg_update(int n, T* __restrict__ x, T* __restrict__ r,
                                                       const T* __restrict__ D, const T* __restrict__ p,
                                                       const T* __restrict__ q, SolveCtl sc, Blk bk)
{
    double alpha_d;
    if (!update_begin(sc, alpha_d, bk.id)) return;
    const T alpha = (T)alpha_d;
    double acc[2] = {0.0, 0.0};
    for (int c = bk.id * blockDim.x + threadIdx.x; c < n; c += bk.n * blockDim.x) {
        const T xc = x[c] + alpha * p[c];
        const T rc = r[c] - alpha * q[c];
        x[c] = xc;
        r[c] = rc;
        const T zc = rc / D[c];
        acc[0] += (double)rc * (double)zc;
        acc[1] += (double)rc * (double)rc;
    }
    block_partials<2, false>(acc, sc.part_out, bk.id);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_pcg_update(int n, T* __restrict__ x, T* __restrict__ r,
                                                       const T* __restrict__ D, const T* __restrict__ p,
                                                       const T* __restrict__ q, SolveCtl sc)
{
    b_pcg_update<T>(n, x, r, D, p, q, sc, hw_blk());
}

// Jacobi scaling of the one-kernel PCG: u = r * jac_inv(D), the hardware reciprocal (FP32) or
// the reciprocal refined by two Newton steps (FP64).  It is a fixed diagonal preconditioner like
// r / D, cheaper than an IEEE division; every kernel of the one-kernel form uses this function,
// so the preconditioner is the same in all of them.
__device__ __forceinline__ float jac_inv(float d) { return __builtin_amdgcn_rcpf(d); }
__device__ __forceinline__ double jac_inv(double d)
{
    double y = __builtin_amdgcn_rcp(d);
    y = fma(y, fma(-d, y, 1.0), y);
    return fma(y, fma(-d, y, 1.0), y);
}

// A copy of a slot's value in a register of its own.  A loop that keeps the loads of the next planes in
// flight reuses the slot's registers for the next load; a value that is still needed then must not
// share them, or the new load goes elsewhere and a move at the end of the loop waits for it.
__device__ __forceinline__ float take(float v)
{
    float r;
    asm volatile("v_mov_b32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}
__device__ __forceinline__ double take(double v)
{
    double r;
    asm volatile("v_mov_b64 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

// Column (vertical line) preconditioner: z = T^-1 r with T the vertical tridiagonal part of the
// 7-point operator -- diagonal D, coupling to the cell above / below -(wz/2)(K_k + K_k-+1), as
// in the SpMV --, i.e. one independent tridiagonal system per column of cells, solved by the
// Thomas algorithm with the column's forward sweep in LDS.  The flow
// operator's vertical couplings exceed the horizontal ones by (dx/dz)^2 (400 at dz = 5 cm);
// Jacobi scaling leaves that stiffness to the Krylov iteration, the column solve removes it.
// Thread = column: the plane-major layout makes every plane access coalesced.
//   INIT:   start of a solve segment: z from r; partials [(r, z), (r, r), S2, S3] with S2, S3
//           the totals of slots 2, 3 of the previous kernel's partials (||b||^2 and the FP64
//           residual of the assembly or reliable update), carried over by block 0.
//   update: alpha = (r, z) / (p, q) from the SpMV partials, x += alpha p, r -= alpha q, then z
//           from the new r; partials [(r, z), (r, r)].
// (r, z) is accumulated as sum_k w_k y_k with w_k = r_k - a_k y_k-1 = den_k y_k (T = L diag(den)
// L^T): the same value as sum_k r_k z_k, as a sum of positive terms.  The reciprocal of the
// pivot is jac_inv, a fixed function of the operator, so every application is the same
// linear map.
//
// A column's planes form a chain (elimination down, substitution up) and a thread owns a column,
// so a surface of some 10^4 columns has one or two waves per SIMD to hide memory latency with:
// the loads of A planes are in flight ahead of the plane in work, in registers.  y_k of every plane
// waits in LDS, and so does c'_k in FP32; in FP64 c'_k waits in z itself (written in the forward
// sweep, read back A planes ahead of the substitution, overwritten by it): 8 B per plane and thread
// in both, two blocks per CU up to 39 planes (the reductions' LDS comes on top; with that folded into
// the same array 40 planes fit twice and 300 x 300 x 40 took the same 57 us).  With y in registers
// instead (arrays of 16, 32 or 64 planes, unrolled) each plane waited for its own loads, since a plane
// that may not exist ends the unrolled block, and the batched form needed a launch per array size.
// Working launches, registers -> LDS: update FP64 333 x 187 x 24 30 -> 24 us (131 MB), 300 x 300 x 40
// 94 -> 57 us, 450 x 450 x 30 126 -> 106 us, 500 x 500 x 30 125 -> 107 us, 800 x 800 x 30 316 -> 294 us
// (bytes); FP32 150 x 150 x 40 26 -> 13 us, 450 x 450 x 30 55 -> 48 us, 1024 x 1024 x 30 232 -> 223 us,
// 400 x 400 x 30 37.0 -> 36.4 us (1.2 rounds of resident blocks), 800 x 800 x 12 51.7 -> 50.4 us; start-up
// FP64 333 x 187 x 24 24 -> 17 us, 300 x 300 x 40 45 -> 39 us, FP32 800 x 800 x 12 44 -> 40 us, but
// 400 x 400 x 30 26 -> 29 us (the 1.2 rounds).  In a batched launch the tallest member sets every
// block's LDS: still less time than a launch per array size (20 models of 32..128 x 32..128 x 10..40 in
// FP64, all iterating, 95 -> 50 us; 40 models of 12 planes and one of 64, all launches of six steps,
// FP64 10.5 -> 7.9 ms, FP32 9.7 -> 7.9).
template <typename T>
struct LinePlane {
    T r, q, p, x, K, D;
};

template <typename T, bool INIT>
__device__ __forceinline__ void b_line(Geo g, const T* __restrict__ K, const T* __restrict__ D,
                                           T* __restrict__ x, T* __restrict__ r, const T* __restrict__ p,
                                           const T* __restrict__ q, T* __restrict__ z, SolveCtl sc, Blk bk)
{
    extern __shared__ double line_lds[];
    double alpha_d = 0.0;
    double carry[2] = {0.0, 0.0};
    if constexpr (INIT) {
        if (sc.st->done) return;
        double in[4];
        sum_partials<4>(sc.part_in, sc.nparts, 4, in);
        carry[0] = in[2];
        carry[1] = in[3];
    } else {
        if (!update_begin(sc, alpha_d, bk.id)) return;
    }
    constexpr int A = INIT ? 8 : 4;   // planes ahead
    constexpr bool kCpInZ = sizeof(T) == 8;
    const T alpha = (T)alpha_d;
    const T hz = (T)(0.5 * g.wz);
    const int nz = g.nz, nxy = g.nxy;
    T* ysh = reinterpret_cast<T*>(line_lds) + threadIdx.x;   // y_k at ysh[k * kBlock]
    T* csh = ysh + nz * kBlock;                              // c'_k (FP32)
    double acc[INIT ? 4 : 2] = {};
    for (int col = bk.id * kBlock + threadIdx.x; col < nxy; col += bk.n * kBlock) {
        // c: the plane in work; ld: the next plane to load (it stays on the last plane once there:
        // those loads are not used)
        int c = col, ld = col, left = nz - 1;
        LinePlane<T> buf[A];
        auto fetch = [&](LinePlane<T>& b) {
            b.r = r[ld];
            if constexpr (!INIT) {
                b.q = q[ld];
                b.p = p[ld];
                b.x = x[ld];
            }
            b.K = K[ld];
            b.D = D[ld];
            ld += left > 0 ? nxy : 0;
            --left;
        };
        T kprev = T(0), yprev = T(0), inv_prev = T(0);   // (K above the first plane: its coupling is 0)
        T *ys = ysh, *cs = csh;
        auto plane = [&](const LinePlane<T>& b, bool top) {
            T rc = b.r;
            if constexpr (!INIT) {
                rc -= alpha * b.q;
                r[c] = rc;
                x[c] = b.x + alpha * b.p;
            }
            T den = b.D, w = rc;
            if (!top) {
                const T a = -hz * (b.K + kprev);   // T[k][k-1] = T[k-1][k]
                const T cpk = a * inv_prev;        // c'_{k-1}
                if constexpr (kCpInZ) {
                    z[c - nxy] = cpk;
                } else {
                    *cs = cpk;
                    cs += kBlock;
                }
                den -= a * cpk;
                w -= a * yprev;
            }
            const T inv = jac_inv(den);
            const T yk = w * inv;
            *ys = yk;
            ys += kBlock;
            acc[0] += (double)w * (double)yk;
            acc[1] += (double)rc * (double)rc;
            kprev = b.K;
            asm volatile("" : "+v"(kprev));   // a copy: the slot's register is free for the next load
            yprev = yk;
            inv_prev = inv;
            c += nxy;
        };
        LinePlane<T> b0;
        fetch(b0);
#pragma unroll
        for (int u = 0; u < A; ++u) fetch(buf[u]);
        plane(b0, true);
        int k = 1;
        for (; k + A <= nz; k += A) {
#pragma unroll
            for (int u = 0; u < A; ++u) {
                plane(buf[u], false);
                fetch(buf[u]);
                __builtin_amdgcn_sched_barrier(0);   // else a later plane's r - alpha q is taken here, and waits
            }
        }
#pragma unroll
        for (int u = 0; u < A; ++u)
            if (k + u < nz) plane(buf[u], false);
        // back substitution
        c -= nxy;
        ys -= kBlock;
        T zn = *ys;
        z[c] = zn;
        if constexpr (kCpInZ) {
            T cb[A];
            int lb = c, bl = nz - 1;   // planes above the one at lb
            auto back = [&](T& b) {
                lb -= bl > 0 ? nxy : 0;
                --bl;
                b = z[lb];
            };
            auto sub = [&](T cp) {
                c -= nxy;
                ys -= kBlock;
                zn = *ys - cp * zn;
                z[c] = zn;
            };
#pragma unroll
            for (int u = 0; u < A; ++u) back(cb[u]);
            int n = nz - 1;
            for (; n >= A; n -= A) {
#pragma unroll
                for (int u = 0; u < A; ++u) {
                    sub(cb[u]);
                    back(cb[u]);
                }
            }
#pragma unroll
            for (int u = 0; u < A; ++u)
                if (u < n) sub(cb[u]);
        } else {
            for (int n = nz - 1; n > 0; --n) {
                c -= nxy;
                ys -= kBlock;
                cs -= kBlock;
                zn = *ys - *cs * zn;
                z[c] = zn;
            }
        }
    }
    if constexpr (INIT) {
        if (bk.id == 0 && threadIdx.x == 0) {
            acc[2] = carry[0];
            acc[3] = carry[1];
        }
        block_partials<4, false>(acc, sc.part_out, bk.id);
    } else {
        block_partials<2, false>(acc, sc.part_out, bk.id);
    }
}

template <typename T, bool INIT>
__global__ __launch_bounds__(kBlock) void k_line(Geo g, const T* __restrict__ K, const T* __restrict__ D,
                                                     T* __restrict__ x, T* __restrict__ r, const T* __restrict__ p,
                                                     const T* __restrict__ q, T* __restrict__ z, SolveCtl sc)
{
    b_line<T, INIT>(g, K, D, x, r, p, q, z, sc, hw_blk());
}

// SpMV kernel of the column-preconditioned PCG: p = z + beta p_old, q = A p, partial (p, q), on a
// TX x TY tile of columns marching through kc planes with the p / K planes staged in LDS (one-cell
// halo, double buffered, one barrier per plane).  The loads of A planes, own column and halo, are in
// flight in register slots that an unrolled loop goes round, without branches (a plane or halo that is
// not there repeats a valid load); with slots moved down by one per plane the moves waited for the
// fresh loads.  In the first iteration p_old is not read (z in its place, from cache).  At the same
// tile this gave 38.9 -> 36.4 us at 400 x 400 x 30 and 211 -> 204 at 1024 x 1024 x 30 in FP32 (the halo's
// requests bound it there), with the tiles of default_zin_tile 28 and 172 us (21 and 140 at copy rate).
template <typename T, int TX, int TY>
__global__ __launch_bounds__(TX * TY) void k_spmv_z(Geo g, const T* __restrict__ K, const T* __restrict__ D,
                                                    const T* __restrict__ z, const T* __restrict__ pold,
                                                    T* __restrict__ pnew, T* __restrict__ q, SolveCtl sc, int kc,
                                                    int ntx, int nty, int nkz)
{
    double beta_d;
    if (!pcg_begin(sc, beta_d, lin_bid())) return;
    const bool first = sc.it == 0;
    const T beta = (T)beta_d;
    __shared__ T sp[2][TY + 2][TX + 2];
    __shared__ T sk[2][TY + 2][TX + 2];
    const int nb = ntx * nty * nkz;
    const int t = xcd_tile(blockIdx.x, nb);
    const int bz = t % nkz, bxy = t / nkz;
    const int bx = bxy % ntx, by = bxy / ntx;
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int i = bx * TX + tx, j = by * TY + ty;
    const int k0 = bz * kc, k1 = min(k0 + kc, g.nz);
    const bool in = (i < g.nx) && (j < g.ny);
    const int col = j * g.nx + i;
    const int lid = ty * TX + tx;
    int hx = -2, hy = -2;
    if (lid < TX) { hx = lid; hy = -1; }
    else if (lid < 2 * TX) { hx = lid - TX; hy = TY; }
    else if (lid < 2 * TX + TY) { hx = -1; hy = lid - 2 * TX; }
    else if (lid < 2 * TX + 2 * TY) { hx = TX; hy = lid - 2 * TX - TY; }
    const int hi = bx * TX + hx, hj = by * TY + hy;
    const bool has_halo = hx > -2 && hi >= 0 && hi < g.nx && hj >= 0 && hj < g.ny;
    const int nxy = g.nxy, nz = g.nz;
    const T wx = (T)g.wx, wy = (T)g.wy, wz = (T)g.wz, half = T(0.5);
    auto pv = [&](T zv, T pov) -> T { return first ? zv : zv + beta * pov; };
    // the columns that a thread loads from: its own, and its halo's (any valid one without)
    const int ccol = min(j, g.ny - 1) * g.nx + min(i, g.nx - 1);
    const int hcol = has_halo ? hj * g.nx + hi : by * TY * g.nx + bx * TX;
    const T* po = first ? z : pold;   // (z again: in cache, p_old is not used)

    constexpr int A = sizeof(T) == 4 ? 4 : 2;
    struct Own { T z, p, K, D; } own[A];   // planes k + 1 .. k + A at step k
    struct Halo { T z, p, K; } halo[A];    // planes k .. k + A - 1
    const int lo = min(k1, nz - 1);        // last plane of the own column that is used
    int fo = k0 + 1, fh = k0;              // next planes to load
    auto fetch_own = [&](Own& o) {
        const int c = min(fo, lo) * nxy + ccol;
        ++fo;
        o.z = z[c]; o.p = po[c]; o.K = K[c]; o.D = D[c];
    };
    auto fetch_halo = [&](Halo& h) {
        const int c = min(fh, k1 - 1) * nxy + hcol;
        ++fh;
        h.z = z[c]; h.p = po[c]; h.K = K[c];
    };
    const int cm = max(k0 - 1, 0) * nxy + ccol, c0 = k0 * nxy + ccol;
    const T zm = z[cm], zc = z[c0], qm = po[cm], qc = po[c0];
    T km = K[cm], kcur = K[c0], dc = D[c0];
#pragma unroll
    for (int u = 0; u < A; ++u) {
        fetch_halo(halo[u]);
        fetch_own(own[u]);
    }
    T pm = pv(zm, qm), pc = pv(zc, qc);
    double acc = 0.0;
    auto plane = [&](int k, Own& o, Halo& h, bool fetch) {
        const int buf = k & 1;
        sp[buf][ty + 1][tx + 1] = pc;
        sk[buf][ty + 1][tx + 1] = kcur;
        if (has_halo) {
            sp[buf][hy + 1][hx + 1] = pv(h.z, h.p);
            sk[buf][hy + 1][hx + 1] = h.K;
        }
        T pn = pv(o.z, o.p);
        asm volatile("" : "+v"(pn));   // computed here, not where it is used
        const T kn = take(o.K), dn = take(o.D);
        if (fetch) {
            fetch_halo(h);
            fetch_own(o);
        }
        __syncthreads();
        if (in) {
            const int c = k * nxy + col;
            T qv = dc * pc;
            if (k > 0) qv -= wz * (half * (kcur + km)) * pm;
            if (j > 0) qv -= wy * (half * (kcur + sk[buf][ty][tx + 1])) * sp[buf][ty][tx + 1];
            if (i > 0) qv -= wx * (half * (kcur + sk[buf][ty + 1][tx])) * sp[buf][ty + 1][tx];
            if (i < g.nx - 1) qv -= wx * (half * (kcur + sk[buf][ty + 1][tx + 2])) * sp[buf][ty + 1][tx + 2];
            if (j < g.ny - 1) qv -= wy * (half * (kcur + sk[buf][ty + 2][tx + 1])) * sp[buf][ty + 2][tx + 1];
            if (k < nz - 1) qv -= wz * (half * (kcur + kn)) * pn;
            pnew[c] = pc;
            q[c] = qv;
            acc += (double)pc * (double)qv;
        }
        pm = pc; km = kcur;
        pc = pn; kcur = kn; dc = dn;
    };
    int k = k0;
    for (; k + A <= k1; k += A) {
#pragma unroll
        for (int u = 0; u < A; ++u) {
            plane(k + u, own[u], halo[u], true);
            __builtin_amdgcn_sched_barrier(0);   // keeps the loads of a plane behind the uses of its slot
        }
    }
#pragma unroll
    for (int u = 0; u < A; ++u)
        if (k + u < k1) plane(k + u, own[u], halo[u], false);
    double v[1] = {acc};
    block_partials<1, false>(v, sc.part_out);
}

// Reliable update of the mixed column-preconditioned PCG after k_refine_add (x += d): the true
// residual r = b - A x in FP64, r32 = (float) r, d = 0, and the start of the next FP32 segment,
// z32 = T32^-1 r32 with T32 the column operator of the FP32 solve ((float) K, (float) D, the
// arithmetic of k_line) -- k_refine_residual_tiled and the k_line start-up in one launch.  (x
// += d stays a launch of its own: a block reads x on its halo, which another block would be
// updating.)  A block owns TX x TY whole columns (the column solve needs them); x and K of each
// plane are staged in LDS with a one-cell halo, the vertical neighbours stay in registers.
// Partials [(r32, z32), (r32, r32), 0, (r, r)] per block, the layout of a segment start.
// FULL = false: the FP64 residual's norm only (partials [0, 0, 0, (r, r)]; r32, d32 and z32 are
// not written), for the outer test of an update after which the solve usually ends; this form
// runs only when the gate (k_refine_gate) is open, so that it can be queued before the host has
// seen the segment end.
template <int NZM, int TX, int TY, bool FULL>
__global__ __launch_bounds__(TX * TY) void k_refine_line(RefineArgs a, float* __restrict__ z32, int ntx, int nty)
{
    if (!FULL && !a.st->gate) return;
    const Geo g = a.g;
    // the next inner solve starts (the check-only form leaves the ended segment's state as it is:
    // the host reads it after the check, and the rest of the update resets it)
    if (FULL && lin_bid() == 0 && lin_tid() == 0) a.st->done = 0;
    __shared__ double sx[2][TY + 2][TX + 2];
    __shared__ double sk[2][TY + 2][TX + 2];
    const int t = xcd_tile(blockIdx.x, ntx * nty);
    const int bx = t % ntx, by = t / ntx;
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int i = bx * TX + tx, j = by * TY + ty;
    const bool in = (i < g.nx) && (j < g.ny);
    const int col = j * g.nx + i;
    const int lid = ty * TX + tx;
    int hx = -2, hy = -2;
    if (lid < TX) { hx = lid; hy = -1; }
    else if (lid < 2 * TX) { hx = lid - TX; hy = TY; }
    else if (lid < 2 * TX + TY) { hx = -1; hy = lid - 2 * TX; }
    else if (lid < 2 * TX + 2 * TY) { hx = TX; hy = lid - 2 * TX - TY; }
    const int hi = bx * TX + hx, hj = by * TY + hy;
    const bool has_halo = hx > -2 && hi >= 0 && hi < g.nx && hj >= 0 && hj < g.ny;
    const int hcol = hj * g.nx + hi;
    const double* __restrict__ x = a.x;
    const double* __restrict__ K = a.K;
    const double wx = g.wx, wy = g.wy, wz = g.wz, half = 0.5;
    const float hz = (float)(0.5 * g.wz);
    const int nz = g.nz, nxy = g.nxy;

    double xm = 0.0, km = 0.0, xc = 0.0, kcur = 0.0, xn = 0.0, kn = 0.0;
    // loads run ahead of their use: the own column's x and K two planes ahead (plane k + 1 is
    // already in the stencil of plane k), its D and b and the halo's x and K one plane ahead.  A
    // block has a whole column per thread (few waves per SIMD), so each plane would otherwise
    // wait a full memory latency after its barrier
    double Dc = 1.0, bc = 0.0, hxc = 0.0, hkc = 0.0;
    if (in) {
        xc = x[col];
        kcur = K[col];
        Dc = a.D[col];
        bc = a.b[col];
        if (nz > 1) {
            xn = x[nxy + col];
            kn = K[nxy + col];
        }
    }
    if (has_halo) {
        hxc = x[hcol];
        hkc = K[hcol];
    }
    float y[NZM], cp[NZM];
    float kprev = 0.0f, yprev = 0.0f, inv_prev = 0.0f;
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < NZM; ++k) {
        if (k < nz) {
            double x2 = 0.0, k2 = 0.0, Dn = 1.0, bn = 0.0, hxn = 0.0, hkn = 0.0;
            if (in && k + 1 < nz) {
                const int cn = (k + 1) * nxy + col;
                Dn = a.D[cn];
                bn = a.b[cn];
                if (k + 2 < nz) {
                    x2 = x[cn + nxy];
                    k2 = K[cn + nxy];
                }
            }
            if (has_halo && k + 1 < nz) {
                hxn = x[(k + 1) * nxy + hcol];
                hkn = K[(k + 1) * nxy + hcol];
            }
            const int buf = k & 1;
            sx[buf][ty + 1][tx + 1] = xc;
            sk[buf][ty + 1][tx + 1] = kcur;
            if (has_halo) {
                sx[buf][hy + 1][hx + 1] = hxc;
                sk[buf][hy + 1][hx + 1] = hkc;
            }
            __syncthreads();
            if (in) {
                const int c = k * nxy + col;
                double ax = Dc * xc;
                if (k > 0) ax -= wz * (half * (kcur + km)) * xm;
                if (j > 0) ax -= wy * (half * (kcur + sk[buf][ty][tx + 1])) * sx[buf][ty][tx + 1];
                if (i > 0) ax -= wx * (half * (kcur + sk[buf][ty + 1][tx])) * sx[buf][ty + 1][tx];
                if (i < g.nx - 1) ax -= wx * (half * (kcur + sk[buf][ty + 1][tx + 2])) * sx[buf][ty + 1][tx + 2];
                if (j < g.ny - 1) ax -= wy * (half * (kcur + sk[buf][ty + 2][tx + 1])) * sx[buf][ty + 2][tx + 1];
                if (k < nz - 1) ax -= wz * (half * (kcur + kn)) * xn;
                const double r = bc - ax;
                acc[3] += r * r;
                if constexpr (FULL) {
                    const float r32 = (float)r;
                    a.r32[c] = r32;
                    a.d32[c] = 0.0f;
                    // forward elimination of the FP32 column system (k_line's arithmetic)
                    const float k32 = (float)kcur;
                    float den = (float)Dc, w = r32;
                    if (k > 0) {
                        const float av = -hz * (k32 + kprev);
                        const float cpk = av * inv_prev;
                        cp[k - 1] = cpk;
                        den -= av * cpk;
                        w -= av * yprev;
                    }
                    const float inv = jac_inv(den);
                    const float yk = w * inv;
                    y[k] = yk;
                    acc[0] += (double)w * (double)yk;
                    acc[1] += (double)r32 * (double)r32;
                    kprev = k32;
                    yprev = yk;
                    inv_prev = inv;
                }
            }
            xm = xc; km = kcur; xc = xn; kcur = kn; xn = x2; kn = k2;
            Dc = Dn; bc = bn; hxc = hxn; hkc = hkn;
        }
    }
    if (FULL && in) {
        float zn = 0.0f;
#pragma unroll
        for (int k = NZM - 1; k >= 0; --k) {
            if (k < nz) {
                const float zk = (k == nz - 1) ? y[k] : y[k] - cp[k] * zn;
                z32[k * nxy + col] = zk;
                zn = zk;
            }
        }
    }
    block_partials<4, false>(acc, a.part_out);
}

// LDS-tiled 2.5D SpMV.  Block = TX x TY threads owning TX x TY columns; the block marches
// through planes k0..k0+kc-1.  For each plane the new search direction p = M^-1 r + beta p
// and the conductivity K are written into a (TY+2) x (TX+2) LDS tile (the one-cell halo is
// computed by the first 2(TX+TY) threads); the k-1 / k+1 values of the thread's own column
// come from registers (one plane of look-ahead).  Two LDS buffers alternate by plane parity,
// so one barrier per plane suffices.  Blocks are numbered so that each XCD (workgroups are
// dealt to the 8 XCDs round-robin) gets a contiguous band of tiles: neighbouring tiles, whose
// halos overlap, then share that XCD's L2.

// Load / store at a 32-bit byte offset from a kernel-argument base (the scalar-base plus vector
// offset addressing form; the caller guarantees that every offset fits in 32 bits).
template <typename T>
__device__ __forceinline__ T ld_off(const T* base, unsigned byte_off)
{
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + byte_off);
}
template <typename T>
__device__ __forceinline__ void st_off(T* base, unsigned byte_off, T v)
{
    *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + byte_off) = v;
}


// INIT: start-up of a one-kernel PCG segment instead -- u = M^-1 r, A u, no stores, partials
// [(r, u), (r, r), (u, A u), (p_old, A u), 0] (p_old: the kept direction, it > 0).  (The
// column-preconditioned form, whose input is z, is k_spmv_z.)
template <typename T, bool DIR, int TX, int TY, bool INIT = false>
__global__ __launch_bounds__(TX * TY) void k_pcg3_spmv_tiled(Geo g, const uint8_t* __restrict__ flags,
                                                             const T* __restrict__ K, const T* __restrict__ D,
                                                             const T* __restrict__ r, const T* __restrict__ pold,
                                                             T* __restrict__ pnew, T* __restrict__ q,
                                                             SolveCtl sc, int kc, int ntx, int nty, int nkz)
{
    double beta_d;
    if (!pcg_begin(sc, beta_d, lin_bid())) return;
    const bool first = INIT || (sc.it == 0);
    const bool kept = INIT && sc.it > 0;
    double acc5[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    const T beta = (T)beta_d;
    __shared__ T sp[2][TY + 2][TX + 2];
    __shared__ T sk[2][TY + 2][TX + 2];

    const int nb = ntx * nty * nkz;
    const int t = xcd_tile(blockIdx.x, nb);
    const int bz = t % nkz;
    const int bxy = t / nkz;
    const int bx = bxy % ntx, by = bxy / ntx;
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int i = bx * TX + tx, j = by * TY + ty;
    const int k0 = bz * kc;
    const int k1 = min(k0 + kc, g.nz);
    const bool in = (i < g.nx) && (j < g.ny);
    const int col = j * g.nx + i;

    // halo cell of this thread (if any): top row, bottom row, left column, right column
    const int lid = ty * TX + tx;
    int hx = -2, hy = -2;
    if (lid < TX) { hx = lid; hy = -1; }
    else if (lid < 2 * TX) { hx = lid - TX; hy = TY; }
    else if (lid < 2 * TX + TY) { hx = -1; hy = lid - 2 * TX; }
    else if (lid < 2 * TX + 2 * TY) { hx = TX; hy = lid - 2 * TX - TY; }
    const int hi = bx * TX + hx, hj = by * TY + hy;
    const bool has_halo = hx > -2 && hi >= 0 && hi < g.nx && hj >= 0 && hj < g.ny;
    const int hcol = hj * g.nx + hi;

    auto jac = [&](T rv, T dv) -> T { return INIT ? rv * jac_inv(dv) : rv / dv; };
    auto pval = [&](int c) -> T {
        const T z = jac(r[c], D[c]);
        return first ? z : z + beta * pold[c];
    };
    const T wx = (T)g.wx, wy = (T)g.wy, wz = (T)g.wz, half = T(0.5);

    T pm = T(0), km = T(0), pc = T(0), kcur = T(0), dc = T(1);
    if (in) {
        if (k0 > 0) {
            const int c = (k0 - 1) * g.nxy + col;
            pm = pval(c);
            km = K[c];
        }
        if (k0 < k1) {
            const int c = k0 * g.nxy + col;
            dc = D[c];
            const T z = jac(r[c], dc);
            pc = first ? z : z + beta * pold[c];
            kcur = K[c];
        }
    }
    double acc = 0.0;
    for (int k = k0; k < k1; ++k) {
        // look-ahead: plane k+1 of the own column
        T pn = T(0), kn = T(0), dn = T(1);
        if (in && k + 1 < g.nz) {
            const int c = (k + 1) * g.nxy + col;
            dn = D[c];
            const T z = jac(r[c], dn);
            pn = first ? z : z + beta * pold[c];
            kn = K[c];
        }
        const int buf = k & 1;
        sp[buf][ty + 1][tx + 1] = pc;
        sk[buf][ty + 1][tx + 1] = kcur;
        if (has_halo) {
            const int c = k * g.nxy + hcol;
            sp[buf][hy + 1][hx + 1] = pval(c);
            sk[buf][hy + 1][hx + 1] = K[c];
        }
        __syncthreads();
        if (in) {
            const int c = k * g.nxy + col;
            T qv;
            const unsigned fl = DIR ? flags[c] : 0u;
            if (DIR && (fl & RF_IDENTITY)) {
                qv = pc;
            } else {
                qv = dc * pc;
                if (k > 0 && !(DIR && (fl & RF_CUT_D))) qv -= wz * (half * (kcur + km)) * pm;
                if (j > 0 && !(DIR && (fl & RF_CUT_S)))
                    qv -= wy * (half * (kcur + sk[buf][ty][tx + 1])) * sp[buf][ty][tx + 1];
                if (i > 0 && !(DIR && (fl & RF_CUT_W)))
                    qv -= wx * (half * (kcur + sk[buf][ty + 1][tx])) * sp[buf][ty + 1][tx];
                if (i < g.nx - 1 && !(DIR && (fl & RF_CUT_E)))
                    qv -= wx * (half * (kcur + sk[buf][ty + 1][tx + 2])) * sp[buf][ty + 1][tx + 2];
                if (j < g.ny - 1 && !(DIR && (fl & RF_CUT_N)))
                    qv -= wy * (half * (kcur + sk[buf][ty + 2][tx + 1])) * sp[buf][ty + 2][tx + 1];
                if (k < g.nz - 1 && !(DIR && (fl & RF_CUT_U))) qv -= wz * (half * (kcur + kn)) * pn;
            }
            if constexpr (INIT) {
                const T rc = r[c];
                acc5[0] += (double)rc * (double)pc;
                acc5[1] += (double)rc * (double)rc;
                acc5[2] += (double)pc * (double)qv;
                if (kept) acc5[3] += (double)pold[c] * (double)qv;
            } else {
                pnew[c] = pc;
                q[c] = qv;
                acc += (double)pc * (double)qv;
            }
        }
        pm = pc;
        km = kcur;
        pc = pn;
        kcur = kn;
        dc = dn;
    }
    if constexpr (INIT) {
        block_partials<5, false>(acc5, sc.part_out);
    } else {
        double v[1] = {acc};
        block_partials<1, false>(v, sc.part_out);
    }
}

// FP64 residual of a reliable update (after k_refine_add), LDS-tiled like the SpMV: r = b - A x,
// r32 = (float) r, d32 = 0, partials [rz32, rr32, 0, rr64].  No Dirichlet rows.  The untiled
// grid-stride form re-reads the k +- 1 and j +- 1 neighbours from HBM (2.4x the algorithmic
// bytes); here x and K of a plane are staged once per tile and the vertical neighbours stay in
// registers.  Same operations in the same order as op3_row.
template <int TX, int TY>
__global__ __launch_bounds__(TX * TY) void k_refine_residual_tiled(RefineArgs a, int kc, int ntx, int nty, int nkz)
{
    const Geo g = a.g;
    if (lin_bid() == 0 && lin_tid() == 0) a.st->done = 0;   // the next inner solve starts
    __shared__ double sx[2][TY + 2][TX + 2];
    __shared__ double sk[2][TY + 2][TX + 2];
    const int nb = ntx * nty * nkz;
    const int t = xcd_tile(blockIdx.x, nb);
    const int bz = t % nkz, bxy = t / nkz;
    const int bx = bxy % ntx, by = bxy / ntx;
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int i = bx * TX + tx, j = by * TY + ty;
    const int k0 = bz * kc, k1 = min(k0 + kc, g.nz);
    const bool in = (i < g.nx) && (j < g.ny);
    const int col = j * g.nx + i;
    const int lid = ty * TX + tx;
    int hx = -2, hy = -2;
    if (lid < TX) { hx = lid; hy = -1; }
    else if (lid < 2 * TX) { hx = lid - TX; hy = TY; }
    else if (lid < 2 * TX + TY) { hx = -1; hy = lid - 2 * TX; }
    else if (lid < 2 * TX + 2 * TY) { hx = TX; hy = lid - 2 * TX - TY; }
    const int hi = bx * TX + hx, hj = by * TY + hy;
    const bool has_halo = hx > -2 && hi >= 0 && hi < g.nx && hj >= 0 && hj < g.ny;
    const int hcol = hj * g.nx + hi;
    const double* __restrict__ x = a.x;
    const double* __restrict__ K = a.K;
    const double wx = g.wx, wy = g.wy, wz = g.wz, half = 0.5;

    double xm = 0.0, km = 0.0, xc = 0.0, kcur = 0.0;
    if (in) {
        if (k0 > 0) { xm = x[(k0 - 1) * g.nxy + col]; km = K[(k0 - 1) * g.nxy + col]; }
        if (k0 < k1) { xc = x[k0 * g.nxy + col]; kcur = K[k0 * g.nxy + col]; }
    }
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (int k = k0; k < k1; ++k) {
        double xn = 0.0, kn = 0.0;
        if (in && k + 1 < g.nz) { xn = x[(k + 1) * g.nxy + col]; kn = K[(k + 1) * g.nxy + col]; }
        const int buf = k & 1;
        sx[buf][ty + 1][tx + 1] = xc;
        sk[buf][ty + 1][tx + 1] = kcur;
        if (has_halo) {
            sx[buf][hy + 1][hx + 1] = x[k * g.nxy + hcol];
            sk[buf][hy + 1][hx + 1] = K[k * g.nxy + hcol];
        }
        __syncthreads();
        if (in) {
            const int c = k * g.nxy + col;
            double ax = a.D[c] * xc;
            if (k > 0) ax -= wz * (half * (kcur + km)) * xm;
            if (j > 0) ax -= wy * (half * (kcur + sk[buf][ty][tx + 1])) * sx[buf][ty][tx + 1];
            if (i > 0) ax -= wx * (half * (kcur + sk[buf][ty + 1][tx])) * sx[buf][ty + 1][tx];
            if (i < g.nx - 1) ax -= wx * (half * (kcur + sk[buf][ty + 1][tx + 2])) * sx[buf][ty + 1][tx + 2];
            if (j < g.ny - 1) ax -= wy * (half * (kcur + sk[buf][ty + 2][tx + 1])) * sx[buf][ty + 2][tx + 1];
            if (k < g.nz - 1) ax -= wz * (half * (kcur + kn)) * xn;
            const double r = a.b[c] - ax;
            const float r32 = (float)r;
            a.r32[c] = r32;
            a.d32[c] = 0.0f;
            const float z32 = r32 / a.D32[c];
            acc[3] += r * r;
            acc[0] += (double)r32 * (double)z32;
            acc[1] += (double)r32 * (double)r32;
        }
        xm = xc; km = kcur; xc = xn; kcur = kn;
    }
    block_partials<4, false>(acc, a.part_out);
}

template <typename T, bool DIR>
__global__ __launch_bounds__(kBlock) void k_apply3(Geo g, const uint8_t* flags, const T* K,
                                                   const T* D, const T* x, T* y)
{
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < g.n; c += gridDim.x * blockDim.x) {
        int i, j, k;
        decompose(g, c, i, j, k);
        auto pf = [&](int cc) { return x[cc]; };
        y[c] = op3_row<T, DIR>(g, c, i, j, k, D[c], x[c], pf, K, DIR ? flags[c] : 0u);
    }
}

__global__ __launch_bounds__(kBlock) void k_cast_f32(int n, const double* in, float* out)
{
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x)
        out[c] = (float)in[c];
}

__global__ __launch_bounds__(kBlock) void k_cast_f64(int n, const float* in, double* out)
{
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x)
        out[c] = (double)in[c];
}

// ---------------------------------------------------------------------------------------
// End of step: mass-balance sums (src/subsurface.cu:494-629, 808-826) and the state copies
// psi^n <- psi^{n+1}, theta^n <- theta carry (836-840).
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ void b_end_step(EndArgs a, Blk bk)
{
    const Geo g = a.g;
    // 0 sum dtheta, 1 sum Ss th/phi dpsi dz, 2 sink volume/area, 3 qt, 4 qb, 5 qw, 6 qe, 7 qs, 8 qn
    double acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int c = bk.id * blockDim.x + threadIdx.x; c < g.n; c += bk.n * blockDim.x) {
        int i, j, k;
        decompose(g, c, i, j, k);
        const double thn = a.theta_new[c];
        const double xc = a.x[c];
        acc[0] += thn - a.theta_n[c];
        acc[1] += (xc - a.psi_n[c]) * (a.Ss / a.dt * thn / a.poros) * g.dz * a.dt;
        const int id2d = j * g.nx + i;
        if (a.has_transp) {
            const double tr = a.transp[id2d];
            if (tr > 0.0) acc[2] += tr * a.dt * a.root[a.procmap[id2d] * g.nz + k];
        }
        const int bi = k * g.ny + j, bj = k * g.nx + i, bk = id2d;
        if (k == 0 && a.bctype[FT][bk] != 0) acc[3] += a.bcq[FT][bk];
        if (k == g.nz - 1 && a.bctype[FB][bk] != 0) acc[4] += a.bcq[FB][bk];
        if (i == 0 && a.bctype[FW][bi] != 0) acc[5] += a.bcq[FW][bi];
        if (i == g.nx - 1 && a.bctype[FE][bi] != 0) acc[6] += a.bcq[FE][bi];
        if (j == 0 && a.bctype[FS][bj] != 0) acc[7] += a.bcq[FS][bj];
        if (j == g.ny - 1 && a.bctype[FN][bj] != 0) acc[8] += a.bcq[FN][bj];
        a.psi_n[c] = xc;
        a.theta_n[c] = a.carry_reference ? a.theta_m[c] : thn;
    }
    block_partials<9, false>(acc, a.part_out, bk.id);
}

__global__ __launch_bounds__(kBlock) void k_end_step(EndArgs a)
{
    b_end_step(a, hw_blk());
}

// ---------------------------------------------------------------------------------------
// Overland
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ bool is_ring(const Geo2& g, int i, int j)
{
    return i == 0 || j == 0 || i == g.nx - 1 || j == g.ny - 1;
}

// Face conductance of the diffusive-wave model (UpdateKOverland, src/overland.cu:193-368):
// S = sqrt(gx^2 + gy^2), K = h_avg^(5/3) / (n_avg sqrt(S)) when the upwind depth, the mean
// depth exceed hmin and |S| > delta, K0 otherwise.  `up_nb` selects the neighbour as the
// upwind cell.
__device__ __forceinline__ double olf_face_k(double gdir, double gcross, double h_nb, double h_c,
                                             double m_nb, double m_c, bool up_nb, double hmin,
                                             double delta, double K0)
{
    const double Ssl = sqrt(gdir * gdir + gcross * gcross);
    const double hup = up_nb ? h_nb : h_c;
    const double hav = (h_nb + h_c) / 2.;
    if (hup > hmin && hav > hmin && fabs(Ssl) > delta)
        return pow(hav, 5. / 3.) / (0.5 * (m_nb + m_c) * sqrt(Ssl));
    return K0;
}

// H = h + z (stored; formed again for the neighbours, from the same two values), and the east and
// north face conductances of every face the eliminated system uses, each evaluated from its
// non-ring cell (the row that owns the coupling in the reference matrix).
__device__ __forceinline__ void b_olf_faces(OlfArgs a, Blk bk)
{
    const Geo2 g = a.g;
    const int nx = g.nx;
    const double* __restrict__ h = a.h;
    const double* __restrict__ z = a.z;
    const double* __restrict__ m = a.mann;
    auto H = [&](int c) { return h[c] + z[c]; };
    for (int c = bk.id * blockDim.x + threadIdx.x; c < g.n; c += bk.n * blockDim.x) {
        const int j = c / nx, i = c - j * nx;
        const double Hc = H(c);
        a.H[c] = Hc;
        double ke = 0.0, kn = 0.0;
        // east face (i,j)-(i+1,j): used when row j is interior
        if (i < nx - 1 && j > 0 && j < g.ny - 1) {
            const double gx = (H(c + 1) - Hc) / g.dx;
            const double gy = (H(c + nx + 1) + H(c + nx) - H(c - nx + 1) - H(c - nx)) / (4 * g.dy);
            const bool west_owner = !is_ring(g, i, j);
            // owner's view: neighbour upwind if its H is strictly higher
            const bool up_east = west_owner ? (H(c + 1) > Hc) : !(Hc > H(c + 1));
            ke = olf_face_k(gx, gy, h[c + 1], h[c], m[c + 1], m[c], up_east, a.hmin, a.delta, a.K0);
            // olf_face_k's "neighbour" is the east cell here
        }
        // north face (i,j)-(i,j+1): used when column i is interior
        if (j < g.ny - 1 && i > 0 && i < nx - 1) {
            const double gyy = (H(c + nx) - Hc) / g.dy;
            const double gxx = (H(c + nx + 1) + H(c + 1) - H(c + nx - 1) - H(c - 1)) / (4 * g.dx);
            const bool south_owner = !is_ring(g, i, j);
            const bool up_north = south_owner ? (H(c + nx) > Hc) : !(Hc > H(c + nx));
            kn = olf_face_k(gyy, gxx, h[c + nx], h[c], m[c + nx], m[c], up_north, a.hmin, a.delta, a.K0);
        }
        a.ke[c] = ke;
        a.kn[c] = kn;
    }
}

__global__ __launch_bounds__(kBlock) void k_olf_faces(OlfArgs a)
{
    b_olf_faces(a, hw_blk());
}

// SetUpLinearSystemsOverland (src/overland.cu:65-189) with the ring eliminated, fused with
// r0 = b - A H.
__device__ __forceinline__ void b_olf_assemble(OlfArgs a, Blk bk)
{
    const Geo2 g = a.g;
    const int nx = g.nx;
    const double dtodx2 = -g.cx, dtody2 = -g.cy;
    const double* __restrict__ H = a.H;
    const double* __restrict__ ke = a.ke;
    const double* __restrict__ kn = a.kn;
    double acc[4] = {0.0, 0.0, 0.0, 0.0};   // rz, rr, bb, rr
    if (bk.id == 0 && threadIdx.x == 0) a.st->done = 0;   // a new solve starts
    for (int c = bk.id * blockDim.x + threadIdx.x; c < g.n; c += bk.n * blockDim.x) {
        const int j = c / nx, i = c - j * nx;
        double D, b, r;
        if (is_ring(g, i, j)) {
            D = 1.0;
            b = H[c] + 0.0;
            r = 0.0;
        } else {
            const double kE = ke[c], kW = ke[c - 1], kN = kn[c], kS = kn[c - nx];
            D = 1.0 - dtodx2 * (kE + kW) - dtody2 * (kN + kS);
            b = H[c] + 0.0 + 0.0 + 0.0;
            double Ax = D * H[c];
            // couplings to ring cells move to the right-hand side
            if (i == 1) b -= dtodx2 * kW * H[c - 1]; else Ax += dtodx2 * kW * H[c - 1];
            if (i == nx - 2) b -= dtodx2 * kE * H[c + 1]; else Ax += dtodx2 * kE * H[c + 1];
            if (j == 1) b -= dtody2 * kS * H[c - nx]; else Ax += dtody2 * kS * H[c - nx];
            if (j == g.ny - 2) b -= dtody2 * kN * H[c + nx]; else Ax += dtody2 * kN * H[c + nx];
            r = b - Ax;
        }
        a.D[c] = D;
        a.b[c] = b;
        a.r[c] = r;
        acc[0] += r * (r / D);
        acc[1] += r * r;
        acc[2] += b * b;
        acc[3] += r * r;
    }
    block_partials<4, false>(acc, a.part_out, bk.id);
}

__global__ __launch_bounds__(kBlock) void k_olf_assemble(OlfArgs a)
{
    b_olf_assemble(a, hw_blk());
}

__device__ __forceinline__ void b_pcg2_spmv(Geo2 g, const double* __restrict__ ke, const double* __restrict__ kn,
                                            const double* __restrict__ D, const double* __restrict__ r,
                                            const double* __restrict__ pold, double* __restrict__ pnew,
                                            double* __restrict__ q, SolveCtl sc, Blk bk)
{
    double beta;
    if (!pcg_begin(sc, beta, bk.id)) return;
    const bool first = (sc.it == 0);
    auto pf = [&](int c) -> double {
        const double z = r[c] / D[c];
        return first ? z : z + beta * pold[c];
    };
    double acc[1] = {0.0};
    for (int c = bk.id * blockDim.x + threadIdx.x; c < g.n; c += bk.n * blockDim.x) {
        const double pc = pf(c);
        pnew[c] = pc;
        const double qc = op2_row(g, c, D[c], pc, pf, ke, kn);
        q[c] = qc;
        acc[0] += pc * qc;
    }
    block_partials<1, false>(acc, sc.part_out, bk.id);
}

__global__ __launch_bounds__(kBlock) void k_pcg2_spmv(Geo2 g, const double* __restrict__ ke,
                                                      const double* __restrict__ kn, const double* __restrict__ D,
                                                      const double* __restrict__ r, const double* __restrict__ pold,
                                                      double* __restrict__ pnew, double* __restrict__ q, SolveCtl sc)
{
    b_pcg2_spmv(g, ke, kn, D, r, pold, pnew, q, sc, hw_blk());
}

// ---------------------------------------------------------------------------------------
// The overland Jacobi-PCG of one model by one workgroup (surfaces of at most kOlfBlockCells
// cells): the whole solve in one launch, its reductions inside the block, instead of two
// launches per iteration; the batched form runs one workgroup per model of an ensemble, each to
// its own stopping point.  The iteration and the stopping rule are those of the grid-wide form:
// z = r / D, ||r|| <= tol ||b|| tested before the first and after every iteration, a zero or
// non-finite step ends the solve as a breakdown.  r holds b - A x on entry (k_olf_assemble).
// ---------------------------------------------------------------------------------------

__device__ __forceinline__ void b_olf_cg_block(const OlfCgArgs& a)
{
    __shared__ double lds[3 * 16];
    const Geo2 g = a.g;
    const int n = g.n, tid = threadIdx.x, nt = blockDim.x;
    const double* __restrict__ D = a.D;
    const double* __restrict__ b = a.b;
    double* __restrict__ x = a.x;
    double* __restrict__ r = a.r;
    double* __restrict__ p = a.p;
    double* __restrict__ zq = a.q;   // z = r / D after an update, then q = A p
    double v[3] = {0.0, 0.0, 0.0};   // (r, z), (r, r), (b, b)
    for (int c = tid; c < n; c += nt) {
        const double rc = r[c], zc = rc / D[c];
        p[c] = zc;
        v[0] += rc * zc;
        v[1] += rc * rc;
        v[2] += b[c] * b[c];
    }
    block_sum3(v, lds);
    double rz = v[0], rr = v[1], beta = 0.0;
    const double bb = v[2], tol2 = a.tol * a.tol * bb;
    int it = 0, conv = 0, nan = !isfinite(bb);
    for (;;) {
        nan |= !isfinite(rr);
        conv = (rr <= tol2) ? 1 : 0;
        if (conv || nan || it >= a.maxit) break;
        if (it > 0)
            for (int c = tid; c < n; c += nt) p[c] = zq[c] + beta * p[c];
        __syncthreads();   // p of the neighbours
        double w[3] = {0.0, 0.0, 0.0};
        for (int c = tid; c < n; c += nt) {
            const double pc = p[c];
            const double qc = op2_row(g, c, D[c], pc, [&](int k) { return p[k]; }, a.ke, a.kn);
            zq[c] = qc;
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
            const double rc = r[c] - alpha * zq[c];
            r[c] = rc;
            const double zc = rc / D[c];
            zq[c] = zc;
            u[0] += rc * zc;
            u[1] += rc * rc;
        }
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

__global__ __launch_bounds__(kOlfBlockThreads) void k_olf_cg_block(OlfCgArgs a)
{
    b_olf_cg_block(a);
}

// One workgroup per model (block m solves model m's system; models whose flag is off return).
__global__ __launch_bounds__(kOlfBlockThreads) void kb_olf_cg_block(const OlfCgArgs* __restrict__ args,
                                                                    const int* __restrict__ active)
{
    if (active && !active[blockIdx.x]) return;
    b_olf_cg_block(args[blockIdx.x]);
}

// WaterDepthOverland (src/overland.cu:371-383) and the discharge into the Dirichlet ring.
__device__ __forceinline__ void b_olf_post(OlfArgs a, Blk bk)
{
    const Geo2 g = a.g;
    const int nx = g.nx;
    const double* __restrict__ H = a.H;
    double acc[2] = {0.0, 0.0};   // x = 0 edge, whole ring
    for (int c = bk.id * blockDim.x + threadIdx.x; c < g.n; c += bk.n * blockDim.x) {
        const int j = c / nx, i = c - j * nx;
        if (!is_ring(g, i, j)) {
            const double Hc = H[c];
            if (i == 1) {
                const double q = a.ke[c - 1] * (Hc - H[c - 1]) / g.dx * g.dy;
                acc[0] += q;
                acc[1] += q;
            }
            if (i == nx - 2) acc[1] += a.ke[c] * (Hc - H[c + 1]) / g.dx * g.dy;
            if (j == 1) acc[1] += a.kn[c - nx] * (Hc - H[c - nx]) / g.dy * g.dx;
            if (j == g.ny - 2) acc[1] += a.kn[c] * (Hc - H[c + nx]) / g.dy * g.dx;
        }
        a.h[c] = fmax(H[c] - a.z[c], 0.0);
    }
    block_partials<2, false>(acc, a.part_out, bk.id);
}

__global__ __launch_bounds__(kBlock) void k_olf_post(OlfArgs a)
{
    b_olf_post(a, hw_blk());
}

// ---------------------------------------------------------------------------------------
// Batched launches over an ensemble of models
// ---------------------------------------------------------------------------------------
template <class A, void (*F)(A, Blk)>
__global__ __launch_bounds__(kBlock) void kb_args(const A* __restrict__ args, const BlkMap* __restrict__ map,
                                                  const int* __restrict__ active)
{
    const BlkMap e = map[blockIdx.x];
    if (active && !active[e.m]) return;
    F(args[e.m], Blk{e.id, e.n});
}

// The Anderson pass of every member the host has decided to update (ungated: a.red is null),
// over a map of ceil(nx ny / kAaCols) blocks per member.
template <int M>
__global__ __launch_bounds__(kBlock) void kb_aa_column(const AaArgs* __restrict__ args,
                                                       const BlkMap* __restrict__ map, const int* __restrict__ active)
{
    const BlkMap e = map[blockIdx.x];
    if (active && !active[e.m]) return;
    b_aa_column<M, kAaCols>(args[e.m], e.id);
}

template <bool MIXED>
__device__ __forceinline__ void b_assemble_flux(AsmArgs a, Blk bk) { b_assemble<false, MIXED>(a, bk); }
__device__ __forceinline__ void b_refine_add_args(RefineArgs a, Blk bk) { b_refine_add(a.g.n, a.x, a.d32, bk); }
__device__ __forceinline__ void b_picard_inc_args(VgArgs a, Blk bk)
{
    b_picard_inc(a.psi, a.psi_m, a.g.n, a.rule, a.part_out, bk);
}
__device__ __forceinline__ void b_refine_res_args(RefineArgs a, Blk bk) { b_refine_residual<false>(a, bk); }

template <typename T>
__global__ __launch_bounds__(kBlock) void kb_spmv3(const KrylovArgs<T>* __restrict__ args,
                                                   const BlkMap* __restrict__ map, const int* __restrict__ active,
                                                   const int* __restrict__ it_base, int k)
{
    const BlkMap e = map[blockIdx.x];
    if (!active[e.m]) return;
    const KrylovArgs<T>& a = args[e.m];
    SolveCtl sc = a.spmv;
    sc.it = *it_base + k;
    b_pcg3_spmv<T, false>(a.g, nullptr, a.K, a.D, a.r, a.p[sc.it & 1], a.p[(sc.it + 1) & 1], a.q, sc,
                          Blk{e.id, e.n});
}

template <typename T>
__global__ __launch_bounds__(kBlock) void kb_update3(const KrylovArgs<T>* __restrict__ args,
                                                     const BlkMap* __restrict__ map, const int* __restrict__ active,
                                                     const int* __restrict__ it_base, int k)
{
    const BlkMap e = map[blockIdx.x];
    if (!active[e.m]) return;
    const KrylovArgs<T>& a = args[e.m];
    SolveCtl sc = a.upd;
    sc.it = *it_base + k;
    b_pcg_update<T>(a.g.n, a.x, a.res, a.D, a.p[(sc.it + 1) & 1], a.q, sc, Blk{e.id, e.n});
}

template <typename T>
__global__ __launch_bounds__(kBlock) void kb_spmv_z(const KrylovArgs<T>* __restrict__ args,
                                                    const BlkMap* __restrict__ map, const int* __restrict__ active,
                                                    const int* __restrict__ it_base, int k)
{
    const BlkMap e = map[blockIdx.x];
    if (!active[e.m]) return;
    const KrylovArgs<T>& a = args[e.m];
    SolveCtl sc = a.spmv;
    sc.it = *it_base + k - a.seg0;
    if (sc.it == 0) sc.part_in = a.part_first;
    b_pcg3_spmv<T, false, true>(a.g, nullptr, a.K, a.D, a.z, a.p[sc.it & 1], a.p[(sc.it + 1) & 1], a.q, sc,
                                Blk{e.id, e.n});
}

template <typename T, bool INIT>
__global__ __launch_bounds__(kBlock) void kb_line(const KrylovArgs<T>* __restrict__ args,
                                                  const BlkMap* __restrict__ map, const int* __restrict__ active,
                                                  const int* __restrict__ it_base, int k)
{
    const BlkMap e = map[blockIdx.x];
    if (!active[e.m]) return;
    const KrylovArgs<T>& a = args[e.m];
    SolveCtl sc = INIT ? a.init : a.upd;
    sc.it = INIT ? 0 : *it_base + k - a.seg0;
    b_line<T, INIT>(a.g, a.K, a.D, a.x, a.res, a.p[(sc.it + 1) & 1], a.q, a.z, sc, Blk{e.id, e.n});
}

__global__ __launch_bounds__(kBlock) void kb_spmv2(const KrylovArgs<double>* __restrict__ args,
                                                   const BlkMap* __restrict__ map, const int* __restrict__ active,
                                                   const int* __restrict__ it_base, int k)
{
    const BlkMap e = map[blockIdx.x];
    if (!active[e.m]) return;
    const KrylovArgs<double>& a = args[e.m];
    SolveCtl sc = a.spmv;
    sc.it = *it_base + k;
    b_pcg2_spmv(a.g2, a.ke, a.kn, a.D, a.r, a.p[sc.it & 1], a.p[(sc.it + 1) & 1], a.q, sc,
                       Blk{e.id, e.n});
}

__global__ __launch_bounds__(kBlock) void kb_update2(const KrylovArgs<double>* __restrict__ args,
                                                     const BlkMap* __restrict__ map, const int* __restrict__ active,
                                                     const int* __restrict__ it_base, int k)
{
    const BlkMap e = map[blockIdx.x];
    if (!active[e.m]) return;
    const KrylovArgs<double>& a = args[e.m];
    SolveCtl sc = a.upd;
    sc.it = *it_base + k;
    b_pcg_update<double>(a.g2.n, a.x, a.res, a.D, a.p[(sc.it + 1) & 1], a.q, sc, Blk{e.id, e.n});
}

__global__ __launch_bounds__(kBlock) void k_advance(int* it_base, int by, const int* __restrict__ st, int words,
                                                    int* __restrict__ out)
{
    if (threadIdx.x == 0) *it_base += by;
    for (int i = threadIdx.x; i < words; i += kBlock) out[i] = st[i];
}

// One launch when the set of active models changes, in place of a copy of the flags, a wait for it
// and per map a copy of its segments and a compaction (about 3 us each and the gaps between them).
// Every block reads all flags (a few lines over the bus) and takes the models m = blockIdx.x mod
// gridDim.x; a model's place in a map is the sum of the counts before it.
__global__ __launch_bounds__(kBlock) void k_activate(const int* __restrict__ flags, int M, int* __restrict__ active,
                                                     ActMaps maps)
{
    __shared__ int sum[kBlock];
    int base[4] = {};
    for (int c0 = 0; c0 < M; c0 += kBlock) {
        const int t = threadIdx.x, m = c0 + t, n = min(M - c0, kBlock);
        const int on = m < M ? flags[m] : 0;
        if (blockIdx.x == 0 && m < M) active[m] = on;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (q >= maps.n) break;
            const ActMap& a = maps.m[q];
            const int cnt = on ? a.count[m] : 0;
            int v = cnt;
            __syncthreads();
            sum[t] = v;
            __syncthreads();
            for (int d = 1; d < n; d <<= 1) {   // inclusive sums
                const int w = t >= d ? sum[t - d] : 0;
                __syncthreads();
                sum[t] = v += w;
                __syncthreads();
            }
            for (int j = (int)((blockIdx.x + gridDim.x - c0 % gridDim.x) % gridDim.x); j < n; j += gridDim.x) {
                const int before = j ? sum[j - 1] : 0, len = sum[j] - before, from = len ? a.start[c0 + j] : 0;
                for (int i = t; i < len; i += kBlock) a.cur[base[q] + before + i] = a.full[from + i];
            }
            base[q] += sum[n - 1];
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_reduce_models(const double* const* __restrict__ part,
                                                          const int* __restrict__ nparts, int nv, int take_max,
                                                          double* __restrict__ out)
{
    const int m = blockIdx.x;
    __shared__ double lds[16];
    for (int v = 0; v < nv; ++v) {
        const double* row = part[m] + (size_t)v * kMaxBlocks;
        double acc[1] = {take_max ? -INFINITY : 0.0};
        for (int b = threadIdx.x; b < nparts[m]; b += blockDim.x)
            acc[0] = take_max ? fmax(acc[0], row[b]) : acc[0] + row[b];
        if (take_max) block_reduce<1, true>(acc, lds);
        else block_reduce<1, false>(acc, lds);
        if (threadIdx.x == 0) out[m * nv + v] = acc[0];
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------------------
// One kernel per Jacobi-PCG iteration: the single-reduction recurrences of Chronopoulos &
// Gear (1989).  With u = M^-1 r (M = diag(A)):
//   p_i = u_i + beta_i p_{i-1},  s_i = A p_i,  x_{i+1} = x_i + alpha_i p_i,  r_{i+1} = r_i - alpha_i s_i
//   gamma_{i+1} = (r_{i+1}, u_{i+1}),  delta_{i+1} = (u_{i+1}, A u_{i+1}),
//   eps_{i+1} = (p_i, A u_{i+1}),  pi_i = (p_i, s_i),  rho_{i+1} = (r_{i+1}, r_{i+1})
//   beta_{i+1} = gamma_{i+1} / gamma_i,  alpha_{i+1} = gamma_{i+1} / pi_{i+1},
//   pi_{i+1} = (p_{i+1}, A p_{i+1}) = delta_{i+1} + 2 beta_{i+1} eps_{i+1} + beta_{i+1}^2 pi_i.
// All five sums come out of the same kernel, so one launch is one iteration.  In exact
// arithmetic the iterates are those of the two-kernel (Hestenes-Stiefel) PCG above, so the
// stopping rule ||r|| <= tol ||b|| is met at the same iteration.  (p, Ap) is expanded from
// inner products computed directly rather than from the classic recurrence
// delta - beta gamma / alpha, which stays valid when the residual is replaced (mixed
// precision) and the search direction kept.
//
// A u_{i+1} needs u_{i+1} on the neighbours, which needs s_i there, which needs p_i on the
// neighbours' neighbours: a block owning TX x TY columns computes p_i on the tile plus a
// two-cell halo (LDS), s_i, r_{i+1}, u_{i+1} on the tile plus a one-cell halo, and A u_{i+1} on
// the tile.  Vertically the block marches through its planes k0..k1-1 as a pipeline: in the
// step of plane m it computes p_i of plane m, u_{i+1} of plane m-1 and A u_{i+1} of plane m-2;
// the own column's values stay in registers, the halo's come from LDS rings (p: 3 planes,
// K: 4, u: 2), two barriers per plane.  Cells outside the domain hold p = u = K = 0, which
// removes exactly the couplings the operator does not have.  Without Dirichlet rows only.
// ---------------------------------------------------------------------------------------
// Start of iteration sc.it: sum the five partials of the previous kernel, stop or return
// alpha_i and beta_i.  After a start-up kernel (sc.after_init) the stopping test has been
// made there and pi_{i-1} comes from the state (the partial is not available).
__device__ __forceinline__ bool cg1_begin(const SolveCtl& sc, double& alpha, double& beta, int bid)
{
    PcgState* st = sc.st;
    if (st->done) return false;
    double in[5];
    sum_partials<5>(sc.part_in, sc.nparts, 5, in);
    const double gam = in[0], rr = in[1], del = in[2], eps = in[3], pi_direct = in[4];
    const bool lead = bid == 0 && lin_tid() == 0;
    if (!sc.after_init) {
        const int conv = (rr <= st->tol2) ? 1 : 0;
        const int nan = !isfinite(rr);
        if (conv || nan || sc.it >= sc.maxit) {
            if (lead) {
                st->iter = sc.it;
                st->conv = conv;
                st->rr = rr;
                st->nan = st->nan | nan;
                if (!sc.mixed_inner) st->outer_conv = conv;
                st->done = 1;
            }
            return false;
        }
    }
    double b = 0.0, pi = del;
    if (sc.it > 0) {
        b = gam / st->rz[(sc.it - 1) & 1];
        const double pi_prev = sc.after_init ? st->pi[(sc.it - 1) & 1] : pi_direct;
        pi = del + 2.0 * b * eps + b * b * pi_prev;
    }
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

// Start-up of a solve segment (fresh residual from the assembly or an FP64 reliable update):
// the stopping test of pcg_begin on the four partials [rz, rr, bb, rr64], then
// [gamma, rho, delta, eps, 0] of u = M^-1 r (eps against the kept direction p_{i-1}).
template <typename T>
__device__ __forceinline__ void b_cg1_init(Geo g, const T* __restrict__ K, const T* __restrict__ D,
                                           const T* __restrict__ r, const T* __restrict__ p_old, SolveCtl sc, Blk bk)
{
    double unused;
    if (!pcg_begin(sc, unused, bk.id)) return;
    const bool kept = sc.it > 0;
    auto uf = [&](int c) -> T { return r[c] * jac_inv(D[c]); };
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (int c = bk.id * blockDim.x + threadIdx.x; c < g.n; c += bk.n * blockDim.x) {
        int i, j, k;
        decompose(g, c, i, j, k);
        const T rc = r[c];
        const T uc = uf(c);
        const T au = op3_row<T, false>(g, c, i, j, k, D[c], uc, uf, K, 0u);
        acc[0] += (double)rc * (double)uc;
        acc[1] += (double)rc * (double)rc;
        acc[2] += (double)uc * (double)au;
        if (kept) acc[3] += (double)p_old[c] * (double)au;
    }
    block_partials<5, false>(acc, sc.part_out, bk.id);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_cg1_init(Geo g, const T* __restrict__ K, const T* __restrict__ D,
                                                     const T* __restrict__ r, const T* __restrict__ p_old,
                                                     SolveCtl sc)
{
    b_cg1_init<T>(g, K, D, r, p_old, sc, hw_blk());
}

// Local position (li, lj) of halo cell h of a TX x TY tile: first the one-cell ring (top row,
// bottom row, left column, right column), then the second ring in the same order.
template <int TX, int TY>
__device__ __forceinline__ int2 cg1_halo_pos(int h)
{
    int li, lj;
    constexpr int W1 = TX + 2, W2 = TX + 4, H1 = TY + 2;
    constexpr int NH1 = 2 * W1 + 2 * TY;
    if (h < NH1) {
        if (h < W1) { lj = -1; li = h - 1; }
        else if (h < 2 * W1) { lj = TY; li = h - W1 - 1; }
        else if (h < 2 * W1 + TY) { li = -1; lj = h - 2 * W1; }
        else { li = TX; lj = h - 2 * W1 - TY; }
    } else {
        const int q = h - NH1;
        if (q < W2) { lj = -2; li = q - 2; }
        else if (q < 2 * W2) { lj = TY + 1; li = q - W2 - 2; }
        else if (q < 2 * W2 + H1) { li = -2; lj = q - 2 * W2 - 1; }
        else { li = TX + 1; lj = q - 2 * W2 - H1 - 1; }
    }
    return make_int2(li, lj);
}


// Global values of one plane for one thread: its own cell and its (up to two) halo cells.
template <typename T>
struct Cg1Plane {
    T r, d, p, k, x;
    T hr0, hd0, hp0, hk0;
    T hr1, hd1, hp1, hk1;
};

// The iteration kernel.  Blocks loop over tiles t = blockIdx.x, blockIdx.x + gridDim.x, ...
// (gridDim.x a multiple of 8, so every tile of a block runs on the block's XCD and xcd_tile
// keeps an XCD's tiles contiguous).  The stencil is evaluated in factored form: with
// h = w / 2 per direction and q = K p,
//   (A p)_c = D_c p_c - sum over directions h (K_c (p_nb1 + p_nb2) + (q_nb1 + q_nb2)),
// which equals the arithmetic-mean face form; p and q (and u, K u for A u) are staged in LDS, so
// a direction costs four operations.  The plane loop is unrolled six times, so the LDS ring
// slots are compile-time constants and the register pipeline shifts are renames.
template <typename T, int TX, int TY>
__device__ __forceinline__ void b_cg1(Geo g, const T* __restrict__ K, const T* __restrict__ D,
                                      const T* __restrict__ r_in, T* __restrict__ r_out,
                                      const T* __restrict__ p_in, T* __restrict__ p_out, T* __restrict__ x,
                                      SolveCtl sc, int kc, int ntx, int nty, int nkz, Blk bk)
{
    constexpr int NT = TX * TY;
    constexpr int W2 = TX + 4, A2 = W2 * (TY + 4);
    constexpr int W1 = TX + 2, A1 = W1 * (TY + 2);
    constexpr int NH1 = A1 - NT, NH2 = A2 - NT;
    static_assert(NH1 <= NT && NH2 <= 2 * NT, "tile too small for its halo");
    double alpha_d, beta_d;
    if (!cg1_begin(sc, alpha_d, beta_d, bk.id)) return;
    const bool first = sc.it == 0;
    const T alpha = (T)alpha_d, beta = (T)beta_d;
    const T hx = (T)(0.5 * g.wx), hy = (T)(0.5 * g.wy), hz = (T)(0.5 * g.wz);

    __shared__ T sp[3][A2], sq[3][A2];     // p, K p of planes m, m-1, m-2
    __shared__ T su[2][A1], squ[2][A1];    // u, K u of planes m-1, m-2

    const int lid = threadIdx.x;
    const int tx = lid % TX, ty = lid / TX;
    const int oq2 = (ty + 2) * W2 + tx + 2;
    const int oq1 = (ty + 1) * W1 + tx + 1;
    // halo slots of this thread: h = lid (if < NH2) and h = lid + NT (if < NH2); for lid < NH1
    // slot 0 is a cell of the one-cell ring, whose s, r, u this thread also computes
    const int2 hp0 = lid < NH2 ? cg1_halo_pos<TX, TY>(lid) : make_int2(0, 0);
    const int2 hp1 = lid + NT < NH2 ? cg1_halo_pos<TX, TY>(lid + NT) : make_int2(0, 0);
    const bool has_h0 = lid < NH2, has_h1 = lid + NT < NH2, ring = lid < NH1;
    const int hq2_0 = (hp0.y + 2) * W2 + hp0.x + 2, hq2_1 = (hp1.y + 2) * W2 + hp1.x + 2;
    const int rq1 = (hp0.y + 1) * W1 + hp0.x + 1;
    // lowest neighbour index of a stencil read (the j-1 neighbour), so that every LDS read of
    // a stencil is a non-negative constant offset from one register
    const unsigned obase = (unsigned)(oq2 - W2), ubase = (unsigned)(oq1 - W1);
    const unsigned rbase = has_h0 && lid < NH1 ? (unsigned)(hq2_0 - W2) : 0u;
    constexpr unsigned ES = sizeof(T);
    const unsigned plane_bytes = (unsigned)g.nxy * ES;

    const int nb = ntx * nty * nkz;
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};   // gamma, rho, delta, eps, pi
    for (int tw = bk.id; tw < nb; tw += bk.n) {
        const int t = xcd_tile(tw, nb);
        const int bz = t % nkz, bxy = t / nkz;
        const int i0 = (bxy % ntx) * TX, j0 = (bxy / ntx) * TY;
        const int k0 = bz * kc, k1 = min(k0 + kc, g.nz);
        const int oi = i0 + tx, oj = j0 + ty;
        const bool own_in = oi < g.nx && oj < g.ny;
        const int h0i = i0 + hp0.x, h0j = j0 + hp0.y, h1i = i0 + hp1.x, h1j = j0 + hp1.y;
        const bool h0_in = has_h0 && h0i >= 0 && h0j >= 0 && h0i < g.nx && h0j < g.ny;
        const bool h1_in = has_h1 && h1i >= 0 && h1j >= 0 && h1i < g.nx && h1j < g.ny;
        const unsigned obyte = (unsigned)(oj * g.nx + oi) * ES;
        const unsigned h0byte = (unsigned)(h0j * g.nx + h0i) * ES, h1byte = (unsigned)(h1j * g.nx + h1i) * ES;

        // loads of plane m, one plane ahead of their use: only lanes whose cell is in the domain
        // load, the others keep the zeros (D = 1) of zero_plane(); planes outside the domain are
        // all zeros.  Lanes without a cell compute garbage where a neighbour is not zero, which
        // is masked before it reaches LDS, memory or a sum.
        Cg1Plane<T> L;
        auto zero_plane = [&]() {
            L.r = 0; L.d = 1; L.k = 0; L.x = 0; L.p = 0;
            L.hr0 = 0; L.hd0 = 1; L.hk0 = 0; L.hp0 = 0;
            L.hr1 = 0; L.hd1 = 1; L.hk1 = 0; L.hp1 = 0;
        };
        auto load_plane = [&](int m) {   // 0 <= m < nz
            const unsigned off = (unsigned)m * plane_bytes;
            if (own_in) {
                const unsigned c = off + obyte;
                L.r = ld_off(r_in, c); L.d = ld_off(D, c); L.k = ld_off(K, c); L.x = ld_off((const T*)x, c);
                if (!first) L.p = ld_off(p_in, c);
            }
            if (h0_in) {
                const unsigned c = off + h0byte;
                L.hr0 = ld_off(r_in, c); L.hd0 = ld_off(D, c); L.hk0 = ld_off(K, c);
                if (!first) L.hp0 = ld_off(p_in, c);
            }
            if (h1_in) {
                const unsigned c = off + h1byte;
                L.hr1 = ld_off(r_in, c); L.hd1 = ld_off(D, c); L.hk1 = ld_off(K, c);
                if (!first) L.hp1 = ld_off(p_in, c);
            }
        };

        // own column pipeline (plane of each register relative to the step m)
        T P1 = 0, P2 = 0, Q1 = 0, Q2 = 0;   // p, K p of planes m-1, m-2
        T K1 = 0, K2 = 0;                   // K(m-1), K(m-2)
        T D1 = 1, D2 = 1, DI1 = 1;          // D(m-1), D(m-2), jac_inv(D(m-1))
        T R1 = 0, X1 = 0;                   // r(m-1), x(m-1)
        T U2 = 0, U3 = 0, QU2 = 0, QU3 = 0; // u, K u of planes m-2, m-3
        T RR1 = 0, RD1 = 1, RDI1 = 1, RK1 = 0;   // ring cell: r, D, jac_inv(D), K of plane m-1

        // step J (mod 6) of plane m.  The LDS ring slots are compile-time constants: sp/sq hold
        // planes m, m-1, m-2 in slots a0, a1, a2, su/squ planes m-1, m-2 in b0, b1.  (A second,
        // check-free copy of the steps for the steady range measured slower: it raises the
        // register count and lowers the occupancy more than it saves.)
        auto step = [&](auto J, int m) {
            constexpr int j = decltype(J)::value;
            constexpr int a0 = (3 - j % 3) % 3, a1 = (4 - j % 3) % 3, a2 = (5 - j % 3) % 3;
            constexpr int b0 = j % 2, b1 = 1 - j % 2;
            // phase 1: p_i, K p_i of plane m on the tile + two-cell halo
            const T DI0 = jac_inv(L.d);
            const T P0 = L.r * DI0 + (first ? T(0) : beta * L.p);
            const T K0 = L.k, Q0 = L.k * P0, D0 = L.d, R0 = L.r, X0 = L.x;
            sp[a0][oq2] = P0;
            sq[a0][oq2] = Q0;
            const T RR0 = L.hr0, RD0 = L.hd0, RK0 = L.hk0;
            const T RDI0 = jac_inv(L.hd0);
            if (has_h0) {
                const T ph = L.hr0 * RDI0 + (first ? T(0) : beta * L.hp0);
                sp[a0][hq2_0] = ph;
                sq[a0][hq2_0] = L.hk0 * ph;
            }
            if (has_h1) {
                const T ph = L.hr1 * jac_inv(L.hd1) + (first ? T(0) : beta * L.hp1);
                sp[a0][hq2_1] = ph;
                sq[a0][hq2_1] = L.hk1 * ph;
            }
            if (m + 1 <= k1 + 1) {
                if (m + 1 >= 0 && m + 1 < g.nz) load_plane(m + 1);
                else zero_plane();
            }
            __syncthreads();
            // phase 3: s_i, r_{i+1}, u_{i+1} of plane m-1 on the tile + one-cell halo
            const int pm = m - 1;
            T U1 = 0, QU1 = 0;
            if (pm >= k0 - 1) {
                const bool pv = pm >= 0 && pm < g.nz;
                if (pv) {
                    const T* pc = &sp[a1][obase];   // obase = oq2 - W2: neighbours at 0, W2-1, W2+1, 2 W2
                    const T* qc = &sq[a1][obase];
                    const T tx_ = fma(K1, pc[W2 - 1] + pc[W2 + 1], qc[W2 - 1] + qc[W2 + 1]);
                    const T ty_ = fma(K1, pc[0] + pc[2 * W2], qc[0] + qc[2 * W2]);
                    const T tz_ = fma(K1, P2 + P0, Q2 + Q0);
                    T sv = D1 * P1;
                    sv = fma(-hx, tx_, sv);
                    sv = fma(-hy, ty_, sv);
                    sv = fma(-hz, tz_, sv);
                    const T rn = own_in ? fma(-alpha, sv, R1) : T(0);
                    U1 = rn * DI1;
                    QU1 = K1 * U1;
                    if (pm >= k0 && pm < k1) {
                        if (own_in) {
                            const unsigned c = (unsigned)pm * plane_bytes + obyte;
                            st_off<T>(r_out, c, rn);
                            st_off<T>(p_out, c, P1);
                            st_off<T>(x, c, fma(alpha, P1, X1));
                        }
                        acc[0] += (double)rn * (double)U1;
                        acc[1] += (double)rn * (double)rn;
                        acc[4] += (double)P1 * (double)sv;
                    }
                }
                su[b0][oq1] = U1;
                squ[b0][oq1] = QU1;
                if (ring) {
                    T ur = 0, qur = 0;
                    if (pv) {
                        const T* pc = &sp[a1][rbase];   // rbase = hq2_0 - W2
                        const T* qc = &sq[a1][rbase];
                        const T tx_ = fma(RK1, pc[W2 - 1] + pc[W2 + 1], qc[W2 - 1] + qc[W2 + 1]);
                        const T ty_ = fma(RK1, pc[0] + pc[2 * W2], qc[0] + qc[2 * W2]);
                        const T tz_ = fma(RK1, sp[a2][hq2_0] + sp[a0][hq2_0], sq[a2][hq2_0] + sq[a0][hq2_0]);
                        T sv = RD1 * pc[W2];
                        sv = fma(-hx, tx_, sv);
                        sv = fma(-hy, ty_, sv);
                        sv = fma(-hz, tz_, sv);
                        ur = h0_in ? fma(-alpha, sv, RR1) * RDI1 : T(0);
                        qur = RK1 * ur;
                    }
                    su[b0][rq1] = ur;
                    squ[b0][rq1] = qur;
                }
            }
            __syncthreads();
            // phase 5: A u_{i+1} of plane m-2 on the tile (lanes without a cell have U2 = P2 = 0)
            const int pm2 = m - 2;
            if (pm2 >= k0 && pm2 < k1) {
                const T* uc = &su[b1][ubase];   // ubase = oq1 - W1
                const T* quc = &squ[b1][ubase];
                const T tx_ = fma(K2, uc[W1 - 1] + uc[W1 + 1], quc[W1 - 1] + quc[W1 + 1]);
                const T ty_ = fma(K2, uc[0] + uc[2 * W1], quc[0] + quc[2 * W1]);
                const T tz_ = fma(K2, U3 + U1, QU3 + QU1);
                T au = D2 * U2;
                au = fma(-hx, tx_, au);
                au = fma(-hy, ty_, au);
                au = fma(-hz, tz_, au);
                acc[2] += (double)U2 * (double)au;
                acc[3] += (double)P2 * (double)au;
            }
            // shift the pipeline
            P2 = P1; P1 = P0; Q2 = Q1; Q1 = Q0;
            K2 = K1; K1 = K0;
            D2 = D1; D1 = D0; DI1 = DI0;
            R1 = R0; X1 = X0;
            U3 = U2; U2 = U1; QU3 = QU2; QU2 = QU1;
            RR1 = RR0; RD1 = RD0; RDI1 = RDI0; RK1 = RK0;
        };

        zero_plane();
        if (k0 - 2 >= 0) load_plane(k0 - 2);
        const int mend = k1 + 1;
        for (int m = k0 - 2; m <= mend; m += 6) {
            step(std::integral_constant<int, 0>{}, m);
            if (m + 1 > mend) break;
            step(std::integral_constant<int, 1>{}, m + 1);
            if (m + 2 > mend) break;
            step(std::integral_constant<int, 2>{}, m + 2);
            if (m + 3 > mend) break;
            step(std::integral_constant<int, 3>{}, m + 3);
            if (m + 4 > mend) break;
            step(std::integral_constant<int, 4>{}, m + 4);
            if (m + 5 > mend) break;
            step(std::integral_constant<int, 5>{}, m + 5);
        }
        __syncthreads();   // the LDS rings are reused by the next tile
    }
    block_partials<5, false>(acc, sc.part_out, bk.id);
}

template <typename T, int TX, int TY>
__global__ __launch_bounds__(TX * TY) void k_cg1(Geo g, const T* __restrict__ K, const T* __restrict__ D,
                                                 const T* __restrict__ r_in, T* __restrict__ r_out,
                                                 const T* __restrict__ p_in, T* __restrict__ p_out,
                                                 T* __restrict__ x, SolveCtl sc, int kc, int ntx, int nty, int nkz)
{
    b_cg1<T, TX, TY>(g, K, D, r_in, r_out, p_in, p_out, x, sc, kc, ntx, nty, nkz, Blk{(int)blockIdx.x, (int)gridDim.x});
}

template <typename T>
__global__ __launch_bounds__(kBlock) void kb_cg1_init(const Cg1Args<T>* __restrict__ args,
                                                      const BlkMap* __restrict__ map, const int* __restrict__ active)
{
    const BlkMap e = map[blockIdx.x];
    if (!active[e.m]) return;
    const Cg1Args<T>& a = args[e.m];
    SolveCtl sc = a.ctl;
    sc.it = 0;
    sc.segment_start = 0;
    sc.part_in = a.part_asm;
    sc.nparts = a.nparts_asm;
    sc.part_out = a.part[1];
    b_cg1_init<T>(a.g, a.K, a.D, a.r[0], a.p[1], sc, Blk{e.id, e.n});
}

template <typename T>
__global__ __launch_bounds__(kBlock) void kb_cg1(const Cg1Args<T>* __restrict__ args, const BlkMap* __restrict__ map,
                                                 const int* __restrict__ active, const int* __restrict__ it_base, int k)
{
    static_assert(kCg1BatchTx * kCg1BatchTy == kBlock, "batched tile = one block of kBlock threads");
    const BlkMap e = map[blockIdx.x];
    if (!active[e.m]) return;
    const Cg1Args<T>& a = args[e.m];
    SolveCtl sc = a.ctl;
    const int it = *it_base + k;
    sc.it = it;
    sc.after_init = it == 0 ? 1 : 0;
    sc.part_in = a.part[(it + 1) & 1];
    sc.nparts = it == 0 ? a.nparts_asm : a.ntiles;
    sc.part_out = a.part[it & 1];
    b_cg1<T, kCg1BatchTx, kCg1BatchTy>(a.g, a.K, a.D, a.r[it & 1], a.r[(it + 1) & 1], a.p[(it + 1) & 1], a.p[it & 1],
                                       a.x, sc, a.kc, a.ntx, a.nty, a.nkz, Blk{e.id, e.n});
}

}  // namespace

// =========================================================================================
// Launchers
// =========================================================================================
// Krylov launches: through hipExtLaunchKernelGGL so that profiling events, when given, carry
// the kernel's own begin/end timestamps.
template <typename F, typename... Args>
static void launch_ev(F kernel, dim3 gr, dim3 bl, hipStream_t s, const LaunchEv& ev, Args... args)
{
    hipExtLaunchKernelGGL(kernel, gr, bl, 0, s, ev.start, ev.stop, 0, args...);
}

void launch_vg(hipStream_t s, const VgArgs& a)
{
    hipLaunchKernelGGL(k_vg, dim3(grid_for(a.g.n)), dim3(kBlock), 0, s, a);
}

void launch_init_state(hipStream_t s, const InitArgs& a, bool from_theta)
{
    const dim3 gr(grid_for(a.g.n)), bl(kBlock);
    if (from_theta) hipLaunchKernelGGL(k_init_state<true>, gr, bl, 0, s, a);
    else hipLaunchKernelGGL(k_init_state<false>, gr, bl, 0, s, a);
}

void launch_vg_picard(hipStream_t s, const VgArgs& a, const Gate& gate)
{
    hipLaunchKernelGGL(k_vg_picard, dim3(grid_for(a.g.n)), dim3(kBlock), 0, s, a, gate);
}

// Fewer columns than one block of 64 per CU leave CUs idle: blocks of 16 there.  Where the blocks of 64
// fill the chip, bytes bound the pass and 16 columns would only shorten the rows of a load to 128 B.
template <int M>
static void picard_next(hipStream_t s, const NextArgs& a, const LaunchEv* ev)
{
    const LaunchEv e = ev ? *ev : LaunchEv{};
    const int n = a.aa.g.nxy;
    if (n < 256 * kAaCols)
        launch_ev(k_picard_next<M, kAaColsSmall>, dim3((n + kAaColsSmall - 1) / kAaColsSmall), dim3(kBlock), s, e, a);
    else
        launch_ev(k_picard_next<M, kAaCols>, dim3(aa_blocks(a.aa.g)), dim3(kBlock), s, e, a);
}

void launch_picard_next(hipStream_t s, const NextArgs& a, int depth, const LaunchEv* ev)
{
    switch (depth) {
    case 1: picard_next<1>(s, a, ev); break;
    case 2: picard_next<2>(s, a, ev); break;
    case 3: picard_next<3>(s, a, ev); break;
    case 4: picard_next<4>(s, a, ev); break;
    default: picard_next<kAaMaxDepth>(s, a, ev); break;
    }
}

void launch_picard_inc(hipStream_t s, const VgArgs& a, const Gate& gate)
{
    hipLaunchKernelGGL(k_picard_inc, dim3(grid_for(a.g.n)), dim3(kBlock), 0, s, a.psi, a.psi_m, a.g.n, a.rule, a.part_out,
                       gate);
}

void launch_refine_conv(hipStream_t s, const double* part, int nparts, double lin_tol, PcgState* st)
{
    hipLaunchKernelGGL(k_refine_conv, dim3(1), dim3(kBlock), 0, s, part, nparts, lin_tol, st);
}

void launch_picard_report(hipStream_t s, const double* part, int nparts, const Gate& gate, HostReport* rep)
{
    hipLaunchKernelGGL(k_picard_report, dim3(1), dim3(kBlock), 0, s, part, nparts, gate, rep);
}

void launch_report(hipStream_t s, const PcgState* st, HostReport* rep)
{
    hipLaunchKernelGGL(k_report, dim3(1), dim3(kWave), 0, s, st, rep);
}

void launch_report_sums(hipStream_t s, const double* part, int nparts, int nv, HostReport* rep)
{
    hipLaunchKernelGGL(k_report_sums, dim3(1), dim3(nv * kWave), 0, s, part, nparts, nv, rep);
}

void launch_vg_inverse(hipStream_t s, const Geo& g, const Soil& soil, const double* theta, double* psi)
{
    hipLaunchKernelGGL(k_vg_inverse, dim3(grid_for(g.n)), dim3(kBlock), 0, s, g, soil, theta, psi);
}

void launch_row_flags(hipStream_t s, const Geo& g, const int* const bctype[6], uint8_t* flags)
{
    BcTypes bt;
    for (int f = 0; f < 6; ++f) bt.t[f] = bctype[f];
    hipLaunchKernelGGL(k_row_flags, dim3(grid_for(g.n)), dim3(kBlock), 0, s, g, bt, flags);
}

void launch_group_scatter(hipStream_t s, int nxy, const int* procmap, const double* groups, double* out)
{
    hipLaunchKernelGGL(k_group_scatter, dim3(grid_for(nxy)), dim3(kBlock), 0, s, nxy, procmap, groups, out);
}

void launch_surface_pre(hipStream_t s, const SurfArgs& a)
{
    hipLaunchKernelGGL(k_surface_pre, dim3(grid_for(a.nxy)), dim3(kBlock), 0, s, a);
}

void launch_surface_post(hipStream_t s, const SurfArgs& a)
{
    hipLaunchKernelGGL(k_surface_post, dim3(grid_for(a.nxy)), dim3(kBlock), 0, s, a);
}

void launch_assemble(hipStream_t s, const AsmArgs& a, bool mixed)
{
    const dim3 gr(grid_for(a.g.n)), bl(kBlock);
    const bool dir = a.flags != nullptr;
    if (dir) {
        if (mixed) hipLaunchKernelGGL((k_assemble<true, true>), gr, bl, 0, s, a);
        else hipLaunchKernelGGL((k_assemble<true, false>), gr, bl, 0, s, a);
    } else {
        if (mixed) hipLaunchKernelGGL((k_assemble<false, true>), gr, bl, 0, s, a);
        else hipLaunchKernelGGL((k_assemble<false, false>), gr, bl, 0, s, a);
    }
}

template <bool MIXED, int TX, int TY>
static void assemble_tiled(hipStream_t s, const AsmArgs& a, int kc)
{
    const int ntx = (a.g.nx + TX - 1) / TX, nty = (a.g.ny + TY - 1) / TY, nkz = (a.g.nz + kc - 1) / kc;
    hipLaunchKernelGGL((k_assemble_tiled<MIXED, TX, TY>), dim3(ntx * nty * nkz), dim3(TX, TY), 0, s, a, kc, ntx,
                       nty, nkz);
}

template <bool MIXED>
static void assemble_tiled_dispatch(hipStream_t s, const AsmArgs& a, const TileCfg& t)
{
    if (t.tx == 32 && t.ty == 8) assemble_tiled<MIXED, 32, 8>(s, a, t.kc);
    else if (t.tx == 64 && t.ty == 4) assemble_tiled<MIXED, 64, 4>(s, a, t.kc);
    else if (t.tx == 16 && t.ty == 16) assemble_tiled<MIXED, 16, 16>(s, a, t.kc);
    else if (t.tx == 32 && t.ty == 4) assemble_tiled<MIXED, 32, 4>(s, a, t.kc);
    else assemble_tiled<MIXED, 64, 8>(s, a, t.kc);
}

int launch_assemble_tiled(hipStream_t s, const AsmArgs& a, bool mixed, const TileCfg& t)
{
    if (a.flags || !t.tx) {
        launch_assemble(s, a, mixed);
        return grid_for(a.g.n);
    }
    if (mixed) assemble_tiled_dispatch<true>(s, a, t);
    else assemble_tiled_dispatch<false>(s, a, t);
    return tile_blocks(a.g, t);
}

void launch_refine(hipStream_t s, const RefineArgs& a)
{
    const dim3 gr(grid_for(a.g.n)), bl(kBlock);
    hipLaunchKernelGGL(k_refine_add, gr, bl, 0, s, a.g.n, a.x, (const float*)a.d32);
    if (a.flags) hipLaunchKernelGGL((k_refine_residual<true>), gr, bl, 0, s, a);
    else hipLaunchKernelGGL((k_refine_residual<false>), gr, bl, 0, s, a);
}

template <int TX, int TY>
static void refine_tiled(hipStream_t s, const RefineArgs& a, int kc)
{
    const int ntx = (a.g.nx + TX - 1) / TX, nty = (a.g.ny + TY - 1) / TY, nkz = (a.g.nz + kc - 1) / kc;
    hipLaunchKernelGGL((k_refine_residual_tiled<TX, TY>), dim3(ntx * nty * nkz), dim3(TX, TY), 0, s, a, kc, ntx,
                       nty, nkz);
}

template <bool FULL>
static void refine_line_dispatch(hipStream_t s, const RefineArgs& a, float* z32, int ntx, int nty)
{
    constexpr int TX = 32, TY = 8;
    const dim3 gr(ntx * nty), bl(TX, TY);
    if (a.g.nz <= 16) hipLaunchKernelGGL((k_refine_line<16, TX, TY, FULL>), gr, bl, 0, s, a, z32, ntx, nty);
    else if (a.g.nz <= 32) hipLaunchKernelGGL((k_refine_line<32, TX, TY, FULL>), gr, bl, 0, s, a, z32, ntx, nty);
    else hipLaunchKernelGGL((k_refine_line<64, TX, TY, FULL>), gr, bl, 0, s, a, z32, ntx, nty);
}

int launch_refine_line(hipStream_t s, const RefineArgs& a, float* z32, RefineLineMode mode)
{
    constexpr int TX = 32, TY = 8;
    const int ntx = (a.g.nx + TX - 1) / TX, nty = (a.g.ny + TY - 1) / TY;
    if (ntx * nty > kMaxBlocks || a.g.nz > kLineMaxNz) return 0;
    if (mode == kRefineCheck) {
        hipLaunchKernelGGL(k_refine_gate, dim3(1), dim3(kWave), 0, s, a.st);
        hipLaunchKernelGGL(k_refine_add_gated, dim3(grid_for(a.g.n)), dim3(kBlock), 0, s, a.g.n, a.x,
                           (const float*)a.d32, (const PcgState*)a.st);
        refine_line_dispatch<false>(s, a, z32, ntx, nty);
    } else {
        if (mode == kRefineFull)
            hipLaunchKernelGGL(k_refine_add, dim3(grid_for(a.g.n)), dim3(kBlock), 0, s, a.g.n, a.x,
                               (const float*)a.d32);
        refine_line_dispatch<true>(s, a, z32, ntx, nty);
    }
    return ntx * nty;
}

int launch_refine_tiled(hipStream_t s, const RefineArgs& a, const TileCfg& t)
{
    if (a.flags || !t.tx) {
        launch_refine(s, a);
        return grid_for(a.g.n);
    }
    hipLaunchKernelGGL(k_refine_add, dim3(grid_for(a.g.n)), dim3(kBlock), 0, s, a.g.n, a.x, (const float*)a.d32);
    if (t.tx == 32 && t.ty == 8) refine_tiled<32, 8>(s, a, t.kc);
    else if (t.tx == 64 && t.ty == 4) refine_tiled<64, 4>(s, a, t.kc);
    else if (t.tx == 16 && t.ty == 16) refine_tiled<16, 16>(s, a, t.kc);
    else if (t.tx == 32 && t.ty == 4) refine_tiled<32, 4>(s, a, t.kc);
    else refine_tiled<64, 8>(s, a, t.kc);
    return tile_blocks(a.g, t);
}

void launch_end_step(hipStream_t s, const EndArgs& a)
{
    hipLaunchKernelGGL(k_end_step, dim3(grid_for(a.g.n)), dim3(kBlock), 0, s, a);
}

template <typename T>
static void pcg3_spmv(hipStream_t s, const Geo& g, const uint8_t* flags, const T* K, const T* D,
                      const T* r, T* const p[2], T* q, const SolveCtl& sc, const LaunchEv& ev)
{
    const dim3 gr(grid_for(g.n)), bl(kBlock);
    const T* pold = p[sc.it & 1];
    T* pnew = p[(sc.it + 1) & 1];
    if (flags) launch_ev(k_pcg3_spmv<T, true>, gr, bl, s, ev, g, flags, K, D, r, pold, pnew, q, sc);
    else launch_ev(k_pcg3_spmv<T, false>, gr, bl, s, ev, g, flags, K, D, r, pold, pnew, q, sc);
}

template <typename T>
static void pcg_update(hipStream_t s, int n, T* x, T* r, const T* D, const T* p, const T* q,
                       const SolveCtl& sc, const LaunchEv& ev)
{
    launch_ev(k_pcg_update<T>, dim3(grid_for(n)), dim3(kBlock), s, ev, n, x, r, D, p, q, sc);
}

void launch_pcg3_spmv_f64(hipStream_t s, const Geo& g, const uint8_t* flags, const double* K,
                          const double* D, const double* r, double* const p[2], double* q,
                          const SolveCtl& sc, const LaunchEv& ev)
{
    pcg3_spmv<double>(s, g, flags, K, D, r, p, q, sc, ev);
}

void launch_pcg3_spmv_f32(hipStream_t s, const Geo& g, const uint8_t* flags, const float* K,
                          const float* D, const float* r, float* const p[2], float* q,
                          const SolveCtl& sc, const LaunchEv& ev)
{
    pcg3_spmv<float>(s, g, flags, K, D, r, p, q, sc, ev);
}

void launch_pcg_update_f64(hipStream_t s, int n, double* x, double* r, const double* D,
                           const double* p, const double* q, const SolveCtl& sc, const LaunchEv& ev)
{
    pcg_update<double>(s, n, x, r, D, p, q, sc, ev);
}

void launch_pcg_update_f32(hipStream_t s, int n, float* x, float* r, const float* D,
                           const float* p, const float* q, const SolveCtl& sc, const LaunchEv& ev)
{
    pcg_update<float>(s, n, x, r, D, p, q, sc, ev);
}

bool tile_supported(const TileCfg& t)
{
    return t.kc >= 1 && ((t.tx == 32 && t.ty == 8) || (t.tx == 64 && t.ty == 4) || (t.tx == 16 && t.ty == 16) ||
                         (t.tx == 32 && t.ty == 4) || (t.tx == 64 && t.ty == 8));
}

int tile_blocks(const Geo& g, const TileCfg& t)
{
    const int ntx = (g.nx + t.tx - 1) / t.tx, nty = (g.ny + t.ty - 1) / t.ty;
    const int nkz = (g.nz + t.kc - 1) / t.kc;
    return ntx * nty * nkz;
}

template <typename T, int TX, int TY, bool ZIN = false>
static void tiled_launch(hipStream_t s, const Geo& g, int kc, const uint8_t* flags, const T* K, const T* D,
                         const T* r, const T* pold, T* pnew, T* q, const SolveCtl& sc, const LaunchEv& ev)
{
    const int ntx = (g.nx + TX - 1) / TX, nty = (g.ny + TY - 1) / TY, nkz = (g.nz + kc - 1) / kc;
    const dim3 gr(ntx * nty * nkz), bl(TX, TY);
    if constexpr (ZIN)
        launch_ev(k_spmv_z<T, TX, TY>, gr, bl, s, ev, g, K, D, r, pold, pnew, q, sc, kc, ntx, nty, nkz);
    else if (flags)
        launch_ev(k_pcg3_spmv_tiled<T, true, TX, TY>, gr, bl, s, ev, g, flags, K, D, r, pold, pnew, q, sc, kc,
                  ntx, nty, nkz);
    else
        launch_ev(k_pcg3_spmv_tiled<T, false, TX, TY>, gr, bl, s, ev, g, flags, K, D, r, pold, pnew, q, sc, kc,
                  ntx, nty, nkz);
}

template <typename T, bool ZIN = false>
static void tiled_dispatch(hipStream_t s, const Geo& g, const TileCfg& t, const uint8_t* flags, const T* K,
                           const T* D, const T* r, T* const p[2], T* q, const SolveCtl& sc, const LaunchEv& ev)
{
    const T* pold = p[sc.it & 1];
    T* pnew = p[(sc.it + 1) & 1];
    if (t.tx == 32 && t.ty == 8) tiled_launch<T, 32, 8, ZIN>(s, g, t.kc, flags, K, D, r, pold, pnew, q, sc, ev);
    else if (t.tx == 64 && t.ty == 4) tiled_launch<T, 64, 4, ZIN>(s, g, t.kc, flags, K, D, r, pold, pnew, q, sc, ev);
    else if (t.tx == 16 && t.ty == 16) tiled_launch<T, 16, 16, ZIN>(s, g, t.kc, flags, K, D, r, pold, pnew, q, sc, ev);
    else if (t.tx == 32 && t.ty == 4) tiled_launch<T, 32, 4, ZIN>(s, g, t.kc, flags, K, D, r, pold, pnew, q, sc, ev);
    else tiled_launch<T, 64, 8, ZIN>(s, g, t.kc, flags, K, D, r, pold, pnew, q, sc, ev);
}

// SpMV kernel of the column-preconditioned PCG: p = z + beta p, q = A p, (p, q); tiled on t, or
// untiled when t.tx = 0.  No Dirichlet rows.
template <typename T>
static void spmv_z(hipStream_t s, const Geo& g, const TileCfg& t, const T* K, const T* D, const T* z, T* const p[2],
                   T* q, const SolveCtl& sc, const LaunchEv& ev)
{
    if (t.tx) {
        tiled_dispatch<T, true>(s, g, t, nullptr, K, D, z, p, q, sc, ev);
    } else {
        launch_ev(k_pcg3_spmv<T, false, true>, dim3(grid_for(g.n)), dim3(kBlock), s, ev, g, (const uint8_t*)nullptr,
                  K, D, z, (const T*)p[sc.it & 1], p[(sc.it + 1) & 1], q, sc);
    }
}

void launch_pcg3_spmv_z_f64(hipStream_t s, const Geo& g, const TileCfg& t, const double* K, const double* D,
                            const double* z, double* const p[2], double* q, const SolveCtl& sc, const LaunchEv& ev)
{
    spmv_z<double>(s, g, t, K, D, z, p, q, sc, ev);
}

void launch_pcg3_spmv_z_f32(hipStream_t s, const Geo& g, const TileCfg& t, const float* K, const float* D,
                            const float* z, float* const p[2], float* q, const SolveCtl& sc, const LaunchEv& ev)
{
    spmv_z<float>(s, g, t, K, D, z, p, q, sc, ev);
}

bool line_supported(const Geo& g) { return g.nz >= 1 && g.nz <= kLineMaxNz; }

// y (FP64) or y and c' (FP32) of a block's columns: 128 KB of the CU's 160 KB at kLineMaxNz planes.
static size_t line_lds_bytes(int nz) { return (size_t)nz * kBlock * 8; }

int line_blocks(const Geo& g) { return std::min((g.nxy + kBlock - 1) / kBlock, kMaxBlocks / 2); }

template <typename T, bool INIT>
static void line_launch(hipStream_t s, const Geo& g, const T* K, const T* D, T* x, T* r, const T* p, const T* q,
                        T* z, const SolveCtl& sc, const LaunchEv& ev)
{
    const dim3 gr(line_blocks(g)), bl(kBlock);
    hipExtLaunchKernelGGL((k_line<T, INIT>), gr, bl, line_lds_bytes(g.nz), s, ev.start, ev.stop, 0, g, K, D, x, r, p,
                          q, z, sc);
}

void launch_line_init_f64(hipStream_t s, const Geo& g, const double* K, const double* D, const double* r, double* z,
                          const SolveCtl& sc, const LaunchEv& ev)
{
    line_launch<double, true>(s, g, K, D, nullptr, const_cast<double*>(r), nullptr, nullptr, z, sc, ev);
}

void launch_line_init_f32(hipStream_t s, const Geo& g, const float* K, const float* D, const float* r, float* z,
                          const SolveCtl& sc, const LaunchEv& ev)
{
    line_launch<float, true>(s, g, K, D, nullptr, const_cast<float*>(r), nullptr, nullptr, z, sc, ev);
}

void launch_line_update_f64(hipStream_t s, const Geo& g, const double* K, const double* D, double* x, double* r,
                            const double* p, const double* q, double* z, const SolveCtl& sc, const LaunchEv& ev)
{
    line_launch<double, false>(s, g, K, D, x, r, p, q, z, sc, ev);
}

void launch_line_update_f32(hipStream_t s, const Geo& g, const float* K, const float* D, float* x, float* r,
                            const float* p, const float* q, float* z, const SolveCtl& sc, const LaunchEv& ev)
{
    line_launch<float, false>(s, g, K, D, x, r, p, q, z, sc, ev);
}

void launch_pcg3_spmv_tiled_f64(hipStream_t s, const Geo& g, const TileCfg& t, const uint8_t* flags,
                                const double* K, const double* D, const double* r, double* const p[2],
                                double* q, const SolveCtl& sc, const LaunchEv& ev)
{
    tiled_dispatch<double>(s, g, t, flags, K, D, r, p, q, sc, ev);
}

void launch_pcg3_spmv_tiled_f32(hipStream_t s, const Geo& g, const TileCfg& t, const uint8_t* flags,
                                const float* K, const float* D, const float* r, float* const p[2],
                                float* q, const SolveCtl& sc, const LaunchEv& ev)
{
    tiled_dispatch<float>(s, g, t, flags, K, D, r, p, q, sc, ev);
}

void launch_apply3_f64(hipStream_t s, const Geo& g, const uint8_t* flags, const double* K,
                       const double* D, const double* x, double* y)
{
    const dim3 gr(grid_for(g.n)), bl(kBlock);
    if (flags) hipLaunchKernelGGL((k_apply3<double, true>), gr, bl, 0, s, g, flags, K, D, x, y);
    else hipLaunchKernelGGL((k_apply3<double, false>), gr, bl, 0, s, g, flags, K, D, x, y);
}

void launch_apply3_f32(hipStream_t s, const Geo& g, const uint8_t* flags, const float* K,
                       const float* D, const float* x, float* y)
{
    const dim3 gr(grid_for(g.n)), bl(kBlock);
    if (flags) hipLaunchKernelGGL((k_apply3<float, true>), gr, bl, 0, s, g, flags, K, D, x, y);
    else hipLaunchKernelGGL((k_apply3<float, false>), gr, bl, 0, s, g, flags, K, D, x, y);
}

void launch_cast_f32(hipStream_t s, int n, const double* in, float* out)
{
    hipLaunchKernelGGL(k_cast_f32, dim3(grid_for(n)), dim3(kBlock), 0, s, n, in, out);
}

void launch_cast_f64(hipStream_t s, int n, const float* in, double* out)
{
    hipLaunchKernelGGL(k_cast_f64, dim3(grid_for(n)), dim3(kBlock), 0, s, n, in, out);
}

void launch_olf_faces(hipStream_t s, const OlfArgs& a)
{
    hipLaunchKernelGGL(k_olf_faces, dim3(grid_for(a.g.n)), dim3(kBlock), 0, s, a);
}

void launch_olf_assemble(hipStream_t s, const OlfArgs& a)
{
    hipLaunchKernelGGL(k_olf_assemble, dim3(grid_for(a.g.n)), dim3(kBlock), 0, s, a);
}

void launch_pcg2_spmv(hipStream_t s, const Geo2& g, const double* ke, const double* kn,
                      const double* D, const double* r, double* const p[2], double* q, const SolveCtl& sc)
{
    hipLaunchKernelGGL(k_pcg2_spmv, dim3(grid_for(g.n)), dim3(kBlock), 0, s, g, ke, kn, D, r, p[sc.it & 1],
                       p[(sc.it + 1) & 1], q, sc);
}

void launch_olf_cg_block(hipStream_t s, const OlfCgArgs& a)
{
    hipLaunchKernelGGL(k_olf_cg_block, dim3(1), dim3(kOlfBlockThreads), 0, s, a);
}

void launch_batched_olf_cg_block(hipStream_t s, const OlfCgArgs* args, int nmodels, const int* active)
{
    if (nmodels > 0)
        hipLaunchKernelGGL(kb_olf_cg_block, dim3(nmodels), dim3(kOlfBlockThreads), 0, s, args, active);
}

void launch_olf_post(hipStream_t s, const OlfArgs& a)
{
    hipLaunchKernelGGL(k_olf_post, dim3(grid_for(a.g.n)), dim3(kBlock), 0, s, a);
}

void launch_batched(hipStream_t s, BatchKind kind, const void* args, const BlkMap* map, int nblocks,
                    const int* active)
{
    const dim3 gr(nblocks), bl(kBlock);
    switch (kind) {
    case BK_VG:
        hipLaunchKernelGGL((kb_args<VgArgs, b_vg>), gr, bl, 0, s, (const VgArgs*)args, map, active); break;
    case BK_VG_PICARD:
        hipLaunchKernelGGL((kb_args<VgArgs, b_vg_picard>), gr, bl, 0, s, (const VgArgs*)args, map, active); break;
    case BK_SURF_PRE:
        hipLaunchKernelGGL((kb_args<SurfArgs, b_surface_pre>), gr, bl, 0, s, (const SurfArgs*)args, map, active);
        break;
    case BK_SURF_POST:
        hipLaunchKernelGGL((kb_args<SurfArgs, b_surface_post>), gr, bl, 0, s, (const SurfArgs*)args, map, active);
        break;
    case BK_ASM_F64:
        hipLaunchKernelGGL((kb_args<AsmArgs, b_assemble_flux<false>>), gr, bl, 0, s, (const AsmArgs*)args, map,
                           active);
        break;
    case BK_ASM_MIXED:
        hipLaunchKernelGGL((kb_args<AsmArgs, b_assemble_flux<true>>), gr, bl, 0, s, (const AsmArgs*)args, map,
                           active);
        break;
    case BK_REFINE_ADD:
        hipLaunchKernelGGL((kb_args<RefineArgs, b_refine_add_args>), gr, bl, 0, s, (const RefineArgs*)args, map,
                           active);
        break;
    case BK_REFINE_RES:
        hipLaunchKernelGGL((kb_args<RefineArgs, b_refine_res_args>), gr, bl, 0, s, (const RefineArgs*)args, map,
                           active);
        break;
    case BK_END:
        hipLaunchKernelGGL((kb_args<EndArgs, b_end_step>), gr, bl, 0, s, (const EndArgs*)args, map, active); break;
    case BK_OLF_FACES:
        hipLaunchKernelGGL((kb_args<OlfArgs, b_olf_faces>), gr, bl, 0, s, (const OlfArgs*)args, map, active);
        break;
    case BK_OLF_ASM:
        hipLaunchKernelGGL((kb_args<OlfArgs, b_olf_assemble>), gr, bl, 0, s, (const OlfArgs*)args, map, active);
        break;
    case BK_OLF_POST:
        hipLaunchKernelGGL((kb_args<OlfArgs, b_olf_post>), gr, bl, 0, s, (const OlfArgs*)args, map, active);
        break;
    case BK_PICARD_INC:
        hipLaunchKernelGGL((kb_args<VgArgs, b_picard_inc_args>), gr, bl, 0, s, (const VgArgs*)args, map, active);
        break;
    }
}

void launch_batched_aa(hipStream_t s, int depth, const AaArgs* args, const BlkMap* map, int nblocks,
                       const int* active)
{
    const dim3 gr(nblocks), bl(kBlock);
    switch (depth) {
    case 1: hipLaunchKernelGGL(kb_aa_column<1>, gr, bl, 0, s, args, map, active); break;
    case 2: hipLaunchKernelGGL(kb_aa_column<2>, gr, bl, 0, s, args, map, active); break;
    case 3: hipLaunchKernelGGL(kb_aa_column<3>, gr, bl, 0, s, args, map, active); break;
    case 4: hipLaunchKernelGGL(kb_aa_column<4>, gr, bl, 0, s, args, map, active); break;
    default: hipLaunchKernelGGL(kb_aa_column<kAaMaxDepth>, gr, bl, 0, s, args, map, active); break;
    }
}

int aa_blocks(const Geo& g) { return (g.nxy + kAaCols - 1) / kAaCols; }

void launch_batched_spmv_z(hipStream_t s, bool fp32, const void* kargs, const BlkMap* map, int nblocks,
                           const int* active, const int* it_base, int k)
{
    if (fp32)
        hipLaunchKernelGGL(kb_spmv_z<float>, dim3(nblocks), dim3(kBlock), 0, s, (const KrylovArgs<float>*)kargs, map,
                           active, it_base, k);
    else
        hipLaunchKernelGGL(kb_spmv_z<double>, dim3(nblocks), dim3(kBlock), 0, s, (const KrylovArgs<double>*)kargs,
                           map, active, it_base, k);
}

void launch_batched_line(hipStream_t s, bool fp32, bool init, int nz_max, const void* kargs, const BlkMap* map,
                         int nblocks, const int* active, const int* it_base, int k)
{
    const dim3 gr(nblocks), bl(kBlock);
    const size_t lds = line_lds_bytes(nz_max);
    if (fp32) {
        const KrylovArgs<float>* a = (const KrylovArgs<float>*)kargs;
        if (init) hipLaunchKernelGGL((kb_line<float, true>), gr, bl, lds, s, a, map, active, it_base, k);
        else hipLaunchKernelGGL((kb_line<float, false>), gr, bl, lds, s, a, map, active, it_base, k);
    } else {
        const KrylovArgs<double>* a = (const KrylovArgs<double>*)kargs;
        if (init) hipLaunchKernelGGL((kb_line<double, true>), gr, bl, lds, s, a, map, active, it_base, k);
        else hipLaunchKernelGGL((kb_line<double, false>), gr, bl, lds, s, a, map, active, it_base, k);
    }
}

void launch_batched_spmv3(hipStream_t s, bool fp32, const void* kargs, const BlkMap* map, int nblocks,
                          const int* active, const int* it_base, int k)
{
    if (fp32)
        hipLaunchKernelGGL(kb_spmv3<float>, dim3(nblocks), dim3(kBlock), 0, s, (const KrylovArgs<float>*)kargs, map,
                           active, it_base, k);
    else
        hipLaunchKernelGGL(kb_spmv3<double>, dim3(nblocks), dim3(kBlock), 0, s, (const KrylovArgs<double>*)kargs,
                           map, active, it_base, k);
}

void launch_batched_update3(hipStream_t s, bool fp32, const void* kargs, const BlkMap* map, int nblocks,
                            const int* active, const int* it_base, int k)
{
    if (fp32)
        hipLaunchKernelGGL(kb_update3<float>, dim3(nblocks), dim3(kBlock), 0, s, (const KrylovArgs<float>*)kargs,
                           map, active, it_base, k);
    else
        hipLaunchKernelGGL(kb_update3<double>, dim3(nblocks), dim3(kBlock), 0, s,
                           (const KrylovArgs<double>*)kargs, map, active, it_base, k);
}

void launch_batched_spmv2(hipStream_t s, const void* kargs, const BlkMap* map, int nblocks, const int* active,
                          const int* it_base, int k)
{
    hipLaunchKernelGGL(kb_spmv2, dim3(nblocks), dim3(kBlock), 0, s, (const KrylovArgs<double>*)kargs, map, active,
                       it_base, k);
}

void launch_batched_update2(hipStream_t s, const void* kargs, const BlkMap* map, int nblocks, const int* active,
                            const int* it_base, int k)
{
    hipLaunchKernelGGL(kb_update2, dim3(nblocks), dim3(kBlock), 0, s, (const KrylovArgs<double>*)kargs, map,
                       active, it_base, k);
}

void launch_batched_cg1_init(hipStream_t s, bool fp32, const void* args, const BlkMap* map, int nblocks,
                             const int* active)
{
    if (fp32)
        hipLaunchKernelGGL(kb_cg1_init<float>, dim3(nblocks), dim3(kBlock), 0, s, (const Cg1Args<float>*)args, map,
                           active);
    else
        hipLaunchKernelGGL(kb_cg1_init<double>, dim3(nblocks), dim3(kBlock), 0, s, (const Cg1Args<double>*)args, map,
                           active);
}

void launch_batched_cg1(hipStream_t s, bool fp32, const void* args, const BlkMap* map, int nblocks,
                        const int* active, const int* it_base, int k)
{
    if (fp32)
        hipLaunchKernelGGL(kb_cg1<float>, dim3(nblocks), dim3(kBlock), 0, s, (const Cg1Args<float>*)args, map, active,
                           it_base, k);
    else
        hipLaunchKernelGGL(kb_cg1<double>, dim3(nblocks), dim3(kBlock), 0, s, (const Cg1Args<double>*)args, map,
                           active, it_base, k);
}

void launch_advance(hipStream_t s, int* it_base, int by, const PcgState* st, int nst, PcgState* out)
{
    static_assert(sizeof(PcgState) % sizeof(int) == 0);
    hipLaunchKernelGGL(k_advance, dim3(1), dim3(kBlock), 0, s, it_base, by, (const int*)st,
                       nst * (int)(sizeof(PcgState) / sizeof(int)), (int*)out);
}

void launch_activate(hipStream_t s, const int* flags, int M, int* active, const ActMaps& maps)
{
    hipLaunchKernelGGL(k_activate, dim3(maps.n ? std::min(M, 128) : 1), dim3(kBlock), 0, s, flags, M, active, maps);
}

void launch_reduce_models(hipStream_t s, int nmodels, const double* const* part, const int* nparts, int nv,
                          bool take_max, double* out)
{
    hipLaunchKernelGGL(k_reduce_models, dim3(nmodels), dim3(kBlock), 0, s, part, nparts, nv, take_max ? 1 : 0,
                       out);
}

// ---- one-kernel PCG iteration ----------------------------------------------------------
bool cg1_tile_supported(const TileCfg& t)
{
    return t.kc >= 1 && t.grid >= 0 && (t.grid % 8) == 0 &&
           ((t.tx == 32 && t.ty == 8) || (t.tx == 16 && t.ty == 16) || (t.tx == 32 && t.ty == 16) ||
            (t.tx == 64 && t.ty == 8));
}

// A block marches its planes one after the other (two barriers each), so a surface of few tiles
// is bound by that chain, not by its bytes: 20 to 30 planes of a 32 x 32 or 64 x 64 surface took
// 25 to 34 us a launch.  Splitting the columns adds four halo planes of arithmetic per chunk,
// which idle CUs do for nothing: chunks are taken as long as the blocks stay at about 1.5 per CU.
// Jacobi-PCG steps with whole columns / with this rule (FP64, MI355X, us): 32x32x20 1455 / 979,
// 64x64x30 3470 / 1975, 150x97x40 2274 / 1632, 200x200x30 2813 / 2590; beyond the line (300x300x20,
// 380 tiles) whole columns are within 2 % of the best split, and at 400x400x30 every split loses
// (9689 whole, 10475 with two chunks).
int cg1_default_planes(const Geo& g)
{
    const int nt = ((g.nx + 31) / 32) * ((g.ny + 7) / 8);
    const int nkz = std::max(1, std::min(g.nz, kCg1FillTiles / nt));
    return (g.nz + nkz - 1) / nkz;
}

int cg1_blocks(const Geo& g, const TileCfg& t)
{
    const int nb = tile_blocks(g, t);
    return (t.grid > 0 && t.grid < nb) ? t.grid : nb;
}

template <typename T, int TX, int TY>
static void cg1_launch(hipStream_t s, const Geo& g, const TileCfg& t, const T* K, const T* D, const T* r_in,
                       T* r_out, const T* p_in, T* p_out, T* x, const SolveCtl& sc, const LaunchEv& ev)
{
    const int ntx = (g.nx + TX - 1) / TX, nty = (g.ny + TY - 1) / TY, nkz = (g.nz + t.kc - 1) / t.kc;
    launch_ev(k_cg1<T, TX, TY>, dim3(cg1_blocks(g, t)), dim3(TX * TY), s, ev, g, K, D, r_in, r_out, p_in, p_out,
              x, sc, t.kc, ntx, nty, nkz);
}

template <typename T>
static void cg1_dispatch(hipStream_t s, const Geo& g, const TileCfg& t, const T* K, const T* D, const T* r_in,
                         T* r_out, const T* p_in, T* p_out, T* x, const SolveCtl& sc, const LaunchEv& ev)
{
    if (t.tx == 32 && t.ty == 8) cg1_launch<T, 32, 8>(s, g, t, K, D, r_in, r_out, p_in, p_out, x, sc, ev);
    else if (t.tx == 16 && t.ty == 16) cg1_launch<T, 16, 16>(s, g, t, K, D, r_in, r_out, p_in, p_out, x, sc, ev);
    else if (t.tx == 32 && t.ty == 16) cg1_launch<T, 32, 16>(s, g, t, K, D, r_in, r_out, p_in, p_out, x, sc, ev);
    else cg1_launch<T, 64, 8>(s, g, t, K, D, r_in, r_out, p_in, p_out, x, sc, ev);
}

void launch_cg1_f64(hipStream_t s, const Geo& g, const TileCfg& t, const double* K, const double* D,
                    const double* r_in, double* r_out, const double* p_in, double* p_out, double* x,
                    const SolveCtl& sc, const LaunchEv& ev)
{
    cg1_dispatch<double>(s, g, t, K, D, r_in, r_out, p_in, p_out, x, sc, ev);
}

void launch_cg1_f32(hipStream_t s, const Geo& g, const TileCfg& t, const float* K, const float* D,
                    const float* r_in, float* r_out, const float* p_in, float* p_out, float* x,
                    const SolveCtl& sc, const LaunchEv& ev)
{
    cg1_dispatch<float>(s, g, t, K, D, r_in, r_out, p_in, p_out, x, sc, ev);
}

template <typename T, int TX, int TY>
static void cg1_init_tiled(hipStream_t s, const Geo& g, int kc, const T* K, const T* D, const T* r,
                           const T* p_old, const SolveCtl& sc, const LaunchEv& ev)
{
    const int ntx = (g.nx + TX - 1) / TX, nty = (g.ny + TY - 1) / TY, nkz = (g.nz + kc - 1) / kc;
    launch_ev(k_pcg3_spmv_tiled<T, false, TX, TY, true>, dim3(ntx * nty * nkz), dim3(TX, TY), s, ev, g,
              (const uint8_t*)nullptr, K, D, r, p_old, (T*)nullptr, (T*)nullptr, sc, kc, ntx, nty, nkz);
}

template <typename T>
static void cg1_init(hipStream_t s, const Geo& g, const TileCfg& t, const T* K, const T* D, const T* r,
                     const T* p_old, const SolveCtl& sc, const LaunchEv& ev)
{
    if (t.tx == 32 && t.ty == 8) cg1_init_tiled<T, 32, 8>(s, g, t.kc, K, D, r, p_old, sc, ev);
    else if (t.tx == 64 && t.ty == 4) cg1_init_tiled<T, 64, 4>(s, g, t.kc, K, D, r, p_old, sc, ev);
    else if (t.tx == 16 && t.ty == 16) cg1_init_tiled<T, 16, 16>(s, g, t.kc, K, D, r, p_old, sc, ev);
    else if (t.tx == 32 && t.ty == 4) cg1_init_tiled<T, 32, 4>(s, g, t.kc, K, D, r, p_old, sc, ev);
    else if (t.tx == 64 && t.ty == 8) cg1_init_tiled<T, 64, 8>(s, g, t.kc, K, D, r, p_old, sc, ev);
    else launch_ev(k_cg1_init<T>, dim3(grid_for(g.n)), dim3(kBlock), s, ev, g, K, D, r, p_old, sc);
}

int cg1_init_blocks(const Geo& g, const TileCfg& t)
{
    return t.tx ? tile_blocks(g, t) : grid_for(g.n);
}

void launch_cg1_init_f64(hipStream_t s, const Geo& g, const TileCfg& t, const double* K, const double* D,
                         const double* r, const double* p_old, const SolveCtl& sc, const LaunchEv& ev)
{
    cg1_init<double>(s, g, t, K, D, r, p_old, sc, ev);
}

void launch_cg1_init_f32(hipStream_t s, const Geo& g, const TileCfg& t, const float* K, const float* D,
                         const float* r, const float* p_old, const SolveCtl& sc, const LaunchEv& ev)
{
    cg1_init<float>(s, g, t, K, D, r, p_old, sc, ev);
}

}  // namespace dh

// ctx.h -- the context object behind the C-ABI handle and the host-side helpers shared by
// the forward solver (capi.hip) and the discrete adjoint (adjoint.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>
#include <vector>

#include "../../include/dhara_hip.h"
#include "kernels.h"

struct dhara_adjoint;   // reverse-sweep buffers, allocated on the first adjoint call

// One context = one HIP stream + every device buffer of one model.
struct dhara_ctx {
    dhara_grid grid{};
    dhara_params p{};
    int dev = 0;
    hipStream_t s = nullptr;
    std::string err;
    int N = 0, S = 0;
    dh::Geo g{};
    dh::Geo2 g2{};

    // 3D FP64 state
    double *psi_n = nullptr, *psi_m = nullptr, *x = nullptr;
    double *theta_n = nullptr, *theta_m = nullptr, *theta_new = nullptr;
    double *K = nullptr, *C = nullptr, *Ks = nullptr, *alpha_f = nullptr, *n_f = nullptr;
    double *D = nullptr, *b = nullptr, *r = nullptr, *pv[2] = {nullptr, nullptr}, *q = nullptr;
    // 3D FP32 solver arrays (mixed precision)
    float *K32 = nullptr, *D32 = nullptr, *r32 = nullptr, *d32 = nullptr;
    float *p32[2] = {nullptr, nullptr}, *q32 = nullptr;
    uint8_t* flags = nullptr;
    // surface
    double *z = nullptr, *mann = nullptr, *h = nullptr, *H = nullptr;
    double *rain = nullptr, *evap = nullptr, *transp = nullptr, *hpoten = nullptr, *qcapa = nullptr;
    double *bcpsi[6] = {}, *bcq[6] = {};
    int* bctype[6] = {};
    int* procmap = nullptr;
    double* root = nullptr;
    // overland solver
    double *D2 = nullptr, *b2 = nullptr, *r2 = nullptr, *p2[2] = {nullptr, nullptr}, *q2 = nullptr;
    double *ke = nullptr, *kn = nullptr;
    // overland multigrid hierarchy (allocated on first use) and the preconditioned residual
    dh::MgHier mg{};
    bool mg_ready = false;
    double* z2 = nullptr;
    double* r2b = nullptr;   // second residual buffer: the single-reduction overland CG alternates r2 / r2b
    double *w2 = nullptr, *s2b = nullptr;   // single-reduction overland CG: A z, second A p buffer (with q2)
    // reductions: partial buffers A (written by assembly/update kernels) and B (SpMV kernels)
    double* part[2] = {nullptr, nullptr};
    // column-preconditioned PCG (allocated on first use): z = T^-1 r in FP64 / FP32 and the
    // partials of its segment start-up kernel
    double* zl = nullptr;
    float* zl32 = nullptr;
    double* part_line = nullptr;
    bool vg_ready = false;    // the solve ended with the Picard pass already run (its maxima in rep)
    // Anderson-accelerated Picard update (picard_accel > 0; allocated on first use): the ring of f
    // and y of the last picard_accel + 1 passes, pass p of a step in slot p mod (picard_accel + 1);
    // aa_count: passes of this step that have run.
    double* aa_f[dh::kAaMaxDepth + 1] = {};
    double* aa_y[dh::kAaMaxDepth + 1] = {};
    int aa_count = 0;
    int aa_active = 0;        // the Picard pass after the current solve may update (not the last)
    hipEvent_t aa_ev[2] = {nullptr, nullptr};   // kernel timestamps of the last queued pass (profiling)
    dh::PcgState* st_sub = nullptr;
    dh::PcgState* st_olf = nullptr;
    // pinned host memory that kernels write (HostReport), and the state in it
    dh::HostReport* rep = nullptr;
    dh::PcgState* h_st = nullptr;

    bool face_dirichlet[6] = {false, false, false, false, false, false};
    bool has_alpha = false, has_n = false, has_transp = false;
    bool initialized = false;
    bool theta_m_current = true;
    // iterations of the last solve of each kind: of the subsurface solves one per Picard iteration of
    // a step (a step's solves get shorter as it converges, and the next step's follow them), in
    // mixed precision for the solve's first segment and, seg_hint, the segments after it
    static constexpr int kHints = 16;
    int pcg_hints[kHints], seg_hint = 8, olf_hint = 8, adj_hint = 8;
    int upd_hint = 1;         // reliable updates of the last mixed solve
    int picard_it = 0;        // Picard iteration of the step being solved
    dhara_ctx() { std::fill(pcg_hints, pcg_hints + kHints, 8); }
    int& pcg_hint() { return pcg_hints[std::min(picard_it, kHints - 1)]; }
    std::vector<void*> allocs;
    // Tile shapes: [0] FP64, [1] FP32 (tx = 0: untiled kernels).  A tile that the caller sets is all three;
    // the defaults differ, and the autotuner sets the one that it timed.
    dh::TileCfg tile[2] = {{32, 8, 0}, {32, 8, 0}};         // assembly, refinement, two-kernel SpMV
    dh::TileCfg zin_tile[2] = {{32, 8, 0}, {32, 8, 0}};     // SpMV of the column form
    dh::TileCfg start_tile[2] = {{32, 8, 0}, {32, 8, 0}};   // start-up of the one-kernel PCG
    // one-kernel PCG tiles: [0] FP64, [1] FP32; cg1_set: chosen by the caller or the autotuner
    dh::TileCfg cg1_tile[2] = {{32, 8, 0, 0}, {32, 8, 0, 0}};
    bool cg1_set[2] = {false, false};
    // kernel profiling (dhara_profile_enable)
    bool prof = false;
    std::vector<hipEvent_t> ev;
    dhara_kernel_profile prof_acc{};
    dhara_adjoint* adj = nullptr;
};

namespace dhc {

constexpr int kMaxBatch = 64;   // Krylov iterations queued between two host checks

int set_err(dhara_ctx* c, int code, const std::string& msg);

#define HIPCHK(ctx, call)                                                                   \
    do {                                                                                    \
        hipError_t e_ = (call);                                                             \
        if (e_ != hipSuccess)                                                               \
            return set_err((ctx), DHARA_E_DEVICE,                                           \
                           std::string(#call) + ": " + hipGetErrorString(e_));              \
    } while (0)

#define LAUNCHCHK(ctx)                                                                      \
    do {                                                                                    \
        hipError_t e_ = hipGetLastError();                                                  \
        if (e_ != hipSuccess)                                                               \
            return set_err((ctx), DHARA_E_DEVICE,                                           \
                           std::string("kernel launch: ") + hipGetErrorString(e_));         \
    } while (0)

template <typename T>
int dalloc(dhara_ctx* c, T** ptr, size_t count)
{
    void* v = nullptr;
    hipError_t e = hipMalloc(&v, std::max<size_t>(count, 1) * sizeof(T));
    if (e != hipSuccess) return set_err(c, DHARA_E_ALLOC, std::string("hipMalloc: ") + hipGetErrorString(e));
    e = hipMemsetAsync(v, 0, std::max<size_t>(count, 1) * sizeof(T), c->s);
    if (e != hipSuccess) return set_err(c, DHARA_E_DEVICE, "hipMemset");
    c->allocs.push_back(v);
    *ptr = static_cast<T*>(v);
    return DHARA_OK;
}

int host_reduce(dhara_ctx* c, int nparts, int nv, double* out);   // sums of the first nv rows of part[0]
int read_state(dhara_ctx* c, dh::PcgState* dev);
int sync_stream(dhara_ctx* c);
bool has_dirichlet(const dhara_ctx* c);
dh::Soil soil_of(const dhara_ctx* c);
dh::VgArgs vg_args(dhara_ctx* c, const double* psi, double* theta);
dh::OlfArgs olf_args(dhara_ctx* c);
dh::OlfCgArgs olf_cg_args(dhara_ctx* c, dh::PcgState* st);   // the one-workgroup overland solve
dh::SurfArgs surf_args(dhara_ctx* c);
dh::AsmArgs asm_args(dhara_ctx* c, bool dir);
int alloc_mixed(dhara_ctx* c);
int alloc_line(dhara_ctx* c, bool mixed);
// Anderson pass after the current solve
int alloc_aa(dhara_ctx* c);
dh::AaArgs aa_args(dhara_ctx* c);
void queue_picard_pass(dhara_ctx* c, dh::GateKind gate);
dh::SolveCtl solve_ctl(dhara_ctx* c, dh::PcgState* st, int maxit, int nparts, bool mixed_inner,
                       bool first_sweep);
int do_subsurface_step(dhara_ctx* c, dhara_step_stats* st);
int do_overland_step(dhara_ctx* c, dhara_step_stats* st);
int ensure_mg(dhara_ctx* c);   // allocates the overland multigrid hierarchy
void free_adjoint(dhara_ctx* c);   // adjoint.hip
// noalloc.hip: the device address of this device's scratch array of the allocation-free entry
// point, taken once per device (called by dhara_create with the context's device current)
int noalloc_setup(dhara_ctx* c);

// Queue Krylov iterations in batches; the kernels stop doing work once the device-side
// state says the solve is done, so over-queued iterations cost one launch each.  The SpMV
// kernel of iteration `it` reads partials A and writes B, the update kernel reads B and
// writes A.  With profiling on, events bracket each SpMV and update launch of the batch and
// only the launches that did work (the first ones of the batch) are accumulated.
// after() queues further work behind every batch; it returns true if that work leaves the state in
// the host's report, so that a synchronisation is enough to read it.
template <class SpmvFn, class UpdFn, class AfterFn>
int run_krylov_then(dhara_ctx* c, dh::PcgState* st, int maxit, int& hint, bool prof, double elem,
                    SpmvFn spmv, UpdFn upd, AfterFn after, int it_start, int first_batch)
{
    int it = it_start;
    // first batch: the previous solve's count + the launch that detects the end (the next
    // solve is usually within +-2 of it), or first_batch when the caller knows better; then
    // small batches, since an over-queued iteration costs two empty launches and an
    // under-queued one a host round trip
    int batch = first_batch > 0 ? first_batch : std::max(2, std::min(kMaxBatch, hint + 1));
    for (;;) {
        const int it0 = it;
        for (int b = 0; b < batch; ++b, ++it) {
            dh::LaunchEv e_spmv, e_upd;
            if (prof) {
                e_spmv = dh::LaunchEv{c->ev[4 * b], c->ev[4 * b + 1]};
                e_upd = dh::LaunchEv{c->ev[4 * b + 2], c->ev[4 * b + 3]};
            }
            spmv(it, e_spmv);
            upd(it, e_upd);
        }
        const bool reported = after();
        LAUNCHCHK(c);
        int rc = reported ? sync_stream(c) : read_state(c, st);
        if (rc) return rc;
        const int done_iters = c->h_st->done ? c->h_st->iter : it;
        if (prof) {
            const int real = std::max(0, std::min(batch, done_iters - it0));
            for (int b = 0; b < real; ++b) {
                float m0 = 0.f, m1 = 0.f;
                HIPCHK(c, hipEventElapsedTime(&m0, c->ev[4 * b], c->ev[4 * b + 1]));
                HIPCHK(c, hipEventElapsedTime(&m1, c->ev[4 * b + 2], c->ev[4 * b + 3]));
                c->prof_acc.spmv_ms += m0;
                c->prof_acc.update_ms += m1;
            }
            c->prof_acc.spmv_launches += real;
            c->prof_acc.update_launches += real;
            c->prof_acc.spmv_bytes = 6.0 * elem * c->N;
            c->prof_acc.update_bytes = 7.0 * elem * c->N;
            c->prof_acc.elem_bytes = (int)elem;
        }
        if (c->h_st->done) break;
        if (it > maxit + 1) return set_err(c, DHARA_E_STATE, "Krylov loop did not terminate");
        batch = 3;
    }
    if (first_batch <= 0) hint = std::max(1, c->h_st->iter - it_start);
    return DHARA_OK;
}

template <class SpmvFn, class UpdFn>
int run_krylov(dhara_ctx* c, dh::PcgState* st, int maxit, int& hint, bool prof, double elem,
               SpmvFn spmv, UpdFn upd, int it_start = 0, int first_batch = 0)
{
    return run_krylov_then(c, st, maxit, hint, prof, elem, spmv, upd, [] { return false; }, it_start, first_batch);
}

// One launch per iteration (one-kernel PCG): the same batching as run_krylov; iteration `it`
// of the batch is queued by kern(it, events).  Profiling counts every launch that did work
// as an "spmv" launch of 8 algorithmic arrays.
template <class KernFn, class AfterFn>
int run_krylov1(dhara_ctx* c, dh::PcgState* st, int maxit, int& hint, bool prof, double elem, KernFn kern, AfterFn after,
                int it_start = 0)
{
    int it = it_start;
    int batch = std::max(2, std::min(kMaxBatch, hint + 1));
    for (;;) {
        const int it0 = it;
        for (int b = 0; b < batch; ++b, ++it) {
            dh::LaunchEv e;
            if (prof) e = dh::LaunchEv{c->ev[2 * b], c->ev[2 * b + 1]};
            kern(it, e);
        }
        const bool reported = after();
        LAUNCHCHK(c);
        int rc = reported ? sync_stream(c) : read_state(c, st);
        if (rc) return rc;
        const int done_iters = c->h_st->done ? c->h_st->iter : it;
        if (prof) {
            const int real = std::max(0, std::min(batch, done_iters - it0));
            for (int b = 0; b < real; ++b) {
                float m0 = 0.f;
                HIPCHK(c, hipEventElapsedTime(&m0, c->ev[2 * b], c->ev[2 * b + 1]));
                c->prof_acc.spmv_ms += m0;
            }
            c->prof_acc.spmv_launches += real;
            c->prof_acc.spmv_bytes = 8.0 * elem * c->N;
            c->prof_acc.update_bytes = 0.0;
            c->prof_acc.elem_bytes = (int)elem;
        }
        if (c->h_st->done) break;
        if (it > maxit + 1) return set_err(c, DHARA_E_STATE, "Krylov loop did not terminate");
        batch = 3;
    }
    hint = std::max(1, c->h_st->iter - it_start);
    return DHARA_OK;
}

}  // namespace dhc

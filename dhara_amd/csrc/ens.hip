// ens.hip -- a batched ensemble: many independent models of uneven size stepped together.
//
// No reference counterpart (the reference runs one model per process).  The members are
// ordinary contexts (created, filled and initialised through the C-ABI); the ensemble steps
// all of them at once on its own stream:
//   * every kernel is launched once for all members: a block map sends physical block b to
//     block map[b].id of model map[b].m, which reads that model's argument struct, so one
//     launch covers ~sum N cells (>> 256 workgroups even when each member is small); the maps
//     are compacted on the device to the members still iterating (set_active);
//   * members run in lockstep through the step -- surface pass, Picard iterations, Krylov
//     solves, end of step, overland solve -- and a member that has converged drops out through
//     its active flag (its blocks return at once); every member keeps its own Picard and
//     Krylov stopping decisions, so each member's result is its own, not a batch average;
//   * a batch of 1, 2, 4 or 8 Krylov iterations (SpMV + update kernels for every member) is
//     captured once per size as a hipGraph and replayed while every member is active (eager
//     launches over compacted maps otherwise); the kernels take the iteration index from a
//     device counter that the batch's last node advances, so every replay is the same graph;
//   * per-member reductions go through one kernel that writes all members' sums to pinned host
//     memory; the members' solver states sit in one array, which a batch's last node writes there;
//   * what the host sends (active sets, changed argument images) goes through pinned staging and
//     waits for nothing, so the host waits once per Krylov batch and once per reduction.  With a
//     copy and a wait for each of them: 26.7 -> 24.9 ms (two steps of 20 models of 32..128 x 32..128 x
//     10..40, FP64), 26.1 -> 22.3 ms (12 models, mixed: a refinement round changes the set twice).
// Mixed precision here is FP32 PCG with FP64 iterative refinement that restarts the FP32
// recurrence after each refinement: in lockstep rounds for the Jacobi forms, per member inside
// the running batches for the column form (mixed_line_solve).  A member's overland solve is the
// one-workgroup CG (multigrid or Jacobi) for a surface of at most kOlfBlockCells cells, one
// launch for all such members (the DHARA_OLF_PRECOND_*_BLOCK forms of a single model), else the
// batched lockstep Jacobi-PCG.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <string>
#include <unordered_map>
#include <vector>

#include "ctx.h"

using namespace dhc;

struct dhara_ensemble {
    int M = 0;
    std::vector<dhara_ctx*> mem;
    hipStream_t s = nullptr;
    bool mixed = false, use_graph = true, overland = false;
    std::string err;
    std::vector<void*> allocs;
    dh::BlkMap *map3 = nullptr, *map2 = nullptr;
    int nb3 = 0, nb2 = 0;
    int* active = nullptr;        // device, M
    // Pinned staging of what the host sends between two waits for the stream: active sets (slots of
    // M flags, read by k_activate) and argument images.  Every wait frees all of it; a full one waits.
    static constexpr int kFlagSlots = 64;
    int* h_flags = nullptr;
    int flags_used = 0;
    char* stage = nullptr;
    size_t stage_size = 0, stage_used = 0;
    int* it_base = nullptr;
    dh::PcgState* st = nullptr;   // device, 2M: subsurface then overland
    dh::PcgState* h_st = nullptr; // pinned, written by k_advance
    double** parts = nullptr;     // device, M (each member's partial buffer A)
    int *np3 = nullptr, *np2 = nullptr;
    double* h_red = nullptr;      // pinned, M * kMaxSums, written by k_reduce_models
    // argument arrays (device) and their host images
    dh::VgArgs* a_vg = nullptr;
    dh::SurfArgs* a_surf = nullptr;
    dh::AsmArgs* a_asm = nullptr;
    dh::RefineArgs* a_ref = nullptr;
    dh::EndArgs* a_end = nullptr;
    dh::OlfArgs* a_olf = nullptr;
    dh::OlfCgArgs* a_ocg = nullptr;   // one-workgroup overland solves (olf_kind 1, 2)
    dh::OlfMgArgs* a_omg = nullptr;
    int *olf_jac = nullptr, *olf_mgm = nullptr;   // per-member masks of those launches
    void* a_k3 = nullptr;
    dh::KrylovArgs<double>* a_k2 = nullptr;
    std::vector<dh::VgArgs> h_vg;
    std::vector<dh::SurfArgs> h_surf;
    std::vector<dh::AsmArgs> h_asm;
    std::vector<dh::RefineArgs> h_ref;
    std::vector<dh::EndArgs> h_end;
    std::vector<dh::OlfArgs> h_olf;
    std::vector<dh::OlfCgArgs> h_ocg;
    std::vector<dh::OlfMgArgs> h_omg;
    // each member's overland form: a surface of at most kOlfBlockCells cells the one-workgroup
    // solve (1: Jacobi, 2: multigrid), one launch for all such members, each workgroup to its
    // own member's stopping point; a larger one (0) the batched lockstep Jacobi-PCG
    std::vector<int> olf_kind;
    std::vector<dh::KrylovArgs<double>> h_k3d, h_k2;
    std::vector<dh::KrylovArgs<float>> h_k3f;
    // Krylov batches of 1, 2, 4 or 8 iterations (index log2 of the size), each captured once
    static constexpr int kBatchSizes = 4;
    hipGraphExec_t graph3[kBatchSizes] = {}, graph2[kBatchSizes] = {};
    // first batch of the next solve of each kind: the iterations the last one took, plus the
    // launch that detects the end (subsurface first round, subsurface refinement round, overland)
    int hint[3] = {8, 8, 8};
    // one-kernel PCG of the subsurface solves (every member with DHARA_KRYLOV_ONE_KERNEL)
    bool one = false;
    dh::BlkMap* map_c1 = nullptr;   // one block per 32 x 8 tile of every member
    int nb_c1 = 0;
    void* a_c1 = nullptr;
    std::vector<dh::Cg1Args<double>> h_c1d;
    std::vector<dh::Cg1Args<float>> h_c1f;
    bool c1_full = false;           // the members' whole-column tiles fill the chip together
    int kc_div = 0;                 // dhara_ensemble_autotune: planes per tile = ceil(nz / kc_div); 0: member's tile
    // column-preconditioned PCG (every member with DHARA_PRECOND_COLUMN): the column kernel's
    // block map and the planes of the tallest member
    bool line = false;
    dh::BlkMap* map_l = nullptr;
    int line_nz = 0;
    // Anderson-accelerated Picard update (every member with the same picard_accel > 0): the
    // batched pass over aa_blocks(g) blocks per member
    int aa_depth = 0;
    dh::BlkMap* map_aa = nullptr;
    dh::AaArgs* a_aa = nullptr;
    std::vector<dh::AaArgs> h_aa;
    // Block maps restricted to the active members: a batched launch over the full map spends a
    // block's dependent loads (map entry, active flag, solver state) on every block of an
    // inactive member, which is most of the grid once most members have converged.  k_activate
    // makes all of them when the active set changes.
    struct CMap {
        const dh::BlkMap* full = nullptr;
        int n_full = 0;
        dh::BlkMap* cur = nullptr;          // device, n_full entries
        int n_cur = 0;                      // 0: the full map
        std::vector<int> start, count;      // member m's blocks are full[start[m] ..)
        int *d_start = nullptr, *d_count = nullptr;
    };
    CMap cm3, cm2, cml, cmaa;
    std::vector<int> act;                   // host copy of the active flags
    // the last image uploaded to each argument array: an unchanged image is not sent again (the
    // arrays are read-only on the device), which saves a host synchronisation per launch group
    std::unordered_map<const void*, std::vector<unsigned char>> uploaded;
};

namespace {

int eset(dhara_ensemble* e, int code, const std::string& msg)
{
    if (e) e->err = msg;
    return code;
}

#define EHIP(e, call)                                                                        \
    do {                                                                                     \
        hipError_t e_ = (call);                                                              \
        if (e_ != hipSuccess) return eset((e), DHARA_E_DEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

template <typename T>
int ealloc(dhara_ensemble* e, T** p, size_t n)
{
    void* v = nullptr;
    if (hipMalloc(&v, std::max<size_t>(n, 1) * sizeof(T)) != hipSuccess) return eset(e, DHARA_E_ALLOC, "hipMalloc");
    e->allocs.push_back(v);
    *p = static_cast<T*>(v);
    return DHARA_OK;
}

template <typename T>
int upload(dhara_ensemble* e, T* dev, const std::vector<T>& host)
{
    EHIP(e, hipMemcpyAsync(dev, host.data(), host.size() * sizeof(T), hipMemcpyHostToDevice, e->s));
    EHIP(e, hipStreamSynchronize(e->s));   // the host image may change after this
    return DHARA_OK;
}

// Waits for the stream; the staging memory is free again.
int wait(dhara_ensemble* e)
{
    EHIP(e, hipStreamSynchronize(e->s));
    e->flags_used = 0;
    e->stage_used = 0;
    return DHARA_OK;
}

// Upload of an argument array, skipped when the image equals the last one sent.
template <typename T>
int upload_args(dhara_ensemble* e, T* dev, const std::vector<T>& host)
{
    const size_t nb = host.size() * sizeof(T);
    std::vector<unsigned char>& last = e->uploaded[dev];
    if (last.size() == nb && std::memcmp(last.data(), host.data(), nb) == 0) return DHARA_OK;
    int rc;
    if (nb > e->stage_size) {
        if ((rc = upload(e, dev, host))) return rc;
    } else {
        if (e->stage_used + nb > e->stage_size && (rc = wait(e))) return rc;
        char* at = e->stage + e->stage_used;
        std::memcpy(at, host.data(), nb);
        EHIP(e, hipMemcpyAsync(dev, at, nb, hipMemcpyHostToDevice, e->s));
        e->stage_used += (nb + 63) / 64 * 64;
    }
    last.assign(reinterpret_cast<const unsigned char*>(host.data()),
                reinterpret_cast<const unsigned char*>(host.data()) + nb);
    return DHARA_OK;
}

// The active flags of the members for the launches that follow (unchanged flags are not sent
// again) and the block maps restricted to them, in one launch that reads the flags from pinned
// memory: the host neither copies nor waits.
int set_active(dhara_ensemble* e, const std::vector<int>& on)
{
    if (e->act == on) return DHARA_OK;
    int rc;
    if (e->flags_used == dhara_ensemble::kFlagSlots && (rc = wait(e))) return rc;
    int* flags = e->h_flags + (size_t)e->flags_used++ * e->M;
    std::copy(on.begin(), on.end(), flags);
    dh::ActMaps maps{};
    for (dhara_ensemble::CMap* cm : {&e->cm3, &e->cm2, &e->cml, &e->cmaa}) {
        int tot = 0;
        for (int m = 0; m < e->M; ++m)
            if (on[m] && cm->n_full) tot += cm->count[m];
        cm->n_cur = tot == cm->n_full ? 0 : tot;
        if (cm->n_cur) maps.m[maps.n++] = dh::ActMap{cm->full, cm->d_start, cm->d_count, cm->cur};
    }
    e->act = on;
    dh::launch_activate(e->s, flags, e->M, e->active, maps);
    EHIP(e, hipGetLastError());
    return DHARA_OK;
}

struct MapRef {
    const dh::BlkMap* map;
    int n;
};

// The block map `cm` restricted to the active members (the full map when all, or none, are: the
// kernels test the active flags).
MapRef use_map(const dhara_ensemble::CMap& cm) { return cm.n_cur ? MapRef{cm.cur, cm.n_cur} : MapRef{cm.full, cm.n_full}; }

// Compacted maps: device buffers and the members' block ranges of a full map.
int init_cmap(dhara_ensemble* e, dhara_ensemble::CMap& cm, const dh::BlkMap* full_dev,
              const std::vector<dh::BlkMap>& full)
{
    cm.full = full_dev;
    cm.n_full = (int)full.size();
    cm.start.assign(e->M, 0);
    cm.count.assign(e->M, 0);
    for (int i = (int)full.size() - 1; i >= 0; --i) {   // members' blocks are contiguous
        cm.start[full[i].m] = i;
        ++cm.count[full[i].m];
    }
    if (cm.n_full == 0) return DHARA_OK;
    int rc = ealloc(e, &cm.cur, full.size());
    if (!rc) rc = ealloc(e, &cm.d_start, e->M);
    if (!rc) rc = ealloc(e, &cm.d_count, e->M);
    if (!rc) rc = upload(e, cm.d_start, cm.start);
    if (!rc) rc = upload(e, cm.d_count, cm.count);
    return rc;
}

// The members' sums or maxima in e->h_red.
int reduce(dhara_ensemble* e, bool two_d, int nv, bool take_max)
{
    dh::launch_reduce_models(e->s, e->M, e->parts, two_d ? e->np2 : e->np3, nv, take_max, e->h_red);
    EHIP(e, hipGetLastError());
    return wait(e);
}

// One batch of 1 << lg Krylov iterations for every member whose active flag is set; leaves the
// solver states in e->h_st.
void krylov_batch(dhara_ensemble* e, bool two_d, int lg)
{
    const int nb = 1 << lg;
    for (int k = 0; k < nb; ++k) {
        if (two_d) {
            const MapRef r = use_map(e->cm2);
            dh::launch_batched_spmv2(e->s, e->a_k2, r.map, r.n, e->active, e->it_base, k);
            dh::launch_batched_update2(e->s, e->a_k2, r.map, r.n, e->active, e->it_base, k);
        } else if (e->line) {
            const MapRef r = use_map(e->cm3);
            dh::launch_batched_spmv_z(e->s, e->mixed, e->a_k3, r.map, r.n, e->active, e->it_base, k);
            const MapRef l = use_map(e->cml);
            dh::launch_batched_line(e->s, e->mixed, false, e->line_nz, e->a_k3, l.map, l.n, e->active, e->it_base, k);
        } else if (e->one) {
            dh::launch_batched_cg1(e->s, e->mixed, e->a_c1, e->map_c1, e->nb_c1, e->active, e->it_base, k);
        } else {
            dh::launch_batched_spmv3(e->s, e->mixed, e->a_k3, e->map3, e->nb3, e->active, e->it_base, k);
            dh::launch_batched_update3(e->s, e->mixed, e->a_k3, e->map3, e->nb3, e->active, e->it_base, k);
        }
    }
    dh::launch_advance(e->s, e->it_base, nb, e->st, 2 * e->M, e->h_st);
}

int ensure_graph(dhara_ensemble* e, bool two_d, int lg)
{
    hipGraphExec_t& ex = two_d ? e->graph2[lg] : e->graph3[lg];
    if (ex) return DHARA_OK;
    hipGraph_t g = nullptr;
    EHIP(e, hipStreamBeginCapture(e->s, hipStreamCaptureModeThreadLocal));
    krylov_batch(e, two_d, lg);
    EHIP(e, hipStreamEndCapture(e->s, &g));
    EHIP(e, hipGraphInstantiate(&ex, g, nullptr, nullptr, 0));
    (void)hipGraphDestroy(g);
    return DHARA_OK;
}

void drop_graphs(dhara_ensemble* e, bool three_d_only)
{
    for (int i = 0; i < dhara_ensemble::kBatchSizes; ++i) {
        if (e->graph3[i]) (void)hipGraphExecDestroy(e->graph3[i]);
        e->graph3[i] = nullptr;
        if (three_d_only) continue;
        if (e->graph2[i]) (void)hipGraphExecDestroy(e->graph2[i]);
        e->graph2[i] = nullptr;
    }
}

// Krylov iterations until every active member's solve is done (`two_d`: the overland solves).
// The first batch is sized from the last solve of the same kind (`kind` indexes e->hint), the
// following ones take 8 iterations: a solve of a few iterations then queues few launches that
// only find their member done.  Members whose solve has ended leave the launches of the later
// batches; the caller's active set is restored at the end.
int krylov_solve(dhara_ensemble* e, bool two_d, const std::vector<int>& on, int maxit, int kind)
{
    EHIP(e, hipMemsetAsync(e->it_base, 0, sizeof(int), e->s));   // outside any captured graph
    if (!two_d && e->one) {
        dh::launch_batched_cg1_init(e->s, e->mixed, e->a_c1, e->map3, e->nb3, e->active);
        EHIP(e, hipGetLastError());
    }
    if (!two_d && e->line) {   // z = T^-1 r of the fresh residual
        const MapRef l = use_map(e->cml);
        dh::launch_batched_line(e->s, e->mixed, true, e->line_nz, e->a_k3, l.map, l.n, e->active, e->it_base, 0);
        EHIP(e, hipGetLastError());
    }
    const int off = two_d ? e->M : 0;
    int lg = 0;
    while (lg < dhara_ensemble::kBatchSizes - 1 && (1 << lg) < e->hint[kind]) ++lg;
    std::vector<int> still = on;
    for (int launched = 0;;) {
        // a captured batch holds the full maps: replayed while every member is active
        const bool full = std::all_of(e->act.begin(), e->act.end(), [](int a) { return a != 0; });
        if (e->use_graph && full) {
            int rc = ensure_graph(e, two_d, lg);
            if (rc) return rc;
            EHIP(e, hipGraphLaunch(two_d ? e->graph2[lg] : e->graph3[lg], e->s));
        } else {
            krylov_batch(e, two_d, lg);
        }
        EHIP(e, hipGetLastError());
        launched += 1 << lg;
        int rc = wait(e);
        if (rc) return rc;
        bool all = true;
        int most = 0;
        for (int m = 0; m < e->M; ++m) {
            if (!on[m]) continue;
            if (!e->h_st[off + m].done) all = false;
            most = std::max(most, e->h_st[off + m].iter);
        }
        if (all) {
            e->hint[kind] = most + 1;
            if (still != on && (rc = set_active(e, on))) return rc;   // as the caller set it
            break;
        }
        if (launched > maxit + 16) return eset(e, DHARA_E_STATE, "batched Krylov loop did not terminate");
        lg = dhara_ensemble::kBatchSizes - 1;
        bool shrink = false;   // members whose solve has ended leave the launches
        for (int m = 0; m < e->M; ++m)
            if (still[m] && e->h_st[off + m].done) {
                still[m] = 0;
                shrink = true;
            }
        if (shrink && (rc = set_active(e, still))) return rc;
    }
    return DHARA_OK;
}

dh::SolveCtl ctl(dhara_ctx* c, dh::PcgState* st, int maxit, double tol, bool mixed_inner, bool first_sweep,
                 double* part_in, int nparts, double* part_out)
{
    dh::SolveCtl sc{};
    sc.maxit = maxit;
    sc.mixed_inner = mixed_inner ? 1 : 0;
    sc.first_sweep = first_sweep ? 1 : 0;
    sc.lin_tol = tol;
    sc.inner_tol = c->p.inner_tol;
    sc.part_in = part_in;
    sc.nparts = nparts;
    sc.part_out = part_out;
    sc.st = st;
    return sc;
}

void build_k3(dhara_ensemble* e, bool first_sweep)
{
    for (int m = 0; m < e->M; ++m) {
        dhara_ctx* c = e->mem[m];
        const int np = dh::grid_for(c->N);
        if (e->mixed) {
            dh::KrylovArgs<float>& k = e->h_k3f[m];
            k = dh::KrylovArgs<float>{};
            k.g = c->g;
            k.K = c->K32; k.D = c->D32; k.r = c->r32;
            k.x = c->d32; k.res = c->r32; k.p[0] = c->p32[0]; k.p[1] = c->p32[1]; k.q = c->q32;
            k.spmv = ctl(c, &e->st[m], c->p.inner_maxiter, c->p.lin_tol, true, first_sweep, c->part[0], np, c->part[1]);
            k.upd = ctl(c, &e->st[m], c->p.inner_maxiter, c->p.lin_tol, true, first_sweep, c->part[1], np, c->part[0]);
            if (e->line) {
                k.z = c->zl32;
                k.init = ctl(c, &e->st[m], c->p.inner_maxiter, c->p.lin_tol, true, first_sweep, c->part[0], np,
                             c->part_line);
                k.part_first = c->part_line;
                k.spmv.nparts = dh::line_blocks(c->g);
            }
        } else {
            dh::KrylovArgs<double>& k = e->h_k3d[m];
            k = dh::KrylovArgs<double>{};
            k.g = c->g;
            k.K = c->K; k.D = c->D; k.r = c->r;
            k.x = c->x; k.res = c->r; k.p[0] = c->pv[0]; k.p[1] = c->pv[1]; k.q = c->q;
            k.spmv = ctl(c, &e->st[m], c->p.lin_maxiter, c->p.lin_tol, false, true, c->part[0], np, c->part[1]);
            k.upd = ctl(c, &e->st[m], c->p.lin_maxiter, c->p.lin_tol, false, true, c->part[1], np, c->part[0]);
            if (e->line) {
                k.z = c->zl;
                k.init = ctl(c, &e->st[m], c->p.lin_maxiter, c->p.lin_tol, false, true, c->part[0], np, c->part_line);
                k.part_first = c->part_line;
                k.spmv.nparts = dh::line_blocks(c->g);
            }
        }
    }
}

int upload_k3(dhara_ensemble* e)
{
    return e->mixed ? upload_args(e, (dh::KrylovArgs<float>*)e->a_k3, e->h_k3f)
                    : upload_args(e, (dh::KrylovArgs<double>*)e->a_k3, e->h_k3d);
}

// Tiles of a member in the batched one-kernel PCG: 32 x 8 columns; the member's own planes per
// tile when its tile is 32 x 8, whole columns otherwise.  The default planes of a small member split
// its columns to fill the chip; members that fill it together (e->c1_full: more whole-column tiles
// than kCg1FillTiles) keep whole columns unless their tile was set or tuned, since the chunks' halo
// planes would then only add work (the solve is the same to rounding: other partial sums).
void c1_tiles(const dhara_ensemble* e, const dhara_ctx* c, int& kc, int& ntx, int& nty, int& nkz, int kc_div)
{
    const int pr = e->mixed ? 1 : 0;
    const dh::TileCfg& t = c->cg1_tile[pr];
    if (kc_div > 0) kc = (c->g.nz + kc_div - 1) / kc_div;
    else if (e->c1_full && !c->cg1_set[pr]) kc = c->g.nz;
    else kc = (t.tx == dh::kCg1BatchTx && t.ty == dh::kCg1BatchTy && t.kc > 0) ? std::min(t.kc, c->g.nz) : c->g.nz;
    ntx = (c->g.nx + dh::kCg1BatchTx - 1) / dh::kCg1BatchTx;
    nty = (c->g.ny + dh::kCg1BatchTy - 1) / dh::kCg1BatchTy;
    nkz = (c->g.nz + kc - 1) / kc;
}

template <typename T>
void fill_c1(dhara_ensemble* e, dhara_ctx* c, int m, bool first_sweep, const T* K, const T* D, T* r0, T* r1, T* p0,
             T* p1, T* x, dh::Cg1Args<T>& a)
{
    a = dh::Cg1Args<T>{};
    a.g = c->g;
    a.K = K; a.D = D;
    a.r[0] = r0; a.r[1] = r1; a.p[0] = p0; a.p[1] = p1; a.x = x;
    a.part_asm = c->part[0];
    a.part[0] = c->part[0]; a.part[1] = c->part[1];
    a.nparts_asm = dh::grid_for(c->N);
    c1_tiles(e, c, a.kc, a.ntx, a.nty, a.nkz, e->kc_div);
    a.ntiles = a.ntx * a.nty * a.nkz;
    const int maxit = e->mixed ? c->p.inner_maxiter : c->p.lin_maxiter;
    a.ctl = ctl(c, &e->st[m], maxit, c->p.lin_tol, e->mixed, first_sweep, nullptr, 0, nullptr);
}

// Block map of the batched one-kernel PCG for a planes-per-tile policy (kc_div, see c1_tiles).
int c1_map(dhara_ensemble* e, int kc_div, std::vector<dh::BlkMap>& map)
{
    map.clear();
    for (int m = 0; m < e->M; ++m) {
        int kc, ntx, nty, nkz;
        c1_tiles(e, e->mem[m], kc, ntx, nty, nkz, kc_div);
        const int nt = ntx * nty * nkz;
        if (nt > dh::kMaxBlocks) return eset(e, DHARA_E_UNSUPPORTED, "member has more tiles than partial slots");
        for (int b = 0; b < nt; ++b) map.push_back(dh::BlkMap{m, b, nt});
    }
    return DHARA_OK;
}

// Arguments of the one-kernel PCG of every member (first_sweep: ||b||^2 from the assembly).
void build_c1(dhara_ensemble* e, bool first_sweep)
{
    for (int m = 0; m < e->M; ++m) {
        dhara_ctx* c = e->mem[m];
        if (e->mixed)
            fill_c1<float>(e, c, m, first_sweep, c->K32, c->D32, c->r32, c->q32, c->p32[0], c->p32[1], c->d32,
                           e->h_c1f[m]);
        else
            fill_c1<double>(e, c, m, first_sweep, c->K, c->D, c->r, c->q, c->pv[0], c->pv[1], c->x, e->h_c1d[m]);
    }
}

int upload_c1(dhara_ensemble* e)
{
    return e->mixed ? upload_args(e, (dh::Cg1Args<float>*)e->a_c1, e->h_c1f)
                    : upload_args(e, (dh::Cg1Args<double>*)e->a_c1, e->h_c1d);
}

// Kernel arguments of the subsurface Krylov solve of every member.
int build_krylov(dhara_ensemble* e, bool first_sweep)
{
    if (e->one) {
        build_c1(e, first_sweep);
        return upload_c1(e);
    }
    build_k3(e, first_sweep);
    return upload_k3(e);
}

// The mixed column-preconditioned solve of every member in `on` with per-member reliable
// updates: after each batch, a member whose FP32 segment has ended without passing the outer
// test folds its correction into x and restarts from the FP64 residual (refinement add,
// FP64 residual, column start-up), and its next segment's iterations run in the batches that
// the other members are still iterating in (its iteration index restarts at 0 through the
// argument seg0), so no member waits for the slowest one between refinement rounds.
int mixed_line_solve(dhara_ensemble* e, const std::vector<int>& on, std::vector<dhara_step_stats>& st)
{
    const int M = e->M;
    int rc;
    std::vector<int> solving = on, rounds(M, 0);
    for (int m = 0; m < M; ++m) e->h_k3f[m].seg0 = 0;
    if ((rc = upload_k3(e)) || (rc = set_active(e, solving))) return rc;
    EHIP(e, hipMemsetAsync(e->it_base, 0, sizeof(int), e->s));   // outside any captured graph
    {   // z = T^-1 r of the assembly's residual
        const MapRef l = use_map(e->cml);
        dh::launch_batched_line(e->s, true, true, e->line_nz, e->a_k3, l.map, l.n, e->active, e->it_base, 0);
    }
    EHIP(e, hipGetLastError());
    const int maxit = e->mem[0]->p.inner_maxiter, maxr = e->mem[0]->p.refine_maxiter;
    int lg = 0;
    while (lg < dhara_ensemble::kBatchSizes - 1 && (1 << lg) < e->hint[0]) ++lg;
    int seg_most = 0;   // the longest segment of the first batch's members (next solve's hint)
    bool first = true;
    for (int launched = 0;;) {
        const bool full = std::all_of(e->act.begin(), e->act.end(), [](int a) { return a != 0; });
        if (e->use_graph && full) {
            if ((rc = ensure_graph(e, false, lg))) return rc;
            EHIP(e, hipGraphLaunch(e->graph3[lg], e->s));
        } else {
            krylov_batch(e, false, lg);
        }
        EHIP(e, hipGetLastError());
        launched += 1 << lg;
        if ((rc = wait(e))) return rc;
        std::vector<int> restart(M, 0), next(M, 0);
        bool any_next = false, any_restart = false;
        int most = 0;
        for (int m = 0; m < M; ++m) {
            if (!solving[m]) continue;
            const dh::PcgState& ps = e->h_st[m];
            if (!ps.done) {
                next[m] = 1;
                any_next = true;
                continue;
            }
            st[m].lin_iters += ps.iter;
            most = std::max(most, ps.iter);
            if (ps.nan) st[m].nan_seen = 1;
            if (ps.outer_conv || ps.nan) {
                if (!ps.outer_conv) st[m].lin_converged = 0;
                continue;
            }
            if (rounds[m] >= maxr) {
                st[m].lin_converged = 0;
                continue;
            }
            ++rounds[m];
            st[m].refine_sweeps += 1;
            restart[m] = next[m] = 1;
            any_next = any_restart = true;
        }
        if (first) seg_most = most;
        first = false;
        if (!any_next) break;
        if (launched > (maxr + 1) * (maxit + 16))
            return eset(e, DHARA_E_STATE, "batched Krylov loop did not terminate");
        if (any_restart) {
            for (int m = 0; m < M; ++m) {
                if (!restart[m]) continue;
                dhara_ctx* c = e->mem[m];
                dh::KrylovArgs<float>& k = e->h_k3f[m];
                k.seg0 = launched;                                   // the next batch starts at 0
                k.spmv.first_sweep = k.upd.first_sweep = k.init.first_sweep = 0;   // keep ||b||
                dh::RefineArgs& ra = e->h_ref[m];
                ra = dh::RefineArgs{};
                ra.g = c->g; ra.K = c->K; ra.D = c->D; ra.b = c->b; ra.x = c->x; ra.flags = nullptr;
                ra.r32 = c->r32; ra.D32 = c->D32; ra.d32 = c->d32; ra.part_out = c->part[0]; ra.st = &e->st[m];
            }
            if ((rc = upload_k3(e)) || (rc = upload_args(e, e->a_ref, e->h_ref)) || (rc = set_active(e, restart)))
                return rc;
            const MapRef r = use_map(e->cm3);
            dh::launch_batched(e->s, dh::BK_REFINE_ADD, e->a_ref, r.map, r.n, e->active);
            dh::launch_batched(e->s, dh::BK_REFINE_RES, e->a_ref, r.map, r.n, e->active);
            const MapRef l = use_map(e->cml);
            dh::launch_batched_line(e->s, true, true, e->line_nz, e->a_k3, l.map, l.n, e->active, e->it_base, 0);
            EHIP(e, hipGetLastError());
            // a restarted segment is as long as the refinement segments before it
            lg = 0;
            while (lg < dhara_ensemble::kBatchSizes - 1 && (1 << lg) < e->hint[1]) ++lg;
            e->hint[1] = std::max(1, most) + 1;
        } else {
            lg = dhara_ensemble::kBatchSizes - 1;
        }
        if ((rc = set_active(e, next))) return rc;
        solving = next;
    }
    e->hint[0] = seg_most + 1;
    return set_active(e, on);
}

// Subsurface step of every member (do_subsurface_step in lockstep).
int subsurface_step(dhara_ensemble* e, std::vector<dhara_step_stats>& st)
{
    const int M = e->M;
    int rc;
    for (int m = 0; m < M; ++m) {
        dhara_ctx* c = e->mem[m];
        if (c->p.am != 0.0 || e->aa_depth)
            EHIP(e, hipMemcpyAsync(c->psi_m, c->psi_n, (size_t)c->N * 8, hipMemcpyDeviceToDevice, e->s));
        c->aa_count = 0;
        e->h_surf[m] = surf_args(c);
    }
    std::vector<int> all(M, 1), surf(M, 0);
    for (int m = 0; m < M; ++m) surf[m] = e->mem[m]->p.top_bc == DHARA_TOP_SURFACE;
    if ((rc = upload_args(e, e->a_surf, e->h_surf)) || (rc = set_active(e, surf))) return rc;
    {
        const MapRef r = use_map(e->cm2);
        dh::launch_batched(e->s, dh::BK_SURF_PRE, e->a_surf, r.map, r.n, e->active);
    }
    for (int m = 0; m < M; ++m) {
        dhara_ctx* c = e->mem[m];
        if (!c->theta_m_current) {
            std::swap(c->theta_m, c->theta_new);
            c->theta_m_current = true;
        }
        st[m].lin_converged = 1;
    }
    std::vector<int> pic(M, 1), niter(M, 0), conv(M, 0);
    std::vector<double> delta(M, 0.0);
    auto any = [](const std::vector<int>& v) { return std::any_of(v.begin(), v.end(), [](int x) { return x != 0; }); };
    while (any(pic)) {
        // assembly (D, b, r0 = b - A x) of every member still iterating
        for (int m = 0; m < M; ++m) {
            dhara_ctx* c = e->mem[m];
            e->h_asm[m] = asm_args(c, false);
            e->h_asm[m].st = &e->st[m];
        }
        if ((rc = upload_args(e, e->a_asm, e->h_asm)) || (rc = set_active(e, pic))) return rc;
        {
            const MapRef r = use_map(e->cm3);
            dh::launch_batched(e->s, e->mixed ? dh::BK_ASM_MIXED : dh::BK_ASM_F64, e->a_asm, r.map, r.n, e->active);
        }
        if ((rc = build_krylov(e, true))) return rc;
        std::vector<int> solving = pic;
        int round = 0;
        if (e->mixed && e->line) {
            if ((rc = mixed_line_solve(e, pic, st))) return rc;
            solving.assign(M, 0);   // the rounds below are done
        }
        for (; std::any_of(solving.begin(), solving.end(), [](int v) { return v != 0; });) {
            if ((rc = set_active(e, solving))) return rc;
            const int maxit = e->mixed ? e->mem[0]->p.inner_maxiter : e->mem[0]->p.lin_maxiter;
            if ((rc = krylov_solve(e, false, solving, maxit, round == 0 ? 0 : 1))) return rc;
            std::vector<int> refine(M, 0);
            for (int m = 0; m < M; ++m) {
                if (!solving[m]) continue;
                const dh::PcgState& s = e->h_st[m];
                st[m].lin_iters += s.iter;
                if (s.nan) st[m].nan_seen = 1;
                if (!e->mixed) {
                    st[m].lin_converged &= s.conv;
                    continue;
                }
                if (s.outer_conv || s.nan) {
                    if (!s.outer_conv) st[m].lin_converged = 0;
                    continue;
                }
                refine[m] = 1;   // fold d into x and restart from the FP64 residual
            }
            if (!e->mixed || !any(refine)) break;
            for (int m = 0; m < M; ++m) {
                dhara_ctx* c = e->mem[m];
                dh::RefineArgs& ra = e->h_ref[m];
                ra = dh::RefineArgs{};
                ra.g = c->g; ra.K = c->K; ra.D = c->D; ra.b = c->b; ra.x = c->x; ra.flags = nullptr;
                ra.r32 = c->r32; ra.D32 = c->D32; ra.d32 = c->d32; ra.part_out = c->part[0]; ra.st = &e->st[m];
                if (refine[m]) st[m].refine_sweeps += 1;
            }
            if ((rc = upload_args(e, e->a_ref, e->h_ref)) || (rc = set_active(e, refine))) return rc;
            {
                const MapRef r = use_map(e->cm3);
                dh::launch_batched(e->s, dh::BK_REFINE_ADD, e->a_ref, r.map, r.n, e->active);
                dh::launch_batched(e->s, dh::BK_REFINE_RES, e->a_ref, r.map, r.n, e->active);
            }
            ++round;
            if (round > e->mem[0]->p.refine_maxiter) {
                for (int m = 0; m < M; ++m)
                    if (refine[m]) st[m].lin_converged = 0;
                break;
            }
            if (round == 1 && (rc = build_krylov(e, false))) return rc;   // later rounds keep the first round's ||b||
            solving = refine;
        }
        // theta, K, C of the new iterate and the Picard increment (k_vg_picard) for every member;
        // with the Anderson update and a rule on psi the increment alone (theta, K, C then come
        // from the Anderson pass, or from a pass over x once the member stops)
        std::vector<int> inc_only(M, 0), full(M, 0);
        for (int m = 0; m < M; ++m) {
            if (!pic[m]) continue;
            dhara_ctx* c = e->mem[m];
            e->h_vg[m] = vg_args(c, c->x, c->theta_new);
            (e->aa_depth && c->p.picard_rule != DHARA_PICARD_REL_THETA ? inc_only : full)[m] = 1;
        }
        if ((rc = upload_args(e, e->a_vg, e->h_vg))) return rc;
        if (any(full)) {
            if ((rc = set_active(e, full))) return rc;
            const MapRef r = use_map(e->cm3);
            dh::launch_batched(e->s, dh::BK_VG_PICARD, e->a_vg, r.map, r.n, e->active);
        }
        if (any(inc_only)) {
            if ((rc = set_active(e, inc_only))) return rc;
            const MapRef r = use_map(e->cm3);
            dh::launch_batched(e->s, dh::BK_PICARD_INC, e->a_vg, r.map, r.n, e->active);
        }
        if ((rc = reduce(e, false, 2, true))) return rc;
        std::vector<int> relax(M, 0), accel(M, 0);
        for (int m = 0; m < M; ++m) {
            if (!pic[m]) continue;
            dhara_ctx* c = e->mem[m];
            ++niter[m];
            delta[m] = e->h_red[2 * m];
            if (e->h_red[2 * m + 1] > 0.0 || st[m].nan_seen) {
                st[m].nan_seen = 1;
                pic[m] = 0;
                c->theta_m_current = false;
            } else if (delta[m] < c->p.picard_tol) {
                conv[m] = 1;
                pic[m] = 0;
                c->theta_m_current = false;
            } else if (niter[m] < c->p.picard_maxiter) {
                if (e->aa_depth) accel[m] = 1;
                else if (c->p.am == 0.0) std::swap(c->theta_m, c->theta_new);
                else relax[m] = 1;
                c->theta_m_current = true;
            } else {
                pic[m] = 0;
                c->theta_m_current = false;
            }
        }
        std::vector<int> final_vg(M, 0);   // members that stopped after an increment-only pass
        for (int m = 0; m < M; ++m) final_vg[m] = inc_only[m] && !accel[m];
        if (any(final_vg)) {
            if ((rc = set_active(e, final_vg))) return rc;
            const MapRef r = use_map(e->cm3);
            dh::launch_batched(e->s, dh::BK_VG, e->a_vg, r.map, r.n, e->active);
        }
        if (any(accel)) {   // the Anderson pass: next iterate psi_m and theta, K, C at it
            for (int m = 0; m < M; ++m) {
                if (!accel[m]) continue;
                dhara_ctx* c = e->mem[m];
                c->aa_active = 1;
                e->h_aa[m] = aa_args(c);
                ++c->aa_count;
            }
            if ((rc = upload_args(e, e->a_aa, e->h_aa)) || (rc = set_active(e, accel))) return rc;
            const MapRef r = use_map(e->cmaa);
            dh::launch_batched_aa(e->s, e->aa_depth, e->a_aa, r.map, r.n, e->active);
            EHIP(e, hipGetLastError());
        }
        if (any(relax)) {   // theta, K, C at the relaxed iterate psi_m
            for (int m = 0; m < M; ++m) e->h_vg[m] = vg_args(e->mem[m], e->mem[m]->psi_m, e->mem[m]->theta_m);
            if ((rc = upload_args(e, e->a_vg, e->h_vg)) || (rc = set_active(e, relax))) return rc;
            const MapRef r = use_map(e->cm3);
            dh::launch_batched(e->s, dh::BK_VG, e->a_vg, r.map, r.n, e->active);
        }
    }
    // ponding update and end of step for every member
    if ((rc = set_active(e, surf))) return rc;
    {
        const MapRef r = use_map(e->cm2);
        dh::launch_batched(e->s, dh::BK_SURF_POST, e->a_surf, r.map, r.n, e->active);
    }
    for (int m = 0; m < M; ++m) {
        dhara_ctx* c = e->mem[m];
        dh::EndArgs& ea = e->h_end[m];
        ea = dh::EndArgs{};
        ea.g = c->g;
        ea.dt = c->p.dt;
        ea.Ss = c->p.Ss;
        ea.poros = c->p.porosity;
        ea.x = c->x;
        ea.theta_new = c->theta_new;
        ea.theta_m = c->theta_m;
        ea.psi_n = c->psi_n;
        ea.theta_n = c->theta_n;
        ea.transp = c->transp;
        ea.root = c->root;
        ea.procmap = c->procmap;
        ea.has_transp = c->has_transp ? 1 : 0;
        ea.carry_reference = c->p.theta_carry == DHARA_THETA_CARRY_REFERENCE ? 1 : 0;
        for (int f = 0; f < 6; ++f) {
            ea.bctype[f] = c->bctype[f];
            ea.bcq[f] = c->bcq[f];
        }
        ea.part_out = c->part[0];
    }
    if ((rc = upload_args(e, e->a_end, e->h_end)) || (rc = set_active(e, all))) return rc;
    {
        const MapRef r = use_map(e->cm3);
        dh::launch_batched(e->s, dh::BK_END, e->a_end, r.map, r.n, e->active);
    }
    if ((rc = reduce(e, false, 9, false))) return rc;
    for (int m = 0; m < M; ++m) {
        dhara_ctx* c = e->mem[m];
        c->theta_m_current = false;
        dhara_step_stats& o = st[m];
        o.picard_iters = niter[m];
        o.picard_converged = conv[m];
        o.picard_delta = o.nan_seen ? NAN : delta[m];
        const double* s = e->h_red + 9 * m;
        const double dx = c->grid.dx, dy = c->grid.dy, dz = c->grid.dz, dt = c->p.dt;
        const double qt = s[3], qb = s[4], qw = s[5], qe = s[6], qs = s[7], qn = s[8];
        o.mb_ref = s[0] * dz + ((qe - qw) + (qn - qs) + (qb - qt)) * dt + s[2] + s[1];
        o.storage_change = (s[0] * dz + s[1]) * dx * dy;
        const double inflow = (qt - qb) * dx * dy * dt + (qw - qe) * dy * dz * dt + (qs - qn) * dx * dz * dt -
                              s[2] * dx * dy;
        o.boundary_inflow = inflow;
        const double flux_scale = (std::fabs(qt) + std::fabs(qb)) * dx * dy * dt +
                                  (std::fabs(qw) + std::fabs(qe)) * dy * dz * dt +
                                  (std::fabs(qs) + std::fabs(qn)) * dx * dz * dt + s[2] * dx * dy;
        const double scale = std::max({std::fabs(o.storage_change), std::fabs(inflow), flux_scale, 1e-300});
        o.mb_rel = std::fabs(o.storage_change - inflow) / scale;
    }
    return DHARA_OK;
}

int overland_step(dhara_ensemble* e, std::vector<dhara_step_stats>& st)
{
    const int M = e->M;
    int rc;
    std::vector<int> on(M, 0);
    for (int m = 0; m < M; ++m) {   // the form from the member's current parameters
        dhara_ctx* c = e->mem[m];
        const int op = c->p.olf_precond;
        const bool mg = op == DHARA_OLF_PRECOND_MG || op == DHARA_OLF_PRECOND_MG_BLOCK;
        e->olf_kind[m] = c->S > dh::kOlfBlockCells ? 0 : mg ? 2 : 1;
        if (e->olf_kind[m] == 2 && (rc = ensure_mg(c))) return eset(e, rc, c->err);
    }
    for (int m = 0; m < M; ++m) {
        dhara_ctx* c = e->mem[m];
        on[m] = c->p.overland ? 1 : 0;
        e->h_olf[m] = olf_args(c);
        e->h_olf[m].st = &e->st[M + m];
        dh::KrylovArgs<double>& k = e->h_k2[m];
        k = dh::KrylovArgs<double>{};
        k.g2 = c->g2;
        k.D = c->D2; k.r = c->r2; k.x = c->H; k.res = c->r2; k.p[0] = c->p2[0]; k.p[1] = c->p2[1]; k.q = c->q2;
        k.ke = c->ke; k.kn = c->kn;
        const int np = dh::grid_for(c->S);
        k.spmv = ctl(c, &e->st[M + m], c->p.olf_maxiter, c->p.olf_tol, false, true, c->part[0], np, c->part[1]);
        k.upd = ctl(c, &e->st[M + m], c->p.olf_maxiter, c->p.olf_tol, false, true, c->part[1], np, c->part[0]);
        e->h_ocg[m] = olf_cg_args(c, &e->st[M + m]);
        if (e->olf_kind[m] == 2) e->h_omg[m] = dh::OlfMgArgs{e->h_ocg[m], c->mg};
    }
    std::vector<int> jac(M, 0), mgm(M, 0), lock(M, 0);
    for (int m = 0; m < M; ++m) {
        jac[m] = on[m] && e->olf_kind[m] == 1;
        mgm[m] = on[m] && e->olf_kind[m] == 2;
        lock[m] = on[m] && e->olf_kind[m] == 0;
    }
    const bool any_jac = std::count(jac.begin(), jac.end(), 1) > 0, any_mg = std::count(mgm.begin(), mgm.end(), 1) > 0;
    const bool any_lock = std::count(lock.begin(), lock.end(), 1) > 0;
    if ((rc = upload_args(e, e->a_olf, e->h_olf)) || (rc = upload_args(e, e->a_k2, e->h_k2)) || (rc = set_active(e, on)))
        return rc;
    if ((any_jac && ((rc = upload_args(e, e->a_ocg, e->h_ocg)) || (rc = upload_args(e, e->olf_jac, jac)))) ||
        (any_mg && ((rc = upload_args(e, e->a_omg, e->h_omg)) || (rc = upload_args(e, e->olf_mgm, mgm)))))
        return rc;
    const MapRef r2 = use_map(e->cm2);
    dh::launch_batched(e->s, dh::BK_OLF_FACES, e->a_olf, r2.map, r2.n, e->active);
    dh::launch_batched(e->s, dh::BK_OLF_ASM, e->a_olf, r2.map, r2.n, e->active);
    if (any_mg) dh::launch_batched_olf_mgcg_block(e->s, e->a_omg, M, e->olf_mgm);
    if (any_jac) dh::launch_batched_olf_cg_block(e->s, e->a_ocg, M, e->olf_jac);
    EHIP(e, hipGetLastError());
    // the lockstep solve leaves every member's state on the host; without it, they are sent here
    if (any_lock) {
        if ((rc = set_active(e, lock)) || (rc = krylov_solve(e, true, lock, e->mem[0]->p.olf_maxiter, 2)) ||
            (rc = set_active(e, on)))
            return rc;
    } else {
        dh::launch_advance(e->s, e->it_base, 0, e->st, 2 * M, e->h_st);
        EHIP(e, hipGetLastError());
        if ((rc = wait(e))) return rc;
    }
    for (int m = 0; m < M; ++m) {
        if (!on[m]) continue;
        st[m].olf_iters = e->h_st[M + m].iter;
        st[m].olf_converged = e->h_st[M + m].conv;
        if (e->h_st[M + m].nan) st[m].nan_seen = 1;
    }
    {
        const MapRef r = use_map(e->cm2);
        dh::launch_batched(e->s, dh::BK_OLF_POST, e->a_olf, r.map, r.n, e->active);
    }
    if ((rc = reduce(e, true, 2, false))) return rc;
    for (int m = 0; m < M; ++m) {
        if (!on[m]) continue;
        st[m].outlet_discharge = e->h_red[2 * m];
        st[m].ring_outflow = e->h_red[2 * m + 1];
    }
    return DHARA_OK;
}

}  // namespace

extern "C" {

int dhara_ensemble_create(int32_t n, dhara_ctx* const* members, dhara_ensemble** out)
{
    if (n < 1 || !members || !out) return DHARA_E_ARG;
    *out = nullptr;
    dhara_ensemble* e = new dhara_ensemble;
    e->M = n;
    e->mem.assign(members, members + n);
    for (dhara_ctx* c : e->mem) {
        if (!c || !c->initialized) { delete e; return DHARA_E_STATE; }
        if (has_dirichlet(c)) { delete e; return DHARA_E_UNSUPPORTED; }
        // one batched Anderson pass serves every member: one depth for all
        if (c->p.picard_accel != e->mem[0]->p.picard_accel) { delete e; return DHARA_E_ARG; }
    }
    e->mixed = e->mem[0]->p.precision == DHARA_MIXED;
    for (dhara_ctx* c : e->mem) {
        if ((c->p.precision == DHARA_MIXED) != e->mixed) { delete e; return DHARA_E_ARG; }
        if (e->mixed && alloc_mixed(c)) { delete e; return DHARA_E_ALLOC; }
        if (hipStreamSynchronize(c->s) != hipSuccess) { delete e; return DHARA_E_DEVICE; }
    }
    if (hipStreamCreateWithFlags(&e->s, hipStreamNonBlocking) != hipSuccess) { delete e; return DHARA_E_DEVICE; }
    std::vector<dh::BlkMap> m3, m2;
    std::vector<double*> parts(n);
    std::vector<int> np3(n), np2(n);
    for (int m = 0; m < n; ++m) {
        dhara_ctx* c = e->mem[m];
        np3[m] = dh::grid_for(c->N);
        np2[m] = dh::grid_for(c->S);
        for (int b = 0; b < np3[m]; ++b) m3.push_back(dh::BlkMap{m, b, np3[m]});
        for (int b = 0; b < np2[m]; ++b) m2.push_back(dh::BlkMap{m, b, np2[m]});
        parts[m] = c->part[0];
    }
    e->nb3 = (int)m3.size();
    e->nb2 = (int)m2.size();
    // column preconditioner when every member asks for it (and its columns fit the kernel)
    e->line = true;
    for (dhara_ctx* c : e->mem)
        if (c->p.precond != DHARA_PRECOND_COLUMN || !dh::line_supported(c->g)) e->line = false;
    std::vector<dh::BlkMap> ml;
    if (e->line) {
        for (int m = 0; m < n; ++m) {
            dhara_ctx* c = e->mem[m];
            if (alloc_line(c, e->mixed) || hipStreamSynchronize(c->s) != hipSuccess) {
                dhara_ensemble_destroy(e);
                return DHARA_E_ALLOC;
            }
            const int nb = dh::line_blocks(c->g);
            for (int i = 0; i < nb; ++i) ml.push_back(dh::BlkMap{m, i, nb});
            e->line_nz = std::max(e->line_nz, c->g.nz);
        }
    }
    // otherwise the one-kernel Jacobi PCG when every member asks for it (32-bit plane offsets)
    e->one = !e->line;
    for (dhara_ctx* c : e->mem)
        if (c->p.krylov != DHARA_KRYLOV_ONE_KERNEL || (size_t)c->N * 8 >= (size_t(1) << 32)) e->one = false;
    std::vector<dh::BlkMap> mc1;
    if (e->one) {
        e->h_c1d.resize(n);
        e->h_c1f.resize(n);
        long tiles = 0;
        for (dhara_ctx* c : e->mem)
            tiles += (long)((c->g.nx + dh::kCg1BatchTx - 1) / dh::kCg1BatchTx) *
                     ((c->g.ny + dh::kCg1BatchTy - 1) / dh::kCg1BatchTy);
        e->c1_full = tiles > dh::kCg1FillTiles;
        // room for the finest policy the autotuner tries (a third of the planes per tile)
        std::vector<dh::BlkMap> finest;
        if (c1_map(e, 0, mc1) || c1_map(e, 3, finest)) {
            dhara_ensemble_destroy(e);
            return DHARA_E_UNSUPPORTED;
        }
        e->nb_c1 = (int)mc1.size();
        mc1.resize(std::max(mc1.size(), finest.size()), dh::BlkMap{0, 0, 1});
    }
    int rc = 0;
    if ((rc = ealloc(e, &e->map3, m3.size())) || (rc = ealloc(e, &e->map2, m2.size())) ||
        (rc = ealloc(e, &e->active, n)) || (rc = ealloc(e, &e->it_base, 1)) || (rc = ealloc(e, &e->st, 2 * n)) ||
        (rc = ealloc(e, &e->parts, n)) || (rc = ealloc(e, &e->np3, n)) || (rc = ealloc(e, &e->np2, n)) ||
        (rc = ealloc(e, &e->a_vg, n)) ||
        (rc = ealloc(e, &e->a_surf, n)) || (rc = ealloc(e, &e->a_asm, n)) || (rc = ealloc(e, &e->a_ref, n)) ||
        (rc = ealloc(e, &e->a_end, n)) || (rc = ealloc(e, &e->a_olf, n)) || (rc = ealloc(e, &e->a_k2, n)) ||
        (rc = ealloc(e, &e->a_ocg, n)) || (rc = ealloc(e, &e->a_omg, n)) || (rc = ealloc(e, &e->olf_jac, n)) ||
        (rc = ealloc(e, &e->olf_mgm, n))) {
        dhara_ensemble_destroy(e);
        return rc;
    }
    if (e->mixed) rc = ealloc(e, (dh::KrylovArgs<float>**)&e->a_k3, n);
    else rc = ealloc(e, (dh::KrylovArgs<double>**)&e->a_k3, n);
    if (!rc && e->one) {
        if (e->mixed) rc = ealloc(e, (dh::Cg1Args<float>**)&e->a_c1, n);
        else rc = ealloc(e, (dh::Cg1Args<double>**)&e->a_c1, n);
        if (!rc) rc = ealloc(e, &e->map_c1, mc1.size());
        if (!rc) rc = upload(e, e->map_c1, mc1);   // the first nb_c1 entries are live
    }
    if (!rc && e->line && !(rc = ealloc(e, &e->map_l, ml.size()))) rc = upload(e, e->map_l, ml);
    e->aa_depth = e->mem[0]->p.picard_accel;
    std::vector<dh::BlkMap> ma;
    if (!rc && e->aa_depth > 0) {
        for (int m = 0; m < n && !rc; ++m) {
            const int nb = dh::aa_blocks(e->mem[m]->g);
            for (int b = 0; b < nb; ++b) ma.push_back(dh::BlkMap{m, b, nb});
            rc = alloc_aa(e->mem[m]);
        }
        if (!rc) rc = ealloc(e, &e->map_aa, ma.size());
        if (!rc) rc = upload(e, e->map_aa, ma);
        if (!rc) rc = ealloc(e, &e->a_aa, n);
        e->h_aa.resize(n);
    }
    if (rc) { dhara_ensemble_destroy(e); return rc; }
    e->stage_size = std::max<size_t>(size_t(1) << 20, (size_t)n * 8192);
    if (hipHostMalloc((void**)&e->h_flags, (size_t)dhara_ensemble::kFlagSlots * n * sizeof(int)) != hipSuccess ||
        hipHostMalloc((void**)&e->stage, e->stage_size) != hipSuccess ||
        hipHostMalloc((void**)&e->h_st, 2 * n * sizeof(dh::PcgState)) != hipSuccess ||
        hipHostMalloc((void**)&e->h_red, (size_t)n * dh::kMaxSums * sizeof(double)) != hipSuccess) {
        dhara_ensemble_destroy(e);
        return DHARA_E_ALLOC;
    }
    if ((rc = upload(e, e->map3, m3)) || (rc = upload(e, e->map2, m2)) || (rc = upload(e, e->parts, parts)) ||
        (rc = upload(e, e->np3, np3)) || (rc = upload(e, e->np2, np2))) {
        dhara_ensemble_destroy(e);
        return rc;
    }
    e->act.assign(n, -1);   // matches no active set: the first set_active records one
    if ((rc = init_cmap(e, e->cm3, e->map3, m3)) || (rc = init_cmap(e, e->cm2, e->map2, m2)) ||
        (rc = init_cmap(e, e->cml, e->map_l, ml))) {
        dhara_ensemble_destroy(e);
        return rc;
    }
    if ((rc = init_cmap(e, e->cmaa, e->map_aa, ma))) { dhara_ensemble_destroy(e); return rc; }
    std::vector<dh::PcgState> zero(2 * n);
    if ((rc = upload(e, e->st, zero))) { dhara_ensemble_destroy(e); return rc; }
    e->h_vg.resize(n); e->h_surf.resize(n); e->h_asm.resize(n); e->h_ref.resize(n); e->h_end.resize(n);
    e->h_olf.resize(n); e->h_k3d.resize(n); e->h_k3f.resize(n); e->h_k2.resize(n); e->h_ocg.resize(n);
    e->h_omg.resize(n);
    e->olf_kind.assign(n, 0);
    for (int m = 0; m < n; ++m) {
        dhara_ctx* c = e->mem[m];
        if (c->S > dh::kOlfBlockCells) continue;
        const int op = c->p.olf_precond;
        e->olf_kind[m] = (op == DHARA_OLF_PRECOND_MG || op == DHARA_OLF_PRECOND_MG_BLOCK) ? 2 : 1;
        if (e->olf_kind[m] == 2 && (rc = ensure_mg(c))) {
            dhara_ensemble_destroy(e);
            return rc;
        }
    }
    *out = e;
    return DHARA_OK;
}

int dhara_ensemble_set_graph(dhara_ensemble* e, int32_t on)
{
    if (!e) return DHARA_E_ARG;
    e->use_graph = on != 0;
    return DHARA_OK;
}

const char* dhara_ensemble_last_error(const dhara_ensemble* e) { return e ? e->err.c_str() : "null ensemble"; }

int dhara_ensemble_step(dhara_ensemble* e, int32_t nsteps, dhara_step_stats* stats)
{
    if (!e || nsteps < 0) return DHARA_E_ARG;
    for (int s = 0; s < nsteps; ++s) {
        const auto t0 = std::chrono::steady_clock::now();
        std::vector<dhara_step_stats> st(e->M);
        for (auto& x : st) std::memset(&x, 0, sizeof(x));
        int rc = subsurface_step(e, st);
        if (rc == DHARA_OK) rc = overland_step(e, st);
        const double ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
        for (int m = 0; m < e->M; ++m) {
            st[m].wall_ms = ms;
            if (stats) stats[(size_t)s * e->M + m] = st[m];
        }
        if (rc) return rc;
        for (int m = 0; m < e->M; ++m)
            if (st[m].nan_seen) return eset(e, DHARA_E_NUMERIC, "NaN/Inf in member " + std::to_string(m));
    }
    return DHARA_OK;
}

// Ensemble-level tile autotuner of the batched one-kernel PCG: planes per tile = all, 1/2 or 1/3
// of each member's columns (the 32 x 8 tile is fixed by the batched kernel), 3 + 10 launches of
// every member's iteration kernel on scratch outputs and a never-converging scratch state; the
// members' own arrays are only read.  Keeps the fastest (a later policy must be 3 % faster).
int dhara_ensemble_autotune(dhara_ensemble* e, double* best_us, int32_t* planes_div)
{
    if (!e) return DHARA_E_ARG;
    if (!e->one)
        return eset(e, DHARA_E_UNSUPPORTED, "autotune: members do not use the one-kernel Jacobi PCG (the column "
                                            "form's column kernel and untiled SpMV have no tile to tune)");
    const int M = e->M;
    const size_t es = e->mixed ? 4 : 8;
    std::vector<void*> scratch;
    auto cleanup = [&]() {
        (void)hipStreamSynchronize(e->s);
        for (void* v : scratch) (void)hipFree(v);
    };
    dh::PcgState* st = nullptr;
    int* it1 = nullptr;
    std::vector<void*> xs(M), r0s(M), r1s(M), ps(M), qs(M);   // x, r[0], r[1], p[0], p[1]
    {
        void* v = nullptr;
        if (hipMalloc(&v, M * sizeof(dh::PcgState)) != hipSuccess) return eset(e, DHARA_E_ALLOC, "hipMalloc");
        scratch.push_back(v);
        st = (dh::PcgState*)v;
        if (hipMalloc(&v, sizeof(int)) != hipSuccess) { cleanup(); return eset(e, DHARA_E_ALLOC, "hipMalloc"); }
        scratch.push_back(v);
        it1 = (int*)v;
        for (int m = 0; m < M; ++m) {
            const size_t nb = (size_t)e->mem[m]->N * es;
            for (void** slot : {&xs[m], &r0s[m], &r1s[m], &ps[m], &qs[m]}) {
                if (hipMalloc(slot, nb) != hipSuccess) { cleanup(); return eset(e, DHARA_E_ALLOC, "hipMalloc"); }
                scratch.push_back(*slot);
                (void)hipMemsetAsync(*slot, 0, nb, e->s);
            }
        }
    }
    dh::PcgState tune{};
    tune.rz[0] = tune.rz[1] = 1.0;
    tune.pi[0] = tune.pi[1] = 1.0;
    tune.tol2 = -1.0;
    std::vector<dh::PcgState> tunes(M, tune);
    std::vector<double> ones(5 * dh::kMaxBlocks, 1.0);
    const int one = 1;
    EHIP(e, hipMemcpyAsync(st, tunes.data(), M * sizeof(dh::PcgState), hipMemcpyHostToDevice, e->s));
    EHIP(e, hipMemcpyAsync(it1, &one, sizeof(int), hipMemcpyHostToDevice, e->s));
    for (dhara_ctx* c : e->mem)
        for (int b = 0; b < 2; ++b)
            for (int v = 0; v < 5; ++v)
                EHIP(e, hipMemcpyAsync(c->part[b] + v * dh::kMaxBlocks, ones.data(), dh::kMaxBlocks * sizeof(double),
                                       hipMemcpyHostToDevice, e->s));
    std::vector<int> all(M, 1);
    int rc = set_active(e, all);
    if (rc) { cleanup(); return rc; }
    hipEvent_t e0, e1;
    EHIP(e, hipEventCreate(&e0));
    EHIP(e, hipEventCreate(&e1));
    const int old_div = e->kc_div;
    // 0: the members' own tiles, which split a small ensemble's columns finer than any policy; they stay
    // unless a policy is 3 % faster
    float best = 1e30f, best_policy = 1e30f;
    int keep = 0, best_div = 1;
    for (int div : {0, 1, 2, 3}) {
        std::vector<dh::BlkMap> map;
        if ((rc = c1_map(e, div, map))) break;
        e->kc_div = div;
        build_c1(e, false);
        for (int m = 0; m < M; ++m) {   // scratch outputs and state
            dhara_ctx* c = e->mem[m];
            if (e->mixed) {
                dh::Cg1Args<float>& a = e->h_c1f[m];
                a.r[0] = (float*)r0s[m]; a.r[1] = (float*)r1s[m]; a.p[0] = (float*)ps[m]; a.p[1] = (float*)qs[m]; a.x = (float*)xs[m];
                a.ctl.st = st + m;
            } else {
                dh::Cg1Args<double>& a = e->h_c1d[m];
                a.r[0] = (double*)r0s[m]; a.r[1] = (double*)r1s[m]; a.p[0] = (double*)ps[m]; a.p[1] = (double*)qs[m]; a.x = (double*)xs[m];
                a.ctl.st = st + m;
            }
            (void)c;
        }
        if ((rc = upload_c1(e)) || (rc = upload(e, e->map_c1, map))) break;
        float ms = 0.f;
        for (int rep = 0; rep < 13; ++rep) {
            if (rep == 3) EHIP(e, hipEventRecord(e0, e->s));
            // iteration 1 every time: reads part[0] (the ones, never written) and state slot 0,
            // writes part[1] and slot 1, so every launch does the same full iteration
            dh::launch_batched_cg1(e->s, e->mixed, e->a_c1, e->map_c1, (int)map.size(), e->active, it1, 0);
        }
        EHIP(e, hipEventRecord(e1, e->s));
        EHIP(e, hipEventSynchronize(e1));
        EHIP(e, hipGetLastError());
        EHIP(e, hipEventElapsedTime(&ms, e0, e1));
        const float us = ms * 1e3f / 10.f;
        if (us < 0.97f * best || best >= 1e29f) { best = us; keep = div; }
        if (div > 0 && (us < 0.97f * best_policy || best_policy >= 1e29f)) { best_policy = us; best_div = div; }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    cleanup();
    if (rc) { e->kc_div = old_div; return rc; }
    // keep the winner: its tile map (the solves rebuild their arguments from the members)
    e->kc_div = keep;
    std::vector<dh::BlkMap> map;
    if ((rc = c1_map(e, keep, map)) || (rc = upload(e, e->map_c1, map))) return rc;
    e->nb_c1 = (int)map.size();
    drop_graphs(e, true);   // their launches carry the old grid size: captured again at the next solve
    if (best_us) *best_us = best;
    if (planes_div) *planes_div = best_div;
    return DHARA_OK;
}

int dhara_ensemble_destroy(dhara_ensemble* e)
{
    if (!e) return DHARA_OK;
    if (e->s) (void)hipStreamSynchronize(e->s);
    drop_graphs(e, false);
    for (void* v : e->allocs) (void)hipFree(v);
    if (e->h_flags) (void)hipHostFree(e->h_flags);
    if (e->stage) (void)hipHostFree(e->stage);
    if (e->h_st) (void)hipHostFree(e->h_st);
    if (e->h_red) (void)hipHostFree(e->h_red);
    if (e->s) (void)hipStreamDestroy(e->s);
    delete e;
    return DHARA_OK;
}

}  // extern "C"

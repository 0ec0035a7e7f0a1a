// noalloc.hip -- the allocation-free variant of dhara_overland_precond.
//
// For callers that cannot allocate device memory (code under HIP graph capture, tight serving
// loops, harnesses that forbid hipMalloc): r and z are device pointers, and the multigrid
// hierarchy the V-cycle works in -- level weights, right-hand sides, iterates and the dense
// inverse of the coarsest level -- lives in `scratch`, a file-scope device array of fixed size.
// Each device the library runs on holds its own copy until the process ends.  Every call on one
// device shares that device's copy and leaves the last call's contents in it: the hierarchy is
// cleared by a fill kernel at the start of every call, and calls that overlap on one device race.
#include <hip/hip_runtime.h>

#include <mutex>
#include <string>

#include "../../include/dhara_hip.h"
#include "ctx.h"

namespace {

constexpr size_t kScratchDoubles = DHARA_NOALLOC_SCRATCH_BYTES / sizeof(double);
constexpr size_t kAlign = 32;   // doubles: every array of the hierarchy starts on 256 bytes

__device__ __align__(256) double scratch[kScratchDoubles];

// Device address of each device's copy of `scratch` (the array's name in host code is only a
// host-side stand-in), taken once per device with that device current.
constexpr int kMaxDevices = 64;
double* g_scratch[kMaxDevices] = {};
std::mutex g_scratch_mu;

__global__ void k_fill_zero(double* p, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = 0.0;
}

size_t round_up(size_t n) { return (n + kAlign - 1) / kAlign * kAlign; }

}  // namespace

namespace dhc {

int noalloc_setup(dhara_ctx* c)
{
    if (c->dev < 0 || c->dev >= kMaxDevices) return set_err(c, DHARA_E_DEVICE, "device index out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch[c->dev]) return DHARA_OK;
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
        return set_err(c, DHARA_E_DEVICE, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    g_scratch[c->dev] = static_cast<double*>(p);
    return DHARA_OK;
}

}  // namespace dhc

using namespace dhc;

int dhara_overland_precond_noalloc(dhara_ctx* c, const double* r, double* z)
{
    if (!c || !r || !z) return DHARA_E_ARG;
    double* base = g_scratch[(c->dev >= 0 && c->dev < kMaxDevices) ? c->dev : 0];
    if (!base) return set_err(c, DHARA_E_STATE, "no scratch address for this device");
    // the hierarchy of ensure_mg down to the exactly solved level, laid out in the scratch:
    // level 0 keeps the context's diagonal D2 and residual r2 and writes its result into z
    int dims[dh::kMgMaxLevels][2];
    const int nl = dh::mg_levels(c->grid.nx, c->grid.ny, dims);
    if (nl > dh::kMgMaxLevels) return set_err(c, DHARA_E_UNSUPPORTED, "surface grid too large for the multigrid");
    dh::MgHier h{};
    h.nlev = nl;
    for (int l = 0; l < nl; ++l) {
        h.lv[l].nx = dims[l][0];
        h.lv[l].ny = dims[l][1];
    }
    h.le = dh::mg_exact_level(h);
    h.nlev = h.le + 1;   // levels below the exact one are never touched
    size_t used = 0;
    auto take = [&](size_t n) {
        double* p = base + used;
        used += round_up(n);
        return p;
    };
    for (int l = 0; l <= h.le; ++l) {
        dh::MgLevel& L = h.lv[l];
        const size_t n = (size_t)L.nx * L.ny;
        if (used + 6 * round_up(n) > kScratchDoubles) break;   // reported below
        L.we = take(n);
        L.wn = take(n);
        L.x = take(n);
        if (l == 0) {
            L.d = c->D2;
            L.b = c->r2;
            L.y = z;
        } else {
            L.d = take(n);
            L.b = take(n);
            L.y = take(n);
        }
    }
    const size_t ninv = (size_t)dh::kMgExactCells * dh::kMgExactCells;
    size_t need = 0;
    for (int l = 0; l <= h.le; ++l) need += (l == 0 ? 3 : 6) * round_up((size_t)h.lv[l].nx * h.lv[l].ny);
    need += round_up(ninv);
    if (need > kScratchDoubles)
        return set_err(c, DHARA_E_ARG,
                       "surface of " + std::to_string(c->grid.nx) + " x " + std::to_string(c->grid.ny) +
                           " cells needs " + std::to_string(need * sizeof(double)) +
                           " bytes of multigrid scratch, more than the " +
                           std::to_string(DHARA_NOALLOC_SCRATCH_BYTES) + " the allocation-free entry point has");
    h.inv = take(ninv);
    const unsigned grid = (unsigned)std::min<size_t>((used + 255) / 256, 4096);
    hipLaunchKernelGGL(k_fill_zero, dim3(grid), dim3(256), 0, c->s, base, used);
    dh::OlfArgs a = olf_args(c);
    dh::launch_olf_faces(c->s, a);
    dh::launch_olf_assemble(c->s, a);
    dh::launch_mg_setup(c->s, c->g2, c->ke, c->kn, h);
    HIPCHK(c, hipMemcpyAsync(c->r2, r, (size_t)c->S * sizeof(double), hipMemcpyDeviceToDevice, c->s));
    dh::launch_mg_vcycle(c->s, h);
    LAUNCHCHK(c);
    HIPCHK(c, hipStreamSynchronize(c->s));
    return DHARA_OK;
}

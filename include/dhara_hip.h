/*
 * dhara_hip.h -- C-ABI of the MI355X (gfx950) integrated surface/subsurface flow solver.
 *
 * Plain C: fixed-width integers, doubles, opaque handles.  No HIP, torch or C++ types cross
 * this boundary.  Every function returns 0 on success or a negative DHARA_E* code; the text
 * of the last error of a context is returned by dhara_last_error().  Nothing here calls
 * exit(); the reference terminated the process on any device error
 * (src/device.cu:162-171 CheckCudaCall, include/main.h:58-68 cudaCheckError).
 *
 * Units are SI throughout: psi [m], alpha [1/m], K [m/s], dt [s], rain/evaporation/
 * transpiration rates [m/s].  The reference kept psi in m but alpha in 1/cm, dt in hours
 * and K in m per time step (include/devconst.h:6-21, src/global.cu:79,96, src/host.cc:53);
 * the reference-named shims in dhara_shim.h do that conversion.
 *
 * Layout (identical to the reference, so uploads are plain copies):
 *   3D cell (i,j,k):   k*nx*ny + j*nx + i, k = 0 is the TOP layer, z positive downward
 *                      (src/subsurface.cu:401-410)
 *   surface (i,j):     j*nx + i
 *   W/E face arrays:   k*ny + j;  S/N face arrays: k*nx + i;  top/bottom: j*nx + i
 *                      (src/subsurface.cu:139-142)
 *
 * Threading: one context is used by one host thread at a time; it owns one HIP stream and
 * all device memory it needs.  Separate contexts are independent.  Calls are synchronous
 * on return.
 */
#ifndef DHARA_HIP_H
#define DHARA_HIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define DHARA_ABI_VERSION 4

/* ---- status codes ---------------------------------------------------------------- */
#define DHARA_OK            0
#define DHARA_E_ARG        -1   /* bad argument / size mismatch                        */
#define DHARA_E_DEVICE     -2   /* HIP runtime error                                    */
#define DHARA_E_ALLOC      -3   /* device or host allocation failed                     */
#define DHARA_E_STATE      -4   /* call made in the wrong state (e.g. step before init) */
#define DHARA_E_NUMERIC    -5   /* NaN/Inf detected in the state                        */
#define DHARA_E_UNSUPPORTED -6  /* option not supported by this library                 */

/* ---- enumerations ---------------------------------------------------------------- */
/* Picard stopping rule.  src/subsurface.cu:762-780: PICARD_METHOD 0 uses
 * max|(psi^{m+1}-psi^m)/psi^{m+1}|, PICARD_METHOD 1 the same on theta. */
#define DHARA_PICARD_ABS_PSI   0   /* max|psi^{m+1}-psi^m| [m]  (default)               */
#define DHARA_PICARD_REL_PSI   1   /* reference PICARD_METHOD = 0                        */
#define DHARA_PICARD_REL_THETA 2   /* reference PICARD_METHOD = 1                        */

/* Linear-solver precision of the subsurface solve. */
#define DHARA_FP64   0   /* Jacobi-PCG in FP64 end to end                                */
#define DHARA_MIXED  1   /* FP32 Jacobi-PCG inner solves + FP64 residual refinement      */

/* theta carried to the next step.  The reference copies theta^{n+1,m} (the iterate
 * BEFORE the last solve) into theta^n (src/subsurface.cu:839). */
#define DHARA_THETA_CARRY_CONSISTENT 0   /* theta^n <- theta(psi^{n+1})  (default)       */
#define DHARA_THETA_CARRY_REFERENCE  1   /* theta^n <- theta^{n+1,m}     (reference)      */

/* Top boundary of the subsurface.  The reference always derives it from the surface
 * (EstimateFluxes + IdentifyTopBoundary, src/global.cu:172-257, which force type 1 on every
 * Picard iteration) and updates the ponding depth from it (src/subsurface.cu:465-491). */
#define DHARA_TOP_SURFACE    0   /* reference coupling (default)                          */
#define DHARA_TOP_PRESCRIBED 1   /* use the uploaded DHARA_F_BCTYPE_T/BCPSI_T/BCQ_T; the
                                    ponding depth is left unchanged                       */

/* Preconditioner of the overland CG (the reference's CUSP CG had none, src/overland.cu:410),
 * and the form of the solve.  The *_BLOCK forms solve a surface of at most 128 x 128 cells in
 * one workgroup and one launch (the form a batched ensemble uses for such members, so that a
 * member stepped alone can match it bit for bit; for a single model the other forms are
 * faster); larger surfaces take the grid-wide form of the same preconditioner.  Multigrid on a single
 * model's surface of up to about 64 x 64 cells runs on chip in one workgroup, else grid-wide. */
#define DHARA_OLF_PRECOND_JACOBI       0
#define DHARA_OLF_PRECOND_MG           1   /* aggregation-multigrid V-cycle (same solution, far
                                              fewer iterations on ponded surfaces)            */
#define DHARA_OLF_PRECOND_MG_BLOCK     2
#define DHARA_OLF_PRECOND_JACOBI_BLOCK 3

/* Kernel structure of the subsurface Jacobi-PCG (same method, same stopping rule)          */
#define DHARA_KRYLOV_TWO_KERNEL 0   /* Hestenes-Stiefel recurrences, the reference's CUSP CG:
                                       two launches per iteration                           */
#define DHARA_KRYLOV_ONE_KERNEL 1   /* single-reduction recurrences (Chronopoulos-Gear): one
                                       launch per iteration (default); without Dirichlet rows
                                       only, the two-kernel form is used otherwise          */

/* Preconditioner of the subsurface PCG (the reference ran unpreconditioned BiCGStab,
 * src/subsurface.cu:750-751; the converged solution is the same, ||r|| <= lin_tol ||b||)    */
#define DHARA_PRECOND_JACOBI 0      /* diagonal scaling (default)                            */
#define DHARA_PRECOND_COLUMN 1      /* exact solve of each column's vertical tridiagonal part
                                       (the stiff dz^-2 couplings): ~4x fewer iterations on
                                       thin layers; two-kernel recurrences with a column-solve
                                       kernel; needs nz <= 64 and no Dirichlet rows (Jacobi is
                                       used otherwise)                                      */

/* State initialisation. */
#define DHARA_INIT_FROM_THETA 0   /* psi <- vG^-1(theta), then theta,K,C <- vG(psi)
                                     (src/device.cu:323-330, src/global.cu:289)          */
#define DHARA_INIT_FROM_PSI   1   /* theta,K,C <- vG(psi)                                 */

/* Boundary types (src/subsurface.cu:126-353): 0 = Dirichlet (pressure head), else flux. */
#define DHARA_BC_DIRICHLET 0
#define DHARA_BC_FLUX      1

/* ---- field identifiers ------------------------------------------------------------ */
enum dhara_field {
    /* 3D cell fields, n = nx*ny*nz */
    DHARA_F_PSI = 0,        /* pressure head psi^n [m]                      (in/out)   */
    DHARA_F_THETA,          /* water content theta^n [-]                    (in/out)   */
    DHARA_F_KSAT,           /* saturated conductivity [m/s]                 (in)       */
    DHARA_F_ALPHA,          /* van Genuchten alpha per cell [1/m]  (optional, in)      */
    DHARA_F_NVG,            /* van Genuchten n per cell [-]        (optional, in)      */
    DHARA_F_K,              /* unsaturated conductivity K(psi) [m/s]        (out)      */
    DHARA_F_C,              /* specific moisture capacity dtheta/dpsi [1/m] (out)      */
    /* surface fields, n = nx*ny */
    DHARA_F_ZTOPO,          /* ground elevation z [m]                       (in)       */
    DHARA_F_MANNING,        /* Manning n [s m^-1/3]                         (in)       */
    DHARA_F_PONDING,        /* ponding / overland water depth h [m]         (in/out)   */
    DHARA_F_WATERELEV,      /* water surface elevation H = h + z [m]        (out)      */
    DHARA_F_RAIN,           /* rain (throughfall) rate [m/s]                (in)       */
    DHARA_F_EVAP,           /* soil evaporation rate [m/s]                  (in)       */
    DHARA_F_TRANSP,         /* transpiration rate [m/s]                     (in)       */
    DHARA_F_QTOP,           /* infiltration flux into layer 0 [m/s], +down  (out)      */
    DHARA_F_QBOT,           /* free-drainage flux out of the bottom [m/s]   (out)      */
    DHARA_F_HPOTEN,         /* potential surface head [m]                   (out)      */
    DHARA_F_QCAPA,          /* infiltration capacity [m/s]                  (out)      */
    /* boundary values, n = size of the face (W/E: ny*nz, S/N: nx*nz, T/B: nx*ny) */
    DHARA_F_BCPSI_W, DHARA_F_BCPSI_E, DHARA_F_BCPSI_S, DHARA_F_BCPSI_N,
    DHARA_F_BCPSI_T, DHARA_F_BCPSI_B,
    DHARA_F_BCQ_W, DHARA_F_BCQ_E, DHARA_F_BCQ_S, DHARA_F_BCQ_N,
    DHARA_F_BCQ_T, DHARA_F_BCQ_B,
    /* root-uptake distribution: n = nroot_groups*nz, row g is the profile of group g */
    DHARA_F_ROOT,
    /* integer fields (dhara_upload_field_i32 / dhara_download_field_i32) */
    DHARA_F_BCTYPE_W, DHARA_F_BCTYPE_E, DHARA_F_BCTYPE_S, DHARA_F_BCTYPE_N,
    DHARA_F_BCTYPE_T, DHARA_F_BCTYPE_B,
    DHARA_F_PROCMAP,        /* surface cell -> root group (reference: MPI rank map)    */
    DHARA_F__COUNT
};

/* ---- structures -------------------------------------------------------------------- */
typedef struct dhara_grid {
    int32_t nx, ny, nz;
    int32_t nroot_groups;   /* rows of DHARA_F_ROOT (reference: MPI process count)     */
    double  dx, dy, dz;     /* [m]                                                      */
} dhara_grid;

typedef struct dhara_params {
    double  dt;                                   /* time step [s]                      */
    /* Mualem-van Genuchten scalars (per-cell alpha/n override when uploaded)           */
    double  theta_s, theta_r, alpha, n_vg, Ss, porosity;
    /* Picard loop (src/subsurface.cu:715-790)                                          */
    int32_t picard_maxiter, picard_rule;
    double  picard_tol, am;
    /* subsurface linear solve                                                          */
    int32_t lin_maxiter, precision;
    double  lin_tol;                              /* ||r||_2 <= lin_tol * ||b||_2         */
    int32_t refine_maxiter, inner_maxiter;        /* DHARA_MIXED: max FP64 reliable updates
                                                     per solve, max FP32 iterations        */
    double  inner_tol;                            /* DHARA_MIXED: FP32 residual reduction
                                                     between two FP64 reliable updates     */
    /* overland flow (src/overland.cu:387-419, include/devconst.h:25-28)                 */
    int32_t overland, olf_maxiter;
    double  olf_tol;
    double  hmin, delta, K0;
    /* compatibility switches                                                           */
    int32_t theta_carry;                          /* DHARA_THETA_CARRY_*                  */
    int32_t dirichlet_face_quirk;                 /* 1: reference's opposite-face K in
                                                     inner Dirichlet rows
                                                     (src/subsurface.cu:223,259,294,328) */
    int32_t top_bc;                               /* DHARA_TOP_*                          */
    int32_t olf_precond;                          /* DHARA_OLF_PRECOND_* (overland CG)    */
    int32_t krylov;                               /* DHARA_KRYLOV_* (subsurface PCG)      */
    int32_t precond;                              /* DHARA_PRECOND_* (subsurface PCG)     */
    /* Picard update.  0: the reference's psi^m <- am psi^m + (1-am) psi^{m+1}
     * (src/subsurface.cu:450-461).  1..DHARA_PICARD_ACCEL_MAX: Anderson acceleration of the
     * same map over that many previous iterations, with damping 1-am (Walker & Ni 2011); the
     * fixed point and the stopping test are unchanged.  Not in the reference. */
    int32_t picard_accel;
} dhara_params;

#define DHARA_PICARD_ACCEL_MAX 5

typedef struct dhara_step_stats {
    int32_t picard_iters, picard_converged;
    int32_t lin_iters;          /* Krylov iterations of the subsurface solves (all sweeps) */
    int32_t lin_converged;      /* 1 if every linear solve of the step converged         */
    int32_t refine_sweeps;      /* FP64 residual sweeps (DHARA_MIXED)                      */
    int32_t olf_iters, olf_converged;
    int32_t nan_seen;
    double  picard_delta;       /* last Picard increment (rule units)                      */
    double  mb_ref;             /* reference mass-balance formula, src/subsurface.cu:825 [m] */
    double  storage_change;     /* sum of storage change over the domain [m^3]            */
    double  boundary_inflow;    /* net inflow through all faces minus sinks, times dt [m^3] */
    double  mb_rel;             /* |storage_change - boundary_inflow| / scale              */
    double  outlet_discharge;   /* overland discharge into the x = 0 edge [m^3/s]          */
    double  ring_outflow;       /* overland discharge into the whole Dirichlet ring [m^3/s] */
    double  wall_ms;            /* wall time of the call                                   */
} dhara_step_stats;

/* Device-time profile of the subsurface Krylov kernels (measurement hook; no reference
 * counterpart).  Only launches that did work are counted. */
typedef struct dhara_kernel_profile {
    int64_t spmv_launches;      /* p-update + stencil SpMV + (p, Ap) kernel                  */
    double  spmv_ms;            /* summed device time of those launches                      */
    double  spmv_bytes;         /* algorithmic HBM bytes of one launch                       */
    int64_t update_launches;    /* x/r update + (r, M^-1 r), (r, r) kernel                   */
    double  update_ms;
    double  update_bytes;
    int32_t elem_bytes;         /* 8 (FP64) or 4 (FP32 inner solves) of the profiled solves  */
    int32_t reserved;
    int64_t aa_launches;        /* Anderson Picard passes (k_picard_next) that ran            */
    double  aa_ms;              /* summed device time of those passes                         */
    double  aa_bytes;           /* summed algorithmic HBM bytes of those passes                */
} dhara_kernel_profile;

typedef struct dhara_ctx dhara_ctx;

/* ---- defaults ------------------------------------------------------------------------ */
/* Parameter defaults: homogeneous loam (Carsel & Parrish), Picard 1e-6 m absolute,
 * Jacobi-PCG to 1e-12, overland constants of include/devconst.h:25-28 in SI. */
static inline void dhara_params_defaults(dhara_params* p)
{
    p->dt = 60.0;
    p->theta_s = 0.43; p->theta_r = 0.078; p->alpha = 3.6; p->n_vg = 1.56;
    p->Ss = 1e-5; p->porosity = 0.43;
    p->picard_maxiter = 20; p->picard_rule = DHARA_PICARD_ABS_PSI;
    p->picard_tol = 1e-6; p->am = 0.0;
    p->lin_maxiter = 2000; p->precision = DHARA_FP64; p->lin_tol = 1e-12;
    p->refine_maxiter = 16; p->inner_maxiter = 2000; p->inner_tol = 1e-5;
    p->overland = 1; p->olf_maxiter = 2000; p->olf_tol = 1e-12;
    p->hmin = 1e-5; p->delta = 1e-7; p->K0 = 1e-5;
    p->theta_carry = DHARA_THETA_CARRY_CONSISTENT;
    p->dirichlet_face_quirk = 1;
    p->top_bc = DHARA_TOP_SURFACE;
    p->olf_precond = DHARA_OLF_PRECOND_MG;
    p->krylov = DHARA_KRYLOV_ONE_KERNEL;
    p->precond = DHARA_PRECOND_JACOBI;
    p->picard_accel = 0;
}

/* ---- lifecycle ------------------------------------------------------------------------ */
/* Replaces AllocateMemoryFlowModel's device half (src/numerical.cc:127-188) and the CUSP
 * containers of ResizeCuspMemory (src/device.cu:27-72). */
int dhara_create(const dhara_grid* grid, const dhara_params* params, dhara_ctx** out);
/* Replaces FreeDeviceMemory (src/numerical.cc:279-336). */
int dhara_destroy(dhara_ctx* ctx);
const char* dhara_last_error(const dhara_ctx* ctx);
int dhara_abi_version(void);
/* Writes "<device name> <gcnArchName> CUs=<n>" into buf. */
int dhara_device_info(char* buf, size_t n);

int dhara_set_params(dhara_ctx* ctx, const dhara_params* params);
int dhara_get_params(const dhara_ctx* ctx, dhara_params* params);
int dhara_set_precision(dhara_ctx* ctx, int32_t precision);

/* ---- data movement ------------------------------------------------------------------- */
/* Replace the cudaMemcpy H2D block of CopyDataToDevice (src/device.cu:223-321) and the
 * root-density H2D of GatherRootDensityToMasterAndFilter (src/host.cc:256-257). */
int dhara_upload_field(dhara_ctx* ctx, int32_t field, const double* host, size_t n);
int dhara_upload_field_i32(dhara_ctx* ctx, int32_t field, const int32_t* host, size_t n);
/* Replace SaveModelResults' D2H (src/io.cc:866-901) and SubsurfaceFlowModel's per-step
 * psiout/thetaout copies (src/subsurface.cu:842-846; here only on request). */
int dhara_download_field(dhara_ctx* ctx, int32_t field, double* host, size_t n);
int dhara_download_field_i32(dhara_ctx* ctx, int32_t field, int32_t* host, size_t n);
/* Device-to-device variants: `dev` is a device pointer of the same element type. */
int dhara_upload_field_device(dhara_ctx* ctx, int32_t field, const void* dev, size_t n);
int dhara_download_field_device(dhara_ctx* ctx, int32_t field, void* dev, size_t n);

/* Per-group forcing (reference: one value per MPI rank gathered to rank 0): field[cell] =
 * values[procmap[cell]] for a surface field (DHARA_F_RAIN, _EVAP, _TRANSP).  Replaces the
 * H2D copy + SendFluxDataToGrids of GatherFluxesDomain (src/subsurface.cu:643-659,
 * 364-378); `values` has nroot_groups entries (host memory). */
int dhara_scatter_group_field(dhara_ctx* ctx, int32_t field, const double* values, size_t ngroups);

/* psi <-> theta initialisation: CopyDataToDevice's vanGenuchtenInverse
 * (src/device.cu:323-330) followed by PreRunningFlowModel (src/global.cu:270-296). */
int dhara_init_state(dhara_ctx* ctx, int32_t mode);

/* ---- time stepping -------------------------------------------------------------------- */
/* One subsurface step: SubsurfaceFlowModel (src/subsurface.cu:686-847). */
int dhara_subsurface_step(dhara_ctx* ctx, dhara_step_stats* stats);
/* One overland step: OverlandFlowModel (src/overland.cu:387-419). */
int dhara_overland_step(dhara_ctx* ctx, dhara_step_stats* stats);
/* nsteps coupled steps (subsurface then overland when params.overland != 0): the body of
 * RunCoupledFlowModel's time loop (src/device.cu:426-469) without the canopy model.
 * `stats` (may be NULL) receives nsteps records. */
int dhara_step(dhara_ctx* ctx, int32_t nsteps, dhara_step_stats* stats);

/* ---- measurement ------------------------------------------------------------------------ */
/* Turn HIP-event timing of the subsurface Krylov kernels on (1) or off (0).  The events are
 * recorded on the context's stream around every SpMV / update launch. */
int dhara_profile_enable(dhara_ctx* ctx, int32_t on);
/* Accumulated profile since the last read; resets the accumulators. */
int dhara_profile_read(dhara_ctx* ctx, dhara_kernel_profile* out);

/* ---- tuning ------------------------------------------------------------------------------ */
/* Tile shape of the LDS-tiled subsurface SpMV kernel for one precision (elem_bytes 8: FP64
 * solves, 4: FP32 inner solves).  tx = 0 selects the untiled one-cell-per-thread kernel.
 * Supported (tx, ty): (32,8) (64,4) (16,16) (32,4) (64,8); kc >= 1 planes per block.  A tile set here
 * is also the assembly's (FP64) and the start-up's of the one-kernel PCG; without one, each kernel has
 * a default of its own, and dhara_get_tile gives the SpMV's. */
int dhara_set_tile(dhara_ctx* ctx, int32_t elem_bytes, int32_t tx, int32_t ty, int32_t kc);
int dhara_get_tile(const dhara_ctx* ctx, int32_t elem_bytes, int32_t* tx, int32_t* ty, int32_t* kc);
/* Tile of the one-kernel PCG (DHARA_KRYLOV_ONE_KERNEL): (tx, ty) in (32,8) (16,16) (32,16)
 * (64,8), kc >= 1 planes per tile, grid = 0 (one block per tile) or a multiple of 8 capping
 * the blocks, which then loop over tiles.  No reference counterpart (tuning hook). */
int dhara_set_krylov_tile(dhara_ctx* ctx, int32_t elem_bytes, int32_t tx, int32_t ty, int32_t kc, int32_t grid);
int dhara_get_krylov_tile(const dhara_ctx* ctx, int32_t elem_bytes, int32_t* tx, int32_t* ty, int32_t* kc,
                          int32_t* grid);
/* Times the candidate tile shapes, the one in use first, on the context's current operator (HIP events,
 * a few launches each) for the precisions the context uses -- of the SpMV kernel (its z-input form
 * with DHARA_PRECOND_COLUMN) and, with DHARA_KRYLOV_ONE_KERNEL and Jacobi, of the one-kernel
 * PCG; there, and in DHARA_MIXED with DHARA_PRECOND_COLUMN, where no SpMV runs on the FP64 tile,
 * that tile is timed on the assembly (which rewrites the system from the current state, as every
 * Picard iteration does) -- keeps the fastest (the earlier candidate unless another is 3 %
 * faster) for the kernel timed, and records it in a process-wide table keyed by (nx, ny, nz,
 * elem_bytes, kernel) that later contexts of the same shape reuse without timing.  best_us (may be
 * NULL) receives the winner's time per launch for [FP64, FP32]. */
int dhara_autotune(dhara_ctx* ctx, double* best_us);

/* ---- kernel-level entry points used by the parity tests ------------------------------ */
/* theta, K, C of the context's soil at the given psi (vanGenuchten, src/global.cu:66-105).
 * All arrays have nx*ny*nz host doubles. */
int dhara_eval_constitutive(dhara_ctx* ctx, const double* psi, double* theta, double* K,
                            double* C);
/* psi of the given theta (vanGenuchtenInverse, src/global.cu:32-52). */
int dhara_eval_inverse(dhara_ctx* ctx, const double* theta, double* psi);
/* Assembles the subsurface system at the current state the way the first Picard iteration
 * of a step does (src/subsurface.cu:704-732) and returns its diagonal D and right-hand
 * side b (either may be NULL). */
int dhara_assemble_subsurface(dhara_ctx* ctx, double* diag, double* rhs);
/* y = A x with the operator of the last dhara_assemble_subsurface / Picard iteration
 * (the matrix-free equivalent of CUSP's DIA SpMV on a3d,
 * cusp/system/cuda/detail/multiply/dia_spmv.h:60-111). */
int dhara_apply_subsurface_operator(dhara_ctx* ctx, const double* x, double* y);
/* Same operator evaluated in FP32 (K and D rounded to float, x rounded to float). */
int dhara_apply_subsurface_operator_f32(dhara_ctx* ctx, const double* x, double* y);
/* Overland face conductivities at the current ponding depth: ke[nx*ny] is the east face
 * of each cell, kn[nx*ny] the north face (UpdateKOverland, src/overland.cu:193-368, seen
 * from the non-ring cell of the face). */
int dhara_overland_conductance(dhara_ctx* ctx, double* ke, double* kn);
/* z = M^-1 r for the overland system at the current ponding depth, M^-1 one V-cycle of the
 * overland multigrid preconditioner (no reference counterpart: the reference's CG was
 * unpreconditioned, src/overland.cu:410).  r and z: nx*ny host doubles; r must be zero on the
 * outer ring (the Dirichlet rows). */
int dhara_overland_precond(dhara_ctx* ctx, const double* r, double* z);
/* Allocation-free variant of dhara_overland_precond.  No counterpart in the reference: it is for
 * callers that cannot allocate device memory (code under HIP graph capture, tight serving loops,
 * harnesses that forbid hipMalloc).  r and z are DEVICE pointers to nx*ny doubles (r zero on the
 * outer ring).  The multigrid hierarchy lives in a library-owned device array of
 * DHARA_NOALLOC_SCRATCH_BYTES per GPU, held until the process ends; a surface whose hierarchy
 * does not fit (any surface up to 512 x 512 cells fits) is rejected with DHARA_E_ARG.  The call
 * allocates nothing.  Every call on one GPU shares that GPU's array: calls that overlap on one
 * GPU race. */
#define DHARA_NOALLOC_SCRATCH_BYTES (12u << 20)
int dhara_overland_precond_noalloc(dhara_ctx* ctx, const double* r, double* z);

/* ---- discrete adjoint ------------------------------------------------------------------
 * No reference counterpart (the reference has no sensitivities).  The adjoint is that of the
 * converged implicit step: each step solves F(psi^{n+1}; psi^n, h^n, p) = 0 (the mixed-form
 * Richards residual whose modified-Picard fixed point the forward iterates to), followed by
 * the ponding update and the semi-implicit overland solve of that step.  The reverse sweep
 * solves J^T lambda = dL/dpsi^{n+1} with J = dF/dpsi^{n+1} (BiCGStab on the transposed
 * 7-point Jacobian stencil) and A2^T mu = dL/dH^{n+1} for the overland system, and recomputes
 * the forward states of every checkpoint interval from its checkpoint.
 * Requirements: FP64 precision, DHARA_THETA_CARRY_CONSISTENT, no Dirichlet faces, and a
 * forward whose Picard iterations converge (the adjoint is that of the converged step).
 * The forcing fields in place at the call stay fixed for the whole run. */
typedef struct dhara_loss_spec {
    int32_t nsteps;           /* steps run from the current state                          */
    int32_t checkpoint_every; /* a forward checkpoint (psi, ponding) every k steps, k >= 1  */
    double w_q;               /* weight of sum_t (Q_t - Q*_t)^2, Q = outlet discharge
                                 across the x = 0 edge after step t [m^3/s]               */
    double w_w;               /* weight of sum_t sum_cols (W_t - W*_t)^2, W = column storage
                                 sum_k theta dz after step t [m]                           */
    const double* q_target;   /* nsteps host doubles, or NULL for zeros                    */
    const double* w_target;   /* nsteps * nx*ny host doubles (step-major), or NULL         */
    double adj_tol;           /* relative tolerance of the reverse linear solves           */
    int32_t adj_maxiter;      /* iteration limit of each reverse linear solve              */
    int32_t reserved;
} dhara_loss_spec;

/* Runs nsteps steps from the current state and records, after every step t, the outlet
 * discharge q[t] (may be NULL) and the column storage w[t*nx*ny + col] (may be NULL). */
int dhara_observe(dhara_ctx* ctx, int32_t nsteps, double* q, double* w);
/* Forward run of spec->nsteps steps with checkpoints, the loss, and (when any gradient
 * pointer is non-NULL) the reverse sweep.  Gradients are with respect to per-cell ln Ks,
 * alpha [1/m] and n (nx*ny*nz host doubles each; NULL skips one).  On return the state is
 * the one after the forward run.  stats (may be NULL) gets the reverse-solve totals:
 * lin_iters = BiCGStab iterations, olf_iters = overland CG iterations, lin_converged and
 * olf_converged = every reverse solve converged, picard_iters = forward steps whose Picard
 * iteration ended at its limit, picard_converged = every forward step (the forward pass and
 * every recompute) converged -- when it is 0, the gradient is not that of converged steps --,
 * wall_ms. */
int dhara_adjoint_run(dhara_ctx* ctx, const dhara_loss_spec* spec, double* loss,
                      double* grad_lnks, double* grad_alpha, double* grad_n,
                      dhara_step_stats* stats);
/* Residual F(psi_new) of the implicit subsurface step that starts from the current state
 * (top flux from the current ponding depth), nx*ny*nz host doubles; F = 0 at the converged
 * step.  Units: 1/s (volume balance per cell volume). */
int dhara_adjoint_residual(dhara_ctx* ctx, const double* psi_new, double* F);
/* out = J v (transpose = 0) or J^T v (transpose = 1), J = dF/dpsi_new at psi_new. */
int dhara_adjoint_jvp(dhara_ctx* ctx, const double* psi_new, int32_t transpose, const double* v,
                      double* out);

/* ---- batched ensemble -------------------------------------------------------------------
 * No reference counterpart (the reference runs one model per process).  Many independent
 * models of uneven size, each an initialised context, stepped together: every kernel is
 * launched once over the blocks of the members still iterating, members run the step in
 * lockstep and drop out of each solve when their own stopping rule is met, and batches of
 * Krylov iterations are replayed from captured hipGraphs while every member is active.  All
 * members must have the same precision, the same picard_accel and flux faces only.  The
 * subsurface solves are column-preconditioned when every member asks for it
 * (DHARA_PRECOND_COLUMN) and fits the column kernel, else Jacobi-preconditioned.  Mixed
 * precision is FP32 PCG with FP64 iterative refinement: a member whose FP32 segment ends folds
 * its correction into x and restarts from the FP64 residual (with the column preconditioner,
 * inside the batches the other members are still iterating in).  The overland solve of a member
 * whose surface has at most 128 x 128 cells is the whole CG in one workgroup (multigrid- or
 * Jacobi-preconditioned after the member's olf_precond), one launch for all such members -- the
 * form a member created with DHARA_OLF_PRECOND_*_BLOCK takes stepped alone; a larger surface
 * takes the batched lockstep Jacobi-PCG.  The members stay
 * usable through the other entry points between ensemble steps
 * and must outlive the ensemble. */
typedef struct dhara_ensemble dhara_ensemble;
int dhara_ensemble_create(int32_t n, dhara_ctx* const* members, dhara_ensemble** out);
int dhara_ensemble_destroy(dhara_ensemble* ens);
const char* dhara_ensemble_last_error(const dhara_ensemble* ens);
/* Krylov batches from a captured hipGraph (1, default) or as individual launches (0). */
int dhara_ensemble_set_graph(dhara_ensemble* ens, int32_t on);
/* nsteps coupled steps of every member; stats (may be NULL) holds nsteps*n entries,
 * stats[step*n + member]. */
int dhara_ensemble_step(dhara_ensemble* ens, int32_t nsteps, dhara_step_stats* stats);
/* Tile autotuner of the ensemble's batched one-kernel PCG (members with DHARA_KRYLOV_ONE_KERNEL):
 * times planes-per-tile policies (planes = ceil(nz / div), div = 1, 2, 3, on 32 x 8 tiles) on the
 * members' current operators and keeps the fastest, or the members' own tiles where no policy is 3 %
 * faster than these (a small ensemble's are finer); best_us and planes_div (may be NULL) receive the
 * time per batched launch of what is kept and the fastest policy's div.  The members' states are not
 * changed.  No reference counterpart. */
int dhara_ensemble_autotune(dhara_ensemble* ens, double* best_us, int32_t* planes_div);

#ifdef __cplusplus
}
#endif
#endif /* DHARA_HIP_H */

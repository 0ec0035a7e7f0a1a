"""Column-preconditioned PCG (DHARA_PRECOND_COLUMN) against the oracle's PCG with the same
preconditioner (a Thomas solve of every column's vertical tridiagonal system, pinned against
dense solves in test_oracle_known_answers.py).

Same method and stopping rule (||r|| <= 1e-12 ||b||): heads within the FP64 parity bound
(1e-8 m) of the oracle, Krylov counts within one per solve, and several times fewer Krylov
iterations than Jacobi on the thin-layer (dz = 5 cm) workloads.  Column lengths cover the
range of the column kernel (up to 64 planes); nz > 64 and Dirichlet rows
fall back to Jacobi.
"""
import numpy as np
import pytest

from dhara_amd import _abi, inputs

pytestmark = pytest.mark.gpu

HEAD_TOL = 1e-8


def cp(p):
    return _abi.Params.from_buffer_copy(p)


def model(hip, w, precond, **overrides):
    p = cp(w.params)
    p.precond = precond
    for k, v in overrides.items():
        setattr(p, k, v)
    m = hip.FlowModel(w.grid, p)
    w.apply(m)
    return m


def oracle(orc, w, line=True, **overrides):
    p = cp(w.params)
    for k, v in overrides.items():
        setattr(p, k, v)
    o = orc.OracleModel(w.grid, p, lin_solver=orc.LIN_PCG_LINE if line else orc.LIN_PCG_JACOBI)
    w.apply(o)
    return o


def test_column_fp64_coupled_matches_oracle(hip, orc):
    w = inputs.c2_coupled(nx=37, ny=21, nz=30)
    col = model(hip, w, _abi.PRECOND_COLUMN)
    jac = model(hip, w, _abi.PRECOND_JACOBI)
    om = oracle(orc, w)
    oj = oracle(orc, w, line=False)
    lin_c = lin_j = 0
    for s in range(6):
        a = w.run(col, 1, start=s)[0]
        b = w.run(jac, 1, start=s)[0]
        so = w.run(om, 1, start=s)[0]
        w.run(oj, 1, start=s)
        dpsi = np.max(np.abs(col.download("PSI") - om.download("PSI")))
        dh = np.max(np.abs(col.download("PONDING") - om.download("PONDING")))
        dj = np.max(np.abs(col.download("PSI") - oj.download("PSI")))
        print(f"step {s}: picard {a['picard_iters']}/{so['picard_iters']} lin col {a['lin_iters']} "
              f"oracle {so['lin_iters']} jacobi {b['lin_iters']} dpsi {dpsi:.2e} dh {dh:.2e} "
              f"vs jacobi oracle {dj:.2e} mb {a['mb_rel']:.1e}", flush=True)
        assert dpsi <= HEAD_TOL and dh <= HEAD_TOL
        # the Jacobi solver meets the same residual test (||r|| <= 1e-12 ||b||) at another point
        # of the Krylov space: the heads differ by the solve tolerance times the conditioning
        # (~1e-6 m here, amplified by Picard iterations that stop at their limit)
        assert dj <= 1e-5
        assert a["picard_iters"] == so["picard_iters"]
        assert abs(a["lin_iters"] - so["lin_iters"]) <= a["picard_iters"]
        assert a["lin_converged"] == 1
        if a["picard_converged"]:
            assert a["mb_rel"] < 1e-10
        lin_c += a["lin_iters"]
        lin_j += b["lin_iters"]
    # fewer Krylov iterations than Jacobi (the early, dry steps need only a few of either)
    assert lin_c * 3 < lin_j * 2


@pytest.mark.parametrize("nz", [16, 40, 64])
def test_column_lengths_match_oracle(hip, orc, nz):
    nx, ny = 12, 10
    w = inputs.c1_column(nx=nx, ny=ny, nz=nz)
    rng = np.random.default_rng(nz)
    w.fields["KSAT"] = inputs.KS_LOAM * np.exp(rng.normal(0.0, 1.0, nx * ny * nz))
    gm = model(hip, w, _abi.PRECOND_COLUMN)
    om = oracle(orc, w)
    # four steps: the deep columns' Picard iterations stop at their limit at every step, where
    # rounding-level differences grow from step to step (1e-11 m after one, 1e-8 m after five)
    for s in range(4):
        sg = gm.step(1)[0]
        so = om.step(1)[0]
        dpsi = np.max(np.abs(gm.download("PSI") - om.download("PSI")))
        print(f"nz {nz} step {s}: picard {sg['picard_iters']}/{so['picard_iters']} "
              f"lin {sg['lin_iters']}/{so['lin_iters']} dpsi {dpsi:.2e}", flush=True)
        assert dpsi <= HEAD_TOL
        assert sg["picard_iters"] == so["picard_iters"]
        assert abs(sg["lin_iters"] - so["lin_iters"]) <= sg["picard_iters"]
        if sg["picard_converged"]:
            assert sg["mb_rel"] < 1e-10


def test_column_untiled_spmv(hip, orc):
    w = inputs.c2_coupled(nx=20, ny=17, nz=30)
    gm = model(hip, w, _abi.PRECOND_COLUMN)
    gm.set_tile(8, 0)                              # untiled SpMV kernel
    om = oracle(orc, w)
    for s in range(3):
        w.run(gm, 1, start=s)
        w.run(om, 1, start=s)
        assert np.max(np.abs(gm.download("PSI") - om.download("PSI"))) <= HEAD_TOL


def test_column_mixed_head_error(hip, orc):
    w = inputs.c2_coupled(nx=24, ny=20, nz=30)
    gm = model(hip, w, _abi.PRECOND_COLUMN, precision=_abi.MIXED)
    om = oracle(orc, w)
    sg = w.run(gm, 8)
    w.run(om, 8)
    err = np.max(np.abs(gm.download("PSI") - om.download("PSI")))
    print("mixed column max head error", err, "sweeps", [s["refine_sweeps"] for s in sg],
          "lin", [s["lin_iters"] for s in sg], flush=True)
    assert all(s["lin_converged"] for s in sg)
    assert err <= 1e-6


def test_column_falls_back_to_jacobi(hip, orc):
    # Dirichlet rows, and columns longer than the column kernel holds
    nx, ny, nz = 10, 9, 12
    w = inputs.c1_column(nx=nx, ny=ny, nz=nz)
    w.fields["BCTYPE_W"] = np.zeros(ny * nz, np.int32)
    w.fields["BCPSI_W"] = np.full(ny * nz, -0.3)
    w2 = inputs.c1_column(nx=6, ny=5, nz=70)
    for wk in (w, w2):
        gm = model(hip, wk, _abi.PRECOND_COLUMN)
        om = oracle(orc, wk, line=False)
        for s in range(3):
            gm.step(1)
            om.step(1)
            assert np.max(np.abs(gm.download("PSI") - om.download("PSI"))) <= HEAD_TOL


def test_column_autotuned_tiles(hip, orc):
    w = inputs.c2_coupled(nx=48, ny=40, nz=20, precision=_abi.MIXED)
    gm = model(hip, w, _abi.PRECOND_COLUMN, precision=_abi.MIXED)
    om = oracle(orc, w, precision=_abi.MIXED)
    best = gm.autotune()
    print("autotune:", best, flush=True)
    w.run(gm, 3)
    w.run(om, 3)
    assert np.max(np.abs(gm.download("PSI") - om.download("PSI"))) <= 1e-6


@pytest.mark.parametrize("inner_tol", [1e-5, 1e-7])
def test_mixed_column_tight_tolerance_matches_fp64(hip, inner_tol):
    """Mixed column PCG at ||r|| <= 1e-14 ||b|| (the FP64 attainable end): several FP32 segments
    and reliable updates per solve, through the queued update with its outer test on the device,
    the rate-sized batches and the rest of an update after a failed test.  Every solve converges,
    with the Picard counts of the FP64 column run, and the heads are that run's to within the
    solve tolerance."""
    w = inputs.c2_coupled(nx=48, ny=40, nz=20)
    wm = inputs.c2_coupled(nx=48, ny=40, nz=20, precision=_abi.MIXED)
    f64 = model(hip, w, _abi.PRECOND_COLUMN, lin_tol=1e-14)
    mix = model(hip, wm, _abi.PRECOND_COLUMN, lin_tol=1e-14, inner_tol=inner_tol)
    steps = 4
    sf, sm = w.run(f64, steps), wm.run(mix, steps)
    picard = sum(s["picard_iters"] for s in sm)
    updates = sum(s["refine_sweeps"] for s in sm)
    err = np.max(np.abs(mix.download("PSI") - f64.download("PSI")))
    print(f"inner_tol {inner_tol}: picard {picard} (fp64 {sum(s['picard_iters'] for s in sf)}), "
          f"reliable updates {updates}, max |dpsi| {err:.2e} m", flush=True)
    assert all(s["lin_converged"] for s in sm) and all(s["lin_converged"] for s in sf)
    assert [s["picard_iters"] for s in sm] == [s["picard_iters"] for s in sf]
    assert updates >= picard
    assert err <= 1e-8


def test_column_huge_surface_fallbacks(hip):
    """A surface with more 32 x 8 column tiles than partial slots (1056 x 1000: 4125 > 4096):
    the SpMV and assembly run untiled, the mixed reliable update falls back to the separate FP64
    residual and column start-up, the one-kernel Jacobi PCG caps its grid; all three agree."""
    w = inputs.c1_column(nx=1056, ny=1000, nz=2)
    col = model(hip, w, _abi.PRECOND_COLUMN)
    mix = model(hip, w, _abi.PRECOND_COLUMN, precision=_abi.MIXED)
    jac = model(hip, w, _abi.PRECOND_JACOBI)
    assert col.get_tile(8) == (0, 0, 0)
    sc, sm, sj = col.step(1)[0], mix.step(1)[0], jac.step(1)[0]
    print("lin iters column / mixed / jacobi:", sc["lin_iters"], sm["lin_iters"], sj["lin_iters"], flush=True)
    assert sc["lin_converged"] and sm["lin_converged"] and sj["lin_converged"]
    pc, pm, pj = col.download("PSI"), mix.download("PSI"), jac.download("PSI")
    assert np.max(np.abs(pc - pj)) <= 1e-8
    assert np.max(np.abs(pm - pc)) <= 1e-6


@pytest.mark.parametrize("inner_maxiter,refine_maxiter", [(2, 16), (2000, 0), (3, 1)])
def test_mixed_column_iteration_limits(hip, inner_maxiter, refine_maxiter):
    """The mixed column solve stopped by its FP32 iteration limit or its limit on FP64 reliable
    updates: the step reports lin_converged = 0, stays within the limits, and its heads carry the
    last correction (closer to the converged FP64 solution of the same system than the start)."""
    w = inputs.c2_coupled(nx=48, ny=40, nz=30)
    w.params.picard_maxiter = 1          # one linear solve per step
    w.params.lin_tol = 1e-14
    ref = model(hip, w, _abi.PRECOND_COLUMN)
    psi0 = ref.download("PSI")
    sr = ref.step(1)[0]
    assert sr["lin_converged"] == 1
    x_star = ref.download("PSI")
    m = model(hip, w, _abi.PRECOND_COLUMN, precision=_abi.MIXED, inner_maxiter=inner_maxiter,
              refine_maxiter=refine_maxiter)
    st = m.step(1)[0]
    x = m.download("PSI")
    err, err0 = np.max(np.abs(x - x_star)), np.max(np.abs(psi0 - x_star))
    print(f"inner {inner_maxiter} refine {refine_maxiter}: lin {st['lin_iters']} updates {st['refine_sweeps']} "
          f"converged {st['lin_converged']} err {err:.2e} (start {err0:.2e})", flush=True)
    assert st["lin_converged"] == 0
    assert np.all(np.isfinite(x))
    assert st["refine_sweeps"] <= refine_maxiter + 1
    assert st["lin_iters"] <= inner_maxiter + 1
    assert err < 0.5 * err0

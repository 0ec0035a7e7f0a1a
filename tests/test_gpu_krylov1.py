"""One-kernel PCG (single-reduction recurrences) against the oracle and the two-kernel PCG.

The one-kernel form computes the same iterates as the two-kernel Hestenes-Stiefel PCG in exact
arithmetic, so with the same stopping rule (||r|| <= 1e-12 ||b||) the heads agree with the
oracle to the FP64 parity bound (1e-8 m) and the iteration counts with the two-kernel form to
within one per solve.  Tiles: partial tiles in x and y, chunks of planes that do not divide nz,
and grids capped below the tile count (blocks looping over several tiles).
"""
import numpy as np
import pytest

from dhara_amd import _abi, inputs

pytestmark = pytest.mark.gpu

HEAD_TOL = 1e-8


def cp(p):
    return _abi.Params.from_buffer_copy(p)


def model(hip, w, krylov, **overrides):
    p = cp(w.params)
    p.krylov = krylov
    for k, v in overrides.items():
        setattr(p, k, v)
    m = hip.FlowModel(w.grid, p)
    w.apply(m)
    return m


def oracle(orc, w, **overrides):
    p = cp(w.params)
    for k, v in overrides.items():
        setattr(p, k, v)
    o = orc.OracleModel(w.grid, p)
    w.apply(o)
    return o


def test_one_kernel_fp64_coupled_matches_oracle(hip, orc):
    w = inputs.c2_coupled(nx=37, ny=21, nz=30)
    one = model(hip, w, _abi.KRYLOV_ONE_KERNEL)
    two = model(hip, w, _abi.KRYLOV_TWO_KERNEL)
    om = oracle(orc, w)
    for s in range(6):
        a = w.run(one, 1, start=s)[0]
        b = w.run(two, 1, start=s)[0]
        w.run(om, 1, start=s)
        dpsi = np.max(np.abs(one.download("PSI") - om.download("PSI")))
        dh = np.max(np.abs(one.download("PONDING") - om.download("PONDING")))
        print(f"step {s}: picard {a['picard_iters']}/{b['picard_iters']} lin {a['lin_iters']}/{b['lin_iters']} "
              f"dpsi {dpsi:.2e} dh {dh:.2e} mb {a['mb_rel']:.1e}", flush=True)
        assert dpsi <= HEAD_TOL and dh <= HEAD_TOL
        assert a["picard_iters"] == b["picard_iters"]
        assert abs(a["lin_iters"] - b["lin_iters"]) <= a["picard_iters"]
        assert a["lin_converged"] == 1
        if a["picard_converged"]:
            assert a["mb_rel"] < 1e-10


def test_one_kernel_c1_steps_match_oracle(hip, orc):
    nx, ny, nz = 12, 10, 16
    w = inputs.c1_column(nx=nx, ny=ny, nz=nz)
    rng = np.random.default_rng(3)
    w.fields["KSAT"] = inputs.KS_LOAM * np.exp(rng.normal(0.0, 1.0, nx * ny * nz))
    gm = model(hip, w, _abi.KRYLOV_ONE_KERNEL)
    gm.set_krylov_tile(8, 16, 16, 5)
    om = oracle(orc, w)
    for s in range(10):
        sg = gm.step(1)[0]
        so = om.step(1)[0]
        dpsi = np.max(np.abs(gm.download("PSI") - om.download("PSI")))
        print(f"step {s}: picard {sg['picard_iters']}/{so['picard_iters']} lin {sg['lin_iters']}/{so['lin_iters']} "
              f"dpsi {dpsi:.2e}", flush=True)
        assert dpsi <= HEAD_TOL
        assert sg["picard_iters"] == so["picard_iters"]
        assert abs(sg["lin_iters"] - so["lin_iters"]) <= sg["picard_iters"]
        assert sg["mb_rel"] < 1e-10


@pytest.mark.parametrize("tile", [(32, 8, 30, 0), (16, 16, 7, 0), (32, 16, 4, 8), (64, 8, 11, 16), (32, 8, 1, 24)])
def test_one_kernel_tiles(hip, tile):
    w = inputs.c2_coupled(nx=37, ny=21, nz=30)
    ref = model(hip, w, _abi.KRYLOV_TWO_KERNEL)
    one = model(hip, w, _abi.KRYLOV_ONE_KERNEL)
    one.set_krylov_tile(8, *tile)
    assert one.get_krylov_tile(8) == tile
    for s in range(3):
        a = w.run(ref, 1, start=s)[0]
        b = w.run(one, 1, start=s)[0]
        d = np.max(np.abs(ref.download("PSI") - one.download("PSI")))
        print(f"tile {tile} step {s}: lin {a['lin_iters']}/{b['lin_iters']} dpsi {d:.2e}", flush=True)
        assert a["picard_iters"] == b["picard_iters"]
        assert abs(a["lin_iters"] - b["lin_iters"]) <= a["picard_iters"]
        assert d < 1e-9


def test_one_kernel_mixed_head_error(hip, orc):
    w = inputs.c2_coupled(nx=24, ny=20, nz=30)
    gm = model(hip, w, _abi.KRYLOV_ONE_KERNEL, precision=_abi.MIXED)
    gm.set_krylov_tile(4, 32, 8, 9, 8)
    om = oracle(orc, w)
    sg = w.run(gm, 8)
    w.run(om, 8)
    err = np.max(np.abs(gm.download("PSI") - om.download("PSI")))
    print("mixed one-kernel max head error", err, "sweeps", [s["refine_sweeps"] for s in sg],
          "lin", [s["lin_iters"] for s in sg], flush=True)
    assert all(s["lin_converged"] for s in sg)
    assert err <= 1e-6


def test_one_kernel_falls_back_with_dirichlet_rows(hip, orc):
    nx, ny, nz = 10, 9, 12
    w = inputs.c1_column(nx=nx, ny=ny, nz=nz)
    w.fields["BCTYPE_W"] = np.zeros(ny * nz, np.int32)
    w.fields["BCPSI_W"] = np.full(ny * nz, -0.3)
    gm = model(hip, w, _abi.KRYLOV_ONE_KERNEL)
    om = oracle(orc, w)
    for s in range(3):
        gm.step(1)
        om.step(1)
        assert np.max(np.abs(gm.download("PSI") - om.download("PSI"))) <= HEAD_TOL


def test_one_kernel_autotune_then_parity(hip, orc):
    w = inputs.c2_coupled(nx=48, ny=40, nz=20, precision=_abi.MIXED)
    gm = model(hip, w, _abi.KRYLOV_ONE_KERNEL, precision=_abi.MIXED)
    om = oracle(orc, w, precision=_abi.MIXED)
    best = gm.autotune()
    print("autotune:", best, gm.get_krylov_tile(8), gm.get_krylov_tile(4), flush=True)
    assert best[0] > 0 and best[1] > 0
    w.run(gm, 3)
    w.run(om, 3)
    assert np.max(np.abs(gm.download("PSI") - om.download("PSI"))) <= 1e-6
    # a second context of the same shape picks the tuned tiles from the table
    g2 = model(hip, w, _abi.KRYLOV_ONE_KERNEL, precision=_abi.MIXED)
    assert g2.get_krylov_tile(4) == gm.get_krylov_tile(4)
    assert g2.get_krylov_tile(8) == gm.get_krylov_tile(8)


@pytest.mark.parametrize("prec", [_abi.FP64, _abi.MIXED])
def test_autotune_of_a_fresh_context_times_full_iterations(hip, prec):
    """Before any step too, a timed launch is a whole iteration: no faster than its 8 arrays at 8 TB/s."""
    w = inputs.c2_coupled(nx=400, ny=300, nz=30, precision=prec)
    gm = model(hip, w, _abi.KRYLOV_ONE_KERNEL, precision=prec)
    us = gm.autotune()
    n = 400 * 300 * 30
    print("autotune:", us, gm.get_krylov_tile(8), gm.get_krylov_tile(4), flush=True)
    assert us[0] >= n * 8 * 8 / 8e6
    assert prec == _abi.FP64 or us[1] >= n * 8 * 4 / 8e6


def test_autotune_keeps_the_defaults_that_it_does_not_beat(hip):
    """A small surface's default splits its columns finer than any fixed candidate (whole, halves,
    thirds: 7 planes of 20) and is faster by a third; and a tile timed in one form of the solver is
    not taken over by another kernel in a later context of the same grid."""
    w = inputs.c2_coupled(nx=64, ny=47, nz=20)
    before = model(hip, w, _abi.KRYLOV_TWO_KERNEL).get_tile(8)
    col = model(hip, w, _abi.KRYLOV_ONE_KERNEL, precond=_abi.PRECOND_COLUMN)
    col.set_tile(8, 64, 8, 13)          # in use, so a candidate
    col.autotune()
    assert model(hip, w, _abi.KRYLOV_TWO_KERNEL).get_tile(8) == before
    one = model(hip, w, _abi.KRYLOV_ONE_KERNEL)
    one.step(1)
    one.autotune()
    assert one.get_krylov_tile(8)[2] < 7

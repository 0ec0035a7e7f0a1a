"""The overland multigrid CG that runs on chip in one workgroup (surfaces whose level 0 has at most one
2 x 2 aggregate per thread) against the oracle: the exact level alone, one and several smoothed
levels, odd edges, the largest square it takes and a shape just beyond it (grid-wide form), strips up
to the longest it takes and one of two rows that goes to the one-workgroup form in memory."""
import numpy as np
import pytest

from dhara_amd import _abi, inputs

pytestmark = pytest.mark.gpu

TOL = 1e-8   # m: ponding and heads of every coupled parity case


@pytest.mark.parametrize("nx,ny", [(8, 8), (9, 8), (16, 17), (33, 31), (47, 86), (64, 64), (65, 64), (3, 200),
                                   (3, 600), (470, 5), (6, 480), (3, 750), (2, 800)])
@pytest.mark.parametrize("form", [_abi.OLF_PRECOND_MG])
def test_small_surfaces_match_oracle(hip, orc, nx, ny, form):
    w = inputs.c2_coupled(nx=nx, ny=ny, nz=3, rain_mm_h=150.0)
    p = _abi.Params.from_buffer_copy(w.params)
    q = _abi.Params.from_buffer_copy(p)
    p.olf_precond = form
    g, o = hip.FlowModel(w.grid, p), orc.OracleModel(w.grid, q)
    w.apply(g)
    w.apply(o)
    sg = g.step(6)
    o.step(6)
    assert all(s["olf_converged"] for s in sg)
    assert np.max(np.abs(g.download("PONDING") - o.download("PONDING"))) <= TOL
    assert np.max(np.abs(g.download("PSI") - o.download("PSI"))) <= TOL


def test_iteration_limit_is_reported(hip):
    w = inputs.c2_coupled(nx=40, ny=33, nz=3, rain_mm_h=150.0)
    p = _abi.Params.from_buffer_copy(w.params)
    p.olf_maxiter = 2
    m = hip.FlowModel(w.grid, p)
    w.apply(m)
    s = m.step(4)[-1]
    assert s["olf_iters"] == 2 and not s["olf_converged"]


# columns, rows, seed, wetted fraction, depth, surface wiggle, dt, cell size
@pytest.mark.parametrize("nx,ny,seed,wet,depth,wiggle,dt,dx", [
    (26, 40, 1023104, 0.414, 83.644, 1.27e-05, 7313.1, 0.329), (38, 31, 1042317, 0.406, 89.815, 2.64e-06, 3555.0, 0.32),
    (45, 19, 641173, 0.43, 69.547, 0.00133, 1458.1, 0.415), (13, 24, 190083, 0.405, 30.476, 2.13e-06, 8631.3, 0.443)])
def test_flat_pools_between_islands_converge(hip, nx, ny, seed, wet, depth, wiggle, dt, dx):
    """Deep water at rest around dry islands: conductances of 1e-2 next to 1e12.  CG that sums (p, A p)
    directly solves these in 100 to 500 iterations in numpy; with a recurrence for it the sum comes
    out negative on the way."""
    rng = np.random.default_rng(seed)
    w = rng.random((ny, nx)) < wet
    z = np.where(w, -depth * rng.uniform(0.5, 1.0, (ny, nx)), rng.uniform(0.1, 1.0, (ny, nx)))
    h = np.where(w, wiggle * rng.random((ny, nx)) - z, 0.0)
    g = _abi.Grid(nx=nx, ny=ny, nz=1, nroot_groups=1, dx=dx, dy=dx, dz=0.05)
    m = hip.FlowModel(g, _abi.default_params(dt=dt))
    m.upload_many({"ZTOPO": z.ravel(), "PONDING": h.ravel(), "MANNING": np.full(nx * ny, 0.03)})
    s = m.overland_step()
    assert s["olf_converged"] and not s["nan_seen"] and s["olf_iters"] > 0
    assert np.all(np.isfinite(m.download("PONDING")))

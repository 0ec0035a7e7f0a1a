"""The overland multigrid CG that runs on chip in one workgroup (surfaces whose level 0 has at most one
2 x 2 aggregate per thread) against the oracle: the exact level alone, one and several smoothed
levels, odd edges, the largest square it takes and a shape just beyond it (grid-wide form)."""
import numpy as np
import pytest

from dhara_amd import _abi, inputs

pytestmark = pytest.mark.gpu

TOL = 1e-8   # m: ponding and heads of every coupled parity case


@pytest.mark.parametrize("nx,ny", [(8, 8), (9, 8), (16, 17), (33, 31), (47, 86), (64, 64), (65, 64), (3, 200)])
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

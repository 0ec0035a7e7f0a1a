"""The one-launch initial state against the separate evaluations (same formulas, so to a few rounding
errors): one cell, ragged sizes, more cells than one round of the grid (1024 x 256), per-cell soils,
both modes and precisions; the copies for the first iteration through a step from it."""
import numpy as np
import pytest

from dhara_amd import _abi, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [_abi.INIT_FROM_PSI, _abi.INIT_FROM_THETA])
@pytest.mark.parametrize("shape,soils,precision", [((1, 1, 1), False, _abi.FP64), ((13, 7, 5), True, _abi.MIXED),
                                                   ((97, 71, 41), True, _abi.FP64)])
def test_initial_state(hip, orc, shape, soils, precision, mode):
    nx, ny, nz = shape
    n = nx * ny * nz
    w = inputs.c1_column(nx=nx, ny=ny, nz=nz)
    rng = np.random.default_rng(n)
    if soils:
        w.fields["ALPHA"] = rng.uniform(1.0, 4.0, n)
        w.fields["NVG"] = rng.uniform(1.3, 2.2, n)
    p = _abi.Params.from_buffer_copy(w.params)
    p.precision = precision
    m = hip.FlowModel(w.grid, p)
    o = orc.OracleModel(w.grid, _abi.Params.from_buffer_copy(w.params))
    for x in (m, o):
        w.apply(x)
    psi = rng.uniform(-5.0, 0.2, n)
    theta = rng.uniform(0.1, 0.425, n)
    if mode == _abi.INIT_FROM_THETA:
        psi = m.eval_inverse(theta)
        m.upload("THETA", theta)
    else:
        m.upload("PSI", psi)
    m.init_state(mode)
    th, K, C = m.eval_constitutive(psi)
    for f, ref in (("PSI", psi), ("THETA", th), ("K", K), ("C", C)):
        np.testing.assert_allclose(m.download(f), ref, rtol=1e-13, atol=0.0)
    if n < 1000:
        o.upload("PSI", psi)
        o.init_state(_abi.INIT_FROM_PSI)
        m.step(1)
        o.step(1)
        assert np.max(np.abs(m.download("PSI") - o.download("PSI"))) <= (1e-8 if precision == _abi.FP64 else 1e-6)

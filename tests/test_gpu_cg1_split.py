"""The default planes per block of the one-kernel PCG on the GPU: surfaces on both sides of the line
between split and whole columns, planes that do not divide, against the oracle; and an ensemble whose
members fill the chip together against its members stepped alone."""
import numpy as np
import pytest

import dhara_amd
from dhara_amd import _abi, inputs

pytestmark = pytest.mark.gpu

HEAD_TOL = 1e-8   # m, as for every FP64 parity case (solves end at ||r|| <= 1e-12 ||b||)


# (nx, ny, nz): one tile; 4 tiles of 7 planes (one plane a block); 66 tiles of 13 planes (chunks of 3,
# the last of 1); 209 tiles (one chunk)
@pytest.mark.parametrize("shape", [(7, 5, 3), (33, 9, 7), (161, 88, 13), (333, 152, 4)])
@pytest.mark.parametrize("prec", [_abi.FP64, _abi.MIXED])
def test_default_split_matches_oracle(hip, orc, shape, prec):
    w = inputs.c2_coupled(*shape)
    p = _abi.Params.from_buffer_copy(w.params)
    p.overland = 0
    q = _abi.Params.from_buffer_copy(p)
    p.precision = prec
    g, o = hip.FlowModel(w.grid, p), orc.OracleModel(w.grid, q)
    w.apply(g)
    w.apply(o)
    sg, so = g.step(2), o.step(2)
    assert [s["picard_iters"] for s in sg] == [s["picard_iters"] for s in so]
    assert np.max(np.abs(g.download("PSI") - o.download("PSI"))) <= (HEAD_TOL if prec == _abi.FP64 else 1e-6)


def test_full_ensemble_matches_members_alone():
    spec = [dict(nx=100, ny=80 - i, nz=6, sigma_lnk=1.0, rain_mm_h=20.0 + i, seed=3000 + i) for i in range(12)]

    def make(s):
        w = inputs.c5_member(s, precision=_abi.FP64)
        m = dhara_amd.FlowModel(w.grid, _abi.Params.from_buffer_copy(w.params))
        w.apply(m)
        return m
    ms = [make(s) for s in spec]   # 464 whole-column tiles: beyond the line
    st = dhara_amd.Ensemble(ms).step(2)
    for i in (0, 11):
        alone = make(spec[i])
        sa = alone.step(2)
        assert [s["picard_iters"] for s in sa] == [st[k][i]["picard_iters"] for k in range(2)]
        assert np.max(np.abs(ms[i].download("PSI") - alone.download("PSI"))) <= HEAD_TOL

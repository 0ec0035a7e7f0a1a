"""The Anderson pass's ring on the GPU against the oracle: depths 1 to the largest, each with a case whose
steps wrap the ring (depth 5: 14 passes of the 45-plane case), columns shorter and longer than the
planes it keeps on chip, widths that are not a multiple of its 16 or 64 columns, surfaces on both sides
of the rule between these two."""
import numpy as np
import pytest

from dhara_amd import _abi, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,depth", [((9, 7, 5), 1), ((13, 11, 32), 2), ((16, 8, 33), 3), ((11, 7, 45), 4),
                                         ((10, 13, 30), 5), ((12, 9, 45), 5), ((129, 127, 3), 3), ((129, 128, 3), 3)])
def test_ring_matches_oracle(hip, orc, shape, depth):
    w = inputs.c2_coupled(*shape)
    p = _abi.Params.from_buffer_copy(w.params)
    p.overland = 0
    p.picard_accel = depth
    g = hip.FlowModel(w.grid, _abi.Params.from_buffer_copy(p))
    o = orc.OracleModel(w.grid, _abi.Params.from_buffer_copy(p))
    w.apply(g)
    w.apply(o)
    sg, so = g.step(4), o.step(4)
    assert [s["picard_iters"] for s in sg] == [s["picard_iters"] for s in so]
    assert np.max(np.abs(g.download("PSI") - o.download("PSI"))) <= 1e-8   # m, every FP64 parity case
    assert np.max(np.abs(g.download("THETA") - o.download("THETA"))) <= 1e-9

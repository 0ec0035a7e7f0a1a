"""The block maps of an ensemble follow its active set: more members than one pass of the map
kernel takes (256) that stop at different iterations, each against the same model stepped alone.
Bitwise, as for every FP64 ensemble whose members use the batched forms alone too."""
import numpy as np
import pytest

from dhara_amd import _abi, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("members", [1, 3, 259])
def test_members_equal_models_alone(hip, members):
    shapes = [(5 + m % 7, 4 + m % 5, 3 + m % 4) for m in range(members)]

    def build(m):
        w = inputs.c2_coupled(*shapes[m])
        p = _abi.Params.from_buffer_copy(w.params)
        p.precond = _abi.PRECOND_COLUMN
        p.olf_precond = _abi.OLF_PRECOND_JACOBI_BLOCK
        p.picard_accel = 3
        p.dt = 20.0 * (1 + m % 6)          # different Picard and Krylov counts
        g = hip.FlowModel(w.grid, p)
        w.apply(g)
        g.set_tile(8, 0)                   # the untiled SpMV of the batched form
        return g

    models = [build(m) for m in range(members)]
    ens = hip.Ensemble(models)
    ens.step(2)
    for m in range(0, members, 1 if members < 9 else 37):
        alone = build(m)
        alone.step(2)
        for f in ("PSI", "THETA", "PONDING"):
            assert np.array_equal(models[m].download(f), alone.download(f)), (m, f)

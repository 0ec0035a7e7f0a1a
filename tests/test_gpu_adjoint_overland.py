"""Reverse overland solve in its two forms (one-workgroup multigrid CG; Jacobi-CG) over surfaces from
3 x 2 inner cells to the largest square that fits one workgroup and the first size that does not: the
gradients of a run with outlet discharge agree to the forward's and reverse's tolerances (1e-14, 1e-12)
times the conditioning: 1e-6 of the largest entry, the bound of the oracle parity test."""
import numpy as np
import pytest

from dhara_amd import _abi

from test_gpu_adjoint import make_gpu
from test_oracle_adjoint import small_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(5, 4), (17, 9), (33, 64), (64, 64), (65, 40), (65, 64)])
def test_gradient_of_both_overland_forms(nx, ny):
    grads = []
    steps = 6
    for form in (_abi.OLF_PRECOND_MG, _abi.OLF_PRECOND_JACOBI):
        w = small_workload(nx=nx, ny=ny, nz=4)
        w.params.olf_precond = form
        m = make_gpu(w)
        _, *g, st = m.adjoint_run(steps, checkpoint_every=2, q_target=np.zeros(steps),
                                  w_target=np.zeros((steps, nx * ny)), w_q=1e6, w_w=1.0)
        assert st["olf_converged"] and st["lin_converged"]
        grads.append(g)
    for a, b in zip(*grads):
        assert np.max(np.abs(b)) > 0.0
        assert np.max(np.abs(a - b)) <= 1e-6 * np.max(np.abs(b))

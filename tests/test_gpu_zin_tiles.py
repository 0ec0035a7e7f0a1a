"""SpMV of the column form over its tiles and plane chunks (remainders of the planes in flight, chunks
of one plane, whole columns, rows narrower and wider than a tile) against the oracle's PCG with the same
preconditioner, FP64: the parity bound on heads (1e-8 m), equal Picard counts, Krylov counts within one
a solve.  Tile (0, 0, 0) is the default's choice."""
import numpy as np
import pytest

from dhara_amd import _abi, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,tile", [((70, 9, 11), (0, 0, 0)), ((33, 40, 6), (0, 0, 0)), ((65, 5, 1), (0, 0, 0)),
                                        ((37, 21, 13), (32, 8, 1)), ((37, 21, 13), (64, 4, 5)),
                                        ((70, 17, 10), (64, 8, 10)), ((18, 19, 7), (16, 16, 3))])
def test_column_spmv_tiles(hip, orc, shape, tile):
    nx, ny, nz = shape
    w = inputs.c1_column(nx=nx, ny=ny, nz=nz)
    rng = np.random.default_rng(nx * ny)
    w.fields["KSAT"] = inputs.KS_LOAM * np.exp(rng.normal(0.0, 1.0, nx * ny * nz))
    p = _abi.Params.from_buffer_copy(w.params)
    p.precond = _abi.PRECOND_COLUMN
    g = hip.FlowModel(w.grid, p)
    o = orc.OracleModel(w.grid, _abi.Params.from_buffer_copy(w.params), lin_solver=orc.LIN_PCG_LINE)
    w.apply(g)
    w.apply(o)
    if tile[0]:
        g.set_tile(8, *tile)
    for _ in range(3):
        sg, so = g.step(1)[0], o.step(1)[0]
        assert np.max(np.abs(g.download("PSI") - o.download("PSI"))) <= 1e-8
        assert sg["picard_iters"] == so["picard_iters"]
        assert abs(sg["lin_iters"] - so["lin_iters"]) <= sg["picard_iters"]


def test_default_takes_whole_columns_while_they_are_resident(hip):
    """64 x 8 tiles: 504 (resident at once) keep their columns whole, 560 (a second round nearly
    empty) are halved."""
    for nx, ny, kc in ((500, 500, 12), (512, 560, 6)):
        m = hip.FlowModel(_abi.Grid(nx=nx, ny=ny, nz=12, nroot_groups=1, dx=1.0, dy=1.0, dz=0.05),
                          _abi.default_params(precond=_abi.PRECOND_COLUMN))
        assert m.get_tile(8) == (64, 8, kc)
        m.close()

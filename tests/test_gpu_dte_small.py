"""core_dTe at the line between meshes that one workgroup sweeps in one launch
(up to 1,024 cells) and tiled ones, against the oracle, and bitwise the same
for every workgroup size and under a captured graph. 100 updates a cell of a few
ulp each stay far below TOL."""
import numpy as np
import pytest

from spilady_amd.constants import BOLTZ
from spilady_amd.engine import Engine
from oracle import orcpy

from helpers import assert_close
from test_gpu_dte_tiles import _system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [(3, 3, 3), (5, 3, 4), (16, 8, 8), (11, 31, 3), (5, 5, 41), (3, 18, 19)])
def test_core_dte_around_the_line(cells):
    p, at = _system(cells)
    o = orcpy.Oracle(p, at, compute_initial_forces=True, rng=orcpy.RNG_PHILOX)
    assert tuple(o.ncell3) == cells
    te = BOLTZ * np.random.default_rng(9).uniform(200.0, 1500.0, o.ncells)
    o.set_cells_te(te)
    o.core_dTe(0.5e-15)
    want = o.cells()
    o.close()
    got = []
    e = Engine(p, at, compute_initial_forces=True)
    for block, graph in ((64, 0), (128, 0), (256, 0), (256, 1), (256, 1)):
        e.set_graph_mode(graph)
        e.set_shapes(dict(sweep_block=block))
        e.set_cells_te(te)
        e.core_dTe(0.5e-15)
        got.append(e.cells())
    e.close()
    for k in ("te", "ee"):
        assert_close(want[k], got[0][k], f"{cells} {k}")
        for g in got[1:]:
            np.testing.assert_array_equal(g[k], got[0][k])

"""core_dTe on a mesh of more than 512 tiles (648 tiles of 4 x 4 x 4 cells, one
launch a sweep), whose sweep keeps eight slots a thread in flight, against the
oracle and bitwise the same for every workgroup size: with 64 threads a tile's
slots go past the eighth. The oracle sweeps in the same order; 100 updates a
cell of a few ulp each stay far below TOL."""
import numpy as np
import pytest

from spilady_amd.constants import BOLTZ
from spilady_amd.engine import Engine
from oracle import orcpy

from helpers import assert_close
from test_gpu_dte_tiles import _system

pytestmark = pytest.mark.gpu


def test_core_dte_on_many_tiles():
    cells = (35, 33, 31)
    p, at = _system(cells)
    o = orcpy.Oracle(p, at, compute_initial_forces=True, rng=orcpy.RNG_PHILOX)
    assert tuple(o.ncell3) == cells
    te = BOLTZ * np.random.default_rng(8).uniform(200.0, 1500.0, o.ncells)
    o.set_cells_te(te)
    o.core_dTe(0.5e-15)
    want = o.cells()
    o.close()
    got = []
    e = Engine(p, at, compute_initial_forces=True)
    for block in (64, 128, 256):
        e.set_shapes(dict(sweep_block=block))
        e.set_cells_te(te)
        e.core_dTe(0.5e-15)
        got.append(e.cells())
    e.close()
    for k in ("te", "ee"):
        assert_close(want[k], got[0][k], k)
        for g in got[1:]:
            np.testing.assert_array_equal(g[k], got[0][k])

"""core_dTe over tiled meshes of every kind of side (even, odd, below a tile,
remainder tiles; one launch for both sweeps and one each) against the oracle,
and bitwise the same for every workgroup size.

The oracle sweeps group by group in the same order, so what differs is
rounding: 100 updates a cell of a few ulp each stay far below TOL."""
import numpy as np
import pytest

from spilady_amd import abi, configs
from spilady_amd.constants import BOLTZ, FE_A_LATTICE
from spilady_amd.engine import Engine
from oracle import orcpy

from helpers import assert_close

pytestmark = pytest.mark.gpu


def _system(cells, seed=5):
    """a bcc block whose link mesh has the given sides"""
    n = [int(np.ceil(c * 4.11 / FE_A_LATTICE)) for c in cells]
    r = configs.bcc100_positions(*n, FE_A_LATTICE)
    rng = np.random.default_rng(seed)
    natom = len(r)
    box = [n[0] * FE_A_LATTICE, 0.0, n[1] * FE_A_LATTICE, 0.0, 0.0, n[2] * FE_A_LATTICE]
    v = configs.fe_variables(300.0, seed, thermostats=True, eltemp=True, localcolmot=True)
    p = abi.params_from_variables(v, box, natom)
    s = np.array([0.0, 0.0, 1.1]) + rng.normal(0.0, 0.05, (natom, 3))
    at = dict(r=r, p=rng.normal(0.0, np.sqrt(p.atmass * BOLTZ * 300.0), (natom, 3)), s=s, f=np.zeros((natom, 3)))
    return p, at


@pytest.mark.parametrize("cells", [(3, 4, 5), (4, 4, 4), (7, 7, 7), (9, 3, 11), (8, 8, 8), (13, 12, 6), (17, 10, 9),
                                   (23, 22, 21), (33, 25, 13), (24, 24, 20)])
def test_core_dte_on_any_mesh(cells):
    p, at = _system(cells)
    o = orcpy.Oracle(p, at, compute_initial_forces=True, rng=orcpy.RNG_PHILOX)
    assert tuple(o.ncell3) == cells
    te = BOLTZ * np.random.default_rng(7).uniform(200.0, 1500.0, o.ncells)
    o.set_cells_te(te)
    o.core_dTe(0.5e-15)
    want = o.cells()
    o.close()
    got = []
    for block in (64, 128, 256):
        e = Engine(p, at, compute_initial_forces=True)
        e.set_shapes(dict(sweep_block=block))
        e.set_cells_te(te)
        e.core_dTe(0.5e-15)
        got.append(e.cells())
        e.close()
    for k in ("te", "ee"):
        assert_close(want[k], got[0][k], f"{cells} {k}")
        for g in got[1:]:
            np.testing.assert_array_equal(g[k], got[0][k])


@pytest.mark.parametrize("lo,hi", [(0.5, 20.0), (2.0, 20000.0), (5000.0, 8000.0)])
def test_core_dte_outside_the_polynomials(lo, hi):
    """Electron temperatures below and above the fitted range and relaxations
    past |u| = 1/4, cell by cell next to ordinary ones: waves with both kinds
    of lanes."""
    p, at = _system((7, 6, 8))
    o = orcpy.Oracle(p, at, compute_initial_forces=True, rng=orcpy.RNG_PHILOX)
    te = BOLTZ * np.exp(np.random.default_rng(11).uniform(np.log(lo), np.log(hi), o.ncells))
    o.set_cells_te(te)
    o.core_dTe(0.5e-15)
    want = o.cells()
    o.close()
    e = Engine(p, at, compute_initial_forces=True)
    e.set_cells_te(te)
    e.core_dTe(0.5e-15)
    got = e.cells()
    e.close()
    for k in ("te", "ee"):
        assert_close(want[k], got[k], f"{lo}-{hi} K {k}")

"""core_dTe on meshes of more than 1,024 tiles (11 x 11 x 9 of 10^3 cells), whose
final-energy partials are reduced by a launch of their own before a sub-step is
normalised. Without thermostats nothing but diffusion acts on the electrons, so
their energy stays: each of 50 sub-steps normalises it from two sums of about 10^6
terms, good to 1e-14 at worst, 5e-13 in all. The mesh needs few atoms; kappa_e is
scaled to their number, which the conductivity's volume per atom goes by."""
import numpy as np
import pytest

from spilady_amd import abi, configs
from spilady_amd.constants import BOLTZ
from spilady_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [(101, 101, 81), (102, 102, 82)])
def test_energy_is_kept(cells):
    n, C = 64, int(np.prod(cells))
    box = [c * 4.12 for c in cells]
    rng = np.random.default_rng(2)
    r = rng.uniform(0.0, 1.0, (n, 3)) * box
    v = configs.fe_variables(300.0, 3, thermostats=False, eltemp=True)
    p = abi.params_from_variables(v, [box[0], 0.0, box[1], 0.0, 0.0, box[2]], n)
    p.kappa_e *= (n / (6.0 * C)) ** 2
    s = np.tile([0.0, 0.0, 1.1], (n, 1))
    e = Engine(p, dict(r=r, p=np.zeros((n, 3)), s=s, f=np.zeros((n, 3))), compute_initial_forces=True)
    assert e.ncell3 == cells
    te = BOLTZ * rng.uniform(200.0, 1500.0, C)
    e.set_cells_te(te)
    before = e.cells()["ee"].astype(np.longdouble).sum()
    e.core_dTe(0.5e-15)
    c = e.cells()
    e.close()
    after = c["ee"].astype(np.longdouble).sum()
    assert abs(after - before) <= 5e-13 * before
    # and the cells have mixed
    assert np.std(c["te"]) < 0.99 * np.std(te)

"""The neighbour build's density and exchange field over cells of any
occupation (more pairs than its buffer holds, more candidates than its
registers hold), against the oracle, and the capacity errors at its edges.
Sums run in another order: a few roundings of 1e-16 a pair, far below TOL."""
import numpy as np
import pytest

from spilady_amd import abi, configs
from spilady_amd.engine import Engine, SldError
from oracle import orcpy

from helpers import assert_close

pytestmark = pytest.mark.gpu


def _pair(nu, mlc, sigma, seed=4, a=2.8665):
    at = configs.make_bcc_fe(nu, 300.0, seed, displace_sigma=sigma, tilt_max_deg=40.0, a=a)
    v = configs.fe_variables(300.0, seed, thermostats=False)
    v["min_length_link_cell"] = mlc
    return abi.params_from_variables(v, at.box, at.natom), at


# cells of up to 9 atoms (4.11 A), 16 (432 candidates) and about 20 (displaced by 0.25 A)
@pytest.mark.parametrize("nu,mlc,sigma", [(5, 4.11, 0.0), (6, 4.11, 0.1), (8, 5.7, 0.05), (8, 5.7, 0.25), (11, 5.2, 0.15),
                                          (12, 4.11, 0.2)])
def test_density_and_field_match_the_oracle(nu, mlc, sigma):
    p, at = _pair(nu, mlc, sigma)
    o = orcpy.Oracle(p, at, compute_initial_forces=True)
    e = Engine(p, at, compute_initial_forces=True)
    for x in (o, e):
        x.links()
        x.calculate_rho()
        x.core_ds(1e-15)
        x.calculate_force_energy()
    a, b = o.download(), e.download()
    o.close()
    e.close()
    for k in ("rho", "f", "pe", "me", "s", "heff_h"):
        assert_close(a[k], b[k], k)


# 35 atoms in a link cell of 32; more neighbours within rcut_max than a list holds (lattice constant 2.2 A)
@pytest.mark.parametrize("nu,mlc,sigma,a", [(7, 6.6, 0.1, 2.8665), (8, 4.11, 0.0, 2.2)])
def test_what_does_not_fit_is_an_error(nu, mlc, sigma, a):
    p, at = _pair(nu, mlc, sigma, a=a)
    with pytest.raises(SldError) as err:
        Engine(p, at, compute_initial_forces=True)
    assert "SLD_ERR_CAPACITY" in str(err.value)

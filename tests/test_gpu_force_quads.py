"""The force pass over lists of every length modulo its four lanes, empty ones
included, against the oracle: forces, energies, virial and stress, with and
without the local volume. Sums run in another order: a few roundings of 1e-16 a
pair, far below TOL."""
import numpy as np
import pytest

from spilady_amd import abi, configs
from spilady_amd.engine import Engine
from oracle import orcpy

from helpers import assert_close

pytestmark = pytest.mark.gpu


def _sparse(nu, keep, seed):
    """A displaced lattice of which a share of the atoms is kept."""
    rng = np.random.default_rng(seed)
    at = configs.make_bcc_fe(nu, 300.0, seed, displace_sigma=0.08, tilt_max_deg=60.0)
    k = rng.random(len(at.r)) < keep
    return at.box, at.r[k], at.s[k], rng.normal(0.0, 1.0, (int(k.sum()), 3))


# lists of 0 to 3, 7 to 20, 2 to 12, 12 to 24 and 18 to 26 atoms; an atom without
# neighbours has no local volume
@pytest.mark.parametrize("nu,keep,localvol", [(5, 0.1, 0), (5, 0.5, 0), (5, 0.5, 1), (6, 0.3, 1), (7, 0.8, 0),
                                              (9, 1.0, 1)])
def test_every_list_length_matches_the_oracle(nu, keep, localvol):
    box, r, s, p0 = _sparse(nu, keep, 31 + nu)
    n = len(r)
    v = configs.fe_variables(300.0, 31, thermostats=False)
    v["localvol"] = localvol
    p = abi.params_from_variables(v, box, n)
    at = dict(r=r, p=p0, s=s, f=np.zeros((n, 3)))
    o = orcpy.Oracle(p, at, compute_initial_forces=True)
    e = Engine(p, at, compute_initial_forces=True)
    a, b = o.download(), e.download()
    o.close()
    e.close()
    for k in ("f", "pe", "me", "me0", "stress"):
        assert_close(a[k], b[k], k)
    # the oracle books a pair's virial on one of its atoms, the engine half on each
    assert_close(a["vir"].sum(), b["vir"].sum(), "virial")

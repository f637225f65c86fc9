"""The model's device-built tables over all branches of the pair term: knots,
the quintic bridge (1.8 to 2 A) and the ZBL core, against the oracle's
host-built tables through energies, forces, fields and the gradient.

The bridge and the knot sums are evaluated in the oracle's order, so what
differs is the rounding of exp, log and cubes: 1e-16 of a value, times 45/60
over dx = r/1000 (about 500) in a derivative, far below the TOL that the
pair sums are held to.
"""
import numpy as np
import pytest

from oracle import orcpy
from spilady_amd import configs, fit

from helpers import TOL, assert_close

pytestmark = pytest.mark.gpu
RC = dict(rcut_max=4.1001, rcut_pot=4.1001, rcut_mag=3.7501)


@pytest.mark.parametrize("rel", [0.0, 0.02, -0.05])
def test_tables_in_the_bridge_and_the_core(rel):
    at = configs.make_bcc_fe(5, 300.0, 41, displace_sigma=0.3, tilt_max_deg=30.0)
    L = at.box[0]
    d = at.r[:, None, :] - at.r[None, :, :]
    d -= L * np.round(d / L)
    dist = np.sqrt((d * d).sum(-1))[np.triu_indices(len(at.r), 1)]
    assert np.sum(dist <= 1.8) > 0 and np.sum((dist > 1.8) & (dist <= 2.0)) > 0
    th = fit.perturbed_params(fit.default_params(), rel, 5)
    m = fit.PotentialModel([at])
    m.set_params(th)
    E, F, H = m.eval()
    rng = np.random.default_rng(3)
    gE, gF, gH = rng.normal(size=1), rng.normal(size=F.shape), rng.normal(size=H.shape)
    g = m.vjp(gE, gF, gH)
    m.close()
    tab = orcpy.ModelTables(th, RC["rcut_max"])
    e, f, h, gr = tab.eval_grad(at, **RC, gE=gE[0], gF=gF, gH=gH)
    tab.close()
    assert abs(E[0] - e) <= TOL * abs(e)
    assert_close(f, F, "force")
    assert_close(h, H, "field")
    assert_close(gr, g, "gradient")

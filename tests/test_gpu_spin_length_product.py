"""|s_i| |s_j| of the force pass's exchange energy against long double, for spins
whose common length rounds badly: pairs of atoms out of everyone else's reach, so
that me0 of an atom is J/2 |s_i| |s_j|, with J/2 from spins of length one.

In units of 2^-53: the two squared lengths round about twice each, which the root
halves, the product, the root and J/2's product once each at 0.4 root mean square:
0.7 in all, 1.0 allowed. Lengths rounded first would share one error of 0.6 on each
side, 1.2 for every pair alike."""
import numpy as np
import pytest

from spilady_amd import abi, configs
from spilady_amd.engine import Engine

from test_gpu_model_knots import _pairs

pytestmark = pytest.mark.gpu


def test_product_of_lengths_is_rounded_once():
    at, _, _ = _pairs(2.5, 71, n=8)
    rng = np.random.default_rng(72)
    unit = rng.normal(size=(len(at.r), 3)).astype(np.longdouble)
    unit /= np.sqrt((unit * unit).sum(axis=1, keepdims=True))
    length = np.longdouble(1.03125) + np.longdouble(0.3) * np.spacing(1.03125)   # 0.3 of a place past a double
    s = (length * unit).astype(np.float64)
    at.s = np.tile([1.0, 0.0, 0.0], (len(at.r), 1))
    v = configs.fe_variables(300.0, 3, thermostats=False)
    e = Engine(abi.params_from_variables(v, at.box, len(at.r)), at, compute_initial_forces=True)
    half_j = e.download()["me0"].astype(np.longdouble)
    e.upload(dict(r=at.r, p=at.p, s=s))
    e.calculate_force_energy()
    me0 = e.download()["me0"].astype(np.longdouble)
    e.close()
    exact = np.sqrt((s.astype(np.longdouble) ** 2).sum(axis=1))
    want = half_j * np.repeat(exact[0::2] * exact[1::2], 2)
    err = (me0 - want) / want * np.longdouble(2.0) ** 53
    assert np.sqrt((err ** 2).mean()) <= 1.0, (err.mean(), np.sqrt((err ** 2).mean()))

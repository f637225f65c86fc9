"""Launch shapes where they change the launches: 24^3 link cells (levels of 1,728
cells, so that a wave of the spin sweep takes 1, 2 or 4 cells as spin_block and
spin_lanes say, and an electron mesh in 216 tiles, whose workgroups sweep_block
sizes). The trajectory is the same bit for bit, and the autotuner's twin too."""
import numpy as np
import pytest

from helpers import consistent_state, fe_params
from spilady_amd.engine import Engine

pytestmark = pytest.mark.gpu

FIELDS = ("r", "p", "f", "s", "rho", "pe", "ke", "me", "me0", "stress", "heff_h", "heff_l")
SETS = [dict(spin_block=b, spin_lanes=l, sweep_block=w) for b, l, w in
        ((32, 1, 64), (64, 1, 128), (128, 1, 256), (64, 2, 64), (32, 2, 128), (128, 4, 64))]


@pytest.fixture(scope="module")
def system():
    v, p, at = fe_params(35, 600.0, 41, thermostats=True, eltemp=True, localcolmot=True)
    return p, consistent_state(p, at)


def _run(e, steps, first=0):
    return e.step(first, steps)


def _same(a, b):
    return len(a) == len(b) and all(x.keys() == y.keys() and all(np.array_equal(x[k], y[k]) for k in x)
                                    for x, y in zip(a, b))


@pytest.fixture(scope="module")
def plain(system):
    p, st = system
    e = Engine(p, st)
    assert e.ncell3 == (24, 24, 24)
    out = _run(e, 3), e.download(), e.cells()
    e.close()
    return out


@pytest.mark.parametrize("shapes", SETS, ids=str)
def test_trajectory_does_not_depend_on_the_shapes(system, plain, shapes):
    p, st = system
    e = Engine(p, st)
    e.set_shapes(shapes)
    obs, a, c = _run(e, 3), e.download(), e.cells()
    e.close()
    assert _same(obs, plain[0])
    for f in FIELDS:
        np.testing.assert_array_equal(a[f], plain[1][f], err_msg=f)
    for f in ("te", "ee"):
        np.testing.assert_array_equal(c[f], plain[2][f], err_msg=f)


def test_autotuned_twin(system, plain):
    p, st = system
    e = Engine(p, st)
    obs = _run(e, 1)
    e.autotune(1)
    obs += _run(e, 2, 1)
    a = e.download()
    e.close()
    assert _same(obs, plain[0])
    for f in FIELDS:
        np.testing.assert_array_equal(a[f], plain[1][f], err_msg=f)

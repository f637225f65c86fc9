"""The rotation of a spin about its field at every angle: atoms out of each
other's reach in an external field, whose core_ds is two rotations by |H| dt / 2
hbar, against the Rodrigues formula in long double.

In units of 2^-53: an angle is off by the roundings of dt / hbar, of its product
with H, of the square and of the root, together below 1.25 of it; the two
rotations themselves round a few times, 4 allowed, of which the spin's length
takes part in the latter only."""
import numpy as np
import pytest

from spilady_amd import abi, configs
from spilady_amd.constants import HBAR
from spilady_amd.engine import Engine

pytestmark = pytest.mark.gpu

U = 2.0 ** -53
DT = 1e-15


@pytest.fixture(scope="module")
def isolated():
    n, spacing = 14, 9.0
    r = np.stack(np.meshgrid(*[np.arange(n)] * 3, indexing="ij"), axis=-1).reshape(-1, 3) * spacing + spacing / 2
    rng = np.random.default_rng(4)
    s = rng.normal(size=r.shape)
    s *= 1.1 / np.linalg.norm(s, axis=1, keepdims=True)
    v = configs.fe_variables(300.0, 3, thermostats=False)
    v["extfield"] = 1
    p = abi.params_from_variables(v, [n * spacing, 0.0, n * spacing, 0.0, 0.0, n * spacing], len(r))
    e = Engine(p, dict(r=r, p=np.zeros_like(r), s=s, f=np.zeros_like(r)), compute_initial_forces=True)
    yield e, r, s, rng
    e.close()


def _turn(isolated, angle):
    e, r, s, rng = isolated
    axis = rng.normal(size=r.shape)
    axis /= np.linalg.norm(axis, axis=1, keepdims=True)
    H = axis * (angle * rng.uniform(0.8, 1.2, len(r)) * HBAR / (DT / 2))[:, None]
    e.set_external(H, None)
    e.upload(dict(r=r, p=np.zeros_like(r), s=s))
    e.core_ds(DT)
    got = e.download()["s"].astype(np.longdouble)
    S = s.astype(np.longdouble)
    length = np.sqrt((got ** 2).sum(axis=1) / (S ** 2).sum(axis=1)) - 1
    return H, S, got, np.sqrt((length ** 2).mean())


@pytest.mark.parametrize("angle", [0.01, 0.3, 0.9, 1.5, 2.5, 5.0, 10.0, 30.0, 100.0, 1000.0, 1e4])
def test_rotation(isolated, angle):
    H, S, got, length = _turn(isolated, angle)
    w = -(np.longdouble(DT) / 2 / np.longdouble(HBAR)) * H.astype(np.longdouble)
    t = np.sqrt((w * w).sum(axis=1, keepdims=True))
    k = w / t
    want = S * np.cos(2 * t) + np.cross(k, S) * np.sin(2 * t) + k * (k * S).sum(axis=1, keepdims=True) * (1 - np.cos(2 * t))
    err = np.sqrt(((got - want) ** 2).sum(axis=1).mean()) / 1.1
    assert err <= U * (1.25 * 2 * angle + 4.0), (err, U)
    assert length <= 4.0 * U, (length, U)


@pytest.mark.parametrize("angle", [1e12, 1e16, 1e30])
def test_an_angle_without_meaning_is_still_a_rotation(isolated, angle):
    _, _, _, length = _turn(isolated, angle)
    assert length <= 4.0 * U, (length, U)

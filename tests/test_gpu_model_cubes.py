"""The cubes of the pair spline in the device's tables are rounded once. Pairs of
atoms out of everyone else's reach feel one knot's spline alone, with the
coefficient 1: their force is the table's 6-point derivative, whose noise is the
rounding of its cubes. The reference evaluates the same stencil at the same
points (doubles, as the device places them) with long double cubes.

A correctly rounded cube is uniform within half a place, 1/sqrt(12) of one root
mean square; the stencil adds 2 x (45^2 + 9^2 + 1) such squares over 60 dx, and the
interpolation takes w and 1 - w of two entries. 1.2 of that is allowed (512 pairs:
1 +- 0.03); d * d * d rounds twice and has 1.4."""
import numpy as np
import pytest

from spilady_amd import fit

from test_gpu_model_knots import VR, _pairs

pytestmark = pytest.mark.gpu

N = 1000000
RMAX = 4.1001   # rcut_max of the potential fit
LD = np.longdouble


def _entry(R, n):
    """value of the derivative entry n, and its expected rounding"""
    x = RMAX / N * (n + 1).astype(np.float64)
    dx = x / 1000.0
    c = lambda p: np.maximum(LD(R) - p.astype(LD), 0) ** 3
    d = LD(0)
    for k, w in ((1, 45), (2, -9), (3, 1)):
        step = float(k) * dx
        d = d + w * (c(x + step) - c(x - step))
    place = np.spacing(np.maximum(R - x, 1e-3) ** 3)
    return d / (60 * dx.astype(LD)), np.sqrt(2 * (45 ** 2 + 9 ** 2 + 1) / 12.0) * place / (60 * dx)


@pytest.mark.parametrize("k", [0, 2])
def test_cubes_are_rounded_once(k):
    at, pull, _ = _pairs(2.6, 90 + k, n=8)
    rng = np.random.default_rng(91 + k)
    axis = pull[1::2]
    mid = 0.5 * (at.r[0::2] + at.r[1::2])
    half = 0.5 * rng.uniform(2.1, 2.9, len(mid))[:, None] * axis
    at.r = np.stack([mid - half, mid + half], axis=1).reshape(-1, 3)
    th = np.zeros(fit.NPARAM)
    th[6 + k] = 1.0
    th[17] = 3.75
    m = fit.PotentialModel([at])
    m.set_params(th)
    _, F, _ = m.eval()
    m.close()
    rij = (at.r[1::2] - at.r[0::2]).astype(LD)
    r = np.sqrt((rij ** 2).sum(axis=1))
    got = -(F[1::2].astype(LD) * rij).sum(axis=1) / r
    fn = r * LD(N / RMAX)
    n = fn.astype(np.int64)
    w = (n + 1) - fn
    a, ea = _entry(VR[k], n - 1)
    b, eb = _entry(VR[k], n)
    err = (got - (a * w + b * (1 - w))) / np.sqrt((ea * w) ** 2 + (eb * (1 - w)) ** 2)
    assert np.sqrt((err ** 2).mean()) <= 1.2, np.sqrt((err ** 2).mean())

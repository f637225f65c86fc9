"""The gradient of the pair splines and of the exchange amplitude for pairs near
a knot, against differences of the forward pass. Energies, forces and fields are
linear in these parameters, so a central difference of any width is the exact
derivative of the interpolated tables that the forward pass reads, up to rounding.

The configuration is pairs of atoms r apart and out of everyone else's reach,
r within 0.2 % of the knot R, pulled along their axis: the component of knot R is
the sum of the splines' derivatives there. The bound on a pair is the rounding of
a table's derivative entry (its 6-point stencil adds 110 values of magnitude v in
units of 60 dx) over the width of the difference, and a few ulp of the basis
function's own derivative and of the forces."""
import numpy as np
import pytest

from spilady_amd import configs, fit

pytestmark = pytest.mark.gpu

U = 2.0 ** -53
VR = (4.1, 3.8, 3.5, 3.2, 2.9, 2.6, 2.4, 2.3)
WIDTH = 1000.0


def _pairs(knot, seed, n=6, spacing=9.0):
    rng = np.random.default_rng(seed)
    site = np.stack(np.meshgrid(*[np.arange(n)] * 3, indexing="ij"), axis=-1).reshape(-1, 3) * spacing + spacing / 2
    axis = rng.normal(size=site.shape)
    axis /= np.linalg.norm(axis, axis=1, keepdims=True)
    r = knot * (1.0 + rng.uniform(-0.002, 0.002, len(site)))
    at = configs.make_bcc_fe(5, 300.0, seed)
    half = 0.5 * r[:, None] * axis
    at.r = np.stack([site - half, site + half], axis=1).reshape(-1, 3)
    k = len(at.r)
    at.box = [n * spacing, 0.0, n * spacing, 0.0, 0.0, n * spacing]
    at.p = np.zeros((k, 3))
    at.s = np.stack([np.array([0.0, 0.0, 1.1]), np.array([0.6, 0.0, 0.9])])[np.arange(k) % 2]
    for f in ("f", "heff_h", "heff_l"):
        setattr(at, f, np.zeros((k, 3)))
    for f in ("rho", "pe", "ke", "me", "me0"):
        setattr(at, f, np.zeros(k))
    at.stress = np.zeros((k, 6))
    # along the axis, outwards: every pair's terms have the same sign
    pull = np.stack([-axis, axis], axis=1).reshape(-1, 3)
    return at, pull, r


def _difference(m, th, k, gF):
    side = []
    for sign in (1.0, -1.0):
        t = th.copy()
        t[k] += sign * WIDTH
        m.set_params(t)
        _, F, _ = m.eval()
        side.append(F)
    round_off = 16.0 * U * np.abs(side).sum() / WIDTH  # of the forces and of their sum
    return float((gF * ((side[0] - side[1]) / (2.0 * WIDTH))).sum()), round_off


# knots past the quintic bridge; r below rcut_pot for the first
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 6, 7])
def test_pair_spline_near_its_knot(k):
    R = VR[k]
    at, pull, r = _pairs(R, 50 + k)
    th = fit.default_params()
    m = fit.PotentialModel([at])
    m.set_params(th)
    got = m.vjp(None, pull, None)[6 + k]
    want, round_off = _difference(m, th, 6 + k, pull)
    m.close()
    d = np.maximum(1.004 * R - r, 0.0)       # how far the stencil reaches inside
    v = sum(abs(th[6 + q]) * np.maximum(VR[q] - r + 0.01, 0.0) ** 3 for q in range(8))
    entry = 110.0 * 4.0 * U * (v / WIDTH + d ** 3) / (60.0 * 1e-3 * r)
    bound = round_off + 2.0 * np.sum(entry + 16.0 * U * 3.0 * d * d)
    assert abs(got - want) <= bound, (got, want, bound)


def test_exchange_amplitude_near_its_cutoff():
    th = fit.default_params()
    A, rc = th[16], th[17]
    at, pull, r = _pairs(rc, 60)
    m = fit.PotentialModel([at])
    m.set_params(th)
    got = m.vjp(None, pull, None)[16]
    want, round_off = _difference(m, th, 16, pull)
    m.close()
    s = at.s[:2]
    x = abs(s[0] @ s[1] - np.linalg.norm(s[0]) * np.linalg.norm(s[1]))
    q = np.maximum(1.004 - r / rc, 0.0)
    v = sum(abs(th[6 + k]) * np.maximum(VR[k] - r + 0.01, 0.0) ** 3 for k in range(8))
    entry = 110.0 * 8.0 * U * (v / WIDTH + x * (abs(A) / WIDTH + 1.0) * q ** 3) / (60.0 * 1e-3 * r)
    bound = round_off + 2.0 * np.sum(entry + 32.0 * U * x * 3.0 * q * q / rc)
    assert abs(got - want) <= bound, (got, want, bound)

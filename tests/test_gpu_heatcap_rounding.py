"""E(T) and T(E) of the electron mesh as the device leaves them in a cell,
against long double: no bias and about one rounding, so that the conversions of a
run do not add up. In units of 2^-53 of the value: the product and the sums that
make either function round three times, each by up to half a unit in the last
place, 0.4 root mean square over the values' mantissas, and the polynomials' other
terms are smaller: 0.7 in all, 1.0 allowed. A coefficient rounded badly is a bias
of a whole unit; a quarter is allowed."""
import numpy as np
import pytest

from spilady_amd.constants import BOLTZ
from spilady_amd.engine import Engine

from test_gpu_dte_tiles import _system

pytestmark = pytest.mark.gpu

B = np.longdouble(2e-4 / BOLTZ)
U = np.longdouble(2.0) ** -53


def _check(got, want, what):
    err = (got.astype(np.longdouble) - want) / want / U
    assert abs(err.mean()) <= 0.25 and np.sqrt((err ** 2).mean()) <= 1.0, (what, err.mean(), np.sqrt((err ** 2).mean()))


@pytest.mark.parametrize("cells", [(10, 10, 10), (23, 22, 21)])   # one workgroup; tiles
def test_conversions_have_no_bias(cells):
    p, at = _system(cells)
    e = Engine(p, at, compute_initial_forces=True)
    n = int(np.prod(cells))
    te = BOLTZ * np.random.default_rng(3).uniform(100.0, 4000.0, n)
    e.set_cells_te(te)
    c = e.cells()
    x = B * te.astype(np.longdouble)
    _check(c["ee"], 3 / B * np.log1p(2 * np.sinh(x / 2) ** 2), "E(T)")
    e.core_dTe(0.5e-15)
    c = e.cells()
    y = B / 3 * c["ee"].astype(np.longdouble)
    _check(c["te"], (y + np.log1p(np.sqrt(-np.expm1(-2 * y)))) / B, "T(E)")
    e.close()

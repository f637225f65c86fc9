"""The model's passes over one large context (several rounds of atoms a block,
a last round and a last block that are not full) against its configurations
each alone: the same pairs in sums of another order. A gradient component adds
up to 10^6 terms of either sign, about 150 times larger together than a
configuration's result: roundings of 1e-16 stay below TOL of the results'
absolute sum."""
import numpy as np
import pytest

from spilady_amd import fit

from helpers import TOL, assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(5,), (5, 7, 6), (8,) * 33, (11,) * 26, (7, 9, 8) * 30])
def test_a_large_context_is_the_sum_of_its_configurations(sizes):
    confs = [fit.frozen_configs(n, [400 + k])[0] for k, n in enumerate(sizes)]
    th = fit.perturbed_params(fit.default_params(), 0.02, 7)
    rng = np.random.default_rng(len(sizes))
    nat = [len(c.r) for c in confs]
    gE = rng.normal(size=len(confs))
    gF = rng.normal(size=(sum(nat), 3))
    gH = rng.normal(size=(sum(nat), 3))
    m = fit.PotentialModel(confs)
    m.set_params(th)
    E, F, H = m.eval()
    g = m.vjp(gE, gF, gH)
    m.close()
    one = []
    off = 0
    for k, c in enumerate(confs):
        m = fit.PotentialModel([c])
        m.set_params(th)
        e, f, h = m.eval()
        assert abs(E[k] - e[0]) <= TOL * abs(e[0])
        assert_close(f, F[off:off + nat[k]], f"force {k}")
        assert_close(h, H[off:off + nat[k]], f"field {k}")
        one.append(m.vjp(gE[k:k + 1], gF[off:off + nat[k]], gH[off:off + nat[k]]))
        off += nat[k]
        m.close()
    one = np.array(one)
    assert np.all(np.abs(g - one.sum(axis=0)) <= TOL * np.abs(one).sum(axis=0))

"""Momentum and kinetic-energy sums of a replica: added inside the next kernel
for replicas of few partial sums, by a launch of their own in a batch that also
holds a larger one (more than 4,096 link cells). Bitwise the same either way."""
import numpy as np
import pytest

from spilady_amd import abi, configs
from spilady_amd.engine import BatchEngine, Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("small,large", [(5, 26), (11, 26), (22, 26)])
def test_small_replica_beside_a_large_one(small, large):
    reps = []
    for k, nu in enumerate((small, large)):
        at = configs.make_bcc_fe(nu, 300.0, 60 + k, tilt_max_deg=30.0)
        v = configs.fe_variables(300.0, k, thermostats=True)
        reps.append((abi.params_from_variables(v, at.box, at.natom, replica=k), at))
    b = BatchEngine([p for p, _ in reps], [a for _, a in reps], compute_initial_forces=True)
    one = Engine(*reps[0], compute_initial_forces=True)
    for e in (b, one):
        e.core_dp(1e-15)
        e.core_dp(1e-15)
    want, got = one.download(), b.download_replica(0)
    one.close()
    b.close()
    for f in ("p", "ke"):
        np.testing.assert_array_equal(want[f], got[f], err_msg=f)

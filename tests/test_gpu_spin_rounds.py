"""The spin sweep with many cells a wave: uneven cells whose atoms fill a wave's
64 lanes and overflow into further passes, against the same replica alone,
where a wave takes one cell. A cell's rounds and sums depend on its own atoms
only, so the two are bitwise the same."""
import numpy as np
import pytest

from spilady_amd import abi, configs
from spilady_amd.constants import FE_A_LATTICE
from spilady_amd.engine import BatchEngine, Engine

pytestmark = pytest.mark.gpu


def _replica(k, nu, thermostats):
    """A lattice with a third of its 2 x 2 x 2 blocks empty: cells of 0 to 11 atoms."""
    at = configs.make_bcc_fe(nu, 300.0, 50 + k, tilt_max_deg=60.0)
    block = np.floor(at.r / (2 * FE_A_LATTICE) + 1e-9).astype(int).sum(axis=1)
    keep = block % 3 != k % 3
    n = int(keep.sum())
    v = configs.fe_variables(300.0 + k, k, thermostats=thermostats)
    p = abi.params_from_variables(v, at.box, n, replica=k)
    return p, dict(r=at.r[keep], p=np.zeros((n, 3)), s=at.s[keep], f=np.zeros((n, 3)))


@pytest.mark.parametrize("nu,nrep", [(12, 72), (10, 170)])
@pytest.mark.parametrize("spin_block", [32, 64, 128])
@pytest.mark.parametrize("thermostats", [True, False])
def test_many_cells_a_wave_equal_one(nu, nrep, spin_block, thermostats):
    reps = [_replica(k, nu, thermostats) for k in range(nrep)]
    b = BatchEngine([p for p, _ in reps], [a for _, a in reps], compute_initial_forces=True)
    b.set_shapes(dict(spin_block=spin_block, spin_lanes=1))
    b.core_ds(1e-15)
    for k in (0, 1, nrep // 2, nrep - 1):
        one = Engine(*reps[k], compute_initial_forces=True)
        one.core_ds(1e-15)
        want, got = one.download(), b.download_replica(k)
        one.close()
        for f in ("s", "heff_h", "heff_l"):
            np.testing.assert_array_equal(want[f], got[f], err_msg=f"replica {k} {f}")
    b.close()

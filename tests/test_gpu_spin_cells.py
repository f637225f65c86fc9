"""core_ds over cells of very different occupation (empty ones, ones of up to
30 atoms next to them), so that a wave's cells need several passes through
LDS, odd link-cell counts, and angles past the series' range, against the
oracle. Both sweeps run in the same order; a field is summed in another order
and corrected, a few roundings of 1e-16 an atom, far below TOL."""
import numpy as np
import pytest

from spilady_amd import abi, configs
from spilady_amd.constants import FE_A_LATTICE
from spilady_amd.engine import Engine
from oracle import orcpy

from helpers import assert_close

pytestmark = pytest.mark.gpu


def _system(nu, kind, thermostats):
    rng = np.random.default_rng(17)
    at = configs.make_bcc_fe(nu, 300.0, 9, tilt_max_deg=60.0)
    r, s = at.r, at.s
    if kind == "clumps":
        # half the atoms drawn towards the middle of coarse blocks, the other
        # half removed from them: cells of 0 to about 25 atoms, none closer
        # than 2.2 A so that the neighbour lists hold them
        block = 3 * FE_A_LATTICE
        mid = (np.floor(r / block) + 0.5) * block
        r = mid + 0.93 * (r - mid)
    keep = np.ones(len(r), bool)
    if kind == "holes":
        c = np.floor(r / (2 * FE_A_LATTICE)).astype(int).sum(axis=1)
        keep = (c % 3 != 0) | (rng.random(len(r)) < 0.1)
    r, s = r[keep], s[keep]
    n = len(r)
    v = configs.fe_variables(300.0, 9, thermostats=thermostats)
    p = abi.params_from_variables(v, at.box, n)
    return p, dict(r=r, p=np.zeros((n, 3)), s=s, f=np.zeros((n, 3)))


@pytest.mark.parametrize("nu,kind", [(5, "full"), (7, "clumps"), (9, "holes"), (12, "clumps"), (13, "full")])
@pytest.mark.parametrize("thermostats,dt", [(True, 1e-15), (False, 1e-15), (False, 3e-14)])
def test_core_ds_matches_the_oracle(nu, kind, thermostats, dt):
    p, at = _system(nu, kind, thermostats)
    o = orcpy.Oracle(p, at, compute_initial_forces=True, rng=orcpy.RNG_PHILOX)
    e = Engine(p, at, compute_initial_forces=True)
    for k in range(2):
        o.core_ds(dt)
        e.core_ds(dt)
    a, b = o.download(), e.download()
    o.close()
    e.close()
    # a step of 3e-14 s turns a spin by tens of radians: the angle's rounding
    # is that much larger
    tol = 1e-10 if dt < 1e-14 else 1e-8
    for k in ("s", "heff_h"):
        assert_close(a[k], b[k], f"{kind} {k}", tol)


def test_waves_of_several_passes_equal_single_cells():
    """312 replicas whose cells hold 16 atoms each: levels of 8,424 cells put
    five cells (80 atoms, 600 pairs) on a wave, more than a pass holds. Alone,
    a replica's levels have 27 cells and a wave takes one: bitwise the same."""
    nu, nrep = 12, 312
    plist, alist = [], []
    for k in range(nrep):
        at = configs.make_bcc_fe(nu, 300.0, 1000 + k, tilt_max_deg=40.0)
        v = configs.fe_variables(300.0 + k, k, thermostats=True)
        v["min_length_link_cell"] = 5.7
        plist.append(abi.params_from_variables(v, at.box, at.natom, replica=k))
        alist.append(at)
    from spilady_amd.engine import BatchEngine
    b = BatchEngine(plist, alist, compute_initial_forces=True)
    assert b.ncell3 == (6, 6, 6) and np.max(b.cell_lists()[0]) == 16
    b.core_ds(0.5e-15)
    for k in (0, 1, 157, 311):
        one = Engine(plist[k], alist[k], compute_initial_forces=True)
        one.core_ds(0.5e-15)
        want, got = one.download(), b.download_replica(k)
        one.close()
        for f in ("s", "heff_h", "heff_l"):
            np.testing.assert_array_equal(want[f], got[f], err_msg=f"replica {k} {f}")
    b.close()

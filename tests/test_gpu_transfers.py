"""Arrays through sld_upload / sld_download: exact values at sizes around a
block (256 elements) and past a transfer piece (2^20 doubles), any subset of
arrays, replicas in the middle of the slots."""
import numpy as np
import pytest

from spilady_amd import abi, configs
from spilady_amd.engine import BatchEngine, Engine

pytestmark = pytest.mark.gpu


def _make(n_unit, seed=3):
    at = configs.make_bcc_fe(n_unit, 300.0, seed)
    v = configs.fe_variables(300.0, seed, thermostats=False)
    return abi.params_from_variables(v, at.box, at.natom), at


@pytest.mark.parametrize("n_unit", [5, 8, 13, 56])   # 250, 1,024, 4,394 and 351,232 atoms (1.05 M doubles a vector)
def test_round_trip_is_exact(n_unit):
    p, at = _make(n_unit)
    rng = np.random.default_rng(n_unit)
    stress = rng.normal(size=(at.natom, 6))
    at.stress = stress
    e = Engine(p, at)
    d = e.download()
    for k in ("r", "p", "s"):
        np.testing.assert_array_equal(d[k], getattr(at, k))
    np.testing.assert_array_equal(d["stress"], stress)
    new = {k: rng.normal(size=(at.natom, 3)) for k in ("p", "f", "s")}
    new["rho"] = rng.random(at.natom)
    e.upload(new)
    d = e.download()
    for k in new:
        np.testing.assert_array_equal(d[k], new[k])
    np.testing.assert_array_equal(d["r"], at.r)
    e.close()


def test_a_single_array_and_a_middle_replica():
    made = [_make(n, n) for n in (5, 7, 6)]
    b = BatchEngine([p for p, _ in made], [a for _, a in made])
    s = np.random.default_rng(1).normal(size=(made[1][1].natom, 3))
    b.select(1)
    b.upload(dict(s=s))
    for k, (p, a) in enumerate(made):
        d = b.download_replica(k)
        np.testing.assert_array_equal(d["s"], s if k == 1 else a.s)
        np.testing.assert_array_equal(d["p"], a.p)
    out = abi.AtomBuffers({"rho": np.full(made[2][1].natom, -1.0)})
    b.select(2)
    b._rc(b.L.sld_download(b.h, out.view()))
    np.testing.assert_array_equal(out.as_dict()["rho"], b.download()["rho"])
    b.close()

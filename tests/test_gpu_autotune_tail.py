"""The autotuner neither times nor changes sweep_tail, which no launch reads: its
entries repeat the chosen sweep_block's time, and the value that was set stays."""
import pytest

from helpers import consistent_state, fe_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [0, 2048, 8192])
def test_sweep_tail_is_not_tuned(value):
    from spilady_amd.engine import Engine
    v, p, at = fe_params(8, 600.0, 41, thermostats=True, eltemp=True, localcolmot=True)
    e = Engine(p, consistent_state(p, at))
    e.set_shapes(dict(sweep_tail=value))
    best, table = e.autotune(1)
    e.close()
    assert best["sweep_tail"] == value
    assert set(table["sweep_tail"].values()) == {table["sweep_block"][best["sweep_block"]]}

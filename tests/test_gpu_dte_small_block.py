"""Every sweep_block costs a small electron mesh the same: the workgroup that
takes the whole core_dTe call of 10^3 cells does not shrink with it. The launches
are alike, so the fastest of five calls differs by the clock only: 10 % allowed,
where a workgroup of a quarter of the threads takes 2.4 times as long."""
import pytest

from spilady_amd.engine import Engine

from test_gpu_dte_tiles import _system

pytestmark = pytest.mark.gpu


def test_sweep_block_does_not_slow_a_small_mesh():
    p, at = _system((10, 10, 10))
    e = Engine(p, at, compute_initial_forces=True)
    e.time_kernel("k_dte_sweep")
    ms = {}
    for block in (256, 128, 64):
        e.set_shapes(dict(sweep_block=block))
        calls = []
        for _ in range(5):
            e.core_dTe(0.5e-15)
            calls.append(e.kernel_timing()[1])
        ms[block] = min(calls)
    e.close()
    assert max(ms.values()) <= 1.1 * min(ms.values()), ms

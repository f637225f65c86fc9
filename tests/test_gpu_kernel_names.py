"""sld_time_kernel by the names of the electron diffusion's kernels: a small
mesh's one launch a core_dTe call answers to its own name and the sweeps', a
tiled mesh's launches to the sweeps' only."""
import pytest

from spilady_amd.engine import Engine

from test_gpu_dte_tiles import _system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,small", [((7, 7, 7), True), ((12, 12, 12), False)])
def test_names_of_the_diffusion(cells, small):
    p, at = _system(cells)
    e = Engine(p, at, compute_initial_forces=True)
    n = {}
    for name in ("k_dte_small", "k_dte_sweep"):
        e.time_kernel(name)
        e.core_dTe(0.5e-15)
        n[name], ms = e.kernel_timing()
        assert (ms > 0.0) == (n[name] > 0)
    e.close()
    assert n["k_dte_small"] == (1 if small else 0)
    assert n["k_dte_sweep"] == 1 if small else n["k_dte_sweep"] in (50, 100)

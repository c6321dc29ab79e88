"""Membrane cycles (M) far longer than any run."""
import numpy as np
import pytest

from tests.pairs import gpu_of, small_cells

pytestmark = pytest.mark.gpu


def _free():
    """Bytes free on the device, from the runtime that the library uses."""
    import ctypes as C
    from preprocess_src_amd import native
    free, total = C.c_size_t(), C.c_size_t()
    assert native.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("m", [2 ** 30, 2 ** 31 - 2, 2 ** 31 - 1])
def test_cycles_longer_than_a_run_cost_no_memory(m):
    """The steps' values are kept for the blocks that are replayed, and a cycle
    longer than the run is not; the run is the eager one."""
    shape = (24, 18, 22)
    cells = small_cells(*shape, nc=2, radius=3.0)
    print(f"[cycle] {m}", flush=True)
    before = _free()
    sims = [gpu_of(*shape, "f64", cells=cells, m=m, p=1e-5, b=5e-3) for _ in range(2)]
    assert before - _free() < 1 << 30
    for sim, graph in zip(sims, (True, False)):
        sim.volume_init()
        sim.run(0, 12, graph=graph)
    assert np.array_equal(sims[0].populations(), sims[1].populations())
    for sim in sims:
        sim.close()

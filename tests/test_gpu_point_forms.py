"""The two forms of the point-by-point interpolation (FP32 values under an
indicator)."""
import numpy as np
import pytest

from tests.pairs import gpu_of, rel
from tests.test_gpu_paths import _advected, _scattered

pytestmark = pytest.mark.gpu


def _advect(shape, nc, amp, runge_kutta=4, **kw):
    """Velocities of vertices in a rough field, and the same in plain FP64."""
    lx, ly, lz = shape
    cells, pos = _scattered(lx, ly, lz, nc, 2, seed=2)
    if nc > 2:  # crowd them into two tiles
        pos = [(p / v) * w + o for p, v, w, o in zip(pos, shape, (14.0, 6.0, 6.0), (1.0, 0.0, 1.0))]
    g = gpu_of(lx, ly, lz, "f32", cells=cells, vof_period=1000, runge_kutta=runge_kutta, **kw)
    g.set_cells_state(x=pos[0], y=pos[1], z=pos[2])
    U = amp * np.random.default_rng(9).standard_normal((3, lz, ly, lx))
    pad = np.zeros((3, lz + 4, ly + 4, lx + 4))
    pad[:, 2:-2, 2:-2, 2:-2] = U
    g.set_macros(*[a.reshape(-1) for a in pad])
    g.ibm_st2()
    s = g.cells_state()
    report = g.autotune_report()
    g.close()
    return s, _advected(np.stack(pos, 1), U, shape), report


# slow: the stages stay in a cell; fast: they leave it, and the staged box
@pytest.mark.parametrize("amp", [0.02, 1.5, 6.0])
@pytest.mark.parametrize("shape,nc", [((9, 8, 17), 2), ((16, 8, 8), 1), ((40, 24, 40), 11), ((50, 23, 31), 2)])
def test_the_two_forms_give_the_same_bits(shape, nc, amp, monkeypatch):
    print(f"[point forms] {shape} {amp}", flush=True)
    out = []
    for form in "01":
        monkeypatch.setenv("LBMIBM_INTERP_FORM", form)
        s, ref, report = _advect(shape, nc, amp)
        assert "fixed by LBMIBM_INTERP_FORM" in report
        out.append(s)
    for k in ("x", "y", "z", "u", "v", "w", "xd"):
        assert np.array_equal(out[0][k], out[1][k]), k
    if amp < 2.0:  # FP32: the bound of the rough field of 1.5 in test_gpu_paths; slower fields come nearer
        for d, k in enumerate("uvw"):
            assert rel(out[0][k], ref[:, d]) < 3e-5, k


def test_both_forms_are_timed(monkeypatch):
    """No form is taken unseen: 3204 vertices prefer rows from memory, those of a
    thousand cells tiles in LDS."""
    for name in ("LBMIBM_INTERP_FORM", "LBMIBM_AUTOTUNE"):
        monkeypatch.delenv(name, raising=False)
    _, _, report = _advect((40, 24, 40), 11, 0.02)
    for line in ("interp form tiles in LDS: ", "interp form rows from memory: ", "interp: using "):
        assert line in report

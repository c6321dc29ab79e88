"""The sums of the spreading: what they are rounded to, and that their bits do
not depend on the order in which the binning places the vertices."""
import numpy as np
import pytest

from tests.pairs import gpu_of
from tests.test_gpu_paths import CROWDS, _crowded

pytestmark = pytest.mark.gpu

SHAPE = (48, 40, 40)
EPS = {"f64": 2.0 ** -53, "f32": 2.0 ** -24}  # half a unit in the last place, relative


def _on_nodes(level, lo, hi, seed, on_node=None):
    """One cell whose vertices sit on lattice nodes lo <= i <= hi: their weights
    are 1/4, 1/2, 1/4 per axis, with no rounding."""
    from preprocess_src_amd import mesh
    cells = mesh.assemble([level], np.zeros((1, 3)), np.eye(3)[None], 3.0)
    rng = np.random.default_rng(seed)
    n = cells["x"].size
    at = np.stack([rng.integers(a, b + 1, n) for a, b in zip(lo, hi)], 1)
    return cells, at, [at[:, d] - (SHAPE[d] - 1) / 2.0 for d in range(3)]


def _exact(at, force):
    """Sums of the forces on each node with those weights, and of their absolute
    values: whole numbers of 2^-6 of the force's unit, in 64-bit integers."""
    lx, ly, lz = SHAPE
    s, a = np.zeros((2, lz, ly, lx), np.int64)
    w = {-1: 1, 0: 2, 1: 1}
    for i in w:
        for j in w:
            for k in w:
                q = w[i] * w[j] * w[k]
                idx = (at[:, 2] + k, at[:, 1] + j, at[:, 0] + i)
                np.add.at(s, idx, q * force)
                np.add.at(a, idx, q * np.abs(force))
    return s, a


def _spread(prec, cells, pos, forces):
    g = gpu_of(*SHAPE, prec, cells=cells)
    g.set_cells_state(x=pos[0], y=pos[1], z=pos[2], fx=forces[0], fy=forces[1], fz=forces[2])
    g.ibm_st1()
    F = [f.reshape(SHAPE[2] + 4, SHAPE[1] + 4, SHAPE[0] + 4)[2:-2, 2:-2, 2:-2] for f in g.lattice_force()]
    g.close()
    return F


# vertices of one tile (nodes 9..16 of each axis, whose stencils start in 8..15)
# below the share of 800, shared out between 4 and 13 work groups, and in so few
# lattice cells that a chunk does not fit the sort
FULL = [(3, (9, 9, 9), (16, 16, 16)), (4, (9, 9, 9), (16, 16, 16)), (5, (9, 9, 9), (16, 16, 16)),
        (5, (11, 12, 12), (12, 13, 12))]


@pytest.mark.parametrize("signs", ["one", "by stretch"])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("k", range(len(FULL)))
def test_sum_of_one_tile_is_rounded_once(k, prec, signs, monkeypatch):
    """The forces of a tile's vertices on a node, whole numbers here, are summed
    exactly and rounded once, however many work groups share the tile: half a
    unit in the last place of the result and the quantum of the fixed point
    (one per term: 2^-46 of the bound that the scale is taken from in FP32,
    2^-61 in FP64)."""
    monkeypatch.setenv("LBMIBM_SPREAD_FORM", "1")
    level, lo, hi = FULL[k]
    print(f"[one tile] {k} {prec} {signs}", flush=True)
    cells, at, pos = _on_nodes(level, lo, hi, 3 + k)
    n = len(at)
    rng = np.random.default_rng(k)
    forces = []
    for _ in range(3):
        f = rng.integers(1, 1 << 22, n)
        if signs != "one":  # the sums of the lower and the upper half nearly cancel
            f = np.where(at[:, 2] <= (lo[2] + hi[2]) / 2 if hi[2] > lo[2] else at[:, 0] <= lo[0], f, -f)
        forces.append(f)
    F = _spread(prec, cells, pos, [f.astype(np.float64) for f in forces])
    bound = n * float(1 << 22) / 8.0
    quantum = n * bound * 2.0 ** (-46 if prec == "f32" else -61)
    for got, f in zip(F, forces):
        s, _ = _exact(at, f)
        want = s / 64.0  # exact: fewer than 53 bits
        assert np.all(np.abs(got - want) <= EPS[prec] * np.abs(want) + quantum)


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_sum_of_several_tiles_is_rounded_once(prec, monkeypatch):
    """Vertices around a corner of eight tiles: whole-number forces whose sums
    fit 24 bits in every tile's box, but not together.  The nodes hold the
    exact sum rounded once."""
    monkeypatch.setenv("LBMIBM_SPREAD_FORM", "1")
    print(f"[eight tiles] {prec}", flush=True)
    cells, at, pos = _on_nodes(3, (16, 16, 16), (17, 17, 17), 11)  # stencils start in 15 and 16, the tiles at 16
    tile = ((at == 17) * [1, 2, 4]).sum(1)
    T = np.float32 if prec == "f32" else np.float64
    rng = np.random.default_rng(2)
    wide = 0
    for _ in range(8):
        forces = [rng.integers(1 << 14, 1 << 15, len(at)) >> 1 for _ in range(3)]
        F = _spread(prec, cells, pos, [f.astype(np.float64) for f in forces])
        for got, f in zip(F, forces):
            for t in range(8):
                assert _exact(at[tile == t], f[tile == t])[1].max() < 1 << 24
            s = _exact(at, f)[0]
            wide += int((s >= 1 << 24).sum())
            assert np.array_equal(got, (s / 64.0).astype(T).astype(np.float64))
    assert wide >= 100  # sums that FP32 does not hold


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("k", [1, 3, 4, 5])
def test_home_boxes_do_not_depend_on_the_order_of_the_binning(k, prec, monkeypatch):
    """Tiles of more than 800 vertices, cells of many, chunks beyond the sort's
    capacity: every repeated binning places a tile's vertices in the order in
    which its work groups arrive; the lattice force keeps its bits."""
    monkeypatch.setenv("LBMIBM_SPREAD_FORM", "1")
    levels, lo, hi = CROWDS[k]
    print(f"[binning order] {k} {prec}", flush=True)
    cells, pos = _crowded(*SHAPE, levels, 17 + k, lo, hi)
    rng = np.random.default_rng(4)
    n = pos[0].size
    forces = [1e-3 * rng.standard_normal(n) * 10.0 ** rng.uniform(-4, 0, n) for _ in range(3)]
    g = gpu_of(*SHAPE, prec, cells=cells)
    first = None
    for _ in range(8):
        g.set_cells_state(x=pos[0], y=pos[1], z=pos[2], fx=forces[0], fy=forces[1], fz=forces[2])
        g.ibm_st1()
        F = np.concatenate(g.lattice_force())
        if first is None:
            first = F
        assert np.array_equal(F, first)
    g.close()
    assert np.abs(first).max() > 0.0


@pytest.mark.parametrize("form", [0, 1])
def test_more_tiles_than_the_scan_takes_at_once(form, monkeypatch):
    """4913 tiles, 4096 at a time and four per thread, an odd number of them: full
    tiles on both sides of the border and in the last rows, nearly all others empty."""
    monkeypatch.setenv("LBMIBM_SPREAD_FORM", str(form))
    shape = (135, 135, 129)
    print(f"[many tiles] form={form}", flush=True)
    from preprocess_src_amd import mesh
    cells = mesh.assemble([4, 4, 4, 3], np.zeros((4, 3)), np.repeat(np.eye(3)[None], 4, 0), 3.0)
    rng = np.random.default_rng(8)
    n = cells["x"].size
    at = rng.uniform(0.0, 1.0, (n, 3)) * 7.0
    per = np.repeat(np.arange(4), np.diff(cells["voff"]))
    # tiles 4095 and 4096 (x = 15 and 16, y = 2, z = 14), the last rows, anywhere
    corner = np.array([[121.0, 17.0, 113.0], [129.0, 17.0, 113.0], [128.0, 128.0, 121.0]])
    at[per < 3] += corner[per[per < 3]]
    at[per == 3] = rng.uniform(0.0, 1.0, ((per == 3).sum(), 3)) * (np.array(shape) - 1.0)
    forces = [1e-3 * rng.standard_normal(n) for _ in range(3)]
    pos = [at[:, d] - (shape[d] - 1) / 2.0 for d in range(3)]
    g = gpu_of(*shape, "f64", cells=cells)
    g.set_cells_state(x=pos[0], y=pos[1], z=pos[2], fx=forces[0], fy=forces[1], fz=forces[2])
    g.ibm_st1()
    F = [f.reshape([v + 4 for v in shape[::-1]])[2:-2, 2:-2, 2:-2] for f in g.lattice_force()]
    g.close()
    first = np.floor(at)
    t = np.pi / 2 * (at - first)
    w = np.stack([1 - np.sin(t), 1 + np.cos(t), 1 + np.sin(t), 1 - np.cos(t)], 2) / 4.0
    i = first.astype(int)[:, :, None] - 1 + np.arange(4)
    want = np.zeros((3,) + shape[::-1])
    for a in range(4):
        for b in range(4):
            for c in range(4):
                ok = (i[:, 1, b] >= 0) & (i[:, 1, b] < shape[1])
                q = w[:, 0, a] * w[:, 1, b] * w[:, 2, c] * ok
                idx = (i[:, 2, c] % shape[2], np.clip(i[:, 1, b], 0, shape[1] - 1), i[:, 0, a] % shape[0])
                for d in range(3):
                    np.add.at(want[d], idx, q * forces[d])
    for d in range(3):  # FP64 sums of at most a few thousand terms, as the other spreading tests
        assert np.max(np.abs(F[d] - want[d])) < 1e-11 * np.max(np.abs(want[d]))

"""Kernel paths at the sizes where they can go wrong (tile and work-group
edges, remainders, smallest and largest inputs), against the oracle or a plain
FP64 evaluation."""
import numpy as np
import pytest

from tests.pairs import gpu_of, oracle_of, rel

pytestmark = pytest.mark.gpu


def _scattered(lx, ly, lz, nc, level, seed):
    """nc cells whose vertices lie anywhere in the box, in random order: every
    work group of the binning meets most of the tiles."""
    from preprocess_src_amd import mesh
    c = np.zeros((nc, 3))
    cells = mesh.assemble([level] * nc, c, np.repeat(np.eye(3)[None], nc, 0), 3.0)
    rng = np.random.default_rng(seed)
    n = cells["x"].size
    pos = [rng.uniform(-0.5, 0.5, n) * (v - 1e-6) for v in (lx, ly, lz)]
    return cells, pos


def _spread_both(lx, ly, lz, prec, cells, pos, forces, **kw):
    """Lattice force of the oracle and of the library for the given positions
    and nodal forces (COMP nodes)."""
    o = oracle_of(lx, ly, lz, cells=cells, **kw)
    g = gpu_of(lx, ly, lz, prec, cells=cells, **kw)
    for k, v in zip("xyz", pos):
        o.cells[k][:] = v
    g.set_cells_state(x=pos[0], y=pos[1], z=pos[2])
    for k, v in zip(("cfx", "cfy", "cfz"), forces):
        o.cells[k][:] = v
    g.set_cells_state(fx=forces[0], fy=forces[1], fz=forces[2])
    o.ibm_st1()
    g.ibm_st1()
    comp = o.bc == 0
    F = [f[comp] for f in g.lattice_force()]
    g.close()
    return F, [f[comp] for f in (o.fx, o.fy, o.fz)]


# FP64: sums of at most a few hundred terms, 1e-11 of max |F| as the other
# spreading tests; FP32: the weights' FP32 rounding, 1e-5
SPREAD_TOL = {"f64": 1e-11, "f32": 1e-5}


@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("nc", [1, 6, 7, 13])  # 162, 972, 1134, 2106 vertices: the binning's work groups hold 1024
def test_binning_of_vertices_in_random_order(nc, prec, form, monkeypatch):
    monkeypatch.setenv("LBMIBM_SPREAD_FORM", str(form))
    lx, ly, lz = 64, 40, 64
    print(f"[binning] nc={nc} prec={prec} form={form}", flush=True)
    cells, pos = _scattered(lx, ly, lz, nc, 2, seed=5 + nc)
    rng = np.random.default_rng(3)
    forces = [1e-3 * rng.standard_normal(pos[0].size) for _ in range(3)]
    F, ref = _spread_both(lx, ly, lz, prec, cells, pos, forces)
    for a, b in zip(F, ref):
        assert rel(a, b) < SPREAD_TOL[prec]


def _crowded(lx, ly, lz, levels, seed, lo, hi):
    """Cells whose vertices lie anywhere between the corners lo and hi (in
    lattice nodes of the fluid frame), in random order."""
    from preprocess_src_amd import mesh
    nc = len(levels)
    cells = mesh.assemble(levels, np.zeros((nc, 3)), np.repeat(np.eye(3)[None], nc, 0), 3.0)
    rng = np.random.default_rng(seed)
    n = cells["x"].size
    # node i of an axis of m nodes sits at i - (m - 1) / 2
    return cells, [rng.uniform(a, b, n) - (m - 1) / 2.0 for a, b, m in zip(lo, hi, (lx, ly, lz))]


# corners of the first stencil nodes (a vertex between nodes i and i + 1 starts
# its stencil at i - 1): within two tiles (8 x 8 x 8 nodes) below and above the share
# of 800 vertices that a work group takes, in one lattice cell below and above the
# sort's capacity, and more vertices than 16-bit indices hold; across the lower wall
CROWDS = [([3, 3], (2.0, 9.0, 9.0), (16.9, 16.9, 16.9)), ([4, 4], (2.0, 9.0, 9.0), (16.9, 16.9, 16.9)),
          ([3], (5.1, 12.1, 12.1), (5.9, 12.9, 12.9)), ([4], (5.1, 12.1, 12.1), (5.9, 12.9, 12.9)),
          ([5, 3], (5.1, 12.1, 12.1), (6.9, 12.9, 12.9)), ([5] * 7, (2.0, 9.0, 9.0), (16.9, 16.9, 16.9)),
          ([4, 4], (2.0, -0.5, 9.0), (16.9, 1.0, 16.9))]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("k", range(len(CROWDS)))
def test_spread_of_crowded_tiles(k, prec, monkeypatch):
    """Home boxes summed per lattice cell: tiles and cells around the
    capacities of the sort; forces over several decades."""
    monkeypatch.setenv("LBMIBM_SPREAD_FORM", "1")
    levels, lo, hi = CROWDS[k]
    lx, ly, lz = 48, 40, 40
    print(f"[crowd] {k} {prec}", flush=True)
    cells, pos = _crowded(lx, ly, lz, levels, 17 + k, lo, hi)
    rng = np.random.default_rng(4)
    n = pos[0].size
    forces = [1e-3 * rng.standard_normal(n) * 10.0 ** rng.uniform(-4, 0, n) for _ in range(3)]
    F, ref = _spread_both(lx, ly, lz, prec, cells, pos, forces)
    for a, b in zip(F, ref):
        assert rel(a, b) < SPREAD_TOL[prec]


def test_spread_of_crowded_tiles_does_not_depend_on_the_order():
    """Repeated binning places the vertices of a tile in another order; the
    lattice force keeps its bits."""
    lx, ly, lz = 48, 40, 40
    cells, pos = _crowded(lx, ly, lz, [4, 4, 3], 3, (2.0, 2.0, 2.0), (40.0, 34.0, 34.0))
    rng = np.random.default_rng(4)
    forces = [1e-3 * rng.standard_normal(pos[0].size) for _ in range(3)]
    g = gpu_of(lx, ly, lz, "f32", cells=cells)
    out = []
    for _ in range(6):
        g.set_cells_state(x=pos[0], y=pos[1], z=pos[2], fx=forces[0], fy=forces[1], fz=forces[2])
        g.ibm_st1()
        out.append(np.concatenate(g.lattice_force()))
    g.close()
    for a in out[1:]:
        assert np.array_equal(a, out[0])


def _advected(pos, U, shape):
    """RK4 advection (M dt = 1) of positions through a velocity field U [3][z, y,
    x], periodic in x and z, at rest beyond the y walls, in plain FP64."""
    lx, ly, lz = shape

    def vel(X):
        s = X + np.array([(n - 1) / 2.0 for n in shape])  # node i sits at i
        first = np.floor(s)
        t = np.pi / 2 * (s - first)
        w = np.stack([1 - np.sin(t), 1 + np.cos(t), 1 + np.sin(t), 1 - np.cos(t)], 2) / 4.0
        i = first.astype(int)[:, :, None] - 1 + np.arange(4)
        ok = (i[:, 1] >= 0) & (i[:, 1] < ly)
        ix, iy, iz = i[:, 0] % lx, np.clip(i[:, 1], 0, ly - 1), i[:, 2] % lz
        f = U[:, iz[:, :, None, None], iy[:, None, :, None], ix[:, None, None, :]]
        return np.einsum("dvzyx,vz,vy,vx->vd", f, w[:, 2], w[:, 1] * ok, w[:, 0])

    k1 = vel(pos)
    k2 = vel(pos + k1 / 2)
    k3 = vel(pos + k2 / 2)
    k4 = vel(pos + k3)
    return (k1 + 2 * k2 + 2 * k3 + k4) / 6


def _rough_field(shape, nc, prec, **kw):
    lx, ly, lz = shape
    cells, pos = _scattered(lx, ly, lz, nc, 2, seed=2)
    if nc > 2:  # crowd them into two tiles
        pos = [(p / v) * w + o for p, v, w, o in zip(pos, shape, (14.0, 6.0, 6.0), (1.0, 0.0, 1.0))]
    g = gpu_of(lx, ly, lz, prec, cells=cells, **kw)
    g.set_cells_state(x=pos[0], y=pos[1], z=pos[2])
    U = 1.5 * np.random.default_rng(9).standard_normal((3, lz, ly, lx))
    pad = np.zeros((3, lz + 4, ly + 4, lx + 4))
    pad[:, 2:-2, 2:-2, 2:-2] = U
    g.set_macros(*[a.reshape(-1) for a in pad])
    g.ibm_st2()
    s = g.cells_state()
    g.close()
    ref = _advected(np.stack(pos, 1), U, shape)
    # FP32: the stage positions carry the velocity's rounding (1e-7 of 1.5
    # nodes), which the next stage multiplies by the field's slope (about 3 per
    # node), three times: 1e-7 * 27, with a margin of 10
    tol = {"f64": 1e-11, "f32": 3e-5}[prec]
    for d, k in enumerate("uvw"):
        assert rel(s[k], ref[:, d]) < tol, k


@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("shape,nc", [((9, 8, 17), 2), ((40, 24, 40), 11)])  # boxes that wrap onto themselves; full tiles
def test_interpolation_of_a_fast_rough_field(shape, nc, prec, form, monkeypatch):
    """Vertices that leave their lattice cell, and the staged box, between the
    RK stages; tiles shared out between work groups (1782 vertices in two of
    them); rough velocities of order one node per step.  Against a plain FP64
    evaluation: stages beyond the reference's two halo layers, which the oracle
    has too, take the periodic images here."""
    monkeypatch.setenv("LBMIBM_INTERP_FORM", str(form))
    print(f"[interp rough] {shape} {prec} form={form}", flush=True)
    _rough_field(shape, nc, prec)


@pytest.mark.parametrize("k", [0, 1, 2, 6])
def test_spread_point_by_point(k, monkeypatch):
    """FP32 values under an indicator: boxes of 16 x 8 x 8 tiles."""
    monkeypatch.setenv("LBMIBM_SPREAD_FORM", "1")
    levels, lo, hi = CROWDS[k]
    lx, ly, lz = 45, 37, 40
    print(f"[spread points] {k}", flush=True)
    cells, pos = _crowded(lx, ly, lz, levels, 17 + k, lo, hi)
    rng = np.random.default_rng(4)
    n = pos[0].size
    forces = [1e-3 * rng.standard_normal(n) * 10.0 ** rng.uniform(-4, 0, n) for _ in range(3)]
    F, ref = _spread_both(lx, ly, lz, "f32", cells, pos, forces, vof_period=1000)
    for a, b in zip(F, ref):
        assert rel(a, b) < SPREAD_TOL["f32"]


@pytest.mark.parametrize("shape,nc", [((9, 8, 17), 2), ((40, 24, 40), 11)])
def test_interpolation_point_by_point(shape, nc):
    """The rough field, FP32 values under an indicator."""
    print(f"[interp points] {shape}", flush=True)
    _rough_field(shape, nc, "f32", vof_period=1000)


# several pieces of the ring in one plane, rows longer than a piece, helper
# threads (above 8 MB in all), the smallest lattice; a tube
FRAMES = [((4, 4, 4), {}), ((77, 46, 51), {}), ((77, 46, 51), {"periodic_y": True}), ((140001, 4, 4), {}),
          ((160, 128, 130), {"periodic_y": True}), ((33, 34, 40), {"tube_radius": 14.0, "e": (0.0, 0.0, 1.0)})]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("k", range(len(FRAMES)))
def test_downloads_fill_the_padded_frame(k, prec):
    """Velocities with their periodic images, wall nodes left as they were; the
    values are whole numbers, so equal to the last bit."""
    from preprocess_src_amd import native
    (lx, ly, lz), kw = FRAMES[k]
    print(f"[frame] {lx}x{ly}x{lz} {kw} {prec}", flush=True)
    g = gpu_of(lx, ly, lz, prec, store_macros=False, **kw)
    rng = np.random.default_rng(k)
    comp = rng.integers(1, 1 << 20, (3, lz, ly, lx)).astype(np.float64)
    pad = np.zeros((3, lz + 4, ly + 4, lx + 4))
    pad[:, 2:-2, 2:-2, 2:-2] = comp
    g.set_macros(*[np.ascontiguousarray(a).reshape(-1) for a in pad])
    want = np.full_like(pad, -7.0)
    if "tube_radius" in kw:
        want[:, :, 2:-2, 2:-2] = np.pad(comp, ((0, 0), (2, 2), (0, 0), (0, 0)), mode="wrap")
        x, y = np.arange(lx + 4) - 1.5 - lx / 2.0, np.arange(ly + 4) - 1.5 - ly / 2.0
        want[:, :, np.sqrt(x[None, :] ** 2 + y[:, None] ** 2) > kw["tube_radius"]] = -7.0
    else:
        wy = 2 if kw.get("periodic_y") else 0
        want[:, :, 2 - wy:ly + 2 + wy] = np.pad(comp, ((0, 0), (2, 2), (wy, wy), (2, 2)), mode="wrap")
    for order in ((0, 1, 2), (2,)):  # all, one alone
        got = [np.full(g.np_, -7.0) for _ in range(3)]
        native.check(g.L.lbmibm_download_macros(g.ctx, *([None] * 5),
                                                *[native.dp(got[d]) if d in order else None for d in range(3)]), g.ctx)
        for d in range(3):
            assert np.array_equal(got[d].reshape(want[d].shape), want[d] if d in order else np.full_like(want[d], -7.0))
    force = [np.full(g.np_, -7.0) for _ in range(3)]  # at rest: 0 on the fluid nodes alone
    native.check(g.L.lbmibm_download_lattice_force(g.ctx, *map(native.dp, force)), g.ctx)
    inner = np.full(want[0].shape, -7.0)
    inner[2:-2, 2:-2, 2:-2] = 0.0
    for f in force:
        assert np.array_equal(f.reshape(inner.shape), inner)
    g.close()


def test_download_of_the_indicator_zeroes_the_walls():
    from preprocess_src_amd import native
    lx, ly, lz = 29, 18, 23
    cells, _ = _scattered(lx, ly, lz, 1, 2, seed=1)
    g = gpu_of(lx, ly, lz, "f32", cells=cells, vof_period=1000)
    comp = np.random.default_rng(3).uniform(0, 1, (lz, ly, lx))
    pad = np.zeros((lz + 4, ly + 4, lx + 4))
    pad[2:-2, 2:-2, 2:-2] = comp
    native.check(g.L.lbmibm_upload_vf(g.ctx, native.dp(np.ascontiguousarray(pad))), g.ctx)
    got = np.full(g.np_, -7.0)
    native.check(g.L.lbmibm_download_vf(g.ctx, native.dp(got)), g.ctx)
    want = np.zeros_like(pad)
    want[:, 2:-2] = np.pad(comp, ((2, 2), (0, 0), (2, 2)), mode="wrap")
    g.close()
    assert np.array_equal(got.reshape(want.shape), want)


# more receptors in range than the search holds in LDS, and long lists; few
# receptors for many springs, which lose round after round; one candidate each
SPRINGS = [dict(receptor_density=64.0, max_neighwall=100), dict(receptor_density=1.0, springs_per_knob=12),
           dict(max_neighwall=1), dict(receptor_density=16.0, max_neighwall=100, springs_per_knob=40)]


@pytest.mark.parametrize("k", range(len(SPRINGS)))
def test_receptor_lists_and_attachment_rounds(k):
    """Lists and attachments are whole numbers: equal to the oracle's."""
    from tests.test_adhesion import LY, _pair
    print(f"[springs] {SPRINGS[k]}", flush=True)
    o, g, st, nrec = _pair("f64", extra=SPRINGS[k], tau=0.9, p=5e-6, b=5e-3)
    X, Y, Z = o.node_coords()
    vel = 4e-3 * (Y + LY / 2) / LY
    vel[o.bc == 2] = 0.0
    o.init_fluid(None, vel, None, None)
    g.set_equilibrium(None, vel, None, None)
    o.volume_init()
    g.volume_init()
    for it in range(5):
        gs = g.adhesion_state(nrec)
        for name in ("id_wall", "attach", "is_attached"):
            assert np.array_equal(gs[name], st[name]), (it, name)
        if it < 4:
            assert o.step(it + 1)[0] == 0
            g.step(it + 1)
    assert (st["attach"] >= 0).sum() > 5
    g.close()


# the halo's image of either colour on each axis, the smallest lattice, several
# work groups
SORS = [(20, 16, 18), (21, 16, 18), (20, 17, 19), (23, 16, 21), (4, 14, 4), (70, 30, 61)]


@pytest.mark.parametrize("k", range(len(SORS)))
def test_front_tracking_of_every_halo_parity(k):
    from preprocess_src_amd import mesh
    shape = SORS[k]
    print(f"[front parity] {shape}", flush=True)
    cells = mesh.assemble([2], np.array([[0.3, 0.2, -0.4]]), np.eye(3)[None], min(shape) / 4.5, shape="sphere")
    kw = dict(sor_itrmax=200000, sor_residual=1e-10)
    o = oracle_of(*shape, cells=cells, **kw)
    g = gpu_of(*shape, "f64", cells=cells, vof_period=4, **kw)
    rc, its, att = o.front_tracking()
    assert rc == 0
    gits, gatt = g.front_tracking()
    assert gatt == att and abs(gits - its) <= 1, (gits, its)
    keep = o.bc != 2
    # two solves of the same system, stopped at a residual of 1e-10
    assert rel(g.vf()[keep], o.vf[keep]) < 1e-8
    first = g.vf()
    g.front_tracking()
    assert np.array_equal(g.vf(), first)
    g.close()


def test_front_tracking_of_several_stretches_per_group():
    """More x pairs than 1024 work groups of 512 take in one stretch each."""
    from preprocess_src_amd import mesh
    shape = (300, 10, 300)
    print(f"[front stretches] {shape}", flush=True)
    cells = mesh.assemble([2], np.array([[0.3, 0.2, -0.4]]), np.eye(3)[None], 2.5, shape="sphere")
    kw = dict(sor_itrmax=200000, sor_residual=1e-2)
    o = oracle_of(*shape, cells=cells, **kw)
    g = gpu_of(*shape, "f64", cells=cells, vof_period=4, **kw)
    rc, its, att = o.front_tracking()
    assert rc == 0
    gits, gatt = g.front_tracking()
    assert gatt == att and gits == its, (gits, its)
    keep = o.bc != 2
    assert rel(g.vf()[keep], o.vf[keep]) < 1e-10  # the same iterate of the same sweeps
    g.close()


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("normal", [(1, 1, -1), (1, 2, 3), (0, 0, 1)])
def test_spread_of_a_flat_membrane_through_full_tiles(normal, prec, monkeypatch):
    """Vertices on a plane through one tile, which is shared out: the plane's
    cells are a few diagonals, rows or one layer of the tile."""
    monkeypatch.setenv("LBMIBM_SPREAD_FORM", "1")
    lx, ly, lz = 40, 32, 40
    print(f"[membrane] {normal} {prec}", flush=True)
    cells, pos = _crowded(lx, ly, lz, [4], 5, (9.0, 9.0, 9.0), (16.9, 16.9, 16.9))
    n = np.array(normal, float)
    mid = [13.0 - (m - 1) / 2.0 for m in (lx, ly, lz)]
    off = sum(a * (p - c) for a, p, c in zip(n, pos, mid)) / (n @ n)
    pos = [np.clip(p - a * off, c - 3.9, c + 3.9) for p, a, c in zip(pos, n, mid)]
    rng = np.random.default_rng(4)
    forces = [1e-3 * rng.standard_normal(pos[0].size) for _ in range(3)]
    F, ref = _spread_both(lx, ly, lz, prec, cells, pos, forces)
    for a, b in zip(F, ref):
        assert rel(a, b) < SPREAD_TOL[prec]

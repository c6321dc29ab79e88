"""Attachment rounds of so many springs that they run over the whole chip."""
import numpy as np
import pytest

from tests.test_adhesion import LY, _knobs, _cell, _pair

pytestmark = pytest.mark.gpu

# more springs than one work group takes without further launches (8192), more
# losers than it takes (1024): rounds beyond the eight launches, fewer of them than
# launches, one; springs that find few receptors
MANY = [dict(springs_per_knob=420, max_neighwall=100, receptor_density=16.0),
        dict(springs_per_knob=420, max_neighwall=5), dict(springs_per_knob=420, max_neighwall=1),
        dict(springs_per_knob=600, max_neighwall=9, receptor_density=1.0)]


@pytest.mark.parametrize("k", range(len(MANY)))
def test_rounds_of_many_springs(k):
    """Lists and attachments are whole numbers: equal to the oracle's."""
    print(f"[many springs] {MANY[k]}", flush=True)
    assert int(_knobs(_cell()).sum()) * MANY[k]["springs_per_knob"] > 8192
    o, g, st, nrec = _pair("f64", extra=MANY[k], tau=0.9, p=5e-6, b=5e-3)
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
    near = (st["id_wall"].reshape(-1, MANY[k]["max_neighwall"])[:, 0] >= 0).sum()
    assert near * MANY[k]["springs_per_knob"] > 2 * 1024
    assert (st["attach"] >= 0).sum() > 5
    g.close()


# several hundred to ten thousand receptors in range: the list is cut over and
# over, to one entry, to the longest that it can be cut to, and where it cannot
DENSE = [(64.0, 1), (64.0, 16), (64.0, 100), (64.0, 192), (64.0, 193), (100.0, 64), (900.0, 16), (900.0, 300)]


@pytest.mark.parametrize("density,maxn", DENSE)
def test_lists_of_dense_receptors(density, maxn):
    print(f"[dense] {density} {maxn}", flush=True)
    extra = dict(receptor_density=density, max_neighwall=maxn, springs_per_knob=1)
    o, g, st, nrec = _pair("f64", extra=extra, tau=0.9, p=5e-6, b=5e-3)
    gs = g.adhesion_state(nrec)
    g.close()
    assert np.array_equal(gs["id_wall"], st["id_wall"])
    assert np.allclose(gs["r_wall"], st["r_wall"], rtol=1e-14, atol=0)
    assert np.array_equal(gs["attach"], st["attach"])
    assert (st["id_wall"].reshape(-1, maxn)[:, -1] >= 0).any()  # full lists


# two springs on each of 5124 knobs: eight launches, and what is left in one group
CROWDED = [dict(receptor_density=4.0, max_neighwall=40), dict(receptor_density=1.0, max_neighwall=12, k_on0=3.0),
           dict(receptor_density=16.0, max_neighwall=100, k_on0=3.0, k_off0=2.0)]


@pytest.mark.parametrize("k", range(len(CROWDED)))
def test_rounds_of_crowded_knobs(k):
    from preprocess_src_amd import mesh
    from tests.pairs import gpu_of, oracle_of
    from tests.test_adhesion import ADH, LX, LZ
    print(f"[crowded knobs] {CROWDED[k]}", flush=True)
    y = -LY / 2 + 3.5
    cells = mesh.assemble([4, 4], np.array([[-6.0, y, -0.4], [6.2, y, 0.3]]), np.repeat(np.eye(3)[None], 2, 0), 3.0,
                          shape="sphere")
    kw = dict(tau=0.9, p=5e-6, b=5e-3)
    o = oracle_of(LX, LY, LZ, cells=cells, **kw)
    g = gpu_of(LX, LY, LZ, "f64", cells=cells, **kw)
    kn = np.ones(len(cells["x"]), np.uint8)
    adh = dict(ADH, springs_per_knob=2, **CROWDED[k])
    assert 8192 < 2 * kn.size <= 65536
    g.adhesion_setup(adh, kn)
    st = o.adhesion_setup(adh, kn)
    nrec = o._adhs.nxw * o._adhs.nzw
    o.volume_init()
    g.volume_init()
    assert (st["id_wall"].reshape(-1, adh["max_neighwall"])[:, 0] >= 0).sum() * 2 > 2048
    for it in range(7):
        gs = g.adhesion_state(nrec)
        for name in ("id_wall", "attach", "is_attached"):
            assert np.array_equal(gs[name], st[name]), (it, name)
        if it < 6:
            assert o.step(it + 1)[0] == 0
            g.step(it + 1)
    g.close()

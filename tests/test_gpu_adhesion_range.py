"""A search range beyond the box."""
import numpy as np
import pytest

from tests.pairs import gpu_of
from tests.test_adhesion import ADH, LX, LY, LZ, _cell, _knobs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("density,limit", [(1.0, 12), (1.0, 30), (4.0, 25), (4.0, 70)])
def test_rows_beyond_a_period_are_no_receptors(density, limit):
    """Rows of receptors up to LIMIT dx away, each taken as it is or one period
    further; with LIMIT dx longer than the box some would lie beyond both, at
    numbers that no receptor has."""
    print(f"[range] {density} {limit}", flush=True)
    maxn, ns = 40, 2
    cells = _cell()
    g = gpu_of(LX, LY, LZ, "f64", cells=cells)
    kn = _knobs(cells)
    g.adhesion_setup(dict(ADH, receptor_density=density, limit=limit, max_neighwall=maxn, springs_per_knob=ns), kn)
    d = np.sqrt(1.0 / density)
    nzw, nxw = int(LZ / d + 1e-3), int(LX / d + 1e-3)
    dzw, dxw = LZ / nzw, LX / nxw
    gs = g.adhesion_state(nzw * nxw)
    g.close()
    span = limit * int(1.0 / dzw)
    jx = np.arange(nxw)
    lists = gs["id_wall"].reshape(-1, maxn)
    beyond = 0
    for v in np.flatnonzero(kn):
        x, y, z = (cells[k][v] for k in "xyz")
        iz = int((z + LZ / 2.0) / dzw)
        ids, rs = [], []
        for i in range(2 * span):
            jz = iz + i - (span - 1)
            zj = (jz - nzw // 2) * dzw
            if jz < 0:
                jz, zj = jz + nzw, zj + LZ
            elif jz >= nzw:
                jz, zj = jz - nzw, zj - LZ
            if not 0 <= jz < nzw:
                beyond += 1
                continue
            r = np.sqrt(((jx - nxw // 2) * dxw - x) ** 2 + (-0.5 * LY - y) ** 2 + (zj - z) ** 2)
            ids.append(jz * nxw + jx)
            rs.append(r)
        ids, rs = np.concatenate(ids), np.concatenate(rs)
        near = rs <= limit
        order = np.argsort(rs[near], kind="stable")[:maxn]
        want = ids[near][order]
        # distances that agree to rounding may change places
        got = lists[v][:len(want)]
        assert (got >= 0).all() and (got < nzw * nxw).all() and (lists[v][len(want):] == -1).all()
        where = {}
        for a, b in zip(ids[near], rs[near]):
            where.setdefault(int(a), []).append(b)
        dist = np.sort([min(where[int(a)]) for a in got])
        assert np.allclose(gs["r_wall"].reshape(-1, maxn)[v][:len(want)], rs[near][order], rtol=1e-13, atol=0)
        assert dist[-1] <= rs[near][order][-1] * (1 + 1e-13)
    assert (beyond > 0) == (limit >= 30)  # the cell in the middle reaches a period and a half
    assert ((gs["attach"] >= -1) & (gs["attach"] < nzw * nxw)).all() and (gs["attach"] >= 0).any()

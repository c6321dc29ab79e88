"""Downloads whose host arrays share memory."""
import numpy as np
import pytest

from tests.pairs import gpu_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(12, 9, 10), (128, 120, 100), (2000, 16, 64)])
def test_the_last_field_remains_in_a_shared_place(shape):
    """One place for several fields keeps the last of them, also where the
    fields are large enough for helper threads (above 8 MB)."""
    from preprocess_src_amd import native
    lx, ly, lz = shape
    print(f"[shared place] {shape}", flush=True)
    g = gpu_of(lx, ly, lz, "f32", store_macros=False)
    rng = np.random.default_rng(1)
    pad = np.zeros((3, lz + 4, ly + 4, lx + 4))
    pad[:, 2:-2, 2:-2, 2:-2] = rng.integers(1, 1 << 20, (3, lz, ly, lx))
    g.set_macros(*[np.ascontiguousarray(a).reshape(-1) for a in pad])
    out = np.zeros(g.np_)
    for _ in range(5):
        for order in ((0, 0, 0), (0, 0, None), (None, 0, 0)):
            native.check(g.L.lbmibm_download_macros(g.ctx, *([None] * 5),
                                                    *[None if o is None else native.dp(out) for o in order]), g.ctx)
            last = 1 if order[2] is None else 2
            got = out.reshape(pad[0].shape)[2:-2, 2:-2, 2:-2]
            assert np.array_equal(got, pad[last, 2:-2, 2:-2, 2:-2])
            out[:] = 0.0
    g.close()

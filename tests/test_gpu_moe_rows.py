"""gv_model_moe's rows on their way in and out through the staging slots (1 MB each, eight in turn): counts whose rows
end inside, at and past a slot's end and past the whole ring give, row for row, what small calls of the same rows give,
bit for bit (a row's result does not depend on the others)."""
import numpy as np
import pytest

from model_helpers import SMALL, SMALL_ROUTER_SIGMA

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 17, 18, 1024, 1025, 9000])
def test_rows_in_slots(M):
    import geode_amd as g
    g.init(0)
    gm = g.VerifyModel(SMALL)
    gm.randomize(3, 0.02, float(SMALL_ROUTER_SIGMA), 0)
    rng = np.random.default_rng(M)
    h = rng.standard_normal((M, SMALL["hidden"]), np.float32)
    lg = rng.standard_normal((M, SMALL["n_experts"]), np.float32)
    out, ids, wts = gm.moe(0, h, lg)
    # (small calls of the same path: more rows than max_rows take the prefill's, fewer the verify step's)
    n = min(M, 40)
    for a in sorted({0, min(1000, M - n), M // 2 - n // 2, M - n} if M > 17 else {0}):
        o, i, w = gm.moe(0, h[a:a + n], lg[a:a + n])
        assert np.array_equal(o, out[a:a + n]) and np.array_equal(i, ids[a:a + n]) and np.array_equal(w, wts[a:a + n])
    # the routed weights against a float64 softmax over the picked experts: 32-bit exponentials and quotients
    p = np.exp(np.take_along_axis(lg.astype(np.float64), ids, 1))
    assert np.abs(wts - p / p.sum(1, keepdims=True)).max() <= 1e-6
    gm.close()

"""gv_model_moe's rows on their way in and out through the staging slots (1 MB each, eight in turn): counts whose rows
end inside, at and past a slot's end and past the whole ring give, row for row, what smaller calls of the same rows give,
bit for bit (a row's result does not depend on the others), and what the CPU oracle gives."""
import numpy as np
import pytest

import pyoracle as po
from model_helpers import SMALL, SMALL_ROUTER_SIGMA, adopt_oracle_model, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 17, 18, 1024, 1025, 9000])
def test_rows_in_slots(M):
    import geode_amd as g
    g.init(0)
    om = po.Model(SMALL, seed=3, router_sigma=SMALL_ROUTER_SIGMA, ctx=0)
    gm = g.VerifyModel(SMALL)
    adopt_oracle_model(gm, om, 0)
    rng = np.random.default_rng(M)
    h = rng.standard_normal((M, SMALL["hidden"]), np.float32)
    lg = rng.standard_normal((M, SMALL["n_experts"]), np.float32)
    out, ids, wts = gm.moe(0, h, lg)
    # (smaller calls of the same path: more rows than max_rows take the prefill's, fewer the verify step's)
    if M > 17:
        n = min(M, 40)
        windows = {(a, n) for a in (0, min(1000, M - n), M // 2 - n // 2, M - n)}
    else:
        windows = {(0, 1), (M - 1, 1), (M // 2, M - M // 2), (0, max(1, M - 1))}
    for a, n in sorted(windows):
        o, i, w = gm.moe(0, h[a:a + n], lg[a:a + n])
        assert np.array_equal(o, out[a:a + n]) and np.array_equal(i, ids[a:a + n]) and np.array_equal(w, wts[a:a + n])
        want, wids, wwts = po.moe_layer(om, 0, h[a:a + n], lg[a:a + n])
        # the bounds of the block's other tests (test_gpu_configs.py)
        assert np.array_equal(ids[a:a + n], wids) and np.abs(wts[a:a + n] - wwts).max() <= 1e-6
        assert rel_err(out[a:a + n], want) <= 1e-2
    # every row's picks and weights: the largest logits (ties, none here, to the lower index), a float64 softmax over them
    assert np.array_equal(ids, np.argsort(-lg, axis=1, kind="stable")[:, :SMALL["top_k"]])
    p = np.exp(np.take_along_axis(lg.astype(np.float64), ids, 1))
    assert np.abs(wts - p / p.sum(1, keepdims=True)).max() <= 1e-6   # 32-bit exponentials and quotients
    gm.close()

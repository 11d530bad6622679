"""The draft's pick over few logits (mtp.hip): fewer than its 64 chunks (empty ones), a chunk's edge, equal logits in
every chunk (their probability exactly 1 / n), the maximum in the first, a middle and the last place."""
import numpy as np
import pytest

import pyoracle as po
from model_helpers import adopt_oracle_model

pytestmark = pytest.mark.gpu

CTX = 20
CFG = dict(hidden=256, vocab=2000, n_layers=1, n_experts=16, top_k=4, moe_ff=128, shared_ff=128, n_heads=4,
           n_kv_heads=2, head_dim=64, rope_dim=16, rope_theta=1e7, eps=1e-6, max_ctx=64, max_rows=8, mtp=1)


@pytest.fixture(scope="module")
def model():
    import geode_amd as gv

    gv.init(0)
    om = po.Model(CFG, seed=5, router_sigma=1.0 / np.sqrt(CFG["hidden"]), ctx=CTX)
    gm = gv.VerifyModel(CFG)
    adopt_oracle_model(gm, om, CTX)
    yield gm
    gm.close()


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 1999])
def test_pick(model, n):
    rng = np.random.default_rng(3)
    toks = rng.integers(0, CFG["vocab"], 2).astype(np.int32)
    hid = rng.normal(0, 1, (2, CFG["hidden"])).astype(np.float32)
    try:
        model.set_draft_vocab(None)
        model.draft(toks, CTX, hid)
        full = model.draft_logits().astype(np.float64)
        hi, lo = int(full.argmax()), int(full.argmin())
        model.set_draft_vocab(np.full(n, hi, np.int32))
        d, p = model.draft(toks, CTX, hid)
        assert d == hi and p == np.float32(1.0 / n)   # n equal terms exp(0) = 1: an exact sum
        for at in {0, n // 2, n - 1}:
            ids = np.full(n, lo, np.int32)
            ids[at] = hi
            model.set_draft_vocab(ids)
            d, p = model.draft(toks, CTX, hid)
            want = 1.0 / (1.0 + (n - 1) * np.exp(np.float64(np.float32(full[lo]) - np.float32(full[hi]))))
            # the sum's own rounding ~n 2^-53 and the float32 result
            assert d == hi and abs(p - want) <= 2.0 ** -23 * want
    finally:
        model.set_draft_vocab(None)

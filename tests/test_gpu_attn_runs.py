"""The attention over long contexts and where a KV head's queries make several groups: contexts at block edges, a ragged
last block, chains and trees, against the CPU oracle on the exact path (fp32 activations) and, for the int8 cache, on the
int8 path; a row's result for itself, whatever rows go with it; the softmax weights of large scores that 32 bits hold
exactly."""
import numpy as np
import pytest

import pyoracle as po
from model_helpers import SMALL, SMALL_ROUTER_SIGMA, adopt_oracle_model, rel_err, route_margins, tree_parents

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gv():
    import geode_amd
    geode_amd.init(0)
    return geode_amd


# (n_heads, head_dim): 8 query heads a KV head make 3 groups at 17 rows, 2 make one
@pytest.mark.parametrize("heads,hd,M,tree,ctx", [
    (16, 64, 17, True, 5437), (16, 64, 17, True, 5424), (16, 64, 17, False, 11000), (16, 256, 17, True, 6000),
    (16, 96, 9, False, 9001), (4, 64, 1, False, 16384), (4, 64, 5, False, 16379), (4, 64, 5, False, 16500),
    (16, 64, 17, True, 130)])
@pytest.mark.parametrize("kv8", [False, True])
def test_attention_runs(gv, heads, hd, M, tree, ctx, kv8):
    cfg = dict(SMALL, n_heads=heads, head_dim=hd, n_layers=1, max_ctx=ctx + 40, kv_int8=int(kv8), exact=int(not kv8))
    om = po.Model({k: v for k, v in cfg.items() if k != "exact"}, seed=5, router_sigma=SMALL_ROUTER_SIGMA, ctx=ctx)
    gm = gv.VerifyModel(cfg)
    adopt_oracle_model(gm, om, ctx)
    toks = ((np.arange(M) * 37 + 11) % cfg["vocab"]).astype(np.int32)
    parents = tree_parents() if tree else None
    want, ids, trace = om.verify_trace(toks, parents, mode=0 if kv8 else 1)
    got = gm.verify(toks, parents)
    # exact path: 32-bit sums in another order (test_gpu_exact.py's bound); int8 path: the codes' own sensitivity. Only a
    # row whose K-th and (K+1)-th router logits are nearer than that may take another expert
    tol = 1e-2 if kv8 else 1e-4
    swapped = (np.sort(gm.route_ids(M), axis=2) != np.sort(ids, axis=2)).any(axis=(0, 2))
    assert np.all(route_margins(om, trace).min(axis=0)[swapped] < tol)
    assert swapped.sum() <= 1
    if not swapped.all():
        assert rel_err(got[~swapped], want[~swapped]) <= tol
    gm.close()


# 16 query heads a KV head: 4 rows make one group, 5 rows two, a workgroup each over the short context and one after the
# other over the long one
@pytest.mark.parametrize("ctx", [1003, 8300])
@pytest.mark.parametrize("kv8", [False, True])
def test_row_for_itself(gv, kv8, ctx):
    cfg = dict(SMALL, n_heads=32, head_dim=32, n_layers=1, max_ctx=ctx + 40, kv_int8=int(kv8))
    gm = gv.VerifyModel(cfg)
    gm.randomize(7, 0.05, float(SMALL_ROUTER_SIGMA), 0 if kv8 else ctx)
    rng = np.random.default_rng(3)
    if kv8:
        rows = rng.integers(-127, 128, 2 * ctx * 64, np.int8)
        gm.adopt(gv.KV_I8, np.concatenate([rows.view(np.uint8), np.full(2 * ctx * 2, 0.02, np.float32).view(np.uint8)]))
        gm.position = ctx
    x = rng.standard_normal((8, cfg["hidden"]), np.float32)
    mid, out, ids = gm.layer(0, x)
    for n in (1, 4, 5):
        m, o, i = gm.layer(0, x[:n])
        assert np.array_equal(m, mid[:n]) and np.array_equal(o, out[:n]) and np.array_equal(i, ids[:n])
    gm.close()


def test_weights_of_large_scores(gv):
    """Keys whose scores are near 2,000 and exact in 32 bits (whole numbers times powers of two all the way), a few units
    apart: each weight is one exponential of an exact difference, so its error is the
    exponential's own and does not grow with the scores. One value a position, one-hot in dim position mod 64."""
    ctx, hd, H, nkv = 200, 64, SMALL["hidden"], 2
    cfg = dict(SMALL, n_layers=1, exact=1, eps=1e-30, max_ctx=ctx + 40)
    gm = gv.VerifyModel(cfg)
    gm.randomize(7, 0.02, float(SMALL_ROUTER_SIGMA), ctx)
    rng = np.random.default_rng(11)
    nh, cols = cfg["n_heads"], cfg["n_heads"] * hd
    gm.adopt(gv.IN_NORM, np.zeros(H, np.float32))
    gm.adopt(gv.Q_NORM, np.zeros(hd, np.float32))
    gm.adopt(gv.K_NORM, np.zeros(hd, np.float32))
    # a pack row: codes (0: level 1), then a block's scale in E4M3 (0x38: 1). The rows' input is 1 in every dim, so a
    # query row with one block is 16 x the global: dims 40..43 of a head 8, over the root mean square 2 (past the 16
    # rotated dims); gates, keys and values of the new rows 0
    qkv = np.zeros((nh * 2 * hd + 2 * nkv * hd, H // 2 + H // 16), np.uint8)
    for h in range(nh):
        qkv[h * 2 * hd + 40:h * 2 * hd + 44, H // 2] = 0x38
    gm.adopt(gv.QKV, qkv, globals_=[0.5, 0.5, 0.5])
    level = rng.integers(0, 8, (H, cols))
    sign = rng.integers(0, 2, (H, cols))
    code = (level | (sign << 3)).astype(np.uint8)
    o = np.concatenate([code[:, 0::2] | (code[:, 1::2] << 4), np.full((H, cols // 16), 0x38, np.uint8)], 1)
    gm.adopt(gv.O, np.ascontiguousarray(o), globals_=[0.25])
    W = 0.25 * (2.0 * level + 1) * (1 - 2 * sign)
    # score = (4 dims of 4) . key / 8, the keys' dims whole numbers
    k4 = rng.integers(996, 1001, (ctx, nkv, 4))
    score = k4.sum(-1) * 4 / 8
    kv = np.zeros((2, ctx, nkv, hd))
    kv[0, :, :, 40:44] = k4
    kv[1, np.arange(ctx), :, np.arange(ctx) % hd] = 1.0
    gm.adopt(gv.KV, kv.astype(np.float16).view(np.uint16).reshape(2, ctx, nkv * hd))
    gm.position = ctx
    x = np.ones((3, H), np.float32)
    mid, _, _ = gm.layer(0, x)
    w = np.exp(score - score.max(0))
    w /= w.sum(0)
    att = np.zeros((nh, hd))
    for h in range(nh):
        np.add.at(att[h], np.arange(ctx) % hd, w[:, h // (nh // nkv)])
    att = 0.5 * att.reshape(-1)   # (the sigmoid of a gate of 0)
    want, mag = 1.0 + W @ att, np.abs(W) @ att
    # two exponentials of 1 ulp (2^-23 each), weights and operands as two halves (2^-22 each), the normalization and the
    # 32-bit sums of a few terms a dim and of cols products: 16 units of 2^-23 of the products' magnitude; the residual's
    # own rounding
    assert np.all(np.abs(mid - want) <= 16 * 2.0 ** -23 * mag + 2.0 ** -24 * np.abs(want)), (np.abs(mid - want) / mag).max()
    gm.close()

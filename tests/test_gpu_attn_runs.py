"""The attention where a workgroup takes a run of several blocks of positions (a long context, or many query tiles) and
where a KV head's queries make several groups: contexts at the edge between one block a workgroup and runs of two, a
ragged last run, chains and trees, against the CPU oracle on the exact path (fp32 activations) and, for the int8
cache, on the int8 path."""
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


# (n_heads, head_dim): 8 query heads a KV head make 3 groups at 17 rows (runs from 5,441 positions on), 2 make one (from
# 16,385 on)
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

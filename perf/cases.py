"""The work that is measured on an MI355X: the calls a program makes around one speculative-decoding step, from a
one-row dense MLP to the whole 40-layer verify step, each through the package's public entry points.

`listed()` are the measured cases, `draw(rng)` makes one more of the same ranges, `prepare` / `run` are what a
program holds before a call and the call, `work` the bytes and operations no implementation can do without,
`tolerance` how far two correct implementations may be apart, `exact` the same result in 64 bits by plain torch.

The shapes are those of the benchmark and the tests: hidden 2048, 256 experts (8 a row) plus a shared one of width
512, gated attention of 16 query and 2 key/value heads of 256, Gated DeltaNet of 16 key and 32 value heads of 128
behind a conv of 4, vocabularies of 151,936 and 248,320.
"""
import collections
import ctypes

import numpy as np
import torch

import geode_amd as g

H, EXPERTS, TOP_K, MOE_FF = 2048, 256, 8, 512
HEADS, KV_HEADS, HEAD_DIM, ROPE_DIM, THETA, EPS = 16, 2, 256, 64, 1e7, 1e-6
GDN = dict(gdn_k_heads=16, gdn_v_heads=32, gdn_k_dim=128, gdn_v_dim=128, conv_kernel=4)
LAYER_VOCAB = 4096      # a single layer's cases end in a small head: the layer is what they are about
VOCAB = 151936
STEP_CTX = 8192         # the whole model's context at most
STEP_LAYERS = 40
DRAFT_HEAD = 32768      # a draft vocabulary's rows
DEV = "cuda"


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest call: one row (plain decoding, no draft stands) through one dense MLP; launches and latency
        dict(name="ffn_row", kind="ffn", rows=1, ff=6144, layers=1),
        # the dense MLPs of a 12-layer model at a step of 4 drafts: every layer's weights from memory
        dict(name="ffn_stack", kind="ffn", rows=5, ff=6144, layers=12),
        # the final norm and the vocabulary head over a draft tree's 17 rows
        dict(name="head_tree", kind="head", rows=17, vocab=VOCAB),
        # one attention + MoE layer decoding a single row in a short chat (a ragged context)
        dict(name="layer_decode", kind="layer", mixer="attention", rows=1, ctx=1003, int8=False, branch=""),
        # the same layer verifying a draft tree of 16 nodes in a long document, the int8 cache
        dict(name="layer_tree_long", kind="layer", mixer="attention", rows=17, ctx=32001, int8=True, branch="4,3"),
        # a Gated DeltaNet + MoE layer verifying 4 drafts, then keeping the rows that stand
        dict(name="gdn_chain", kind="layer", mixer="gdn", rows=5, ctx=1003, int8=True, branch=""),
        # a prompt's chunk through one MoE block (host rows in and out, as the engine calls it)
        dict(name="moe_prefill", kind="moe", rows=512),
        # textbook acceptance of 4 drafts by their full distributions
        dict(name="accept_textbook", kind="textbook", drafts=4, vocab=VOCAB, temperature=0.7, top_p=0.95, greedy=False),
        # sample-and-match of a step at a chat's usual sampler, the large vocabulary
        dict(name="accept_match", kind="match", rows=5, vocab=248320, temperature=0.7, top_p=0.95, top_k=20),
        # one MTP draft from a step's 5 rows over a draft vocabulary, its logits read back
        dict(name="draft", kind="draft", rows=5, ctx=2001, int8=True),
        # the whole verify step, 4 chained drafts: the headline
        dict(name="step_chain", kind="step", rows=5, ctx=8192, branch=""),
        # the whole verify step over the draft tree
        dict(name="step_tree", kind="step", rows=17, ctx=8192, branch="4,3"),
    ]


def _log_int(rng, lo, hi):
    """an integer of [lo, hi], spread over its logarithm"""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["ffn", "head", "layer", "layer", "layer", "moe", "textbook", "match", "draft", "step"])
    branch = lambda: rng.choice(["", "", "4,3", "2,2,2", "3,1,1,1"])   # noqa: E731  chains and trees of drafts
    if kind == "ffn":
        return dict(kind=kind, rows=_log_int(rng, 1, 32), ff=256 * _log_int(rng, 4, 32), layers=rng.randint(1, 12))
    if kind == "head":
        return dict(kind=kind, rows=_log_int(rng, 1, 32), vocab=_log_int(rng, 4096, 248320))
    if kind == "layer":
        gdn = rng.random() < 0.4
        return dict(kind=kind, mixer="gdn" if gdn else "attention", rows=_log_int(rng, 1, 24),
                    ctx=_log_int(rng, 64, 4096 if gdn else 32768), int8=rng.random() < 0.5, branch=branch())
    if kind == "moe":
        return dict(kind=kind, rows=_log_int(rng, 2, 2048))
    if kind == "textbook":
        return dict(kind=kind, drafts=rng.randint(1, 8), vocab=_log_int(rng, 32000, 248320),
                    temperature=round(rng.uniform(0.5, 1.2), 3), top_p=round(rng.uniform(0.8, 0.99), 3),
                    greedy=rng.random() < 0.3)
    if kind == "match":
        return dict(kind=kind, rows=rng.randint(1, 9), vocab=_log_int(rng, 32000, 248320),
                    temperature=0.0 if rng.random() < 0.3 else round(rng.uniform(0.5, 1.2), 3),
                    top_p=round(rng.uniform(0.8, 0.99), 3), top_k=rng.choice([0, 20, 50, 200]))
    if kind == "draft":
        return dict(kind=kind, rows=_log_int(rng, 1, 17), ctx=_log_int(rng, 64, 8192), int8=rng.random() < 0.5)
    return dict(kind=kind, rows=_log_int(rng, 1, 17), ctx=_log_int(rng, 128, STEP_CTX), branch=branch())


# ------------------------------------------------------------------ q4 matrices (the pack's rows)
def _gen(seed, *salt):
    x = seed & 0xFFFFFFFF
    for s in salt:
        x = (x * 6364136223846793005 + 1442695040888963407 + s) & 0x7FFFFFFFFFFFFFFF
    return torch.Generator(device=DEV).manual_seed(x)


def _q4_pack(w, sigma):
    """float [rows, cols] of spread 1 to the pack's rows (a code nibble a value, an E4M3 scale a 16-value block) and
    the matrix's global: level x E4M3 x global is the value times sigma, to a 4-bit step"""
    rows, cols = w.shape
    b = w.view(rows, cols // 16, 16)
    scale = (b.abs().amax(-1) * (256.0 / 15.0)).to(torch.float8_e4m3fn)
    s = scale.float().clamp_min(2.0 ** -9).unsqueeze(-1) / 256.0
    code = ((b.abs() / s - 1.0) * 0.5).round_().clamp_(0, 7).to(torch.uint8) | ((b < 0).to(torch.uint8) << 3)
    code = code.view(rows, cols // 2, 2)
    return torch.cat([code[..., 0] | (code[..., 1] << 4), scale.view(torch.uint8)], 1).contiguous(), sigma / 256.0


def _q4_random(gen, rows, cols, sigma):
    return _q4_pack(torch.randn(rows, cols, device=DEV, generator=gen), sigma)


def _q4_values(pack, cols, glob):
    """the matrix in 64 bits from its pack rows"""
    rows = pack.shape[0]
    by = pack[:, :cols // 2]
    code = torch.stack([by & 15, by >> 4], -1).view(rows, cols).to(torch.int64)
    level = ((code & 7) * 2 + 1) * (1 - 2 * (code >> 3))
    scale = pack[:, cols // 2:].contiguous().view(torch.float8_e4m3fn).double()
    return level.double() * scale.repeat_interleave(16, 1) * float(np.float32(glob))


def _q4_device(pack, cols, glob):
    """the matrix in the library's layout: (its device bytes, its descriptor)"""
    rows = pack.shape[0]
    buf = torch.empty(g.lib.gv_q4_device_bytes(rows, cols), dtype=torch.uint8, device=DEV)
    desc = g.GvQ4()
    torch.cuda.synchronize()   # (the library works on a stream of its own)
    g.check(g.lib.gv_q4_from_pack(pack.data_ptr(), rows, cols, glob, buf.data_ptr(), ctypes.byref(desc)), "gv_q4_from_pack")
    g.check(g.lib.gv_synchronize(), "gv_synchronize")
    return buf, desc


def _codes(x):
    """a float32 row's values as the int8 path takes them, q x (amax / 127) of each 16-value block, in 64 bits"""
    b = x.float().reshape(*x.shape[:-1], -1, 16)
    amax = b.abs().amax(-1, keepdim=True)
    inv = torch.where(amax > 0, 127.0 / amax, torch.zeros_like(amax))
    return (torch.round(b * inv).clamp(-127, 127).double() * (amax / 127.0).double()).reshape(x.shape)


# ------------------------------------------------------------------ a decoder layer's tensors
def _host(t):
    return t.cpu().numpy()


def _cfg(case):
    c = dict(hidden=H, vocab=LAYER_VOCAB, n_layers=1, n_experts=EXPERTS, top_k=TOP_K, moe_ff=MOE_FF, shared_ff=MOE_FF,
             n_heads=HEADS, n_kv_heads=KV_HEADS, head_dim=HEAD_DIM, rope_dim=ROPE_DIM, rope_theta=THETA, eps=EPS,
             max_ctx=case["ctx"] + 96, max_rows=max(17, case["rows"]), kv_int8=int(case.get("int8", False)))
    if case.get("mixer") == "gdn":
        c.update(GDN, gdn_layers=[1])
    if case["kind"] == "draft":
        c.update(mtp=1, vocab=VOCAB)
    return c


def _experts(gen, layer_tensors):
    """every expert's gate_up and down rows (the shared one last), as the pack's expert blocks [E + 1, bytes]"""
    gu, dn = [], []
    for e0 in range(0, EXPERTS + 1, 64):
        n = min(64, EXPERTS + 1 - e0)
        p, layer_tensors["gu_global"] = _q4_random(gen, n * 2 * MOE_FF, H, 0.02)
        gu.append(p.view(n, 2 * MOE_FF, -1))
        p, layer_tensors["dn_global"] = _q4_random(gen, n * H, MOE_FF, 0.02)
        dn.append(p.view(n, H, -1))
    layer_tensors["gu"], layer_tensors["dn"] = torch.cat(gu), torch.cat(dn)


def _layer_tensors(case, seed, salt):
    """one layer's tensors on the GPU, from the seed: weights of spread 0.02, norms near 1, a router of unit logits"""
    gen = _gen(seed, salt)
    f = lambda n, s: torch.randn(n, device=DEV, generator=gen) * s   # noqa: E731
    L = dict(in_norm=f(H, 0.02), post_norm=f(H, 0.02),
             router=f((EXPERTS, H), H ** -0.5).bfloat16(), shared_gate=f(H, 0.02).bfloat16())
    _experts(gen, L)
    if case.get("mixer") == "gdn":
        nk, nv, dk, dv, K = (GDN[k] for k in ("gdn_k_heads", "gdn_v_heads", "gdn_k_dim", "gdn_v_dim", "conv_kernel"))
        conv = 2 * nk * dk + nv * dv
        L["qkv"], L["z"], L["out"] = (_q4_random(gen, r, c, 0.02) for r, c in ((conv, H), (nv * dv, H), (H, nv * dv)))
        L["a"], L["b"] = f((nv, H), H ** -0.5).bfloat16(), f((nv, H), H ** -0.5).bfloat16()
        L["a_log"], L["dt_bias"], L["gnorm"] = f(nv, 0.5), f(nv, 0.5), 1.0 + f(dv, 0.02)
        L["conv"], L["conv_state"], L["S"] = f((conv, K), 0.3), f((conv, K - 1), 1.0), f((nv, dk, dv), 0.05)
        return L
    L["q_norm"], L["k_norm"] = f(HEAD_DIM, 0.02), f(HEAD_DIM, 0.02)
    L["q"], L["k"], L["v"] = (_q4_random(gen, r, H, 0.02) for r in (HEADS * 2 * HEAD_DIM, KV_HEADS * HEAD_DIM,
                                                                 KV_HEADS * HEAD_DIM))
    L["o"] = _q4_random(gen, H, HEADS * HEAD_DIM, 0.02)
    kv = f((2, case["ctx"], KV_HEADS, HEAD_DIM), 1.0)
    if case.get("int8"):   # int8 rows of a (position, head), a float scale each
        sc = kv.abs().amax(-1) / 127.0
        L["kv"], L["kv_scale"] = torch.round(kv / sc.unsqueeze(-1)).clamp(-127, 127).to(torch.int8), sc
    else:
        L["kv"] = kv.half()
    return L


def _adopt_layer(m, L, layer):
    """the layer's tensors into the model, as an engine hands over its pack"""
    for kind, name in ((g.IN_NORM, "in_norm"), (g.POST_NORM, "post_norm")):
        m.adopt(kind, _host(L[name]), layer=layer)
    for kind, name in ((g.ROUTER, "router"), (g.SHARED_GATE, "shared_gate")):
        m.adopt(kind, _host(L[name].view(torch.int16)), layer=layer)
    blocks = _host(torch.cat([L["gu"].flatten(1), L["dn"].flatten(1)], 1))
    gu, dn = L["gu_global"], L["dn_global"]
    for e in range(EXPERTS):
        m.adopt(g.EXPERT, blocks[e], layer=layer, expert=e, globals_=[gu, dn])
    m.adopt(g.SHARED_EXPERT, blocks[EXPERTS], layer=layer, globals_=[gu, gu, dn])
    if "z" in L:
        for kind, name in ((g.GDN_QKV, "qkv"), (g.GDN_Z, "z"), (g.GDN_OUT, "out")):
            m.adopt(kind, _host(L[name][0]), layer=layer, globals_=[L[name][1]])
        for kind, name in ((g.GDN_A, "a"), (g.GDN_B, "b")):
            m.adopt(kind, _host(L[name].view(torch.int16)), layer=layer)
        for kind, name in ((g.GDN_ALOG, "a_log"), (g.GDN_DTB, "dt_bias"), (g.GDN_NORM, "gnorm"), (g.GDN_CONV, "conv"),
                           (g.GDN_CONV_ST, "conv_state"), (g.GDN_S, "S")):
            m.adopt(kind, _host(L[name]), layer=layer)
        return
    m.adopt(g.Q_NORM, _host(L["q_norm"]), layer=layer)
    m.adopt(g.K_NORM, _host(L["k_norm"]), layer=layer)
    m.adopt(g.QKV, _host(torch.cat([L["q"][0], L["k"][0], L["v"][0]])), layer=layer,
            globals_=[L[n][1] for n in "qkv"])
    m.adopt(g.O, _host(L["o"][0]), layer=layer, globals_=[L["o"][1]])
    if "kv_scale" in L:
        m.adopt(g.KV_I8, np.concatenate([_host(L["kv"]).reshape(-1).view(np.uint8),
                                         _host(L["kv_scale"]).reshape(-1).view(np.uint8)]), layer=layer)
    else:
        m.adopt(g.KV, _host(L["kv"]).view(np.uint16), layer=layer)


def _ends(case, seed, vocab):
    """embedding, head and final norm. The embedding's rows have unit spread: a row that reaches a layer of a trained
    model carries the sum of the layers before, to which one layer adds a small part."""
    return dict(embed=_q4_random(_gen(seed, 1), vocab, H, 1.0), head=_q4_random(_gen(seed, 2), vocab, H, 0.02),
                final_norm=torch.randn(H, device=DEV, generator=_gen(seed, 3)) * 0.02)


def _mtp_tensors(seed):
    gen = _gen(seed, 8)
    n = lambda: torch.randn(H, device=DEV, generator=gen) * 0.02   # noqa: E731
    return dict(fc=_q4_random(gen, H, 2 * H, 0.02), norm=n(), pre_e=n(), pre_h=n(),
                ids=torch.arange(DRAFT_HEAD, device=DEV) * (VOCAB // DRAFT_HEAD))


def _tokens(seed, n, vocab):
    return np.random.default_rng(seed).integers(0, vocab, n).astype(np.int32)


def _hidden(seed, n):
    return np.random.default_rng(seed + 77).standard_normal((n, H)).astype(np.float32)


def _parents(case):
    """the rows' parents: a chain ("") or a tree in breadth-first order, so many children of a node at each depth,
    cut to the case's rows (the last node's first children go on as a chain where the tree is smaller)"""
    if not case["branch"] or case["rows"] == 1:
        return None
    parents, frontier = [-1], [0]
    for b in (int(x) for x in case["branch"].split(",")):
        nxt = []
        for p in frontier:
            for _ in range(b):
                parents.append(p)
                nxt.append(len(parents) - 1)
        frontier = nxt
    while len(parents) < case["rows"]:
        parents.append(len(parents) - 1)
    return np.array(parents[:case["rows"]], np.int32)


class _Logits:
    """the model's logits on the device as an array (it keeps the model)"""

    def __init__(self, model, rows, vocab):
        self.model = model
        self.__cuda_array_interface__ = {"shape": (rows, vocab), "typestr": "<f4", "version": 3,
                                         "data": (int(g.lib.gv_model_logits(model.h)), False)}


_WHOLE = collections.OrderedDict()   # the whole model, as a program loads it once for all its conversations


def _whole_model():
    if "model" not in _WHOLE:
        m = g.VerifyModel(dict(_cfg(dict(kind="step", ctx=STEP_CTX, rows=17)), vocab=VOCAB, n_layers=STEP_LAYERS))
        m.randomize(20261201, 0.02, H ** -0.5, STEP_CTX)
        # the residual stream of a trained model's rows: each layer adds a few percent to it (_ends)
        pack, glob = _q4_random(_gen(20261201, 1), VOCAB, H, 4.0)
        m.adopt(g.EMBED, _host(pack), globals_=[glob])
        _WHOLE["model"] = m
    return _WHOLE["model"]


# ------------------------------------------------------------------ what a program holds before the call
def prepare(case, seed):
    g.init(0)
    s = dict(case=case)
    kind = case["kind"]
    if kind == "ffn":
        s["x"], s["packs"] = _ffn_inputs(case, seed)
        s["mats"] = [[_q4_device(p, c, gl) for p, c, gl in layer] for layer in s.pop("packs")]
        s["y"] = torch.empty(case["layers"], case["rows"], H, device=DEV)
        s["ws"] = torch.empty(g.lib.gv_ffn_workspace_bytes(H, case["ff"], case["rows"]), dtype=torch.uint8, device=DEV)
        s["calls"] = [[ctypes.byref(desc) for _, desc in layer] + [case["rows"], s["x"][l].data_ptr(),
                                                                  s["y"][l].data_ptr(), s["ws"].data_ptr()]
                      for l, layer in enumerate(s["mats"])]
    elif kind == "head":
        s["x"], s["norm"], (pack, glob) = _head_inputs(case, seed)
        s["w"] = _q4_device(pack, H, glob)
        s["act"] = torch.empty(case["rows"] * g.act_bytes(H), dtype=torch.uint8, device=DEV)
        s["y"] = torch.empty(case["rows"], case["vocab"], device=DEV)
    elif kind == "layer":
        m = s["model"] = g.VerifyModel(_cfg(case))
        ends = _ends(case, seed, LAYER_VOCAB)
        m.adopt(g.EMBED, _host(ends["embed"][0]), globals_=[ends["embed"][1]])
        m.adopt(g.LM_HEAD, _host(ends["head"][0]), globals_=[ends["head"][1]])
        m.adopt(g.FINAL_NORM, _host(ends["final_norm"]))
        _adopt_layer(m, _layer_tensors(case, seed, 4), 0)
        s["tokens"], s["parents"] = _tokens(seed, case["rows"], LAYER_VOCAB), _parents(case)
        s["logits"] = torch.as_tensor(_Logits(m, case["rows"], LAYER_VOCAB), device=DEV)
    elif kind == "moe":
        m = s["model"] = g.VerifyModel(_cfg(dict(case, ctx=64, rows=17)))
        _adopt_layer(m, _layer_tensors(dict(case, ctx=64), seed, 4), 0)
        s["h"], s["router_logits"] = _moe_inputs(case, seed)
    elif kind == "textbook":
        gen, k, V = _gen(seed, 5), case["drafts"], case["vocab"]
        s["target"] = torch.randn(k + 1, V, device=DEV, generator=gen) * 3.0
        s["draft"] = s["target"][:k] + torch.randn(k, V, device=DEV, generator=gen) * 0.5
        r = np.random.default_rng(seed)
        s["u_draft"], s["u_acc"], s["u_res"] = r.random(k, np.float32), r.random(k, np.float32), float(r.random())
    elif kind == "match":
        n, V = case["rows"], case["vocab"]
        s["logits"] = torch.randn(n, V, device=DEV, generator=_gen(seed, 6)) * 3.0
        best = _host(s["logits"].argmax(1)).astype(np.int32)
        s["batch"] = np.concatenate([[7], best[:-1]]).astype(np.int32)   # (the drafts: each row's likeliest token)
        s["u"] = np.random.default_rng(seed).random(n)
    elif kind == "draft":
        m = s["model"] = g.VerifyModel(_cfg(case))
        ends, mtp = _ends(case, seed, VOCAB), _mtp_tensors(seed)
        m.adopt(g.EMBED, _host(ends["embed"][0]), globals_=[ends["embed"][1]])
        m.adopt(g.LM_HEAD, _host(ends["head"][0]), globals_=[ends["head"][1]])
        m.adopt(g.MTP_FC, _host(mtp["fc"][0]), globals_=[mtp["fc"][1]])
        for kd, name in ((g.MTP_NORM, "norm"), (g.MTP_PRE_E, "pre_e"), (g.MTP_PRE_H, "pre_h")):
            m.adopt(kd, _host(mtp[name]))
        _adopt_layer(m, _layer_tensors(case, seed, 4), 1)   # (the decoder layer of the MTP layer)
        m.set_draft_vocab(_host(mtp["ids"]))
        s["tokens"], s["hidden"] = _tokens(seed, case["rows"], VOCAB), _hidden(seed, case["rows"])
    else:
        m = s["model"] = _whole_model()
        s["tokens"], s["parents"] = _tokens(seed, case["rows"], VOCAB), _parents(case)
        s["logits"] = torch.as_tensor(_Logits(m, case["rows"], VOCAB), device=DEV)
    return s


def _ffn_inputs(case, seed):
    gen, F = _gen(seed, 10), case["ff"]
    x = torch.randn(case["layers"], case["rows"], H, device=DEV, generator=gen).half()
    shapes = ((F, H), (F, H), (H, F))   # gate, up, down
    return x, [[(p, c, gl) for r, c in shapes for p, gl in [_q4_random(gen, r, c, 0.02)]] for _ in range(case["layers"])]


def _head_inputs(case, seed):
    gen = _gen(seed, 11)
    x = torch.randn(case["rows"], H, device=DEV, generator=gen) * 2.0
    return x, torch.randn(H, device=DEV, generator=gen) * 0.02, _q4_random(gen, case["vocab"], H, 0.02)


def _moe_inputs(case, seed):
    r = np.random.default_rng(seed)
    return (r.standard_normal((case["rows"], H), np.float32),
            r.standard_normal((case["rows"], EXPERTS), np.float32))


# ------------------------------------------------------------------ one pass
def _p(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "ffn":
        for args in s["calls"]:
            g.check(g.lib.gv_ffn_swiglu(*args), "gv_ffn_swiglu")
        return s["y"]
    if kind == "head":
        M, V = case["rows"], case["vocab"]
        g.check(g.lib.gv_quantize(s["x"].data_ptr(), H, M, H, s["norm"].data_ptr(), EPS, s["act"].data_ptr(), None),
                "gv_quantize")
        g.check(g.lib.gv_gemv_q4(ctypes.byref(s["w"][1]), s["act"].data_ptr(), M, s["y"].data_ptr(), V, 0), "gv_gemv_q4")
        return s["y"]
    if kind in ("layer", "step"):
        m = s["model"]
        m.position = case["ctx"]
        m.verify(s["tokens"], s["parents"], want_logits=False)
        if case.get("mixer") == "gdn" and s["parents"] is None:
            m.keep((case["rows"] + 1) // 2)   # (some of the drafts stand)
        return s["logits"]
    if kind == "moe":
        out, _, weights = s["model"].moe(0, s["h"], s["router_logits"])
        return out, weights
    if kind == "textbook":
        V, out = case["vocab"], np.full(case["drafts"] + 1, -1, np.int32)
        n = g.lib.gv_accept_textbook(s["target"].data_ptr(), s["draft"].data_ptr(), V, V, case["drafts"],
                                     case["temperature"], case["top_p"], int(case["greedy"]), _p(s["u_draft"]),
                                     _p(s["u_acc"]), s["u_res"], _p(out))
        g.check(-1 if n < 0 else 0, "gv_accept_textbook")
        return out, n
    if kind == "match":
        V, kept, out = case["vocab"], ctypes.c_int(0), np.full(case["rows"], -1, np.int32)
        n = g.lib.gv_accept_match(s["logits"].data_ptr(), V, V, _p(s["batch"]), case["rows"], case["temperature"],
                                  case["top_p"], case["top_k"], 1024, _p(s["u"]), _p(out), ctypes.byref(kept))
        g.check(-1 if n < 0 else 0, "gv_accept_match")
        return out, n, kept.value
    m = s["model"]
    _, prob = m.draft(s["tokens"], case["ctx"], hidden=s["hidden"])
    return m.draft_logits(), prob


# ------------------------------------------------------------------ what no implementation can do without
def _q4_bytes(rows, cols):
    return rows * cols // 16 * 9


def _touched(rows):
    """distinct experts that so many rows of 8 picks are expected to touch, and the shared one"""
    return EXPERTS * (1.0 - (1.0 - TOP_K / EXPERTS) ** rows) + 1.0


def _moe_work(rows):
    b = _touched(rows) * (_q4_bytes(2 * MOE_FF, H) + _q4_bytes(H, MOE_FF))
    return b, 2.0 * 3 * H * MOE_FF * rows * (TOP_K + 1)


def _layer_work(case):
    """a layer: its projections, mixer state or cache, router and touched experts, each read once"""
    M, ctx = case["rows"], case["ctx"]
    b, fl = _moe_work(M)
    b += (EXPERTS + 1) * H * 2
    fl += 2.0 * M * EXPERTS * H
    if case.get("mixer") == "gdn":
        nk, nv, dk, dv = (GDN[k] for k in ("gdn_k_heads", "gdn_v_heads", "gdn_k_dim", "gdn_v_dim"))
        rows = 2 * nk * dk + 2 * nv * dv
        b += _q4_bytes(rows, H) + _q4_bytes(H, nv * dv) + 2 * nv * H * 2 + nv * dk * dv * 4 * (1 + M)
        return b, fl + 2.0 * M * (rows * H + H * nv * dv + 3 * nv * dk * dv)
    rows = HEADS * 2 * HEAD_DIM + 2 * KV_HEADS * HEAD_DIM
    b += _q4_bytes(rows, H) + _q4_bytes(H, HEADS * HEAD_DIM)
    b += 2 * KV_HEADS * (ctx + M) * (HEAD_DIM + 4 if case.get("int8") else 2 * HEAD_DIM)
    return b, fl + 2.0 * M * (rows * H + H * HEADS * HEAD_DIM + 2 * HEADS * HEAD_DIM * ctx)


def work(case):
    kind = case["kind"]
    if kind == "ffn":
        M, F, n = case["rows"], case["ff"], case["layers"]
        b = n * (2 * _q4_bytes(F, H) + _q4_bytes(H, F) + M * H * 6)
        return {"bytes": b, "flops": n * 2.0 * 3 * H * F * M}
    if kind == "head":
        M, V = case["rows"], case["vocab"]
        return {"bytes": _q4_bytes(V, H) + M * (H + V) * 4, "flops": 2.0 * M * V * H}
    if kind == "moe":
        b, fl = _moe_work(case["rows"])
        return {"bytes": b + case["rows"] * (2 * H + EXPERTS) * 4, "flops": fl}
    if kind == "textbook":
        return {"bytes": (2 * case["drafts"] + 1) * case["vocab"] * 4, "flops": 0}
    if kind == "match":
        return {"bytes": case["rows"] * case["vocab"] * 4, "flops": 0}
    b, fl = _layer_work(case)
    M = case["rows"]
    if kind == "draft":
        return {"bytes": b + _q4_bytes(H, 2 * H) + _q4_bytes(DRAFT_HEAD, H) + DRAFT_HEAD * 4,
                "flops": fl + 2.0 * (M * 2 * H * H + DRAFT_HEAD * H)}
    layers, V = (STEP_LAYERS, VOCAB) if kind == "step" else (1, LAYER_VOCAB)
    return {"bytes": layers * b + _q4_bytes(V, H) + M * V * 4, "flops": layers * fl + 2.0 * M * V * H}


# ------------------------------------------------------------------ how far two correct implementations may be apart
def tolerance(case):
    kind = case["kind"]
    if kind in ("textbook", "match"):
        return "exact"   # tokens: the uniforms decide, and lie nowhere near a boundary of 64-bit sums
    if kind == "head":
        return {"rel": 1e-5, "max": 1e-4}   # one product of given int8 codes: 32-bit sums in another order
    # Beyond one product, the int8 path rounds values that it has computed to codes (1/127 of the block's largest): a
    # last-bit difference before moves some codes by a step. Measured on the paths with every matrix's scale one ulp up
    # or the sums in another order (relative, largest): dense MLP 1e-4, 1.7e-3 (a single moved code of one row: 2.5e-4);
    # MoE block 1.8e-5, 1e-3; a layer 1.1e-3, 8.4e-3; 40 layers 6e-3, 5.7e-2 (0.4% of the routed experts change).
    if kind in ("ffn", "moe"):
        return {"rel": 1e-3, "max": 2e-2}
    if kind == "step":
        return {"rel": 2.5e-2, "max": 0.25}
    return {"rel": 5e-3, "max": 5e-2}


# ------------------------------------------------------------------ the same in 64 bits
# The products take the activations as they are: the int8 rounding of values computed on the way (1/254 of a block's
# largest, about 0.5 percent of a product) is the path's own distance from this. Where the rows to be rounded are
# given (the head), their codes are given too and the result is that of the same codes.
def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * (1.0 + w.double())


def _mm(q, x, cols):
    return x @ _q4_values(q[0], cols, q[1]).T


def _silu(x):
    return x * torch.sigmoid(x)


def _moe64(L, h, logits=None):
    lg, hx = (h @ L["router"].double().T, h) if logits is None else (logits, _codes(h))   # (given rows: their codes)
    p = torch.softmax(lg, -1)
    w, ids = torch.sort(p, dim=-1, descending=True, stable=True)
    w, ids = w[:, :TOP_K], ids[:, :TOP_K]
    w = w / w.sum(-1, keepdim=True)

    def expert(e, x):
        gu = x @ _q4_values(L["gu"][e], H, L["gu_global"]).T
        return (_silu(gu[:, :MOE_FF]) * gu[:, MOE_FF:]) @ _q4_values(L["dn"][e], MOE_FF, L["dn_global"]).T

    out = torch.sigmoid(h @ L["shared_gate"].double()).unsqueeze(1) * expert(EXPERTS, hx)
    for e in torch.unique(ids).tolist():
        r, k = torch.nonzero(ids == e, as_tuple=True)
        out[r] += w[r, k].unsqueeze(1) * expert(e, hx[r])
    return out, w


def _tree(case):
    """each row's depth and which new rows it sees"""
    n, par = case["rows"], _parents(case)
    depth, vis = np.zeros(n, np.int64), np.zeros((n, n), bool)
    for i in range(n):
        p = i - 1 if par is None else int(par[i])
        if p >= 0:
            depth[i] = depth[p] + 1
            vis[i] = vis[p]
        vis[i, i] = True
    return depth, vis


def _attention64(case, L, h):
    n, ctx, half = case["rows"], case["ctx"], ROPE_DIM // 2
    depth, vis = _tree(case)
    q = _mm(L["q"], h, H).view(n, HEADS, 2, HEAD_DIM)
    k, v = (_mm(L[x], h, H).view(n, KV_HEADS, HEAD_DIM) for x in "kv")
    # the rotary angles: float(position) x inv_freq in 32 bits, as the table is defined
    inv = (np.float32(1) / np.power(np.float32(THETA), np.arange(0, ROPE_DIM, 2, dtype=np.float32) / np.float32(ROPE_DIM)))
    ang = torch.from_numpy(((ctx + depth).astype(np.float32)[:, None] * inv.astype(np.float32)).astype(np.float64)).to(DEV)
    cs, sn = torch.cos(ang).unsqueeze(1), torch.sin(ang).unsqueeze(1)

    def rope(x):
        a, b = x[..., :half], x[..., half:2 * half]
        return torch.cat([a * cs - b * sn, b * cs + a * sn, x[..., 2 * half:]], -1)

    gate, q = q[:, :, 1], rope(_rms(q[:, :, 0], L["q_norm"]))
    k = rope(_rms(k, L["k_norm"]))
    kv = L["kv"].double()
    if "kv_scale" in L:
        kv = kv * L["kv_scale"].double().unsqueeze(-1)
    keys, vals = torch.cat([kv[0], k]), torch.cat([kv[1], v])
    seen = torch.from_numpy(np.concatenate([np.ones((n, ctx), bool), vis], 1)).to(DEV)
    group, core = HEADS // KV_HEADS, torch.empty(n, HEADS, HEAD_DIM, device=DEV, dtype=torch.float64)
    for kh in range(KV_HEADS):
        for t in range(n):
            s = q[t, kh * group:(kh + 1) * group] @ keys[:, kh].T / HEAD_DIM ** 0.5
            core[t, kh * group:(kh + 1) * group] = torch.softmax(s.masked_fill(~seen[t], -torch.inf), -1) @ vals[:, kh]
    return _mm(L["o"], (core * torch.sigmoid(gate)).reshape(n, -1), HEADS * HEAD_DIM)


def _gdn64(case, L, h):
    nk, nv, dk, dv, K = (GDN[k] for k in ("gdn_k_heads", "gdn_v_heads", "gdn_k_dim", "gdn_v_dim", "conv_kernel"))
    n, kd, par = case["rows"], nk * dk, _parents(case)
    proj, z = _mm(L["qkv"], h, H), _mm(L["z"], h, H)
    a, b = h @ L["a"].double().T, h @ L["b"].double().T
    decay = torch.exp(-torch.exp(L["a_log"].double()) * torch.nn.functional.softplus(a + L["dt_bias"].double()))
    beta = torch.sigmoid(b)
    convs, states, core = [], [], []
    for t in range(n):
        p = t - 1 if par is None else int(par[t])
        win = torch.cat([convs[p] if p >= 0 else L["conv_state"].double(), proj[t].unsqueeze(1)], 1)
        convs.append(win[:, 1:])
        x = _silu((win * L["conv"].double()).sum(1))
        q, k, v = x[:kd].view(nk, dk), x[kd:2 * kd].view(nk, dk), x[2 * kd:].view(nv, dv)
        unit = lambda y: y / torch.sqrt((y * y).sum(1, keepdim=True) + 1e-6)   # noqa: E731
        q, k = (unit(y).repeat_interleave(nv // nk, 0) for y in (q, k))
        S = (states[p] if p >= 0 else L["S"].double()) * decay[t].view(nv, 1, 1)
        delta = (v - (S * k.unsqueeze(2)).sum(1)) * beta[t].unsqueeze(1)
        S = S + k.unsqueeze(2) * delta.unsqueeze(1)
        states.append(S)
        o = (S * q.unsqueeze(2)).sum(1) / dk ** 0.5
        o = o / torch.sqrt((o * o).mean(1, keepdim=True) + EPS) * L["gnorm"].double()
        core.append((o * _silu(z[t].view(nv, dv))).reshape(-1))
    return _mm(L["out"], torch.stack(core), nv * dv)


def _layer64(case, L, x):
    mix = _gdn64 if case.get("mixer") == "gdn" else _attention64
    x = x + mix(case, L, _rms(x, L["in_norm"]))
    return x + _moe64(L, _rms(x, L["post_norm"]))[0]


def exact(case, seed):
    kind = case["kind"]
    if kind == "ffn":
        x, layers = _ffn_inputs(case, seed)
        out = []
        for l, (gate, up, down) in enumerate(layers):
            w = [_q4_values(*q) for q in (gate, up, down)]
            h = _codes(x[l])
            out.append((_silu(h @ w[0].T) * (h @ w[1].T)) @ w[2].T)
        return torch.stack(out)
    if kind == "head":
        x, norm, (pack, glob) = _head_inputs(case, seed)
        # the normalized rows in 32 bits, so that their codes are the given ones
        inv = 1.0 / torch.sqrt((x.double() ** 2).mean(1, keepdim=True).float() + EPS)
        return torch.cat([_codes(x * inv * (1.0 + norm)) @ _q4_values(p, H, glob).T for p in pack.split(32768)], 1)
    if kind == "layer":
        ends = _ends(case, seed, LAYER_VOCAB)
        tok = torch.from_numpy(_tokens(seed, case["rows"], LAYER_VOCAB)).long().to(DEV)
        x = _layer64(case, _layer_tensors(case, seed, 4), _q4_values(ends["embed"][0][tok], H, ends["embed"][1]))
        return _mm(ends["head"], _rms(x, ends["final_norm"]), H)
    if kind == "moe":
        h, lg = (torch.from_numpy(a).double().to(DEV) for a in _moe_inputs(case, seed))
        out, w = _moe64(_layer_tensors(dict(case, ctx=64), seed, 4), h, lg)
        return out, w
    if kind == "draft":
        ends, mtp, L = _ends(case, seed, VOCAB), _mtp_tensors(seed), _layer_tensors(case, seed, 4)
        tok = torch.from_numpy(_tokens(seed, case["rows"], VOCAB)).long().to(DEV)
        e = _rms(_q4_values(ends["embed"][0][tok], H, ends["embed"][1]), mtp["pre_e"])
        hid = _rms(torch.from_numpy(_hidden(seed, case["rows"])).double().to(DEV), mtp["pre_h"])
        x = _layer64(dict(case, branch=""), L, _mm(mtp["fc"], torch.cat([e, hid], 1), 2 * H))
        head = (ends["head"][0][mtp["ids"]], ends["head"][1])
        lg = _mm(head, _rms(x[-1:], mtp["norm"]), H)[0]
        return lg, float(torch.softmax(lg, 0).max())
    return None   # (tokens; and the whole model, whose 20 GB of weights are made on the device)

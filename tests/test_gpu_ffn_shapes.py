"""The dense MLP and the skinny product where their launches change form: rows at the edges of the 8-, 16- and 32-row
forms, K ranges of one launch and of several (12 waves at K 4608..6144 and at most 256 row tiles, row groups at 17..32
rows over few tiles, both K ranges of 4096 in one launch over more), ragged last row tiles, against the CPU oracle's int8
path."""
import numpy as np
import pytest

import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gv():
    import geode_amd
    geode_amd.init(0)
    return geode_amd


@pytest.mark.parametrize("H,F,M", [(2048, 6144, 1), (2048, 6144, 16), (2048, 6144, 32), (2048, 4608, 8),
                                   (2048, 1152, 17), (128, 256, 9), (4096, 512, 5), (4096, 512, 20), (640, 5376, 8)])
def test_ffn_shapes(gv, H, F, M):
    gq, gg = po.q4_random(1001, F, H)
    uq, ug = po.q4_random(1002, F, H)
    dq, dg = po.q4_random(1003, H, F)
    x16 = po.f32_to_f16_bits(po.normal(2001, M * H).reshape(M, H))
    G, U, D = gv.Q4Matrix(gq, F, H, gg), gv.Q4Matrix(uq, F, H, ug), gv.Q4Matrix(dq, H, F, dg)
    dx = gv.DeviceBuffer.from_array(x16)
    y = gv.DeviceBuffer(M * H * 4)
    ws = gv.DeviceBuffer(gv.lib.gv_ffn_workspace_bytes(H, F, M))
    gv.check(gv.lib.gv_ffn_swiglu(G.ref(), U.ref(), D.ref(), M, dx.ptr, y.ptr, ws.ptr), "ffn")
    got = y.download(np.float32, (M, H))
    want = po.ffn_swiglu(gq, uq, dq, gg, ug, dg, H, F, x16, mode=0)
    # each row on its own: fp32 sums in another order (1e-5 of the row, as a single product), and where they move a
    # SwiGLU value over a rounding boundary of its code, a step of 1/127 of a block's largest value out of F values:
    # at most a few codes a row, each at most 3 / 127 / sqrt(F) of the row
    rms = np.sqrt(np.mean(want.astype(np.float64) ** 2, axis=1))
    err = np.sqrt(np.mean((got.astype(np.float64) - want) ** 2, axis=1))
    assert np.all(err <= (1e-5 + 3 * 3 / 127 / np.sqrt(F)) * rms), (err / rms).max()
    exact = po.ffn_swiglu(gq, uq, dq, gg, ug, dg, H, F, x16, mode=1)
    # the gpu_check.cpp:80-94 criterion against the exact path
    assert np.abs(got - exact).max() <= 1.5 * np.abs(want - exact).max() + 1e-6 * np.abs(exact).max()


@pytest.mark.parametrize("H,F,M,taken", [(2048, 8448, 8, True), (2048, 8448, 9, False), (2048, 8192, 9, True)])
def test_ffn_width_limit(gv, H, F, M, taken):
    """ff beyond 8192: up to 8 rows; more rows are refused before anything is launched (the workspace and the output as
    they were)."""
    gq, gg = po.q4_random(1001, F, H)
    dq, dg = po.q4_random(1003, H, F)
    x16 = po.f32_to_f16_bits(po.normal(2001, M * H).reshape(M, H))
    G, D = gv.Q4Matrix(gq, F, H, gg), gv.Q4Matrix(dq, H, F, dg)
    dx = gv.DeviceBuffer.from_array(x16)
    n = gv.lib.gv_ffn_workspace_bytes(H, F, M) // 4
    y, ws = (gv.DeviceBuffer.from_array(np.full(k, 7.0, np.float32)) for k in (M * H, n))
    rc = gv.lib.gv_ffn_swiglu(G.ref(), G.ref(), D.ref(), M, dx.ptr, y.ptr, ws.ptr)
    gv.check(gv.lib.gv_synchronize(), "synchronize")
    got = y.download(np.float32, (M, H))
    if taken:
        want = po.ffn_swiglu(gq, gq, dq, gg, gg, dg, H, F, x16, mode=0)
        # (test_ffn_shapes' bound, a row's)
        assert rc == 0 and np.abs(got - want).max() <= 1e-2 * np.abs(want).max()
    else:
        assert rc != 0 and b"at most 8192" in gv.lib.gv_last_error()
        assert np.all(got == 7.0) and np.all(ws.download(np.float32, (n,)) == 7.0)


@pytest.mark.parametrize("rows,cols,M", [(2048, 6144, 1), (600, 6144, 8), (16, 4608, 3), (600, 6144, 17),
                                         (600, 2048, 17), (2048, 1152, 32), (4096, 4096, 31), (40, 128, 20),
                                         (2100, 2048, 17), (4112, 4608, 8), (4112, 4096, 17), (8192, 4096, 32)])
@pytest.mark.parametrize("accumulate", [False, True])
def test_gemv_few_tiles(gv, rows, cols, M, accumulate):
    wq, s2 = po.q4_random(31 + rows + cols, rows, cols)
    m = gv.Q4Matrix(wq, rows, cols, s2)
    x = po.normal(41 + M, M * cols, 1.0).reshape(M, cols)
    base = po.normal(79, M * rows).reshape(M, rows) if accumulate else None
    got = gv.gemv(m, x, accumulate_into=base)
    want = np.stack([po.matvec_q(wq, cols, s2, x[t]) for t in range(M)])
    if accumulate:
        want = want + base
    # the integer block sums are exact; only the fp32 sums over blocks are in another order
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()

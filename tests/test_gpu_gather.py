"""GPU: convolutions over channels-last copies (vh_gather.hip) at the edges of
their tiles, stages and stride phases, against the oracle under the parity gate."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from tests.parity import k_conv_dgrad, k_conv_fwd, k_conv_wgrad
from tests.test_gpu_parity import DEV, DTYPES, check, host, prep, rng
from volta_amd import lib, nn as vnn

pytestmark = pytest.mark.gpu

# (B, C, O, H, W, K, S, P): shapes outside the specialised kernels (odd widths, strides)
CASES = [
    (1, 3, 5, 3, 1, 3, 1, 1),        # one column, channels below one 16-byte unit
    (2, 33, 31, 7, 7, 3, 1, 1),      # 31 and 33 rows: one 32-row tile / one row of a second
    (1, 64, 65, 9, 15, 3, 1, 1),     # 65 rows, 135 positions: one past the tile both ways
    (3, 130, 129, 9, 9, 3, 2, 1),    # 129 and 130 channels, phases of 4, 2, 2 and 1 taps
    (2, 8, 200, 5, 5, 1, 2, 0),      # K = 8: less than one stage; phases without taps
    (2, 20, 12, 6, 7, 5, 3, 2),      # nine phases
    (2, 7, 9, 10, 3, 2, 4, 0),       # stride 4 past the width, taps missing in most phases
    (2, 12, 20, 11, 13, 3, 1, 3),    # padding wider than the kernel reaches
    (64, 9, 80, 33, 31, 3, 1, 1),    # 128-row tiles, channels 9 -> 16 padded
    (80, 24, 64, 33, 31, 3, 1, 1),   # 64-row tiles of many positions
    (16, 16, 16, 45, 45, 3, 1, 1),   # weight gradient split many ways
    (2, 72, 136, 5, 7, 3, 1, 1),     # weight gradient split a few ways, channels past 64
]


def _ids(c):
    return "B{}C{}O{}H{}W{}K{}S{}P{}".format(*c)


@pytest.mark.parametrize("case", CASES, ids=_ids)
@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_gather_conv_all_passes(case, dt):
    B, C, O, H, W, K, S, P = case
    g = rng(sum(case) + 11)
    x, xt = prep(g.standard_normal((B, C, H, W)), dt)
    w, wt = prep(g.standard_normal((O, C, K, K)) * np.sqrt(2.0 / (C * K * K)), dt)
    b, bt = prep(g.uniform(-1, 1, (O,)), dt)
    conv = vnn.Conv2d(C, O, K, S, P, device=DEV, dtype=DTYPES[dt])
    conv.weight, conv.bias = wt, bt
    conv.set_algo(vnn.ConvAlgo.IGEMM)
    kw = dict(stride=(S, S), pad=(P, P))
    y = conv.forward(xt)
    bb = b[None, :, None, None]
    check(y, oracle.direct_conv, (x, w), dt, "y", kw, extra_ref=bb, extra_scale=np.abs(bb), k=k_conv_fwd(C, K, K))
    assert np.array_equal(host(conv.forward(xt, relu=True)), np.maximum(host(y), 0))
    dy, dyt = prep(g.standard_normal(tuple(y.shape)), dt)
    kwg = k_conv_wgrad(B, y.shape[2], y.shape[3])
    dx, dw, db = conv.backward(dyt, xt)  # one call: the copy of dy is shared
    check(dx, oracle.direct_conv_backward_input, (dy, w, x.shape), dt, "dx", kw, k=k_conv_dgrad(O, K, K))
    check(dw, oracle.direct_conv_backward_weight, (dy, x, w.shape), dt, "dw", kw, k=kwg)
    check(db, oracle.conv_bias_grad, (dy,), dt, "db", k=kwg)
    # each gradient alone, and the input gradient under a ReLU mask
    assert np.array_equal(host(conv.backward(dyt, xt, weight_grad=False)[0]), host(dx))
    _, dw1, db1 = conv.backward(dyt, xt, input_grad=False)
    assert np.array_equal(host(dw1), host(dw)) and np.array_equal(host(db1), host(db))
    masked = host(conv.backward(dyt, xt, weight_grad=False, relu_input=True)[0])
    assert np.array_equal(masked, np.where(x > 0, host(dx), 0))


@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_gather_padding_does_not_leak(dt):
    """An infinity reaches the outputs whose window or channel holds it and no
    other: the channel, position and stage padding is never multiplied with it."""
    B, C, O, H, W = 2, 5, 7, 9, 11
    conv = vnn.Conv2d(C, O, 3, 1, 1, device=DEV, dtype=DTYPES[dt])
    conv.set_algo(vnn.ConvAlgo.IGEMM)
    x = torch.ones((B, C, H, W), device=DEV, dtype=DTYPES[dt])
    dy = torch.ones((B, O, H, W), device=DEV, dtype=DTYPES[dt])
    x[1, 4, 8, 10] = float("inf")
    y = np.isfinite(host(conv.forward(x)))
    assert y[0].all() and y[1, :, :7].all() and y[1, :, :, :9].all() and not y[1, :, 7:, 9:].any()
    dw = np.isfinite(host(conv.backward(dy, x)[1]))
    # the corner (8, 10) is under tap rows and columns 1 and 2 only
    assert dw[:, :4].all() and dw[:, 4, 0].all() and dw[:, 4, :, 0].all() and not dw[:, 4, 1:, 1:].any()
    x[1, 4, 8, 10] = 1
    dy[1, 6, 8, 10] = float("inf")
    dx, dw, db = (np.isfinite(host(t)) for t in conv.backward(dy, x))
    assert dx[0].all() and dx[1, :, :7].all() and not dx[1, :, 7:, 9:].any()
    assert dw[:6].all() and db[:6].all() and not db[6]


@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_gather_conv_transpose(dt):
    B, CI, CO, H, W, K, S, P = 3, 24, 20, 7, 5, 4, 2, 1
    g = rng(5)
    x, xt = prep(g.standard_normal((B, CI, H, W)), dt)
    w, wt = prep(g.normal(0, 0.1, (CI, CO, K, K)), dt)
    b, bt = prep(g.uniform(-1, 1, (CO,)), dt)
    ct = vnn.ConvTranspose2d(CI, CO, K, S, P, device=DEV, dtype=DTYPES[dt])
    ct.weight, ct.bias = wt, bt
    y = ct.forward(xt)
    kw = dict(stride=(S, S), pad=(P, P))
    check(y, oracle.conv_transpose_forward, (x, w, b), dt, "y", kw, k=CI * K * K + 1)
    dy, dyt = prep(g.standard_normal(tuple(y.shape)), dt)
    got = ct.backward(dyt, xt)
    ks = (CO * K * K, B * H * W, B * y.shape[2] * y.shape[3])
    for i, (what, t) in enumerate(zip(("dx", "dw", "db"), got)):
        check(t, lambda *a, i=i, **k: oracle.conv_transpose_backward(*a, **k)[i], (dy, x, w), dt, what, kw, k=ks[i])
    assert np.array_equal(host(ct.backward(dyt, xt, weight_grad=False)[0]), host(got[0]))


def _workspace(stream):
    n = ctypes.c_size_t()
    assert lib().vh_workspace_info(ctypes.c_void_p(stream.cuda_stream), None, ctypes.byref(n), None) == 0
    return n.value


def test_gather_falls_back_without_workspace():
    """A capture on a stream whose workspace holds what the generic path needs
    but not the copies is still accepted, and right; the workspace does not move."""
    conv = vnn.Conv2d(16, 16, 3, 1, 1, use_bias=False, device=DEV)
    conv.set_algo(vnn.ConvAlgo.IGEMM)
    small, big = torch.randn(1, 16, 31, 31, device=DEV), torch.randn(64, 16, 31, 31, device=DEV)
    want = conv.forward(big)
    out = torch.empty_like(want)
    cap = torch.cuda.Stream()  # (its handle may be one that earlier work has grown a workspace on)
    torch.cuda.synchronize()
    assert lib().vh_release_cache() == 0
    cap.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(cap):
        conv.forward(small)
    torch.cuda.synchronize()
    have = _workspace(cap)
    assert 0 < have < big.shape[0] * 33 * 33 * 16 * 4, "the copy of the input fits: nothing falls back"
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=cap):
        conv.forward(big, out=out)
    assert _workspace(cap) == have
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert float((out - want).abs().max()) <= 2 * 144 * 2.0 ** -24 * float(want.abs().max()) * 16


@pytest.mark.parametrize("B", [3, 33, 60, 64, 65])
def test_narrow_fp32_layer_on_either_kernel(B):
    """32 -> 64 channels at 28 x 28: all passes on the channels-last path (3), on the
    halo kernels (60, 64), the weight and the input gradient on them (33), none (65)."""
    g = rng(B)
    conv = vnn.Conv2d(32, 64, 3, 1, 1, device=DEV)
    conv.set_algo(vnn.ConvAlgo.IGEMM)
    x, xt = prep(g.standard_normal((B, 32, 28, 28)), "f32")
    dy, dyt = prep(g.standard_normal((B, 64, 28, 28)), "f32")
    w, kw = host(conv.weight), dict(stride=(1, 1), pad=(1, 1))
    check(conv.forward(xt), oracle.direct_conv, (x, w), "f32", "y", kw, k=288)
    dx, dw, db = conv.backward(dyt, xt)
    check(dx, oracle.direct_conv_backward_input, (dy, w, x.shape), "f32", "dx", kw, k=576)
    check(dw, oracle.direct_conv_backward_weight, (dy, x, w.shape), "f32", "dw", kw, k=B * 784)
    check(db, oracle.conv_bias_grad, (dy,), "f32", "db", k=B * 784)


@pytest.mark.parametrize("C", [60, 120, 190, 250, 300, 550])  # 1x1: 1, 2, 3, 4, 5 and 9 stages
@pytest.mark.parametrize("B,O", [(2, 40), (96, 130)])  # 32 x 64 tiles, K over two wave groups
def test_gather_bf16_stages_in_flight(C, B, O):
    g = rng(C + B)
    x, xt = prep(g.standard_normal((B, C, 13, 11)), "bf16")
    w, wt = prep(g.standard_normal((O, C, 1, 1)) * np.sqrt(2.0 / C), "bf16")
    conv = vnn.Conv2d(C, O, 1, 2, 0, device=DEV, dtype=DTYPES["bf16"])
    conv.weight = wt
    conv.bias.zero_()
    check(conv.forward(xt), oracle.direct_conv, (x, w), "bf16", "y", dict(stride=(2, 2), pad=(0, 0)), k=C)


# copies of all images above the workspace's bound: chunks of images, the last smaller
@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_gather_gradients_in_chunks(dt):
    B, C, O, H, W, K, S = (41, 96, 24, 131, 130, 1, 1) if dt == "f32" else (67, 72, 24, 171, 165, 2, 2)
    g = rng(B)
    x, xt = prep(g.standard_normal((B, C, H, W)), dt)
    w, wt = prep(g.standard_normal((O, C, K, K)) * np.sqrt(2.0 / (C * K * K)), dt)
    conv = vnn.Conv2d(C, O, K, S, 0, device=DEV, dtype=DTYPES[dt])
    conv.weight = wt
    conv.set_algo(vnn.ConvAlgo.IGEMM)
    kw = dict(stride=(S, S), pad=(0, 0))
    HO, WO = (H - K) // S + 1, (W - K) // S + 1
    dy, dyt = prep(g.standard_normal((B, O, HO, WO)), dt)
    dx, dw, db = conv.backward(dyt, xt)
    check(dx, oracle.direct_conv_backward_input, (dy, w, x.shape), dt, "dx", kw, k=k_conv_dgrad(O, K, K))
    check(dw, oracle.direct_conv_backward_weight, (dy, x, w.shape), dt, "dw", kw, k=k_conv_wgrad(B, HO, WO))
    check(db, oracle.conv_bias_grad, (dy,), dt, "db", k=B * HO * WO)
    masked = host(conv.backward(dyt, xt, weight_grad=False, relu_input=True)[0])
    assert np.array_equal(masked, np.where(x > 0, host(dx), 0))


def test_gather_forward_in_chunks():
    B, C, O, H, W = 37, 32, 8, 270, 247
    g = rng(B)
    x, xt = prep(g.standard_normal((B, C, H, W)), "f32")
    w, wt = prep(g.standard_normal((O, C, 1, 1)), "f32")
    b, bt = prep(g.uniform(-1, 1, (O,)), "f32")
    conv = vnn.Conv2d(C, O, 1, 1, 0, device=DEV)
    conv.weight, conv.bias = wt, bt
    conv.set_algo(vnn.ConvAlgo.IGEMM)
    bb = b[None, :, None, None]
    check(conv.forward(xt), oracle.direct_conv, (x, w), "f32", "y", extra_ref=bb, extra_scale=np.abs(bb), k=C + 1)


def test_narrow_fp32_layer_with_passes_on_both_paths():
    """64 -> 32 channels at 20 x 20, 128 images: the weight gradient on the halo kernel,
    the input gradient and the forward pass over channels-last copies."""
    g = rng(20)
    conv = vnn.Conv2d(64, 32, 3, 1, 1, device=DEV)
    conv.set_algo(vnn.ConvAlgo.IGEMM)
    x, xt = prep(g.standard_normal((128, 64, 20, 20)), "f32")
    dy, dyt = prep(g.standard_normal((128, 32, 20, 20)), "f32")
    w, kw = host(conv.weight), dict(stride=(1, 1), pad=(1, 1))
    check(conv.forward(xt), oracle.direct_conv, (x, w), "f32", "y", kw, k=576)
    dx, dw, db = conv.backward(dyt, xt)
    check(dx, oracle.direct_conv_backward_input, (dy, w, x.shape), "f32", "dx", kw, k=288)
    check(dw, oracle.direct_conv_backward_weight, (dy, x, w.shape), "f32", "dw", kw, k=128 * 400)
    check(db, oracle.conv_bias_grad, (dy,), "f32", "db", k=128 * 400)


# fp32: forward / input gradient with K too long for their positions (the implicit GEMM
# with K split), next to a weight gradient over the copies
@pytest.mark.parametrize("case", [(1, 130, 33, 5, 7, 5, 1, 2), (2, 9, 310, 4, 6, 3, 1, 1), (1, 300, 20, 7, 9, 3, 1, 1)], ids=_ids)
@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_few_positions(case, dt):
    test_gather_conv_all_passes(case, dt)


# fp32 1x1 layers on either side of the rule for a forward or a lone input gradient: one row of tiles
# over the implicit GEMM (48, 64 and 24 rows), two rows or few positions over the copies; stride 2
# forward over the implicit GEMM and (257 rows, few positions) the copies
@pytest.mark.parametrize("case", [(100, 64, 48, 13, 13, 1), (65, 65, 64, 16, 16, 1), (64, 64, 64, 16, 16, 1), (3, 24, 66, 77, 73, 1),
                                  (2, 24, 8, 257, 256, 1), (8, 20, 70, 65, 67, 2), (8, 12, 257, 65, 67, 2), (8, 20, 70, 64, 64, 2)])
@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_pointwise_layer_on_either_kernel(case, dt):
    B, C, O, H, W, S = case
    g = rng(B + C)
    conv = vnn.Conv2d(C, O, 1, S, 0, device=DEV, dtype=DTYPES[dt])
    conv.set_algo(vnn.ConvAlgo.IGEMM)
    x, xt = prep(g.standard_normal((B, C, H, W)), dt)
    w, wt = prep(g.standard_normal((O, C, 1, 1)) / np.sqrt(C), dt)
    b, bt = prep(g.standard_normal(O), dt)
    dy, dyt = prep(g.standard_normal((B, O, (H - 1) // S + 1, (W - 1) // S + 1)), dt)
    conv.weight, conv.bias = wt, bt
    kw = dict(stride=(S, S), pad=(0, 0))
    y = conv.forward(xt)
    bb = b[None, :, None, None]
    check(y, oracle.direct_conv, (x, w), dt, "y", kw, extra_ref=bb, extra_scale=np.abs(bb), k=C + 1)
    assert np.array_equal(host(conv.forward(xt, relu=True)), np.maximum(host(y), 0))
    check(conv.backward(dyt, xt, weight_grad=False)[0], oracle.direct_conv_backward_input, (dy, w, x.shape), dt, "dx", kw, k=O)
    dx, dw, db = conv.backward(dyt, xt)
    check(dx, oracle.direct_conv_backward_input, (dy, w, x.shape), dt, "dx together", kw, k=O)
    check(dw, oracle.direct_conv_backward_weight, (dy, x, w.shape), dt, "dw", kw, k=B * H * W)
    check(db, oracle.conv_bias_grad, (dy,), dt, "db", k=B * H * W)


# bf16 on the tiles that the cases above do not pick (host_check pins the choice): 64 x 64 and
# 64 x 128 with three LDS stages of 1 .. 5, 64 x 64 with two wave groups of 9 and 8 stages
@pytest.mark.parametrize("case", [(64, 60, 64, 39, 41, 1, 2), (64, 120, 64, 39, 41, 1, 2), (64, 190, 64, 39, 41, 1, 2),
                                  (64, 250, 64, 39, 41, 1, 2), (64, 300, 64, 39, 41, 1, 2), (128, 60, 64, 39, 41, 1, 2),
                                  (128, 190, 64, 39, 41, 1, 2), (128, 250, 64, 39, 41, 1, 2), (16, 120, 130, 21, 23, 3, 1),
                                  (5, 120, 250, 33, 31, 3, 1)])
def test_gather_bf16_tiles(case):
    B, C, O, H, W, K, S = case
    g = rng(C + B)
    x, xt = prep(g.standard_normal((B, C, H, W)), "bf16")
    w, wt = prep(g.standard_normal((O, C, K, K)) * np.sqrt(2.0 / (C * K * K)), "bf16")
    conv = vnn.Conv2d(C, O, K, S, K // 2, use_bias=False, device=DEV, dtype=DTYPES["bf16"])
    conv.weight = wt
    conv.set_algo(vnn.ConvAlgo.IGEMM)
    kw = dict(stride=(S, S), pad=(K // 2, K // 2))
    y = conv.forward(xt)
    check(y, oracle.direct_conv, (x, w), "bf16", "y", kw, k=C * K * K)
    if S == 1:  # the same tiles in the input gradient, O and C changing places
        dy, dyt = prep(g.standard_normal(tuple(y.shape)), "bf16")
        dx = conv.backward(dyt, xt, weight_grad=False)[0]
        check(dx, oracle.direct_conv_backward_input, (dy, w, x.shape), "bf16", "dx", kw, k=O * K * K)

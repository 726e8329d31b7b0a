"""GPU: products of any size (vh_mm.hip) at the edges of their tiles, stages, K
splits and padded rows, against the oracle under the parity gate."""
import numpy as np
import pytest
import torch

import oracle
from tests.parity import assert_parity
from tests.test_gpu_parity import DEV, DTYPES, check, host, prep, rng
from volta_amd import nn as vnn
from volta_amd import ops

pytestmark = pytest.mark.gpu

# (m, k, n)
CASES = [
    (1, 1, 1), (31, 9, 33),      # below one tile, one unit of k and a bit
    (33, 64, 65), (65, 65, 31),  # one past a tile, one past a stage
    (40, 3000, 24),              # few tiles: K split over blocks
    (129, 4097, 70),             # the same with padded rows, a split's last stage partial
    (300, 96, 1000), (257, 130, 255),
    (520, 250, 520),             # 32 x 64 tiles in two K groups, dA and dB of 9 stages
    (1030, 72, 1100),            # bf16 64 x 128 tiles with remainders; dA 32 x 64, dB 32 x 32 of 17 stages
    (2060, 40, 2072),            # many 64 x 64 tiles of one stage, aligned rows; dB split
    (2050, 33, 2310),            # the same, padded rows
    (4100, 16, 2056),            # 2145 tiles of a quarter stage; dA and dB of few deep tiles
]


@pytest.mark.parametrize("mkn", CASES)
@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_mm_family(mkn, dt):
    m, k, n = mkn
    g = rng(m * 3 + k * 5 + n)
    a, at = prep(g.standard_normal((m, k)), dt)
    b, bt = prep(g.standard_normal((k, n)), dt)
    gr, grt = prep(g.standard_normal((m, n)), dt)
    check(ops.gpu_matmul(at, bt, m, k, n), oracle.matmul, (a, b), dt, "matmul", k=k)
    check(ops.gpu_matmul_backward_a(grt, bt, m, k, n), oracle.matmul_backward_a, (gr, b), dt, "dA", k=n)
    check(ops.gpu_matmul_backward_b(at, grt, m, k, n), oracle.matmul_backward_b, (a, gr), dt, "dB", k=m)


@pytest.mark.parametrize("shape", [(3, 5, 7), (34, 3846, 80), (256, 784, 512), (1000, 60, 44), (70, 1030, 900)])
@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_mm_linear(shape, dt):
    m, i, o = shape
    g = rng(m + i + o)
    x, xt = prep(g.standard_normal((m, i)), dt)
    w, wt = prep(g.uniform(-0.5, 0.5, (i, o)), dt)
    b, bt = prep(g.uniform(-1, 1, (o,)), dt)
    dy, dyt = prep(g.standard_normal((m, o)), dt)
    lin = vnn.Linear(i, o, device=DEV, dtype=DTYPES[dt])
    lin.weight, lin.bias = wt, bt
    check(lin.forward(xt), oracle.linear_forward, (x, w, b), dt, "y", k=i + 1)
    got = lin.backward(dyt, xt)  # dX and dW in one launch
    for q, (what, k) in enumerate((("dx", o), ("dw", m), ("db", m))):
        check(got[q], lambda *a, q=q: oracle.linear_backward(*a)[q], (dy, x, w), dt, what, k=k)
    one = lin.backward(dyt, xt, input_grad=False)
    for q, what in ((1, "dw"), (2, "db")):
        check(one[q], lambda *a, q=q: oracle.linear_backward(*a)[q], (dy, x, w), dt, what + " alone", k=m)
    assert lin.backward(dyt, xt, weight_grad=False)[0].shape == xt.shape


@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_mm_unaligned_operands(dt):
    """Views that start off a 16-byte boundary take the padded copies."""
    m, k, n = 70, 64, 48
    g = rng(9)
    a, _ = prep(g.standard_normal((m, k)), dt)
    b, _ = prep(g.standard_normal((k, n)), dt)

    def view(x):
        t = torch.empty(x.size + 1, device=DEV, dtype=DTYPES[dt])[1:].view(x.shape)
        t.copy_(torch.from_numpy(x))
        return t

    check(ops.gpu_matmul(view(a), view(b), m, k, n), oracle.matmul, (a, b), dt, "matmul", k=k)


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("mkn", [(5, 7, 9), (40, 3001, 24)])
def test_mm_padding_does_not_leak(mkn, dt):
    """An infinity stays in its row and column: stage, row and unit padding is zero."""
    m, k, n = mkn
    a, b = torch.ones((m, k), device=DEV, dtype=DTYPES[dt]), torch.ones((k, n), device=DEV, dtype=DTYPES[dt])
    a[m - 1, k - 1] = float("inf")
    c = np.isfinite(host(ops.gpu_matmul(a, b, m, k, n)))
    assert c[: m - 1].all() and not c[m - 1].any()
    db = np.isfinite(host(ops.gpu_matmul_backward_b(a, torch.ones((m, n), device=DEV, dtype=DTYPES[dt]), m, k, n)))
    assert db[: k - 1].all() and not db[k - 1].any()


@pytest.mark.parametrize("k", [700, 768, 772, 896, 1030])  # 11 stages (two in LDS) .. 17 (three), on every tile
@pytest.mark.parametrize("m,n", [(40, 1200), (520, 264), (1024, 1024), (1500, 1111), (1536, 2048), (1537, 2048)])
def test_mm_bf16_stages_in_flight(m, k, n):
    g = rng(m + k + n)
    a, at = prep(g.standard_normal((m, k)), "bf16")
    b, bt = prep(g.standard_normal((k, n)), "bf16")
    check(ops.gpu_matmul(at, bt, m, k, n), oracle.matmul, (a, b), "bf16", "matmul", k=k)
    gr, grt = prep(g.standard_normal((m, k)), "bf16")  # dA = G [m][k] . B^T, reduced over k
    w, wt = prep(g.standard_normal((n, k)), "bf16")
    check(ops.gpu_matmul_backward_a(grt, wt, m, n, k), oracle.matmul_backward_a, (gr, w), "bf16", "dA", k=k)


# a long batch over few features (dW: few tiles of a deep K, split beside dX's many), then
# the pair on 64 x 128 and 128 x 128 tiles (bf16) with remainders, aligned rows and padded ones
@pytest.mark.parametrize("shape", [(5000, 12, 30), (4100, 70, 64), (1030, 1032, 2056), (1700, 1544, 1800), (2056, 1290, 2312)])
@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_mm_linear_gradients_in_one_launch(shape, dt):
    m, i, o = shape
    g = rng(m + i + o)
    x, xt = prep(g.standard_normal((m, i)), dt)
    w, wt = prep(g.uniform(-0.5, 0.5, (i, o)), dt)
    dy, dyt = prep(g.standard_normal((m, o)), dt)
    lin = vnn.Linear(i, o, device=DEV, dtype=DTYPES[dt])
    lin.weight = wt
    ref = oracle.linear_backward(dy, x, w)
    scale = oracle.linear_backward(np.abs(dy), np.abs(x), np.abs(w))
    for got, r, s, what, k in zip(lin.backward(dyt, xt), ref, scale, ("dx", "dw", "db"), (o, m, m)):
        assert_parity(host(got), r, s, dt, what, k=k)


# K short or an operand long: the implicit GEMM's side of the rule, and just past it
@pytest.mark.parametrize("mkn", [(30, 38, 139), (60, 161, 120), (4000, 9, 37), (4000, 25, 150), (3, 2050, 1003), (17, 1030, 3001)])
@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_mm_or_implicit_gemm(mkn, dt):
    test_mm_family(mkn, dt)


# dB alone on 128 x 128 tiles (bf16) with remainders, aligned rows and padded ones
@pytest.mark.parametrize("mkn", [(300, 2056, 2064), (289, 2299, 2308)])
def test_mm_bf16_backward_b_128x128_tiles(mkn):
    m, k, n = mkn
    g = rng(m + k + n)
    a, at = prep(g.standard_normal((m, k)), "bf16")
    gr, grt = prep(g.standard_normal((m, n)), "bf16")
    check(ops.gpu_matmul_backward_b(at, grt, m, k, n), oracle.matmul_backward_b, (a, gr), "bf16", "dB", k=m)


def test_stream_of_a_device():
    """The current stream by a tensor's device, an index, a name or nothing; no other device has one."""
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        for d in (torch.zeros(1, device=DEV).device, 0, "cuda", "cuda:0", torch.device("cuda"), None):
            assert ops.stream_ptr(d) == side.cuda_stream
    for d in ("cpu", torch.device("cpu")):
        with pytest.raises(ValueError):
            ops.stream_ptr(d)


def test_algorithm_given_as_a_plain_number():
    conv = vnn.Conv2d(3, 4, 3, 1, 1, device=DEV)
    x = torch.randn(2, 3, 6, 6, device=DEV)
    conv.algo = np.int64(int(vnn.ConvAlgo.IGEMM))
    y = conv.forward(x)
    assert conv.last_algo == vnn.ConvAlgo.IGEMM
    conv.algo = vnn.ConvAlgo.IGEMM
    assert torch.equal(conv.forward(x), y)


# fp32 dX + dW in one launch: whole tiles with sums in two levels (no product fills the chip with
# 256 x 256 tiles), dX or a dW without db in one level (it does: 16384 x 1024, 4096 x 4096),
# smaller tiles; where a product alone has the same groups and splits of K, its bits (dW of
# 16384 x 1024 x 256 is split alone)
@pytest.mark.parametrize("shape", [(4096, 2048, 2048), (16384, 1024, 128), (4096, 4096, 4096), (300, 200, 260), (16384, 1024, 256),
                                   (1024, 4096, 4096)])
@pytest.mark.parametrize("bias", [True, False])
def test_linear_gradients_together_and_alone(shape, bias):
    m, i, o = shape
    torch.manual_seed(m + i + o)
    lin = vnn.Linear(i, o, use_bias=bias, device=DEV)
    x, dy = torch.randn(m, i, device=DEV), torch.randn(m, o, device=DEV)
    dx, dw, db = lin.backward(dy, x)
    assert torch.equal(lin.backward(dy, x, weight_grad=False)[0], dx)
    _, dw1, db1 = lin.backward(dy, x, input_grad=False)
    if shape != (16384, 1024, 256):
        assert torch.equal(dw1, dw)
    if not bias:
        return
    # (db: column sums of the staged tiles, or of dY: the bound of m additions in any order)
    bound = 2.0 ** -24 * m * dy.double().abs().sum(0)
    assert bool(((db.double() - dy.double().sum(0)).abs() <= bound).all())
    assert bool(((db1.double() - dy.double().sum(0)).abs() <= bound).all())


# dW deep beside a dX that fills the chip: two launches (fp32; whole tiles of either type), whose
# outputs are those of separate calls
@pytest.mark.parametrize("shape", [(20600, 260, 50), (16384, 512, 256)])
@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_linear_gradients_of_a_long_batch(shape, dt):
    m, i, o = shape
    torch.manual_seed(m + i + o)
    lin = vnn.Linear(i, o, device=DEV, dtype=DTYPES[dt])
    x, dy = (torch.randn(m, n, device=DEV).to(DTYPES[dt]) for n in (i, o))
    dx, dw, db = (t.double().cpu() for t in lin.backward(dy, x))
    x, dy, w = (t.double().cpu() for t in (x, dy, lin.weight))
    u = 2.0 ** (-24 if dt == "f32" else -8)
    for got, a, b in ((dx, dy, w.t()), (dw, x.t(), dy)):  # random signs: the error is far below k u S
        ref, s, k = a @ b, a.abs() @ b.abs(), a.shape[1]
        assert bool(((got - ref).abs() <= 2.0 ** -24 * k * s + u * ref.abs()).all())
    assert bool(((db - dy.sum(0)).abs() <= 2.0 ** -24 * m * dy.abs().sum(0) + u * dy.sum(0).abs()).all())

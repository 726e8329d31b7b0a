"""GPU: fp32 results against 64 bits, at sums long enough for their order to show.

A sum of n products of N(0, 1) values taken one after the other rounds n partial
sums, the k-th of about sqrt(k): each by at most u / sqrt(3) of it in the root mean
square (u = 2^-24), u sqrt(n / 6) of the result together.  Taken as sums of 64 products
that are then added up it is u sqrt((64 + n / 64) / 6): 4.6 u at n = 4096, where one long
sum may show 26 u (19 u measured).  Column sums go through at most three levels of 16
additions each: u sqrt(3 * 16 / 6).  The bounds below are these; one long sum exceeds
them at every size here."""
import pytest
import torch
import torch.nn.functional as F

from volta_amd import nn as vnn, ops

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
U = 2.0 ** -24


def _rand(*shape, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(DEV)


def _check(got, ref, n, what, column_sum=False):
    err = float((got.double() - ref).norm() / ref.norm())
    bound = U * ((3 * 16 if column_sum else 64 + n / 64) / 6) ** 0.5
    print(f"{what}: n {n} error {err:.2e} bound {bound:.2e}", flush=True)
    assert err <= bound, f"{what}: error {err:.2e} against 64 bits, bound {bound:.2e} for {n} products"


# few channels, many splits; many channels, all positions in one split; a narrow layer on neither
@pytest.mark.parametrize("case", [(4, 512, 512, 32, 32), (8, 64, 96, 31, 33), (16, 256, 256, 14, 15)])
def test_conv_gradients(case):
    B, C, O, H, W = case
    conv = vnn.Conv2d(C, O, 3, 1, 1, device=DEV)
    conv.set_algo(vnn.ConvAlgo.IGEMM)
    x, dy = _rand(B, C, H, W, seed=1), _rand(B, O, H, W, seed=2)
    _, dw, db = conv.backward(dy, x, input_grad=False)
    d = dy[:, :16].double().permute(1, 0, 2, 3).reshape(16, -1)
    xp = F.pad(x.double(), (1, 1, 1, 1))
    for r, q in ((0, 0), (1, 1), (2, 0)):
        v = xp[:, :, r:r + H, q:q + W].permute(0, 2, 3, 1).reshape(-1, C)
        _check(dw[:16, :, r, q], d @ v, B * H * W, f"dW tap {r},{q}")
    _check(db, dy.double().sum((0, 2, 3)), B * H * W, "db", column_sum=True)


@pytest.mark.parametrize("case", [(1, 512, 512, 7, 7), (2, 300, 200, 14, 13), (8, 128, 128, 31, 29)])
def test_conv_forward_and_input_gradient(case):
    B, C, O, H, W = case
    conv = vnn.Conv2d(C, O, 3, 1, 1, use_bias=False, device=DEV)
    conv.set_algo(vnn.ConvAlgo.IGEMM)
    conv.weight = _rand(O, C, 3, 3, seed=3)
    x, dy = _rand(B, C, H, W, seed=1), _rand(B, O, H, W, seed=2)
    w = conv.weight.double()
    wf = w.reshape(O, -1)
    cols = F.unfold(x.double(), 3, padding=1).permute(1, 0, 2).reshape(C * 9, -1)
    y = (wf @ cols).reshape(O, B, H, W).permute(1, 0, 2, 3)
    _check(conv.forward(x), y, 9 * C, "y")
    wt = w.flip(2, 3).permute(1, 0, 2, 3).reshape(C, -1).contiguous()
    cols = F.unfold(dy.double(), 3, padding=1).permute(1, 0, 2).reshape(O * 9, -1)
    dx = (wt @ cols).reshape(C, B, H, W).permute(1, 0, 2, 3)
    _check(conv.backward(dy, x, weight_grad=False)[0], dx, 9 * O, "dX")


@pytest.mark.parametrize("mkn", [(512, 8192, 512), (1000, 4096, 900), (64, 16384, 64), (3, 4096, 1000)])
def test_products(mkn):
    m, k, n = mkn
    a, b = _rand(m, k, seed=1), _rand(k, n, seed=2)
    _check(ops.gpu_matmul(a, b, m, k, n), a.double() @ b.double(), k, "A B")
    g, bt = _rand(m, k, seed=3), _rand(n, k, seed=4)
    _check(ops.gpu_matmul_backward_a(g, bt, m, n, k), g.double() @ bt.double().t(), k, "G B^T")
    at, h = _rand(k, m, seed=5), _rand(k, n, seed=6)
    _check(ops.gpu_matmul_backward_b(at, h, k, m, n), at.double().t() @ h.double(), k, "A^T G")


@pytest.mark.parametrize("mio", [(16384, 64, 64), (4096, 100, 36), (2048, 500, 300)])
def test_linear_gradients(mio):
    m, i, o = mio
    layer = vnn.Linear(i, o, device=DEV)
    x, dy = _rand(m, i, seed=1), _rand(m, o, seed=2)
    _, dw, db = layer.backward(dy, x)
    _check(dw, x.double().t() @ dy.double(), m, "dW")
    _check(db, dy.double().sum(0), m, "db", column_sum=True)

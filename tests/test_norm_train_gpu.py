"""Trainer RMSNorm backward at the edges of its blocks (rows a block walks)
and words (columns a thread holds), against float64 autograd."""
import pytest
import torch

import polyrl_amd.ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("t,h", [(1, 8), (3, 2048), (1023, 256), (1025, 2056),
                                 (2100, 4096), (5, 8192), (7, 16384),
                                 (3, 16392)])
@pytest.mark.parametrize("use", ["both", "norm", "sum", "no residual"])
def test_backward(t, h, use):
    torch.manual_seed(4)
    x, res = (torch.randn(t, h, device=DEV).bfloat16().requires_grad_()
              for _ in range(2))
    w = torch.randn(h, device=DEV).bfloat16().requires_grad_()
    gy, gh = (torch.randn(t, h, device=DEV).bfloat16() for _ in range(2))
    eps = 1e-5
    if use == "no residual":
        ops.rmsnorm_train(x, w, eps).backward(gy)
        s = x.detach().double()
    else:
        y, s = ops.fused_add_rmsnorm_train(x, res, w, eps)
        outs = {"both": (y, s), "norm": (y,), "sum": (s,)}[use]
        grads = {"both": (gy, gh), "norm": (gy,), "sum": (gh,)}[use]
        torch.autograd.backward(outs, grads)
        assert torch.equal(x.grad, res.grad)
        s = s.detach().double()
    s.requires_grad_()
    w64 = w.detach().double().requires_grad_()
    y64 = s / (s.square().mean(-1, keepdim=True) + eps).sqrt() * w64
    loss = 0.0
    if use != "sum":
        loss = loss + (y64 * gy.double()).sum()
    if use in ("both", "sum"):
        loss = loss + (s * gh.double()).sum()
    loss.backward()
    # rounded once to bf16; 32-bit sums over a row and over t rows.  Rows
    # wider than 16384 take two steps: the norm's share is rounded before the
    # sum's gradient is added
    bound = 2 ** -8 * s.grad.abs() + 1e-5
    if h > 16384 and use == "both":
        bound = bound + 2 ** -8 * (s.grad - gh.double()).abs()
    off = (x.grad.double() - s.grad).abs()
    assert (off <= bound).all()
    if use != "sum":
        size = (gy.double() * y64 / w64).abs().sum(0)
        off = (w.grad.double() - w64.grad).abs()
        assert (off <= 2 ** -8 * w64.grad.abs() + 1e-5 * size + 1e-6).all()


def test_backward_of_the_sum_alone():
    """Where only the sum is used the weight's gradient is zero, not absent."""
    x, res = (torch.randn(5, 64, device=DEV).bfloat16().requires_grad_()
              for _ in range(2))
    w = torch.randn(64, device=DEV).bfloat16().requires_grad_()
    _, s = ops.fused_add_rmsnorm_train(x, res, w, 1e-5)
    g = torch.randn(5, 64, device=DEV).bfloat16()
    dx, dres, dw = torch.autograd.grad(s, (x, res, w), g)
    assert torch.equal(dx, g) and torch.equal(dres, g)
    assert dw.dtype == w.dtype and (dw == 0).all()


def test_backward_of_nothing():
    """No gradient reaches either output: zeros."""
    class Drop(torch.autograd.Function):
        @staticmethod
        def forward(ctx, a, b):
            return a + b

        @staticmethod
        def backward(ctx, g):
            return None, None

    x, res = (torch.randn(5, 64, device=DEV).bfloat16().requires_grad_()
              for _ in range(2))
    w = torch.randn(64, device=DEV).bfloat16().requires_grad_()
    out = Drop.apply(*ops.fused_add_rmsnorm_train(x, res, w, 1e-5))
    for g, t in zip(torch.autograd.grad(out.sum(), (x, res, w)), (x, res, w)):
        assert g.shape == t.shape and (g == 0).all()

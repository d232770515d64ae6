"""Log-probability and sampling kernels over the vocabulary at the edges of
their words, blocks and row splits.  References: float64 log-softmax."""
import pytest
import torch

import polyrl_amd.ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,v", [(1, 1), (3, 7), (5, 8), (4, 1023),
                                 (1025, 333), (2, 50257), (1030, 8192 + 5),
                                 (3, 151936)])
def test_logprobs_rows_and_entropy(n, v, dtype):
    torch.manual_seed(1)
    x = (torch.randn(n, v, device=DEV) * 3).to(dtype)
    if v > 20:                       # masked entries of both kinds, and a row
        x[:, 5] = torch.finfo(dtype).min      # that starts with one
        x[0, 0] = torch.finfo(dtype).min
    lab = torch.randint(v, (n,), device=DEV)
    lp, ent = ops.gather_logprobs(x, lab, want_entropy=True)
    want = torch.log_softmax(x.double(), -1)
    at = want.gather(1, lab[:, None])[:, 0]
    # 32-bit: the label's logit and the log-sum-exp are each rounded, the sum
    # of v terms adds less than 1e-6 relative
    tol = 2e-6 * (1 + at.abs()) + 4e-7 * x.double().gather(
        1, lab[:, None])[:, 0].abs()
    assert ((lp.double() - at).abs() <= tol).all()
    p = want.exp()
    h = -(p * want.clamp_min(-1e30)).sum(-1)
    assert (ent.double() - h).abs().max() <= 2e-5 * (1 + h.abs().max())
    assert torch.equal(ops.gather_logprobs(x, lab), lp)
    if dtype == torch.bfloat16:
        g = x.clone().requires_grad_()
        lp2 = ops.gather_logprobs_train(g, lab)
        assert torch.equal(lp2, lp)
        dlp = torch.randn(n, device=DEV)
        lp2.backward(dlp)
        dx = -dlp[:, None].double() * p
        dx.scatter_add_(1, lab[:, None], dlp[:, None].double())
        # rounded once to bf16, the label's entry twice
        tol = 2 ** -7 * dx.abs() + 1e-6
        tol.scatter_add_(1, lab[:, None], 2 ** -8 * dlp[:, None].abs().double())
        assert ((g.grad.double() - dx).abs() <= tol).all()


@pytest.mark.parametrize("v", [64, 50257])
def test_logprobs_minus_infinity(v):
    """Banned tokens (-inf): probability 0, everything else as without them."""
    x = torch.randn(2, v, device=DEV).bfloat16()
    x[:, : v // 2] = -float("inf")
    lab = torch.tensor([v - 1, v // 2], device=DEV)
    want = torch.log_softmax(x.double(), -1).gather(1, lab[:, None])[:, 0]
    assert (ops.gather_logprobs(x, lab).double() - want).abs().max() < 1e-5

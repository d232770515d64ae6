"""Weight gradients dY^T X: the edges of stages and tiles, tiles whose rows are
shared among blocks, the trainer's use of them."""
import pytest
import torch

import polyrl_amd.ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rand(m, n, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(m, n, generator=g, device=DEV).bfloat16()


def check(dy, x, got):
    a, b = dy.double(), x.double()
    want, mass = a.t() @ b, a.abs().t() @ b.abs()
    # 32-bit sums of M products, each off by 2^-24 of the sum of magnitudes at
    # most, and one rounding to bf16
    bound = 2 ** -8 * want.abs() + len(dy) * 2.0 ** -24 * mass
    assert got.shape == want.shape
    assert ((got.double() - want).abs() <= bound).all()


def direct(m, n, k):
    dy, x = rand(m, n, m + n), rand(m, k, m + k + 1)
    check(dy, x, ops._require_ext().linear_wgrad(dy, x))


@pytest.mark.parametrize("m", [1, 31, 32, 33, 64, 65, 127, 128, 129, 160, 200,
                               257, 450])
def test_rows(m):
    """Fewer stages than are on their way at once, odd ones, a last one of some
    rows."""
    direct(m, 256, 264)


@pytest.mark.parametrize("n,k", [(8, 8), (8, 520), (248, 256), (264, 1000),
                                 (2048, 256), (2312, 512), (4360, 264)])
def test_columns(n, k):
    """Columns short of a tile, one tile more than a group of rows of tiles."""
    direct(96, n, k)


@pytest.mark.parametrize("m", [1280, 1283, 1950, 5121, 8191])
@pytest.mark.parametrize("n,k", [(256, 256), (264, 520), (1024, 1304)])
def test_shared_rows(m, n, k):
    """Two blocks and more for a tile, unequal parts, edges in the sums."""
    direct(m, n, k)


def test_rows_behind_the_last_are_zero():
    """What stands in memory behind an operand has no part in its product."""
    m, n, k = 70, 136, 72
    dy = torch.full((m + 64, n), float("nan"), device=DEV).bfloat16()
    x = torch.full((m + 64, k), float("inf"), device=DEV).bfloat16()
    dy[:m], x[:m] = rand(m, n, 3), rand(m, k, 4)
    check(dy[:m], x[:m], ops._require_ext().linear_wgrad(dy[:m], x[:m]))


@pytest.mark.parametrize("m,n,k", [
    (511, 5120, 2048), (512, 5120, 2048), (600, 5112, 2040),  # 160 tiles
    (5119, 512, 256), (5120, 512, 256), (600, 5116, 2048)])
def test_linear_backward(m, n, k):
    """Both sides of the lines where the trainer's linears take the kernel, and
    columns that it does not take."""
    x = rand(m, k, 5).requires_grad_()
    w = (rand(n, k, 6) / 8).requires_grad_()
    dy = rand(m, n, 7)
    ops.tuned_linear(x, w).backward(dy)
    check(dy, x.detach(), w.grad)


def test_refused():
    ext = ops._require_ext()
    with pytest.raises(RuntimeError):
        ext.linear_wgrad(rand(64, 12, 0), rand(64, 16, 0))
    with pytest.raises(RuntimeError):
        ext.linear_wgrad(rand(0, 16, 0), rand(0, 16, 0))
    with pytest.raises(RuntimeError):
        ext.linear_wgrad(rand(64, 16, 0), rand(65, 16, 0))

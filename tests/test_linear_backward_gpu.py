"""Gradients of linear layers, dY^T X and dY W: the edges of steps and tiles, tiles
whose inner numbers are shared among blocks, the trainer's use of them."""
import pytest
import torch

import polyrl_amd.ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rand(m, n, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(m, n, generator=g, device=DEV).bfloat16()


def check(a, b, got):
    """got = a b"""
    a, b = a.double(), b.double()
    want, mass = a @ b, a.abs() @ b.abs()
    # 32-bit sums of the inner products, each off by 2^-24 of the sum of
    # magnitudes at most, and one rounding to bf16
    bound = 2 ** -8 * want.abs() + a.shape[1] * 2.0 ** -24 * mass
    assert got.shape == want.shape
    assert ((got.double() - want).abs() <= bound).all()


def wgrad(m, n, k):
    dy, x = rand(m, n, m + n), rand(m, k, m + k + 1)
    check(dy.t(), x, ops._require_ext().linear_wgrad(dy, x))


def dgrad(m, n, k):
    dy, w = rand(m, n, m + n), rand(n, k, n + k + 1)
    check(dy, w, ops._require_ext().linear_dgrad(dy, w))


@pytest.mark.parametrize("m", [1, 31, 32, 33, 64, 65, 127, 128, 129, 160, 200,
                               257, 450])
def test_wgrad_inner(m):
    """Fewer steps than are on their way at once, odd ones, a last one of some
    rows."""
    wgrad(m, 256, 264)


@pytest.mark.parametrize("n,k", [(8, 8), (8, 520), (248, 256), (264, 1000),
                                 (2048, 256), (2312, 512), (4360, 264)])
def test_wgrad_outer(n, k):
    """Columns short of a tile, one tile more than a group of rows of tiles."""
    wgrad(96, n, k)


@pytest.mark.parametrize("n", [64, 128, 192, 256, 320, 384, 448, 576])
@pytest.mark.parametrize("m,k", [(256, 264), (3, 256)])
def test_dgrad_inner(m, n, k):
    """One pair of steps to more than two rounds of the three that LDS holds."""
    dgrad(m, n, k)


@pytest.mark.parametrize("m,k", [(1, 8), (8, 520), (255, 256), (257, 1000),
                                 (2049, 256), (2311, 512), (4353, 264)])
def test_dgrad_outer(m, k):
    """Rows and columns short of a tile, one tile more than a group of rows of
    tiles."""
    dgrad(m, 192, k)


@pytest.mark.parametrize("n", [64, 128, 192, 256, 320])
@pytest.mark.parametrize("m", [1500, 1791, 1799, 2041])
def test_dgrad_rows(m, n):
    """Tiles of 192 rows, 224 and 256: one round of them each."""
    dgrad(m, n, 8184)


@pytest.mark.parametrize("inner", [193, 256, 320, 384, 448])
def test_tiles_in_turn(inner):
    """More tiles than blocks that run at once: a block's second tile and third,
    whose first units are loaded during the one before; fewer units than that
    takes."""
    wgrad(inner, 4360, 4104)
    dgrad(4353, (inner + 63) // 64 * 64, 8200)


@pytest.mark.parametrize("n", [256, 320, 384])
@pytest.mark.parametrize("m,parts", [(189, 6), (221, 7), (445, 7), (253, 8), (509, 8)])
def test_dgrad_rows_in_turn(m, parts, n):
    """A block's second tile and third of every number of row parts: a tile's sums
    leave beside the next one's first step."""
    cols = 290                         # (more tiles than blocks that run at once)
    assert ops._require_ext().product_rows(m, cols, n, 6)[0] == parts
    dgrad(m, n, 256 * cols - 8)


@pytest.mark.parametrize("inner", [1280, 1344, 1984, 5120, 8192])
@pytest.mark.parametrize("n,k", [(256, 256), (264, 520), (1024, 1304)])
def test_shared(inner, n, k):
    """Two blocks and more for a tile, unequal parts, edges in the sums."""
    wgrad(inner - 1, n, k)
    dgrad(n, inner, k)


def test_behind_the_last():
    """What stands in memory behind an operand has no part in its product."""
    m, n, k = 70, 192, 72
    dy = torch.full((m + 64, n), float("nan"), device=DEV).bfloat16()
    x = torch.full((m + 64, k), float("inf"), device=DEV).bfloat16()
    w = torch.full((n + 64, k), float("inf"), device=DEV).bfloat16()
    dy[:m], x[:m], w[:n] = rand(m, n, 3), rand(m, k, 4), rand(n, k, 5)
    ext = ops._require_ext()
    check(dy[:m].t(), x[:m], ext.linear_wgrad(dy[:m], x[:m]))
    check(dy[:m], w[:n], ext.linear_dgrad(dy[:m], w[:n]))


def same_kinds(got, want):
    for kind in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(kind(got), kind(want))
    live = want.isfinite()
    assert live.any() and not live.all()
    assert (got.double() - want)[live].norm() <= 5e-3 * want[live].norm()


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_not_finite(bad):
    """Numbers that are not finite reach the sums that they are a part of, and no
    other ones."""
    ext = ops._require_ext()
    m, n, k = 600, 320, 264
    dy, x, w = rand(m, n, 3), rand(m, k, 4), rand(n, k, 5)
    dy[17, 3] = dy[m - 1, n - 1] = x[40, 9] = w[250, 100] = bad
    x[17, 5] = w[3, 7] = 0             # (times infinity)
    d, f, v = dy.double(), x.double(), w.double()
    same_kinds(ext.linear_wgrad(dy, x), d.t() @ f)
    same_kinds(ext.linear_dgrad(dy, w), d @ v)
    same_kinds(ext.linear_dgrad_sum([dy, dy[:, :64].contiguous()],
                                    [w, w[:64].contiguous()]),
               d @ v + d[:, :64] @ v[:64])
    m, k = 1700, 192
    x, wg, wu = rand(m, k, 6), rand(4096, k, 7), rand(4096, k, 8)
    x[m - 1, 0] = wg[2000, k - 1] = wu[4095, 5] = bad
    y, gate, up = ext.linear_gated(x, wg, wu, True)
    g, u = x.double() @ wg.double().t(), x.double() @ wu.double().t()
    same_kinds(gate, g)
    same_kinds(up, u)
    same_kinds(y, g * torch.sigmoid(g) * u)
    out = rand(m, 4096, 9)
    out[5, 6] = out[m - 1, 2000] = -bad
    old = out.double()
    ops.linear_rows_add(out, x, wg)
    same_kinds(out, old + g)


@pytest.mark.parametrize("m,n,k", [
    (511, 5120, 2048), (512, 5120, 2048), (600, 5112, 2040),  # 160 tiles of dW
    (5119, 512, 256), (5120, 512, 256), (600, 5116, 2048),
    (2600, 256, 4096), (2700, 256, 4096), (5200, 320, 4096),  # 176, 336 of dX
    (64, 8128, 264), (63, 8192, 264), (64, 8192, 264), (130, 8224, 520),
    (270, 8192, 11264), (460, 8192, 11264)])          # two blocks a tile of dX
def test_linear_backward(m, n, k):
    """Both sides of the lines where the trainer's linears take the kernels, and
    columns that they do not take."""
    x = rand(m, k, 5).requires_grad_()
    w = (rand(n, k, 6) / 8).requires_grad_()
    dy = rand(m, n, 7)
    ops.tuned_linear(x, w).backward(dy)
    check(dy.t(), x.detach(), w.grad)
    check(dy, w.detach(), x.grad)


def test_refused():
    ext = ops._require_ext()
    for dy, x in (((64, 12), (64, 16)), ((0, 16), (0, 16)), ((64, 16), (65, 16))):
        with pytest.raises(RuntimeError):
            ext.linear_wgrad(rand(*dy, 0), rand(*x, 0))
    for dy, w in (((64, 96), (96, 16)), ((64, 64), (64, 12)), ((0, 64), (64, 8)),
                  ((64, 64), (128, 16))):
        with pytest.raises(RuntimeError):
            ext.linear_dgrad(rand(*dy, 0), rand(*w, 0))


@pytest.mark.parametrize("m", [1, 190, 449])
@pytest.mark.parametrize("ns", [(64, 128), (256, 64, 320), (448, 64, 64),
                                (512, 512)])
def test_dgrad_sum(m, ns):
    """Products of unequal inner dimensions, from one unit on, edges of tiles."""
    dys = [rand(m, n, 3 + i) for i, n in enumerate(ns)]
    ws = [rand(n, 520, 13 + i) for i, n in enumerate(ns)]
    got = ops._require_ext().linear_dgrad_sum(dys, ws)
    check(torch.cat(dys, 1), torch.cat(ws), got)


@pytest.mark.parametrize("m", [1500, 1791, 1799, 2041, 4700])
def test_dgrad_sum_rows(m):
    """Tiles of 192, 224 and 256 rows; blocks with a second tile and third."""
    dys, ws = [rand(m, 192, 3), rand(m, 64, 4)], [rand(192, 8184, 5), rand(64, 8184, 6)]
    got = ops._require_ext().linear_dgrad_sum(dys, ws)
    check(torch.cat(dys, 1), torch.cat(ws), got)


def test_dgrad_sum_refused():
    ext = ops._require_ext()
    dy, w = rand(64, 64, 1), rand(64, 128, 2)
    for dys, ws in (([dy], [w]), ([dy, dy], [w]), ([dy] * 4, [w] * 4),
                    ([dy, dy[:32]], [w, w]), ([dy, dy], [w, rand(64, 136, 3)]),
                    ([dy, rand(64, 72, 1)], [w, rand(72, 128, 2)])):
        with pytest.raises(RuntimeError):
            ext.linear_dgrad_sum(dys, ws)
        assert len(dys) == len(ws) == 2 or not ext.linear_dgrad_sum_takes(dys, ws)


@pytest.mark.parametrize("m,ns,k", [(760, (8192, 7936, 256), 128),
                                    (1700, (6144, 2048), 192),
                                    (4400, (2048, 512, 512), 256)])
def test_joint_linear(m, ns, k):
    """Forward and gradients of layers of one input, against each layer's own."""
    mods = [torch.nn.Linear(k, n, bias=i == 1, device=DEV, dtype=torch.bfloat16)
            for i, n in enumerate(ns)]
    x = rand(m, k, 5).requires_grad_()
    ys = ops.joint_linear(x, mods)
    assert ys is not None
    dys = [rand(m, n, 7 + i) for i, n in enumerate(ns)]
    torch.autograd.backward(ys, dys)
    for y, dy, mod in zip(ys, dys, mods):
        want = x.detach().double() @ mod.weight.detach().double().t()
        if mod.bias is None:
            check(x.detach(), mod.weight.detach().t(), y.detach())
        else:
            want += mod.bias.detach().double()
            assert (y - want).norm() <= 5e-3 * want.norm()
            assert (mod.bias.grad - dy.sum(0)).norm() <= 1e-2 * dy.sum(0).norm()
        check(dy.t(), x.detach(), mod.weight.grad)
    want = sum(dy.double() @ m.weight.detach().double() for dy, m in zip(dys, mods))
    assert (x.grad - want).norm() <= 5e-3 * want.norm()


@pytest.mark.parametrize("m,n,k", [(760, 8192, 128), (1700, 4096, 192),
                                   (2041, 4096, 320), (4400, 1664, 256)])
def test_gated_linear(m, n, k, monkeypatch):
    """Gate, up and activation of one kernel with their gradients; the products are
    stored for a way back alone, and the result is the same without."""
    gate, up = (torch.nn.Linear(k, n, bias=False, device=DEV, dtype=torch.bfloat16)
                for _ in range(2))
    x = rand(m, k, 5).requires_grad_()
    ext, kept = ops._require_ext(), []
    real = ext.linear_gated
    monkeypatch.setattr(ext, "linear_gated",
                        lambda *a: kept.append(a[-1]) or real(*a))
    y = ops.gated_linear(x, gate, up)
    with torch.no_grad():              # (a log-probability pass)
        assert torch.equal(ops.gated_linear(x, gate, up), y)
    for l in (gate, up):
        l.requires_grad_(False)
    assert torch.equal(ops.gated_linear(x.detach(), gate, up), y)
    for l in (gate, up):
        l.requires_grad_(True)
    assert kept == [True, False, False]
    alone, = real(x.detach(), gate.weight, up.weight, False)
    assert torch.equal(alone, y)
    dy = rand(m, n, 7)
    y.backward(dy)
    xd = x.detach().double().requires_grad_()
    wd = [l.weight.detach().double().requires_grad_() for l in (gate, up)]
    want = torch.nn.functional.silu(xd @ wd[0].t()) * (xd @ wd[1].t())
    want.backward(dy.double())
    for got, exact in ((y, want), (x.grad, xd.grad), (gate.weight.grad, wd[0].grad),
                       (up.weight.grad, wd[1].grad)):
        # (roundings to bf16 of the products, their gradients and the result)
        assert (got - exact).norm() <= 1e-2 * exact.norm()


def test_joint_other_layers():
    """Who is not a plain layer of bf16 weights has its own forward."""
    class Other(torch.nn.Linear):
        pass

    def lin(cls=torch.nn.Linear, k=128, bias=False, **kw):
        return cls(k, 8192, bias=bias, device=DEV, **{"dtype": torch.bfloat16, **kw})

    x = rand(760, 128, 1)
    assert ops.joint_linear(x, (lin(), lin())) is not None
    for bad in (lin(Other), lin(dtype=torch.float32)):
        assert ops.joint_linear(x, (lin(), bad)) is None
        assert ops.gated_linear(x, lin(), bad) is None
    assert ops.gated_linear(x, lin(), lin(bias=True)) is None
    assert ops.joint_linear(x[:500], (lin(), lin())) is None
    assert ops.joint_linear(x.cpu(), (lin(), lin())) is None


@pytest.mark.parametrize("m,n,k", [(512, 5120, 2048), (520, 4104, 2568),
                                   (700, 14336, 1000)])
def test_wgrad_pair(m, n, k):
    """Two layers of one input: as a product each, edges of tiles at both ends."""
    ext = ops._require_ext()
    x, dys = rand(m, k, 1), [rand(m, n, 2), rand(m, n, 3)]
    assert ext.linear_wgrad_pair_takes(*dys, x)
    for dy, got in zip(dys, ext.linear_wgrad_pair(*dys, x)):
        assert torch.equal(got, ext.linear_wgrad(dy, x))
    for other in (rand(m, n + 8, 4), rand(m + 1, n, 4)):
        assert not ext.linear_wgrad_pair_takes(dys[0], other, x)
        with pytest.raises(RuntimeError):
            ext.linear_wgrad_pair(dys[0], other, x)

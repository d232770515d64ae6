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


# ------------------------------------------------------------------ sampling


def noise(seed, row, v):
    """Gumbel noise of a row's entries, from the documented generator:
    splitmix64 keyed by (seed, row, entry), 24 bits, -log(-log u); -log u of
    the largest number is 2^-25."""
    import numpy as np
    with np.errstate(over="ignore"):
        u64 = np.uint64
        key = u64(seed) + u64(row) * u64(0x9e3779b97f4a7c15)
        z = key ^ (np.arange(v, dtype=u64) * u64(0xd1342543de82ef95)
                   + u64(0x2545f4914f6cdd1d))
        z = z + u64(0x9e3779b97f4a7c15)
        z = (z ^ (z >> u64(30))) * u64(0xbf58476d1ce4e5b9)
        z = (z ^ (z >> u64(27))) * u64(0x94d049bb133111eb)
        u = ((z >> u64(40)).astype("f8") + 1) / 16777216.0
        return torch.from_numpy(-np.log(np.where(u == 1.0, 2.0 ** -25,
                                                 -np.log(u))))


def kept(x, temp, k, p):
    """Mask of the kept entries, and of those within 1e-4 of the top-p
    boundary (32-bit mass)."""
    v = x.numel()
    s, order = x.sort(descending=True)
    low = s[k - 1] if 0 < k < v else torch.tensor(-float("inf"))
    sure, maybe = x >= low, x >= low
    if p < 1.0:
        mass = torch.softmax(s / temp, -1).cumsum(-1)
        for slack, which in ((1e-4, "maybe"), (-1e-4, "sure")):
            j = int((mass < p + slack).sum().clamp(max=v - 1))
            cut = x >= s[j]
            if which == "maybe":
                maybe = maybe & cut
            else:
                sure = sure & cut
    return sure, maybe


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,v", [(1, 9), (3, 1000), (2, 50257), (70, 4099),
                                 (2100, 300), (4, 151936)])
@pytest.mark.parametrize("temp,k,p", [(1.0, -1, 1.0), (0.7, 5, 1.0),
                                      (1.3, -1, 0.9), (0.7, 50, 0.6),
                                      (0.0, 3, 0.5), (1.0, 10 ** 6, 0.999)])
def test_sample_against_its_definition(n, v, dtype, temp, k, p):
    torch.manual_seed(3)
    x = (torch.randn(n, v, device=DEV) * 2.5).to(dtype)
    if v > 20:
        x[:, 7] = -float("inf")
    seed = 12345
    full = lambda t, ty: torch.full((n,), t, dtype=ty, device=DEV)
    args = (x, full(temp, torch.float32), full(k, torch.int32),
            full(p, torch.float32), seed)
    plain = (k <= 0 or k >= v) and p >= 1.0
    tok, lp = ops.sample(*args, no_filter=plain)
    again = ops.sample(*args, no_filter=plain)
    assert torch.equal(tok, again[0])
    if plain:      # the filtered path keeps everything: the same draw
        assert torch.equal(tok, ops.sample(*args, no_filter=False)[0])
    want = torch.log_softmax(x.double(), -1).gather(1, tok[:, None])[:, 0]
    assert (lp.double() - want).abs().max() <= 1e-5 * (1 + want.abs().max())
    for r in list(range(min(n, 3))) + [n - 1]:
        row = x[r].double().cpu()
        t = int(tok[r])
        assert 0 <= t < v
        if temp == 0.0:
            assert t == int(row.argmax())
            continue
        sure, maybe = kept(row, temp, k, p)
        assert maybe[t]
        z = row / temp + noise(seed, r, v)
        # 32-bit logarithms of 24-bit numbers: 1e-4 where the noise is large
        assert z[t] >= z[sure].max() - 1e-3


@pytest.mark.parametrize("b1,b2", [(0, 0), (1, 63), (5, 64), (64, 255),
                                   (255, 200), (256, 256), (2047, 1023)])
def test_sample_low_bins_of_later_digits(b1, b2):
    """fp32 rows whose k-th largest entry has small second and third digits
    (bin numbers like thread numbers and like the block size among them):
    what is kept is exactly the k largest."""
    n, v, k = 128, 3000, 40
    g = torch.Generator().manual_seed(b1 * 4096 + b2)

    def number(d0, d1, d2):           # its bits but the sign, as digits
        return ((d0 << 21) | (d1 << 10) | d2).to(torch.int32).view(
            torch.float32)

    rand = lambda lo, hi, m: torch.randint(lo, hi, (m,), generator=g)
    top = 0x7f << 2                   # exponent of numbers from 1 on
    rows = []
    for _ in range(n):
        m = v - 1
        x = number(torch.full((m,), top), rand(0, 2048, m), rand(0, 1024, m))
        # the larger ones share as many digits with the k-th as there are
        at = torch.tensor([top, b1, b2])
        kth = number(*at.view(3, 1))
        x = torch.where(x > kth, kth - x, x)     # not above: below zero
        up = number(torch.full((k - 1,), top),
                    torch.full((k - 1,), b1).minimum(torch.tensor(2047)),
                    rand(b2, 1024, k - 1))
        x = torch.cat([up, kth, x])
        rows.append(x[torch.randperm(v, generator=g)])
    x = torch.stack(rows)
    full = lambda t, ty: torch.full((n,), t, dtype=ty, device=DEV)
    temp, seed = 0.7, 77
    tok, _ = ops.sample(x.to(DEV), full(temp, torch.float32),
                        full(k, torch.int32), full(1.0, torch.float32), seed,
                        no_filter=False)
    for r in range(n):
        row = x[r].double()
        sure, _ = kept(row, temp, k, 1.0)
        t = int(tok[r])
        assert sure[t]
        z = row / temp + noise(seed, r, v)
        assert z[t] >= z[sure].max() - 1e-3


@pytest.mark.parametrize("seed,at", [(4116, 1462), (5128, 2925)])
@pytest.mark.parametrize("filtered", [False, True])
def test_sample_largest_random_number(seed, at, filtered):
    """An entry whose 24 random bits are all ones has the largest noise there
    is, but finite noise: it does not win against any logit."""
    v = 4096
    assert noise(seed, 0, v).argmax() == at
    x = torch.zeros(1, v, device=DEV)
    x[0, at] = -40.0
    full = lambda t, ty: torch.full((1,), t, dtype=ty, device=DEV)
    tok, _ = ops.sample(x, full(1.0, torch.float32), full(-1, torch.int32),
                        full(1.0, torch.float32), seed,
                        no_filter=not filtered)
    assert int(tok) == int((x[0].double().cpu() + noise(seed, 0, v)).argmax())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_sample_negative_temperature(dtype):
    """The draw at a negative temperature, with and without top-p: the
    filter's mass is exp(x / T) also there, from the largest logit down."""
    torch.manual_seed(7)
    n, v, temp, seed = 64, 3000, -0.8, 21
    x = torch.randn(n, v, device=DEV).to(dtype)
    full = lambda t, ty: torch.full((n,), t, dtype=ty, device=DEV)
    for p in (1.0, 0.3):
        tok, lp = ops.sample(x, full(temp, torch.float32),
                             full(-1, torch.int32), full(p, torch.float32),
                             seed, no_filter=p >= 1.0)
        want = torch.log_softmax(x.double(), -1).gather(1, tok[:, None])[:, 0]
        assert (lp.double() - want).abs().max() <= 1e-4
        for r in range(n):
            row = x[r].double().cpu()
            sure, maybe = kept(row, temp, -1, p)
            t = int(tok[r])
            assert maybe[t]
            z = row / temp + noise(seed, r, v)
            assert z[t] >= z[sure].max() - 1e-3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("v", [300, 9000])
@pytest.mark.parametrize("filtered", [False, True])
@pytest.mark.parametrize("temp", [0.0, 1.0])
def test_sample_nan_logits(v, dtype, filtered, temp):
    """A NaN anywhere in a row shows in its log-probability, also where a
    whole word of the row is NaN and no number was seen before it."""
    x = torch.randn(3, v, device=DEV).to(dtype)
    x[0, :8] = float("nan")
    x[1, v - 1] = float("nan")
    full = lambda t, ty: torch.full((3,), t, dtype=ty, device=DEV)
    tok, lp = ops.sample(x, full(temp, torch.float32), full(-1, torch.int32),
                         full(0.9 if filtered else 1.0, torch.float32), 3,
                         no_filter=not filtered)
    assert lp.isnan().tolist() == [True, True, False]
    assert ((tok >= 0) & (tok < v)).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("p", [0.0, 1e-30, 1e-6])
def test_sample_smallest_top_p(p, dtype):
    """top-p always keeps the largest logit."""
    torch.manual_seed(2)
    x = torch.randn(5, 5000, device=DEV).to(dtype)
    x[:, 100] = 9.0
    x[2] -= 100.0                      # all below zero
    full = lambda t, ty: torch.full((5,), t, dtype=ty, device=DEV)
    tok, _ = ops.sample(x, full(1.0, torch.float32), full(-1, torch.int32),
                        full(p, torch.float32), 5, no_filter=False)
    assert tok.tolist() == [100] * 5


@pytest.mark.parametrize("temp,p", [(0.01, 0.99), (0.01, 0.999), (0.003, 0.9)])
def test_sample_top_p_far_from_zero(temp, p):
    """Large logits at a low temperature (x / T in the thousands): the filter
    still ends where the mass reaches p."""
    torch.manual_seed(11)
    n, v = 4096, 1000
    x = 30 + torch.randn(n, v, device=DEV) * temp
    full = lambda t, ty: torch.full((n,), t, dtype=ty, device=DEV)
    tok, _ = ops.sample(x, full(temp, torch.float32), full(-1, torch.int32),
                        full(p, torch.float32), 9, no_filter=False)
    s, order = (x.double() / temp).sort(-1, descending=True)
    mass = torch.softmax(s, -1)
    above = torch.empty_like(mass).scatter_(1, order, mass.cumsum(-1) - mass)
    # 32-bit 1 / T moves every x / T here by less than 1e-4 of itself times
    # the logits' spread, and so the mass above an entry by less than 1e-4
    assert (above.gather(1, tok[:, None]) < p + 1e-4).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,v", [(2, 64), (2, 50257), (1030, 500)])
def test_entropy_with_banned_tokens(n, v, dtype):
    """-inf logits take no part in the entropy."""
    torch.manual_seed(6)
    x = (torch.randn(n, v, device=DEV) * 2).to(dtype)
    x[:, : v // 3] = -float("inf")
    x[0, v // 2] = -float("inf")
    lab = torch.full((n,), v - 1, device=DEV)
    p = torch.softmax(x.double(), -1)
    want = -torch.special.xlogy(p, p).sum(-1)
    _, ent = ops.gather_logprobs(x, lab, want_entropy=True)
    assert (ent.double() - want).abs().max() <= 2e-5 * (1 + want.max())


@pytest.mark.parametrize("n,v,skip", [(3, 50257, 0), (5, 333, 3), (4, 4096, 1),
                                      (2, 5, 0), (6, 11, 1), (3, 64, 8)])
def test_logprob_gradients_of_unaligned_rows(n, v, skip):
    """Rows that do not start at 16-byte addresses, and logits that do not
    start where their gradient does."""
    torch.manual_seed(2)
    flat = torch.randn(skip + n * v, device=DEV).bfloat16()
    x = flat[skip:].view(n, v)
    lab = torch.arange(n, device=DEV) * 7 % v
    dlp = torch.randn(n, device=DEV)
    g = x.detach().requires_grad_()
    ops.gather_logprobs_train(g, lab).backward(dlp)
    dx = -dlp[:, None].double() * torch.softmax(x.double(), -1)
    dx.scatter_add_(1, lab[:, None], dlp[:, None].double())
    # rounded once to bf16, the label's entry twice
    tol = 2 ** -7 * dx.abs() + 1e-6
    tol.scatter_add_(1, lab[:, None], 2 ** -8 * dlp[:, None].abs().double())
    assert ((g.grad.double() - dx).abs() <= tol).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("v", [4095, 4096, 4097, 8191, 8192, 8193])
@pytest.mark.parametrize("temp,k,p", [(1.0, -1, 1.0), (0.7, 15, 0.9),
                                      (0.7, 17, 1.0), (0.0, 3, 0.5)])
def test_sample_short_rows(v, dtype, temp, k, p):
    """Rows on both sides of the lengths up to which one block takes a row;
    k on both sides of the maxima that such a block keeps."""
    test_sample_against_its_definition(5, v, dtype, temp, k, p)


@pytest.mark.parametrize("n,v", [(5, 2047), (5, 2049), (3, 16384), (3, 16385),
                                 (2, 32768), (2, 32769), (191, 17000),
                                 (192, 17000), (257, 2049), (257, 20481),
                                 (192, 65537)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("temp,k,p", [(1.0, -1, 1.0), (0.7, 64, 0.9),
                                      (0.7, 65, 1.0)])
def test_sample_one_launch(n, v, dtype, temp, k, p):
    """Both sides of the sizes up to which one block takes a row, and of those
    from which it has 1024 threads; k on both sides of the maxima of such a
    block.  Many rows: the first and the last are enough."""
    torch.manual_seed(8)
    x = (torch.randn(n, v, device=DEV) * 3).to(dtype)
    full = lambda t, ty: torch.full((n,), t, dtype=ty, device=DEV)
    seed = 31
    tok, lp = ops.sample(x, full(temp, torch.float32), full(k, torch.int32),
                         full(p, torch.float32), seed, no_filter=k < 0)
    want = torch.log_softmax(x.double(), -1).gather(1, tok[:, None])[:, 0]
    assert (lp.double() - want).abs().max() <= 1e-5 * (1 + want.abs().max())
    for r in {0, 1, n - 1}:
        row = x[r].double().cpu()
        sure, maybe = kept(row, temp, k, p)
        t = int(tok[r])
        assert maybe[t]
        z = row / temp + noise(seed, r, v)
        # (as above)
        assert z[t] >= z[sure].max() - 1e-3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("k,p", [(50, 1.0), (-1, 0.9), (50, 0.5), (900, 1.0),
                                 (1500, 0.99)])
@pytest.mark.parametrize("what", ["random", "cluster", "ties", "peak",
                                  "about_full"])
def test_sample_candidate_lists(what, k, p, dtype):
    """Rows in pieces whose candidates are few (a list), many, more than a list
    holds though the lanes' groups show few (neighbours), all alike, or about
    as many as a list holds; an odd row length."""
    torch.manual_seed(11)
    n, v, temp, seed = 3, 70001, 0.8, 77
    x = torch.randn(n, v, device=DEV)
    if what == "cluster":
        x[:, 5000:7000] = 8 + torch.rand(n, 2000, device=DEV)
    elif what == "ties":
        x[:] = 1.0
    elif what == "peak":
        x[:, 12345] = 40.0
    elif what == "about_full":
        for r in range(n):
            at = torch.randperm(v, device=DEV)[:1010 + 14 * r]
            x[r, at] = 9 + torch.rand(len(at), device=DEV)
    x = x.to(dtype)
    full = lambda t, ty: torch.full((n,), t, dtype=ty, device=DEV)
    tok, lp = ops.sample(x, full(temp, torch.float32), full(k, torch.int32),
                         full(p, torch.float32), seed, no_filter=False)
    want = torch.log_softmax(x.double(), -1).gather(1, tok[:, None])[:, 0]
    assert (lp.double() - want).abs().max() <= 1e-5 * (1 + want.abs().max())
    for r in range(n):
        row = x[r].double().cpu()
        sure, maybe = kept(row, temp, k, p)
        t = int(tok[r])
        assert maybe[t]
        z = row / temp + noise(seed, r, v)
        # 32-bit logarithms of 24-bit numbers: 1e-4 where the noise is large
        assert z[t] >= z[sure].max() - 1e-3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [9, 40])
def test_sample_rows_of_every_kind(n, dtype):
    """One call whose rows go every way that a long row can: the largest logit,
    no filter, few candidates, many, neighbours that a list does not hold
    (from one piece, or from several), all alike, NaN; an odd row length."""
    torch.manual_seed(15)
    v, seed = 70001, 123
    x = torch.randn(n, v, device=DEV) * 2
    temp, k, p = [], [], []
    kinds = [("greedy", 0.0, 40, 0.9), ("plain", 0.9, -1, 1.0),
             ("few", 0.7, 50, 0.9), ("flat", 1.3, -1, 0.95),
             ("next", 0.8, -1, 0.9), ("wide", 0.8, 90, 0.97),
             ("alike", 1.0, 20, 1.0), ("greedy", 0.0, -1, 1.0),
             ("nan", 0.8, 30, 0.9)]
    what = [kinds[(r * 7) % len(kinds)] for r in range(n)]
    for r, (kind, t, kk, pp) in enumerate(what):
        temp.append(t), k.append(kk), p.append(pp)
        if kind == "flat":
            x[r] = torch.rand(v, device=DEV)
        elif kind == "next":
            x[r, 3000:4500] = 12 + torch.rand(1500, device=DEV)
        elif kind == "wide":            # several pieces list, the last do not fit
            x[r, 1000:20000:9] = 12 + torch.rand(2112, device=DEV)
        elif kind == "alike":
            x[r] = 1.0
        elif kind == "nan":
            x[r, 777] = float("nan")
    x = x.to(dtype)
    tok, lp = ops.sample(x, torch.tensor(temp, device=DEV),
                         torch.tensor(k, dtype=torch.int32, device=DEV),
                         torch.tensor(p, device=DEV), seed, no_filter=False)
    for r, (kind, t, kk, pp) in enumerate(what):
        row, got = x[r].double().cpu(), int(tok[r])
        if kind == "nan":
            assert 0 <= got < v and torch.isnan(lp[r])
            continue
        want = torch.log_softmax(row, -1)[got]
        assert abs(float(lp[r]) - want) <= 1e-5 * (1 + abs(want)), r
        if t == 0.0:
            assert row[got] == row.max(), r
            continue
        sure, maybe = kept(row, t, kk, pp)
        assert maybe[got], (r, kind)
        z = row / t + noise(seed, r, v)
        # (as above)
        assert z[got] >= z[sure].max() - 1e-3, (r, kind)


@pytest.mark.parametrize("n,v", [(5, 16383), (3, 16384), (1100, 16385),
                                 (896, 65536), (897, 65536), (2048, 65536),
                                 (2049, 65536)])
def test_logprobs_on_both_sides_of_the_caches(n, v):
    """Rows that the gradient's blocks of 256 and of 1024 threads take, and
    logits that the cache behind the L2s just holds, alone or with their
    gradient, and just does not."""
    x = torch.randn(n, v, generator=torch.Generator(DEV).manual_seed(7),
                    device=DEV).bfloat16().requires_grad_()
    lab = torch.arange(n, device=DEV) * 7 % v
    dlp = torch.randn(n, device=DEV)
    lp = ops.gather_logprobs_train(x, lab)
    lp.backward(dlp)
    assert torch.equal(ops.gather_logprobs(x.detach(), lab), lp)
    for a in range(0, n, 256):
        b = slice(a, min(a + 256, n))
        want = torch.log_softmax(x.detach()[b].double(), -1)
        at = want.gather(1, lab[b, None])
        assert (lp[b].double() - at[:, 0]).abs().max() < 1e-5 * at.abs().max()
        g = dlp[b, None].double()
        dx = -g * want.exp()
        dx.scatter_add_(1, lab[b, None], g)
        # rounded once to bf16, the label's entry twice
        tol = 2 ** -7 * dx.abs() + 1e-6
        tol.scatter_add_(1, lab[b, None], 2 ** -8 * g.abs())
        assert ((x.grad[b].double() - dx).abs() <= tol).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,v", [(64, 98305), (100, 33001), (128, 65537),
                                 (180, 40003), (256, 65539), (257, 66001),
                                 (700, 65540), (1030, 65537), (16, 128256)])
def test_sample_block_sizes(n, v, dtype):
    """Without a filter, over the numbers of rows at which blocks of 256, 512
    and 1024 threads take the pieces: the draw is the filtered path's, which
    has other pieces, entry by entry (both judge first words by approximate
    noise; the next test's other side does not).  Rows of few possible entries,
    of one, of large logits and of a temperature that is not positive among them."""
    torch.manual_seed(21)
    x = (torch.randn(n, v, device=DEV) * 3).to(dtype)
    x[1, 100:] = -float("inf")
    x[2, :] = -float("inf")
    x[2, v - 1] = -5.0
    x[3] *= 1000
    x[4, 300:] -= 40
    full = lambda t, ty: torch.full((n,), t, dtype=ty, device=DEV)
    temp = full(0.9, torch.float32)
    temp[5], temp[6], temp[7] = 0.0, -1.0, 1e-6
    args = (x, temp, full(-1, torch.int32), full(1.0, torch.float32), 77)
    tok, lp = ops.sample(*args, no_filter=True)
    other, _ = ops.sample(*args, no_filter=False)
    assert torch.equal(tok, other)
    assert int(tok[2]) == v - 1 and int(tok[1]) < 100
    want = torch.log_softmax(x.double(), -1).gather(1, tok[:, None])[:, 0]
    assert ((lp.double() - want).abs() <= 1e-5 * (1 + want.abs())).all()
    for r in (0, 1, 4, n - 1):
        z = x[r].double().cpu() / float(temp[r]) + noise(77, r, v)
        # 32-bit logarithms of 24-bit numbers: 1e-4 where the noise is large
        assert z[int(tok[r])] >= z.max() - 1e-3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,v", [(64, 98305), (128, 65537), (180, 40003),
                                 (256, 65539), (1030, 65537), (16, 128256),
                                 (300, 9000)])
def test_sample_draw_without_approximate_noise(n, v, dtype):
    """Without a filter the draw is that of a filter which keeps the entries that
    can win: that one has a threshold, and takes the exact noise of all of them.
    Half of the entries stand in the words that the blocks' waves read first."""
    m = 12
    g = torch.Generator().manual_seed(n)
    x = torch.full((n, v), -200.0)
    at = torch.stack([torch.cat([
        torch.randperm(4096, generator=g)[:m // 2],
        4096 + torch.randperm(v - 4096, generator=g)[:m // 2]])
        for _ in range(n)])
    x = x.scatter_(1, at, torch.randn(n, m, generator=g)).to(dtype).to(DEV)
    full = lambda t, ty: torch.full((n,), t, dtype=ty, device=DEV)
    for seed in range(8):
        temp, p = full(0.9, torch.float32), full(1.0, torch.float32)
        tok, lp = ops.sample(x, temp, full(-1, torch.int32), p, seed,
                             no_filter=True)
        other, olp = ops.sample(x, temp, full(m, torch.int32), p, seed,
                                no_filter=False)
        assert torch.equal(tok, other), seed
        assert (x.gather(1, tok[:, None]) > -100).all()
        assert (lp - olp).abs().max() <= 1e-5


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,v,ks", [(300, 40001, (1, 16, 17, 64, 65)),
                                    (64, 131073, (1, 64, 65, 256, 257)),
                                    (52, 200003, (79, 80, 303, 320, 321)),
                                    (16, 262147, (200, 256, 257, 1000, 1024))])
def test_sample_cut_of_few_and_many_pieces(n, v, ks, dtype):
    """The cut below the k-th largest of the pieces' maxima: 4, 16, 20 and 64
    pieces, 16 maxima each, and a k on both sides of where waves' maxima, all of
    them and no cut take turns.  Rows whose k-th largest is positive, negative,
    tied, zero, infinite."""
    torch.manual_seed(23)
    x = torch.randn(n, v, device=DEV) * 2
    x[1::5] -= 300
    x[2::5] = x[2::5].round()
    # (zeros of one sign: the kernels' order has -0 below +0, the oracle's does not,
    # and a row of ties of both keeps the positive ones only)
    x[3::5] = x[3::5].clamp(max=0.0)
    x[4::5, 11:] = -float("inf")
    x = x.to(dtype)
    k = torch.tensor([ks[(r // 5) % len(ks)] for r in range(n)],
                     dtype=torch.int32, device=DEV)
    p = torch.tensor([1.0 if r % 2 else 0.95 for r in range(n)], device=DEV)
    temp = torch.full((n,), 0.8, device=DEV)
    tok, lp = ops.sample(x, temp, k, p, 31, no_filter=False)
    want = torch.log_softmax(x.double(), -1).gather(1, tok[:, None])[:, 0]
    assert ((lp.double() - want).abs() <= 1e-5 * (1 + want.abs())).all()
    for r in range(min(n, 25)):
        row, got = x[r].double().cpu(), int(tok[r])
        sure, maybe = kept(row, float(temp[r]), int(k[r]), float(p[r]))
        assert maybe[got], r
        z = row / float(temp[r]) + noise(31, r, v)
        # 32-bit logarithms of 24-bit numbers: 1e-4 where the noise is large; at
        # 300 / T a multiply-add of 32 bits is off by another 3e-5
        assert z[got] >= z[sure].max() - 1e-3, r


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n,v", [(64, 9000), (128, 40001), (256, 65539),
                                 (100, 98305)])
def test_sample_ties_of_rounded_sums(n, v, dtype):
    """At a temperature of 1e-6 logits of 11 are 1.1e7, where 32-bit numbers are
    whole: of equal logits those whose noise rounds alike tie, and the first of them
    wins, whichever wave is first.  Without a filter and with one that keeps all."""
    m = 200
    g = torch.Generator().manual_seed(n)
    x = torch.randn(n, v, generator=g)
    at = torch.stack([torch.randperm(v, generator=g)[:m].sort()[0]
                      for _ in range(n)])
    x.scatter_(1, at, 11.0)
    full = lambda t, ty: torch.full((n,), t, dtype=ty, device=DEV)
    temp = full(1e-6, torch.float32)
    by = torch.tensor(1.0) / torch.tensor(1e-6)
    checked = 0
    for seed in (5, 1 << 40):
        args = (x.to(dtype).to(DEV), temp, full(-1, torch.int32),
                full(1.0, torch.float32), seed)
        got = [ops.sample(*args, no_filter=f)[0].cpu() for f in (True, False)]
        for r in range(n):
            # 32-bit logarithms of 24-bit numbers: 1e-4 where the noise is large;
            # rows that this could decide are passed over
            z = 11.0 * by.double() + noise(seed, r, v)[at[r]]
            lo, hi = ((z + d).float() for d in (-2e-4, 2e-4))
            if not torch.equal(lo, hi):
                sure = hi < lo.max()
                if not torch.equal(lo[~sure], hi[~sure]):
                    continue
            checked += 1
            first = int(at[r][(lo == lo.max()).nonzero()[0, 0]])
            assert [int(t[r]) for t in got] == [first, first], (seed, r)
    assert checked > n

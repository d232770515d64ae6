"""Matrix-core attention of the dense decoders at the edges of its tiles:
32-row units, 64-row and 64-key tiles, head groups that do not fill a block,
rows behind cached keys.  Reference: float64 softmax attention of the same
bf16 inputs."""
import pytest
import torch

import polyrl_amd.ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda"

LENS = {
    "one": [1],
    "edges": [1, 31, 32, 33, 63, 64, 65, 127, 128, 129],
    "ragged": [200, 7, 321, 64],
    "many": [3] * 70 + [65],            # more sequences than a scan step
    "shares": [65] * 20 + [33] * 130,   # dK/dV blocks of 2 to 4 heads of 7
}


def cu_of(lens):
    return torch.tensor([0] + lens).cumsum(0).int()


def heads(x, hq):
    return x.repeat_interleave(hq // x.shape[1], 1)


def attend(q, k, v, hist, causal, scale):
    """(rows, heads, d) and the log-sum-exp (rows, heads), float64."""
    s = torch.einsum("qhd,khd->hqk", q, k) * scale
    if causal:
        i = torch.arange(q.shape[0], device=q.device)[:, None] + hist
        s = s.masked_fill(torch.arange(k.shape[0], device=q.device)[None] > i,
                          -float("inf"))
    return torch.einsum("hqk,khd->qhd", torch.softmax(s, -1), v), \
        torch.logsumexp(s, -1).t()


@pytest.mark.parametrize("table", [False, True])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("hist", [0, 77])
@pytest.mark.parametrize("name,hq,hk,d", [
    ("edges", 8, 2, 128), ("edges", 7, 1, 64), ("one", 3, 3, 128),
    ("ragged", 12, 2, 128), ("ragged", 4, 4, 64), ("many", 8, 1, 64),
    ("ragged", 10, 2, 64)])
def test_forward(name, hq, hk, d, hist, causal, table):
    torch.manual_seed(5)
    lens = LENS[name]
    klens = [n + hist for n in lens]
    cu_q, cu_k = cu_of(lens), cu_of(klens)
    # rows of a fused projection: the token stride is not heads * size
    q = torch.randn(sum(lens), hq * d + 16, device=DEV).bfloat16()[
        :, :hq * d].unflatten(1, (hq, d))
    k = torch.randn(sum(klens), hk, d, device=DEV).bfloat16()
    v = torch.randn(sum(klens), hk, d, device=DEV).bfloat16()
    scale = d ** -0.5
    if table:
        out = torch.empty(q.shape, dtype=q.dtype, device=DEV)
        lse = torch.empty(q.shape[:2], device=DEV)
        t = ops.build_varlen_tiles(cu_q, DEV)
        ops._require_ext().varlen_prefill_attention(
            out, q, k, v, cu_q.to(DEV), cu_k.to(DEV), t[0], t[1], scale,
            causal, lse)
    else:
        out, lse = ops.varlen_prefill_attention(
            q, k, v, cu_q.to(DEV), cu_k.to(DEV), scale, causal,
            return_lse=True)
    for i, n in enumerate(lens):
        a, b = slice(cu_q[i], cu_q[i + 1]), slice(cu_k[i], cu_k[i + 1])
        kk, vv = heads(k[b].double(), hq), heads(v[b].double(), hq)
        want, wl = attend(q[a].double(), kk, vv, hist, causal, scale)
        mass, _ = attend(q[a].double(), kk, vv.abs(), hist, causal, scale)
        # a weight and the result are each rounded once to bf16 (2^-9, and as
        # much again for the 32-bit sums and exponentials)
        bound = 2 ** -8 * (mass + want.abs())
        assert ((out[a].double() - want).abs() <= bound).all(), (name, n)
        # 32-bit scores (|s| < 64) and sums
        assert (lse[a].double() - wl).abs().max() < 1e-4


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("name,hq,hk,d", [
    ("edges", 8, 2, 128), ("edges", 7, 1, 64), ("one", 3, 3, 128),
    ("ragged", 12, 2, 128), ("ragged", 4, 4, 64), ("many", 8, 1, 64),
    ("ragged", 10, 2, 64), ("shares", 14, 2, 128), ("shares", 4, 2, 64)])
def test_backward(name, hq, hk, d, causal):
    """Gradients of every sequence against float64 autograd.  With P and dS
    rounded once to bf16, sums in 32 bits and the result rounded once, an
    entry is off by at most 2^-8 of the sum of its terms' magnitudes, plus
    what the bf16 output in delta = rowsum(dO * O) adds."""
    torch.manual_seed(6)
    lens, scale = LENS[name], d ** -0.5
    cu = cu_of(lens)
    n = sum(lens)
    q, k, v = (torch.randn(n, h, d, device=DEV).bfloat16().requires_grad_()
               for h in (hq, hk, hk))
    dout = torch.randn(n, hq, d, device=DEV).bfloat16()
    out = ops.flash_attn_varlen(q, k, v, cu.to(DEV), scale, causal)
    got = torch.autograd.grad(out, (q, k, v), dout)
    again = torch.autograd.grad(
        ops.flash_attn_varlen(q, k, v, cu.to(DEV), scale, causal), (q, k, v),
        dout)
    for a, b in zip(got, again):
        assert torch.equal(a, b)            # no atomics: the same bits
    for i in range(len(lens)):
        a = slice(cu[i], cu[i + 1])
        x = [t.detach()[a].double() for t in (q, k, v)]
        kk, vv, do = heads(x[1], hq), heads(x[2], hq), dout[a].double()
        s = torch.einsum("qhd,khd->hqk", x[0], kk) * scale
        if causal:
            r = torch.arange(lens[i], device=DEV)
            s = s.masked_fill(r[None] > r[:, None], -float("inf"))
        p = torch.softmax(s, -1)
        dp = torch.einsum("qhd,khd->hqk", do, vv)
        o = torch.einsum("hqk,khd->qhd", p, vv)
        delta = (do * o).sum(-1).t()[..., None]
        ds = p * (dp - delta)
        # the magnitudes: |dS| plus the share of delta that rounding O moves
        big = p * ((dp - delta).abs()
                   + (do * o).abs().sum(-1).t()[..., None])
        group = lambda t: t.unflatten(1, (hk, hq // hk)).sum(2)
        pair = lambda w, t: torch.einsum("hqk,qhd->khd", w, t)
        want = (torch.einsum("hqk,khd->qhd", ds, kk) * scale,
                group(pair(ds, x[0])) * scale, group(pair(p, do)))
        size = (torch.einsum("hqk,khd->qhd", big, kk.abs()) * scale,
                group(pair(big, x[0].abs())) * scale,
                group(pair(p, do.abs())))
        for name_, g, w, m in zip(("dq", "dk", "dv"), got, want, size):
            off = (g[a].double() - w).abs() - 2 ** -8 * (m + w.abs())
            assert off.max() <= 0, (name_, lens[i], off.max())


@pytest.mark.parametrize("page_size,wide", [(16, False), (16, True), (1, False),
                                            (7, True)])
@pytest.mark.parametrize("hq,hk,d", [(8, 8, 128), (7, 1, 128), (12, 4, 64),
                                     (16, 2, 64), (28, 4, 128), (5, 1, 64),
                                     (6, 2, 128)])
def test_decode(hq, hk, d, page_size, wide):
    """Paged decode at the edges of its 32-key rounds and 128-key stretches;
    ``wide``: a page table far wider than the contexts (a captured graph's),
    which divides them further.  The weights are 32-bit ones, so an entry is
    off by its rounding to bf16 and 2^-14 of its terms."""
    torch.manual_seed(9)
    lens = [1, 31, 32, 33, 127, 128, 129, 300, 1025, 2]
    need = [-(-n // page_size) for n in lens]
    pages = torch.randperm(sum(need), device=DEV).int()
    table = torch.zeros(len(lens), max(need) * (4 if wide else 1),
                        dtype=torch.int32, device=DEV)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = pages[at:at + n]
        at += n
    k, v = (torch.randn(sum(need), page_size, hk, d, device=DEV).bfloat16()
            for _ in range(2))
    q = torch.randn(len(lens), (hq + 2) * d, device=DEV).bfloat16()[
        :, :hq * d].unflatten(1, (hq, d))
    out = ops.paged_attention_decode(
        q, k, v, table, torch.tensor(lens, dtype=torch.int32, device=DEV),
        d ** -0.5)
    for i, n in enumerate(lens):
        p = table[i, :need[i]].long()
        kk = heads(k[p].view(-1, hk, d)[:n].double(), hq)
        vv = heads(v[p].view(-1, hk, d)[:n].double(), hq)
        want, _ = attend(q[i:i + 1].double(), kk, vv, n - 1, True, d ** -0.5)
        mass, _ = attend(q[i:i + 1].double(), kk, vv.abs(), n - 1, True,
                         d ** -0.5)
        bound = 2 ** -8 * want.abs() + 2 ** -14 * mass
        assert ((out[i:i + 1].double() - want).abs() <= bound).all(), n


@pytest.mark.parametrize("hq,hk,d", [(8, 2, 64), (7, 1, 64), (4, 4, 128),
                                     (12, 2, 128)])
@pytest.mark.parametrize("window,keep,chunk", [(1 << 20, 0, 0), (100, 0, 0),
                                               (64, 4, 0), (70, 130, 0),
                                               (1 << 20, 0, 96), (1, 0, 0)])
@pytest.mark.parametrize("extras", [False, True])
def test_window_prompts(hq, hk, d, window, keep, chunk, extras):
    """Paged window attention of prompt portions (some behind cached rows):
    tile edges, windows shorter and longer than a tile, kept first tokens
    before the window, chunks; sink, gate, row temperature and an output
    column slice together."""
    torch.manual_seed(8)
    lens, hist = [1, 31, 33, 64, 65, 200, 7], [0, 5, 0, 300, 63, 0, 129]
    page = 16
    need = [-(-(n + m) // page) for n, m in zip(lens, hist)]
    pages = torch.randperm(sum(need), device=DEV).int()
    table = torch.zeros(len(lens), max(need), dtype=torch.int32, device=DEV)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = pages[at:at + n]
        at += n
    rows = torch.randn(sum(need), page, 2 * hk * d, device=DEV).bfloat16()
    n = sum(lens)
    q = torch.randn(n, hq * d, device=DEV).bfloat16()
    i32 = dict(dtype=torch.int32, device=DEV)
    seq = torch.repeat_interleave(torch.arange(len(lens), **i32),
                                  torch.tensor(lens, device=DEV))
    pos = torch.cat([torch.arange(m, m + x, **i32)
                     for x, m in zip(lens, hist)])
    sink = torch.randn(hq, device=DEV) * 3 if extras else None
    gate = torch.randn(n, hq, device=DEV).bfloat16() if extras else None
    wide = torch.zeros(n, hq * d + 24, device=DEV).bfloat16()
    out = wide[:, 8:8 + hq * d] if extras else None
    coef, scale, mult = (0.1, d ** -0.5, 0.5) if extras else \
        (0.0, d ** -0.5, 1.0)
    got = ops.seq.gqa_window_attention(
        q, rows, table, seq, pos, hq, hk, d, d, window, keep, None, None,
        gate, scale, torch.bfloat16, tiles=ops.seq.attention_tiles(lens, DEV),
        sink=sink, q_temp_coef=coef, q_temp_every=16, chunk=chunk, out=out,
        out_scale=mult)
    a = 0
    for i, (x, m) in enumerate(zip(lens, hist)):
        kv = rows[table[i, :need[i]].long()].view(-1, 2, hk, d)[:x + m].double()
        k, v = heads(kv[:, 0], hq), heads(kv[:, 1], hq)
        r = pos[a:a + x].long()[:, None]
        j = torch.arange(x + m, device=DEV)[None]
        live = (r - j < window)
        if chunk:
            live = live & (j // chunk == r // chunk)
        live = (live | (j < keep)) & (j <= r)
        temp = 1 + coef * torch.log((r[:, 0].double() + 1).div(
            16, rounding_mode="floor") + 1)
        s = torch.einsum("qhd,khd->hqk", q[a:a + x].double().view(x, hq, d),
                         k) * scale * temp[None, :, None]
        s = s.masked_fill(~live, -float("inf"))
        if sink is not None:
            s = torch.cat([s, sink.double()[:, None, None].expand(
                -1, x, 1)], -1)
        p = torch.softmax(s, -1)[..., :x + m]
        want = torch.einsum("hqk,khd->qhd", p, v)
        mass = torch.einsum("hqk,khd->qhd", p, v.abs())
        f = mult * (torch.sigmoid(gate[a:a + x].double())[..., None]
                    if gate is not None else 1.0)
        bound = 2 ** -8 * (mass + want.abs()) * f
        off = (got[a:a + x].double().view(x, hq, d) - want * f).abs() - bound
        assert off.max() <= 0, (i, off.max())
        a += x
    if extras:                         # nothing written beside the slice
        assert (wide[:, :8] == 0).all() and (wide[:, 8 + hq * d:] == 0).all()


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("name,hq,hk,d", [("edges", 8, 2, 128),
                                          ("ragged", 7, 1, 64)])
def test_scale_zero(name, hq, hk, d, causal):
    """Scores of zero: the mean of the values a row sees, and no gradient for
    queries and keys."""
    torch.manual_seed(3)
    lens = LENS[name]
    cu, n = cu_of(lens), sum(lens)
    q, k, v = (torch.randn(n, h, d, device=DEV).bfloat16().requires_grad_()
               for h in (hq, hk, hk))
    out = ops.flash_attn_varlen(q, k, v, cu.to(DEV), 0.0, causal)
    same = ops.varlen_prefill_attention(q.detach(), k.detach(), v.detach(),
                                        cu.to(DEV), cu.to(DEV), 0.0, causal)
    assert torch.equal(out, same)
    dout = torch.randn(n, hq, d, device=DEV).bfloat16()
    dq, dk, dv = torch.autograd.grad(out, (q, k, v), dout)
    assert (dq == 0).all() and (dk == 0).all() and dv.isfinite().all()
    for i in range(len(lens)):
        a = slice(cu[i], cu[i + 1])
        x = [t.detach()[a].double() for t in (q, k, v)]
        kk, vv = heads(x[1], hq), heads(x[2], hq)
        want, _ = attend(x[0], kk, vv, 0, causal, 0.0)
        mass, _ = attend(x[0], kk, vv.abs(), 0, causal, 0.0)
        bound = 2 ** -8 * (mass + want.abs())
        assert ((out[a].double() - want).abs() <= bound).all(), lens[i]


@pytest.mark.parametrize("hq,hk,d", [(8, 2, 128), (7, 1, 64), (4, 4, 64)])
def test_infinite_value_of_the_last_key(hq, hk, d):
    """An infinite entry of a sequence's last value row gives an infinite
    entry where that row is seen: what stands in for rows past the end takes
    no part."""
    torch.manual_seed(4)
    lens, page, scale = [1, 33, 200], 16, d ** -0.5
    cu, n = cu_of(lens).to(DEV), sum(lens)
    q = torch.randn(n, hq, d, device=DEV).bfloat16()
    k, v = (torch.randn(n, hk, d, device=DEV).bfloat16() for _ in range(2))
    ends = (cu[1:] - 1).long()
    v[ends, :, 5] = float("inf")
    need = [-(-x // page) for x in lens]
    table = torch.zeros(3, max(need), dtype=torch.int32, device=DEV)
    rows = torch.zeros(sum(need) * page, 2, hk, d, device=DEV).bfloat16()
    at = 0
    for i, x in enumerate(need):
        table[i, :x] = torch.arange(at, at + x, device=DEV)
        a = slice(int(cu[i]), int(cu[i + 1]))
        rows[at * page:at * page + lens[i], 0] = k[a]
        rows[at * page:at * page + lens[i], 1] = v[a]
        at += x
    i32 = dict(dtype=torch.int32, device=DEV)
    pos = torch.cat([torch.arange(x, **i32) for x in lens])
    seq = torch.repeat_interleave(torch.arange(3, **i32),
                                  torch.tensor(lens, device=DEV))
    paged = rows.view(-1, page, 2, hk, d)
    got = {
        "prompt": ops.varlen_prefill_attention(q, k, v, cu, cu, scale,
                                               True)[ends],
        "window": ops.seq.gqa_window_attention(
            q.flatten(1), paged.flatten(2), table, seq, pos, hq, hk, d, d,
            1 << 20, 0, None, None, None, scale, torch.bfloat16,
            tiles=ops.seq.attention_tiles(lens, DEV)).view(n, hq, d)[ends],
        "decode": ops.paged_attention_decode(
            q[ends], paged[:, :, 0].contiguous(), paged[:, :, 1].contiguous(),
            table, torch.tensor(lens, **i32), scale),
    }
    other = [j for j in range(d) if j != 5]
    for name, out in got.items():
        assert (out[:, :, 5] == float("inf")).all(), name
        assert out[:, :, other].isfinite().all(), name


@pytest.mark.parametrize("hq,hk,d", [(8, 2, 128), (7, 1, 64), (4, 4, 64)])
def test_infinite_gradient_of_the_last_row(hq, hk, d):
    """An infinite entry of the gradient of a sequence's last output row gives
    infinite entries of dV, which all of its keys share in, and no NaN: what
    stands in for rows past the end takes no part."""
    torch.manual_seed(4)
    lens = [1, 33, 200]
    cu = cu_of(lens).to(DEV)
    q, k, v = (torch.randn(sum(lens), h, d, device=DEV).bfloat16()
               .requires_grad_() for h in (hq, hk, hk))
    dout = torch.randn(sum(lens), hq, d, device=DEV).bfloat16()
    dout[(cu[1:] - 1).long(), :, 5] = float("inf")
    out = ops.flash_attn_varlen(q, k, v, cu, d ** -0.5, True)
    dv = torch.autograd.grad(out, (q, k, v), dout)[2]
    assert (dv[:, :, 5] == float("inf")).all()
    assert dv[:, :, [j for j in range(d) if j != 5]].isfinite().all()


@pytest.mark.parametrize("hq,hk,d", [(8, 2, 128), (7, 1, 64)])
@pytest.mark.parametrize("sign", [1, -1])
def test_very_large_scores(hq, hk, d, sign):
    """Scores far beyond 2^31, where an exponent is larger than the range of
    the exponential even in its rounding: each row gets the value of its
    largest score."""
    torch.manual_seed(4)
    lens = [1, 33, 200]
    cu = cu_of(lens)
    q, k, v = (torch.randn(sum(lens), h, d, device=DEV).bfloat16()
               for h in (hq, hk, hk))
    q = q * 2.0 ** 40
    got = ops.varlen_prefill_attention(q, k, v, cu.to(DEV), cu.to(DEV),
                                       sign * d ** -0.5, True)
    for i in range(len(lens)):
        a = slice(cu[i], cu[i + 1])
        want, _ = attend(q[a].double(), heads(k[a].double(), hq),
                         heads(v[a].double(), hq), 0, True, sign * d ** -0.5)
        assert torch.equal(got[a].double(), want.bfloat16().double())


@pytest.mark.parametrize("d", [64, 128])
def test_decode_weights(d):
    """Weights are held in 32 bits: the difference of two almost equal ones
    (values +1 and -1, beside a larger weight with the value 0) is exact to a
    bf16 rounding and a few 2^-24, where weights of 16 or 17 bits would be off
    by 2^-20."""
    hq, n, scale = 8, 64, 0.125
    q = torch.zeros(n, hq, d)
    q[:, :, 0] = 4 + 12 * torch.rand(
        n, hq, generator=torch.Generator().manual_seed(1))
    q[:, :, 1] = 2.0 ** -5
    q = q.to(DEV).bfloat16()
    k = torch.zeros(1, 16, 1, d, device=DEV).bfloat16()
    v = torch.zeros(1, 16, 1, d, device=DEV).bfloat16()
    k[0, 0, 0, 0], k[0, 1:3, 0, 0], k[0, 2, 0, 1] = 1.0, 0.75, 2.0 ** -5
    v[0, 1], v[0, 2] = 1.0, -1.0
    out = ops.paged_attention_decode(
        q, k, v, torch.zeros(n, 1, dtype=torch.int32, device=DEV),
        torch.full((n,), 3, dtype=torch.int32, device=DEV), scale)
    p = torch.softmax(torch.einsum("nhd,kd->nhk", q.double(),
                                   k[0, :3, 0].double()) * scale, -1)
    want = (p[..., 1] - p[..., 2])[..., None]
    # a score, its exponential and the sums are each rounded to 24 bits
    bound = 2 ** -8 * want.abs() + 2.0 ** -22
    assert ((out.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("rows,heads_,most", [(11, 3, 64), (11, 3, 65),
                                              (11, 3, 512), (11, 3, 513),
                                              (255, 8, 700), (256, 8, 700),
                                              (128, 16, 3000)])
def test_decode_one_head_a_group(rows, heads_, most, d):
    """Groups of one head on both sides of the sizes at which the vector kernel
    takes them: few rows divided among blocks, many rows undivided."""
    torch.manual_seed(5)
    page = 1 if most % 16 else 16
    lens = ([most, 1, 2, 7, 8, 9, 16, 17, 31, 33, 64]
            + [1 + 37 * i % 90 for i in range(rows)])[:rows]
    need = [-(-n // page) for n in lens]
    table = torch.zeros(rows, max(need), dtype=torch.int32, device=DEV)
    pages = torch.randperm(sum(need), device=DEV).int()
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = pages[at:at + n]
        at += n
    k, v = (torch.randn(sum(need), page, heads_, d, device=DEV).bfloat16()
            for _ in range(2))
    q = torch.randn(rows, heads_, d, device=DEV).bfloat16()
    out = ops.paged_attention_decode(
        q, k, v, table, torch.tensor(lens, dtype=torch.int32, device=DEV),
        d ** -0.5)
    for i in list(range(11)) + [rows - 1]:
        n = lens[i]
        p = table[i, :need[i]].long()
        kk = k[p].view(-1, heads_, d)[:n].double()
        vv = v[p].view(-1, heads_, d)[:n].double()
        want, _ = attend(q[i:i + 1].double(), kk, vv, n - 1, True, d ** -0.5)
        mass, _ = attend(q[i:i + 1].double(), kk, vv.abs(), n - 1, True,
                         d ** -0.5)
        bound = 2 ** -8 * want.abs() + 2 ** -14 * mass
        assert ((out[i:i + 1].double() - want).abs() <= bound).all(), (i, n)


@pytest.mark.parametrize("nseq", [1, 63, 64, 65])
@pytest.mark.parametrize("d", [64, 128])
def test_every_tile_once(nseq, d):
    """Blocks take row tiles by the length of their walk, up to 64 sequences:
    with empty sequences, equal and different lengths and histories, and keys
    fewer than rows, every row is written.  Values that do not depend on the
    key make the result exact whatever the weights."""
    r = torch.Generator().manual_seed(nseq)
    lens = torch.randint(0, 200, (nseq,), generator=r)
    lens[nseq // 2] = 129
    hist = torch.randint(-3, 5, (nseq,), generator=r) * 32
    klens = (lens + hist).clamp(min=0)
    cu_q, cu_k = cu_of(lens.tolist()), cu_of(klens.tolist())
    n, hq, hk = int(lens.sum()), 6, 2
    q = torch.randn(n, hq, d, device=DEV).bfloat16()
    k = torch.randn(int(klens.sum()) + 1, hk, d, device=DEV).bfloat16()[:-1]
    value = torch.arange(1, nseq + 1, device=DEV)
    v = value.repeat_interleave(klens.to(DEV)).bfloat16()[:, None, None] \
        .expand(-1, hk, d).contiguous()
    for causal in (True, False):
        out = torch.full((n, hq, d), -7.0, device=DEV).bfloat16()
        ops._require_ext().varlen_prefill_attention(
            out, q, k, v, cu_q.to(DEV), cu_k.to(DEV), torch.empty(0),
            torch.empty(0), d ** -0.5, causal, torch.empty(0))
        for i in range(nseq):
            a = out[cu_q[i]:cu_q[i + 1]].float()
            blind = min(max(-int(hist[i]), 0), int(lens[i])) if causal else (
                0 if klens[i] else int(lens[i]))
            assert (a[:blind] == 0).all()    # rows that see no key
            assert ((a[blind:] - (i + 1)).abs() <= 2 ** -8 * (i + 1)).all()


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("offset,pad", [(1, 0), (0, 1), (4, 0), (0, 4)])
def test_unaligned_rows(offset, pad, d):
    """Keys, values, queries and gradients whose rows do not start at 16-byte
    addresses give the bits that aligned copies give."""
    torch.manual_seed(8)
    lens, hq, hk, scale = [65, 130], 4, 2, d ** -0.5
    cu, n = cu_of(lens).to(DEV), 195

    def rows(h):
        flat = torch.randn(n * (h * d + pad) + offset, device=DEV).bfloat16()
        return flat[offset:].view(n, h * d + pad)[:, :h * d].unflatten(
            1, (h, d))
    q, k, v, dout = rows(hq), rows(hk), rows(hk), rows(hq)
    got = ops.varlen_prefill_attention(q, k, v, cu, cu, scale, True)
    want = ops.varlen_prefill_attention(*(t.clone() for t in (q, k, v)), cu,
                                        cu, scale, True)
    assert torch.equal(got, want)
    ext, tiles = ops._require_ext(), ops.build_varlen_tiles(cu.cpu(), DEV)
    out, lse = ops.varlen_prefill_attention(q, k, v, cu, cu, scale, True,
                                            return_lse=True)
    both = []
    for make in (lambda t: t, lambda t: t.clone(
            memory_format=torch.contiguous_format)):
        grads = [torch.empty(t.shape, device=DEV).bfloat16()
                 for t in (q, k, v)]
        ext.varlen_attention_backward_v3(
            *grads, make(q), make(k), make(v), out,
            make(dout) if dout.is_contiguous() else dout.clone(
                memory_format=torch.contiguous_format), lse, cu, cu,
            tiles[0], tiles[1], scale, True)
        both.append(grads)
    for a, b in zip(*both):
        assert torch.equal(a, b)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("scale", [-0.1, 0.0, 2.0 ** 40, -2.0 ** 40])
def test_window_scales(scale, d):
    """Window attention at scales that are not positive (the largest score is
    not the largest product) or so large that an exponent's rounding passes
    the exponential's range: each row gets the value of its largest score."""
    torch.manual_seed(9)
    lens, hq, hk, page, window, keep = [3, 150], 4, 2, 16, 70, 2
    table = torch.arange(20, dtype=torch.int32, device=DEV).view(2, 10)
    rows = torch.randn(20, page, 2 * hk * d, device=DEV).bfloat16()
    n = sum(lens)
    q = torch.randn(n, hq * d, device=DEV).bfloat16()
    i32 = dict(dtype=torch.int32, device=DEV)
    seq = torch.repeat_interleave(torch.arange(2, **i32),
                                  torch.tensor(lens, device=DEV))
    pos = torch.cat([torch.arange(x, **i32) for x in lens])
    got = ops.seq.gqa_window_attention(
        q, rows, table, seq, pos, hq, hk, d, d, window, keep, None, None,
        None, scale, torch.bfloat16, tiles=ops.seq.attention_tiles(lens, DEV))
    a = 0
    for i, x in enumerate(lens):
        kv = rows[table[i].long()].view(-1, 2, hk, d)[:x].double()
        k, v = heads(kv[:, 0], hq), heads(kv[:, 1], hq)
        r, j = torch.arange(x, device=DEV)[:, None], torch.arange(x, device=DEV)
        live = ((r - j < window) | (j < keep)) & (j <= r)
        s = torch.einsum("qhd,khd->hqk", q[a:a + x].double().view(x, hq, d),
                         k) * scale
        p = torch.softmax(s.masked_fill(~live, -float("inf")), -1)
        want = torch.einsum("hqk,khd->qhd", p, v)
        mass = torch.einsum("hqk,khd->qhd", p, v.abs())
        assert ((got[a:a + x].double().view(x, hq, d) - want).abs()
                <= 2 ** -8 * (mass + want.abs())).all(), i
        a += x


@pytest.mark.parametrize("hq,hk,d", [(12, 4, 128), (16, 4, 128), (8, 4, 64),
                                     (28, 4, 64)])
def test_decode_table_of_long_contexts(hq, hk, d):
    """A page table that could hold more than the caches do: values are then
    read past them.  Short and ragged contexts in it."""
    torch.manual_seed(10)
    lens, page, scale = [1, 31, 129, 700], 16, d ** -0.5
    wide = (128 << 20) // (len(lens) * page * hk * d * 4) + 1
    need = [-(-n // page) for n in lens]
    table = torch.zeros(len(lens), wide, dtype=torch.int32, device=DEV)
    pages = torch.randperm(sum(need), device=DEV).int()
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = pages[at:at + n]
        at += n
    k, v = (torch.randn(sum(need), page, hk, d, device=DEV).bfloat16()
            for _ in range(2))
    q = torch.randn(len(lens), hq, d, device=DEV).bfloat16()
    got = ops.paged_attention_decode(
        q, k, v, table, torch.tensor(lens, dtype=torch.int32, device=DEV),
        scale)
    for i, n in enumerate(lens):
        rows = table[i, :need[i]].long()
        kk = heads(k[rows].view(-1, hk, d)[:n].double(), hq)
        vv = heads(v[rows].view(-1, hk, d)[:n].double(), hq)
        want, _ = attend(q[i:i + 1].double(), kk, vv, n - 1, True, scale)
        mass, _ = attend(q[i:i + 1].double(), kk, vv.abs(), n - 1, True, scale)
        # weights have all their bits, the result is rounded once
        bound = 2 ** -8 * want.abs() + 2 ** -14 * mass
        assert ((got[i:i + 1].double() - want).abs() <= bound).all(), n


@pytest.mark.parametrize("hq,hk,d", [(4, 4, 128), (8, 2, 128), (4, 4, 64)])
def test_window_many_tiles(hq, hk, d):
    """More row tiles than run at a time with two blocks per CU: heads of 128
    then have one buffer of values."""
    torch.manual_seed(12)
    lens, page, window, keep, scale = [3, 70, 64, 300] * 33, 16, 90, 5, d ** -0.5
    need = [-(-n // page) for n in lens]
    table = torch.zeros(len(lens), max(need), dtype=torch.int32, device=DEV)
    pages = torch.randperm(sum(need), device=DEV).int()
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = pages[at:at + n]
        at += n
    rows = torch.randn(sum(need), page, 2 * hk * d, device=DEV).bfloat16()
    n = sum(lens)
    q = torch.randn(n, hq * d, device=DEV).bfloat16()
    i32 = dict(dtype=torch.int32, device=DEV)
    seq = torch.repeat_interleave(torch.arange(len(lens), **i32),
                                  torch.tensor(lens, device=DEV))
    pos = torch.cat([torch.arange(x, **i32) for x in lens])
    got = ops.seq.gqa_window_attention(
        q, rows, table, seq, pos, hq, hk, d, d, window, keep, None, None,
        None, scale, torch.bfloat16, tiles=ops.seq.attention_tiles(lens, DEV))
    a = 0
    for i, x in enumerate(lens):
        kv = rows[table[i, :need[i]].long()].view(-1, 2, hk, d)[:x].double()
        k, v = heads(kv[:, 0], hq), heads(kv[:, 1], hq)
        r, j = torch.arange(x, device=DEV)[:, None], torch.arange(x, device=DEV)
        live = ((r - j < window) | (j < keep)) & (j <= r)
        s = torch.einsum("qhd,khd->hqk", q[a:a + x].double().view(x, hq, d),
                         k) * scale
        p = torch.softmax(s.masked_fill(~live, -float("inf")), -1)
        want = torch.einsum("hqk,khd->qhd", p, v)
        mass = torch.einsum("hqk,khd->qhd", p, v.abs())
        assert ((got[a:a + x].double().view(x, hq, d) - want).abs()
                <= 2 ** -8 * (mass + want.abs())).all(), i
        a += x


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("stride", [1 << 24, 1 << 25, 1 << 27])
def test_window_rows_far_apart(stride, d):
    """Output rows whose distances 32-bit offsets hold, just do not, and do not."""
    torch.manual_seed(22)
    hq, hk, n, page = 8, 2, 70, 16
    i32 = dict(dtype=torch.int32, device=DEV)
    rows = torch.randn(5, page, 2 * hk * d, device=DEV).bfloat16()
    q = torch.randn(n, hq * d, device=DEV).bfloat16()
    far = torch.empty((n - 1) * stride + hq * d, dtype=torch.bfloat16,
                      device=DEV).as_strided((n, hq * d), (stride, 1))
    got, want = (ops.seq.gqa_window_attention(
        q, rows, torch.randperm(5, generator=torch.Generator().manual_seed(1))
        .int().to(DEV)[None], torch.zeros(n, **i32), torch.arange(n, **i32), hq,
        hk, d, d, 40, 0, None, None, None, d ** -0.5, torch.bfloat16,
        tiles=ops.seq.attention_tiles([n], DEV), out=out) for out in (far, None))
    # two kernels, each within 2^-7 of the values' magnitude of the true result
    assert (got - want).abs().max() <= 2 ** -6 * rows.abs().max()


@pytest.mark.parametrize("hq,hk,d", [(4, 4, 128), (8, 2, 128)])
def test_forward_many_tiles(hq, hk, d):
    """More row tiles than run at a time with two blocks per CU: heads of 128
    then have one buffer of values."""
    torch.manual_seed(13)
    lens, scale = [3, 70, 64, 300] * 33 + [129], d ** -0.5
    cu, n = cu_of(lens), sum(lens)
    q = torch.randn(n, hq, d, device=DEV).bfloat16()
    k, v = (torch.randn(n, hk, d, device=DEV).bfloat16() for _ in range(2))
    out = ops.varlen_prefill_attention(q, k, v, cu.to(DEV), cu.to(DEV), scale,
                                       True)
    for i in range(len(lens)):
        a = slice(cu[i], cu[i + 1])
        kk, vv = heads(k[a].double(), hq), heads(v[a].double(), hq)
        want, _ = attend(q[a].double(), kk, vv, 0, True, scale)
        mass, _ = attend(q[a].double(), kk, vv.abs(), 0, True, scale)
        bound = 2 ** -8 * (mass + want.abs())
        assert ((out[a].double() - want).abs() <= bound).all(), i


@pytest.mark.parametrize("what", ["some", "turned", "one_of_them"])
@pytest.mark.parametrize("nseq", [3, 60, 66])
@pytest.mark.parametrize("d", [64, 128])
def test_tables_of_some_tiles(nseq, d, what):
    """A table names the tiles that are computed, in any order: rows of named
    tiles get what a call without a table gives, others are left alone."""
    torch.manual_seed(14)
    lens, h, scale = ([130, 65, 200] * 22)[:nseq], 4, d ** -0.5
    cu_cpu, n = cu_of(lens), sum(lens)
    cu = cu_cpu.to(DEV)
    q, k, v, dout = (torch.randn(n, h, d, device=DEV).bfloat16()
                     for _ in range(4))
    ext, (t_seq, t_r0) = ops._require_ext(), ops.build_varlen_tiles(
        cu_cpu, DEV)[:2]
    pick = {"some": torch.arange(1, len(t_seq), 3),
            "turned": torch.arange(len(t_seq)).flip(0),
            "one_of_them": torch.full((len(t_seq),), 2)}[what].to(DEV)
    some = t_seq[pick].contiguous(), t_r0[pick].contiguous()
    named = torch.zeros(n, dtype=torch.bool, device=DEV)
    for s, r in zip(some[0].tolist(), some[1].tolist()):
        named[cu_cpu[s] + r:min(cu_cpu[s] + r + 64, cu_cpu[s + 1])] = True

    want, lse = ops.varlen_prefill_attention(q, k, v, cu, cu, scale, True,
                                             return_lse=True)
    got = torch.full_like(want, -7.0)
    ext.varlen_prefill_attention(got, q, k, v, cu, cu, *some, scale, True,
                                 torch.empty(0))
    assert torch.equal(got[named], want[named])
    assert (got[~named] == -7).all()

    def grads(tiles):
        g = [torch.full_like(q, -7.0) for _ in range(3)]
        ext.varlen_attention_backward_v3(*g, q, k, v, want, dout, lse, cu, cu,
                                         *tiles, scale, True)
        return g
    # (dK takes sums of the gradient from dQ's tiles)
    for a, b in list(zip(grads(some), grads((t_seq, t_r0))))[::2]:
        assert torch.equal(a[named], b[named])
        assert (a[~named] == -7).all()


@pytest.mark.parametrize("scale", [0.125, 0.0, -0.125])
@pytest.mark.parametrize("d", [64, 128])
def test_values_of_keys_that_a_nan_row_does_not_see(d, scale):
    """A row whose log-sum-exp is NaN: gradients of the values behind it are
    what they are without it, those that it sees are NaN."""
    torch.manual_seed(16)
    n, bad, hq, hk = 70, 5, 4, 2
    cu_cpu = cu_of([n])
    cu, tiles = cu_cpu.to(DEV), ops.build_varlen_tiles(cu_cpu, DEV)[:2]
    q, dout = (torch.randn(n, hq, d, device=DEV).bfloat16() for _ in range(2))
    k, v = (torch.randn(n, hk, d, device=DEV).bfloat16() for _ in range(2))
    out, lse = ops.varlen_prefill_attention(q, k, v, cu, cu, scale, True,
                                            return_lse=True)

    def grad_v(lse):
        g = [torch.empty_like(t) for t in (q, k, v)]
        ops._require_ext().varlen_attention_backward_v3(
            *g, q, k, v, out, dout, lse, cu, cu, *tiles, scale, True)
        return g[2]
    want = grad_v(lse)
    lse[bad] = float("nan")
    got = grad_v(lse)
    assert torch.equal(got[bad + 1:], want[bad + 1:])
    assert torch.isnan(got[:bad + 1]).all()


@pytest.mark.parametrize("rows,hk,most", [
    (256, 1, 720), (257, 1, 704), (257, 1, 720), (383, 1, 1024), (384, 1, 1024),
    (255, 1, 1040), (128, 2, 1040), (341, 1, 1040), (342, 1, 1040),
    (64, 2, 4112), (53, 3, 4112), (160, 1, 4112)])
@pytest.mark.parametrize("d", [64, 128])
def test_decode_stretches(rows, hk, most, d):
    """Both sides of the numbers of rows, and of tokens that the table holds,
    at which a row is divided otherwise; contexts that end in each stretch."""
    torch.manual_seed(17)
    hq, page, scale = 4 * hk, 16, d ** -0.5
    lens = [1 + (most - 1) * i // (rows - 1) for i in range(rows)]
    pages = torch.randperm(40, device=DEV).int()      # shared by the rows
    at = torch.randint(40, (rows, -(-most // page)), device=DEV)
    table = pages[at]
    k, v = (torch.randn(40, page, hk, d, device=DEV).bfloat16()
            for _ in range(2))
    q = torch.randn(rows, hq, d, device=DEV).bfloat16()
    got = ops.paged_attention_decode(
        q, k, v, table, torch.tensor(lens, dtype=torch.int32, device=DEV),
        scale)
    for i in sorted({0, 1, rows // 3, rows // 2, rows - 2, rows - 1}):
        n = lens[i]
        kk = heads(k[table[i].long()].view(-1, hk, d)[:n].double(), hq)
        vv = heads(v[table[i].long()].view(-1, hk, d)[:n].double(), hq)
        want, _ = attend(q[i:i + 1].double(), kk, vv, n - 1, True, scale)
        mass, _ = attend(q[i:i + 1].double(), kk, vv.abs(), n - 1, True, scale)
        # weights have all their bits, the result is rounded once
        bound = 2 ** -8 * want.abs() + 2 ** -14 * mass
        assert ((got[i:i + 1].double() - want).abs() <= bound).all(), n


@pytest.mark.parametrize("rows,hk,most", [
    (8, 1, 384), (8, 1, 400), (127, 1, 400), (128, 1, 1024), (255, 1, 2064),
    (256, 1, 2064), (342, 1, 1040), (85, 12, 1040), (128, 8, 1040),
    (127, 1, 2064), (128, 1, 2064), (146, 1, 2064), (147, 1, 2064)])
@pytest.mark.parametrize("d", [64, 128])
def test_decode_divided_or_not(rows, hk, most, d):
    """Both sides of the lines from which on rows are divided at all, and among
    an odd number of blocks."""
    test_decode_stretches(rows, hk, most, d)


@pytest.mark.parametrize("page", [1, 12, 16])
@pytest.mark.parametrize("group", [1, 4, 5, 8])
@pytest.mark.parametrize("d", [64, 128])
def test_decode_past_the_caches(d, group, page):
    """Tables that could hold more than the caches do, whose entries past the
    contexts name no page: keys go through LDS, and the weights' parts take the
    columns that the heads leave free."""
    torch.manual_seed(18)
    lens, hk, scale = [1, 32, 33, 161, 640], 4, d ** -0.5
    hq = group * hk
    wide = (128 << 20) // (len(lens) * page * hk * d * 4) + 1
    need = [-(-n // page) for n in lens]
    table = torch.full((len(lens), wide), -(1 << 30), dtype=torch.int32,
                       device=DEV)
    pages = torch.randperm(sum(need), device=DEV).int()
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = pages[at:at + n]
        at += n
    k, v = (torch.randn(sum(need), page, hk, d, device=DEV).bfloat16()
            for _ in range(2))
    q = torch.randn(len(lens), hq, d, device=DEV).bfloat16()
    got = ops.paged_attention_decode(
        q, k, v, table, torch.tensor(lens, dtype=torch.int32, device=DEV),
        scale)
    for i, n in enumerate(lens):
        rows = table[i, :need[i]].long()
        kk = heads(k[rows].view(-1, hk, d)[:n].double(), hq)
        vv = heads(v[rows].view(-1, hk, d)[:n].double(), hq)
        want, _ = attend(q[i:i + 1].double(), kk, vv, n - 1, True, scale)
        mass, _ = attend(q[i:i + 1].double(), kk, vv.abs(), n - 1, True, scale)
        # weights have all their bits, the result is rounded once
        bound = 2 ** -8 * want.abs() + 2 ** -14 * mass
        assert ((got[i:i + 1].double() - want).abs() <= bound).all(), n


@pytest.mark.parametrize("count", [1, 15, 16, 17])
@pytest.mark.parametrize("hist", [0, 130])
def test_row_tiles_of_few_and_long_sequences(count, hist):
    """Both sides of the number of sequences up to which a row tile is found 64
    lengths at a time, walks on both sides of 64 and 128 tiles: every sequence's
    rows and their gradients are those of a call of its own."""
    torch.manual_seed(19)
    hq, hk, d = 2, 1, 64
    lens = ([4097, 1, 64, 65, 8200, 130, 4032, 4096, 63, 2, 200, 128, 129, 1000,
             5, 77, 300])[:count]
    cu = torch.tensor([0] + lens).cumsum(0).int()
    cuk = torch.tensor([0] + [n + hist for n in lens]).cumsum(0).int()
    q, do = (torch.randn(sum(lens), hq, d, device=DEV).bfloat16()
             for _ in range(2))
    k, v = (torch.randn(int(cuk[-1]), hk, d, device=DEV).bfloat16()
            for _ in range(2))
    out = ops.varlen_prefill_attention(q, k, v, cu.to(DEV), cuk.to(DEV),
                                       d ** -0.5, causal=True)
    grads = []
    if hist == 0:
        x = [t.clone().requires_grad_() for t in (q, k, v)]
        y = ops.flash_attn_varlen(*x, cu.to(DEV), d ** -0.5, causal=True)
        assert torch.equal(y, out)
        grads = torch.autograd.grad(y, x, do)
    for i, n in enumerate(lens):
        a, b = slice(int(cu[i]), int(cu[i + 1])), slice(int(cuk[i]),
                                                        int(cuk[i + 1]))
        one = torch.tensor([0, n], dtype=torch.int32, device=DEV)
        onek = torch.tensor([0, n + hist], dtype=torch.int32, device=DEV)
        assert torch.equal(out[a], ops.varlen_prefill_attention(
            q[a], k[b], v[b], one, onek, d ** -0.5, causal=True)), i
        if grads:
            x = [t[a].clone().requires_grad_() for t in (q, k, v)]
            y = ops.flash_attn_varlen(*x, one, d ** -0.5, causal=True)
            own = torch.autograd.grad(y, x, do[a])
            assert torch.equal(grads[0][a], own[0]), i
            # (heads are divided otherwise: 32-bit sums in another order)
            for g, w in zip(grads[1:], own[1:]):
                assert (g[a] - w).abs().max() <= 2 ** -7 * w.abs().max(), i


FORMS = ["plain", "extras", "negative", "zero", "large", "negative_large",
         "infinite"]


def form_of(what, d):
    """Scale and, for the window kernel, further arguments of a form."""
    scale = {"negative": -0.1, "zero": 0.0, "large": 2.0 ** 40,
             "negative_large": -2.0 ** 40}.get(what, d ** -0.5)
    return scale, dict(q_temp_coef=0.1, q_temp_every=16, chunk=96,
                       out_scale=0.5) if what == "extras" else {}


@pytest.mark.parametrize("what", FORMS)
@pytest.mark.parametrize("hq,hk", [(8, 2), (4, 4), (7, 1)])
def test_window_copies_of_a_batch(hq, hk, what):
    """Heads of 128 with more blocks than run at a time have one buffer of
    values: a batch many times over gives each copy the bits that it has alone,
    with two, in every form that the tests above check there; and an infinite
    entry of a sequence's last value row shows where that row is seen, beside
    finite ones."""
    torch.manual_seed(18)
    d, page, window, keep, copies = 128, 16, 70, 3, 50
    lens, hist = [1, 31, 33, 64, 65, 200, 7], [0, 5, 0, 300, 63, 0, 129]
    need = [-(-(n + m) // page) for n, m in zip(lens, hist)]
    table = torch.zeros(len(lens), max(need), dtype=torch.int32, device=DEV)
    pages = torch.randperm(sum(need), device=DEV).int()
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = pages[at:at + n]
        at += n
    rows = torch.randn(sum(need), page, 2 * hk * d, device=DEV).bfloat16()
    n = sum(lens)
    ends = torch.tensor(lens, device=DEV).cumsum(0) - 1
    if what == "infinite":
        for i, (x, m) in enumerate(zip(lens, hist)):
            last = x + m - 1
            rows[table[i, last // page].long(), last % page].view(2, hk, d)[
                1, :, 5] = float("inf")
    q = torch.randn(n, hq * d, device=DEV).bfloat16()
    i32 = dict(dtype=torch.int32, device=DEV)
    pos = torch.cat([torch.arange(m, m + x, **i32)
                     for x, m in zip(lens, hist)])
    gate = torch.randn(n, hq, device=DEV).bfloat16()
    sink = torch.randn(hq, device=DEV) * 3 if what == "extras" else None
    scale, more = form_of(what, d)

    def run(times):
        many = lens * times
        seq = torch.repeat_interleave(torch.arange(len(many), **i32),
                                      torch.tensor(many, device=DEV))
        return ops.seq.gqa_window_attention(
            q.repeat(times, 1), rows, table.repeat(times, 1), seq,
            pos.repeat(times), hq, hk, d, d, window, keep, None, None,
            gate.repeat(times, 1) if what == "extras" else None, scale,
            torch.bfloat16, tiles=ops.seq.attention_tiles(many, DEV),
            sink=sink, **more).view(times, n, hq * d)
    alone, got = run(1), run(copies)
    # (bits: rows that do not see an infinite value weigh it with 0)
    assert torch.equal(got.view(torch.int16),
                       alone.view(torch.int16).expand(copies, -1, -1))
    if what == "infinite":
        seen = got[:, ends].view(copies, len(lens), hq, d)
        assert (seen[..., 5] == float("inf")).all()
        assert seen[..., [j for j in range(d) if j != 5]].isfinite().all()


@pytest.mark.parametrize("what", [f for f in FORMS if f != "extras"])
@pytest.mark.parametrize("hq,hk", [(8, 2), (4, 4), (7, 1)])
def test_forward_copies_of_a_batch(hq, hk, what):
    """The same for packed prompts, some of them behind cached keys."""
    torch.manual_seed(19)
    d, copies = 128, 60
    lens, hist = [1, 31, 33, 64, 65, 200, 7], [0, 5, 0, 300, 63, 0, 129]
    klens = [x + m for x, m in zip(lens, hist)]
    n, nk = sum(lens), sum(klens)
    q = torch.randn(n, hq, d, device=DEV).bfloat16()
    k, v = (torch.randn(nk, hk, d, device=DEV).bfloat16() for _ in range(2))
    if what == "infinite":
        v[torch.tensor(klens, device=DEV).cumsum(0) - 1, :, 5] = float("inf")
    ends = torch.tensor(lens, device=DEV).cumsum(0) - 1
    scale, _ = form_of(what, d)

    def run(times):
        return ops.varlen_prefill_attention(
            *(t.repeat(times, 1, 1) for t in (q, k, v)),
            cu_of(lens * times).to(DEV), cu_of(klens * times).to(DEV), scale,
            True).view(times, n, hq, d)
    alone, got = run(1), run(copies)
    assert torch.equal(got.view(torch.int16),
                       alone.view(torch.int16).expand(copies, -1, -1, -1))
    if what == "infinite":
        seen = got[:, ends]
        assert (seen[..., 5] == float("inf")).all()
        assert seen[..., [j for j in range(d) if j != 5]].isfinite().all()

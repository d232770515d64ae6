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

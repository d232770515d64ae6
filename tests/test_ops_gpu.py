"""GPU numerics: every HIP kernel vs the plain-PyTorch fp32 reference (ops.ref).

All tests are @pytest.mark.gpu and run on a real MI355X via gpurun / the
driver's round-end GPU tier.
"""
import math

import pytest
import torch

import polyrl_amd.ops as ops
from polyrl_amd.ops import ref

pytestmark = pytest.mark.gpu

DEV = "cuda"


def setup_module():
    assert ops.extension_loaded(), "HIP extension must be loaded on GPU"


def rel_err(a, b):
    a, b = a.float(), b.float()
    return ((a - b).abs().max() / (b.abs().max() + 1e-6)).item()


# ---------------------------------------------------------------- norms/elem


@pytest.mark.parametrize("shape", [(4, 512), (37, 4096), (128, 8192)])
def test_rmsnorm(shape):
    torch.manual_seed(0)
    x = torch.randn(shape, dtype=torch.bfloat16, device=DEV)
    w = torch.randn(shape[-1], dtype=torch.bfloat16, device=DEV)
    out = ops.rmsnorm(x, w)
    expect = ref.rmsnorm(x.cpu(), w.cpu())
    assert rel_err(out.cpu(), expect) < 2e-2


def test_fused_add_rmsnorm():
    torch.manual_seed(1)
    x = torch.randn(33, 2048, dtype=torch.bfloat16, device=DEV)
    res = torch.randn_like(x)
    w = torch.randn(2048, dtype=torch.bfloat16, device=DEV)
    expect_norm, expect_res = ref.fused_add_rmsnorm(x.cpu(), res.cpu().clone(), w.cpu())
    out, new_res = ops.fused_add_rmsnorm(x, res, w)
    assert rel_err(new_res.cpu(), expect_res) < 2e-2
    assert rel_err(out.cpu(), expect_norm) < 2e-2


@pytest.mark.parametrize("d", [8, 504, 512, 520, 1024, 1032, 2048, 2056, 3064,
                               3072, 4096, 4104, 8192, 8200, 12288])
@pytest.mark.parametrize("rows", [1, 130, 1024, 1792])
def test_rmsnorm_widths(rows, d):
    """Both sides of the widths from which a row takes more waves and more words
    a thread, and rows that are read again."""
    g = torch.Generator(device=DEV).manual_seed(d + rows)
    x, res = (torch.randn(rows, d, generator=g, device=DEV).bfloat16()
              for _ in range(2))
    w = torch.randn(d, generator=g, device=DEV).bfloat16()

    def close(got, y):
        want = y.double() * (y.double().square().mean(-1, keepdim=True)
                             + 1e-6).rsqrt() * w.double()
        # one rounding to bf16, 32-bit sums of squares
        assert ((got.double() - want).abs() <= (2 ** -8 + 1e-5)
                * want.abs()).all()
    close(ops.rmsnorm(x, w), x)
    total = (x.float() + res.float()).bfloat16()
    out, new = ops.fused_add_rmsnorm(x, res, w)
    assert torch.equal(new, total)
    close(out, total)


def test_silu_mul():
    torch.manual_seed(2)
    g = torch.randn(64, 5632, dtype=torch.bfloat16, device=DEV)
    u = torch.randn_like(g)
    out = ops.silu_mul(g, u)
    expect = ref.silu_mul(g.cpu(), u.cpu())
    assert rel_err(out.cpu(), expect) < 2e-2


def test_rope():
    torch.manual_seed(3)
    N, Hq, Hk, D = 40, 8, 2, 128
    q = torch.randn(N, Hq, D, dtype=torch.bfloat16, device=DEV)
    k = torch.randn(N, Hk, D, dtype=torch.bfloat16, device=DEV)
    pos = torch.randint(0, 1000, (N,), dtype=torch.int32, device=DEV)
    table = ops.RopeTable(D, 2048, 10000.0, DEV)
    cos, sin = ref.rope_cos_sin(pos.cpu(), D, 10000.0)
    eq, ek = ref.apply_rope(q.cpu(), k.cpu(), cos, sin)
    ops.apply_rope_inplace(q, k, pos, table)
    assert rel_err(q.cpu(), eq) < 2e-2
    assert rel_err(k.cpu(), ek) < 2e-2


# ------------------------------------------------------------------ logprobs


@pytest.mark.parametrize("V", [128, 32000, 151936])
def test_gather_logprobs(V):
    torch.manual_seed(4)
    N = 33
    logits = torch.randn(N, V, dtype=torch.bfloat16, device=DEV) * 4
    labels = torch.randint(0, V, (N,), device=DEV)
    lp, ent = ops.gather_logprobs(logits, labels, want_entropy=True)
    elp, eent = ref.gather_logprobs_entropy(logits.cpu(), labels.cpu())
    assert torch.allclose(lp.cpu(), elp, atol=1e-2, rtol=1e-3)
    assert torch.allclose(ent.cpu(), eent, atol=1e-2, rtol=1e-3)


def test_gather_logprobs_fp32():
    torch.manual_seed(5)
    logits = torch.randn(7, 5000, device=DEV) * 3
    labels = torch.randint(0, 5000, (7,), device=DEV)
    lp = ops.gather_logprobs(logits, labels)
    elp = ref.gather_logprobs(logits.cpu(), labels.cpu())
    assert torch.allclose(lp.cpu(), elp, atol=1e-4, rtol=1e-5)


# ------------------------------------------------------------------ sampling


def test_sample_greedy_exact():
    torch.manual_seed(6)
    N, V = 16, 32000
    logits = torch.randn(N, V, dtype=torch.bfloat16, device=DEV) * 3
    temp = torch.zeros(N, device=DEV)
    tk = torch.full((N,), -1, dtype=torch.int32, device=DEV)
    tp = torch.ones(N, device=DEV)
    tokens, lps = ops.sample(logits, temp, tk, tp, seed=7)
    expect = logits.float().argmax(-1)
    assert torch.equal(tokens, expect)
    elp = ref.gather_logprobs(logits.cpu(), expect.cpu())
    assert torch.allclose(lps.cpu(), elp, atol=1e-2, rtol=1e-3)


def test_sample_top_k_stays_in_set():
    torch.manual_seed(7)
    N, V, K = 64, 4096, 20
    logits = (torch.randn(N, V, device=DEV) * 5).bfloat16()
    temp = torch.ones(N, device=DEV)
    tk = torch.full((N,), K, dtype=torch.int32, device=DEV)
    tp = torch.ones(N, device=DEV)
    topk_sets = torch.topk(logits.float(), K, dim=-1).indices
    for seed in range(5):
        tokens, _ = ops.sample(logits, temp, tk, tp, seed=seed)
        for i in range(N):
            # allow boundary ties: sampled logit >= k-th largest logit
            kth = logits[i].float()[topk_sets[i][-1]]
            assert logits[i, tokens[i]].float() >= kth - 1e-3


def test_sample_top_p_mass():
    torch.manual_seed(8)
    N, V = 32, 1024
    logits = (torch.randn(N, V, device=DEV) * 6).bfloat16()
    temp = torch.ones(N, device=DEV)
    tk = torch.full((N,), -1, dtype=torch.int32, device=DEV)
    tp = torch.full((N,), 0.7, device=DEV)
    probs = torch.softmax(logits.float(), -1)
    sorted_p, sorted_idx = probs.sort(-1, descending=True)
    cum = sorted_p.cumsum(-1)
    # nucleus boundary VALUE per row: smallest sorted logit still in nucleus
    # (ties at the boundary are all kept by the kernel, which is valid)
    boundary = torch.empty(N)
    for i in range(N):
        j = int((cum[i] - sorted_p[i] < 0.7).sum().item()) - 1  # last kept rank
        boundary[i] = logits[i].float()[sorted_idx[i, j]].cpu()
    for seed in range(5):
        tokens, _ = ops.sample(logits, temp, tk, tp, seed=seed)
        for i in range(N):
            got = logits[i, tokens[i]].float().cpu()
            assert got >= boundary[i] - 1e-3, \
                f"row {i}: sampled logit {got} below nucleus boundary {boundary[i]}"


def test_sample_categorical_distribution():
    """statistical check: sampled frequencies track softmax probs on small V"""
    V = 8
    logits = torch.tensor([[0., 1., 2., 0.5, -1., 3., 0., 1.5]],
                          device=DEV).bfloat16()
    logits = logits.repeat(4096, 1).contiguous()
    temp = torch.ones(4096, device=DEV)
    tk = torch.full((4096,), -1, dtype=torch.int32, device=DEV)
    tp = torch.ones(4096, device=DEV)
    counts = torch.zeros(V)
    for seed in range(4):
        tokens, _ = ops.sample(logits, temp, tk, tp, seed=seed * 7919 + 13)
        counts += torch.bincount(tokens.cpu(), minlength=V).float()
    freq = counts / counts.sum()
    expect = torch.softmax(logits[0].float().cpu(), -1)
    assert (freq - expect).abs().max().item() < 0.02


# ------------------------------------------------------------------ KV cache


def test_kv_cache_append():
    torch.manual_seed(9)
    num_pages, page_size, Hk, D = 16, 16, 4, 128
    kc = torch.zeros(num_pages, page_size, Hk, D, dtype=torch.bfloat16, device=DEV)
    vc = torch.zeros_like(kc)
    N = 23
    k = torch.randn(N, Hk, D, dtype=torch.bfloat16, device=DEV)
    v = torch.randn_like(k)
    slots = torch.randperm(num_pages * page_size, device=DEV)[:N].int()
    ops.kv_cache_append(kc, vc, k, v, slots)
    flat = kc.view(-1, Hk, D)
    for i in range(N):
        assert torch.equal(flat[slots[i].long()], k[i])


# ----------------------------------------------------------------- attention


@pytest.mark.parametrize("Hq,Hk,D", [(8, 8, 128), (8, 2, 128), (32, 8, 128),
                                     (12, 2, 128), (28, 4, 128), (12, 12, 64)])
def test_paged_attention_decode(Hq, Hk, D):
    torch.manual_seed(10)
    B, page_size = 9, 16
    lens = torch.tensor([1, 5, 16, 17, 60, 64, 100, 255, 300], dtype=torch.int32)
    max_pages = int((-(-lens.max().item() // page_size)))
    num_pages = int(sum(-(-int(l) // page_size) for l in lens)) + 4
    kc = torch.randn(num_pages, page_size, Hk, D, dtype=torch.bfloat16, device=DEV)
    vc = torch.randn_like(kc)
    # random page table (distinct pages)
    perm = torch.randperm(num_pages)
    pt = torch.zeros(B, max_pages, dtype=torch.int32)
    pi = 0
    for b in range(B):
        for j in range(-(-int(lens[b]) // page_size)):
            pt[b, j] = perm[pi]
            pi += 1
    q = torch.randn(B, Hq, D, dtype=torch.bfloat16, device=DEV)
    scale = 1.0 / math.sqrt(D)
    out = ops.paged_attention_decode(q, kc, vc, pt.to(DEV), lens.to(DEV), scale)
    expect = ref.paged_attention_decode(q.cpu(), kc.cpu(), vc.cpu(), pt,
                                        lens, scale)
    assert rel_err(out.cpu(), expect) < 3e-2


@pytest.mark.parametrize("Hq,Hk,D", [(8, 8, 128), (32, 8, 128),
                                     (8, 2, 128), (16, 4, 64)])
def test_paged_attention_decode_mfma(Hq, Hk, D):
    """Decode attention against the CPU form: groups of one to four heads."""
    torch.manual_seed(10)
    B, page_size = 9, 16
    lens = torch.tensor([1, 5, 16, 17, 60, 64, 100, 255, 300],
                        dtype=torch.int32)
    max_pages = int((-(-lens.max().item() // page_size)))
    num_pages = int(sum(-(-int(l) // page_size) for l in lens)) + 4
    kc = torch.randn(num_pages, page_size, Hk, D, dtype=torch.bfloat16,
                     device=DEV)
    vc = torch.randn_like(kc)
    perm = torch.randperm(num_pages)
    pt = torch.zeros(B, max_pages, dtype=torch.int32)
    pi = 0
    for b in range(B):
        for j in range(-(-int(lens[b]) // page_size)):
            pt[b, j] = perm[pi]
            pi += 1
    q = torch.randn(B, Hq, D, dtype=torch.bfloat16, device=DEV)
    scale = 1.0 / math.sqrt(D)
    out = ops.paged_attention_decode(q, kc, vc, pt.to(DEV), lens.to(DEV),
                                     scale)
    expect = ref.paged_attention_decode(q.cpu(), kc.cpu(), vc.cpu(), pt,
                                        lens, scale)
    assert rel_err(out.cpu(), expect) < 3e-2


@pytest.mark.parametrize("Hq,Hk", [(8, 8), (8, 2), (32, 8)])
def test_varlen_prefill_attention(Hq, Hk):
    torch.manual_seed(11)
    D = 128
    seqlens = [1, 17, 64, 63, 200, 256]
    cu = torch.tensor([0] + list(torch.tensor(seqlens).cumsum(0)), dtype=torch.int32)
    total = int(cu[-1])
    q = torch.randn(total, Hq, D, dtype=torch.bfloat16, device=DEV) / 4
    k = torch.randn(total, Hk, D, dtype=torch.bfloat16, device=DEV) / 4
    v = torch.randn(total, Hk, D, dtype=torch.bfloat16, device=DEV)
    scale = 1.0 / math.sqrt(D)
    out = ops.varlen_prefill_attention(q, k, v, cu.to(DEV), cu.to(DEV), scale)
    expect = ref.varlen_prefill_attention(q.cpu(), k.cpu(), v.cpu(), cu, cu, scale)
    assert rel_err(out.cpu(), expect) < 3e-2


def test_varlen_prefill_chunked_alignment():
    """seqlen_k > seqlen_q: query block aligned to the end of keys."""
    torch.manual_seed(12)
    Hq, Hk, D = 8, 2, 128
    cu_q = torch.tensor([0, 32, 96], dtype=torch.int32)
    cu_k = torch.tensor([0, 100, 228], dtype=torch.int32)
    q = torch.randn(96, Hq, D, dtype=torch.bfloat16, device=DEV) / 4
    k = torch.randn(228, Hk, D, dtype=torch.bfloat16, device=DEV) / 4
    v = torch.randn(228, Hk, D, dtype=torch.bfloat16, device=DEV)
    scale = 1.0 / math.sqrt(D)
    out = ops.varlen_prefill_attention(q, k, v, cu_q.to(DEV), cu_k.to(DEV), scale)
    expect = ref.varlen_prefill_attention(q.cpu(), k.cpu(), v.cpu(), cu_q, cu_k,
                                          scale)
    assert rel_err(out.cpu(), expect) < 3e-2


# ------------------------------------------------- strided (fused-qkv) views


def test_silu_mul_strided_gate_up():
    """gate/up as strided row views into a fused (N, 2I) projection."""
    torch.manual_seed(31)
    N, I = 33, 5632
    gate_up = torch.randn(N, 2 * I, dtype=torch.bfloat16, device=DEV)
    out = ops.silu_mul(gate_up.narrow(1, 0, I), gate_up.narrow(1, I, I))
    expect = ref.silu_mul(gate_up[:, :I].cpu(), gate_up[:, I:].cpu())
    assert rel_err(out.cpu(), expect) < 2e-2


def test_rope_and_kv_append_strided_qkv():
    """rope + kv-append on head views straight into a fused qkv row."""
    torch.manual_seed(32)
    N, Hq, Hk, D = 17, 8, 2, 128
    table = ops.RopeTable(D, 256, 10000.0, DEV)
    qkv = torch.randn(N, (Hq + 2 * Hk) * D, dtype=torch.bfloat16, device=DEV)
    qkv_ref = qkv.clone()
    pos = torch.randint(0, 256, (N,), dtype=torch.int32, device=DEV)

    q = qkv.narrow(1, 0, Hq * D).unflatten(1, (Hq, D))
    k = qkv.narrow(1, Hq * D, Hk * D).unflatten(1, (Hk, D))
    v = qkv.narrow(1, (Hq + Hk) * D, Hk * D).unflatten(1, (Hk, D))
    ops.apply_rope_inplace(q, k, pos, table)

    qr = qkv_ref.narrow(1, 0, Hq * D).unflatten(1, (Hq, D)).contiguous()
    kr = qkv_ref.narrow(1, Hq * D, Hk * D).unflatten(1, (Hk, D)).contiguous()
    cos = table.cos[pos.long()]
    sin = table.sin[pos.long()]
    q2, k2 = ref.apply_rope(qr.cpu().float(), kr.cpu().float(),
                            cos.cpu(), sin.cpu())
    assert rel_err(q.cpu(), q2) < 2e-2
    assert rel_err(k.cpu(), k2) < 2e-2

    # kv append from the strided views
    pages, psz = 8, 16
    k_cache = torch.zeros(pages, psz, Hk, D, dtype=torch.bfloat16, device=DEV)
    v_cache = torch.zeros_like(k_cache)
    slots = torch.randperm(pages * psz, device=DEV)[:N].int()
    ops.kv_cache_append(k_cache, v_cache, k, v, slots)
    flat_k = k_cache.view(-1, Hk, D)
    flat_v = v_cache.view(-1, Hk, D)
    assert torch.equal(flat_k[slots.long()], k)
    assert torch.equal(flat_v[slots.long()], v)


def test_decode_attention_strided_q():
    torch.manual_seed(33)
    B, Hq, Hk, D = 4, 8, 2, 128
    pages, psz = 16, 16
    qkv = torch.randn(B, (Hq + 2 * Hk) * D, dtype=torch.bfloat16, device=DEV)
    q = qkv.narrow(1, 0, Hq * D).unflatten(1, (Hq, D))
    k_cache = torch.randn(pages, psz, Hk, D, dtype=torch.bfloat16, device=DEV)
    v_cache = torch.randn_like(k_cache)
    pt = torch.arange(pages, dtype=torch.int32, device=DEV).reshape(B, -1)
    ctx = torch.tensor([7, 30, 48, 1], dtype=torch.int32, device=DEV)
    scale = 1.0 / math.sqrt(D)
    out = ops.paged_attention_decode(q, k_cache, v_cache, pt, ctx, scale)
    expect = ref.paged_attention_decode(
        q.contiguous().cpu().float(), k_cache.cpu().float(),
        v_cache.cpu().float(), pt.cpu(), ctx.cpu(), scale)
    assert rel_err(out.cpu(), expect) < 2e-2


def test_prefill_attention_strided_qkv():
    torch.manual_seed(34)
    Hq, Hk, D = 8, 2, 128
    lens = [33, 64, 7]
    total = sum(lens)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)),
                      dtype=torch.int32, device=DEV)
    qkv = torch.randn(total, (Hq + 2 * Hk) * D, dtype=torch.bfloat16,
                      device=DEV)
    q = qkv.narrow(1, 0, Hq * D).unflatten(1, (Hq, D))
    k = qkv.narrow(1, Hq * D, Hk * D).unflatten(1, (Hk, D))
    v = qkv.narrow(1, (Hq + Hk) * D, Hk * D).unflatten(1, (Hk, D))
    scale = 1.0 / math.sqrt(D)
    out = ops.varlen_prefill_attention(q, k, v, cu, cu, scale, causal=True)
    expect = ref.varlen_prefill_attention(
        q.contiguous().cpu().float(), k.contiguous().cpu().float(),
        v.contiguous().cpu().float(), cu.cpu(), cu.cpu(), scale, True)
    assert rel_err(out.cpu(), expect) < 2e-2


def test_sample_fast_path_statistics():
    """Fused single-pass sampler: empirical distribution tracks softmax."""
    torch.manual_seed(35)
    N, V = 512, 4096
    base = (torch.randn(V, device=DEV) * 3).bfloat16()
    logits = base.expand(N, V).contiguous()
    temp = torch.ones(N, device=DEV)
    tk = torch.full((N,), -1, dtype=torch.int32, device=DEV)
    tp = torch.ones(N, device=DEV)
    counts = torch.zeros(V)
    draws = 0
    for seed in range(20):
        tokens, lps = ops.sample(logits, temp, tk, tp, seed=seed * 977 + 1,
                                 no_filter=True)
        counts += torch.bincount(tokens.cpu(), minlength=V).float()
        draws += N
        # reported logprob is the raw softmax logprob of the sampled token
        expect_lp = ref.gather_logprobs(logits.cpu(), tokens.cpu())
        assert torch.allclose(lps.cpu(), expect_lp, atol=2e-2, rtol=1e-2)
    probs = torch.softmax(base.float().cpu(), -1)
    top = probs.topk(5).indices
    emp = counts / draws
    for t in top:
        assert abs(emp[t] - probs[t]) < 0.05 + 0.3 * probs[t], \
            (t, emp[t], probs[t])


# ------------------------------------------- flash-attn backward (training)


def test_flash_attn_varlen_backward():
    """Custom MFMA backward vs torch-autograd of the fp32 reference."""
    torch.manual_seed(40)
    Hq, Hk, D = 8, 2, 128
    lens = [48, 64, 33]
    total = sum(lens)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)),
                      dtype=torch.int32, device=DEV)
    scale = 1.0 / math.sqrt(D)

    q = (torch.randn(total, Hq, D, device=DEV) / 4).bfloat16().requires_grad_()
    k = (torch.randn(total, Hk, D, device=DEV) / 4).bfloat16().requires_grad_()
    v = (torch.randn(total, Hk, D, device=DEV) / 4).bfloat16().requires_grad_()
    w = torch.randn(total, Hq, D, device=DEV)

    out = ops.flash_attn_varlen(q, k, v, cu, scale, causal=True)
    (out.float() * w).sum().backward()
    dq, dk, dv = q.grad.clone(), k.grad.clone(), v.grad.clone()

    # reference: fp32 torch autograd on CPU
    q2 = q.detach().cpu().float().requires_grad_()
    k2 = k.detach().cpu().float().requires_grad_()
    v2 = v.detach().cpu().float().requires_grad_()
    out2 = ref.varlen_prefill_attention(q2, k2, v2, cu.cpu(), cu.cpu(),
                                        scale, True)
    (out2 * w.cpu()).sum().backward()

    assert rel_err(out.cpu(), out2.detach()) < 2e-2
    assert rel_err(dq.cpu(), q2.grad) < 3e-2, rel_err(dq.cpu(), q2.grad)
    assert rel_err(dk.cpu(), k2.grad) < 3e-2, rel_err(dk.cpu(), k2.grad)
    assert rel_err(dv.cpu(), v2.grad) < 3e-2, rel_err(dv.cpu(), v2.grad)


def test_prefill_lse_output():
    torch.manual_seed(41)
    Hq, Hk, D = 4, 2, 128
    lens = [40, 17]
    total = sum(lens)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)),
                      dtype=torch.int32, device=DEV)
    scale = 1.0 / math.sqrt(D)
    q = (torch.randn(total, Hq, D, device=DEV) / 4).bfloat16()
    k = (torch.randn(total, Hk, D, device=DEV) / 4).bfloat16()
    v = (torch.randn(total, Hk, D, device=DEV) / 4).bfloat16()
    out, lse = ops.varlen_prefill_attention(q, k, v, cu, cu, scale,
                                            causal=True, return_lse=True)
    lse_ref = ref.varlen_lse(q.cpu(), k.cpu(), cu.cpu(), cu.cpu(), scale, True)
    assert (lse.cpu() - lse_ref).abs().max().item() < 5e-2


def test_packed_model_forward_gpu():
    """Trainer model packed path on GPU (flash kernels) vs dense SDPA."""
    from polyrl_amd.models import create_model, get_model_config
    from polyrl_amd.models.registry import DecoderConfig
    cfg = DecoderConfig(arch="llama", vocab_size=512, hidden_size=256,
                        intermediate_size=512, num_hidden_layers=2,
                        num_attention_heads=2, num_key_value_heads=1,
                        head_dim=128, max_position_embeddings=128,
                        rope_theta=10000.0, rms_norm_eps=1e-6)
    torch.manual_seed(42)
    m = create_model(cfg, kind="actor", dtype="bfloat16", device=DEV)
    B, L = 3, 32
    ids = torch.randint(0, cfg.vocab_size, (B, L), device=DEV)
    am = torch.ones(B, L, dtype=torch.long, device=DEV)
    am[0, :7] = 0
    pos = (torch.cumsum(am, dim=1) - 1).clamp(min=0)
    with torch.no_grad():
        dense = m(ids, attention_mask=am, position_ids=pos).float()
        m.model.use_remove_padding = True
        packed = m(ids, attention_mask=am, position_ids=pos).float()
    valid = am.bool()
    err = rel_err(packed[valid], dense[valid])
    assert err < 5e-2, err


# ----------------------------------------------------- engine-level on GPU


def test_engine_greedy_matches_trainer_model_gpu():
    """Greedy engine decode (HIP kernel path + hipGraphs) must match the
    trainer model's argmax chain on GPU."""
    from polyrl_amd.models import create_model
    from polyrl_amd.models.registry import DecoderConfig
    from polyrl_amd.rollout.engine import Engine, SamplingParams
    cfg = DecoderConfig(arch="llama", vocab_size=512, hidden_size=256,
                        intermediate_size=512, num_hidden_layers=2,
                        num_attention_heads=2, num_key_value_heads=1,
                        head_dim=128, max_position_embeddings=128,
                        rope_theta=10000.0, rms_norm_eps=1e-6)
    torch.manual_seed(50)
    model = create_model(cfg, kind="actor", dtype="bfloat16", device=DEV)
    eng = Engine(cfg, device=DEV, dtype=torch.bfloat16,
                 kv_bytes_budget=32 << 20, decode_chunk_size=4)
    eng.model.load_state_dict(model.state_dict())
    torch.manual_seed(51)
    prompt = torch.randint(0, cfg.vocab_size, (9,)).tolist()
    outs = eng.generate([prompt], SamplingParams(temperature=0.0,
                                                 max_new_tokens=8), "g")
    got = outs[0].output_ids
    ids = list(prompt)
    expect = []
    with torch.no_grad():
        for _ in range(8):
            x = torch.tensor([ids], device=DEV)
            logits = model(x).float()
            t = int(logits[0, -1].argmax())
            expect.append(t)
            ids.append(t)
    # margin-aware fp32 oracle: teacher-force the
    # ENGINE's own chain through an fp32 copy of the same weights; every
    # engine token must either be the fp32 argmax or lie within bf16 noise
    # of it (a genuine near-tie).  A wrong-math engine token would sit many
    # logits below the fp32 argmax and fail regardless of position.
    model32 = create_model(cfg, kind="actor", dtype="float32", device=DEV)
    model32.load_state_dict(
        {k: v.float() for k, v in model.state_dict().items()})
    MARGIN = 0.15
    ids = list(prompt)
    n_exact = 0
    with torch.no_grad():
        for t_engine in got:
            logits = model32(torch.tensor([ids], device=DEV)).float()[0, -1]
            top = int(logits.argmax())
            if t_engine == top:
                n_exact += 1
            else:
                margin = float(logits[top] - logits[t_engine])
                assert margin < MARGIN, \
                    (t_engine, top, margin, got, expect)
            ids.append(t_engine)
    assert n_exact >= 6, (n_exact, got, expect)


def test_engine_sampling_replay_determinism_gpu():
    """Same seed + same submission order => identical sampled outputs
    (counter-based RNG, deterministic kernels; hipGraph replays included).
    Note: outputs are keyed by batch-row like other engines, so different
    chunk sizes/batch compositions legitimately draw differently."""
    from polyrl_amd.models import create_model
    from polyrl_amd.models.registry import DecoderConfig
    from polyrl_amd.rollout.engine import Engine, SamplingParams
    cfg = DecoderConfig(arch="llama", vocab_size=512, hidden_size=256,
                        intermediate_size=512, num_hidden_layers=2,
                        num_attention_heads=2, num_key_value_heads=1,
                        head_dim=128, max_position_embeddings=256,
                        rope_theta=10000.0, rms_norm_eps=1e-6)
    torch.manual_seed(52)
    model = create_model(cfg, kind="actor", dtype="bfloat16", device=DEV)
    prompts = [torch.randint(0, cfg.vocab_size, (n,)).tolist()
               for n in (5, 11)]
    results = []
    for _ in range(2):
        eng = Engine(cfg, device=DEV, dtype=torch.bfloat16,
                     kv_bytes_budget=32 << 20, decode_chunk_size=16,
                     seed=7)
        eng.model.load_state_dict(model.state_dict())
        outs = eng.generate(prompts,
                            SamplingParams(temperature=1.0,
                                           max_new_tokens=12), "c")
        results.append([o.output_ids for o in outs])
    assert results[0] == results[1], results
    lens = [len(o) for o in results[0]]
    assert lens == [12, 12], lens


def test_group_prefix_sharing_gpu():
    """Group API on GPU: shared-prefill greedy == separate requests (fork
    copies + shared page tables through the HIP decode kernels)."""
    from polyrl_amd.models import create_model
    from polyrl_amd.models.registry import DecoderConfig
    from polyrl_amd.rollout.engine import Engine, SamplingParams
    cfg = DecoderConfig(arch="llama", vocab_size=512, hidden_size=256,
                        intermediate_size=512, num_hidden_layers=2,
                        num_attention_heads=2, num_key_value_heads=1,
                        head_dim=128, max_position_embeddings=128,
                        rope_theta=10000.0, rms_norm_eps=1e-6)
    torch.manual_seed(60)
    model = create_model(cfg, kind="actor", dtype="bfloat16", device=DEV)
    eng = Engine(cfg, device=DEV, dtype=torch.bfloat16,
                 kv_bytes_budget=32 << 20, decode_chunk_size=4, page_size=16)
    eng.model.load_state_dict(model.state_dict())
    prompt = torch.randint(0, cfg.vocab_size, (13,)).tolist()  # partial page
    sp = SamplingParams(temperature=0.0, max_new_tokens=6)

    eng.enable_prefix_sharing = False
    sep = eng.generate([prompt] * 3, sp, "sep")
    eng.enable_prefix_sharing = True
    eng.add_request_group("grp", prompt, sp, 3)
    outs = {}
    while eng.has_work():
        for o in eng.step():
            outs[o.rid] = o
    for s in range(3):
        assert outs[f"grp-s{s}"].output_ids == sep[s].output_ids, \
            (s, outs[f"grp-s{s}"].output_ids, sep[s].output_ids)
    assert eng.kv.free_pages == eng.kv.num_pages


@pytest.mark.gpu
def test_engine_radix_cache_greedy_equality_gpu():
    """Radix prefix cache on the HIP kernel path: a request hitting a
    cached system prompt must produce the same greedy tokens as a fresh
    no-cache engine (cached KV pages == recomputed KV pages)."""
    from polyrl_amd.models import create_model
    from polyrl_amd.models.registry import DecoderConfig
    from polyrl_amd.rollout.engine import Engine, SamplingParams
    cfg = DecoderConfig(arch="llama", vocab_size=512, hidden_size=256,
                        intermediate_size=512, num_hidden_layers=2,
                        num_attention_heads=2, num_key_value_heads=1,
                        head_dim=128, max_position_embeddings=256,
                        rope_theta=10000.0, rms_norm_eps=1e-6)
    torch.manual_seed(60)
    model = create_model(cfg, kind="actor", dtype="bfloat16", device=DEV)
    sys_prefix = [int(t) for t in
                  torch.randint(0, cfg.vocab_size, (40,))]
    p1 = sys_prefix + [7, 8, 9]
    p2 = sys_prefix + [21, 22]
    sp = SamplingParams(temperature=0.0, max_new_tokens=6)

    e0 = Engine(cfg, device=DEV, dtype=torch.bfloat16,
                kv_bytes_budget=32 << 20)
    e0.model.load_state_dict(model.state_dict())
    ref1 = e0.generate([p1], sp, "r1")[0].output_ids
    ref2 = e0.generate([p2], sp, "r2")[0].output_ids

    e = Engine(cfg, device=DEV, dtype=torch.bfloat16,
               kv_bytes_budget=32 << 20, enable_radix_cache=True)
    e.model.load_state_dict(model.state_dict())
    o1 = e.generate([p1], sp, "a")[0].output_ids
    assert e.radix.num_nodes > 0
    h0 = e.radix.hit_tokens
    o2 = e.generate([p2], sp, "b")[0].output_ids
    assert e.radix.hit_tokens - h0 >= 32, "no radix hit on shared prefix"
    assert o1 == ref1, (o1, ref1)
    assert o2 == ref2, (o2, ref2)
    e.flush_radix()
    assert e.kv.free_pages == e.kv.num_pages


# ------------------------------------- flash-attn backward v3 (atomic-free)


@pytest.mark.parametrize("D,Hq,Hk", [(128, 8, 2), (64, 8, 8), (64, 16, 4)])
def test_flash_attn_backward_v3_vs_ref(D, Hq, Hk, monkeypatch):
    """v3 dkv+dq split vs torch-autograd fp32 reference, D in {64, 128},
    with GQA and ragged sequence lengths."""
    monkeypatch.setenv("POLYRL_ATTN_BWD", "v3")
    torch.manual_seed(42)
    lens = [100, 64, 31, 1, 130]
    total = sum(lens)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)),
                      dtype=torch.int32, device=DEV)
    scale = 1.0 / math.sqrt(D)
    q = (torch.randn(total, Hq, D, device=DEV) / 4).bfloat16().requires_grad_()
    k = (torch.randn(total, Hk, D, device=DEV) / 4).bfloat16().requires_grad_()
    v = (torch.randn(total, Hk, D, device=DEV) / 4).bfloat16().requires_grad_()
    w = torch.randn(total, Hq, D, device=DEV)
    out = ops.flash_attn_varlen(q, k, v, cu, scale, causal=True)
    (out.float() * w).sum().backward()
    dq, dk, dv = q.grad.clone(), k.grad.clone(), v.grad.clone()

    q2 = q.detach().cpu().float().requires_grad_()
    k2 = k.detach().cpu().float().requires_grad_()
    v2 = v.detach().cpu().float().requires_grad_()
    out2 = ref.varlen_prefill_attention(q2, k2, v2, cu.cpu(), cu.cpu(),
                                        scale, True)
    (out2 * w.cpu()).sum().backward()
    assert rel_err(out.cpu(), out2.detach()) < 2e-2
    assert rel_err(dq.cpu(), q2.grad) < 3e-2, rel_err(dq.cpu(), q2.grad)
    assert rel_err(dk.cpu(), k2.grad) < 3e-2, rel_err(dk.cpu(), k2.grad)
    assert rel_err(dv.cpu(), v2.grad) < 3e-2, rel_err(dv.cpu(), v2.grad)


def test_flash_attn_backward_v3_matches_v1(monkeypatch):
    """v3 and v1 compute the same math from identical saved tensors —
    agreement should be much tighter than either-vs-fp32."""
    torch.manual_seed(43)
    Hq, Hk, D = 8, 2, 128
    lens = [512, 200, 64]
    total = sum(lens)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)),
                      dtype=torch.int32, device=DEV)
    scale = 1.0 / math.sqrt(D)
    qv = (torch.randn(total, Hq, D, device=DEV) / 4).bfloat16()
    kv_ = (torch.randn(total, Hk, D, device=DEV) / 4).bfloat16()
    vv = (torch.randn(total, Hk, D, device=DEV) / 4).bfloat16()
    w = torch.randn(total, Hq, D, device=DEV)
    grads = {}
    for ver in ("v1", "v3"):
        monkeypatch.setenv("POLYRL_ATTN_BWD", ver)
        q = qv.clone().requires_grad_()
        k = kv_.clone().requires_grad_()
        v = vv.clone().requires_grad_()
        out = ops.flash_attn_varlen(q, k, v, cu, scale, causal=True)
        (out.float() * w).sum().backward()
        grads[ver] = (q.grad.clone(), k.grad.clone(), v.grad.clone())
    for a, b in zip(grads["v1"], grads["v3"]):
        assert rel_err(a, b) < 5e-3, rel_err(a, b)


def test_prefill_d64_forward():
    """head_dim-64 forward vs fp32 reference (qwen-small / llama3-1b class
    models take the packed path too)."""
    torch.manual_seed(44)
    Hq, Hk, D = 12, 4, 64
    lens = [70, 128, 5]
    total = sum(lens)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)),
                      dtype=torch.int32, device=DEV)
    scale = 1.0 / math.sqrt(D)
    q = (torch.randn(total, Hq, D, device=DEV) / 4).bfloat16()
    k = (torch.randn(total, Hk, D, device=DEV) / 4).bfloat16()
    v = (torch.randn(total, Hk, D, device=DEV) / 4).bfloat16()
    out = ops.varlen_prefill_attention(q, k, v, cu, cu, scale)
    expect = ref.varlen_prefill_attention(q.cpu(), k.cpu(), v.cpu(),
                                          cu.cpu(), cu.cpu(), scale)
    assert rel_err(out.cpu(), expect) < 2e-2


# -------------------------------------------- algo-pinned hipBLASLt linears


def test_tuned_linear_numerics():
    """tuned_linear fwd/dgrad/wgrad vs fp32 reference (gemm_tuned.cpp does
    an in-process algo search on first use per shape)."""
    torch.manual_seed(50)
    M, N, K = 1000, 512, 256     # deliberately odd M
    x = (torch.randn(M, K, device=DEV) / 4).bfloat16().requires_grad_()
    w = (torch.randn(N, K, device=DEV) / 4).bfloat16().requires_grad_()
    b = torch.randn(N, device=DEV).bfloat16().requires_grad_()
    y = ops.tuned_linear(x, w, b)
    g = torch.randn(M, N, device=DEV).bfloat16()
    y.backward(g)

    x2 = x.detach().float().requires_grad_()
    w2 = w.detach().float().requires_grad_()
    b2 = b.detach().float().requires_grad_()
    y2 = torch.nn.functional.linear(x2, w2, b2)
    y2.backward(g.float())
    assert rel_err(y.float(), y2.detach()) < 1e-2
    assert rel_err(x.grad.float(), x2.grad) < 1e-2
    assert rel_err(w.grad.float(), w2.grad) < 1e-2
    assert rel_err(b.grad.float(), b2.grad) < 1e-2
    # 3-D input path (padded layout)
    x3 = (torch.randn(4, 32, K, device=DEV) / 4).bfloat16()
    y3 = ops.tuned_linear(x3, w.detach())
    y3r = torch.nn.functional.linear(x3.float(), w.detach().float())
    assert rel_err(y3.float(), y3r) < 1e-2


def test_rmsnorm_train_fwd_bwd():
    """Fused trainer RMSNorm (+residual) fwd/bwd vs fp32 autograd ref."""
    torch.manual_seed(55)
    T, H = 777, 512
    x = (torch.randn(T, H, device=DEV) / 2).bfloat16().requires_grad_()
    res = (torch.randn(T, H, device=DEV) / 2).bfloat16().requires_grad_()
    w = torch.randn(H, device=DEV).bfloat16().requires_grad_()
    eps = 1e-6
    y, h = ops.fused_add_rmsnorm_train(x, res, w, eps)
    g = torch.randn(T, H, device=DEV)
    gh = torch.randn(T, H, device=DEV)
    (y.float() * g + h.float() * gh).sum().backward()

    x2 = x.detach().float().requires_grad_()
    r2 = res.detach().float().requires_grad_()
    w2 = w.detach().float().requires_grad_()
    h2 = x2 + r2
    y2 = torch.nn.functional.rms_norm(h2, (H,), None, eps) * w2
    (y2 * g + h2 * gh).sum().backward()
    assert rel_err(y.float(), y2.detach()) < 1e-2
    assert rel_err(h.float(), h2.detach()) < 1e-2
    assert rel_err(x.grad.float(), x2.grad) < 2e-2
    assert rel_err(res.grad.float(), r2.grad) < 2e-2
    assert rel_err(w.grad.float(), w2.grad) < 2e-2

    # no-residual variant
    xx = (torch.randn(T, H, device=DEV) / 2).bfloat16().requires_grad_()
    yy = ops.rmsnorm_train(xx, w.detach(), eps)
    yy.float().mul(g).sum().backward()
    xr = xx.detach().float().requires_grad_()
    yr = torch.nn.functional.rms_norm(xr, (H,), None, eps) * w.detach().float()
    yr.mul(g).sum().backward()
    assert rel_err(yy.float(), yr.detach()) < 1e-2
    assert rel_err(xx.grad.float(), xr.grad) < 2e-2


def test_tuned_mm_nt_decode_shapes():
    """Engine decode projection path: algo-pinned nt matmul at skinny M."""
    torch.manual_seed(56)
    for M, N, K in ((32, 6144, 4096), (128, 4096, 4096), (64, 512, 256)):
        x = (torch.randn(M, K, device=DEV) / 4).bfloat16()
        w = (torch.randn(N, K, device=DEV) / 4).bfloat16()
        y = ops.tuned_mm_nt(x, w)
        yr = (x.float() @ w.float().t())
        assert rel_err(y.float(), yr) < 1e-2, (M, N, K)


def test_rope_train_fwd_bwd():
    """Fused trainer RoPE vs the eager rotate-half composition + autograd."""
    torch.manual_seed(57)
    T, H, D = 333, 8, 128
    x = (torch.randn(T, H, D, device=DEV) / 2).bfloat16().requires_grad_()
    pos = torch.randint(0, 500, (T,), device=DEV)
    inv = 1.0 / (10000.0 ** (torch.arange(0, D, 2, device=DEV,
                                          dtype=torch.float32) / D))
    freqs = pos.float()[:, None] * inv[None, :]
    cos, sin = freqs.cos().contiguous(), freqs.sin().contiguous()
    y = ops.rope_train(x, cos, sin)
    g = torch.randn(T, H, D, device=DEV)
    (y.float() * g).sum().backward()

    x2 = x.detach().float().requires_grad_()
    c2 = cos.unsqueeze(1)
    s2 = sin.unsqueeze(1)
    d = D // 2
    y2 = torch.cat([x2[..., :d] * c2 - x2[..., d:] * s2,
                    x2[..., d:] * c2 + x2[..., :d] * s2], dim=-1)
    (y2 * g).sum().backward()
    assert rel_err(y.float(), y2.detach()) < 1e-2
    assert rel_err(x.grad.float(), x2.grad) < 1e-2


def test_fused_trainer_paths_update_equivalence(monkeypatch):
    """One actor update step with ALL fused trainer paths (norm, rope,
    tuned linears) vs the eager composition: logprobs and grad-norm must
    agree within bf16 noise — guards against silent training corruption
    from any fused kernel."""
    from polyrl_amd.config import ActorConfig
    from polyrl_amd.models import create_model
    from polyrl_amd.models.registry import DecoderConfig
    from polyrl_amd.protocol import TensorBatch
    from polyrl_amd.trainer.workers import ActorWorker

    cfg = DecoderConfig(arch="llama", vocab_size=512, hidden_size=256,
                        intermediate_size=512, num_hidden_layers=2,
                        num_attention_heads=4, num_key_value_heads=2,
                        head_dim=64, max_position_embeddings=256,
                        rope_theta=10000.0, rms_norm_eps=1e-6)
    torch.manual_seed(80)
    B, Lp, Lr = 6, 10, 8
    ids = torch.randint(0, cfg.vocab_size, (B, Lp + Lr))
    am = torch.ones(B, Lp + Lr, dtype=torch.long)
    am[0, :4] = 0
    pos = (torch.cumsum(am, 1) - 1).clamp(min=0)
    batch = TensorBatch(tensors={
        "input_ids": ids, "attention_mask": am, "position_ids": pos,
        "responses": ids[:, Lp:],
        "response_mask": torch.ones(B, Lr),
        "old_log_probs": torch.zeros(B, Lr),
        "advantages": torch.randn(B, Lr),
    })

    def run(fused):
        monkeypatch.setenv("POLYRL_FUSED_NORM", "1" if fused else "0")
        monkeypatch.setenv("POLYRL_TUNED_GEMM", "1" if fused else "0")
        torch.manual_seed(81)
        model = create_model(cfg, kind="actor", dtype="bfloat16", device=DEV)
        model.model.use_remove_padding = True
        acfg = ActorConfig()
        acfg.use_dynamic_bsz = False
        acfg.ppo_micro_batch_size_per_gpu = B
        w = ActorWorker(model, acfg, device=DEV)
        lp, _ = w.compute_log_prob(batch)
        m = w.update_policy_stream(batch, is_opt_step=True, is_lr_step=True,
                                   accum_scale=1.0)
        return lp, m["actor/grad_norm"][0]

    lp_f, gn_f = run(True)
    lp_e, gn_e = run(False)
    assert rel_err(lp_f, lp_e) < 5e-2, rel_err(lp_f, lp_e)
    assert abs(gn_f - gn_e) / max(gn_e, 1e-6) < 0.1, (gn_f, gn_e)


def test_gather_logprobs_train_fwd_bwd():
    """Fused training logprob gather (fwd lp+lse, streaming bwd) vs fp32
    autograd log_softmax-gather."""
    torch.manual_seed(58)
    N, V = 64, 32000
    logits = (torch.randn(N, V, device=DEV) * 3).bfloat16().requires_grad_()
    labels = torch.randint(0, V, (N,), device=DEV)
    lp = ops.gather_logprobs_train(logits, labels)
    g = torch.randn(N, device=DEV)
    (lp * g).sum().backward()

    l2 = logits.detach().float().requires_grad_()
    lp2 = torch.log_softmax(l2, -1).gather(-1, labels[:, None]).squeeze(-1)
    (lp2 * g).sum().backward()
    assert torch.allclose(lp, lp2.detach(), atol=1e-2, rtol=1e-3)
    # grads: bf16 vs fp32 reference — compare at bf16 tolerance, and the
    # onehot slot must carry the dominant term
    ge = l2.grad
    gf = logits.grad.float()
    assert rel_err(gf, ge) < 2e-2, rel_err(gf, ge)
    for i in range(0, N, 7):
        assert abs(gf[i, labels[i]] - ge[i, labels[i]]) < 2e-2


def test_silu_mul_train_fwd_bwd():
    torch.manual_seed(59)
    T, I = 500, 1024
    g = (torch.randn(T, I, device=DEV)).bfloat16().requires_grad_()
    u = (torch.randn(T, I, device=DEV)).bfloat16().requires_grad_()
    y = ops.silu_mul_train(g, u)
    w = torch.randn(T, I, device=DEV)
    (y.float() * w).sum().backward()
    g2 = g.detach().float().requires_grad_()
    u2 = u.detach().float().requires_grad_()
    y2 = torch.nn.functional.silu(g2) * u2
    (y2 * w).sum().backward()
    assert rel_err(y.float(), y2.detach()) < 1e-2
    assert rel_err(g.grad.float(), g2.grad) < 2e-2
    assert rel_err(u.grad.float(), u2.grad) < 2e-2


def test_silu_mul_train_3d():
    """Padded-layout (B, L, I) inputs flatten inside the Function."""
    torch.manual_seed(60)
    g = torch.randn(3, 17, 344, device=DEV).bfloat16().requires_grad_()
    u = torch.randn_like(g).requires_grad_()
    y = ops.silu_mul_train(g, u)
    assert y.shape == g.shape
    y.float().sum().backward()
    assert g.grad.shape == g.shape and torch.isfinite(g.grad.float()).all()

"""The trainer's packed rows: maps of padded batches, hidden rows at the places
asked for, the embedding's gradient."""
import numpy as np
import pytest
import torch

import polyrl_amd.ops as ops
from polyrl_amd.models import get_model_config
from polyrl_amd.models.llama import CausalLM

pytestmark = pytest.mark.gpu
DEV = "cuda"


def gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def masks(kind, b, l):
    if kind == "left":
        n = torch.randint(0, l + 1, (b, 1), generator=gen(b), device=DEV)
        return torch.arange(l, device=DEV)[None] >= l - n
    if kind == "all":
        return torch.ones(b, l, dtype=torch.bool, device=DEV)
    return torch.rand(b, l, generator=gen(l), device=DEV) < 0.6


@pytest.mark.parametrize("kind", ["left", "all", "holes"])
@pytest.mark.parametrize("b,l,lo,hi", [
    (1, 1, 0, 1), (3, 255, 0, 255), (5, 256, 100, 256), (4, 257, 255, 257),
    (2, 700, 300, 300), (33, 65, 1, 64)])
def test_maps(kind, b, l, lo, hi):
    """Rows of one stretch of threads, of several and a remainder; rows without
    a token; no place, some and all."""
    m = masks(kind, b, l)
    m[0, -1] = True                                # (a token at least)
    ids = torch.randint(1, 999, (b, l), generator=gen(1), device=DEV)
    pos = torch.randint(0, 5000, (b, l), generator=gen(2), device=DEV)
    ext = ops._require_ext()
    lens, most = ext.pack_lengths(m, pos).tolist()
    assert lens == m.sum(-1).tolist()
    assert most == pos.masked_fill(~m, -1).amax(-1).tolist()
    total, pad = sum(lens), 7
    cu, tiles = ops.packed_tables(lens + [pad], DEV)
    want = torch.tensor([0] + lens + [pad]).cumsum(0)
    assert cu.tolist() == want.tolist()
    for got, ref in zip(tiles, ops.build_varlen_tiles(want, DEV)):
        assert torch.equal(got, ref)
    ids_p, pos_p, packed, place = ext.pack_rows(m, ids, pos, cu, total,
                                                total + pad, lo, hi)
    assert torch.equal(ids_p[:total], ids[m]) and not ids_p[total:].any()
    assert torch.equal(pos_p[:total], pos[m])
    assert pos_p[total:].tolist() == list(range(pad))
    number = torch.full((b, l), -1, dtype=torch.int32, device=DEV)
    number[m] = torch.arange(total, dtype=torch.int32, device=DEV)
    assert torch.equal(packed, number[:, lo:hi])
    back = torch.full((total + pad,), -1, dtype=torch.int32, device=DEV)
    flat = packed.reshape(-1)
    live = flat >= 0
    back[flat[live].long()] = torch.arange(len(flat), dtype=torch.int32,
                                           device=DEV)[live]
    assert torch.equal(place, back)

    x = torch.randn(total + pad, 24, generator=gen(3), device=DEV) \
        .bfloat16().requires_grad_()
    out = ops.rows_from_packed(x, packed, place)
    ref = x.detach()[packed.long().clamp(min=0)] * live.view(b, -1, 1)
    assert torch.equal(out, ref)
    dout = torch.randn(out.shape, generator=gen(4), device=DEV).bfloat16()
    out.backward(dout)
    dx = torch.zeros_like(x)
    dx[flat[live].long()] = dout.reshape(-1, 24)[live]
    assert torch.equal(x.grad, dx)


@pytest.mark.parametrize("t,v,h", [
    (1, 1, 8), (31, 3, 24), (32, 1, 8), (33, 1, 40), (64, 2, 2048),
    (255, 9, 2056), (1000, 40, 4104), (1025, 5000, 64), (3000, 7, 16),
    (32768, 4000, 8)])
def test_embed_grad(t, v, h):
    """Ids of one row and of thousands, sums that end with a window of 32 rows
    and go on through many, rows of ids that no token has."""
    ids = torch.randint(v, (t,), generator=gen(t), device=DEV)
    dy = torch.randn(t, h, generator=gen(h), device=DEV).bfloat16()
    w = torch.randn(v, h, generator=gen(5), device=DEV).bfloat16() \
        .requires_grad_()
    out = ops.embed_train(ids, w)
    assert torch.equal(out, w.detach()[ids])
    out.backward(dy)
    zero = torch.zeros(v, h, dtype=torch.float64, device=DEV)
    want = zero.index_add(0, ids, dy.double())
    mass = zero.index_add(0, ids, dy.double().abs())
    # 32-bit sums of at most t rows and one rounding to bf16
    bound = 2 ** -8 * want.abs() + t * 2.0 ** -24 * mass
    assert ((w.grad.double() - want).abs() <= bound).all()


def test_gradients_anywhere():
    """Gradients that are a part of a buffer, at an address of no whole word, and
    strided ones."""
    ids = torch.tensor([3, 0, 3, 2], device=DEV)
    place = torch.tensor([2, 0, -1, 3], dtype=torch.int32, device=DEV)
    packed = torch.tensor([[1, -1], [0, 3]], dtype=torch.int32, device=DEV)
    flat = torch.randn(4 * 24 + 1, generator=gen(1), device=DEV).bfloat16()
    for g in (flat[1:].view(4, 24), flat[:-1].view(24, 4).t()):
        w = torch.randn(5, 24, device=DEV).bfloat16().requires_grad_()
        ops.embed_train(ids, w).backward(g)
        want = torch.zeros(5, 24, device=DEV).index_add(0, ids, g.float())
        assert torch.equal(w.grad, want.bfloat16())
        x = g.detach().requires_grad_()
        out = ops.rows_from_packed(x, packed, place)
        assert torch.equal(out.view(4, 24)[[2, 0, 3]], g[[0, 1, 3]])
        out.backward(g.view(2, 2, 24) if g.is_contiguous() else
                     g.reshape(2, 2, 24))
        assert torch.equal(x.grad[[0, 1, 3]], g[[2, 0, 3]])
        assert not x.grad[2].any() and not out[0, 1].any()


@pytest.mark.parametrize("rows", [slice(-41, -1), slice(None), slice(3, 50, 2), slice(60, 61),
                                  None, -1, [7, 3, 80], np.array([5, 5]),
                                  torch.arange(90) % 3 == 0])
def test_model(rows):
    """A model's logits and gradients against the same with boolean indices: of the
    places of a slice, or of whatever else indexes a dimension."""
    torch.manual_seed(0)
    cfg = get_model_config("llama-tiny")
    m = CausalLM(cfg).to(DEV, torch.bfloat16).train()
    m.model.use_remove_padding = True
    b, l = 5, 90
    mask = masks("left", b, l)
    mask[0] = True
    mask[2, 40:47] = False
    ids = torch.randint(cfg.vocab_size, (b, l), generator=gen(6), device=DEV)
    pos = (mask.long().cumsum(-1) - 1).clamp_(min=0)

    def run():
        out = m(ids, attention_mask=mask, position_ids=pos, logits_slice=rows)
        g = torch.randn(out.shape, generator=gen(7), device=DEV).bfloat16()
        params = list(m.parameters())
        return [out.detach()] + list(torch.autograd.grad(
            out, params, g, allow_unused=True))

    got = run()
    with pytest.MonkeyPatch.context() as p:
        p.setattr(type(m.model), "_pack_gpu", lambda *a: None)
        p.setattr(type(m.model), "_embed", lambda s, i: s.embed_tokens(i))
        want = run()
    assert len(got) == len(want) and torch.equal(got[0], want[0])
    for a, b_ in zip(got[1:], want[1:]):
        if a is None or b_ is None:
            assert a is b_
            continue
        # 32-bit sums in another order, rounded to bf16
        a, b_ = a.double(), b_.double()
        assert (a - b_).norm() <= 2 ** -8 * b_.norm() + 1e-30


def test_checkpointing():
    """A packed step whose layers are computed again on the way back."""
    torch.manual_seed(0)
    cfg = get_model_config("llama-tiny")
    m = CausalLM(cfg).to(DEV, torch.bfloat16).train()
    m.model.use_remove_padding = True
    mask = masks("left", 5, 90)
    ids = torch.randint(cfg.vocab_size, (5, 90), generator=gen(6), device=DEV)
    pos = (mask.long().cumsum(-1) - 1).clamp_(min=0)

    def run():
        out = m(ids, attention_mask=mask, position_ids=pos,
                logits_slice=slice(-41, -1))
        return [out.detach()] + list(torch.autograd.grad(
            out.float().square().sum(), list(m.parameters())))
    want = run()
    m.gradient_checkpointing_enable()
    assert m.model.gradient_checkpointing
    for a, b in zip(run(), want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("how", ["forward", "hook", "global"])
def test_embedding_with_more(how, monkeypatch):
    """An embedding whose forward was replaced, or that hooks watch, is called."""
    cfg = get_model_config("llama-tiny")
    m = CausalLM(cfg).to(DEV, torch.bfloat16)
    m.model.use_remove_padding = True
    emb, ran = m.model.embed_tokens, []
    fused = []
    monkeypatch.setattr(ops, "embed_train",
                        lambda ids, w: fused.append(1) or w[ids])
    ids = torch.arange(12, device=DEV).view(2, 6)

    def step():
        m(ids, attention_mask=torch.ones_like(ids),
          position_ids=ids % 6)

    def hook(mod, *_):
        if mod is emb:
            ran.append(1)
    step()
    assert fused == [1] and not ran
    if how == "forward":
        plain = emb.forward
        emb.forward = lambda x: ran.append(1) or plain(x)
    elif how == "hook":
        emb.register_forward_hook(hook)
    else:
        handle = torch.nn.modules.module.register_module_forward_hook(hook)
    try:
        step()
    finally:
        if how == "global":
            handle.remove()
    assert fused == ran == [1]
    if how == "global":
        step()
        assert fused == [1, 1] and ran == [1]

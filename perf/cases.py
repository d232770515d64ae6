"""The work that users of this framework have it do, as measurable cases.

Each case is one pass through public entry points: the attention, sampling
and log-probability ops that rollouts and PPO updates are made of
(``polyrl_amd.ops``, ``polyrl_amd.ops.seq``), a whole actor micro-step
(``polyrl_amd.models.llama.CausalLM`` forward and backward, as the trainer's
workers call it) and a prompt step of the rollout engine
(``polyrl_amd.rollout.engine.Engine.step_forced``).  Head counts, widths and
vocabularies are those of the model registry; lengths and batches are those
of the default benchmark (16 prompts x 8 samples of 256 + 256 tokens), its
engine comparison (8 x 2048 prompts, 64 decode rows) and long contexts up to
the registry's 8192 positions.

``kind`` says which path a case takes:

decode_attention   one new token per running request against paged K/V
prompt_attention   causal attention of packed prompts (``hist`` tokens of each
                   already cached: a later portion of a chunked prompt)
train_attention    packed causal attention, forward and backward
window_attention   grouped-query window attention over paged rows (hybrids)
sample             next tokens and their log-probabilities from logits
logprob            label log-probabilities: forward and backward, or (without
                   ``grad``) forward with entropies
actor_step         log-probabilities of responses and all weight gradients
prompt_step        an engine step over whole prompts, logits of the last rows
"""
import math
import random

import torch

import polyrl_amd.ops as ops
from polyrl_amd.models import get_model_config
from polyrl_amd.models.llama import CausalLM
from polyrl_amd.rollout.engine import Engine

DEV = "cuda"
PAGE = 16
BF16 = torch.bfloat16

# (query heads, key/value heads, head size) of the registry's dense decoders
HEADS = ((32, 8, 128), (12, 2, 128), (28, 4, 128), (64, 8, 128), (32, 8, 64),
         (16, 4, 64))
# and of the hybrid presets' grouped-query layers
HYBRID_HEADS = ((16, 4, 64), (32, 8, 64), (32, 8, 128))
VOCABS = (32000, 50257, 128256, 151936, 152064)
# (model, layers, most tokens) of the actor micro-steps and prompt steps
ACTORS = (("llama-400m", 6, 8192), ("llama3-1b", 3, 8192),
          ("qwen2.5-1.5b", 3, 4096), ("llama3-8b", 2, 8192))
SERVED = (("llama-400m", 12), ("llama3-1b", 8), ("qwen2.5-1.5b", 8))


def listed():
    return [
        # one request being decoded early on: latency of the smallest call
        dict(name="decode-one", kind="decode_attention", rows=1, low=37,
             high=37, hq=12, hk=2, d=128),
        # the benchmark's decode batch: 128 samples, prompt plus some response
        dict(name="decode-batch", kind="decode_attention", rows=128, low=257,
             high=512, hq=32, hk=8, d=128),
        # long responses: few rows, thousands of cached tokens each
        dict(name="decode-long", kind="decode_attention", rows=33, low=1900,
             high=8192, hq=28, hk=4, d=128),
        # prompts of an engine step, ragged
        dict(name="prompts", kind="prompt_attention", rows=8, low=1200,
             high=2048, hist=0, hq=32, hk=8, d=64),
        # one trainer micro-batch: 16 sequences of at most 512 tokens
        dict(name="train-512", kind="train_attention", rows=16, low=300,
             high=512, hq=32, hk=8, d=128),
        # long-response training: few sequences of thousands of tokens
        dict(name="train-4k", kind="train_attention", rows=2, low=3500,
             high=4096, hq=28, hk=4, d=128),
        # prompts through a hybrid decoder's window layer
        dict(name="window-prompts", kind="window_attention", rows=8, low=1200,
             high=2048, window=1024, keep=4, sink=False, hq=32, hk=8, d=64),
        # the benchmark's sampler call: temperature 1, no filter
        dict(name="sample-plain", kind="sample", rows=128, vocab=128256,
             temperature=1.0, top_k=-1, top_p=1.0, f32=False),
        # served requests with both filters
        dict(name="sample-filtered", kind="sample", rows=64, vocab=151936,
             temperature=0.7, top_k=50, top_p=0.9, f32=False),
        # responses of one trainer micro-batch against the vocabulary
        dict(name="logprob-train", kind="logprob", rows=4096, vocab=128256,
             grad=True),
        # forward and backward of the actor on one micro-batch (two layers of
        # the 8B stack, embedding and vocabulary whole)
        dict(name="actor-step", kind="actor_step", model="llama3-8b",
             layers=2, rows=16, prompt_low=100, prompt=256, response=256),
        # an engine step over fresh prompts of a small model
        dict(name="prompt-step", kind="prompt_step", model="llama-400m",
             layers=12, rows=16, low=130, high=512),
    ]


def _log(rng, low, high):
    """A whole number in [low, high], spread over its logarithm."""
    return min(high, max(low, round(math.exp(
        rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng):
    kind = rng.choice(("decode_attention", "prompt_attention",
                       "train_attention", "window_attention", "sample",
                       "logprob", "actor_step", "prompt_step"))
    if kind == "decode_attention":
        hq, hk, d = rng.choice(HEADS)
        high = _log(rng, 16, 8192)
        rows = _log(rng, 1, max(1, min(256, 33 * 8192 * 4 // (high * hk))))
        return dict(kind=kind, rows=rows, low=rng.randint(high // 4 + 1, high),
                    high=high, hq=hq, hk=hk, d=d)
    if kind in ("prompt_attention", "train_attention"):
        hq, hk, d = rng.choice(HEADS)
        high = _log(rng, 16, 4096)
        rows = _log(rng, 1, max(1, min(64, 8192 // high)))
        case = dict(kind=kind, rows=rows,
                    low=rng.randint(high // 4 + 1, high), high=high, hq=hq,
                    hk=hk, d=d)
        if kind == "prompt_attention":
            case["hist"] = rng.choice((0, 0, _log(rng, 16, 2048)))
        return case
    if kind == "window_attention":
        hq, hk, d = rng.choice(HYBRID_HEADS)
        high = _log(rng, 32, 4096)
        rows = _log(rng, 1, max(1, min(32, 16384 // high)))
        return dict(kind=kind, rows=rows, low=rng.randint(high // 4 + 1, high),
                    high=high, window=rng.choice((512, 1024, 2048)),
                    keep=rng.choice((0, 4)), sink=rng.random() < 0.5, hq=hq,
                    hk=hk, d=d)
    if kind == "sample":
        vocab = rng.choice(VOCABS)
        rows = _log(rng, 1, 256)
        top_k, top_p = rng.choice(((-1, 1.0), (-1, 1.0), (50, 1.0), (20, 0.8),
                                   (-1, 0.95), (50, 0.9)))
        f32 = rng.random() < 0.25
        if top_k > 0 or top_p < 1.0:
            rows = min(rows, 64)
        return dict(kind=kind, rows=rows, vocab=vocab,
                    temperature=rng.choice((1.0, 1.0, 0.7, 0.0)),
                    top_k=top_k, top_p=top_p, f32=f32)
    if kind == "logprob":
        vocab = rng.choice(VOCABS)
        return dict(kind=kind, rows=_log(rng, 16, 4096 * 128256 // max(
            vocab, 128256)), vocab=vocab, grad=rng.random() < 0.7)
    if kind == "actor_step":
        model, layers, most = rng.choice(ACTORS)
        length = _log(rng, 128, 1024)
        rows = _log(rng, 1, max(1, most // (2 * length)))
        return dict(kind=kind, model=model, layers=layers, rows=rows,
                    prompt_low=rng.randint(length // 4, length),
                    prompt=length, response=rng.randint(length // 4, length))
    model, layers = rng.choice(SERVED)
    high = _log(rng, 24, 2048)
    rows = _log(rng, 1, max(1, min(32, 4096 // high)))
    return dict(kind=kind, model=model, layers=layers, rows=rows,
                low=rng.randint(high // 2, high), high=high)


# ------------------------------------------------------------------ helpers


def _lens(case, low="low", high="high"):
    """The sequences' lengths: whole numbers in [low, high], the longest
    among them, the same for every seed (they set a pass's work)."""
    r = random.Random("%d %d %d" % (case["rows"], case[low], case[high]))
    out = [r.randint(case[low], case[high]) for _ in range(case["rows"])]
    out[r.randrange(len(out))] = case[high]
    return out


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, *shape, dtype=BF16):
    return torch.randn(*shape, generator=g, device=DEV).to(dtype)


def _cu(lens):
    out = [0]
    for n in lens:
        out.append(out[-1] + n)
    return torch.tensor(out, dtype=torch.int32)


def _page_table(lens, g):
    """Shuffled pages for every sequence, (rows, most pages) int32."""
    need = [-(-n // PAGE) for n in lens]
    perm = torch.randperm(sum(need), generator=g, device=DEV).int()
    table = torch.zeros(len(lens), max(need), dtype=torch.int32, device=DEV)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = perm[at:at + n]
        at += n
    return table, sum(need)


def _qkv(case, g, tokens, kv_tokens=None):
    """Query, key and value heads as views into one projection's rows, the
    way the model's forward hands them on."""
    hq, hk, d = case["hq"], case["hk"], case["d"]
    if kv_tokens is None:
        row = _normal(g, tokens, (hq + 2 * hk) * d)
        return (row[:, :hq * d].unflatten(1, (hq, d)),
                row[:, hq * d:(hq + hk) * d].unflatten(1, (hk, d)),
                row[:, (hq + hk) * d:].unflatten(1, (hk, d)))
    return (_normal(g, tokens, hq, d), _normal(g, kv_tokens, hk, d),
            _normal(g, kv_tokens, hk, d))


def _model(case):
    return get_model_config(case["model"],
                            {"num_hidden_layers": case["layers"]})


# ---------------------------------------------------------- prepare and run


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    st = {"case": case}
    if kind == "decode_attention":
        lens = _lens(case)
        hq, hk, d = case["hq"], case["hk"], case["d"]
        st["ptab"], pages = _page_table(lens, g)
        st["k"] = _normal(g, pages, PAGE, hk, d)
        st["v"] = _normal(g, pages, PAGE, hk, d)
        st["q"] = _normal(g, case["rows"], (hq + 2 * hk) * d)[
            :, :hq * d].unflatten(1, (hq, d))
        st["lens"] = torch.tensor(lens, dtype=torch.int32, device=DEV)
    elif kind == "prompt_attention":
        lens = _lens(case)
        klens = [n + case["hist"] for n in lens]
        st["cu_q"], st["cu_k"] = _cu(lens).to(DEV), _cu(klens).to(DEV)
        st["qkv"] = _qkv(case, g, sum(lens),
                         sum(klens) if case["hist"] else None)
    elif kind == "train_attention":
        lens = _lens(case)
        cu = _cu(lens)
        st["cu"] = cu.to(DEV)
        st["tiles"] = ops.build_varlen_tiles(cu, DEV)
        st["qkv"] = tuple(t.contiguous().requires_grad_()
                          for t in _qkv(case, g, sum(lens)))
        st["dout"] = _normal(g, sum(lens), case["hq"], case["d"])
    elif kind == "window_attention":
        lens = _lens(case)
        hq, hk, d = case["hq"], case["hk"], case["d"]
        i32 = dict(dtype=torch.int32, device=DEV)
        st["ptab"], pages = _page_table(lens, g)
        st["rows"] = _normal(g, pages, PAGE, 2 * hk * d)
        st["q"] = _normal(g, sum(lens), hq * d)
        st["seq"] = torch.repeat_interleave(
            torch.arange(len(lens), **i32), torch.tensor(lens, device=DEV))
        st["pos"] = torch.cat([torch.arange(n, **i32) for n in lens])
        st["tiles"] = ops.seq.attention_tiles(lens, DEV)
        st["sink"] = _normal(g, hq, dtype=torch.float32) if case["sink"] \
            else None
    elif kind == "sample":
        n = case["rows"]
        st["logits"] = _normal(g, n, case["vocab"], dtype=torch.float32) \
            .mul_(2.5).to(torch.float32 if case["f32"] else BF16)
        st["temp"] = torch.full((n,), case["temperature"], device=DEV)
        st["top_k"] = torch.full((n,), case["top_k"], dtype=torch.int32,
                                 device=DEV)
        st["top_p"] = torch.full((n,), case["top_p"], device=DEV)
        st["seed"] = seed
        st["no_filter"] = case["top_k"] <= 0 and case["top_p"] >= 1.0
    elif kind == "logprob":
        n, v = case["rows"], case["vocab"]
        st["logits"] = _normal(g, n, v).mul_(2.5).requires_grad_(case["grad"])
        st["labels"] = torch.randint(v, (n,), generator=g, device=DEV)
        st["dlp"] = _normal(g, n, dtype=torch.float32)
    elif kind == "actor_step":
        cfg = _model(case)
        with torch.device("meta"):
            m = CausalLM(cfg)
        m = m.to(BF16).to_empty(device=DEV)
        if cfg.tie_word_embeddings:
            m.lm_head.weight = m.model.embed_tokens.weight
        with torch.no_grad():
            for name, p in m.named_parameters():
                if "norm" in name:
                    p.fill_(1.0)
                else:
                    p.normal_(0, 0.02, generator=g)
        m.model.rotary = type(m.model.rotary)(cfg.head_dim, cfg.rope_theta)
        m.model.use_remove_padding = True
        st["model"] = m.train()
        b, lp, lr = case["rows"], case["prompt"], case["response"]
        lens = torch.tensor(_lens(case, "prompt_low", "prompt"), device=DEV)
        st["ids"] = torch.randint(cfg.vocab_size, (b, lp + lr), generator=g,
                                  device=DEV)
        st["mask"] = torch.arange(lp + lr, device=DEV)[None] >= \
            (lp - lens)[:, None]
        st["pos"] = (st["mask"].long().cumsum(-1) - 1).clamp_(min=0)
        st["coef"] = _normal(g, b, lr, dtype=torch.float32) / (b * lr)
    else:
        cfg = _model(case)
        lens = _lens(case)
        eng = Engine(cfg, device=DEV, dtype=BF16, page_size=PAGE,
                     kv_token_capacity=sum(lens) + PAGE * len(lens),
                     max_running_requests=len(lens))
        sd = {}
        for name, t in _served_shapes(cfg).items():
            norm = name.endswith("norm.weight")
            sd[name] = torch.ones(*t, device=DEV, dtype=BF16) if norm else \
                torch.randn(*t, generator=g, device=DEV).mul_(0.02).to(BF16)
        eng.model.load_state_dict(sd)
        st["engine"], st["weights"] = eng, sd
        ids = torch.randint(cfg.vocab_size, (sum(lens),), generator=g,
                            device=DEV).tolist()
        cu = _cu(lens).tolist()
        st["prompts"] = [("r%d" % i, ids[cu[i]:cu[i + 1]], [lens[i] - 1])
                         for i in range(len(lens))]
        st["rids"] = [p[0] for p in st["prompts"]]
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "decode_attention":
        return ops.paged_attention_decode(st["q"], st["k"], st["v"],
                                          st["ptab"], st["lens"],
                                          case["d"] ** -0.5)
    if kind == "prompt_attention":
        return ops.varlen_prefill_attention(*st["qkv"], st["cu_q"],
                                            st["cu_k"], case["d"] ** -0.5,
                                            causal=True)
    if kind == "train_attention":
        out = ops.flash_attn_varlen(*st["qkv"], st["cu"], case["d"] ** -0.5,
                                    causal=True, tiles=st["tiles"])
        return (out.detach(),) + torch.autograd.grad(out, st["qkv"],
                                                     st["dout"])
    if kind == "window_attention":
        return ops.seq.gqa_window_attention(
            st["q"], st["rows"], st["ptab"], st["seq"], st["pos"], case["hq"],
            case["hk"], case["d"], case["d"], case["window"], case["keep"],
            None, None, None, case["d"] ** -0.5, BF16, tiles=st["tiles"],
            sink=st["sink"])
    if kind == "sample":
        return ops.sample(st["logits"], st["temp"], st["top_k"], st["top_p"],
                          st["seed"], no_filter=st["no_filter"])
    if kind == "logprob":
        if not case["grad"]:
            return ops.gather_logprobs(st["logits"], st["labels"],
                                       want_entropy=True)
        lp = ops.gather_logprobs_train(st["logits"], st["labels"])
        return (lp.detach(),) + torch.autograd.grad(lp, st["logits"],
                                                    st["dlp"])
    if kind == "actor_step":
        m, lr = st["model"], case["response"]
        logits = m(st["ids"], attention_mask=st["mask"],
                   position_ids=st["pos"], logits_slice=slice(-lr - 1, -1))
        lp = ops.gather_logprobs_train(
            logits.reshape(-1, logits.shape[-1]),
            st["ids"][:, -lr:].reshape(-1)).view(-1, lr)
        grads = torch.autograd.grad((lp * st["coef"]).sum(),
                                    list(m.parameters()))
        return (lp.detach(),) + grads
    return st["engine"].step_forced(st["prompts"], end=st["rids"])


# ----------------------------------------------------------- work, tolerance


def _pairs(case, lens):
    """(query, key) pairs that a causal pass over these lengths scores."""
    w = case.get("window", 1 << 30)
    total = 0
    for n in lens:
        h = case.get("hist", 0)
        if n <= w:
            total += n * (n + 1) // 2 + n * h
        else:
            total += w * (w + 1) // 2 + (n - w) * (w + case["keep"])
    return total


def _dense_flops(cfg, tokens, pairs, head_rows):
    h, hd = cfg.hidden_size, cfg.head_dim
    att = (2 * cfg.num_attention_heads + 2 * cfg.num_key_value_heads) * hd
    per = 2 * (h * att + 3 * h * cfg.intermediate_size)
    return cfg.num_hidden_layers * (
        per * tokens + 4 * pairs * cfg.num_attention_heads * hd) \
        + 2 * head_rows * h * cfg.vocab_size


def _weight_bytes(cfg, embed_rows):
    h, hd = cfg.hidden_size, cfg.head_dim
    att = (2 * cfg.num_attention_heads + 2 * cfg.num_key_value_heads) * hd
    return 2 * (cfg.num_hidden_layers * (h * att + 3 * h
                                         * cfg.intermediate_size)
                + cfg.vocab_size * h + embed_rows * h)


def work(case):
    kind = case["kind"]
    if kind == "decode_attention":
        lens = _lens(case)
        hq, hk, d = case["hq"], case["hk"], case["d"]
        return {"bytes": sum(lens) * 4 * hk * d + len(lens) * 4 * hq * d,
                "flops": 4 * sum(lens) * hq * d}
    if kind in ("prompt_attention", "train_attention", "window_attention"):
        lens = _lens(case)
        hq, hk, d = case["hq"], case["hk"], case["d"]
        n = sum(lens)
        nk = n + len(lens) * case.get("hist", 0)
        flops = 4 * _pairs(case, lens) * hq * d
        if kind == "train_attention":
            # forward; backward reads q, k, v, dout again and writes three
            return {"bytes": 2 * d * (n * 5 * hq + nk * 6 * hk),
                    "flops": flops * 3.5}
        return {"bytes": 4 * d * (n * hq + nk * hk), "flops": flops}
    if kind == "sample":
        return {"bytes": case["rows"] * (case["vocab"]
                                         * (4 if case["f32"] else 2) + 24),
                "flops": 0}
    if kind == "logprob":
        n, v = case["rows"], case["vocab"]
        return {"bytes": n * v * (4 if case["grad"] else 2) + 20 * n,
                "flops": 0}
    cfg = _model(case)
    if kind == "actor_step":
        lens = [n + case["response"]
                for n in _lens(case, "prompt_low", "prompt")]
        flops = 3 * _dense_flops(cfg, sum(lens), _pairs(case, lens),
                                 case["rows"] * case["response"])
        return {"bytes": 2 * _weight_bytes(cfg, cfg.vocab_size),
                "flops": flops}
    lens = _lens(case)
    return {"bytes": _weight_bytes(cfg, sum(lens)) + sum(lens) * 4
            * cfg.num_hidden_layers * cfg.num_key_value_heads * cfg.head_dim,
            "flops": _dense_flops(cfg, sum(lens), _pairs(case, lens),
                                  len(lens))}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        # the draw is a function of logits, seed and row; log-probabilities
        # are 32-bit sums over the vocabulary
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.0}
    if kind == "logprob":
        # 16-bit gradients against 64-bit ones: 1e-3
        return {"rel": 4e-3} if case["grad"] else {"rel": 2e-5, "max": 1e-4}
    if kind in ("actor_step", "prompt_step"):
        # activations rounded to 16 bits after every op: 1e-2 to 3e-2
        return {"rel": 3e-2}
    return {"rel": 1e-2}        # 16-bit results and weights: 2.5e-3


# -------------------------------------------------------------------- exact


def _attend(q, k, v, live, scale, sink=None):
    """(heads, rows, d) queries over (heads, keys, d): softmax attention of
    64-bit numbers; ``sink`` adds exp(sink) to each head's denominator."""
    s = (q @ k.transpose(1, 2) * scale).masked_fill_(~live, -math.inf)
    if sink is not None:
        z = torch.cat([s, sink.double()[:, None, None].expand(
            -1, s.shape[1], 1)], -1)
        return torch.softmax(z, -1)[..., :-1] @ v
    return torch.softmax(s, -1) @ v


def _sequence(q, k, v, hist, scale, window=None, keep=0, sink=None):
    """One sequence's causal attention, (rows, heads, d) in 64 bits; the rows
    stand at the end of the keys."""
    hq, hk = q.shape[1], k.shape[1]
    i = torch.arange(q.shape[0], device=q.device)[:, None] + hist
    j = torch.arange(k.shape[0], device=q.device)[None]
    live = j <= i
    if window is not None:
        live &= (i - j < window) | (j < keep)
    out = []
    for h in range(hk):
        at = slice(h * (hq // hk), (h + 1) * (hq // hk))
        n = hq // hk
        out.append(_attend(
            q[:, at].transpose(0, 1), k[None, :, h].expand(n, -1, -1),
            v[None, :, h].expand(n, -1, -1), live, scale,
            None if sink is None else sink[at]).transpose(0, 1))
    return torch.cat(out, 1)


def _rope(x, pos, theta):
    """Rotate-half rotary embedding of (..., tokens, heads, d), pairs
    (i, i + d/2)."""
    half = x.shape[-1] // 2
    inv = theta ** (-torch.arange(half, device=x.device).double() / half)
    a = (pos.double()[..., None] * inv).unsqueeze(-2)
    c, s = a.cos(), a.sin()
    p, r = x[..., :half], x[..., half:]
    return torch.cat([p * c - r * s, r * c + p * s], -1)


def _rms(x, w, eps):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * w


def _decoder(cfg, w, ids, pos, live):
    """Hidden rows (batch, length, width) of the dense decoder in 64 bits,
    from weights by their checkpoint names."""
    b, n = ids.shape
    hq, hk, d = (cfg.num_attention_heads, cfg.num_key_value_heads,
                 cfg.head_dim)
    x = w["model.embed_tokens.weight"][ids]
    for i in range(cfg.num_hidden_layers):
        at = "model.layers.%d." % i

        def lin(name, y):
            y = y @ w[at + name + ".weight"].t()
            bias = w.get(at + name + ".bias")
            return y if bias is None else y + bias

        y = _rms(x, w[at + "input_layernorm.weight"], cfg.rms_norm_eps)
        q = _rope(lin("self_attn.q_proj", y).view(b, n, hq, d), pos,
                  cfg.rope_theta).transpose(1, 2)
        k = _rope(lin("self_attn.k_proj", y).view(b, n, hk, d), pos,
                  cfg.rope_theta).transpose(1, 2)
        v = lin("self_attn.v_proj", y).view(b, n, hk, d).transpose(1, 2)
        k = k.repeat_interleave(hq // hk, 1)
        v = v.repeat_interleave(hq // hk, 1)
        s = (q @ k.transpose(2, 3) * d ** -0.5).masked_fill(
            ~live[:, None], -math.inf)
        o = (torch.softmax(s, -1) @ v).transpose(1, 2).reshape(b, n, hq * d)
        x = x + lin("self_attn.o_proj", o)
        y = _rms(x, w[at + "post_attention_layernorm.weight"],
                 cfg.rms_norm_eps)
        gate = lin("mlp.gate_proj", y)
        x = x + lin("mlp.down_proj",
                    gate * torch.sigmoid(gate) * lin("mlp.up_proj", y))
    return _rms(x, w["model.norm.weight"], cfg.rms_norm_eps)


def _served_shapes(cfg):
    h, i, d = cfg.hidden_size, cfg.intermediate_size, cfg.head_dim
    nq, nk = cfg.num_attention_heads * d, cfg.num_key_value_heads * d
    out = {"model.embed_tokens.weight": (cfg.vocab_size, h)}
    for li in range(cfg.num_hidden_layers):
        at = "model.layers.%d." % li
        out.update({at + "self_attn.q_proj.weight": (nq, h),
                    at + "self_attn.k_proj.weight": (nk, h),
                    at + "self_attn.v_proj.weight": (nk, h),
                    at + "self_attn.o_proj.weight": (h, nq),
                    at + "mlp.gate_proj.weight": (i, h),
                    at + "mlp.up_proj.weight": (i, h),
                    at + "mlp.down_proj.weight": (h, i),
                    at + "input_layernorm.weight": (h,),
                    at + "post_attention_layernorm.weight": (h,)})
        if cfg.attention_bias:
            out.update({at + "self_attn.q_proj.bias": (nq,),
                        at + "self_attn.k_proj.bias": (nk,),
                        at + "self_attn.v_proj.bias": (nk,)})
    out["model.norm.weight"] = (h,)
    if not cfg.tie_word_embeddings:
        out["lm_head.weight"] = (cfg.vocab_size, h)
    return out


def exact(case, seed):
    st = prepare(case, seed)
    kind = case["kind"]
    if kind == "decode_attention":
        hq, hk, d = case["hq"], case["hk"], case["d"]
        out = []
        for i, n in enumerate(_lens(case)):
            pages = st["ptab"][i, :-(-n // PAGE)].long()
            k = st["k"][pages].view(-1, hk, d)[:n].double()
            v = st["v"][pages].view(-1, hk, d)[:n].double()
            q = st["q"][i].double().view(hk, hq // hk, d)
            s = torch.softmax(q @ k.permute(1, 2, 0) * d ** -0.5, -1)
            out.append((s @ v.transpose(0, 1)).reshape(hq, d))
        return torch.stack(out)
    if kind == "prompt_attention":
        q, k, v = (t.double() for t in st["qkv"])
        cq, ck = st["cu_q"].tolist(), st["cu_k"].tolist()
        return torch.cat([_sequence(
            q[cq[i]:cq[i + 1]], k[ck[i]:ck[i + 1]], v[ck[i]:ck[i + 1]],
            case["hist"], case["d"] ** -0.5) for i in range(case["rows"])])
    if kind == "train_attention":
        q, k, v = (t.detach().double().requires_grad_() for t in st["qkv"])
        cu, outs, grads = st["cu"].tolist(), [], []
        for i in range(case["rows"]):
            at = slice(cu[i], cu[i + 1])
            out = _sequence(q[at], k[at], v[at], 0, case["d"] ** -0.5)
            out.backward(st["dout"][at].double())
            outs.append(out.detach())
        return (torch.cat(outs), q.grad, k.grad, v.grad)
    if kind == "window_attention":
        hq, hk, d = case["hq"], case["hk"], case["d"]
        out, at = [], 0
        for i, n in enumerate(_lens(case)):
            pages = st["ptab"][i, :-(-n // PAGE)].long()
            kv = st["rows"][pages].view(-1, 2, hk, d)[:n].double()
            out.append(_sequence(
                st["q"][at:at + n].double().view(n, hq, d), kv[:, 0],
                kv[:, 1], 0, d ** -0.5, case["window"], case["keep"],
                st["sink"]))
            at += n
        return torch.cat(out).flatten(1)
    if kind == "sample":
        if case["temperature"] != 0.0:
            return None               # a random draw has no exact value
        x = st["logits"].double()
        tok = st["logits"].float().argmax(-1)
        return tok, torch.log_softmax(x, -1).gather(1, tok[:, None])[:, 0]
    if kind == "logprob":
        first, second = [], []
        for at in range(0, case["rows"], 256):
            x = st["logits"].detach()[at:at + 256].double()
            lab = st["labels"][at:at + 256, None]
            lp = torch.log_softmax(x, -1)
            first.append(lp.gather(1, lab)[:, 0])
            if case["grad"]:
                dlp = st["dlp"][at:at + 256, None].double()
                dx = lp.exp_().mul_(-dlp)
                second.append(dx.scatter_add_(1, lab, dlp))
            else:
                second.append(-(lp.exp() * lp).sum(-1))
        return torch.cat(first), torch.cat(second)
    if kind == "actor_step":
        m, lr = st["model"], case["response"]
        names = [n for n, _ in m.named_parameters()]
        w = {n: p.detach().double().requires_grad_()
             for n, p in m.named_parameters()}
        head = w.get("lm_head.weight", w["model.embed_tokens.weight"])
        n = st["ids"].shape[1]
        i = torch.arange(n, device=DEV)
        # padding rows see themselves, so that every row has a key
        live = (i[:, None] >= i[None]) & st["mask"][:, None, :] \
            | torch.eye(n, dtype=torch.bool, device=DEV)
        lps = []
        hidden = _decoder(m.config, w, st["ids"], st["pos"], live)
        cut = hidden.detach().requires_grad_()
        for r in range(case["rows"]):
            z = cut[r, -lr - 1:-1] @ head.t()
            lp = torch.log_softmax(z, -1).gather(
                1, st["ids"][r, -lr:, None])[:, 0]
            (lp * st["coef"][r].double()).sum().backward()
            lps.append(lp.detach())
        hidden.backward(cut.grad)
        return (torch.stack(lps), *[w[x].grad for x in names])
    cfg = _model(case)
    w = {n: t.double() for n, t in st["weights"].items()}
    head = w.get("lm_head.weight", w["model.embed_tokens.weight"])
    out = []
    for _, toks, _ in st["prompts"]:
        n = len(toks)
        i = torch.arange(n, device=DEV)
        x = _decoder(cfg, w, torch.tensor([toks], device=DEV), i[None],
                     (i[:, None] >= i[None])[None])
        out.append(x[0, -1] @ head.t())
    return torch.stack(out)

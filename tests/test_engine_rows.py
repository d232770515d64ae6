"""Prompt steps carry only the wanted tokens past the last layer's attention."""
import pytest
import torch

from polyrl_amd.models import get_model_config
from polyrl_amd.rollout.engine import Engine, SamplingParams


def engine(name):
    eng = Engine(get_model_config(name), device="cpu", dtype=torch.float32,
                 kv_token_capacity=4096, max_running_requests=8)
    g = torch.Generator().manual_seed(0)
    for buf in eng.model._name_map.values():
        buf.copy_(torch.randn(buf.shape, generator=g) * 0.05 + (buf.dim() == 1))
    return eng


def prompt(n, seed):
    return torch.randint(1, 200, (n,),
                         generator=torch.Generator().manual_seed(seed)).tolist()


@pytest.mark.parametrize("name", ["llama-tiny", "gpt2-debug"])
@pytest.mark.parametrize("wants", [([399], [0, 7]), ([], [299]), ([], []),
                                   ([0, 5, 399], [298, 299])])
def test_forced_rows(name, wants):
    """700 tokens at once against the prompts in portions of up to 200: the same
    rows, in entry order; a later portion sees what the first one cached."""
    once, parts = engine(name), engine(name)
    toks = [prompt(400, 1), prompt(300, 2)]
    got = once.step_forced([("r%d" % i, t, w)
                            for i, (t, w) in enumerate(zip(toks, wants))])
    want = []
    for i, (t, w) in enumerate(zip(toks, wants)):
        for at in range(0, len(t), 200):
            part = t[at:at + 200]
            rows = [x - at for x in w if at <= x < at + len(part)]
            out = parts.step_forced([("r%d" % i, part, rows)])
            if rows:
                want.append(out)
    if not want:
        assert got is None
    else:
        assert torch.allclose(got, torch.cat(want), atol=1e-4)
    a, b = (e.step_forced([("r0", [3, 4], [1]), ("r1", [5], [0])])
            for e in (once, parts))
    assert torch.allclose(a, b, atol=1e-4)


def test_generate_mixed():
    """Prompts whose prefill ends in a step beside ones that go on, and greedy
    tokens as of one prompt at a time."""
    prompts = [prompt(n, 10 + n) for n in (30, 600, 5, 320)]
    greedy = SamplingParams(temperature=0.0, max_new_tokens=4)
    eng = engine("llama-tiny")
    eng.max_batched_tokens = 640
    got = [o.output_ids for o in eng.generate(prompts, greedy)]
    for p, g in zip(prompts, got):
        assert engine("llama-tiny").generate([p], greedy)[0].output_ids == g

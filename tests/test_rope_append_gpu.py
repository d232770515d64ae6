"""RoPE + KV cache rows in one launch: the same bits as the two ops apart."""
import pytest
import torch

import polyrl_amd.ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("n,hq,hk,d", [(1, 1, 1, 8), (3, 7, 1, 64),
                                       (65, 32, 8, 128), (500, 64, 8, 128),
                                       (9, 2, 2, 40)])
def test_same_as_apart(n, hq, hk, d):
    torch.manual_seed(2)
    table = ops.RopeTable(d, 300, 10000.0, DEV)
    row = torch.randn(n, (hq + 2 * hk) * d, device=DEV).bfloat16()
    pos = torch.randint(0, 300, (n,), dtype=torch.int32, device=DEV)
    pages = (n + 15) // 16 + 1
    slots = torch.randperm(pages * 16, device=DEV)[:n].int()
    slots[::3] = -1                         # padding tokens
    got = []
    for fused in (True, False):
        r = row.clone()
        q = r[:, :hq * d].unflatten(1, (hq, d))
        k = r[:, hq * d:(hq + hk) * d].unflatten(1, (hk, d))
        v = r[:, (hq + hk) * d:].unflatten(1, (hk, d))
        kc, vc = (torch.ones(pages, 16, hk, d, device=DEV).bfloat16()
                  for _ in range(2))
        if fused:
            ops.rope_kv_append(q, k, v, pos, table, kc, vc, slots)
        else:
            ops.apply_rope_inplace(q, k, pos, table)
            ops.kv_cache_append(kc, vc, k, v, slots)
        got.append((r, kc, vc))
    for a, b in zip(*got):
        assert torch.equal(a, b)

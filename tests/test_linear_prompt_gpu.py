"""Products of prompts, and the gated MLP's two with its activation: every number
of row tiles a block may have, the edges of its tiles, the engine's use of them."""
import pytest
import torch

import polyrl_amd.ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def check(m, n, k, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(m * 31 + n * 7 + k)
    x = torch.randn(m, k, generator=g, device=DEV).bfloat16()
    w = (torch.randn(2 * n, k, generator=g, device=DEV) * scale
         / k ** 0.5).bfloat16()
    assert ops.linear_takes(x, w)
    got = ops.linear_swiglu(x, w)
    assert got.shape == (m, n)
    for at in range(0, m, 8192):
        gate, up = (x[at:at + 8192].double() @ w.double().t()).chunk(2, -1)
        want = gate * torch.sigmoid(gate) * up
        # 32-bit sums of k products, each off by 2^-24 of the sum of magnitudes
        # at most, and one rounding to bf16
        mass = x[at:at + 8192].double().abs() @ w.double().abs().t()
        mg, mu = mass.chunk(2, -1)
        bound = 2 ** -8 * want.abs() + k * 2.0 ** -24 * (
            1.1 * mg * up.abs() + gate.abs() * mu) + 2.0 ** -30
        assert ((got[at:at + 8192].double() - want).abs() <= bound).all(), at
    return x, w, got


def check_rows(x, w, got):
    k = x.shape[1]
    assert got.shape == (x.shape[0], w.shape[0])
    for at in range(0, x.shape[0], 8192):
        a = x[at:at + 8192].double()
        want, mass = a @ w.double().t(), a.abs() @ w.double().abs().t()
        bound = 2 ** -8 * want.abs() + k * 2.0 ** -24 * mass
        assert ((got[at:at + 8192].double() - want).abs() <= bound).all(), at


def row_parts(m, cols, k):
    """Row parts, 32 rows each, of the tiles that the library takes for ``cols`` tiles
    of columns."""
    return ops._require_ext().product_rows(m, cols, k, 3)[0]


@pytest.mark.parametrize("tiles", [2, 3, 4, 5, 6, 7, 8, 9])
def test_row_tiles(tiles):
    """Rows that fill 256 blocks of ``tiles`` row tiles but for a remainder."""
    check(8192 * tiles - 17, 128, 64)


@pytest.mark.parametrize("parts", [3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("inner", [2, 3, 4, 5, 16])
def test_inner_tiles(parts, inner):
    """Every number of row parts with inner tiles that fill the buffers just, take
    their places in turn and go round; an incomplete last row tile."""
    m, k = 8192 * parts - 17, 64 * inner
    assert row_parts(m, 1, k) == parts
    x, w, _ = check(m, 128, k)
    check_rows(x, w, ops.linear_rows(x, w))


@pytest.mark.parametrize("m", [1, 31, 32, 33, 64, 65, 127, 513, 700])
@pytest.mark.parametrize("n,k", [(128, 64), (128, 192), (640, 128),
                                 (1152, 320)])
def test_edges(m, n, k):
    """Single rows and remainders; one, an odd and an even number of inner
    tiles; column tiles that do not fill a group or the dies."""
    check(m, n, k)


@pytest.mark.parametrize("m", [1, 33, 65, 513, 700] + [
    8192 * t - 17 for t in range(2, 10)])
@pytest.mark.parametrize("n,k", [(256, 64), (768, 192), (1280, 128)])
def test_rows(m, n, k):
    """The product alone at the same edges, column tiles in one group and two."""
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device=DEV).bfloat16()
    w = torch.randn(n, k, generator=g, device=DEV).bfloat16()
    check_rows(x, w, ops.linear_rows(x, w))


def test_large_gates():
    """Gates far from 0: the sigmoid ends at 0 and 1."""
    x, w, got = check(600, 256, 128, scale=60.0)
    assert got.isfinite().all()


def test_gate_times_up_beyond_32_bits():
    """A closed gate gives 0 whatever the up projection, as silu(gate) * up."""
    x = torch.randn(600, 128, device=DEV).abs().add_(1.0).bfloat16()
    w = torch.zeros(512, 128, device=DEV).bfloat16()
    w[:256, 0], w[256:, 0] = -1e25, 1e25
    w[256::2, 0] = -1e25
    got = ops.linear_swiglu(x, w)
    gate, up = (x @ w.t()).chunk(2, -1)
    assert torch.equal(got, ops.silu_mul(gate, up)) and not got.any()


def test_what_it_takes():
    x = torch.randn(600, 128, device=DEV).bfloat16()
    w = torch.randn(512, 128, device=DEV).bfloat16()
    takes = ops.linear_takes
    assert takes(x, w)
    assert not takes(x.float(), w) and not takes(x, w.float())
    assert not takes(x[:, :96], w[:, :96])
    assert not takes(x, w[:384]) and not takes(x.t(), w)
    flat = torch.randn(600 * 128 + 1, device=DEV).bfloat16()
    assert not takes(flat[1:].view(600, 128), w)
    for a, b in ((x, w[:384]), (x[:, :96].contiguous(), w[:, :96].contiguous()),
                 (x, torch.randn(512, 64, device=DEV).bfloat16())):
        with pytest.raises(RuntimeError):
            ops.linear_swiglu(a, b)
    assert ops.linear_swiglu(x[:0], w).shape == (0, 256)
    assert not takes(x, w.cpu())
    # (rows of outputs end at 32-bit offsets)
    far = torch.empty(1 << 26, 64, dtype=torch.bfloat16, device=DEV)
    for op, n in ((ops.linear_rows, 1 << 25), (ops.linear_swiglu, 1 << 26)):
        assert not takes(x[:, :64].contiguous(), far[:n])
        with pytest.raises(RuntimeError):
            op(x[:1, :64].contiguous(), far[:n])


@pytest.mark.parametrize("m,n,k,rows,glu", [
    (512, 1024, 256, False, False), (513, 1024, 256, True, True),
    (8192, 1536, 128, True, True), (8193, 1280, 128, False, True),
    (700, 1024, 1024, True, True), (700, 1024, 1088, False, True),
    (513, 24320, 64, True, True), (513, 24576, 64, False, True),
    (600, 512, 2048, False, True), (600, 512, 2112, False, False),
    (8192, 512, 1536, False, True), (8191, 512, 1600, False, True),
    (8192, 512, 1600, False, False)])
def test_engine_prompts(m, n, k, rows, glu, monkeypatch):
    """Both sides of the rows and widths from which the engine takes it, which
    of the two ran, and that a captured step has the library's product."""
    from polyrl_amd.rollout.engine import _gate_up, _mm_nt
    ran = []
    for name in ("linear_rows", "linear_swiglu"):
        def spy(x, w, name=name, op=getattr(ops, name)):
            ran.append(name)
            return op(x, w)
        monkeypatch.setattr(ops, name, spy)
    g = torch.Generator(device=DEV).manual_seed(m)
    x = torch.randn(m, k, generator=g, device=DEV).bfloat16()
    w = (torch.randn(n, k, generator=g, device=DEV) / k ** 0.5).bfloat16()
    exact = x.double() @ w.double().t()
    gate, up = exact.chunk(2, -1)
    want = gate * torch.sigmoid(gate) * up
    off = (_gate_up(x, w).double() - want).norm() / want.norm()
    assert off <= 5e-3                 # three roundings to bf16 at most
    # (not taken, _gate_up's product goes through _mm_nt)
    assert ran == ["linear_swiglu"] * glu + ["linear_rows"] * (rows and not glu)
    del ran[:]
    both = _mm_nt(x, w)
    assert (both.double() - exact).norm() / exact.norm() <= 5e-3
    assert ran == ["linear_rows"] * rows
    if rows:
        x @ w.t()                      # (the library's handle and workspace)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            both = _mm_nt(x, w)
        for _ in range(3):
            both.zero_()
            graph.replay()
            assert (both.double() - exact).norm() / exact.norm() <= 5e-3
        assert ran == ["linear_rows"]


@pytest.mark.parametrize("n", [8, 248, 264, 504, 1016])
@pytest.mark.parametrize("m", [1, 97, 600])
def test_columns_short_of_a_tile(m, n):
    """Outputs in 8s, what stands behind them is not touched."""
    x = torch.randn(m, 320, device=DEV).bfloat16()
    w = torch.randn(n, 320, device=DEV).bfloat16()
    flat = torch.full((m * n + 4096,), 7.0, device=DEV, dtype=torch.bfloat16)
    out = flat[:m * n].view(m, n)
    ops._require_ext().linear_rows_into(out, x, w)
    want, mass = x.double() @ w.double().t(), x.abs().double() @ w.abs().double().t()
    assert ((out.double() - want).abs()
            <= 2 ** -8 * want.abs() + 320 * 2.0 ** -24 * mass).all()
    assert (flat[m * n:] == 7).all()


def test_linears_search():
    """A linear layer of many rows: whichever product the search finds, again and
    at an address that the kernel does not take."""
    m, n, k = 1400, 1096, 1088
    flat = torch.randn(m * k + 1, device=DEV).bfloat16()
    w = torch.randn(n, k, device=DEV).bfloat16() / k ** 0.5
    for x in (flat[:-1].view(m, k), flat[1:].view(m, k)):
        want = x.double() @ w.double().t()
        for _ in range(2):
            y = ops.tuned_linear(x, w)
            assert (y.double() - want).norm() / want.norm() <= 5e-3


def test_search_from_memory():
    """The search times what a layer finds: 73 us each where one weight of 134 MB is
    repeated, 103 of the kernel and 85 of the library's algorithm from memory."""
    x = torch.randn(513, 8192, device=DEV).bfloat16()
    w = torch.randn(8192, 8192, device=DEV).bfloat16()
    pick = ops._require_ext().tuned_linear_pick
    y = ops.tuned_linear(x, w)
    assert pick(*y.shape, 8192) == 0 and pick(514, 8192, 8192) == -1
    assert (y.float() - x.float() @ w.float().t()).norm() <= 5e-3 * y.float().norm()


@pytest.mark.parametrize("m,n,k,rows", [
    (2300, 2048, 2048, True), (2200, 2048, 2048, False), (4096, 2048, 2048, True),
    (2048, 4096, 2048, True), (4096, 4096, 2048, False), (4095, 4096, 2048, False),
    (4300, 1024, 4096, True), (4200, 1024, 4096, False), (5000, 512, 4096, False)])
def test_engine_wide_prompts(m, n, k, rows, monkeypatch):
    """Both sides of the line for widths beyond 1024."""
    from polyrl_amd.rollout.engine import _mm_nt
    ran = []
    real = ops.linear_rows
    monkeypatch.setattr(ops, "linear_rows",
                        lambda x, w: ran.append(1) or real(x, w))
    x = torch.randn(m, k, device=DEV).bfloat16()
    w = torch.randn(n, k, device=DEV).bfloat16() / k ** 0.5
    want = x.float() @ w.float().t()
    assert (_mm_nt(x, w).float() - want).norm() / want.norm() <= 5e-3
    assert bool(ran) == rows


@pytest.mark.parametrize("parts,m", [(3, 93), (4, 125), (5, 157), (6, 189),
                                     (7, 445), (8, 253)])
@pytest.mark.parametrize("k", [256, 320, 384])
def test_sums_beside_the_next_tile(parts, m, k):
    """Two tiles and three a block, of every number of row parts: a tile's sums
    leave the accumulators while the next one's first step fills them.  Rows and
    columns short of a tile; what stands behind the outputs is not touched."""
    cols = 300
    assert row_parts(m, cols, k) == parts
    n = 256 * cols - 8
    x = torch.randn(m, k, device=DEV).bfloat16()
    w = torch.randn(n, k, device=DEV).bfloat16()
    flat = torch.full((m * n + 65536,), 7.0, device=DEV, dtype=torch.bfloat16)
    ops._require_ext().linear_rows_into(flat[:m * n].view(m, n), x, w)
    check_rows(x, w, flat[:m * n].view(m, n))
    assert (flat[m * n:] == 7).all()
    half = 128 * cols
    wg, wu = w[:half] / k ** 0.5, torch.randn(half, k, device=DEV).bfloat16()
    got = ops.linear_swiglu(x, torch.cat([wg, wu]))
    for at in range(0, half, 128 * 64):
        a = slice(at, min(half, at + 128 * 64))
        assert torch.equal(got[:, a], ops.linear_swiglu(
            x, torch.cat([wg[a], wu[a]])))


@pytest.mark.parametrize("m", [1149, 1300, 1530, 1785])
def test_kept_beside_the_next_tile(m):
    """The same where gate and up projection are kept."""
    x = torch.randn(m, 320, device=DEV).bfloat16()
    wg, wu = (torch.randn(10240, 320, device=DEV).bfloat16() for _ in range(2))
    y, gate, up = ops._require_ext().linear_gated(x, wg, wu, True)
    check_rows(x, wg, gate)
    check_rows(x, wu, up)
    assert torch.equal(y, ops.linear_swiglu(x, torch.cat([wg, wu])))


def test_outputs_beyond_the_cache():
    """More outputs than go past the L2s: the same as in pieces that do."""
    x = torch.randn(1100, 256, device=DEV).bfloat16()
    w = torch.randn(128264, 256, device=DEV).bfloat16()
    op = ops._require_ext().linear_rows_into

    def rows(w):
        out = x.new_empty(x.shape[0], w.shape[0])
        op(out, x, w)
        return out
    assert torch.equal(rows(w), torch.cat([rows(w[:64136]), rows(w[64136:])], 1))


@pytest.mark.parametrize("m,n,k,parts", [
    (1, 256, 64, 3), (97, 512, 128, 3), (700, 1024, 320, 3), (513, 256, 1024, 3),
    (93, 76800, 256, 3), (125, 76800, 256, 4), (157, 76800, 320, 5),
    (189, 76800, 384, 6), (445, 76800, 320, 7), (253, 76800, 384, 8)])
def test_added(m, n, k, parts):
    """Outputs that hold numbers already: one rounding of the whole sum, edges of
    tiles, a block's tiles one after the other; what stands behind is not touched."""
    assert row_parts(m, n // 256, k) == parts
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device=DEV).bfloat16()
    w = torch.randn(n, k, generator=g, device=DEV).bfloat16()
    flat = torch.randn(m * n + 65536, generator=g, device=DEV).bfloat16()
    out, behind, old = flat[:m * n].view(m, n), flat[m * n:].clone(), \
        flat[:m * n].view(m, n).double()
    ops.linear_rows_add(out, x, w)
    a, b = x.double(), w.double().t()
    want = a @ b + old
    bound = 2 ** -8 * want.abs() + (k + 1) * 2.0 ** -24 * (
        a.abs() @ b.abs() + old.abs())
    assert ((out.double() - want).abs() <= bound).all()
    assert torch.equal(flat[m * n:], behind)


@pytest.mark.parametrize("tokens,calls", [(4095, 0), (4096, 2)])
def test_engine_adds(tokens, calls, monkeypatch):
    """From 2^22 outputs on the projections add to the residual: both sides of the
    line, the same logits as by a product and a norm that adds but for roundings."""
    from polyrl_amd.models import get_model_config
    from polyrl_amd.rollout import engine
    cfg = get_model_config("llama-400m", {"num_hidden_layers": 2})
    eng = engine.Engine(cfg, device=DEV, dtype=torch.bfloat16, page_size=16,
                        kv_token_capacity=tokens + 64, max_running_requests=4)
    h, i, d = cfg.hidden_size, cfg.intermediate_size, cfg.head_dim
    assert h == 1024
    g = torch.Generator(device=DEV).manual_seed(5)
    nq, nk = cfg.num_attention_heads * d, cfg.num_key_value_heads * d
    shapes = {"model.embed_tokens": (cfg.vocab_size, h), "model.norm": (h,),
              "lm_head": (cfg.vocab_size, h)}
    for li in range(2):
        at = "model.layers.%d." % li
        for name, shape in (
                ("self_attn.q_proj", (nq, h)), ("self_attn.k_proj", (nk, h)),
                ("self_attn.v_proj", (nk, h)), ("self_attn.o_proj", (h, nq)),
                ("mlp.gate_proj", (i, h)), ("mlp.up_proj", (i, h)),
                ("mlp.down_proj", (h, i)), ("input_layernorm", (h,)),
                ("post_attention_layernorm", (h,))):
            shapes[at + name] = shape
    eng.model.load_state_dict({
        n + ".weight": (torch.ones(s, device=DEV) if len(s) == 1 else 0.03
                        * torch.randn(s, generator=g, device=DEV)).bfloat16()
        for n, s in shapes.items()})
    ids = torch.randint(cfg.vocab_size, (tokens,), generator=g, device=DEV).tolist()
    cuts = [0, 900, 1901, 2600, tokens]
    ran, real = [], ops.linear_rows_add

    def step():
        prompts = [("r%d" % k, ids[a:b], [b - a - 1])
                   for k, (a, b) in enumerate(zip(cuts, cuts[1:]))]
        return eng.step_forced(prompts, end=[p[0] for p in prompts])
    monkeypatch.setattr(ops, "linear_rows_add",
                        lambda *a: ran.append(1) or real(*a))
    got = step()
    # (the first layer's two at most: the last one goes on with few rows)
    assert bool(ran) == bool(calls) and len(ran) <= calls
    monkeypatch.setattr(engine, "_takes_rows", lambda x, w: False)
    want = step()
    assert (got - want).norm() / want.norm() <= 2e-2

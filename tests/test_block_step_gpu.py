"""The linears between two attentions in one launch (nq_block_step) against the launches one by one and the same in float64, and the layouts
it takes."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = {"0.6b": (1024, 3072), "1.7b": (2048, 6144)}
HEADS, KV, EPS, BLOCK = 16, 8, 1e-6, 16
ORDER = (0, 2, 4, 6, 1, 3, 5, 7)


def _packed(gen, K, N, g=128, std=None):
    """Packed weight and its float64 values [K, N]."""
    q = torch.randint(0, 16, (K, N), generator=gen, device="cuda", dtype=torch.int32)
    z = torch.randint(0, 16, (K // g, N), generator=gen, device="cuda", dtype=torch.int32)
    s = ((0.5 + torch.rand(K // g, N, generator=gen, device="cuda")) * (std or K ** -0.5) / 6.5).bfloat16()

    def pack(x):
        x, w = x.view(x.shape[0], -1, 8), torch.zeros(x.shape[0], x.shape[1] // 8, dtype=torch.int32, device="cuda")
        for j, c in enumerate(ORDER):
            w |= x[:, :, c] << (4 * j)
        return w
    rep = lambda t: t.repeat_interleave(g, dim=0)
    return (pack(q), s, pack(z)), (q - rep(z)).double() * rep(s).double(), (q, z, s)


def _tile(x):
    """[rows, K] -> [ceil(rows / 16) * 16, K] in operand order: 16 rows x 32 columns a piece, element ((k / 8 % 4) * 16 + row) * 8 + k % 8."""
    rows, K = x.shape
    padded = torch.zeros(-(-rows // 16) * 16, K, dtype=x.dtype, device=x.device)
    padded[:rows] = x
    return padded.view(-1, 16, K // 32, 4, 8).permute(0, 2, 3, 1, 4).reshape(padded.shape).contiguous()


@pytest.mark.parametrize("K,N,g", [(128, 16, 128), (1024, 48, 128), (768, 32, 256), (384, 64, 384)])
def test_tile_weight(K, N, g):
    from nanoquantization_amd.engine import ops
    gen = torch.Generator(device="cuda").manual_seed(K + N)
    packed, _, (q, z, s) = _packed(gen, K, N, g)
    got = ops.tile_weight(*packed)
    pieces = N // 16 * (K // 128)
    words = got[:pieces * 1024].view(torch.int32).view(N // 16, K // 128, 4, 16, 4)       # [tile, chunk, k / 8 % 4, column, step]
    shifts = torch.tensor([2 * j if j % 2 == 0 else 16 + 2 * (j - 1) for j in range(8)], device="cuda", dtype=torch.int32)
    turned = (torch.arange(16, device="cuda") & 2).bool().view(1, 1, 1, 16, 1)            # columns whose words are three bits further round
    words = torch.where(turned, ((words >> 3) & 0x1FFFFFFF) | (words << 29), words)
    codes = (words.unsqueeze(-1) >> shifts) & 15                                          # .. k % 8
    assert torch.equal(codes.permute(1, 4, 2, 5, 0, 3).reshape(K, N), q)
    affine = got[pieces * 1024:].view(torch.int32).view(N // 16, K // 128, 16)
    rows = torch.arange(0, K, 128, device="cuda") // g
    want = (z[rows] << 16) | (s[rows].view(torch.int16).int() & 0xFFFF)
    assert torch.equal(affine.permute(1, 0, 2).reshape(K // 128, N), want)


# context splits (few rows) and none, a last tile of rows that is not full
@pytest.mark.parametrize("rows,heads", [(1, 8), (7, 16), (16, 16), (33, 16)])
def test_tiled_attention_is_attention(rows, heads):
    from nanoquantization_amd.engine import ops
    gen = torch.Generator(device="cuda").manual_seed(rows)
    blocks = 24
    k, v = (torch.randn(rows * blocks, KV, BLOCK, 128, generator=gen, device="cuda").bfloat16() for _ in range(2))
    q = torch.randn(rows, heads, 128, generator=gen, device="cuda").bfloat16()
    table = torch.randperm(rows * blocks, generator=gen, device="cuda").int().view(rows, blocks)
    context = torch.randint(1, blocks * BLOCK + 1, (rows,), generator=gen, device="cuda").int()
    want = ops.paged_attention_decode(q, k, v, table, context, 128 ** -0.5)
    out = torch.zeros(-(-rows // 16) * 16, heads * 128, dtype=torch.bfloat16, device="cuda")
    ops.paged_attention_decode(q, k, v, table, context, 128 ** -0.5, out)
    assert torch.equal(out, _tile(want))


class _Case:
    def __init__(self, size, rows, seed):
        from nanoquantization_amd.engine import ops
        hidden, inter = SIZES[size]
        gen = torch.Generator(device="cuda").manual_seed(seed)
        self.hidden, self.inter, self.rows = hidden, inter, rows
        randn = lambda *s, std=1.0: (torch.randn(*s, generator=gen, device="cuda") * std).bfloat16()
        norm = lambda n: 1 + randn(n, std=0.1)
        self.packed, self.dense = [], []
        for _ in range(2):
            qkv, o = _packed(gen, hidden, (HEADS + 2 * KV) * 128), _packed(gen, HEADS * 128, hidden)
            gate, up, down = _packed(gen, hidden, inter), _packed(gen, hidden, inter), _packed(gen, inter, hidden)
            self.packed.append((qkv[0], o[0], ops.interleave_gate_up(gate[0], up[0]), down[0]))
            self.dense.append([w[1] for w in (qkv, o, gate, up, down)])
        self.x, self.attn = randn(rows, hidden, std=2.0), randn(rows, HEADS * 128)
        self.norms = [norm(hidden) for _ in range(4)]           # mid and next of either layer
        self.q_norm, self.k_norm = norm(128), norm(128)
        pos = torch.arange(256, device="cuda").double().unsqueeze(1) * 1e6 ** (-torch.arange(64, device="cuda").double() / 64)
        self.cos_sin = torch.cat([pos.cos(), pos.sin()], dim=1).float()
        self.positions = torch.randint(0, 256, (rows,), generator=gen, device="cuda")
        self.slots = torch.randperm(rows * BLOCK, generator=gen, device="cuda")[:rows].contiguous()
        self.slots[rows // 2] = -1 if rows > 1 else self.slots[0]
        self.k, self.v = (torch.zeros(rows, KV, BLOCK, 128, dtype=torch.bfloat16, device="cuda") for _ in range(2))
        self.steps = ops.BlockSteps(self.packed, rows, hidden, inter, HEADS, KV, torch.device("cuda"))
        self.steps.attn.copy_(_tile(self.attn))

    def run(self, **spin):
        """Both layers: the residuals behind them, and the second layer's q, k and v."""
        following = (self.norms[1], self.q_norm, self.k_norm, self.cos_sin, self.positions, self.slots, self.k, self.v, EPS)
        first = self.steps(0, self.x, self.norms[0], EPS, following, **spin)
        out = [first.clone(), self.steps.q.clone(), self.k.clone(), self.v.clone()]
        return out + [self.steps(1, first, self.norms[2], EPS, None, **spin).clone()]

    def exact(self):
        bf = lambda t: t.bfloat16().double()
        rms = lambda x, w: x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()
        out, x = [], self.x.double()
        for i in range(2):
            _, o, gate, up, down = self.dense[i]
            x = x + self.attn.double() @ o
            h = rms(x, self.norms[2 * i])
            g = h @ gate
            x = x + (g * torch.sigmoid(g) * (h @ up)) @ down
            out.append(x)
            if i == 0:
                y = (rms(x, self.norms[1]) @ self.dense[1][0]).view(self.rows, -1, 128)
                cs = self.cos_sin[self.positions].double().unsqueeze(1)
                turn = lambda t: torch.cat([t[..., :64] * cs[..., :64] - t[..., 64:] * cs[..., 64:],
                                            t[..., :64] * cs[..., 64:] + t[..., 64:] * cs[..., :64]], dim=-1)
                q, k, v = y.split([HEADS, KV, KV], dim=1)
                out += [turn(rms(q, self.q_norm)), turn(rms(k, self.k_norm)), v]
        return out


    def one_by_one(self):
        """What `run` returns, from a launch for each linear."""
        from nanoquantization_amd.engine import ops
        x, k, v = self.x.clone(), torch.zeros_like(self.k), torch.zeros_like(self.v)
        out = []
        for i in range(2):
            _, o, gate_up, down = self.packed[i]
            ssq = torch.empty(self.hidden // 128, self.rows, device="cuda")
            ops.awq_gemv_add_residual(self.attn, *o, x, ssq)
            act = ops.awq_gemv_rmsnorm(x, ssq, self.norms[2 * i], EPS, *gate_up, gated=True)
            ops.awq_gemv_add_residual(act, *down, x, ssq)
            out.append(x.clone())
            if i == 0:
                q = ops.awq_gemv_rmsnorm_qkv_rope_store(x, ssq, self.norms[1], EPS, *self.packed[1][0], self.q_norm, self.k_norm, self.cos_sin,
                                                        self.positions, self.slots, k, v, HEADS, KV, EPS)
                out += [q, k, v]
        return out


# one, a full and a barely begun row tile; where a task takes two row tiles, the last one half empty or full
@pytest.mark.parametrize("size,rows", [("0.6b", r) for r in (1, 15, 16, 17, 32, 33, 49, 64)] + [("1.7b", r) for r in (1, 15, 16, 17, 32)])
def test_block_step(size, rows):
    c = _Case(size, rows, seed=rows)
    x1, q, k, v, x2 = c.run()
    # the cuts of K are the same as far as the launches one by one don't share a wave between chunks
    if size == "0.6b" or 4 < rows <= 16:
        for name, a, b in zip(("residual", "q", "k", "v", "residual behind the second layer"), (x1, q, k, v, x2), c.one_by_one()):
            assert torch.equal(a, b), name
    e1, eq, ek, ev, e2 = c.exact()
    rel = lambda a, b: ((a.double() - b).norm() / b.norm()).item()
    # a rounding to bf16 is 2^-9 / sqrt(3) = 1.1e-3 of a value on average; behind one another lie those of the product of o_proj, the
    # residual, the norm (two), gate and up, SiLU, the activation, the product of down_proj and the residual again, each with a weight of at most
    # one in the result: below sqrt(10) 1.1e-3; the second layer adds its own, q, k and v four more
    for name, got, want, bound in (("residual", x1, e1, 3.5e-3), ("q", q, eq, 6e-3), ("residual behind the second layer", x2, e2, 5e-3)):
        assert rel(got, want) <= bound, (name, rel(got, want))
    # k and v in their slots, and nothing for the row without one
    live = (c.slots >= 0).nonzero()[:, 0]
    block, at = c.slots[live] // BLOCK, c.slots[live] % BLOCK
    for name, cache, want in (("k", k, ek), ("v", v, ev)):
        assert rel(cache[block, :, at], want[live]) <= 6e-3, (name, rel(cache[block, :, at], want[live]))
        cache[block, :, at] = 0
        assert not cache.any(), name
    # the sums of squares of the residual between o_proj and gate|up, whole lines of 128 columns a group of workgroups
    mid = c.steps.tiled[0].view(-1, c.hidden // 32, 4, 16, 8).permute(0, 3, 1, 2, 4).reshape(-1, c.hidden).double()
    squares = c.steps.squares[0].view(-1, c.hidden // 128, 16, 16).transpose(1, 2).reshape(-1, c.hidden // 8)
    assert torch.allclose(squares[:rows].double(), mid.square().view(-1, c.hidden // 8, 8).sum(-1)[:rows], rtol=8 * 2.0 ** -24, atol=0)
    # whoever does the work: nobody waits, every workgroup does what it finds missing
    for a, b in zip((x1, q, x2), (lambda t: (t[0], t[1], t[4]))(c.run(spin=0))):
        assert torch.equal(a, b)


def test_sizes_without_a_form_are_refused():
    from nanoquantization_amd import _lib
    from nanoquantization_amd.engine import ops
    ok = lambda rows, hidden, inter, heads=16, layers=2, dtype=torch.bfloat16, kv=8: ops.BlockSteps.supported(rows, hidden, inter, heads, kv, layers, dtype)
    assert ok(64, 1024, 3072) and ok(32, 2048, 6144) and ok(64, 1024, 3072, kv=16)
    assert not any(ok(8, 1024, 3072, kv=kv) or ok(8, 2048, 6144, kv=kv) for kv in (1, 2, 4, 5, 32))
    assert not any((ok(65, 1024, 3072), ok(33, 2048, 6144), ok(0, 1024, 3072), ok(8, 2560, 9728, 32), ok(8, 1024, 3072, 32), ok(8, 1024, 3072, layers=1),
                    ok(8, 1024, 3072, dtype=torch.float16)))
    c = _Case("0.6b", 2, seed=1)
    c.steps.sizes["rows"], c.x = 65, torch.zeros(65, 1024, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(_lib.AwqHipError, match="no form"):
        c.steps(0, c.x, c.norms[0], EPS)


def test_block_steps_repeat_in_a_graph_and_after_a_step_that_broke_off():
    c = _Case("0.6b", 20, seed=3)
    want = c.run()
    c.k.zero_(), c.v.zero_()
    c.steps(0, c.x, c.norms[0], EPS)                # a step that ends behind its first layer
    assert all(torch.equal(a, b) for a, b in zip(c.run(), want))
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        c.run()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = c.run()
    torch.cuda.current_stream().wait_stream(stream)
    for _ in range(4):
        for t in out:
            t.zero_()
        c.k.zero_(), c.v.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, want))
        assert all(torch.equal(a, b) for a, b in zip(c.run(), want))


@pytest.mark.parametrize("size,batch", [("0.6b", 3), ("0.6b", 24), ("1.7b", 10), ("1.7b", 1), ("1.7b", 24)])
def test_engine_decodes_alike_with_and_without_block_steps(size, batch, monkeypatch):
    """The logits of a decode step, some rows idle, with the launches of a block and with one for each linear: the same bits, but for the second size where
    the launches one by one share waves between chunks (up to 4 rows) or take K in one piece (above 16)."""
    from nanoquantization_amd.engine import LLMEngine, ops
    from nanoquantization_amd.models.random_init import QWEN3_0P6B, random_awq_qwen3
    cfg = dict(QWEN3_0P6B, num_hidden_layers=3, vocab_size=4096, max_position_embeddings=512, hidden_size=SIZES[size][0],
               intermediate_size=SIZES[size][1])
    model = random_awq_qwen3(cfg, seed=5, std=0.02)
    torch.manual_seed(6)
    tokens = torch.randint(0, 4096, (batch, 90))
    logits = []
    for on in (False, True):
        if not on:
            monkeypatch.setattr(ops.BlockSteps, "supported", staticmethod(lambda *a: False))
        else:
            monkeypatch.undo()
        eng = LLMEngine(model, max_batch=batch + 2, max_seq_len=128, block_size=32)
        assert (eng.block_steps is not None) == on
        leases = [eng.acquire(4) for _ in range(batch)]
        eng._prefill(tokens[:, :-1].cuda(), leases)
        for _ in range(2):
            logits.append(eng.decode([(l, 89, int(t)) for l, t in zip(leases, tokens[:, -1])]).clone())
    assert torch.equal(logits[0], logits[1]) and torch.equal(logits[2], logits[3])
    if size == "0.6b" or 4 < batch + 2 <= 16:
        assert torch.equal(logits[0], logits[2])
    else:       # each is within sqrt(3 / 2) 5e-3 of the exact ones (test_block_step's two layers, here three), independently of one another
        rel = ((logits[0].double() - logits[2].double()).norm() / logits[0].double().norm()).item()
        print(f"rel {rel:.2e}", flush=True)
        assert rel <= 1e-2, rel


@pytest.mark.parametrize("kv", [1, 2, 4, 16])
def test_engine_decodes_with_other_numbers_of_kv_heads(kv, monkeypatch):
    """16 query heads over 1, 2 and 4 kv heads have no block step and decode one launch for each linear; over 16 they have one, and both ways
    the logits are the same."""
    from nanoquantization_amd.engine import LLMEngine, ops
    from nanoquantization_amd.models.random_init import QWEN3_0P6B, random_awq_qwen3
    cfg = dict(QWEN3_0P6B, num_hidden_layers=2, vocab_size=2048, max_position_embeddings=256, total_num_kv_heads=kv)
    model = random_awq_qwen3(cfg, seed=kv, std=0.02)
    torch.manual_seed(7)
    tokens = torch.randint(0, 2048, (3, 40))
    logits = []
    for on in (True, False):
        if not on:
            monkeypatch.setattr(ops.BlockSteps, "supported", staticmethod(lambda *a: False))
        eng = LLMEngine(model, max_batch=3, max_seq_len=64, block_size=32)
        assert (eng.block_steps is not None) == (on and kv == 16)
        leases = [eng.acquire(2) for _ in range(3)]
        eng._prefill(tokens[:, :-1].cuda(), leases)
        logits.append(eng.decode([(l, 39, int(t)) for l, t in zip(leases, tokens[:, -1])]).clone())
    assert logits[0].isfinite().all() and torch.equal(*logits)


@pytest.mark.parametrize("size,layers,batch", [("0.6b", 6, 32), ("1.7b", 3, 24)])
def test_two_engines_decode_at_once(size, layers, batch):
    """Two engines on two streams, whose block steps each may hold a part of the GPU: the logits of one after the other, and no wait for
    workgroups without room that is longer than a quarter of a millisecond in a launch (three phases)."""
    from nanoquantization_amd.engine import LLMEngine, ops
    from nanoquantization_amd.models.random_init import QWEN3_0P6B, random_awq_qwen3
    assert 3 * ops.BlockSteps.SPIN * 0.6e-6 <= 0.25e-3
    cfg = dict(QWEN3_0P6B, num_hidden_layers=layers, vocab_size=2048, max_position_embeddings=512, hidden_size=SIZES[size][0],
               intermediate_size=SIZES[size][1])
    model = random_awq_qwen3(cfg, seed=5, std=0.02)
    streams, engines, rows, want = [torch.cuda.Stream() for _ in range(2)], [], [], []
    for seed in range(2):
        eng = LLMEngine(model, max_batch=batch, max_seq_len=384, block_size=64)
        assert eng.block_steps is not None
        gen = torch.Generator(device="cuda").manual_seed(seed)
        for t in (*eng.cache.k, *eng.cache.v):
            t.copy_(torch.randn(t.shape, generator=gen, device="cuda"))
        rows.append([(eng.acquire(6), 320, 7 + i + seed) for i in range(batch)])
        engines.append(eng)
        for _ in range(2):
            logits = eng.decode(rows[seed])
        want.append(logits.clone())
    torch.cuda.synchronize()
    for _ in range(4):
        got = []
        for _ in range(5):
            for i in range(2):
                with torch.cuda.stream(streams[i]):
                    logits = engines[i].decode(rows[i])
                    got = got[-1:] + [logits]
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("use_graph", [True, False])
def test_decode_follows_weights_written_behind_the_engine(use_graph):
    """o_proj and down_proj are the module's own: what is written there in place (without a graph also another tensor in its place) is what the next
    decode step multiplies by."""
    from nanoquantization_amd.engine import LLMEngine
    from nanoquantization_amd.models.random_init import QWEN3_0P6B, random_awq_qwen3
    cfg = dict(QWEN3_0P6B, num_hidden_layers=3, vocab_size=2048, max_position_embeddings=256)
    model = random_awq_qwen3(cfg, seed=9, std=0.02)
    tokens = torch.randint(0, 2048, (4, 40), generator=torch.Generator().manual_seed(1))

    def engine():
        eng = LLMEngine(model, max_batch=4, max_seq_len=64, block_size=32, use_graph=use_graph)
        assert eng.block_steps is not None
        return eng, [eng.acquire(2) for _ in range(4)]

    def logits(eng, leases):
        eng._prefill(tokens[:, :-1].cuda(), leases)
        return eng.decode([(l, 39, int(t)) for l, t in zip(leases, tokens[:, -1])]).clone()

    kept = engine()
    before = logits(*kept)
    layers = model.model.layers
    other = random_awq_qwen3(cfg, seed=10, std=0.02).model.layers
    with torch.no_grad():
        layers[0].mlp.down_proj.qscales.mul_(2)
        layers[1].self_attn.o_proj.load_state_dict(other[1].self_attn.o_proj.state_dict())
        if not use_graph:
            layers[2].self_attn.o_proj.qzeros = other[2].self_attn.o_proj.qzeros
    after = logits(*kept)
    assert not torch.equal(before, after) and torch.equal(after, logits(*engine()))
    assert torch.equal(after, logits(*kept))

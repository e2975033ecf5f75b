"""WQLinear_GEMM.forward on the GPU: shapes, dtype, bias, regime switch, state_dict round trip."""
import numpy as np
import pytest
import torch

import nanoquantization_amd as nq
from conftest import to_bits
from oracle import awq_oracle as o

pytestmark = pytest.mark.gpu


def _module(K, N, g, tdt, bias, seed=0):
    torch.manual_seed(seed)
    w = torch.randn(N, K) * 0.02
    dq, s, z = nq.pseudo_quantize(w, g, 4, True)
    lin = torch.nn.Linear(K, N, bias=bias)
    lin.weight.data = dq
    return nq.WQLinear_GEMM.from_linear(lin, 4, g, s.t().contiguous(), z.t().contiguous(), tdt).to("cuda")


@pytest.mark.parametrize("tdt,dt", [(torch.float16, "f16"), (torch.bfloat16, "bf16")])
@pytest.mark.parametrize("bias", [False, True])
def test_forward_matches_oracle_all_regimes(tdt, dt, bias):
    K, N, g = 1024, 3072, 128
    m = _module(K, N, g, tdt, bias)
    qw, qz = m.qweight.cpu().numpy(), m.qzeros.cpu().numpy()
    qs = to_bits(m.qscales)
    b = m.bias.float().cpu().numpy() if bias else None
    for shape in [(16, K), (1, K), (2, 3, K), (4, 40, K), (300, K)]:   # cfg1 is the first
        print(f"forward {dt} bias={bias} x{shape}", flush=True)
        torch.manual_seed(sum(shape))
        x = torch.randn(*shape).to(tdt).cuda()
        y = m(x)
        assert y.shape == x.shape[:-1] + (N,) and y.dtype == tdt
        ref = o.linear_fp32(to_bits(x.reshape(-1, K)), qw, qz, qs, dt, b)
        err = o.max_rel_err(y.float().cpu().numpy().reshape(-1, N), ref)
        assert err <= 1e-2 and err <= (1.5e-3 if dt == "f16" else 6e-3), err


def test_forward_casts_x_to_scale_dtype():
    # the reference's test runs fp16 activations through bf16 scales: x is cast on load (layers/gemm.py:259)
    m = _module(512, 256, 128, torch.bfloat16, False)
    x = torch.randn(8, 512, dtype=torch.float16, device="cuda")
    y = m(x)
    assert y.dtype == torch.bfloat16
    assert torch.equal(y, m(x.to(torch.bfloat16)))


def test_state_dict_roundtrip_keeps_outputs():
    m = _module(512, 256, 128, torch.float16, False)
    m2 = nq.WQLinear_GEMM(4, 128, 512, 256, bias=False, output_dtype=torch.float16)
    m2.load_state_dict({k: v.cpu() for k, v in m.state_dict().items()})
    m2 = m2.to("cuda")
    x = torch.randn(5, 512, dtype=torch.float16, device="cuda")
    assert torch.equal(m(x), m2(x))
    # with a bias the constructor's buffer is bf16 whatever the output dtype (layers/gemm.py:435-443),
    # so a loaded fp16 bias is rounded to bf16: equal only to bf16 precision
    mb = _module(512, 256, 128, torch.float16, True)
    mb2 = nq.WQLinear_GEMM(4, 128, 512, 256, bias=True, output_dtype=torch.float16)
    mb2.load_state_dict({k: v.cpu() for k, v in mb.state_dict().items()})
    mb2 = mb2.to("cuda")
    assert mb2.bias.dtype == torch.bfloat16
    assert (mb(x).float() - mb2(x).float()).abs().max().item() <= 2.0 ** -8 * mb.bias.abs().max().item() + 2e-3


@pytest.mark.parametrize("bias", [False, True])
def test_forward_empty_and_boundary_row_counts(bias):
    """No rows at all, and the row counts where the dispatch changes kernel (16/17 one m-tile vs row blocks, 64/65
    and 128/129 GEMV vs GEMM -- 128 rows on small weights like this one --, 1023/1024 where the reference's own structure
    changes): shape, dtype and the fp32 oracle at every one of them."""
    K, N, g = 512, 384, 128
    m = _module(K, N, g, torch.bfloat16, bias, seed=3)
    for shape in [(0, K), (2, 0, K)]:
        y = m(torch.zeros(*shape, dtype=torch.bfloat16, device="cuda"))
        assert y.shape == tuple(shape[:-1]) + (N,) and y.dtype == torch.bfloat16 and y.numel() == 0
    qw, qz, qs = m.qweight.cpu().numpy(), m.qzeros.cpu().numpy(), to_bits(m.qscales)
    b = m.bias.float().cpu().numpy() if bias else None
    for M in (16, 17, 64, 65, 128, 129, 1023, 1024):
        print(f"forward boundary M={M} bias={bias}", flush=True)
        torch.manual_seed(M)
        x = torch.randn(M, K).to(torch.bfloat16).cuda()
        ref = o.linear_fp32(to_bits(x), qw, qz, qs, "bf16", b)
        err = o.max_rel_err(m(x).float().cpu().numpy(), ref)
        assert err <= 6e-3, (M, err)


@pytest.mark.parametrize("K,N,g", [(1024, 151936, 128), (65536, 1024, 128), (128, 8, 128), (64, 8, 64), (32, 4096, 32),
                                   (256, 262144, 128)])
def test_linear_extreme_widths_default_dispatch(K, N, g):
    """Widths at the ends of what the entry point takes -- a vocabulary-sized N (a quantised lm_head), one packed word
    of N, one group of K, a K of 512 chunks -- at row counts on both sides of every regime switch, through the default
    dispatch.  Reference: x @ awq_dequantize(...) in fp32 on the device (the dequantise kernel is bit-exact against the
    oracle, tests/test_dequant_gpu.py; the CPU oracle would need minutes at these sizes).  Bound: the 1e-2 of the
    task, and the rounding-only bound the other GEMV tests use."""
    from nanoquantization_amd.layers.gemm import _linear
    torch.manual_seed(K + N)
    for tdt, tight in ((torch.float16, 1.5e-3), (torch.bfloat16, 6e-3)):
        qw = torch.randint(-2 ** 31, 2 ** 31 - 1, (K, N // 8), dtype=torch.int32, device="cuda")
        qz = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // g, N // 8), dtype=torch.int32, device="cuda")
        qs = (torch.rand(K // g, N, device="cuda") * 0.02 + 0.001).to(tdt)
        W = nq.awq_dequantize(qw, qs, qz).float()
        for M in (1, 5, 16, 17, 64, 65, 129):
            print(f"extreme widths K={K} N={N} g={g} {tdt} M={M}", flush=True)
            x = (torch.randn(M, K, device="cuda") * 0.5).to(tdt)
            y = _linear("awq_linear", x, qw, qs, qz, None)
            ref = x.float() @ W
            err = ((y.float() - ref).abs().max() / ref.abs().max()).item()
            assert y.shape == (M, N) and y.dtype == tdt and err <= tight, (M, err)
        del W


def _eager(monkeypatch):
    """The modules on torch operations only."""
    from nanoquantization_amd.layers import norm
    from nanoquantization_amd.models import qwen3_quantized as q3
    for mod in (norm, q3):
        monkeypatch.setattr(mod, "plain", lambda *t: False)


@pytest.mark.parametrize("tdt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hd,heads,kv,b,s,first", [(128, 16, 8, 2, 65, 0), (64, 4, 4, 3, 1, 7), (256, 6, 2, 1, 130, -140), (128, 3, 1, 1, 64, 3)])
def test_steps_between_the_linears(tdt, hd, heads, kv, b, s, first):
    """Norms, rotary, SiLU as one kernel each against the torch expressions of the modules: the same two rounding points,
    each of which may fall one place (ulp, relative) apart where fp32 differs, and rarely does.  Attention against softmax in fp64: weights and output are
    each rounded once, and 2^-8 relative covers both."""
    from nanoquantization_amd import _lib
    from nanoquantization_amd.layers.norm import RMSNorm
    from nanoquantization_amd.layers.rope import RoPE
    ops, ulp = _lib.torch_ops(), {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[tdt]
    print(f"steps between the linears {tdt} hd={hd} heads={heads}/{kv} {b}x{s} from {first}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(hd + s)
    rnd = lambda *n: torch.randn(*n, device="cuda", generator=gen).to(tdt)

    def same(got, want):
        assert got.shape == want.shape and got.dtype == want.dtype
        d, w = (got.float() - want.float()).abs(), want.float().abs()
        assert (d <= 2 * ulp * w + 1e-6).all() and (d > 0).float().mean() < 0.02

    # a view that starts in the middle of a 16-byte word: the operators have to move it
    q, k, v = (rnd(b, s, n * hd + 1)[..., 1:] for n in (heads, kv, kv))
    qn, kn, rope = RMSNorm(hd, 1e-6), RMSNorm(hd, 1e-5), RoPE(hd, 512)
    qn.weight.data, kn.weight.data = 1 + rnd(hd), 1 + rnd(hd)
    rope = rope.cuda()
    pos = torch.arange(first, first + s, device="cuda").repeat(b if first else 1, 1)
    tq, tk, tv = ops.qkv_norm_rope(q, k, v, qn.weight.detach(), kn.weight.detach(), rope.cos_sin_cache, pos, heads, kv, 1e-6, 1e-5)
    wq, wk = rope(qn.rms_norm(q.view(b, s, heads, hd)), kn.rms_norm(k.view(b, s, kv, hd)), pos)
    rot = lambda got, want: ((got.float() - want.float()).abs() <= 2 * ulp * want.float().abs().amax(-1, True)).all()
    assert rot(tq, wq) and rot(tk, wk.transpose(1, 2))     # x1 cos - x2 sin: a last place of a term, not of the difference
    assert torch.equal(tv, v.view(b, s, kv, hd).transpose(1, 2))
    bad = ops.qkv_norm_rope(q, k, v, qn.weight.detach(), kn.weight.detach(), rope.cos_sin_cache, pos * 0 + 512, heads, kv, 1e-6, 1e-5)
    assert bad[0].isnan().all() and bad[1].isnan().all() and torch.equal(bad[2], tv)

    n = RMSNorm(max(512, heads * hd), 1e-6)
    x = rnd(b, s, n.norm_size)
    n.weight.data = 1 + rnd(n.norm_size)
    with torch.no_grad():
        same(n(x), n.rms_norm(x))
        same(n(x.transpose(0, 1)), n.rms_norm(x.transpose(0, 1)))
    up = rnd(b, s, n.norm_size)
    same(ops.silu_mul(x * 4, up), torch.nn.functional.silu(x * 4) * up)

    if tdt == torch.bfloat16:
        o = ops.causal_attention(tq, tk, tv, hd ** -0.5)
        rep = lambda t: t.double().repeat_interleave(heads // kv, 1)
        sc = tq.transpose(1, 2).double() @ rep(tk).transpose(-1, -2) * hd ** -0.5
        w = sc.masked_fill(torch.ones(s, s, dtype=torch.bool, device="cuda").triu(1), float("-inf")).softmax(-1)
        ref = (w @ rep(tv)).transpose(1, 2).reshape(b, s, heads * hd)
        scale = (w @ rep(tv).abs()).transpose(1, 2).reshape(b, s, heads * hd)
        assert ((o.double() - ref).abs() <= 2.0 ** -8 * (scale + ref.abs())).all()


def test_when_modules_use_the_operators(monkeypatch):
    """What the fused steps cannot do runs on torch operations as before: gradients, hooks, transforms, other shapes of
    positions; and a prompt forward gives the same logits either way."""
    from nanoquantization_amd.models.qwen3_quantized import Qwen3QuantizedForCausalLM
    torch.manual_seed(0)
    m = Qwen3QuantizedForCausalLM(num_hidden_layers=2, vocab_size=128, hidden_size=512, total_num_heads=4, total_num_kv_heads=2,
                                  max_position_embeddings=64, intermediate_size=256, head_dim=64).to(torch.bfloat16)
    for mod in m.modules():
        if isinstance(mod, nq.WQLinear_GEMM):
            mod.qweight.random_(-2 ** 31, 2 ** 31 - 1)
            mod.qzeros.random_(-2 ** 31, 2 ** 31 - 1)
            mod.qscales.uniform_(0.002, 0.006)
    m = m.cuda()
    ids, pos = torch.randint(0, 128, (2, 33), device="cuda"), torch.arange(33, device="cuda")
    attn = m.model.layers[0].self_attn
    x = torch.randn(2, 33, 512, device="cuda", dtype=torch.bfloat16)
    seen = []
    with torch.no_grad():
        fused, fused_logits = attn(x, pos), m(ids, pos)
        assert torch.equal(attn(x, pos.int()), fused) and torch.equal(attn(x, pos.expand(2, 33)), fused)
        handle = attn.q_norm.register_forward_hook(lambda mod, a, out: seen.append(out.shape))
        hooked = attn(x, pos)
        handle.remove()
        assert seen == [(2, 33, 4, 64)]
        one = attn(x, pos[:1].view(1, 1))                  # one position for all tokens: broadcast by torch
        mixed = attn(x.half(), pos)                        # float16 into bfloat16 projections
        assert one.shape == fused.shape and torch.equal(mixed, attn(x.half().bfloat16(), pos))
    assert not fused.requires_grad
    norm = next(mod for mod in m.modules() if type(mod).__name__ == "RMSNorm" and mod.norm_size == 512)
    xg = x.clone().requires_grad_()
    norm(xg).float().sum().backward()
    assert xg.grad is not None and norm.weight.grad is not None
    assert torch.func.vmap(norm.rms_norm)(x).shape == x.shape and torch.equal(torch.func.vmap(norm)(x), norm.rms_norm(x))
    _eager(monkeypatch)
    with torch.no_grad():
        assert torch.equal(attn(x, pos), hooked)
        for got, want in ((fused, hooked), (fused_logits, m(ids, pos))):
            # a dozen roundings to 8 bits on the way, of which few fall differently
            assert (got.float() - want.float()).norm() <= 2.0 ** -7 * want.float().norm()


@pytest.mark.parametrize("layout", [lambda x: x.transpose(0, 1), lambda x: x[:, -1], lambda x: x.transpose(-1, -2).contiguous().transpose(-1, -2)])
def test_norm_result_keeps_the_layout(layout):
    from nanoquantization_amd.layers.norm import RMSNorm
    norm = RMSNorm(512).to("cuda", torch.bfloat16)
    x = layout(torch.randn(4, 6, 3, 512, device="cuda", generator=torch.Generator(device="cuda").manual_seed(0)).bfloat16())
    with torch.no_grad():
        got, want = norm(x), norm.rms_norm(x)
    assert got.stride() == want.stride()
    assert ((got.float() - want.float()).abs() <= 2.0 ** -6 * want.float().abs() + 1e-6).all()      # one place each, as above


# one to nine key tiles of 64 (32 at a head dim of 256), one to four query tiles of 128, several sequences of each
@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("b,s", [(2, 127), (3, 128), (2, 129), (3, 257), (2, 450), (1, 513)])
def test_causal_attention_tiles(hd, b, s):
    """Attention of whole sequences over several tiles against softmax in fp64, the running maximum rising along the keys.  Weights
    and output are each rounded once, and 2^-8 relative covers both; two runs give the same bits."""
    from nanoquantization_amd import _lib
    print(f"causal attention hd={hd} {b}x{s}", flush=True)
    heads, kv, bf = 6, 2, torch.bfloat16
    gen = torch.Generator(device="cuda").manual_seed(hd + s)
    q = torch.randn(b, s, heads, hd, device="cuda", generator=gen).to(bf)
    k, v = (torch.randn(b, kv, s, hd, device="cuda", generator=gen) for _ in range(2))
    k, v = (k * (1 + torch.arange(s, device="cuda") / 100).view(-1, 1)).to(bf), v.to(bf)
    for scale in (hd ** -0.5, -hd ** -0.5):
        o = _lib.torch_ops().causal_attention(q, k, v, scale)
        rep = lambda t: t.double().repeat_interleave(heads // kv, 1)
        sc = q.transpose(1, 2).double() @ rep(k).transpose(-1, -2) * scale
        w = sc.masked_fill(torch.ones(s, s, dtype=torch.bool, device="cuda").triu(1), float("-inf")).softmax(-1)
        ref = (w @ rep(v)).transpose(1, 2).reshape(b, s, heads * hd)
        size = (w @ rep(v).abs()).transpose(1, 2).reshape(b, s, heads * hd)
        assert ((o.double() - ref).abs() <= 2.0 ** -8 * (size + ref.abs())).all()
        assert torch.equal(o, _lib.torch_ops().causal_attention(q, k, v, scale))


def test_prompt_forward_of_many_tiles(monkeypatch):
    """Several sequences of several attention tiles, rows enough that gate and up are one product: the same hidden states as on
    torch operations, to the few roundings that fall differently."""
    from nanoquantization_amd import _lib
    from nanoquantization_amd.models.qwen3_quantized import Qwen3QuantizedForCausalLM
    b, s, hidden, inter = 3, 700, 512, 1024
    assert _lib.lib().awq_linear_route(b * s, 2 * inter, hidden, 128, _lib.AWQ_BF16, 1, None) == b"dense"
    m = Qwen3QuantizedForCausalLM(num_hidden_layers=2, vocab_size=128, hidden_size=hidden, total_num_heads=6, total_num_kv_heads=2,
                                  max_position_embeddings=1024, intermediate_size=inter, head_dim=128).to(torch.bfloat16)
    torch.manual_seed(0)
    for mod in m.modules():
        if isinstance(mod, nq.WQLinear_GEMM):
            mod.qweight.random_(-2 ** 31, 2 ** 31 - 1)
            mod.qzeros.random_(-2 ** 31, 2 ** 31 - 1)
            mod.qscales.uniform_(0.002, 0.006)
    m = m.cuda()
    ids, pos = torch.randint(0, 128, (b, s), device="cuda"), torch.arange(s, device="cuda")
    with torch.no_grad():
        got = m(ids, pos)
        assert torch.equal(got, m(ids, pos))
        _eager(monkeypatch)
        want = m(ids, pos)
    assert (got.float() - want.float()).norm() <= 2.0 ** -7 * want.float().norm()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("batch,tokens,heads,kv,dim", [
    (1, 1, 1, 1, 128),            # fewer heads than a wave has lanes for
    (3, 5, 16, 8, 128),
    (2, 4099, 24, 8, 128),        # four tokens a workgroup, the last one with three
    (5, 3301, 5, 1, 64),          # an odd head count
    (2, 2050, 40, 8, 256),        # several passes over the heads
    (1, 67, 37, 5, 128),          # fewer waves than the chip holds: heads over workgroups, the last one part full
    (1, 3, 4, 1, 64), (2, 4097, 4, 1, 64), (1, 2, 1, 1, 256),      # a wave has lanes for all heads: five tokens a workgroup, or the sequences there are
    (4098, 1, 4, 1, 64), (513, 3, 1, 1, 128),      # sequences beside one another
    (65537, 1, 5, 1, 128),        # more sequences than the grid's second dimension holds
])
def test_qkv_norm_rope_sizes(dtype, batch, tokens, heads, kv, dim):
    """Head counts and tokens around the kernel's groups, passes and tokens a workgroup, positions per sequence, against the torch expressions in fp32 with
    the module's roundings: the norm and its product with the weight are rounded to the type, the rotary sums only at the end."""
    g = torch.Generator(device="cuda").manual_seed(tokens)
    randn = lambda *n: torch.randn(*n, generator=g, device="cuda")
    q, k, v = (randn(batch, tokens, n * dim).to(dtype) for n in (heads, kv, kv))
    weights = [(1 + 0.1 * randn(dim)).to(dtype) for _ in range(2)]
    angles = randn(64, dim // 2)
    table = torch.cat([angles.cos(), angles.sin()], dim=-1).unsqueeze(1)
    pos = torch.randint(-64, 64, (batch, tokens), generator=g, device="cuda")
    got = torch.ops.nanoquantization_amd.qkv_norm_rope(q, k, v, *weights, table, pos, heads, kv, 1e-6, 1e-5)
    cos, sin = table[pos].chunk(2, dim=-1)
    for x, w, eps, n, out in ((q, weights[0], 1e-6, heads, got[0]), (k, weights[1], 1e-5, kv, got[1])):
        x = x.view(batch, tokens, n, dim).float()
        x = (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)).to(dtype) * w
        a, b = x.float().chunk(2, dim=-1)
        want = torch.cat([a * cos - b * sin, a * sin + b * cos], dim=-1)
        size = torch.cat([(a * cos).abs() + (b * sin).abs(), (a * sin).abs() + (b * cos).abs()], dim=-1)
        out = out if n == heads and out.shape == want.shape else out.view(batch, n, tokens, dim).transpose(1, 2)
        # fp32 sums in another order may move x * r over a rounding's edge: one place (eps of its value at most), carried into the product with
        # the weight, whose own two roundings are half a place away each: 2 eps a term, and half of one for the result's rounding
        assert ((out.view_as(want).float() - want).abs() <= 2.5 * torch.finfo(dtype).eps * size + 1e-6).all()
    assert torch.equal(got[2].view(batch, kv, tokens, dim).transpose(1, 2), v.view(batch, tokens, kv, dim))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,N", [(2048, 512, 1024), (300, 1024, 264), (4097, 256, 1032), (1, 256, 256), (129, 1024, 2560), (2048, 128, 8200)])
def test_linear_with_a_residual(dtype, M, K, N):
    """residual + linear(x) in the product's last step or behind it, whole and part tiles of both sizes: the bits of the two operations."""
    ops = _lib_ops()
    g = torch.Generator(device="cuda").manual_seed(M)
    words = lambda *n: torch.randint(-2 ** 31, 2 ** 31 - 1, n, generator=g, device="cuda", dtype=torch.int64).int()
    w = (words(K, N // 8), (torch.rand(K // 128, N, generator=g, device="cuda") * 0.01 + 0.01).to(dtype), words(K // 128, N // 8))
    x, r = (torch.randn(M, n, generator=g, device="cuda").to(dtype) for n in (K, N))
    want = r + ops.awq_linear(x, *w, None)
    assert torch.equal(ops.awq_linear_add(x, *w, r), want)
    odd = torch.empty(M, N + 1, dtype=dtype, device="cuda")[:, 1:].copy_(r)      # rows that are neither dense nor aligned
    assert torch.equal(ops.awq_linear_add(x, *w, odd), want)
    with pytest.raises(RuntimeError, match="residual must be"):
        ops.awq_linear_add(x, *w, r[:, 8:])


def _lib_ops():
    from nanoquantization_amd import _lib
    return _lib.torch_ops()


def test_block_leaves_its_additions_to_the_products(monkeypatch):
    """The forward of a model with the residual additions in the products before them, and without: the same bits; whoever watches or replaces a part
    of a block hears of every call."""
    import nanoquantization_amd.models.qwen3_quantized as q3
    from nanoquantization_amd.models.random_init import QWEN3_0P6B, random_awq_qwen3
    model = random_awq_qwen3(dict(QWEN3_0P6B, num_hidden_layers=2, vocab_size=512, max_position_embeddings=512), seed=3, std=0.02)
    ids = torch.randint(0, 512, (2, 300), generator=torch.Generator().manual_seed(1)).cuda()
    pos = torch.arange(300, device="cuda").unsqueeze(0)
    calls = []
    with torch.no_grad():
        monkeypatch.setattr(q3, "_ADD_FROM", 1 << 62)
        want = model(ids, pos)
        monkeypatch.setattr(q3, "_ADD_FROM", 0)
        add = q3._add_linear
        monkeypatch.setattr(q3, "_add_linear", lambda *a: (calls.append(a[1]), add(*a))[1])
        assert torch.equal(model(ids, pos), want) and len(calls) == 4
        block = model.model.layers[0]
        for part, expected in ((block.self_attn, 2), (block.mlp, 2), (block.self_attn.o_proj, 4), (block.mlp.down_proj, 4), (block.input_layernorm, 4)):
            heard = []
            hook = part.register_forward_hook(lambda *a: heard.append(1))
            calls.clear()
            assert torch.equal(model(ids, pos), want) and heard == [1] and len(calls) == expected
            hook.remove()
        for part in (block.self_attn, block.mlp, block.self_attn.o_proj, block.mlp.down_proj):
            heard, forward = [], part.forward
            part.forward = lambda *a: (heard.append(1), forward(*a))[1]
            assert torch.equal(model(ids, pos), want) and heard == [1]
            del part.forward

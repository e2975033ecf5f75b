"""What the Qwen3 modules accept around their operators (tracing, scripting, replaced parts), without a device: where the
operators themselves would run, stand-ins do."""
import os
import types
import warnings

import pytest
import torch
import torch.fx

import nanoquantization_amd as nq
from nanoquantization_amd import _lib
from nanoquantization_amd.layers import norm as norm_module
from nanoquantization_amd.layers.norm import RMSNorm
from nanoquantization_amd.layers.rope import RoPE
from nanoquantization_amd.models import qwen3_quantized as q3
from nanoquantization_amd.models.qwen3_quantized import Qwen3QuantizedAttention, Qwen3QuantizedMLP


@pytest.mark.parametrize("n", [64, 1024])
def test_norm_can_be_traced_and_scripted(n):
    norm = RMSNorm(n)
    norm.weight.data = torch.randn(n, generator=torch.Generator().manual_seed(0))
    x = torch.randn(3, n, generator=torch.Generator().manual_seed(1))
    want = norm.rms_norm(x)
    assert torch.equal(torch.fx.symbolic_trace(norm)(x), want)
    assert torch.equal(torch.jit.script(norm)(x), want)
    with warnings.catch_warnings():
        warnings.simplefilter("error", torch.jit.TracerWarning)
        traced = torch.jit.trace(norm, (x,))
    assert torch.equal(traced(x[:2]), want[:2])


LAYOUTS = [lambda x: x, lambda x: x.transpose(0, 1), lambda x: x.permute(2, 0, 1, 3), lambda x: x[:, -1], lambda x: x[:, ::2],
           lambda x: x.transpose(-1, -2).contiguous().transpose(-1, -2), lambda x: x[:1].expand(4, -1, -1, -1),
           lambda x: torch.cat([x, x], -1)[..., :x.shape[-1]].transpose(0, 2)]


@pytest.mark.parametrize("layout", range(len(LAYOUTS)))
def test_norm_result_keeps_the_layout(layout):
    """The operator's result has the strides of the torch expression's."""
    if not os.path.exists(_lib.TORCH_LIB_PATH):
        from nanoquantization_amd.build import build
        build(verbose=False)
    norm = RMSNorm(512).to(torch.bfloat16)
    x = LAYOUTS[layout](torch.randn(4, 6, 3, 512).bfloat16())
    like = torch.empty_strided(x.shape, x.stride(), dtype=x.dtype, device="meta")
    got = _lib.torch_ops().rms_norm(like, norm.weight.detach().to("meta"), norm.eps)
    assert got.shape == x.shape and got.stride() == norm.rms_norm(x).stride()


def test_mlp_can_be_traced_with_its_linears_as_leaves():
    class Tracer(torch.fx.Tracer):
        def is_leaf_module(self, m, name):
            return isinstance(m, nq.WQLinear_GEMM) or super().is_leaf_module(m, name)

    graph = Tracer().trace(Qwen3QuantizedMLP(64, 128, group_size=64))
    called = [n.target for n in graph.nodes if n.op == "call_module"]
    assert sorted(called) == ["down_proj", "gate_proj", "up_proj"]


@pytest.mark.parametrize("what", ["block", "model"])
def test_block_can_be_traced_with_its_parts_as_leaves(what):
    leaves = (Qwen3QuantizedAttention, Qwen3QuantizedMLP, RMSNorm, torch.nn.Embedding)

    class Tracer(torch.fx.Tracer):
        def is_leaf_module(self, m, name):
            return isinstance(m, leaves) or super().is_leaf_module(m, name)

    sizes = dict(group_size=64, hidden_size=64, total_num_heads=4, total_num_kv_heads=2, max_position_embeddings=32, intermediate_size=128, head_dim=64)
    parts = ["input_layernorm", "self_attn", "post_attention_layernorm", "mlp"]
    if what == "block":
        graph = Tracer().trace(q3.Qwen3QuantizedBlock(**sizes))
    else:
        graph = Tracer().trace(q3.Qwen3QuantizedModel(num_hidden_layers=2, vocab_size=96, **sizes))
        parts = ["embed_tokens", *(f"layers.{i}.{p}" for i in range(2) for p in parts), "norm"]
    assert [n.target for n in graph.nodes if n.op == "call_module"] == parts


class Product(torch.nn.Module):
    def __init__(self, n, m):
        super().__init__()
        self.w = torch.nn.Parameter(torch.randn(n, m, generator=torch.Generator().manual_seed(n + m)))

    def forward(self, x):
        return x @ self.w


@pytest.mark.parametrize("how", ["script", "trace", "compile"])
def test_attention_and_mlp_on_other_linears(how):
    """With linears that can be traced, scripted and compiled the modules can be as well, and give the same result."""
    mlp, attn = Qwen3QuantizedMLP(64, 128, group_size=64), Qwen3QuantizedAttention(64, 4, 2, 32, head_dim=64, group_size=64)
    mlp.gate_proj, mlp.up_proj, mlp.down_proj = Product(64, 128), Product(64, 128), Product(128, 64)
    attn.q_proj, attn.k_proj, attn.v_proj, attn.o_proj = Product(64, 256), Product(64, 128), Product(64, 128), Product(256, 64)
    x, pos = torch.randn(2, 5, 64, generator=torch.Generator().manual_seed(0)), torch.arange(5)
    with torch.no_grad():
        for module, args in ((mlp, (x,)), (attn, (x, pos)), (attn, (x, pos.expand(2, 5)))):
            made = {"script": torch.jit.script, "trace": lambda m: torch.jit.trace(m, args),
                    "compile": lambda m: torch.compile(m, backend="eager", fullgraph=True)}[how](module)
            assert torch.allclose(made(*args), module(*args), rtol=1e-5, atol=1e-5)


@pytest.fixture
def operators(monkeypatch):
    """The operators' names in the order they were called, where every tensor counts as one they take; the tensors they return
    have the right shapes."""
    seen = []

    def qkv_norm_rope(q, k, v, qw, kw, table, pos, heads, kv_heads, *eps):
        seen.append("qkv_norm_rope")
        b, s, hd = q.shape[0], q.shape[1], q.shape[2] // heads
        return q.view(b, s, heads, hd), *(t.reshape(b, s, kv_heads, hd).transpose(1, 2).contiguous() for t in (k, v))

    def pair(x, *weights):
        seen.append("awq_swiglu_pair")
        return x.new_zeros(x.shape[0], weights[1].shape[1])

    def rms_norm(x, *rest):
        seen.append("rms_norm")
        return torch.zeros_like(x)

    ops = types.SimpleNamespace(qkv_norm_rope=qkv_norm_rope, awq_swiglu_pair=pair, rms_norm=rms_norm,
                                silu_mul=lambda g, u: g * u, causal_attention=lambda q, k, v, scale: q.flatten(2))
    monkeypatch.setattr(_lib, "torch_ops", lambda: ops)
    for mod in (norm_module, q3):
        monkeypatch.setattr(mod, "plain", lambda *t: True)
    return seen


def _attention():
    attn = Qwen3QuantizedAttention(64, 4, 2, 32, head_dim=64, group_size=64)
    gen = torch.Generator().manual_seed(0)
    for name, heads in (("q_proj", 4), ("k_proj", 2), ("v_proj", 2)):       # the projections run on a device only
        w = torch.randn(64, heads * 64, generator=gen)
        getattr(attn, name).forward = lambda x, w=w: x @ w
    attn.o_proj.forward = lambda x: x
    return attn, torch.randn(2, 5, 64, generator=gen), torch.arange(5)


@pytest.mark.parametrize("where", ["module", "class"])
@pytest.mark.parametrize("part,cls,method", [("q_norm", RMSNorm, "forward"), ("k_norm", RMSNorm, "rms_norm"), ("rope", RoPE, "forward"),
                                             ("rope", RoPE, "apply_rope")])
def test_attention_calls_replaced_parts(operators, monkeypatch, where, part, cls, method):
    attn, x, pos = _attention()
    with torch.no_grad():
        attn(x, pos)
        assert operators == ["qkv_norm_rope"]
        called, before = [], getattr(cls, method)

        def replaced(*args):
            called.append(method)
            return before(*(args if where == "class" or isinstance(cls.__dict__[method], staticmethod) else (getattr(attn, part), *args)))
        if where == "class":
            monkeypatch.setattr(cls, method, staticmethod(replaced) if isinstance(cls.__dict__[method], staticmethod) else replaced)
        else:
            setattr(getattr(attn, part), method, replaced)
        attn(x, pos)
    assert called and operators == ["qkv_norm_rope"]


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_attention_refuses_positions_outside_the_table(operators, dtype):
    attn, x, pos = _attention()                 # a table of 32 positions
    with torch.no_grad():
        for first in (0, 27, -32):
            attn(x, (pos + first).to(dtype))
            attn(x, (pos + first).expand(2, 5).to(dtype))
        assert operators == ["qkv_norm_rope"] * 6
        for first in (28, 1 << 20, -33):
            with pytest.raises(IndexError):
                attn(x, (pos + first).to(dtype))
            with pytest.raises(IndexError):
                attn(x, (pos + first).expand(2, 5).to(dtype))
    assert operators == ["qkv_norm_rope"] * 6


def test_attention_leaves_other_shapes_to_torch(operators):
    """Norm weights per head and a table of other strides, which broadcasting and indexing take; a table of another head size,
    which they refuse."""
    attn, x, pos = _attention()
    with torch.no_grad():
        attn.q_norm.weight = torch.nn.Parameter(torch.rand(4, 64))
        attn(x, pos)
        attn, x, pos = _attention()
        want = attn.qkv(x, pos)
        attn.rope.cos_sin_cache = attn.rope.cos_sin_cache.transpose(0, 2).contiguous().transpose(0, 2)
        attn(x, pos)
        assert all(torch.equal(a, b) for a, b in zip(attn.qkv(x, pos), want))
        attn.rope = RoPE(32, 64)
        with pytest.raises(RuntimeError):
            attn(x, pos)
    assert operators == []


def test_mlp_broadcasts_as_torch_does(operators):
    mlp, x = Qwen3QuantizedMLP(64, 128, group_size=64), torch.randn(2, 3, 64)
    mlp.gate_proj, mlp.up_proj, mlp.down_proj = torch.nn.Linear(64, 128), torch.nn.Linear(64, 1), torch.nn.Identity()
    called = []
    _lib.torch_ops().silu_mul = lambda g, u: called.append("silu_mul") or g * u
    want = torch.nn.functional.silu(mlp.gate_proj(x)) * mlp.up_proj(x)
    assert torch.equal(mlp(x), want) and called == []


@pytest.mark.parametrize("where", ["module", "subclass"])
def test_attention_calls_a_replaced_qkv(operators, where):
    attn, x, pos = _attention()
    called, before = [], attn.qkv

    def replaced(x, position_ids):
        called.append("qkv")
        return before(x, position_ids)
    if where == "module":
        attn.qkv = replaced
    else:
        attn.__class__ = type("Sub", (Qwen3QuantizedAttention,), {"qkv": lambda self, x, position_ids: replaced(x, position_ids)})
    with torch.no_grad():
        attn(x, pos)
    assert called == ["qkv"] and operators == []


@pytest.mark.parametrize("where", ["gate_proj", "up_proj", "class"])
def test_mlp_calls_replaced_linears(operators, monkeypatch, where):
    mlp, x = Qwen3QuantizedMLP(64, 128, group_size=64), torch.randn(2, 3, 64)
    mlp.down_proj.forward = lambda a: a
    mlp(x)
    assert operators == ["awq_swiglu_pair"]
    called = []

    def replaced(*args):
        called.append(where)
        return args[-1].new_ones(*args[-1].shape[:-1], 128)
    if where == "class":
        monkeypatch.setattr(nq.WQLinear_GEMM, "forward", replaced)
        mlp(x)
        assert called == ["class", "class"]
    else:
        setattr(getattr(mlp, where), "forward", replaced)
        with pytest.raises(_lib.AwqHipError):       # the other projection, which needs a device
            mlp(x)
        assert where == "up_proj" or called == ["gate_proj"]
    assert operators == ["awq_swiglu_pair"]


@pytest.mark.parametrize("where", ["module", "class"])
def test_norm_calls_a_replaced_rms_norm(operators, monkeypatch, where):
    norm, x = RMSNorm(1024), torch.randn(2, 1024)
    norm(x)
    assert operators == ["rms_norm"]
    if where == "class":
        monkeypatch.setattr(RMSNorm, "rms_norm", lambda self, x: x + 1)
    else:
        norm.rms_norm = lambda x: x + 1
    assert torch.equal(norm(x), x + 1) and operators == ["rms_norm"]

"""Qwen3 with AWQ linears: the callers of the hot path, same modules, constructor arguments and
parameter/buffer names as nanoquantization/models/qwen3_quantized.py (so its checkpoints load
unchanged), on this package's WQLinear_GEMM.

`forward(x, position_ids)` is the reference's full-sequence causal forward (no cache,
models/qwen3_quantized.py:65-102, 139-153, 194-215, 259-273).  The engine
(nanoquantization_amd/engine) drives the same weights through a paged KV cache; the reference has
no counterpart for that.
"""
from __future__ import annotations

from typing import Optional

import torch
import torch.nn as nn
import torch.nn.functional as F

from .. import _lib
from ..layers.gemm import WQLinear_GEMM
from ..layers.inference import keeps, plain, shipped, unhooked
from ..layers.norm import RMSNorm
from ..layers.rope import RoPE


_ADD_FROM = 1 << 20      # elements from which an addition is worth more than the questions whether it can be left to the product before it


def _add_linear(residual: torch.Tensor, linear: nn.Module, x: torch.Tensor) -> torch.Tensor:
    """residual + linear(x): one operator where the linear is this package's, unchanged and watched by no hook."""
    if (type(linear) is WQLinear_GEMM and linear.bias is None and keeps(linear, WQLinear_GEMM, "forward") and plain(x, linear.qscales, residual)
            and linear.qscales.dim() == 2 and residual.is_contiguous() and x.shape[:-1] == residual.shape[:-1]
            and residual.shape[-1] == linear.qscales.shape[-1] and unhooked(linear)):
        y = _lib.torch_ops().awq_linear_add(x.reshape(-1, x.shape[-1]), linear.qweight, linear.qscales, linear.qzeros,
                                            residual.view(-1, residual.shape[-1]))
        return y.view(residual.shape)
    return residual + linear(x)


@shipped("qkv", "forward")
class Qwen3QuantizedAttention(nn.Module):
    def __init__(self, hidden_size: int, total_num_heads: int, total_num_kv_heads: int,
                 max_position_embeddings: int, w_bits: int = 4, group_size: int = 128,
                 head_dim: Optional[int] = None, rope_theta: float = 10000, rms_norm_eps: float = 1e-6):
        super().__init__()
        self.head_dim = head_dim or hidden_size // total_num_heads
        self.hidden_size = hidden_size
        self.num_heads = total_num_heads
        self.num_kv_heads = total_num_kv_heads
        self.max_position_embeddings = max_position_embeddings
        self.rope = RoPE(self.head_dim, max_position_embeddings, rope_theta)
        mk = lambda i, o: WQLinear_GEMM(w_bits=w_bits, group_size=group_size, in_features=i, out_features=o)
        self.q_proj = mk(hidden_size, total_num_heads * self.head_dim)
        self.k_proj = mk(hidden_size, total_num_kv_heads * self.head_dim)
        self.v_proj = mk(hidden_size, total_num_kv_heads * self.head_dim)
        self.o_proj = mk(total_num_heads * self.head_dim, hidden_size)
        self.q_norm = RMSNorm(self.head_dim, rms_norm_eps)
        self.k_norm = RMSNorm(self.head_dim, rms_norm_eps)

    def qkv(self, x: torch.Tensor, position_ids: torch.Tensor):
        """Projections, per-head q/k RMSNorm, rotary: [b, s, heads, d], [b, s, kv, d], [b, s, kv, d]."""
        return self._norm_rope(self.q_proj(x), self.k_proj(x), self.v_proj(x), position_ids)

    def _norm_rope(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, position_ids: torch.Tensor):
        bs = q.shape[0]
        if position_ids.dim() == 1:
            position_ids = position_ids.unsqueeze(0)
        q = q.view(bs, -1, self.num_heads, self.head_dim)
        k = k.view(bs, -1, self.num_kv_heads, self.head_dim)
        v = v.view(bs, -1, self.num_kv_heads, self.head_dim)
        q, k = self.rope(self.q_norm(q), self.k_norm(k), position_ids)
        return q, k, v

    def _fused(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, pos: torch.Tensor) -> bool:
        """Whether norms, rotary and the move of k and v into head order run as one kernel: the head dims it is built for, a
        position per token, and norms and rotary that are the ones of this package, unchanged and watched by no hook."""
        return (type(pos) is torch.Tensor and plain(q, k, v, self.q_norm.weight, self.k_norm.weight)
                and q.dim() == 3 and self.head_dim in (64, 128, 256) and pos.dtype in (torch.int32, torch.int64) and pos.dim() in (1, 2) and pos.shape[-1] == q.shape[1]
                and (pos.dim() == 1 or pos.shape[0] in (1, q.shape[0]))
                and type(self.q_norm) is type(self.k_norm) is RMSNorm and type(self.rope) is RoPE
                and keeps(self.q_norm, RMSNorm, "forward", "rms_norm") and keeps(self.k_norm, RMSNorm, "forward", "rms_norm")
                and keeps(self.rope, RoPE, "forward", "apply_rope")
                and self.q_norm.weight.shape == self.k_norm.weight.shape == (self.head_dim,)
                and self.rope.cos_sin_cache.dtype == torch.float32 and self.rope.cos_sin_cache.shape[1:] == (1, self.head_dim)
                and self.rope.cos_sin_cache.is_contiguous() and pos.device == q.device == self.rope.cos_sin_cache.device
                and unhooked(self.q_norm, self.k_norm, self.rope))

    def _attend(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
        """Causal attention and output projection of what `qkv` returns."""
        o = F.scaled_dot_product_attention(q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2), is_causal=True,
                                           enable_gqa=self.num_heads != self.num_kv_heads)
        return self.o_proj(o.transpose(1, 2).reshape(q.shape[0], -1, self.num_heads * self.head_dim))

    def _project(self, x: torch.Tensor):
        """q, k and v: one call, which may be one launch, where the projections are this package's, unchanged and watched by no hook."""
        parts = (self.q_proj, self.k_proj, self.v_proj)
        if (all(type(m) is WQLinear_GEMM and m.bias is None and keeps(m, WQLinear_GEMM, "forward") for m in parts)
                and plain(x, *(m.qscales for m in parts)) and x.dim() > 1
                and all(m.qweight.dim() == m.qscales.dim() == m.qzeros.dim() == 2 and m.qweight.shape[0] == x.shape[-1]
                        and m.qscales.shape[0] == parts[0].qscales.shape[0] for m in parts) and unhooked(*parts)):
            out = _lib.torch_ops().awq_linear_three(x.reshape(-1, x.shape[-1]), *(t for m in parts for t in (m.qweight, m.qscales, m.qzeros)))
            return tuple(y.view(*x.shape[:-1], y.shape[-1]) for y in out)
        return self.q_proj(x), self.k_proj(x), self.v_proj(x)

    def _on_operators(self, x: torch.Tensor, position_ids: torch.Tensor, residual: Optional[torch.Tensor] = None) -> torch.Tensor:
        """With a residual: the sum of it and what the module returns."""
        added = (lambda y: y) if residual is None else lambda y: residual + y
        q, k, v = self._project(x)
        if not self._fused(q, k, v, position_ids):
            q, k, v = self._norm_rope(q, k, v, position_ids)
            return added(self._attend(q, k, v))
        pos = (position_ids if position_ids.dim() == 2 else position_ids.unsqueeze(0)).to(torch.int64)
        self.rope.refuse_unknown(pos)
        q, k, v = _lib.torch_ops().qkv_norm_rope(q, k, v, self.q_norm.weight, self.k_norm.weight, self.rope.cos_sin_cache, pos,
                                                 self.num_heads, self.num_kv_heads, self.q_norm.eps, self.k_norm.eps)
        if q.dtype == torch.bfloat16:
            o = _lib.torch_ops().causal_attention(q, k, v, self.head_dim ** -0.5)
            return self.o_proj(o) if residual is None else _add_linear(residual, self.o_proj, o)
        return added(self._attend(q, k.transpose(1, 2), v.transpose(1, 2)))

    def forward(self, x: torch.Tensor, position_ids: torch.Tensor) -> torch.Tensor:
        if not torch.jit.is_scripting():        # script sees the torch expressions only
            if not torch.compiler.is_compiling() and keeps(self, Qwen3QuantizedAttention, "qkv"):
                return self._on_operators(x, position_ids)
        q, k, v = self.qkv(x, position_ids)
        return self._attend(q, k, v)


@shipped("forward")
class Qwen3QuantizedMLP(nn.Module):
    def __init__(self, hidden_size: int, intermediate_size: int, w_bits: int = 4, group_size: int = 128):
        super().__init__()
        self.hidden_size = hidden_size
        self.intermediate_size = intermediate_size
        mk = lambda i, o: WQLinear_GEMM(w_bits=w_bits, group_size=group_size, in_features=i, out_features=o)
        self.up_proj = mk(hidden_size, intermediate_size)
        self.gate_proj = mk(hidden_size, intermediate_size)
        self.down_proj = mk(intermediate_size, hidden_size)

    def _activation(self, x: torch.Tensor) -> torch.Tensor:
        g, u = self.gate_proj, self.up_proj
        if (type(g) is type(u) is WQLinear_GEMM and plain(x, g.qscales, u.qscales) and g.bias is None and u.bias is None
                and g.qweight.shape == u.qweight.shape and g.qscales.shape == u.qscales.shape and x.shape[-1] == g.qweight.shape[0]
                and x.dim() > 1 and keeps(g, WQLinear_GEMM, "forward") and keeps(u, WQLinear_GEMM, "forward") and unhooked(g, u)):
            act = _lib.torch_ops().awq_swiglu_pair(x.reshape(-1, x.shape[-1]), g.qweight, g.qscales, g.qzeros, u.qweight, u.qscales,
                                                   u.qzeros)
            return act.view(*x.shape[:-1], act.shape[-1])
        gate, up = self.gate_proj(x), self.up_proj(x)
        if plain(gate, up) and gate.shape == up.shape and gate.shape[-1] % 8 == 0:
            return _lib.torch_ops().silu_mul(gate, up)
        return F.silu(gate) * up

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if not torch.jit.is_scripting():        # script sees the torch expression only
            return self.down_proj(self._activation(x))
        return self.down_proj(F.silu(self.gate_proj(x)) * self.up_proj(x))


class Qwen3QuantizedBlock(nn.Module):
    def __init__(self, hidden_size: int, total_num_heads: int, total_num_kv_heads: int,
                 max_position_embeddings: int, intermediate_size: int, w_bits: int = 4, group_size: int = 128,
                 head_dim: Optional[int] = None, rope_theta: float = 10000, rms_norm_eps: float = 1e-6):
        super().__init__()
        self.hidden_size = hidden_size
        self.intermediate_size = intermediate_size
        self.self_attn = Qwen3QuantizedAttention(hidden_size, total_num_heads, total_num_kv_heads,
                                                 max_position_embeddings, w_bits, group_size, head_dim,
                                                 rope_theta, rms_norm_eps)
        self.mlp = Qwen3QuantizedMLP(hidden_size, intermediate_size, w_bits, group_size)
        self.input_layernorm = RMSNorm(hidden_size, rms_norm_eps)
        self.post_attention_layernorm = RMSNorm(hidden_size, rms_norm_eps)

    def _adds_in_products(self, x: torch.Tensor) -> bool:
        """Whether the residual additions may go with the products before them: enough rows, and an attention and an MLP that are the ones of
        this package, unchanged and watched by no hook."""
        attn, mlp = self.self_attn, self.mlp
        return (plain(x) and x.numel() >= _ADD_FROM and x.is_contiguous() and type(attn) is Qwen3QuantizedAttention
                and type(mlp) is Qwen3QuantizedMLP and keeps(attn, Qwen3QuantizedAttention, "qkv", "forward")
                and keeps(mlp, Qwen3QuantizedMLP, "forward") and unhooked(attn, mlp))

    def forward(self, x: torch.Tensor, position_ids: torch.Tensor) -> torch.Tensor:
        if not torch.jit.is_scripting():        # script sees the torch expressions only
            if not torch.compiler.is_compiling() and not torch.jit.is_tracing() and self._adds_in_products(x):
                x = self.self_attn._on_operators(self.input_layernorm(x), position_ids, x)
                return _add_linear(x, self.mlp.down_proj, self.mlp._activation(self.post_attention_layernorm(x)))
        x = x + self.self_attn(self.input_layernorm(x), position_ids)
        return x + self.mlp(self.post_attention_layernorm(x))


class Qwen3QuantizedModel(nn.Module):
    def __init__(self, num_hidden_layers: int, vocab_size: int, hidden_size: int, total_num_heads: int,
                 total_num_kv_heads: int, max_position_embeddings: int, intermediate_size: int,
                 w_bits: int = 4, group_size: int = 128, head_dim: Optional[int] = None,
                 rope_theta: float = 10000, rms_norm_eps: float = 1e-6):
        super().__init__()
        self.layers = nn.ModuleList([
            Qwen3QuantizedBlock(hidden_size, total_num_heads, total_num_kv_heads, max_position_embeddings,
                                intermediate_size, w_bits, group_size, head_dim, rope_theta, rms_norm_eps)
            for _ in range(num_hidden_layers)])
        self.norm = RMSNorm(hidden_size, rms_norm_eps)
        self.embed_tokens = nn.Embedding(vocab_size, hidden_size)

    def forward(self, x: torch.Tensor, position_ids: torch.Tensor) -> torch.Tensor:
        x = self.embed_tokens(x)
        for layer in self.layers:
            x = layer(x, position_ids)
        return self.norm(x)


class Qwen3QuantizedForCausalLM(nn.Module):
    def __init__(self, num_hidden_layers: int, vocab_size: int, hidden_size: int, total_num_heads: int,
                 total_num_kv_heads: int, max_position_embeddings: int, intermediate_size: int,
                 w_bits: int = 4, group_size: int = 128, head_dim: Optional[int] = None,
                 tie_word_embeddings: bool = False, rope_theta: float = 10000, rms_norm_eps: float = 1e-6):
        super().__init__()
        self.model = Qwen3QuantizedModel(num_hidden_layers, vocab_size, hidden_size, total_num_heads,
                                         total_num_kv_heads, max_position_embeddings, intermediate_size,
                                         w_bits, group_size, head_dim, rope_theta, rms_norm_eps)
        self.lm_head = nn.Linear(hidden_size, vocab_size)   # un-quantised, with a bias, as in the reference
        if tie_word_embeddings:
            self.lm_head.weight.data = self.model.embed_tokens.weight.data

    def forward(self, x: torch.Tensor, position_ids: torch.Tensor) -> torch.Tensor:
        return self.model(x, position_ids)

    def logits(self, hidden_states: torch.Tensor) -> torch.Tensor:
        return self.lm_head(hidden_states)

    def compute_loss(self, x: torch.Tensor, labels: torch.Tensor) -> torch.Tensor:
        position_ids = torch.arange(x.shape[1], dtype=torch.int32, device=x.device).unsqueeze(0)
        logits = self.lm_head(self.model(x, position_ids))
        return F.cross_entropy(logits.view(-1, logits.shape[-1]).float(), labels.view(-1))

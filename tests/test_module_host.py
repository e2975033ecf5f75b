"""What the Qwen3 modules accept around their operators (tracing, scripting, replaced parts), without a device: where the
operators themselves would run, stand-ins do."""
import warnings

import pytest
import torch
import torch.fx

import nanoquantization_amd as nq
from nanoquantization_amd.layers.norm import RMSNorm
from nanoquantization_amd.models.qwen3_quantized import Qwen3QuantizedMLP


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


def test_mlp_can_be_traced_with_its_linears_as_leaves():
    class Tracer(torch.fx.Tracer):
        def is_leaf_module(self, m, name):
            return isinstance(m, nq.WQLinear_GEMM) or super().is_leaf_module(m, name)

    graph = Tracer().trace(Qwen3QuantizedMLP(64, 128, group_size=64))
    called = [n.target for n in graph.nodes if n.op == "call_module"]
    assert sorted(called) == ["down_proj", "gate_proj", "up_proj"]

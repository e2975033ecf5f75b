"""When the modules may run on this library's operators between the AWQ linears (norms, rotary, attention, SiLU).  Those compute
what the torch expressions beside them do, with the same rounding points, but have no derivatives and no rules for torch's
function transforms: with any of these in play the torch expressions run."""
from __future__ import annotations

import torch
from torch.autograd import forward_ad
from torch.nn import Parameter

_PLAIN = (torch.Tensor, Parameter)


def plain(*tensors: torch.Tensor) -> bool:
    """Ordinary 16-bit HIP tensors of one type and device, no gradient wanted, no tracing, no transform, no autocast.  To be
    asked before any other condition on the tensors."""
    # types and modes before any property: a tracer's stand-in has no device to compare, and a traced size warns
    if torch.compiler.is_compiling() or torch.jit.is_tracing() or any(type(t) not in _PLAIN for t in tensors):
        return False
    if forward_ad._current_level >= 0 or torch._C._are_functorch_transforms_active():
        return False
    first = tensors[0]
    if first.device.type != "cuda" or first.dtype not in (torch.float16, torch.bfloat16) or torch.is_autocast_enabled("cuda"):
        return False
    grad = torch.is_grad_enabled()
    return all(t.dtype == first.dtype and t.device == first.device and not (grad and t.requires_grad) for t in tensors)


def unhooked(*modules: torch.nn.Module) -> bool:
    """No caller wants to see the inputs or outputs of these modules."""
    return not (torch.nn.modules.module._has_any_global_hook() or any(m._forward_hooks or m._forward_pre_hooks for m in modules))

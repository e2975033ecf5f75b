"""When the modules may run on this library's operators between the AWQ linears (norms, rotary, attention, SiLU).  Those compute
what the torch expressions beside them do, with the same rounding points, but have no derivatives and no rules for torch's
function transforms, and they pass over the modules whose work they take: with a gradient, a transform, a hook or a replaced
method in play the torch expressions run."""
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


_SHIPPED = {}      # (class, method name) -> the method as this package defines it


def shipped(*names: str):
    """Class decorator: remembers these methods, for `keeps`."""
    def remember(cls):
        _SHIPPED.update({(cls, n): getattr(cls, n) for n in names})
        return cls
    return remember


def keeps(module: torch.nn.Module, cls: type, *names: str) -> bool:
    """These methods of the module are still those of `cls`: replaced neither on the module nor on its class."""
    return all(n not in module.__dict__ and getattr(type(module), n, None) is _SHIPPED[cls, n] for n in names)


def is_torch_linear(module: torch.nn.Module) -> bool:
    """An nn.Linear with the forward that torch gives it, replaced neither on the module nor on the class."""
    return (type(module) is torch.nn.Linear and "forward" not in module.__dict__
            and getattr(torch.nn.Linear.forward, "__globals__", None) is vars(torch.nn.modules.linear))


def unhooked(*modules: torch.nn.Module) -> bool:
    """No caller wants to see the inputs or outputs of these modules."""
    return not (torch.nn.modules.module._has_any_global_hook() or any(m._forward_hooks or m._forward_pre_hooks for m in modules))

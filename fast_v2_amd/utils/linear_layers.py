"""Linear layers of few token rows on the weight-streaming kernels.

A layer is taken over only where its call is the plain product (an ``nn.Linear`` itself,
without hooks), nothing else has a say in it (``replaceable``) and ``ops.linear_fits`` holds;
every other call runs the module."""
from __future__ import annotations

import torch
import torch.nn as nn
import torch.nn.modules.module as _every_module
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from .. import ops


def plain_linear(mod: nn.Module) -> bool:
    """A torch linear layer whose call is its product alone: no subclass (adapters,
    quantised or parametrised layers), no replaced forward and no hooks to run, the layer's
    own or those on every module (profilers, debuggers)."""
    return (type(mod) is nn.Linear and "forward" not in mod.__dict__ and not mod._forward_hooks and
            not mod._forward_pre_hooks and not mod._backward_hooks and not mod._backward_pre_hooks and
            not _every_module._global_forward_hooks and not _every_module._global_forward_pre_hooks and
            not _every_module._global_backward_hooks and not _every_module._global_backward_pre_hooks)


def replaceable(x: torch.Tensor) -> bool:
    """Whether a layer's call on ``x`` is, as things stand, nothing but its product: no
    autocast to another type, no tracing, and no mode (a FLOP counter, a tracer) that
    expects to see it. A default device is a mode too, but concerns new tensors only."""
    return (x.is_cuda and not torch.compiler.is_compiling() and not torch._C._len_torch_dispatch_stack() and
            (not torch._C._len_torch_function_stack() or
             all(type(m) is DeviceContext for m in _get_current_function_mode_stack())) and
            torch._C._get_tracing_state() is None and
            (not torch.is_autocast_enabled("cuda") or torch.get_autocast_dtype("cuda") == x.dtype))


def streams(x: torch.Tensor, *mods: nn.Module) -> bool:
    """Whether every one of ``mods`` (layers of x) runs on the weight-streaming kernels."""
    return (replaceable(x) and
            all(plain_linear(m) and ops.linear_fits(x, m.weight, bias=m.bias) for m in mods))


def project(mod: nn.Module, x: torch.Tensor) -> torch.Tensor:
    """``mod(x)``. 16 x 8 rows of the 7B layout: down_proj 42 us against 99 in the library's
    GEMM."""
    if replaceable(x) and plain_linear(mod):
        y = ops.try_linear(x, mod.weight, None, mod.bias)
        if y is not None:
            return y
    return mod(x)


def gated(gate: nn.Module, up: nn.Module, x: torch.Tensor) -> torch.Tensor:
    """``silu(gate(x)) * up(x)`` (modeling.py:164). 16 x 8 rows of the 7B layout: 57 us
    against 79 for the two layers and the product kernel."""
    if replaceable(x) and gate.bias is None and up.bias is None and plain_linear(gate) and plain_linear(up):
        y = ops.try_linear(x, gate.weight, up.weight)
        if y is not None:
            return y
    return ops.silu_mul(gate(x), up(x))


__all__ = ["plain_linear", "replaceable", "streams", "project", "gated"]

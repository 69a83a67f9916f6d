"""Linear layers of few token rows on the weight-streaming kernels.

A layer is taken over only where its call is the plain product (an ``nn.Linear`` itself,
without hooks), nothing else has a say in it (``replaceable``), ``ops.linear_fits`` holds and
the kernel is the faster one (``pays``); every other call runs the module."""
from __future__ import annotations

import functools

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


@functools.lru_cache(maxsize=4096)
def pays(rows: int, n: int, k: int, gated: bool) -> bool:
    """Whether the kernel is the faster one for [rows, k] activations and n output columns,
    against the library's GEMM (gated: two of them and the product kernel). Measured on 49
    layers at 1-128 rows (cold weights, bf16); time over the library's in brackets, ranges
    over the rows. The tiles are those of csrc/linear.hip, 64 or 160 columns, for 256 compute
    units; rules are on sizes where the measured ones turn.

    gated, tiles that fit one round (0.35-0.93), more of them up to 32 rows (28672 x 8192:
    0.74-0.82, 0.96-1.08 above).
    n < 8192 (down_proj, o_proj): 0.41-0.99, but small weights above 64 rows (896 x 4864,
    1536 x 1536, 2048 x 2048: 1.11-1.37) and very small ones (896 x 896: 0.90-1.22).
    n = 8192: with longer k (28672: 0.58-1.02), not at 8192 x 8192 (0.95-1.42).
    n up to 16384, not cut over k: up to 16 rows (0.78-0.99; 0.88-1.07 above).
    n from 16384 (lm_head): up to 48 rows where the tiles are one round (0.71-0.99; 0.73-1.18
    above), cut over k only if they nearly fill it (18944, 20480 columns: 0.41-0.97; 16384:
    1.02-1.14). Several rounds at any row count if the last is nearly full (151936 x 896 and
    x 1536: 0.48-0.95; 152064 x 3584 0.72-1.04 by itself, and a two-layer step is shorter by 5-19
    us at every count, 581 against 600 at 128 rows); not 51200 and 128256, which it is not:
    0.99-1.22."""
    wide = n * (2 if gated else 1) >= 16384
    per = (160 if wide else 64) // (2 if gated else 1)
    tiles = -(-n // per)
    if gated:
        return tiles <= 256 or rows <= 32
    if n <= 8192:
        return n * k >= 1 << (21 if rows <= 64 else 23) and (n < 8192 or k > n)
    if not wide:
        return rows <= 16
    wgs = tiles * (2 if tiles <= 128 else 1)
    return (rows <= 48 or tiles > 256) and (128 < tiles <= 256 or wgs >= 0.9 * 256 * -(-wgs // 256))


def _rows(x: torch.Tensor) -> int:
    return x.numel() // max(x.shape[-1], 1) if x.dim() else 0


def streams(x: torch.Tensor, *mods: nn.Module) -> bool:
    """Whether the weight-streaming kernels take every one of ``mods`` (layers of x)."""
    return (replaceable(x) and
            all(plain_linear(m) and ops.linear_fits(x, m.weight, bias=m.bias) for m in mods))


def project(mod: nn.Module, x: torch.Tensor) -> torch.Tensor:
    """``mod(x)``. 16 x 8 rows of the 7B layout: down_proj 42 us against 99 in the library's
    GEMM."""
    if replaceable(x) and plain_linear(mod) and pays(_rows(x), mod.out_features, mod.in_features, False):
        y = ops.try_linear(x, mod.weight, None, mod.bias)
        if y is not None:
            return y
    return mod(x)


def gated(gate: nn.Module, up: nn.Module, x: torch.Tensor) -> torch.Tensor:
    """``silu(gate(x)) * up(x)`` (modeling.py:164). 16 x 8 rows of the 7B layout: 57 us
    against 79 for the two layers and the product kernel."""
    if (replaceable(x) and gate.bias is None and up.bias is None and plain_linear(gate) and plain_linear(up) and
            pays(_rows(x), gate.out_features, gate.in_features, True)):
        y = ops.try_linear(x, gate.weight, up.weight)
        if y is not None:
            return y
    return ops.silu_mul(gate(x), up(x))


__all__ = ["plain_linear", "replaceable", "pays", "streams", "project", "gated"]

"""Which linear layers the weight-streaming kernels may stand in for (no GPU needed: the
rule refuses before any launch)."""
import pytest
import torch
import torch.nn as nn
import torch.nn.modules.module as every
import torch.nn.utils.parametrize as parametrize

from fast_v2_amd import ops
from fast_v2_amd.utils import linear_layers as ll


class _Adapted(nn.Linear):
    pass


def test_only_plain_layers():
    lin = nn.Linear(64, 8)
    assert ll.plain_linear(lin)
    h = lin.register_forward_hook(lambda m, a, o: o + 1)
    assert not ll.plain_linear(lin)
    h.remove()
    assert ll.plain_linear(lin)
    lin.forward = lambda x: x
    assert not ll.plain_linear(lin)
    assert not ll.plain_linear(_Adapted(64, 8))
    par = nn.Linear(64, 8)
    parametrize.register_parametrization(par, "weight", nn.Identity())
    assert not ll.plain_linear(par)


def test_project_runs_the_module_on_cpu():
    lin = nn.Linear(64, 8).to(torch.bfloat16)
    x = torch.randn(3, 64).to(torch.bfloat16)
    assert not ll.streams(x, lin) and not ops.linear_fits(x, lin.weight)
    assert torch.equal(ll.project(lin, x), lin(x))


@pytest.mark.parametrize("register", [
    lambda f: every.register_module_forward_hook(lambda m, a, o: f()),
    lambda f: every.register_module_forward_pre_hook(lambda m, a: f()),
    lambda f: every.register_module_full_backward_hook(lambda m, gi, go: f()),
    lambda f: every.register_module_full_backward_pre_hook(lambda m, go: f())])
def test_hooks_on_every_module_are_run(register):
    lin = nn.Linear(64, 8)
    h = register(lambda: None)
    try:
        assert not ll.plain_linear(lin)
    finally:
        h.remove()
    assert ll.plain_linear(lin)


@pytest.mark.parametrize("n,k,gated,most", [
    (18944, 3584, True, 128), (8960, 1536, True, 128), (28672, 8192, True, 32), (3584, 18944, False, 128),
    (1536, 8960, False, 128), (2048, 2048, False, 64), (896, 896, False, 0), (8192, 8192, False, 0),
    (8192, 28672, False, 128), (11008, 4096, False, 16), (16384, 4096, False, 0), (32000, 4096, False, 48),
    (151936, 1536, False, 128), (152064, 3584, False, 128), (128256, 4096, False, 0), (51200, 2048, False, 0)])
def test_layers_that_pay(n, k, gated, most):
    """The largest row count at which the kernel stands in for a layer."""
    assert [m for m in range(1, 129) if ll.pays(m, n, k, gated)] == list(range(1, most + 1))

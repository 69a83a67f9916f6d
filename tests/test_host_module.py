"""The calls without their native host side (no GPU needed: the choice is made before any
tensor is looked at)."""
import logging

import pytest
import torch

from fast_v2_amd import _ffi, ops


@pytest.mark.parametrize("how", ["missing", "not a module", "another torch"])
def test_the_python_form_stands_in(monkeypatch, tmp_path, caplog, how):
    if how == "another torch":
        monkeypatch.setattr(torch, "__version__", "0.0.0")
    else:
        path = tmp_path / "fdllm_host.so"
        if how == "not a module":
            path.write_bytes(b"no shared library")
        monkeypatch.setattr(_ffi, "HOST_PATH", path)
    host = ops._Host()
    with caplog.at_level(logging.ERROR):
        assert host.gather(None, None, None, 0.0, 0, True) is None
        assert host.attn(*[None] * 13) is None
    assert len([r for r in caplog.records if "native host side" in r.message]) == 1


def test_without_the_kernels_library_calls_still_fail(monkeypatch, tmp_path):
    monkeypatch.setattr(_ffi, "_lib", None)
    monkeypatch.setattr(_ffi, "LIB_PATH", tmp_path / "libfdllm_hip.so")
    with pytest.raises(RuntimeError, match="not built"):
        ops._Host().attn


def test_a_cpu_layer_is_not_taken():
    x, w = torch.zeros(2, 64).bfloat16(), torch.zeros(8, 64).bfloat16()
    assert ops.try_linear(x, w) is None

"""The per-stream workspaces of the calls (ops._Workspace) without a GPU."""
import threading

import torch

from fast_v2_amd import _ffi, ops


def test_a_buffer_that_a_thread_was_given_is_kept(monkeypatch):
    """Two threads that both grow a stream's workspace: whatever either was given stays
    allocated (in use or retired), as its kernels may still be launched on it."""
    monkeypatch.setattr(_ffi, "stream_ptr", lambda device: 7)
    ws, both, zeros = ops._Workspace(), threading.Barrier(2), torch.zeros

    def slow_zeros(*a, **kw):
        try:  # the other thread reaches its own allocation here if it can
            both.wait(timeout=0.5)
        except threading.BrokenBarrierError:
            pass
        return zeros(*a, **kw)

    monkeypatch.setattr(torch, "zeros", slow_zeros)
    got = [None, None]

    def run(i):
        got[i] = ws.get((2 + i) << 20, torch.device("cpu", 0))

    threads = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    kept = [*ws._bufs.values(), *ws._retired]
    for i, t in enumerate(got):
        assert t.numel() >= (2 + i) << 20 and any(t is k for k in kept)

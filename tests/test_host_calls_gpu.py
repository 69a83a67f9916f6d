"""The native host side of the calls (csrc/host_calls.cpp) against the Python statement of
the same calls: equal results in the plain forms, and the Python function's own conversions
and refusals everywhere else."""
import contextlib
import threading

import pytest
import torch

from fast_v2_amd import _ffi, ops

pytestmark = pytest.mark.gpu


class _Recorded:
    """The native module's functions; notes which calls they left to Python."""

    def __init__(self, host):
        self.host, self.native, self.python = host, set(), set()

    def __getattr__(self, name):
        fn = getattr(self.host, name)

        def call(*a):
            try:
                out = fn(*a)
            except Exception:  # refused by the C ABI: the native call got that far
                self.native.add(name)
                raise
            (self.python if out is None else self.native).add(name)
            return out
        return call


class _Off:
    """Every call "not in the plain form"."""

    def __getattr__(self, name):
        return lambda *a: None


@contextlib.contextmanager
def _python():
    saved = ops._HOST
    ops._HOST = _Off()
    try:
        yield
    finally:
        ops._HOST = saved


@contextlib.contextmanager
def _native(python):
    """Only the calls named in ``python`` may be left to the Python form."""
    saved = ops._HOST
    ops._HOST = _Recorded(saved)
    try:
        yield
        assert ops._HOST.python == set(python), (ops._HOST.native, ops._HOST.python)
        assert not ops._HOST.native & set(python)
    finally:
        ops._HOST = saved


def _both(make, python=()):
    """The call's outputs and its tensors afterwards, natively and in Python."""
    res = []
    for off in (False, True):
        fn, state = make()
        with _python() if off else _native(python):
            try:
                out = fn()
            except Exception as exc:  # noqa: BLE001 - compared below
                out = (type(exc), str(exc))
        res.append((out, state))
    return res


def _same(a, b):
    if isinstance(a, torch.Tensor):
        assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b)
    elif isinstance(a, (tuple, list)):
        assert len(a) == len(b)
        for x, y in zip(a, b):
            _same(x, y)
    else:
        assert a == b


def _rnd(seed, *shape, dtype=torch.bfloat16):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, generator=g, device="cuda").to(dtype)


def _attn(form):
    def make():
        dt = torch.float32 if form == "fp32" else torch.bfloat16
        q, k, v = _rnd(1, 2, 8, 14, 128, dtype=dt), _rnd(2, 2, 96, 2, 128, dtype=dt), _rnd(3, 2, 96, 2, 128, dtype=dt)
        lens = torch.tensor([96, 40], dtype=torch.int32, device="cuda")
        kw = {}
        if form == "bhsd":
            q = q.transpose(1, 2).contiguous().transpose(1, 2)
        elif form == "q_strided":
            q = _rnd(1, 2, 8, 14, 256)[..., ::2]
        elif form == "int64_lens":
            lens = lens.long()
        elif form == "paged":
            k, v = k.view(6, 32, 2, 128), v.view(6, 32, 2, 128)
            kw = dict(page_table=torch.tensor([[5, 0, 3], [1, 2, 4]], dtype=torch.int32, device="cuda"), page_size=32)
        elif form == "write":
            kw = dict(k_new=_rnd(4, 2, 8, 2, 128), v_new=_rnd(5, 2, 8, 2, 128), mask_mode=_ffi.MASK_BLOCK_CAUSAL)
        elif form == "write_strides":
            kw = dict(k_new=_rnd(4, 2, 8, 2, 256)[..., :128], v_new=_rnd(5, 2, 8, 2, 128))
        elif form == "q_start":
            kw = dict(q_start=torch.tensor([10, 0], dtype=torch.int32, device="cuda"), mask_mode=_ffi.MASK_CAUSAL)
        elif form == "scale":
            kw = dict(softmax_scale=0.3)
        elif form == "heads":
            q = q[:, :, :13]
        elif form == "types":
            k = k.half()
        elif form == "cpu_lens":
            lens = lens.cpu()
        elif form == "mask":
            kw = dict(mask_mode=9)
        elif form == "grad":
            q = q.requires_grad_()
        elif form == "empty":
            q, k, v, lens = q[:0], k[:0], v[:0], lens[:0]
        return (lambda: ops.block_attn(q, k, v, lens, **kw)), (k, v)
    return make


@pytest.mark.parametrize("form", ["plain", "fp32", "bhsd", "q_strided", "int64_lens", "paged", "write", "write_strides",
                                  "q_start", "scale", "heads", "types", "cpu_lens", "mask", "grad", "empty"])
def test_attention(gpu, form):
    print(f"case attention {form}", flush=True)
    left = form in ("q_strided", "int64_lens", "write_strides", "heads", "types", "cpu_lens")
    a, b = _both(_attn(form), ("attn",) if left else ())
    _same(a, b)


@pytest.mark.parametrize("form", ["plain", "int32", "no_weight", "plain_mode", "columns", "weight_size", "strided", "empty"])
def test_gather_add_scatter(gpu, form):
    print(f"case rows {form}", flush=True)

    def make():
        h, w = _rnd(1, 2, 50, 512), _rnd(2, 512)
        idx = torch.stack([torch.randperm(50, device="cuda", generator=torch.Generator("cuda").manual_seed(3))[:9]] * 2)
        mode = _ffi.NORM_WEIGHT_AFTER_CAST
        if form == "int32":
            idx = idx.int()
        elif form == "no_weight":
            w = None
        elif form == "plain_mode":
            w, mode = None, _ffi.NORM_PLAIN
        elif form == "columns":
            idx = idx.t().contiguous().t()
        elif form == "weight_size":
            w = _rnd(2, 256)
        elif form == "strided":
            h = _rnd(1, 2, 50, 1024)[..., ::2]
        elif form == "empty":
            idx = idx[:, :0]
        cache, cur = torch.zeros(2, 50, 512, device="cuda").bfloat16(), torch.ones(2, 50, 512, device="cuda").bfloat16()

        def fn():
            normed, got = ops.gather_rmsnorm(h, idx, w, 1e-6, mode)
            s, n = ops.add_rmsnorm(got, normed, w, 1e-6, mode)
            assert ops.scatter_rows(got, idx, cache, cur) is cur
            ops.scatter_rows(s, idx, cache)
            return normed, got, s, n
        return fn, (cache, cur)
    left = {"int32": ("gather", "scatter"), "columns": ("gather", "scatter"), "no_weight": ("gather",),
            "weight_size": ("gather",), "strided": ("gather",)}
    _same(*_both(make, left.get(form, ())))


@pytest.mark.parametrize("form", ["plain", "offset", "no_block", "strided_x", "cos2d", "batch_cos", "no_bias", "types", "shape"])
def test_projections(gpu, form):
    print(f"case projections {form}", flush=True)

    def make():
        x, w = _rnd(1, 2, 8, 256), [_rnd(2 + i, n, 256) for i, n in enumerate((512, 128, 128))]
        b = [None if form == "no_bias" else _rnd(7 + i, t.shape[0]) for i, t in enumerate(w)]
        cs = _rnd(9, 2 if form == "batch_cos" else 1, 8, 128)
        if form == "cos2d":
            cs = cs[0]
        kc, vc, kb, vb = (torch.zeros(2, n, 1, 128, device="cuda").bfloat16() for n in (64, 64, 32, 32))
        kw = dict(write_start=torch.tensor([3, 60], dtype=torch.int32, device="cuda"), k_block=kb, v_block=vb,
                  block_offset=8)
        if form == "offset":
            kw.update(write_offset=5)
        elif form == "no_block":
            kw = dict(write_offset=7)
        elif form == "strided_x":
            x = _rnd(1, 2, 8, 512)[..., 256:]
        elif form == "types":
            w[1] = w[1].half()
        elif form == "shape":
            kc = kc[:, :, :, :64]
        return (lambda: ops.qkv_rope_kv_write(x, w[0], b[0], w[1], b[1], w[2], b[2], cs, cs, kc, vc, **kw)), (kc, vc, kb, vb)
    _same(*_both(make, ("qkv",) if form in ("cos2d", "types", "shape") else ()))


@pytest.mark.parametrize("form", ["plain", "stop", "no_finished", "bytes", "strided", "int32_tokens"])
def test_unmask(gpu, form):
    print(f"case unmask {form}", flush=True)

    def make():
        lg = _rnd(1, 3, 8, 4096) * 6
        tok = torch.full((3, 8), 4095, dtype=torch.int64, device="cuda")
        fin = None if form == "no_finished" else torch.zeros(3, dtype=torch.uint8 if form == "bytes" else torch.bool,
                                                             device="cuda")
        if form == "strided":
            lg = _rnd(1, 3, 8, 8192)[..., ::2]
        elif form == "int32_tokens":
            tok = tok.int()

        def fn():
            sc = ops.unmask_step(lg, tok, 4095, 0.9, finished=fin, stop_token=5 if form == "stop" else None)
            return sc.row_tok, sc.row_conf, sc.counts
        return fn, (tok, fin)
    _same(*_both(make))


def test_linear_strided_and_grad(gpu):
    w = _rnd(1, 64, 128)
    for x in (_rnd(2, 4, 8, 128), _rnd(2, 4, 16, 128)[:, 8:], _rnd(2, 8, 256)[:, 128:]):
        _same(*_both(lambda: ((lambda: ops.linear(x, w)), ()), () if x.is_contiguous() else ("linear",)))
    p = torch.nn.Parameter(w)
    with torch.no_grad():
        assert torch.equal(ops.linear(_rnd(2, 8, 128), p), ops.linear(_rnd(2, 8, 128), w))
    assert not ops.linear_fits(_rnd(2, 8, 128), p)
    assert ops.try_linear(_rnd(2, 8, 128), p) is None


def test_transforms_take_the_python_path(gpu):
    """Wrapped tensors never reach the native calls."""
    x = _rnd(1, 3, 4, 8, 14, 128)
    k = _rnd(2, 4, 32, 2, 128)
    lens = torch.full((4,), 32, dtype=torch.int32, device="cuda")
    seen = []
    host = ops._HOST

    def fn(q):
        seen.append(host.attn(q, k, k, lens, None, 0, 32, None, None, 0, None, None, 0))
        return q
    torch.vmap(fn)(x)
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode(allow_non_fake_inputs=True):
        seen.append(host.attn(x[0], k, k, lens, None, 0, 32, None, None, 0, None, None, 0))
    assert seen == [None, None]


def test_streams_and_threads(gpu):
    """Native calls whose workspaces grow on two threads, each on a stream of its own and
    then both on one stream: every result is the one of a call made alone."""
    sizes = [(1, 200), (2, 900), (3, 2000), (4, 4000)]
    data = [(_rnd(1, b, 8, 14, 128), _rnd(2, b, n, 2, 128), _rnd(3, b, n, 2, 128),
             torch.full((b,), n, dtype=torch.int32, device="cuda")) for b, n in sizes]
    want = [ops.block_attn(*a) for a in data]
    torch.cuda.synchronize()
    for streams in ([torch.cuda.Stream(), torch.cuda.Stream()], [torch.cuda.Stream()] * 2):
        print(f"case threads, {len(set(streams))} streams", flush=True)
        bad, gate = [-1, -1], threading.Barrier(2)

        def run(i):
            with torch.cuda.stream(streams[i]):
                gate.wait()
                outs = [(j, ops.block_attn(*data[j])) for _ in range(20) for j in range(4)]
                streams[i].synchronize()
                bad[i] = sum(not torch.equal(o, want[j]) for j, o in outs)

        threads = [threading.Thread(target=run, args=(i,)) for i in range(2)]
        [t.start() for t in threads]
        [t.join() for t in threads]
        assert bad == [0, 0]


def test_inference_mode_and_the_callers_scratch(gpu):
    with torch.inference_mode():
        _same(*_both(_attn("plain")))
        lg = _rnd(1, 3, 8, 4096) * 6
        kept = ops.UnmaskScratch(3, 8, lg.device)

        def make():
            tok = torch.full((3, 8), 4095, dtype=torch.int64, device="cuda")

            def fn():
                sc = ops.unmask_step(lg, tok, 4095, 0.9, scratch=kept)
                assert sc is kept
                return sc.row_tok.clone(), sc.row_conf.clone(), sc.counts.clone()
            return fn, tok
        _same(*_both(make))

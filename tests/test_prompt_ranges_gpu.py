"""Prompts of few row blocks: the ring prefill kernel with and without key ranges against
float64 and against the general kernel (decode_kernel=False) over the forms it takes."""
import ctypes
import itertools
import threading

import pytest
import torch

from fast_v2_amd import _ffi, ops

pytestmark = pytest.mark.gpu
D = 128


def _case(b, sq, heads, cap, layout, dtype, seed):
    hq, hkv = heads
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rnd(*shape):
        return torch.randn(*shape, generator=g, device="cuda").to(dtype)
    q = rnd(b, sq, hq, D)
    if layout == "contiguous":
        k, v, table = rnd(b, cap, hkv, D), rnd(b, cap, hkv, D), None
    else:
        pages = (cap + 31) // 32
        k, v = rnd(b * pages, 32, hkv, D), rnd(b * pages, 32, hkv, D)
        if layout == "paged_hm":
            k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (k, v))
        table = torch.randperm(b * pages, generator=g, device="cuda").to(torch.int32).view(b, pages)
    return q, k, v, table, rnd(b, sq, hkv, D), rnd(b, sq, hkv, D)


def _dense(t, table, b):
    return t[b] if table is None else t[table[b].long()].flatten(0, 1)


def _ref(q, k, v, table, lens, starts, mode, block=32):
    out = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
    b, sq, hq, _ = q.shape
    for i in range(b):
        kk, vv = (_dense(t, table, i).double() for t in (k, v))
        pos = starts[i] + torch.arange(sq, device="cuda")
        lim = torch.full_like(pos, lens[i])
        if mode == _ffi.MASK_CAUSAL:
            lim = torch.minimum(lim, pos + 1)
        elif mode == _ffi.MASK_BLOCK_CAUSAL:
            lim = torch.minimum(lim, torch.where(pos >= 0, (pos // block + 1) * block, torch.zeros_like(pos)))
        hide = torch.arange(kk.shape[0], device="cuda")[None] >= lim[:, None]
        for h in range(hq):
            g = h // (hq // kk.shape[1])
            s = (q[i, :, h].double() @ kk[:, g].t().contiguous() * D ** -0.5).masked_fill(hide, float("-inf"))
            p = torch.nan_to_num(torch.softmax(s, dim=-1))  # a row that sees no key is zero
            out[i, :, h] = p @ vv[:, g].contiguous()
    return out


# rows per KV head: 259 (two row blocks), 1099, 2037 / 2051 (around the whole-range form's
# start), 3500, 7218 that fill the cache (key ranges); key ranges where the capacity is long; visible lengths at, below and far
# below the capacity (one sequence empty of keys to range over)
SHAPES = [(1, 37, (28, 4), 37), (2, 157, (28, 4), 157), (1, 291, (28, 4), 1500), (1, 293, (28, 4), 293),
          (1, 500, (28, 4), 1203), (1, 300, (12, 2), 2048), (1, 1203, (12, 2), 1203), (3, 70, (12, 2), 700), (1, 129, (2, 1), 4096)]


@pytest.mark.parametrize("b,sq,heads,cap", SHAPES)
@pytest.mark.parametrize("mode", [_ffi.MASK_SEQLEN, _ffi.MASK_CAUSAL, _ffi.MASK_BLOCK_CAUSAL])
@pytest.mark.parametrize("layout", ["contiguous", "paged", "paged_hm"])
def test_prompt(gpu, b, sq, heads, cap, mode, layout):
    dtype = torch.float16 if layout == "paged" else torch.bfloat16
    q, k, v, table, kn, vn = _case(b, sq, heads, cap, layout, dtype, cap + sq + mode)
    kw = dict(mask_mode=mode, page_table=table, page_size=32 if table is not None else 0)
    for short, write in itertools.product((False, True), (False, True)):
        lens = [max(sq, cap - 65 * i - (cap // 2 if short else 0)) for i in range(b)]
        seqlens = torch.tensor(lens, dtype=torch.int32, device="cuda")
        print(f"case prompt {b}x{sq} {heads} cap {cap} mode {mode} {layout} lens {lens} write {write}", flush=True)
        ka, va, kb, vb = k.clone(), v.clone(), k.clone(), v.clone()
        new = dict(k_new=kn, v_new=vn) if write else {}
        got = ops.block_attn(q, ka, va, seqlens, **kw, **new)
        gen = ops.block_attn(q, kb, vb, seqlens, decode_kernel=False, **kw, **new)
        assert torch.equal(ka, kb) and torch.equal(va, vb)
        want = _ref(q, ka, va, table, lens, [n - sq for n in lens], mode)
        # probabilities and results are rounded to the type once each
        torch.testing.assert_close(got.double(), want, atol=1e-2, rtol=1e-2)
        torch.testing.assert_close(gen.double(), want, atol=1e-2, rtol=1e-2)


@pytest.mark.parametrize("starts", [[0, 400], [-20, 100]])
def test_prompt_query_starts_and_empty_rows(gpu, starts):
    q, k, v, table, kn, vn = _case(2, 150, (28, 4), 640, "paged", torch.bfloat16, 5)
    qs = torch.tensor(starts, dtype=torch.int32, device="cuda")
    for lens in ([640, 555], [0, 31]):
        seqlens = torch.tensor(lens, dtype=torch.int32, device="cuda")
        for mode in (_ffi.MASK_SEQLEN, _ffi.MASK_CAUSAL, _ffi.MASK_BLOCK_CAUSAL):
            print(f"case starts {starts} lens {lens} mode {mode}", flush=True)
            got = ops.block_attn(q, k, v, seqlens, mask_mode=mode, q_start=qs, page_table=table, page_size=32)
            torch.testing.assert_close(got.double(), _ref(q, k, v, table, lens, starts, mode), atol=1e-2, rtol=1e-2)


@pytest.mark.parametrize("sq,heads", [(500, (28, 4)), (1203, (12, 2)), (280, (28, 4))])
def test_prompt_graph_replay(gpu, sq, heads):
    """A prompt whole (3500 rows in a cache with room for more) and its ranges with their merge
    (7218 rows that fill the cache; 1960 rows) under graph replay, eager calls in between."""
    q, k, v, table, kn, vn = _case(1, sq, heads, 1203, "contiguous", torch.bfloat16, 9)
    seqlens = torch.tensor([1203], dtype=torch.int32, device="cuda")
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        ops.block_attn(q, k, v, seqlens, mask_mode=_ffi.MASK_CAUSAL)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            out = ops.block_attn(q, k, v, seqlens, mask_mode=_ffi.MASK_CAUSAL)
        for n in (1203, 900, 500):
            seqlens.fill_(n)
            graph.replay()
            assert torch.equal(out, ops.block_attn(q, k, v, seqlens, mask_mode=_ffi.MASK_CAUSAL))
            s.synchronize()


def _c_call(q, k, v, seqlens, mode, ws_bytes):
    out = torch.empty_like(q)
    d = ops._attn_desc(q, k, v, seqlens, out, D ** -0.5, mode, 32, None, None, 0, 0)
    need = ctypes.c_size_t(0)
    _ffi.check(_ffi.lib().fdllm_kv_attn_workspace_size(ctypes.byref(d), ctypes.byref(need)), "size")
    assert need.value > ws_bytes
    ws = torch.zeros(max(ws_bytes, 16), dtype=torch.uint8, device="cuda")
    rc = _ffi.lib().fdllm_kv_attn_fwd(ctypes.byref(d), ws.data_ptr() if ws_bytes else None, ws_bytes,
                                      _ffi.stream_ptr(q.device))
    torch.cuda.synchronize()
    return rc, out


def test_workspace_of_a_plan_without_ranges(gpu):
    """A prompt without a workspace runs whole; a decode call with the slots it cannot do
    without runs on those; less is refused."""
    q, k, v, _, _, _ = _case(1, 1203, (12, 2), 1203, "contiguous", torch.bfloat16, 3)
    lens = torch.tensor([1203], dtype=torch.int32, device="cuda")
    rc, out = _c_call(q, k, v, lens, _ffi.MASK_CAUSAL, 0)
    assert rc == _ffi.FDLLM_OK
    torch.testing.assert_close(out.double(), _ref(q, k, v, None, [1203], [0], _ffi.MASK_CAUSAL), atol=1e-2, rtol=1e-2)

    q, k, v, _, _, _ = _case(33, 2, (8, 4), 5152, "contiguous", torch.bfloat16, 4)  # two splits each: 66 slots, or 128
    lens = torch.tensor([40 * i + 5 for i in range(33)], dtype=torch.int32, device="cuda")
    bytes_ = 64 * 1024 + 66 * 4 * 64 * 8 + 66 * 4 * 64 * 128 * 4
    rc, out = _c_call(q, k, v, lens, _ffi.MASK_SEQLEN, bytes_)
    assert rc == _ffi.FDLLM_OK
    want = _ref(q, k, v, None, lens.tolist(), (lens - 2).tolist(), _ffi.MASK_SEQLEN)
    torch.testing.assert_close(out.double(), want, atol=1e-2, rtol=1e-2)
    assert _c_call(q, k, v, lens, _ffi.MASK_SEQLEN, bytes_ - 256)[0] == _ffi.FDLLM_ERR_WORKSPACE


def test_calls_of_two_threads_on_one_stream(gpu):
    """Calls of two kernels (a prompt with key ranges, a whole-block decode) and of one from
    two threads on one stream, which share that stream's workspace."""
    def call(b, sq, n, seed, mode):
        q, k, v, _, _, _ = _case(b, sq, (28, 4), n, "contiguous", torch.bfloat16, seed)
        return q, k, v, torch.full((b,), n, dtype=torch.int32, device="cuda"), mode
    calls = [call(1, 280, 2048, 1, _ffi.MASK_CAUSAL), call(4, 32, 1500, 2, _ffi.MASK_SEQLEN),
             call(4, 8, 1500, 3, _ffi.MASK_SEQLEN)]
    run = [lambda c=c: ops.block_attn(*c[:4], mask_mode=c[4]) for c in calls]
    want = [f() for f in run]
    torch.cuda.synchronize()
    s, gate, bad = torch.cuda.Stream(), threading.Barrier(2), [-1, -1]

    def thread(i):
        with torch.cuda.stream(s):
            gate.wait()
            got = [(j, run[j]()) for n in range(60) for j in ((0, 1, 2), (1, 2, 0))[i]]
            s.synchronize()
            bad[i] = sum(not torch.equal(o, want[j]) for j, o in got)

    threads = [threading.Thread(target=thread, args=(i,)) for i in range(2)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert bad == [0, 0]


def test_prompt_on_the_librarys_scratch(gpu):
    """fdllm_kv_attn_fwd_noalloc runs a prompt of 2048 rows and more as fdllm_kv_attn_fwd
    does without a workspace; a workspace size without a workspace counts as none."""
    q, k, v, _, _, _ = _case(1, 800, (12, 2), 832, "contiguous", torch.bfloat16, 12)
    lens = torch.tensor([832], dtype=torch.int32, device="cuda")
    outs = []
    for form in ("noalloc", "none", "null"):
        out = torch.empty_like(q)
        d = ops._attn_desc(q, k, v, lens, out, D ** -0.5, _ffi.MASK_CAUSAL, 32, None, None, 0, 0)
        st = _ffi.stream_ptr(q.device)
        rc = _ffi.lib().fdllm_kv_attn_fwd_noalloc(ctypes.byref(d), st) if form == "noalloc" else \
            _ffi.lib().fdllm_kv_attn_fwd(ctypes.byref(d), None, 0 if form == "none" else 1 << 30, st)
        _ffi.check(rc, form)
        outs.append(out)
    want = _ref(q, k, v, None, [832], [32], _ffi.MASK_CAUSAL)
    torch.testing.assert_close(outs[0].double(), want, atol=1e-2, rtol=1e-2)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])

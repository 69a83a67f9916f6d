"""ops.linear / ops.gated_linear (fdllm_linear) and the few-row form of
ops.qkv_rope_kv_write against torch in float64."""
import ctypes

import pytest
import torch
import torch.nn.modules.module as every
from torch.autograd import forward_ad

from torch.overrides import TorchFunctionMode
from torch.utils.flop_counter import FlopCounterMode

from fast_v2_amd import _ffi, ops
from fast_v2_amd.utils import linear_layers as ll

pytestmark = pytest.mark.gpu


def _ints(gen, *shape, dtype):
    """Small whole numbers: every fp32 sum of up to 2^20 products of them is exact, in any
    order, so results compare bit for bit."""
    return torch.randint(-3, 4, shape, generator=gen, device="cuda").to(dtype)


# rows at the edges of the 16-row MFMA tile counts; columns and K where a layer is one
# tile, a partial last tile, tiles cut evenly (<= 128 tiles) and ranges that cross tiles;
# wide tiles (from 16384 columns) with K steps beyond the ring's slots, so that slots are
# refilled: in two ranges (103, 105 tiles), in one (129)
@pytest.mark.parametrize("m", [1, 16, 17, 33, 64, 65, 128])
@pytest.mark.parametrize("n,k", [(8, 64), (72, 576), (200, 4096), (8320, 1088), (16648, 192), (16392, 1088), (16648, 1088),
                                 (20488, 1024)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear_exact(gpu, m, n, k, dtype):
    print(f"case linear {m}x{n}x{k} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m * 7 + n)
    x, w, b = _ints(g, m, k, dtype=dtype), _ints(g, n, k, dtype=dtype), _ints(g, n, dtype=dtype)
    want = x.double() @ w.double().t().contiguous()
    for bias in (None, b):
        ref = want if bias is None else want + b.double()
        for _ in range(2):  # the arrival counters are back at zero after a call
            got = ops.linear(x, w, bias)
            assert torch.equal(got, ref.float().to(dtype))


def test_linear_strided_rows(gpu):
    g = torch.Generator(device="cuda").manual_seed(3)
    full = _ints(g, 40, 2, 256, dtype=torch.bfloat16)
    w = _ints(g, 128, 256, dtype=torch.bfloat16)
    for x in (full[:, 1], full[:, 1, :][::2], full.view(40, 512)[:, 8:264], full.view(40, 512)[:, 1:257]):
        assert torch.equal(ops.linear(x, w), (x.double() @ w.double().t().contiguous()).float().to(x.dtype))


@pytest.mark.parametrize("m", [1, 31, 33, 64, 65, 128])
@pytest.mark.parametrize("n,k", [(8, 64), (104, 1536), (4360, 1088), (8200, 1088), (10248, 512), (18952, 1088)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gated_linear(gpu, m, n, k, dtype):
    print(f"case gated {m}x{n}x{k} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + n)
    x, wg, wu = _ints(g, m, k, dtype=dtype), _ints(g, n, k, dtype=dtype), _ints(g, n, k, dtype=dtype)
    wg = wg * 0.015625  # exact, and gates of a few units instead of saturated ones
    gate, up = ((x.double() @ w.double().t().contiguous()).float().to(dtype) for w in (wg, wu))
    want = ops.silu_mul(gate, up)
    assert torch.equal(ops.gated_linear(x, wg, wu), want)


def test_linear_graph_replay(gpu):
    """Partial sums and counters under graph replay, with other calls in between."""
    g = torch.Generator(device="cuda").manual_seed(5)
    x, w = _ints(g, 24, 4096, dtype=torch.bfloat16), _ints(g, 200, 4096, dtype=torch.bfloat16)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        ops.linear(x, w)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            out = ops.linear(x, w)
        for i in range(4):
            x.copy_(_ints(g, 24, 4096, dtype=torch.bfloat16))
            graph.replay()
            assert torch.equal(out, ops.linear(x, w))
            assert torch.equal(out, (x.double() @ w.double().t().contiguous()).float().to(x.dtype))
            s.synchronize()


@pytest.mark.parametrize("bad", ["rows", "k", "n", "dtype", "grad"])
def test_linear_refuses(gpu, bad):
    x = torch.zeros(129 if bad == "rows" else 8, 96 if bad == "k" else 128, device="cuda", dtype=torch.bfloat16)
    w = torch.zeros(12 if bad == "n" else 16, x.shape[1], device="cuda",
                    dtype=torch.float16 if bad == "dtype" else torch.bfloat16, requires_grad=bad == "grad")
    with pytest.raises(RuntimeError):
        ops.linear(x, w)


@pytest.mark.parametrize("hidden", [1536, 1024, 512])  # the last two on the other kernel from 65 rows
@pytest.mark.parametrize("rows", [(1, 1), (4, 8), (8, 8), (5, 13), (4, 32)])
def test_qkv_linear_is_the_fused_kernels_projection(gpu, rows, hidden):
    """Plain projections, and the ones that qkv_rope_kv_write rotates (v rows as they are)."""
    g = torch.Generator(device="cuda").manual_seed(11)
    b, s = rows
    dt = torch.bfloat16
    x = torch.randn(b, s, hidden, generator=g, device="cuda").to(dt)
    w = [(torch.randn(n, hidden, generator=g, device="cuda") * 0.02).to(dt) for n in (768, 256, 256)]
    bias = [torch.randn(t.shape[0], generator=g, device="cuda").to(dt) for t in w]
    args = [t for pair in zip(w, bias) for t in pair]
    q, k, v = ops.qkv_linear(x, *args)
    for got, wt, bt in zip((q, k, v), w, bias):
        want = x.double() @ wt.double().t().contiguous() + bt.double()
        # one rounding to bf16 (half of 2^-7 of the value) and fp32 sums of at most 1536 products
        torch.testing.assert_close(got.reshape(b, s, -1).double(), want, rtol=2.0 ** -8 + 2e-5, atol=2e-4)
    cos, sin = (torch.randn(1, s, 128, generator=g, device="cuda").to(dt) for _ in range(2))
    q_rot, (k_rot, v_out) = ops.qkv_rope_kv_write(x, *args, cos, sin, kv_out=True)
    q2, (k2, v2) = ops.rope_kv_write(q, k, v, cos, sin, kv_out=True)
    assert torch.equal(q_rot, q2) and torch.equal(k_rot, k2) and torch.equal(v_out, v2) and torch.equal(v, v2)


def test_first_calls_of_a_stream_under_capture(gpu):
    """A capture may be the first use of a stream: the workspace is cleared at once, so eager
    calls on that stream before the first replay, the replays and a second graph captured
    there all find their counters at zero."""
    g = torch.Generator(device="cuda").manual_seed(6)
    x, w = _ints(g, 24, 4096, dtype=torch.bfloat16), _ints(g, 200, 4096, dtype=torch.bfloat16)
    big = _ints(g, 4096, 4096, dtype=torch.bfloat16)
    q, k, v = (torch.randn(2, n, h, 128, generator=g, device="cuda").bfloat16() for n, h in ((8, 28), (900, 4), (900, 4)))
    lens = torch.tensor([900, 500], dtype=torch.int32, device="cuda")
    xp = torch.randn(2, 8, 512, generator=g, device="cuda").bfloat16()
    wp = [(torch.randn(n, 512, generator=g, device="cuda") * 0.05).bfloat16() for n in (512, 128, 128)]
    cs = torch.randn(1, 8, 128, generator=g, device="cuda").bfloat16()

    def calls():
        return [ops.block_attn(q, k, v, lens), ops.linear(x, w), ops.linear(x, big),
                ops.qkv_rope_kv_write(xp, wp[0], None, wp[1], None, wp[2], None, cs, cs)]

    want = calls()
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    while (gpu.index, s.cuda_stream) in ops._WORKSPACE._bufs:  # streams come out of a small pool
        s = torch.cuda.Stream()
    graphs = [torch.cuda.CUDAGraph() for _ in range(2)]
    outs = []
    for graph in graphs:
        with torch.cuda.graph(graph, stream=s):
            outs.append(calls())
    with torch.cuda.stream(s):
        print("case eager before the first replay", flush=True)
        assert all(torch.equal(a, b) for a, b in zip(calls(), want))
        for i in (1, 0, 1, 0, 0):  # the graph captured second is replayed first
            print(f"case replay of graph {i}", flush=True)
            [o.zero_() for o in outs[i]]
            graphs[i].replay()
            assert all(torch.equal(a, b) for a, b in zip(outs[i], want))
            assert all(torch.equal(a, b) for a, b in zip(calls(), want))
    s.synchronize()


def _layers(dtype=torch.bfloat16):
    g = torch.Generator(device="cuda").manual_seed(21)
    gate, up, down = (torch.nn.Linear(k, n, bias=False, device="cuda", dtype=dtype) for k, n in
                      ((1024, 2048), (1024, 2048), (2048, 1024)))
    with torch.no_grad():
        for m in (gate, up, down):
            m.weight.copy_(_ints(g, *m.weight.shape, dtype=dtype) * 0.0625)
    assert ll.pays(32, 1024, 2048, False)  # else the module runs anyway
    return gate, up, down, _ints(g, 4, 8, 1024, dtype=dtype)


def _mlp(gate, up, down, x):
    with torch.no_grad():
        return ll.project(down, ll.gated(gate, up, x))


def test_a_hook_on_every_module_sees_the_layers(gpu):
    gate, up, down, x = _layers()
    want, seen = _mlp(gate, up, down, x), []
    h = every.register_module_forward_hook(lambda m, a, o: seen.append(m))
    try:
        got = _mlp(gate, up, down, x)
    finally:
        h.remove()
    assert seen == [gate, up, down]
    torch.testing.assert_close(got, want, rtol=2.0 ** -6, atol=2.0 ** -6 * float(want.abs().max()))


@pytest.mark.parametrize("cast", [torch.float16, torch.bfloat16])
def test_autocast_decides_the_type(gpu, cast):
    gate, up, down, x = _layers()
    with torch.autocast("cuda", dtype=cast):
        got = _mlp(gate, up, down, x)
        with torch.no_grad():
            want = down(ops.silu_mul(gate(x), up(x)))
    assert got.dtype == want.dtype == cast
    torch.testing.assert_close(got, want, rtol=2.0 ** -6, atol=2.0 ** -6 * float(want.abs().max()))


class _Calls(TorchFunctionMode):
    def __init__(self):
        self.linear = 0

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.linear += func is torch.nn.functional.linear
        return func(*args, **(kwargs or {}))


def test_modes_see_the_layers(gpu):
    gate, up, down, x = _layers()
    with FlopCounterMode(display=False) as flops:
        _mlp(gate, up, down, x)
    assert flops.get_total_flops() == 2 * 32 * 3 * 1024 * 2048
    with _Calls() as calls:
        _mlp(gate, up, down, x)
    assert calls.linear == 3
    with torch.device("cuda"):  # a default device changes nothing
        assert ll.replaceable(x)


class _Doubled(torch.Tensor):
    """A weight that is not stored as it reads (as quantised weights are): twice ``inner``."""

    @staticmethod
    def __new__(cls, inner):
        t = torch.Tensor._make_wrapper_subclass(cls, inner.shape, strides=inner.stride(), dtype=inner.dtype,
                                                device=inner.device)
        t.inner = inner
        return t

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        if func is torch.ops.aten.detach.default:
            return cls(args[0].inner)
        return func(*[a.inner * 2 if isinstance(a, cls) else a for a in args], **(kwargs or {}))


def test_layers_on_other_tensors_run_as_modules(gpu):
    """Weights of a tensor subclass, forward-mode tangents and vmap: what the module gives."""
    gate, _, down, x = _layers()
    half = down.weight.detach() * 0.5
    ones = torch.ones(4, 8, 2048, device=gpu, dtype=torch.bfloat16)
    want = down(ones).detach()
    down.weight = torch.nn.Parameter(_Doubled(half), requires_grad=False)
    with torch.no_grad():
        torch.testing.assert_close(ll.project(down, ones), want, rtol=2.0 ** -7, atol=2.0 ** -6)
        with forward_ad.dual_level():
            y = ll.project(gate, forward_ad.make_dual(x, torch.ones_like(x)))
            tangent = forward_ad.unpack_dual(y).tangent
            assert ll.project(gate, x).shape == y.shape  # no tangent: nothing to carry
        rows = torch.vmap(lambda r: ll.project(gate, r))(x)
    torch.testing.assert_close(tangent, gate(torch.ones_like(x)).detach(), rtol=2.0 ** -6, atol=2.0 ** -5)
    torch.testing.assert_close(rows, gate(x).detach(), rtol=2.0 ** -6, atol=2.0 ** -5)
    dual = None
    with forward_ad.dual_level(), pytest.raises(RuntimeError):
        dual = ops.linear(forward_ad.make_dual(x, torch.ones_like(x)), gate.weight.detach())
    assert dual is None


@pytest.mark.parametrize("m,n,k,gated", [(1, 200, 4096, False), (65, 200, 4096, False), (128, 4360, 1088, True),
                                         (33, 16392, 1088, False)])
def test_linear_without_a_workspace(gpu, m, n, k, gated):
    """fdllm_linear with no workspace: one K range, the same sums."""
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    dt = torch.bfloat16
    x, w, u = _ints(g, m, k, dtype=dt), _ints(g, n, k, dtype=dt), _ints(g, n, k, dtype=dt)
    w = w * 0.015625 if gated else w
    out = torch.empty(m, n, dtype=dt, device=gpu)
    _ffi.check(_ffi.lib().fdllm_linear(x.data_ptr(), k, w.data_ptr(), u.data_ptr() if gated else None, None,
                                       out.data_ptr(), m, n, k, _ffi.dtype_code(dt), None, 0, _ffi.stream_ptr(gpu)),
               "fdllm_linear")
    assert torch.equal(out, ops.gated_linear(x, w, u) if gated else ops.linear(x, w))


@pytest.mark.parametrize("rows,hidden", [((4, 8), 1536), ((4, 32), 1536), ((4, 32), 1024), ((5, 32), 1536)])
def test_projections_without_a_workspace(gpu, rows, hidden):
    """fdllm_qkv_rope_kv_write takes none: whole numbers, whose sums are exact in any order."""
    g = torch.Generator(device="cuda").manual_seed(hidden)
    (b, s), dt = rows, torch.bfloat16
    x, w = _ints(g, b, s, hidden, dtype=dt), [_ints(g, n, hidden, dtype=dt) for n in (768, 256, 256)]
    cs = torch.randn(1, s, 128, generator=g, device="cuda").to(dt)
    want, (wk, wv) = ops.qkv_rope_kv_write(x, w[0], None, w[1], None, w[2], None, cs, cs, kv_out=True)
    d, dims, keep = ops._qkv_desc(x, w[0], None, w[1], None, w[2], None, 128)
    q, (k, v), kept = ops._rope_dest_desc(d.rope, *dims[:5], dt, gpu, cs, cs, None, None, None, 0, None, None, 0, None,
                                          True)
    _ffi.check(_ffi.lib().fdllm_qkv_rope_kv_write(ctypes.byref(d), _ffi.stream_ptr(gpu)), "fdllm_qkv_rope_kv_write")
    assert torch.equal(q, want) and torch.equal(k, wk) and torch.equal(v, wv)

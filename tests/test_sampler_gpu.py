"""GPU parity of the fused greedy sampling + unmask step (fdllm_unmask_step) with the
torch statement of the reference rule (fast_v2_amd.e2e.sampler.greedy_with_confidence
+ threshold_unmask, i.e. modeling.py:2263-2270 and generation_functions.py:784-807).

Bar: tokens, unmask decisions, the stop rule and the counters exact; the confidence
within one ulp of the logits' type (the softmax sum is accumulated in another order
than torch's). The logits are drawn so that no confidence lies within an ulp of the
threshold and no two probabilities tie after rounding except where planted (an
exact tie between two equal logits, resolved to the first index).
"""
import ctypes
import threading

import pytest
import torch

from fast_v2_amd import _ffi, ops
from fast_v2_amd.e2e import model as em
from fast_v2_amd.e2e import sampler as es

pytestmark = pytest.mark.gpu


def _torch_step(raw, x_sub, mask_id, thr, row_offset, finished, stop):
    L = x_sub.shape[1]
    logits = torch.cat([raw[:, :1], raw[:, :-1]], dim=1)[:, row_offset:row_offset + L]
    tok, conf = es.greedy_with_confidence(logits)
    masked = (x_sub == mask_id) & ~finished[:, None]
    unmask = es.threshold_unmask(tok, conf, masked, thr)
    new = torch.where(unmask, tok, x_sub)
    fin = finished | ((tok == stop) & unmask).any(dim=1) if stop is not None else finished.clone()
    left = ((new == mask_id) & ~finished[:, None] & ~fin[:, None]).sum()
    return tok, conf, new, fin, [int(unmask.sum()), int(left), int((new[:, 0] == mask_id).sum()), int(fin.sum())]


@pytest.mark.parametrize("V,R,L,row_offset", [(152064, 8, 8, 0), (152064, 32, 8, 8), (1000, 32, 8, 24), (4099, 9, 5, 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_unmask_step_matches_torch(gpu, V, R, L, row_offset, dtype):
    g = torch.Generator().manual_seed(V + R + L + row_offset)
    B, mask_id, thr, stop = 6, V - 1, 0.9, 7
    raw = (torch.randn(B, R, V, generator=g) * 2).to(dtype)
    # peaked rows: confident positions (conf well above the threshold)
    for b in range(B):
        for r in range(R):
            if (b + r) % 3 == 0:
                raw[b, r, (b * 31 + r * 17) % (V - 1)] = 30.0
    raw[0, 0, 5] = raw[0, 0, 9] = 40.0   # an exact tie: the first index wins
    raw[2, 1, stop] = 50.0               # row 2 emits the stop token
    x_sub = torch.randint(0, V - 1, (B, L), generator=g)
    x_sub[torch.rand(B, L, generator=g) < 0.7] = mask_id
    x_sub[4] = mask_id
    finished = torch.zeros(B, dtype=torch.bool)
    finished[5] = True
    raw_g, x_g, fin_g = raw.to(gpu), x_sub.to(gpu), finished.to(gpu)
    print(f"case unmask V={V} R={R} L={L} off={row_offset} {dtype}", flush=True)
    tok, conf, new, fin, counts = _torch_step(raw_g, x_g.clone(), mask_id, thr, row_offset, fin_g.clone(), stop)
    sc = ops.unmask_step(raw_g, x_g, mask_id, thr, row_offset=row_offset, shift=1, finished=fin_g, stop_token=stop)
    assert torch.equal(sc.row_tok, tok)
    ulp = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
    torch.testing.assert_close(sc.row_conf, conf.float(), atol=0, rtol=ulp)
    assert torch.equal(x_g, new)
    assert torch.equal(fin_g, fin)
    assert sc.counts.tolist() == counts


def test_fused_sampler_generation_matches_torch_rule(gpu):
    """The same HIP forwards with the fused step and with the torch rule give the same
    generation (2-layer model, batch 4, 96 new tokens)."""
    cfg = em.BlockDiffusionConfig(num_hidden_layers=2)
    model = em.build_model(cfg, gpu)
    x = torch.randint(0, cfg.vocab_size - 1, (4, 64), generator=torch.Generator().manual_seed(6)).to(gpu)
    a, st_a = es.generate(model, x, max_new_tokens=96, impl=es.HipStaticAttention(fused_sampler=True))
    b, st_b = es.generate(model, x, max_new_tokens=96, impl=es.HipStaticAttention(fused_sampler=False))
    print(f"forwards {st_a.forwards} vs {st_b.forwards}")
    assert torch.equal(a, b)
    assert st_a.step_tokens == st_b.step_tokens


@pytest.mark.parametrize("V", [1, 7, 8185, 8192, 8193, 16384, 24570, 32001])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("scale", [0.3, 2.0])
def test_unmask_chunk_edges(gpu, V, dtype, scale):
    """Rows around the 8192-logit chunks, rows that start off a 16-byte boundary (odd
    vocabularies), leading chunks of -inf and, at the small scale, maxima that smaller
    logits tie with after rounding (the chunks that are read again). Expected: softmax in 64
    bits, rounded to the logits' type, first index of the maximum; the fp32 sum moves a
    probability by under 1e-6 of itself, far inside a rounding step at these draws."""
    g = torch.Generator().manual_seed(V + int(10 * scale))
    B, L = 3, 5
    raw = (torch.randn(B, L, V, generator=g) * scale).to(dtype)
    raw[1, 2, :V // 2] = float("-inf")
    raw[2, 1, V - 1] = 1.5 if scale < 1 else 20.0
    p = torch.softmax(raw.double(), dim=-1).to(dtype).float()
    top = p.max(dim=-1, keepdim=True).values
    tok = (p == top).to(torch.uint8).argmax(dim=-1)
    x = torch.full((B, L), V + 1, dtype=torch.int64, device=gpu)
    print(f"case unmask chunks V={V} {dtype} scale={scale}", flush=True)
    sc = ops.unmask_step(raw.to(gpu), x, V + 1, 2.0, row_offset=0, shift=0)
    assert torch.equal(sc.row_tok.cpu(), tok)
    torch.testing.assert_close(sc.row_conf.cpu(), top[..., 0], atol=0, rtol=0)
    best = top[..., 0].argmax(dim=-1)
    assert x.cpu().gather(1, best[:, None])[:, 0].tolist() == tok.gather(1, best[:, None])[:, 0].tolist()
    assert sc.counts.tolist()[:2] == [B, B * (L - 1)]


def test_a_step_keeps_its_partials_to_itself(gpu):
    """A step is two kernels, and another thread's step may be launched between them on the
    same stream: what they hand over lies in the caller's scratch, not in the memory that a
    stream's callers share."""
    s = torch.cuda.Stream()
    raw = torch.randn(2, 4, 40000, device=gpu).bfloat16()
    x = torch.full((2, 4), 39999, dtype=torch.int64, device=gpu)
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        sc = ops.unmask_step(raw, x, 39999, 2.0)
        again = ops.unmask_step(raw, x, 39999, 2.0, scratch=sc)
        other = ops.unmask_step(raw, x, 39999, 2.0)
    s.synchronize()
    assert (gpu.index, s.cuda_stream) not in ops._WORKSPACE._bufs
    assert again is sc and len(sc._parts) == 1 and sc._parts[0].data_ptr() != other._parts[0].data_ptr()


def test_steps_of_two_threads_on_one_stream(gpu):
    g = torch.Generator().manual_seed(8)
    B, L, V, steps = 2, 4, 33000, 300
    raws = [(torch.randn(B, L, V, generator=g) * 3).bfloat16().to(gpu) for _ in range(2)]
    want = [ops.unmask_step(r, torch.full((B, L), V, dtype=torch.int64, device=gpu), V, 2.0).row_tok for r in raws]
    bad, gate = [0, 0], threading.Barrier(2)

    def run(i):
        x = torch.full((B, L), V, dtype=torch.int64, device=gpu)
        sc = ops.UnmaskScratch(B, L, gpu)
        toks = []
        gate.wait()
        for _ in range(steps):
            x.fill_(V)
            toks.append(ops.unmask_step(raws[i], x, V, 2.0, scratch=sc).row_tok.clone())
        bad[i] = sum(not torch.equal(t, want[i]) for t in toks)

    assert not torch.equal(want[0], want[1])
    threads = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert bad == [0, 0]


def _step_without_workspace(raw, x, mask_id, threshold):
    """fdllm_unmask_step, the entry point that takes no workspace."""
    sc = ops.UnmaskScratch(*x.shape, x.device)
    _ffi.check(_ffi.lib().fdllm_unmask_step(
        raw.data_ptr(), raw.stride(0), raw.stride(1), raw.shape[2], 0, 0, x.data_ptr(), x.stride(0), None, mask_id,
        threshold, -1, sc.row_tok.data_ptr(), sc.row_conf.data_ptr(), sc.counts.data_ptr(), *x.shape,
        _ffi.dtype_code(raw.dtype), _ffi.stream_ptr(x.device)), "fdllm_unmask_step")
    return sc


@pytest.mark.parametrize("workspace", [True, False])
@pytest.mark.parametrize("V", [1000, 9001, 24584])
def test_rows_without_a_finite_probability(gpu, V, workspace):
    """Rows of -inf, of NaN and with one NaN or +inf among finite logits: the token lies in
    the vocabulary (0 where nothing is above -inf, as argmax over NaN), the position stays
    masked, and the others of its sequence follow the rule."""
    B, L = 3, 4
    raw = torch.randn(B, L, V, generator=torch.Generator().manual_seed(V)).bfloat16()
    raw[0, 1] = float("-inf")
    raw[0, 2] = float("nan")
    raw[1] = float("nan")
    raw[1, 3] = float("-inf")
    raw[2, 0, 7] = float("inf")
    raw[2, 1, 9] = float("nan")
    x = torch.full((B, L), V, dtype=torch.int64, device=gpu)
    rawg = raw.to(gpu)
    print(f"case non-finite rows V={V} workspace={workspace}", flush=True)
    sc = ops.unmask_step(rawg, x, V, 0.0, shift=0) if workspace else _step_without_workspace(rawg, x, V, 0.0)
    bad = torch.tensor([[0, 1, 1, 0], [1, 1, 1, 1], [1, 1, 0, 0]], dtype=torch.bool, device=gpu)
    assert torch.equal(sc.row_conf.isnan(), bad)
    assert bool(((sc.row_tok >= 0) & (sc.row_tok < V)).all())
    assert sc.row_tok[0, 1:3].tolist() == [0, 0] and sc.row_tok[1].tolist() == [0] * 4
    # threshold 0: every position with a probability is unmasked
    assert torch.equal(x == V, bad) and torch.equal(x[~bad], rawg.argmax(dim=-1)[~bad])
    assert sc.counts.tolist() == [4, 8, 2, 0]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_sums_of_exponentials_carry_no_bias(gpu, dtype):
    """The chunks' sums of exp(l - max), which the kernel leaves in the workspace, against 64
    bits. Each of a chunk's 8192 terms has a relative error under 2^-22 and the fp32
    additions one of 2^-24 at most, 13 deep; their signs vary, so a chunk is off by some 1e-7
    at most, and the mean over 512 rows by 1e-8. A systematic error of the terms (log2 e
    rounded to 24 bits: 1.3e-8 of |l - max|, about 8 here) shows in that mean, at 4e-8 and
    more."""
    B, L, V = 64, 8, 40960  # five whole chunks per row, and one for rows off a 16-byte boundary
    raw = (torch.randn(B, L, V, generator=torch.Generator().manual_seed(4)) * 2).to(dtype).to(gpu)
    x = torch.full((B, L), V, dtype=torch.int64, device=gpu)
    sc, need = ops.UnmaskScratch(B, L, gpu), ctypes.c_size_t(0)
    _ffi.check(_ffi.lib().fdllm_unmask_workspace_size(V, B, L, ctypes.byref(need)), "size")
    ws = torch.empty(need.value // 4, dtype=torch.float32, device=gpu)
    _ffi.check(_ffi.lib().fdllm_unmask_step_ws(
        raw.data_ptr(), raw.stride(0), raw.stride(1), V, 0, 0, x.data_ptr(), x.stride(0), None, V, 2.0, -1,
        sc.row_tok.data_ptr(), sc.row_conf.data_ptr(), sc.counts.data_ptr(), B, L, _ffi.dtype_code(dtype),
        ws.data_ptr(), need.value, _ffi.stream_ptr(gpu)), "fdllm_unmask_step_ws")
    got = ws.view(B, L, -1, 4)[:, :, :5]  # (max, sum, index, near) per chunk
    r = raw.view(B, L, 5, 8192).double()
    top = r.amax(dim=-1)
    assert torch.equal(got[..., 0].double(), top)
    err = got[..., 1].double() / torch.exp(r - top[..., None]).sum(dim=-1) - 1
    print(f"rms {err.pow(2).mean().sqrt():.2e} mean {err.mean():.2e}")
    assert abs(float(err.mean())) < 2e-8 and float(err.abs().max()) < 5e-7


@pytest.mark.parametrize("V", [1, 1000, 8192, 8193, 24576, 24584, 32001])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_step_without_a_workspace(gpu, V, dtype):
    """The two forms of the step choose the same tokens; confidences within one ulp of the
    logits' type (the sums' order differs); excluded tokens (-inf) take no part."""
    g = torch.Generator().manual_seed(V)
    raw = (torch.randn(5, 6, V, generator=g) * 2).to(dtype).to(gpu)
    raw[1, :, :V // 2] = raw[2, 3, V // 2 + 1:] = float("-inf")  # most of a row may be excluded
    x = torch.full((5, 6), V + 5, dtype=torch.int64, device=gpu)
    y = x.clone()
    a = ops.unmask_step(raw, x, V + 5, 0.4, shift=0)
    b = _step_without_workspace(raw, y, V + 5, 0.4)
    ulp = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
    assert torch.equal(a.row_tok, b.row_tok) and torch.equal(x, y) and torch.equal(a.counts, b.counts)
    torch.testing.assert_close(a.row_conf, b.row_conf, atol=0, rtol=ulp)

// Greedy sampling + threshold unmasking of one diffusion step (fdllm_unmask_step):
// softmax / argmax / confidence over the vocabulary (modeling.py:2263-2270 at
// temperature 0) and the unmask rule of generation_functions.py:784-807, on the GPU,
// so the step leaves its decisions in device memory and the host reads four counters.
//
// The greedy token is the first index whose probability, rounded to the logits' type,
// equals the rounded maximum probability (torch.argmax over the rounded softmax returns
// the first of equal values); only logits within 2^-7 of the maximum can tie.
//
// With a workspace (fdllm_unmask_step_ws) a long row is cut into chunks of kChunk logits, one
// workgroup each (unmask_cut says from where): unmask_chunks_kernel reads its chunk once into registers and writes
// (max, its first index, sum of exp(l - max), whether a smaller logit could still tie);
// unmask_finish_kernel, one workgroup per sequence, folds the chunks of each position,
// re-reads only the chunks in which a tie is possible, and applies the unmask rule.
// What bounds it: the one read of the logits. 16 x 8 positions of 152064 bf16 logits
// (38.9 MB): 10.4 us (3.7 TB/s) + 4.4 us for the finish, against 50.0 us (128 workgroups, an
// online rescale chain per thread and the second read) + 4.4 us for the form below.
// 8192 logits per workgroup (four 16-byte loads per thread in flight, 2432 workgroups)
// keep every compute unit at eight workgroups.
//
// Without one (fdllm_unmask_step), and for short rows: unmask_rows_kernel, one workgroup per position, reads
// its row twice (pass 1: running maximum, its first index and the online sum; pass 2: the
// first tie), then unmask_select_kernel, one wave per sequence, applies the rule.
#include <math.h>

#include "fdllm_common.h"

namespace fdllm {
namespace {

struct UnmaskArgs {
  const uint16_t* logits;
  int64_t lg_sb, lg_sr;
  int V, row_offset, shift;
  int64_t* tokens;
  int64_t tok_sb;
  uint8_t* finished;
  int64_t mask_id, stop_token;
  float threshold;
  int64_t* row_tok;
  float* row_conf;
  int32_t* counts;
  int B, L;
  float4* parts;  // [B * L][n_chunks] partials of the chunked form
  int n_chunks;
};

constexpr int kThreads = 512;

template <typename T>
__device__ __forceinline__ float rnd16(float x) {
  return Elt<T>::round(x);
}

// (max, first index, sum of exp(x - max)) of two partial states
__device__ __forceinline__ void combine(float& m, int& idx, float& s, float m2, int idx2, float s2) {
  if (m2 > m || (m2 == m && idx2 < idx)) {
    const float sc = m == -INFINITY ? 0.f : expf(m - m2);  // (a NaN sum is kept)
    s = s * sc + s2;
    m = m2;
    idx = idx2;
  } else {
    const float sc = m2 == -INFINITY ? 0.f : expf(m2 - m);
    s += s2 * sc;
  }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void unmask_rows_kernel(const UnmaskArgs a) {
  __shared__ float sm[kThreads / 64], ss[kThreads / 64];
  __shared__ int si[kThreads / 64];
  __shared__ float s_fin[2];
  __shared__ int s_fin_idx;
  const int i = blockIdx.x;
  const int b = blockIdx.y;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  if (i == 0 && b == 0 && tid < 4) a.counts[tid] = 0;  // kernel 2 accumulates into these
  const int r = max(a.row_offset + i - a.shift, 0);
  const uint16_t* row = a.logits + b * a.lg_sb + static_cast<int64_t>(r) * a.lg_sr;
  const bool vec = (a.V % 8 == 0) && ((reinterpret_cast<uintptr_t>(row) & 15u) == 0);

  // ---- pass 1: max, its first index, sum of exp(x - max). While a thread has seen nothing
  // above -inf its sum is 0, or NaN after a NaN logit, which then stays
  float m = -INFINITY, s = 0.f;
  int idx = 0x7fffffff;
  if (vec) {
    const int nv = a.V / 8;
    for (int v = tid; v < nv; v += kThreads) {
      const u32x4 w = *reinterpret_cast<const u32x4*>(row + 8 * v);
      float x[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        x[2 * j] = Elt<T>::lo(w[j]);
        x[2 * j + 1] = Elt<T>::hi(w[j]);
      }
      float mv = x[0];
      int iv = 0;
#pragma unroll
      for (int j = 1; j < 8; ++j)
        if (x[j] > mv) {
          mv = x[j];
          iv = j;
        }
      if (mv > m) {  // a strictly larger value: indices grow, so the first one is kept
        if (m != -INFINITY) s *= expf(m - mv);
        m = mv;
        idx = 8 * v + iv;
      }
      const float ref = m == -INFINITY ? 0.f : m;
#pragma unroll
      for (int j = 0; j < 8; ++j) s += expf(x[j] - ref);
    }
  } else {
    for (int v = tid; v < a.V; v += kThreads) {
      const float x = Elt<T>::lo(row[v]);
      if (x > m) {
        if (m != -INFINITY) s *= expf(m - x);
        m = x;
        idx = v;
      }
      s += expf(x - (m == -INFINITY ? 0.f : m));
    }
  }
  // wave then workgroup reduction
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const float m2 = __shfl_xor(m, o, kWave);
    const int i2 = __shfl_xor(idx, o, kWave);
    const float s2 = __shfl_xor(s, o, kWave);
    combine(m, idx, s, m2, i2, s2);
  }
  if (lane == 0) {
    sm[wave] = m;
    si[wave] = idx;
    ss[wave] = s;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < kThreads / 64; ++w) combine(m, idx, s, sm[w], si[w], ss[w]);
    s_fin[0] = m;
    s_fin[1] = s;
    s_fin_idx = idx;
  }
  __syncthreads();
  m = s_fin[0];
  s = m == -INFINITY ? __builtin_nanf("") : s_fin[1];  // no finite logit: no probability
  // ---- pass 2: first index whose rounded probability equals the rounded maximum
  const float pmax = rnd16<T>(1.f / s);
  const float lo_cut = m - 0.0078125f;  // exp(x - m) < 1 - 2^-8 below it: no tie possible
  int cand = s_fin_idx;
  if (vec) {
    const int nv = a.V / 8;
    for (int v = tid; v < nv; v += kThreads) {
      const u32x4 w = *reinterpret_cast<const u32x4*>(row + 8 * v);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float x = (j & 1) ? Elt<T>::hi(w[j >> 1]) : Elt<T>::lo(w[j >> 1]);
        if (x >= lo_cut && 8 * v + j < cand && rnd16<T>(expf(x - m) / s) == pmax) cand = 8 * v + j;
      }
    }
  } else {
    for (int v = tid; v < a.V; v += kThreads) {
      const float x = Elt<T>::lo(row[v]);
      if (x >= lo_cut && v < cand && rnd16<T>(expf(x - m) / s) == pmax) cand = v;
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) cand = min(cand, __shfl_xor(cand, o, kWave));
  __syncthreads();
  if (lane == 0) si[wave] = cand;
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < kThreads / 64; ++w) cand = min(cand, si[w]);
    if (cand >= a.V) cand = 0;  // no logit above -inf: argmax over NaN probabilities
    a.row_tok[b * a.L + i] = cand;
    a.row_conf[b * a.L + i] = pmax;
  }
}

// The unmask rule of one sequence on one wave: lane i < L is position i of the sub-block,
// conf its confidence and tok its token. A position without a confidence (NaN: non-finite
// logits) stays masked, so that the caller sees a step without progress and no token that
// nothing backs.
__device__ __forceinline__ void select_positions(const UnmaskArgs& a, int b, int i, float conf, int64_t tok) {
  const bool live = i < a.L;
  const bool fin = a.finished != nullptr && a.finished[b] != 0;
  int64_t* tp = a.tokens + b * a.tok_sb + i;
  const int64_t t = live ? *tp : 0;
  const bool masked = live && t == a.mask_id && !fin;
  const bool known = masked && conf == conf;
  const float c = known ? conf : -INFINITY;
  bool unmask = c > a.threshold;
  // most confident masked position, first on ties (torch.argmax over the row)
  float cm = live ? c : -INFINITY;
  int im = live ? i : 0x7fffffff;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const float c2 = __shfl_xor(cm, o, kWave);
    const int i2 = __shfl_xor(im, o, kWave);
    if (c2 > cm || (c2 == cm && i2 < im)) {
      cm = c2;
      im = i2;
    }
  }
  if (i == im) unmask = true;
  unmask = unmask && known;
  if (unmask) *tp = tok;
  const bool stop_hit = unmask && a.stop_token >= 0 && tok == a.stop_token;
  const uint64_t stops = __builtin_amdgcn_ballot_w64(stop_hit);
  const bool fin_after = fin || stops != 0;
  const uint64_t n_unmask = __builtin_amdgcn_ballot_w64(unmask);
  const uint64_t n_left = __builtin_amdgcn_ballot_w64(masked && !unmask && !fin_after);
  const bool first_masked = live && i == 0 && !unmask && t == a.mask_id;
  if (i == 0) {
    if (a.finished != nullptr && stops != 0) a.finished[b] = 1;
    atomicAdd(&a.counts[0], static_cast<int>(__builtin_popcountll(n_unmask)));
    atomicAdd(&a.counts[1], static_cast<int>(__builtin_popcountll(n_left)));
    atomicAdd(&a.counts[2], first_masked ? 1 : 0);
    atomicAdd(&a.counts[3], fin_after ? 1 : 0);
  }
}

// One wave per sequence.
__global__ __launch_bounds__(64) void unmask_select_kernel(const UnmaskArgs a) {
  const int b = blockIdx.x;
  const int i = threadIdx.x;
  const bool live = i < a.L;
  select_positions(a, b, i, live ? a.row_conf[b * a.L + i] : -INFINITY, live ? a.row_tok[b * a.L + i] : 0);
}

// ---------------------------------------------------------------------------
// Chunked form.
constexpr int kChunkThreads = 256;
constexpr int kChunkVecs = 4;  // 16-byte vectors per thread, all in flight at once
constexpr int kChunk = kChunkThreads * kChunkVecs * 8;  // logits per workgroup
constexpr int kFinishThreads = 512;

// Row r's logits as 16-byte vectors from the aligned address at or below its start: the
// first `mis` elements of vector 0 belong to whatever precedes the row, and vector nv - 1
// may run past its end. Every vector holds at least one logit of the row, so an aligned
// 16-byte load of it touches no page that the row does not.
struct RowVecs {
  const u32x4* v;
  int mis, nv;
};
__device__ __forceinline__ RowVecs row_vecs(const UnmaskArgs& a, int b, int i) {
  const int r = max(a.row_offset + i - a.shift, 0);
  const uint16_t* row = a.logits + b * a.lg_sb + static_cast<int64_t>(r) * a.lg_sr;
  const int mis = static_cast<int>((reinterpret_cast<uintptr_t>(row) & 15u) >> 1);
  return RowVecs{reinterpret_cast<const u32x4*>(row - mis), mis, (a.V + mis + 7) / 8};
}
// logits 8 v - mis + 0..7 of a row, -inf where there is none
template <typename T>
__device__ __forceinline__ void unpack_vec(const u32x4& w, int v, int mis, int V, float* x) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    x[2 * j] = Elt<T>::lo(w[j]);
    x[2 * j + 1] = Elt<T>::hi(w[j]);
  }
  const int j0 = 8 * v - mis;
  if (j0 < 0 || j0 + 8 > V) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j0 + j < 0 || j0 + j >= V) x[j] = -INFINITY;
  }
}

// Whether T has a value in [m - 2^-7, m): the spacing below m is at most 2^-7 up to these
// magnitudes (bf16: 8 significant bits, fp16: 11), larger above.
template <typename T>
__device__ __forceinline__ bool can_tie_below(float m);
template <>
__device__ __forceinline__ bool can_tie_below<bf16_t>(float m) { return m <= 2.f && m > -2.f; }
template <>
__device__ __forceinline__ bool can_tie_below<f16_t>(float m) { return m <= 16.f && m > -16.f; }

template <typename T>
__global__ __launch_bounds__(kChunkThreads) void unmask_chunks_kernel(const UnmaskArgs a) {
  constexpr int NW = kChunkThreads / 64;
  __shared__ float sm[NW], ss[NW];
  __shared__ int si[NW], sn[NW];
  const int chunk = blockIdx.x, i = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  if (chunk == 0 && i == 0 && b == 0 && tid < 4) a.counts[tid] = 0;  // the finish kernel accumulates into these
  const RowVecs rv = row_vecs(a, b, i);
  const int v0 = chunk * (kChunk / 8) + tid;
  u32x4 w[kChunkVecs];
#pragma unroll
  for (int k = 0; k < kChunkVecs; ++k) {
    const int v = v0 + k * kChunkThreads;
    if (v < rv.nv) w[k] = __builtin_nontemporal_load(rv.v + v);
  }
  float x[kChunkVecs][8];
  float m = -INFINITY;
#pragma unroll
  for (int k = 0; k < kChunkVecs; ++k) {
    const int v = v0 + k * kChunkThreads;
    if (v < rv.nv) {
      unpack_vec<T>(w[k], v, rv.mis, a.V, x[k]);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) x[k][j] = -INFINITY;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) m = fmaxf(m, x[k][j]);
  }
  m = wave_allreduce_max(m);
  if (lane == 0) sm[wave] = m;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < NW; ++u) m = fmaxf(m, sm[u]);
  // exp relative to the chunk's maximum (0 for a chunk of -inf: its sum is then zero; a NaN
  // or +inf logit makes it NaN, as in a softmax), as exp2 of the product with log2 e in two
  // parts: with one, the constant's rounding biases every term the same way. Error of a row's
  // sum against 64 bits, rms over 128 rows of 152064 bf16 logits of N(0, 2): 4.5e-8, 6.9e-8
  // with one part, 4.4e-8 with expf (which takes 4 us more), 7.1e-8 in unmask_rows_kernel;
  // with one clear token per row 1.4e-7, 1.5e-7, 1.4e-7 and 6.5e-7.
  const float ref = m == -INFINITY ? 0.f : m;
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < kChunkVecs; ++k)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float t = x[k][j] - ref;
      s += __builtin_amdgcn_exp2f(__builtin_fmaf(t, 1.44269502f, t * 1.92596299e-8f));
    }
  int idx = 0x7fffffff;
#pragma unroll
  for (int k = kChunkVecs - 1; k >= 0; --k)
#pragma unroll
    for (int j = 7; j >= 0; --j)
      if (x[k][j] == m) idx = 8 * (v0 + k * kChunkThreads) + j - rv.mis;
  int near = 0;
  if (can_tie_below<T>(m)) {  // uniform over the workgroup
#pragma unroll
    for (int k = 0; k < kChunkVecs; ++k)
#pragma unroll
      for (int j = 0; j < 8; ++j) near |= x[k][j] < m && x[k][j] >= m - 0.0078125f;
  }
  s = wave_allreduce_sum(s);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) idx = min(idx, __shfl_xor(idx, o, kWave));
  const bool any_near = __builtin_amdgcn_ballot_w64(near != 0) != 0;
  if (lane == 0) {
    ss[wave] = s;
    si[wave] = idx;
    sn[wave] = any_near;
  }
  __syncthreads();
  if (tid == 0) {
    for (int u = 1; u < NW; ++u) {
      s += ss[u];
      idx = min(idx, si[u]);
    }
    int nr = 0;
    for (int u = 0; u < NW; ++u) nr |= sn[u];
    // a chunk of -inf has no index of its own
    a.parts[(static_cast<int64_t>(b) * a.L + i) * a.n_chunks + chunk] =
        make_float4(m, s, __int_as_float(m == -INFINITY ? 0x7fffffff : idx), __int_as_float(nr));
  }
}

// One workgroup per sequence; wave w folds positions w, w + 8, ...
template <typename T>
__global__ __launch_bounds__(kFinishThreads) void unmask_finish_kernel(const UnmaskArgs a) {
  __shared__ float s_conf[64];
  __shared__ int s_tok[64];
  const int b = blockIdx.x;
  const int lane = threadIdx.x & 63;
  for (int i = threadIdx.x >> 6; i < a.L; i += kFinishThreads / 64) {
    const float4* parts = a.parts + (static_cast<int64_t>(b) * a.L + i) * a.n_chunks;
    float m = -INFINITY;
    for (int c = lane; c < a.n_chunks; c += 64) m = fmaxf(m, parts[c].x);
    m = wave_allreduce_max(m);
    float s = 0.f;
    for (int c = lane; c < a.n_chunks; c += 64) {
      const float4 p = parts[c];
      // a NaN sum is kept; a chunk of -inf adds its zero
      s += p.x == -INFINITY ? p.y : p.y * expf(p.x - m);
    }
    s = wave_allreduce_sum(s);
    if (m == -INFINITY) s = __builtin_nanf("");  // no finite logit: no probability
    const float pmax = rnd16<T>(1.f / s);
    const float lo_cut = m - 0.0078125f;
    int cand = 0x7fffffff;   // first index of the maximum (kept where no comparison holds: NaN)
    int first = 0x7fffffff;  // first index that ties
    for (int c0 = 0; c0 < a.n_chunks; c0 += 64) {
      const int c = c0 + lane;
      const float4 p = c < a.n_chunks ? parts[c] : make_float4(-INFINITY, 0.f, 0.f, 0.f);
      const int idx = c < a.n_chunks ? __float_as_int(p.z) : 0x7fffffff;
      if (c < a.n_chunks && p.x == m) cand = min(cand, idx);
      const bool cut = p.x >= lo_cut;
      if (cut && rnd16<T>(expf(p.x - m) / s) == pmax) first = min(first, idx);
      // chunks that hold other logits close to their maximum are read again
      uint64_t todo = __builtin_amdgcn_ballot_w64(cut && __float_as_int(p.w) != 0);
      if (todo != 0) {
        const RowVecs rv = row_vecs(a, b, i);
        while (todo != 0) {
          const int cc = c0 + __builtin_ctzll(todo);
          todo &= todo - 1;
          const int ve = min((cc + 1) * (kChunk / 8), rv.nv);
          for (int v = cc * (kChunk / 8) + lane; v < ve; v += 64) {
            float x[8];
            unpack_vec<T>(rv.v[v], v, rv.mis, a.V, x);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              const int at = 8 * v + j - rv.mis;
              if (x[j] >= lo_cut && at < first && rnd16<T>(expf(x[j] - m) / s) == pmax) first = at;
            }
          }
        }
      }
    }
    cand = min(cand, first);
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) cand = min(cand, __shfl_xor(cand, o, kWave));
    if (cand >= a.V) cand = 0;  // no logit above -inf: argmax over NaN probabilities
    if (lane == 0) {
      s_conf[i] = pmax;
      s_tok[i] = cand;
      a.row_tok[b * a.L + i] = cand;
      a.row_conf[b * a.L + i] = pmax;
    }
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const bool live = lane < a.L;
    select_positions(a, b, lane, live ? s_conf[lane] : -INFINITY, live ? s_tok[lane] : 0);
  }
}

// Whether rows are cut into chunks, given a workspace: not short ones, which the row kernel
// reads twice in the time of the finish kernel, whose workgroup per sequence folds eight
// positions at a time and alone re-reads the chunks with possible ties. us, cut / whole, at
// N(0, 2) logits (N(0, 0.2): ties possible): vocab 8000, 1 x 8 positions 7.2 / 9.3 (7.6 /
// 9.1), 4 x 64 16.4 / 9.8 (34 / 9.5); 24576, 16 x 8 8.7 / 14.1 (21.1 / 14.0), 4 x 64 19.2 /
// 13.5 (31.5 / 13.7); 32001 (no multiple of 8, read element by element), 16 x 8 9.0 / 29.7
// (14.4 / 29.6); 152064, 16 x 8 13.7 / 53.1.
inline bool unmask_cut(int vocab, int positions) {
  return vocab > (vocab % 8 != 0 ? 1 : positions > 32 ? 6 : 3) * kChunk;
}

// Chunks of a row, one more where a row start off a 16-byte boundary can need it.
inline int64_t unmask_chunks(int vocab) { return (static_cast<int64_t>(vocab) + 7 + kChunk - 1) / kChunk; }

}  // namespace
}  // namespace fdllm

extern "C" int fdllm_unmask_workspace_size(int vocab, int batch, int num_positions, size_t* bytes) {
  using namespace fdllm;
  FDLLM_CHECK_ARG(bytes != nullptr && vocab > 0 && batch >= 0 && num_positions >= 0 && num_positions <= 64,
                  "fdllm_unmask_workspace_size: need 0 <= num_positions <= 64 and vocab > 0");
  *bytes = 0;
  if (unmask_cut(vocab, num_positions))
    *bytes = static_cast<size_t>(unmask_chunks(vocab)) * batch * num_positions * sizeof(float4);
  return FDLLM_OK;
}

namespace fdllm {
namespace {

int unmask_launch(const char* what, const void* logits, int64_t logits_stride_b, int64_t logits_stride_row, int vocab,
                  int row_offset, int shift, int64_t* tokens, int64_t tokens_stride_b, uint8_t* finished,
                  int64_t mask_id, float threshold, int64_t stop_token, int64_t* row_tok, float* row_conf,
                  int32_t* counts, int batch, int num_positions, int dtype, bool chunked, void* workspace,
                  size_t workspace_bytes, void* stream) {
  FDLLM_CHECK_ARG(dtype == FDLLM_DTYPE_BF16 || dtype == FDLLM_DTYPE_F16,
                  "%s: dtype %d unsupported (bf16 or fp16 logits)", what, dtype);
  FDLLM_CHECK_ARG(batch >= 0 && num_positions >= 0 && num_positions <= 64 && vocab > 0,
                  "%s: need 0 <= num_positions <= 64 and vocab > 0", what);
  FDLLM_CHECK_ARG(shift == 0 || shift == 1, "%s: shift must be 0 or 1", what);
  if (batch == 0 || num_positions == 0) return FDLLM_OK;
  FDLLM_CHECK_ARG(batch < 65536, "%s: batch too large", what);
  FDLLM_CHECK_ARG(logits && tokens && row_tok && row_conf && counts, "%s: null pointer", what);
  UnmaskArgs a;
  a.logits = static_cast<const uint16_t*>(logits);
  a.lg_sb = logits_stride_b;
  a.lg_sr = logits_stride_row;
  a.V = vocab;
  a.row_offset = row_offset;
  a.shift = shift;
  a.tokens = tokens;
  a.tok_sb = tokens_stride_b;
  a.finished = finished;
  a.mask_id = mask_id;
  a.stop_token = stop_token;
  a.threshold = threshold;
  a.row_tok = row_tok;
  a.row_conf = row_conf;
  a.counts = counts;
  a.B = batch;
  a.L = num_positions;
  hipStream_t s = static_cast<hipStream_t>(stream);
  a.parts = nullptr;
  a.n_chunks = 0;
  if (chunked && unmask_cut(vocab, num_positions)) {
    const int64_t chunks = unmask_chunks(vocab);
    const size_t need = static_cast<size_t>(chunks) * batch * num_positions * sizeof(float4);
    if (workspace == nullptr || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 15u) != 0) {
      set_last_error("%s: workspace of %zu bytes required (got %zu)", what, need, workspace_bytes);
      return FDLLM_ERR_WORKSPACE;
    }
    a.parts = static_cast<float4*>(workspace);
    a.n_chunks = static_cast<int>(chunks);
    const dim3 g(static_cast<unsigned>(chunks), num_positions, batch);
    if (dtype == FDLLM_DTYPE_BF16) {
      unmask_chunks_kernel<bf16_t><<<g, dim3(kChunkThreads), 0, s>>>(a);
      unmask_finish_kernel<bf16_t><<<dim3(batch), dim3(kFinishThreads), 0, s>>>(a);
    } else {
      unmask_chunks_kernel<f16_t><<<g, dim3(kChunkThreads), 0, s>>>(a);
      unmask_finish_kernel<f16_t><<<dim3(batch), dim3(kFinishThreads), 0, s>>>(a);
    }
    FDLLM_RETURN_LAUNCH_STATUS(what);
  }
  const dim3 g1(num_positions, batch);
  if (dtype == FDLLM_DTYPE_BF16) unmask_rows_kernel<bf16_t><<<g1, dim3(kThreads), 0, s>>>(a);
  else unmask_rows_kernel<f16_t><<<g1, dim3(kThreads), 0, s>>>(a);
  unmask_select_kernel<<<dim3(batch), dim3(64), 0, s>>>(a);
  FDLLM_RETURN_LAUNCH_STATUS(what);
}

}  // namespace
}  // namespace fdllm

extern "C" int fdllm_unmask_step(const void* logits, int64_t logits_stride_b, int64_t logits_stride_row,
                                 int vocab, int row_offset, int shift, int64_t* tokens, int64_t tokens_stride_b,
                                 uint8_t* finished, int64_t mask_id, float threshold, int64_t stop_token,
                                 int64_t* row_tok, float* row_conf, int32_t* counts, int batch, int num_positions,
                                 int dtype, void* stream) {
  return fdllm::unmask_launch("fdllm_unmask_step", logits, logits_stride_b, logits_stride_row, vocab, row_offset, shift,
                              tokens, tokens_stride_b, finished, mask_id, threshold, stop_token, row_tok, row_conf,
                              counts, batch, num_positions, dtype, false, nullptr, 0, stream);
}

extern "C" int fdllm_unmask_step_ws(const void* logits, int64_t logits_stride_b, int64_t logits_stride_row,
                                    int vocab, int row_offset, int shift, int64_t* tokens, int64_t tokens_stride_b,
                                    uint8_t* finished, int64_t mask_id, float threshold, int64_t stop_token,
                                    int64_t* row_tok, float* row_conf, int32_t* counts, int batch, int num_positions,
                                    int dtype, void* workspace, size_t workspace_bytes, void* stream) {
  return fdllm::unmask_launch("fdllm_unmask_step_ws", logits, logits_stride_b, logits_stride_row, vocab, row_offset,
                              shift, tokens, tokens_stride_b, finished, mask_id, threshold, stop_token, row_tok,
                              row_conf, counts, batch, num_positions, dtype, true, workspace, workspace_bytes, stream);
}

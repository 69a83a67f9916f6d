// Linear layers of a few token rows (fdllm_linear), such as the MLP and lm_head products
// of a diffusion step, on the weight-streaming kernel of skinny_gemm.h, plain (with an
// optional bias) or with the MLP's gate and up projections in one pass and their
// SiLU-gated product as the epilogue (modeling.py:153-166).
#include "launch_turn.h"
#include "skinny_gemm.h"

namespace fdllm {
namespace {

template <typename T>
__device__ __forceinline__ void put8(uint16_t* out, const float* y) {
  u32x4 w;
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = Elt<T>::pack(y[2 * i], y[2 * i + 1]);
  *reinterpret_cast<u32x4*>(out) = w;
}

// bytes of weight rows [n0, n0 + count) that exist
__device__ __forceinline__ int row_bytes(int n0, int count, int N, int stride) {
  return max(min(count, N - n0), 0) * stride;
}

template <typename T>
struct LinearEpi {
  const uint16_t* w;
  const uint16_t* bias;
  uint16_t* out;
  int N, K;

  template <int BN>
  __device__ __forceinline__ SkinnyRows rows(int tile) const {
    const int n0 = tile * BN;
    const uint16_t* p = w + static_cast<int64_t>(n0) * K;
    return SkinnyRows{p, p + static_cast<int64_t>(BN / 2) * K, row_bytes(n0, BN / 2, N, K * 2),
                      row_bytes(n0 + BN / 2, BN / 2, N, K * 2)};
  }
  template <int BN>
  __device__ __forceinline__ void store(int tile, int m, int blk, const f32x4 v[4]) const {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int n = tile * BN + h * (BN / 2) + blk * 8;
      if (n >= N) continue;  // N is a multiple of 8
      float y[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = v[2 * h + (j >> 2)][j & 3];
      if (bias != nullptr) {
        const u32x4 bw = *reinterpret_cast<const u32x4*>(bias + n);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          y[2 * j] += Elt<T>::lo(bw[j]);
          y[2 * j + 1] += Elt<T>::hi(bw[j]);
        }
      }
      put8<T>(out + static_cast<int64_t>(m) * N + n, y);
    }
  }
};

// round(round(silu(round(x wg^T))) * round(x wu^T)): the roundings of the separate layers
// and of fdllm_silu_mul.
template <typename T>
struct GatedEpi {
  const uint16_t* wg;
  const uint16_t* wu;
  uint16_t* out;
  int N, K;

  template <int BN>
  __device__ __forceinline__ SkinnyRows rows(int tile) const {
    const int n0 = tile * (BN / 2);
    const int bytes = row_bytes(n0, BN / 2, N, K * 2);
    return SkinnyRows{wg + static_cast<int64_t>(n0) * K, wu + static_cast<int64_t>(n0) * K, bytes, bytes};
  }
  template <int BN>
  __device__ __forceinline__ void store(int tile, int m, int blk, const f32x4 v[4]) const {
    const int n = tile * (BN / 2) + blk * 8;
    if (n >= N) return;
    float y[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float gt = Elt<T>::round(v[j >> 2][j & 3]);
      const float up = Elt<T>::round(v[2 + (j >> 2)][j & 3]);
      y[j] = Elt<T>::round(gt / (1.0f + expf(-gt))) * up;
    }
    put8<T>(out + static_cast<int64_t>(m) * N + n, y);
  }
};

// Columns per workgroup: enough that the tiles fill the compute units about once, which
// keeps the re-reads of the activation rows and the partial sums few.
constexpr int kWide = 160, kNarrow = 64;
constexpr int kWideFrom = 16384;  // columns (gate and up together): 103 wide tiles
inline int bn_of(int64_t columns) { return columns >= kWideFrom ? kWide : kNarrow; }

template <bool F16, typename Epi>
void launch(const SkinnyArgs& a, int bn, const Epi& epi, hipStream_t s) {
  if (bn == kWide) skinny_launch<F16, kWide>(a, epi, s);
  else skinny_launch<F16, kNarrow>(a, epi, s);
}

inline bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int check_sizes(int rows, int N, int K, const char* what) {
  FDLLM_CHECK_ARG(rows >= 0 && rows <= kSkinnyMaxRows, "%s: rows %d unsupported (at most %d)", what, rows, kSkinnyMaxRows);
  FDLLM_CHECK_ARG(N >= 0 && N % 8 == 0 && N <= (1 << 24), "%s: out_features %d must be a multiple of 8 (at most 2^24)", what, N);
  FDLLM_CHECK_ARG(K >= 64 && K % 64 == 0 && K <= 65536, "%s: in_features %d must be a multiple of 64 (at most 65536)", what, K);
  return FDLLM_OK;
}

SkinnyArgs plan(int rows, int N, int K, bool gated, bool workspace, int* bn) {
  SkinnyArgs a = {};
  *bn = bn_of(gated ? int64_t{2} * N : N);
  const int per = gated ? *bn / 2 : *bn;
  a.T = rows;
  a.ku = K / 64;
  a.tiles = (N + per - 1) / per;
  skinny_plan(a, workspace);
  return a;
}

}  // namespace
}  // namespace fdllm

extern "C" int fdllm_linear_workspace_size(int rows, int out_features, int in_features, int gated, size_t* bytes) {
  using namespace fdllm;
  FDLLM_CHECK_ARG(bytes != nullptr, "fdllm_linear_workspace_size: null pointer");
  const int rc = check_sizes(rows, out_features, in_features, "fdllm_linear_workspace_size");
  if (rc != FDLLM_OK) return rc;
  *bytes = 0;
  if (rows == 0 || out_features == 0) return FDLLM_OK;
  int bn;
  const SkinnyArgs a = plan(rows, out_features, in_features, gated != 0, true, &bn);
  *bytes = skinny_workspace(a, bn);
  return FDLLM_OK;
}

extern "C" int fdllm_linear(const void* x, int64_t x_stride_row, const void* w, const void* w_up, const void* bias,
                            void* out, int rows, int out_features, int in_features, int dtype, void* workspace,
                            size_t workspace_bytes, void* stream) {
  using namespace fdllm;
  FDLLM_CHECK_ARG(dtype == FDLLM_DTYPE_BF16 || dtype == FDLLM_DTYPE_F16,
                  "fdllm_linear: dtype %d unsupported (bf16 or fp16)", dtype);
  const int rc = check_sizes(rows, out_features, in_features, "fdllm_linear");
  if (rc != FDLLM_OK) return rc;
  if (rows == 0 || out_features == 0) return FDLLM_OK;
  FDLLM_CHECK_ARG(x && w && out, "fdllm_linear: null pointer");
  FDLLM_CHECK_ARG(w_up == nullptr || bias == nullptr, "fdllm_linear: the gated form takes no bias");
  for (const void* p : {x, w, w_up, bias, static_cast<const void*>(out), static_cast<const void*>(workspace)})
    FDLLM_CHECK_ARG(p == nullptr || al16(p), "fdllm_linear: pointers must be 16-byte aligned");
  FDLLM_CHECK_ARG(x_stride_row >= in_features && x_stride_row % 8 == 0 && x_stride_row <= (1 << 22),
                  "fdllm_linear: x_stride_row %lld must be a multiple of 8, at least in_features",
                  static_cast<long long>(x_stride_row));
  int bn;
  SkinnyArgs a = plan(rows, out_features, in_features, w_up != nullptr, workspace != nullptr, &bn);
  const size_t need = skinny_workspace(a, bn);
  FDLLM_CHECK_ARG(workspace == nullptr || workspace_bytes >= need, "fdllm_linear: workspace of %zu bytes, need %zu",
                  workspace_bytes, need);
  a.x = static_cast<const uint16_t*>(x);
  a.x_bytes = static_cast<int>((static_cast<int64_t>(rows - 1) * x_stride_row + in_features) * 2);
  a.x_stride_b = static_cast<int>(x_stride_row * 2);
  a.w_stride_b = in_features * 2;
  a.cnt = static_cast<int*>(workspace);
  a.part = static_cast<uint8_t*>(workspace) + kSkinnyCounterBytes;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const uint16_t* w0 = static_cast<const uint16_t*>(w);
  const uint16_t* w1 = static_cast<const uint16_t*>(w_up);
  const uint16_t* bi = static_cast<const uint16_t*>(bias);
  uint16_t* o = static_cast<uint16_t*>(out);
  const WorkspaceTurn turn(need > 0 ? workspace : nullptr);
  if (dtype == FDLLM_DTYPE_BF16) {
    if (w1) launch<false>(a, bn, GatedEpi<bf16_t>{w0, w1, o, out_features, in_features}, s);
    else launch<false>(a, bn, LinearEpi<bf16_t>{w0, bi, o, out_features, in_features}, s);
  } else {
    if (w1) launch<true>(a, bn, GatedEpi<f16_t>{w0, w1, o, out_features, in_features}, s);
    else launch<true>(a, bn, LinearEpi<f16_t>{w0, bi, o, out_features, in_features}, s);
  }
  FDLLM_RETURN_LAUNCH_STATUS("fdllm_linear");
}

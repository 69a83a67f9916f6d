// Product of at most 128 activation rows with streamed weight rows, gfx950:
//
//   acc[m][n] = sum_k x[m][k] * w[n][k]      m < T <= 128, k < K (a multiple of 64)
//
// shared by the linear layers (linear.hip) and the q / k / v projections (rope_kv.hip).
// What bounds it: every weight row is read once from HBM (T flop per byte, far below the
// matrix cores' rate), and each workgroup reads the token rows of its K range from L2, so
// the tile is made for few such re-reads and many bytes in flight.
//   * Tile. All T rows (32, 64 or 128) by BN weight rows and one K range; 64-deep K steps of
//     both operands stream through a ring that fills the LDS (direct-to-LDS loads of whole
//     128-byte lines, XOR-swizzled, one barrier per step). Eight waves: two groups of four
//     take the two 32-deep halves of a step, so a quarter tile per wave and 9 LDS reads per
//     20 v_mfma_f32_16x16x32 at 128 x 160.
//   * Split. Layers of many columns take BN = 160: 2 x 18944 columns are 237 tiles for 256
//     compute units, 152064 are 951. Smaller ones take BN = 64 and are cut over K until the
//     compute units have a workgroup each; the parts meet as fp32 partials (device-coherent
//     stores, one arrival counter per tile), which the last workgroup to arrive adds in
//     range order, so the result does not depend on which that was. Layers of 129 to 256
//     tiles are one round that leaves up to half of the compute units idle (a K range of a
//     tile each would be two rounds); utils/linear_layers.py leaves those to the library
//     where that is faster.
// The tile is handed to the epilogue as 8-column blocks of its two halves (columns c and
// c + BN / 2 of one row), which makes a gate / up pair or a RoPE pair one work item.
//
// Measured (cold weights, graph of calls, us at T = 8 / 64 / 128, library GEMMs beside):
//   18944 x 2 x 3584 gated    44 / 48 / 57      127 / 71 / 79 (two GEMMs and the product)
//   3584 x 18944              28 / 35 / 42      49 / 91 / 99
//   3584 x 3584               10.0 / 12.4 / 16.3    12.0 / 13.7 / 22.5
//   152064 x 3584             171 / 206 / 240   233 / 205 / 238
// that is 6.2-6.4 TB/s of weights at 8 rows and 4.5-4.8 at 128 on the large layers. Tried and
// not kept: both operands straight into MFMA registers without LDS (16 rows x 64 bytes per
// load: 403 us for the last layer at 128 rows), separate rings and loader waves for the
// operands, operand reads a step ahead of the products, K ranges started at different steps
// per workgroup, padded token rows (all within 3 %), BN = 96 or 128 for the smaller layers
// (3584 x 3584 19-22 us at 128 rows).
#pragma once

#include "fdllm_common.h"

namespace fdllm {

constexpr int kSkinnyMaxRows = 128;
constexpr int kSkinnyCounterBytes = 64 * 1024;  // arrival counters (int32, zero between calls), one per tile
constexpr int kSkinnyWgs = 256;                 // one workgroup per compute unit

struct SkinnyArgs {
  const uint16_t* x;
  int x_bytes;     // from row 0's first element to row T - 1's last
  int x_stride_b;  // bytes between rows
  int w_stride_b;  // bytes between weight rows (2 K)
  int T;
  int tiles;
  int ku;      // 64-deep K steps
  int splits;  // K ranges per tile
  int* cnt;
  uint8_t* part;
};

inline int skinny_bm(int T) { return T <= 32 ? 32 : T <= 64 ? 64 : 128; }

// K ranges per tile: as many as give each compute unit a workgroup, at least four steps
// each; one without a workspace for their sums or past its counters.
inline void skinny_plan(SkinnyArgs& a, bool workspace) {
  a.splits = 1;
  if (!workspace || a.tiles > kSkinnyWgs / 2) return;
  const int most = a.ku / 4 > 1 ? a.ku / 4 : 1;
  const int s = kSkinnyWgs / a.tiles;
  a.splits = s < most ? s : most;
}

inline size_t skinny_workspace(const SkinnyArgs& a, int bn) {
  if (a.splits == 1) return 0;
  return kSkinnyCounterBytes + static_cast<size_t>(a.tiles) * a.splits * (skinny_bm(a.T) * bn * 4);
}

template <bool F16>
__device__ __forceinline__ f32x4 skinny_mfma(const u32x4& a, const u32x4& b, const f32x4& c) {
  if constexpr (F16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
  }
}

// Weight rows of one tile: the two halves' first rows and the bytes that exist from there.
struct SkinnyRows {
  const uint16_t* w0;
  const uint16_t* w1;
  int bytes0, bytes1;
};

// Epi: rows<BN>(tile) -> SkinnyRows, and store<BN>(tile, m, block, v[4]) with the sums of
// columns 8 block + (0..7) (v[0], v[1]) and BN / 2 + 8 block + (0..7) of row m < T.
template <bool F16, int BM, int BN, int NS, typename Epi>
__global__ __launch_bounds__(512, 2) void skinny_gemm_kernel(const SkinnyArgs a, const Epi epi) {
  constexpr int NW = 8;
  constexpr int SLOT = (BM + BN) * 128;    // token rows, then weight rows, of one K step
  constexpr int LOADS = (BM + BN) / 8;     // 1 KB (eight rows) each, dealt to the waves in turn
  constexpr int MINE = LOADS / NW;         // per wave, one more for the first EXTRA waves
  constexpr int EXTRA = LOADS % NW;
  constexpr int TM = BM / 32, TN = BN / 32;  // 16-row MFMA tiles of a wave's quarter
  constexpr int LS = BN + 4;               // row stride of the summed tile (floats): 16 rows, 16 bank groups
  constexpr int NB = BN / 16;              // 8-column blocks per half row
  constexpr int ITEMS = BM * NB;
  constexpr int PART = BM * BN * 4;        // bytes of a partial tile
  constexpr int kDev = 16;                 // sc1: coherent at device scope
  static_assert(NS * SLOT <= 159 * 1024 && BM * LS * 4 <= NS * SLOT && NS >= 3, "LDS");
  static_assert(BN % 32 == 0 && BM % 32 == 0, "tile");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[NS * SLOT];
  __shared__ int s_last;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15;
  const int g = lane >> 4;
  const int tile = static_cast<int>(blockIdx.x) / a.splits;
  const int split = static_cast<int>(blockIdx.x) - tile * a.splits;
  const int k0 = a.ku * split / a.splits;
  const int nk = a.ku * (split + 1) / a.splits - k0;

  const SkinnyRows rows = epi.template rows<BN>(tile);
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
  const i32x4 xsrd = make_srd(a.x, a.x_bytes);  // token rows past the end read as zero
  const i32x4 wsrd0 = make_srd(rows.w0, rows.bytes0);
  const i32x4 wsrd1 = make_srd(rows.w1, rows.bytes1);
  // load q fills tile rows 8 q .. 8 q + 7: lane -> row + lane / 8, LDS chunk lane % 8, which
  // holds source chunk (lane % 8) ^ ((row >> 1) & 7): the 16 rows of an operand read then hit
  // 16 distinct 16-byte bank groups
  constexpr int LW = MINE + (EXTRA > 0 ? 1 : 0);
  int off[LW];
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int row = 8 * (wave + NW * i) + (lane >> 3);
    const int chunk = ((lane & 7) ^ ((row >> 1) & 7)) * 16 + k0 * 128;
    const int wr = row - BM < BN / 2 ? row - BM : row - BM - BN / 2;
    off[i] = chunk + (row < BM ? row * a.x_stride_b : wr * a.w_stride_b);
  }
  auto issue = [&](int st, int slot) __attribute__((always_inline)) {
    const uint32_t dst = lds0 + slot * SLOT + wave * 1024;
#pragma unroll
    for (int i = 0; i < LW; ++i) {
      if (i == MINE && wave >= EXTRA) break;  // uniform over the wave
      const int row = 8 * (wave + NW * i);
      const bool token = row < BM, low = row < BM + BN / 2;
      i32x4 srd;
#pragma unroll
      for (int c = 0; c < 4; ++c) srd[c] = token ? xsrd[c] : (low ? wsrd0[c] : wsrd1[c]);
      if (st >= nk) srd[2] = 0;  // past the range: zeros, no memory traffic
      if (token) lds_dma16<false>(srd, off[i] + st * 128, dst + NW * 1024 * i);
      else lds_dma16<true>(srd, off[i] + st * 128, dst + NW * 1024 * i);  // weights are read once
    }
  };

  // waves: two groups of four take the two 32-deep halves of each step; within a group a
  // quarter of the tile each
  const int kg = wave >> 2;
  const int wm = wave & 1, wn = (wave >> 1) & 1;
  f32x4 acc[TM][TN];
#pragma unroll
  for (int m = 0; m < TM; ++m)
#pragma unroll
    for (int n = 0; n < TN; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int chunk = 4 * kg + g;
  const int swz = (chunk ^ ((l16 >> 1) & 7)) * 16;  // tile rows differ from l16 by multiples of 16
  const int xat = (wm * (BM / 2) + l16) * 128 + swz;
  const int wat = (BM + wn * (BN / 2) + l16) * 128 + swz;
  auto compute = [&](int slot) __attribute__((always_inline)) {
    const uint8_t* sl = lds + slot * SLOT;
    u32x4 xv[TM], wv[TN];
#pragma unroll
    for (int n = 0; n < TN; ++n) wv[n] = *reinterpret_cast<const u32x4*>(sl + wat + n * 2048);
#pragma unroll
    for (int m = 0; m < TM; ++m) xv[m] = *reinterpret_cast<const u32x4*>(sl + xat + m * 2048);
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int n = 0; n < TN; ++n) acc[m][n] = skinny_mfma<F16>(wv[n], xv[m], acc[m][n]);
  };

  // step j in slot j % NS; step j + NS - 1 is issued into the slot step j - 1 read, after the
  // barrier that ends that step. Every step issues its loads (zero-size past the end), so
  // each count wait is exact.
#pragma unroll
  for (int st = 0; st < NS - 1; ++st) issue(st, st);
  int cur = 0;
  for (int j = 0; j < nk; ++j) {
    if (EXTRA > 0 && wave < EXTRA) wait_vmcnt<(NS - 2) * (MINE + 1)>();
    else wait_vmcnt<(NS - 2) * MINE>();
    lds_barrier();
    issue(j + NS - 1, cur == 0 ? NS - 1 : cur - 1);
    compute(cur);
    cur = cur == NS - 1 ? 0 : cur + 1;
  }
  wait_vmcnt<0>();  // no load may land in LDS after this point
  lds_barrier();

  // ---- the two K halves meet in LDS, rows m, columns n = 16 .. + 4 g + (0..3)
  float* red = reinterpret_cast<float*>(lds);
  float* mine = red + (wm * (BM / 2) + l16) * LS + wn * (BN / 2) + 4 * g;
  if (kg == 1) {
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int n = 0; n < TN; ++n) *reinterpret_cast<f32x4*>(mine + m * 16 * LS + n * 16) = acc[m][n];
  }
  lds_barrier();
  if (kg == 0) {
#pragma unroll
    for (int m = 0; m < TM; ++m)
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        f32x4* p = reinterpret_cast<f32x4*>(mine + m * 16 * LS + n * 16);
        *p = acc[m][n] + *p;
      }
  }
  lds_barrier();
  const auto pr = __builtin_amdgcn_make_buffer_rsrc(
      a.part + static_cast<int64_t>(tile) * a.splits * PART, 0, a.splits * PART, kBufferFlags);
  for (int it = tid; it < ITEMS; it += 64 * NW) {
    const int m = it / NB;
    const int blk = it - m * NB;
    if (m >= a.T) break;  // items are row-major
    f32x4 v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      v[j] = *reinterpret_cast<const f32x4*>(red + m * LS + (j >> 1) * (BN / 2) + blk * 8 + (j & 1) * 4);
    if (a.splits == 1) {
      epi.template store<BN>(tile, m, blk, v);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v[j]), pr,
                                               split * PART + (j * ITEMS + it) * 16, 0, kDev);
    }
  }
  if (a.splits == 1) return;
  // the stores are acknowledged before the arrival is counted; the last workgroup reads them
  // back with device-coherent loads and adds them in range order, whichever came last
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (tid == 0)
    s_last = __hip_atomic_fetch_add(&a.cnt[tile], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.splits - 1;
  __syncthreads();
  if (!s_last) return;
  for (int it = tid; it < ITEMS; it += 64 * NW) {
    const int m = it / NB;
    if (m >= a.T) break;
    f32x4 v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int GS = 4;  // partials per round trip
    for (int s0 = 0; s0 < a.splits; s0 += GS) {
      f32x4 p[GS][4];
#pragma unroll
      for (int s = 0; s < GS; ++s)  // past the last: outside the descriptor, zero
#pragma unroll
        for (int j = 0; j < 4; ++j)
          p[s][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                  pr, (s0 + s) * PART + (j * ITEMS + it) * 16, 0, kDev));
#pragma unroll
      for (int s = 0; s < GS; ++s)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] += p[s][j];
    }
    epi.template store<BN>(tile, m, it - m * NB, v);
  }
  if (tid == 0) __hip_atomic_store(&a.cnt[tile], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // next call
}

// LDS ring slots of a tile: as many as fit, at most twelve.
constexpr int skinny_slots(int bm, int bn) {
  const int n = (159 * 1024) / ((bm + bn) * 128);
  return n < 12 ? n : 12;
}

template <bool F16, int BN, typename Epi>
void skinny_launch(const SkinnyArgs& a, const Epi& epi, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(a.tiles * a.splits));
  switch (skinny_bm(a.T)) {
    case 32: skinny_gemm_kernel<F16, 32, BN, skinny_slots(32, BN), Epi><<<grid, dim3(512), 0, s>>>(a, epi); break;
    case 64: skinny_gemm_kernel<F16, 64, BN, skinny_slots(64, BN), Epi><<<grid, dim3(512), 0, s>>>(a, epi); break;
    default: skinny_gemm_kernel<F16, 128, BN, skinny_slots(128, BN), Epi><<<grid, dim3(512), 0, s>>>(a, epi); break;
  }
}

}  // namespace fdllm

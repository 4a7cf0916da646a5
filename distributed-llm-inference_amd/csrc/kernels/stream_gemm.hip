// Weight-streaming GEMM for 17 … 256 activation rows, dense and grouped over experts:  C[rows, n] = A[rows, :] · W[n, :]ᵀ (bf16).
//
// At these row counts a projection is still a stream of W through the chip (a decode batch of 96: 235 MB of gate/up weights against 0.8 MB
// of activations), but sixteen-column products (skinny_gemm.hip) would re-read W per 16 rows and the 256² tile (gemm256.hip)
// multiplies mostly padding.  What decides is bytes of W in flight per compute unit: HBM needs ≈ 25 GB/s · 1 µs = 25 KB of them.
//   * A workgroup owns 128 weight rows × BM activation rows (BM = 32, 64, 96, 128: the smallest that holds the rows) and walks K in steps of
//     64; a step is 16 KB of W and BM · 128 bytes of A, both by LDS-DMA into a ring of S stages, S − 1 of them in flight.  BM = 32 / 64
//     run as two workgroups per compute unit (80 / 72 KB of LDS each), BM = 96 / 128 as one (140 / 128 KB).
//   * Every column block starts its walk at another step and wraps around.  In lockstep all workgroups read the same few hundred bytes
//     of rows that lie a power of two apart, i.e. from few HBM channels: gate/up of width 4096 at 17 rows 48.3 → 40.5 µs, at 96 51.5 → 47.
//   * A wave is held for ≈ 75 cycles by every LDS-DMA instruction it issues, so four waves do nothing else and the others only read
//     fragments and multiply.
//   * One barrier per step: it says that stage t has landed (the fetching waves waited for their shares with a counted vmcnt) and
//     that stage t − 1 is consumed, so its slot may be refilled at once.
//   * v_mfma_f32_16x16x32_bf16 with W as the A operand: a wave owns 64 weight rows × min(BM, 64) activation rows for HALF of every
//     step's K.  LDS reads bound the step at BM = 128 (all eight waves together read each operand several times): 64 × 64 tiles read
//     64 KB a step, 32 × 64 tiles over the whole step's K 96 KB.  The two halves of a tile meet in LDS at the end.  A lane holds four
//     consecutive output columns of a row (8-byte stores); SwiGLU pairs a wave's first 32 weight rows (gate) with the other 32 (up).
//   * LDS image and bank swizzle as in gemm256.hip: 128-byte rows, slot p of row r holds 16-byte chunk p ^ (r & 7), applied on the
//     source address.
//   * Few column blocks (a down projection has 32) cut K into slices: fp32 slabs, added in fixed order by the reduce pass.
// Weights that no other workgroup reads (one row tile) are fetched with the streaming policy, like a decode step's: 8 experts of 9 rows
// 512 → 460 µs a Mixtral layer (128 × 128 tiles: 558).
// Measured (hipGraph, weights of several layers in turn; library GEMM, with its activation pass for gate/up, in brackets), µs:
//   gate/up 28672 × 4096   M = 17 43.5 (53.7)   64 47.4 (52.9)   96 49.6 (54.0)   128 53.2 (57.0)     36 at 6.5 TB/s
//   down 4096 × 14336      M = 17 25.0 (27.7)   64 29.6 (39.4)   96 33.4 (63.2)   128 37.7 (75.4)     18
//   LM head 128256 × 4096  M = 17 163 (193)     64 184 (211)     96 203 (228)     128 218 (234)      162
#include "common.h"
#include "kernels.h"

namespace dli {

namespace sgemm {

constexpr int BN = 128, BK = 64;
constexpr int W_BYTES = BN * BK * 2;

enum { PLAIN = 0, PLAIN_SLAB = 1, SWIGLU = 2, SWIGLU_SLAB = 3, SCATTER = 4, SCATTER_SLAB = 5 };
constexpr bool paired(int epi) { return epi == SWIGLU || epi == SWIGLU_SLAB; }

constexpr int FETCHERS = 4;                                  // waves that only issue LDS-DMA
constexpr int workers(int bm) { return bm > 64 ? 8 : 4; }
constexpr int threads(int bm) { return (workers(bm) + FETCHERS) * 64; }

__device__ __forceinline__ int lds_off(int r, int c) { return r * 128 + ((c ^ (r & 7)) << 4); }

using gptr_t = const __attribute__((address_space(1))) void*;
using lptr_t = __attribute__((address_space(3))) void*;

template <int BM, int S, int EPI, bool GROUPED, bool NT>
__global__ __launch_bounds__(threads(BM), BM > 64 ? 3 : 4) void stream_gemm_kernel(
    const uint16_t* __restrict__ A, int64_t a_stride, const uint16_t* __restrict__ W, int64_t w_expert_stride,
    const int* __restrict__ sorted_ids, const int* __restrict__ tile_expert, const int* __restrict__ meta,
    const float* __restrict__ topk_w, int top_k, void* __restrict__ out_, int64_t out_stride, int M, int K, int N_half,
    int n_col_blocks, int k_splits, int64_t slab_elems, float act_limit) {
  constexpr int XB = BM > 64 ? BM / 32 : BM / 16;                // 16-row activation blocks of a wave
  constexpr int STAGE = W_BYTES + BM * BK * 2;
  constexpr int WI = W_BYTES / 1024 / FETCHERS, XI = BM * BK * 2 / 1024 / FETCHERS;   // DMA instructions of a fetching wave per stage
  static_assert(XI >= 1 && XI * 1024 * FETCHERS == BM * BK * 2, "every fetching wave moves whole 1 KiB pieces");
  extern __shared__ __attribute__((aligned(1024))) char lds[];

  // block → (K slice, column block, row tile), row tile fastest: tiles that share weights run next to each other.  XCD x takes the
  // x-th eighth of that order, so its L2 holds the activations of one K slice.
  const int n_tiles = GROUPED ? meta[0] : (M + BM - 1) / BM;
  const int total = n_tiles * n_col_blocks * k_splits;
  const int per_xcd = (total + 7) >> 3;
  const int in_xcd = blockIdx.x >> 3;
  const int lin = (blockIdx.x & 7) * per_xcd + in_xcd;
  if (in_xcd >= per_xcd || lin >= total) return;
  const int tile = lin % n_tiles, cv = lin / n_tiles;
  const int split = cv / n_col_blocks, col_block = cv - split * n_col_blocks;
  const int n0 = col_block * (paired(EPI) ? BN / 2 : BN);
  const int expert = GROUPED ? tile_expert[tile] : 0;
  const uint16_t* We = W + expert * w_expert_stride;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kh = wave & 1, pair = wave >> 1;                 // half of the step's K, wave tile
  const int wn = pair & 1, wm = pair >> 1;
  const int col = lane & 15, g = lane >> 4;

  const int nk_total = K / BK;
  const int kt0 = (int)((int64_t)nk_total * split / k_splits);
  const int nk = (int)((int64_t)nk_total * (split + 1) / k_splits) - kt0;
  f32x4 acc[4][XB];

  if (wave >= workers(BM)) {
    // LDS-DMA: piece = 8 rows of 128 bytes in lane order; fetching wave f moves pieces f, f + FETCHERS, …
    const int f = wave - workers(BM);
    const char* w_src[WI];
    const char* x_src[XI];
#pragma unroll
    for (int i = 0; i < WI; ++i) {
      const int r = (f + i * FETCHERS) * 8 + (lane >> 3), c = (lane & 7) ^ (r & 7);
      const int row = paired(EPI) ? ((r & 32) ? N_half : 0) + n0 + (r >> 6) * 32 + (r & 31) : n0 + r;
      w_src[i] = reinterpret_cast<const char*>(We + (int64_t)row * K + kt0 * BK + c * 8);
    }
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int r = (f + i * FETCHERS) * 8 + (lane >> 3), c = (lane & 7) ^ (r & 7);
      int64_t row = (int64_t)tile * BM + r;
      if (GROUPED && paired(EPI)) {
        const int sid = sorted_ids[row];
        row = sid >= 0 ? sid / top_k : 0;                    // padding rows read token 0 (discarded later)
      } else if (!GROUPED) {
        row = min(row, (int64_t)M - 1);                      // rows past M repeat the last one (never stored)
      }
      x_src[i] = reinterpret_cast<const char*>(A + row * a_stride + kt0 * BK + c * 8);
    }
    const int rot = (col_block * 7 + expert * 11) % nk;
    auto stage = [&](int t, int slot) {
      char* dst = lds + slot * STAGE + f * 1024;
      const int turned = t + rot;
      const int64_t k = (int64_t)(turned >= nk ? turned - nk : turned) * (BK * 2);
#pragma unroll
      for (int i = 0; i < WI; ++i)
        __builtin_amdgcn_global_load_lds((gptr_t)(w_src[i] + k), (lptr_t)(dst + i * (FETCHERS * 1024)), 16, 0, NT ? 2 : 0);
#pragma unroll
      for (int i = 0; i < XI; ++i)
        __builtin_amdgcn_global_load_lds((gptr_t)(x_src[i] + k), (lptr_t)(dst + W_BYTES + i * (FETCHERS * 1024)), 16, 0, 0);
    };
#pragma unroll
    for (int t = 0; t < S - 1; ++t)
      if (t < nk) stage(t, t);
    int fill = S - 1;
    for (int t = 0; t < nk; ++t) {
      // stage t has landed once at most the S − 2 younger ones are in flight; the last steps have fewer and drain
      if (t + S - 1 <= nk) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * (WI + XI)) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (t + S - 1 < nk) stage(t + S - 1, fill);
      fill = fill == S - 1 ? 0 : fill + 1;
    }
  } else {
#pragma unroll
    for (int n = 0; n < 4; ++n)
#pragma unroll
      for (int m = 0; m < XB; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    int slot = 0;
    for (int t = 0; t < nk; ++t) {
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      const char* wb = lds + slot * STAGE;
      const char* xb = wb + W_BYTES;
      bf16x8 fw[4], fx[XB];
#pragma unroll
      for (int n = 0; n < 4; ++n) fw[n] = *reinterpret_cast<const bf16x8*>(wb + lds_off(wn * 64 + n * 16 + col, kh * 4 + g));
#pragma unroll
      for (int m = 0; m < XB; ++m) fx[m] = *reinterpret_cast<const bf16x8*>(xb + lds_off(wm * (XB * 16) + m * 16 + col, kh * 4 + g));
#pragma unroll
      for (int m = 0; m < XB; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n) acc[n][m] = mfma16(fw[n], fx[m], acc[n][m]);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // my fragments are in registers before I pass the next barrier
      __builtin_amdgcn_sched_barrier(0);
      slot = slot == S - 1 ? 0 : slot + 1;
    }
  }

  // The two waves of a tile swap halves: kh = 0 finishes weight blocks 0 and 2, kh = 1 blocks 1 and 3 (a SwiGLU pair stays together).
  __syncthreads();
  f32x4* swap = reinterpret_cast<f32x4*>(lds);               // [pair][to wave kh][2][XB][64]
  if (wave < workers(BM)) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int m = 0; m < XB; ++m) swap[(((pair * 2 + (1 - kh)) * 2 + j) * XB + m) * 64 + lane] = kh ? acc[2 * j][m] : acc[2 * j + 1][m];
  }
  __syncthreads();
  if (wave >= workers(BM)) return;
  f32x4 sum[2][XB];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int m = 0; m < XB; ++m)
      sum[j][m] = (kh ? acc[2 * j + 1][m] : acc[2 * j][m]) + swap[(((pair * 2 + kh) * 2 + j) * XB + m) * 64 + lane];

  // sum[j][m][r]: activation row wm·16·XB + m·16 + col, weight row wn·64 + j·32 + kh·16 + 4g + r of the tile
  uint16_t* out = reinterpret_cast<uint16_t*>(out_);
  float* slab = reinterpret_cast<float*>(out_) + split * slab_elems;
#pragma unroll
  for (int m = 0; m < XB; ++m) {
    const int prow = tile * BM + wm * (XB * 16) + m * 16 + col;
    const int row = GROUPED ? ((EPI == SWIGLU) ? prow : sorted_ids[prow]) : (prow < M ? prow : -1);
    if (row < 0) continue;
    if constexpr (paired(EPI)) {
      const int64_t at = (int64_t)row * out_stride + n0 + wn * 32 + kh * 16 + 4 * g;
      if constexpr (EPI == SWIGLU_SLAB) {                    // raw sums: gate at column c, up at N_half + c
        *reinterpret_cast<f32x4*>(slab + at) = sum[0][m];
        *reinterpret_cast<f32x4*>(slab + at + N_half) = sum[1][m];
      } else {                                               // (grouped padding rows hold finite junk, never read back)
        bf16x4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = (short)f2bf(gated_act(sum[0][m][r], sum[1][m][r], act_limit));
        *reinterpret_cast<bf16x4*>(out + at) = o;
      }
    } else {
      const float w = GROUPED ? topk_w[row] : 1.f;
      const int64_t at = (int64_t)row * out_stride + n0 + wn * 64 + kh * 16 + 4 * g;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if constexpr (EPI == PLAIN_SLAB || EPI == SCATTER_SLAB) {
          f32x4 o;
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = sum[j][m][r] * w;
          *reinterpret_cast<f32x4*>(slab + at + j * 32) = o;
        } else {
          bf16x4 o;
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = (short)f2bf(sum[j][m][r] * w);
          *reinterpret_cast<bf16x4*>(out + at + j * 32) = o;
        }
      }
    }
  }
}

template <int BM, int EPI, bool GROUPED, bool NT>
void go(const void* A, int64_t a_stride, const void* W, int64_t w_expert_stride, const int* sorted_ids, const int* tile_expert,
        const int* meta, const float* topk_w, int top_k, void* out, int64_t out_stride, int M, int K, int N_half, int n_col_blocks,
        int max_tiles, int k_splits, int64_t slab_elems, float act_limit, hipStream_t stream) {
  constexpr int S = BM == 64 ? 3 : BM == 96 ? 5 : 4;
  constexpr int LDS = S * (W_BYTES + BM * BK * 2);
  auto kernel = stream_gemm_kernel<BM, S, EPI, GROUPED, NT>;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  (void)attr;                                                // (a refused attribute shows as a failed launch)
  hipLaunchKernelGGL(kernel, dim3((max_tiles * n_col_blocks * k_splits + 7) / 8 * 8), dim3(threads(BM)), LDS, stream,
                     (const uint16_t*)A, a_stride, (const uint16_t*)W, w_expert_stride, sorted_ids, tile_expert, meta, topk_w, top_k, out,
                     out_stride, M, K, N_half, n_col_blocks, k_splits, slab_elems, act_limit);
}

}  // namespace sgemm

// rows of W: N (swiglu: gate rows, then up rows; N_out = N / 2 output columns).  N % 128 == 0, K % 64 == 0, 16-byte aligned rows.
// k_splits > 1: `out` receives fp32 slabs [k_splits][M][N], to be added by launch_splitk_reduce.
void launch_stream_gemm(bool swiglu, const void* x, int64_t x_stride, const void* W, void* out, int64_t out_stride, int M, int K, int N,
                        int k_splits, hipStream_t stream) {
  using namespace sgemm;
  const int bm = M <= 32 ? 32 : M <= 64 ? 64 : M <= 96 ? 96 : 128, tiles = (M + bm - 1) / bm, cols = N / BN;
  const bool slab = k_splits > 1;
#define SG_GO3(BM_, EPI_, NT_)                                                                                                   \
  go<BM_, EPI_, false, NT_>(x, x_stride, W, 0, nullptr, nullptr, nullptr, nullptr, 1, out, slab ? (int64_t)N : out_stride, M, K, N / 2, cols, \
                            tiles, k_splits, (int64_t)M * N, 0.f, stream)
#define SG_GO2(BM_, NT_)                                                                                                         \
  {                                                                                                                              \
    if (swiglu) { if (slab) SG_GO3(BM_, SWIGLU_SLAB, NT_); else SG_GO3(BM_, SWIGLU, NT_); }                                      \
    else { if (slab) SG_GO3(BM_, PLAIN_SLAB, NT_); else SG_GO3(BM_, PLAIN, NT_); }                                               \
  }
  if (bm == 32) SG_GO2(32, true) else if (bm == 64) SG_GO2(64, true) else if (bm == 96) SG_GO2(96, true) else if (tiles == 1) SG_GO2(128, true) else SG_GO2(128, false)
#undef SG_GO2
#undef SG_GO3
}

// Contract of launch_grouped_gemm (moe.hip) for row tiles of 32 or 64 rows (moe_align padded the experts' rows to that).
// epilogue: 0 SwiGLU, 1 scatter, 2 scatter into fp32 slabs.
void launch_grouped_stream_gemm(int epilogue, int tile_rows, const void* A, int64_t a_stride, const void* W, int64_t w_expert_stride,
                                const int* sorted_ids, const int* tile_expert, const int* meta, const float* topk_w, int top_k, void* out,
                                int64_t out_stride, int K, int N_out, int max_tiles, int k_splits, int64_t slab_elems, hipStream_t stream,
                                float act_limit) {
  using namespace sgemm;
  if (max_tiles == 0) return;
  const int cols = (epilogue == 0 ? 2 * N_out : N_out) / BN;
#define SG_GO(BM_, EPI_)                                                                                                         \
  go<BM_, EPI_, true, true>(A, a_stride, W, w_expert_stride, sorted_ids, tile_expert, meta, topk_w, top_k, out, out_stride, 0, K, N_out, cols, \
                             max_tiles, k_splits, slab_elems, act_limit, stream)
#define SG_EPI(BM_)                                                                                                              \
  { if (epilogue == 0) SG_GO(BM_, SWIGLU); else if (epilogue == 1) SG_GO(BM_, SCATTER); else SG_GO(BM_, SCATTER_SLAB); }
  if (tile_rows == 32) SG_EPI(32) else SG_EPI(64)
#undef SG_EPI
#undef SG_GO
}

}  // namespace dli

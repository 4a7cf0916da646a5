// K8: Mixtral-style mixture-of-experts on gfx950: routing, token alignment, grouped GEMM
// on v_mfma_f32_16x16x32_bf16 with fused epilogues, and the weighted un-permute.
//
//   moe_route      softmax over all experts → top-k → renormalise               [T,E] → ids/weights [T,k]
//   moe_align      bucket the (token, slot) pairs of the *local* experts; every expert's segment is
//                  padded to a multiple of the GEMM row tile; all sizes stay on the device, so the
//                  whole block is hipGraph-capturable (grids are launched at their worst-case size and
//                  surplus tiles exit on a device-side count)
//   grouped_gemm   C[rows of expert e] = A[rows] · W[e]ᵀ, 128×128×64 tiles, 4 waves (2×2) of 64×64,
//                  A rows gathered by index straight into the (XOR-swizzled) LDS image, register
//                  prefetch of the next K tile under the MFMAs.
//                  EPI_SWIGLU: the 128 B-rows of a tile are 2×(32 gate + 32 up) weight rows, so each
//                  wave owns matching gate/up columns and applies silu(g)·u in registers — the [rows, 2I]
//                  intermediate never exists.
//                  EPI_SCATTER: rows are scaled by their routing weight and stored at (token·k + slot).
//   moe_sum        out[t] = Σ_slots y[t·k + slot] over the slots served by local experts (no atomics:
//                  bitwise reproducible; non-local slots are summed in by the caller's all-reduce).
#include <algorithm>

#include "common.h"
#include "kernels.h"

namespace dli {

constexpr int BM = 128, BN = 128, BK = 64;
constexpr int MOE_MAX_E = 64;

// ------------------------------------------------------------------------------------------ routing
// One wave per token, one lane per expert (E ≤ 64): softmax numerators in registers, K rounds of a wave-wide
// arg-max (ties → lowest expert id, like torch.topk on the reference path), lane k keeps the k-th pick.
__global__ __launch_bounds__(256) void moe_route_kernel(const uint16_t* __restrict__ logits, int T, int E, int K,
                                                        int* __restrict__ ids, float* __restrict__ weights) {
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (t >= T) return;                                   // whole wave
  const float v = lane < E ? bf2f(logits[(int64_t)t * E + lane]) : -3.0e38f;
  const float mx = wave_max(v);
  float p = lane < E ? __expf(v - mx) : -1.f;           // the softmax denominator cancels in the renormalisation
  float picked = 0.f, my_w = 0.f;
  int my_id = 0;
  for (int k = 0; k < K; ++k) {
    float bv = p;
    int bi = lane;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(bv, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
    }
    if (lane == k) { my_id = bi; my_w = bv; }
    picked += bv;
    if (lane == bi) p = -2.f;
  }
  if (lane < K) {
    ids[t * K + lane] = my_id;
    weights[t * K + lane] = my_w / picked;              // renormalise over the chosen experts
  }
}

// ------------------------------------------------------------------------------------------ alignment
// Down projection on 256 × 256 tiles, one workgroup a compute unit: whole rounds of 256 tiles, and what is left over (all of it, if that is less than a
// round) in K-slices, so that a last round of few tiles does not leave most of the chip idle.  Only the device knows the number of tiles.
// → {tiles in whole rounds, slices of each of the others}.  µs, measured at K = 14336, 4096 columns: a K-step of a tile 1.7 (`full`: a tile's share of that on
// average, tiles of up to 128 rows take 0.58), a workgroup's start and end 6, a slice's 256 KB of sums written and read 0.1.  Slices that are more than a round end
// half a slice apart.  Mixtral's layer, µs, slices by the largest possible number of tiles and fp32 rows for all of them / this: 300 tokens 636 / 592, 777 731 /
// 680, 2048 1403 / 1343; whole rounds only / this: 4096 2415 / 2321 (tiles for a round and a quarter, say, take that and not two).
// (The times are one layer's; at 63 steps of 13 layers, 512 to 8192 columns, K 1024 to 28672, 2 to 16 experts, 0.93 of the former's on average, at most 1.02.)
constexpr int CUT_CUS = 256, CUT_MAX_SLICES = 8, CUT_MAX_TILES = 512;
int grouped_cut_slabs(int blocks) { return std::min(CUT_MAX_TILES, CUT_MAX_SLICES * std::min(blocks, CUT_CUS - 1)); }
__host__ __device__ inline int2 cut_plan(int blocks, int nk, float full) {
  const int rest = blocks % CUT_CUS;
  int best = 1;
  const float top = full < 0.59f ? full : 1.f;              // the longest of the tiles
  float best_us = top * 1.7f * nk + 6.f;
  for (int k = 2; k <= CUT_MAX_SLICES && 4 * k <= nk && rest * k <= CUT_MAX_TILES; ++k) {
    const int waves = (rest * k + CUT_CUS - 1) / CUT_CUS;
    const float rounds = waves == 1 ? top / k : fminf(waves * top / k, rest * full / CUT_CUS + 0.5f * top / k);
    const float us = rounds * 1.7f * nk + waves * 6.f + 0.1f * rest * k * full;
    if (us < best_us) {
      best_us = us;
      best = k;
    }
  }
  return rest > 0 && best > 1 ? make_int2(blocks - rest, best) : make_int2(0, 1);
}

// meta[0] = number of row tiles, meta[1] = padded row count; n_col_blocks > 0: meta[2], meta[3] = cut_plan of that many column blocks and nk
// K-steps, pos[i] = row of pair i in the sorted order
// A wave has a run of neighbouring pairs: it counts them, learns where its share of each expert's rows begins, and places them, in the order of the pair
// index and without atomics: every launch produces the same sorted_ids, so WHICH rows share an expert's last tile never
// changes from launch to launch and a step replays bit-identically whatever the tile variants do with a partly filled tile.  Two barriers in all.  Bound by
// the instructions that one compute unit issues: the pairs of a lane's expert among 64 come from a ballot for every bit of its number, once, whatever the
// number of experts (8192 pairs of 8 experts, µs: an LDS atomic for every pair and a ballot for every expert 21, two of those 18 to 21, this 10).
__global__ __launch_bounds__(1024) void moe_align_kernel(const int* __restrict__ ids, int n, int expert_offset, int E_local,
                                                         int* __restrict__ sorted_ids, int* __restrict__ tile_expert,
                                                         int* __restrict__ meta, int capacity_rows, int tile_rows, int n_col_blocks, int nk,
                                                         int* __restrict__ pos_of) {
  static_assert(MOE_MAX_E == 64, "a lane for every expert, six bits of its number");
  constexpr int HELD = 8;                                  // 64 pairs each: runs of up to 512 pairs are looked at once
  const int BM = tile_rows;                               // row tile of the GEMM that consumes the alignment (32, 64, 128 or 256)
  __shared__ int wave_cnt[16][MOE_MAX_E], off[MOE_MAX_E + 1], cnt[MOE_MAX_E];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n_waves = blockDim.x >> 6;
  const int run = ((n + n_waves - 1) / n_waves + 63) & ~63, begin = wave * run, end = min(n, begin + run);
  const int bits = 32 - __clz(max(E_local - 1, 1));
  // expert (-1: none of these) of pair at + 64 j + lane, how many before it among the 64 have the same one, and how many in all
  int held[HELD], rank[HELD], same_all[HELD];
  auto look = [&](int at) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < HELD; ++j) held[j] = at + 64 * j + lane < end ? ids[at + 64 * j + lane] : -1;
#pragma unroll
    for (int j = 0; j < HELD; ++j) {
      if (at + 64 * j >= end) break;
      const int e = held[j] - expert_offset;
      const bool here = held[j] >= 0 && e >= 0 && e < E_local;
      const unsigned long long any = __ballot(here);
      uint32_t lo = (uint32_t)any, hi = (uint32_t)(any >> 32);
      for (int b = 0; b < bits; ++b) {
        const unsigned long long set = __ballot((e >> b) & 1);
        const uint32_t clear = ((e >> b) & 1) - 1;         // all ones where the lane's bit is 0
        lo &= (uint32_t)set ^ clear;
        hi &= (uint32_t)(set >> 32) ^ clear;
      }
      held[j] = here ? e : -1;
      rank[j] = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0));
      same_all[j] = __popc(lo) + __popc(hi);
    }
  };
  wave_cnt[wave][lane] = 0;                                // (a wave's row is its own until the barrier)
  for (int at = begin; at < end; at += 64 * HELD) {
    look(at);
#pragma unroll
    for (int j = 0; j < HELD; ++j) {
      wave_lds_order();                                    // the expert's last count may be another lane's
      if (at + 64 * j < end && held[j] >= 0 && rank[j] == 0) wave_cnt[wave][held[j]] += same_all[j];
    }
  }
  __syncthreads();
  if (wave == 0) {                                         // per expert: the waves' counts → places before them, the sum
    int c[16], sum = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) c[w] = w < n_waves ? wave_cnt[w][lane] : 0;
    int total = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) total += c[w];
    const int tiles = lane < E_local ? (total + BM - 1) / BM : 0;
    int before = tiles;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int up = __shfl_up(before, o, 64);
      if (lane >= o) before += up;
    }
    const int all = __builtin_amdgcn_readlane(before, 63);
    before -= tiles;
    cnt[lane] = total;
    off[lane] = before * BM;
    if (lane == 0) off[MOE_MAX_E] = all * BM;
    sum = before * BM;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      if (w < n_waves) wave_cnt[w][lane] = sum;            // the wave's first row of this expert
      sum += c[w];
    }
    for (int t = 0; t < tiles; ++t) tile_expert[before + t] = lane;
    const int half = __popcll(__ballot(tiles * BM - total >= BM / 2 && tiles > 0));
    if (lane == 0) {
      meta[0] = all;
      meta[1] = all * BM;
      if (n_col_blocks > 0) {
        const int2 plan = cut_plan(all * n_col_blocks, nk, 1.f - 0.42f * half / max(all, 1));
        meta[2] = plan.x;
        meta[3] = plan.y;
      }
    }
  }
  __syncthreads();
  // rows without a pair: the end of every expert's last tile, and what no tile has
  for (int e = wave; e < E_local; e += n_waves)
    for (int i = off[e] + cnt[e] + lane; i < (off[e] + cnt[e] + BM - 1) / BM * BM; i += 64) sorted_ids[i] = -1;
  for (int i = off[MOE_MAX_E] + threadIdx.x; i < capacity_rows; i += blockDim.x) sorted_ids[i] = -1;
  for (int at = begin; at < end; at += 64 * HELD) {
    if (run > 64 * HELD) look(at);
#pragma unroll
    for (int j = 0; j < HELD; ++j) {
      const int i = at + 64 * j + lane, e = held[j];       // (e < 0 from the run's end on)
      const int first = e >= 0 ? wave_cnt[wave][e] : 0, to = first + rank[j];
      wave_lds_order();                                    // all lanes have read before the first of an expert moves its place on …
      if (e >= 0 && rank[j] == 0) wave_cnt[wave][e] = first + same_all[j];
      wave_lds_order();                                    // … and the next pairs' lanes read after it
      if (e >= 0) {
        sorted_ids[to] = i;
        if (n_col_blocks > 0) pos_of[i] = to;
      }
    }
  }
}

// ------------------------------------------------------------------------------------------ grouped GEMM
enum { EPI_SWIGLU = 0, EPI_SCATTER = 1, EPI_SCATTER_SPLITK = 2, EPI_RELU2 = 3 };   // SPLITK: fp32 partial slabs, summed by moe_sum
// EPI_RELU2: rows gathered like EPI_SWIGLU, 128 plain output columns per tile, stored as relu(·)² (experts without a gate)

// byte offset of 16-byte chunk c (0..7) of row r inside a [128][64] bf16 LDS tile, XOR-swizzled so that
// the 16 rows a ds_read_b128 lane group touches fall on different bank groups
__device__ __forceinline__ int lds_off(int r, int c) { return r * 128 + ((c ^ (r & 7)) << 4); }

template <int EPI>
__global__ __launch_bounds__(256) void grouped_gemm_kernel(
    const uint16_t* __restrict__ A, int64_t a_stride,         // EPI_SWIGLU: x [T, K], rows gathered; EPI_SCATTER: act [P, K]
    const uint16_t* __restrict__ W, int64_t w_expert_stride,  // [E_local, N_total, K]
    const int* __restrict__ sorted_ids, const int* __restrict__ tile_expert, const int* __restrict__ meta,
    const float* __restrict__ topk_w, int top_k, void* __restrict__ out_, int64_t out_stride, int K, int N_half,
    int n_col_blocks, int k_splits, int64_t slab_elems, float act_limit) {
  uint16_t* out = reinterpret_cast<uint16_t*>(out_);
  constexpr int STAGE = 2 * BM * BK * 2;                     // A tile + B tile of one K-step
  __shared__ __attribute__((aligned(1024))) char lds[2 * STAGE];   // double-buffered, filled by LDS-DMA
  // ---- block → (row tile, column block), XCD-aware.  The hardware deals workgroups round-robin over the 8
  // XCDs (id % 8), each with a private 4 MB L2.  Work is cut into super-tiles of 8 row tiles × 8 column
  // blocks; XCD k runs super-tiles k, k+8, …, 64 consecutive workgroups each, so the blocks resident on
  // one XCD at a time share 8 A tiles and (row tiles being sorted by expert) 8–16 W tiles: each operand
  // K-slice is fetched into that L2 once and reused 8×, instead of every block streaming a private
  // 1 MB W tile from HBM (the round-robin default puts the 8 row tiles of an expert on 8 different XCDs).
  // With fewer than 8 row tiles (decode-sized batches) the super-tile narrows to 4/2/1 row tiles × 16/32/64
  // column blocks, so that the live blocks still spread over all XCDs.
  const int n_tiles = meta[0];
  const int gx_log = n_tiles >= 5 ? 3 : n_tiles >= 3 ? 2 : n_tiles >= 2 ? 1 : 0;
  const int gy_log = 6 - gx_log;
  const int j = blockIdx.x >> 3;
  const int super = (j >> 6) * 8 + (blockIdx.x & 7);
  const int n_virtual = n_col_blocks * k_splits;             // split-K slices are extra "columns" (slowest index)
  const int sy_count = (n_virtual + (1 << gy_log) - 1) >> gy_log;
  const int sx = super / sy_count, sy = super - sx * sy_count;
  const int tile = (sx << gx_log) + (j & ((1 << gx_log) - 1));
  const int col_virtual = (sy << gy_log) + ((j & 63) >> gx_log);
  if (tile >= n_tiles || col_virtual >= n_virtual) return;
  const int split = col_virtual / n_col_blocks;
  const int col_block = col_virtual - split * n_col_blocks;
  const int e = tile_expert[tile];
  const uint16_t* We = W + (int64_t)e * w_expert_stride;
  const int n0 = col_block * (EPI == EPI_SWIGLU ? BN / 2 : BN);   // SWIGLU: 64 output columns per tile
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int col = lane & 15, g = lane >> 4;

  // ---- staging: LDS-DMA (global_load_lds, 16 bytes per lane, no VGPRs, no ds_write).  DMA instruction i of wave w
  // fills the 1 KiB at (w + 4i)·1024 of a tile in lane order, i.e. lane → LDS chunk q = tid + 256 i: row q/8,
  // slot q%8.  The bank swizzle of lds_off is applied on the source side: slot p of row r receives global chunk
  // p ^ (r & 7).
  const uint16_t* a_src[4];
  const uint16_t* b_src[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int q = tid + 256 * i, r = q >> 3, c = (q & 7) ^ (r & 7);
    int64_t arow;
    if (EPI == EPI_SWIGLU || EPI == EPI_RELU2) {
      const int sid = sorted_ids[tile * BM + r];
      arow = sid >= 0 ? sid / top_k : 0;                     // padding rows read token 0 (discarded later)
    } else {
      arow = (int64_t)tile * BM + r;
    }
    a_src[i] = A + arow * a_stride + c * 8;
    int wrow;
    if (EPI == EPI_SWIGLU) {
      const int w_ = r >> 6, within = r & 63;                 // wave-column half, position inside it
      wrow = (within < 32 ? 0 : N_half) + n0 + w_ * 32 + (within & 31);
    } else {
      wrow = n0 + r;
    }
    b_src[i] = We + (int64_t)wrow * K + c * 8;
  }

  f32x4 acc[4][4];
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int n = 0; n < 4; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};

  // this block's K-steps: slice `split` of k_splits (contiguous, sizes differ by at most one step)
  const int nk_total = K / BK;
  const int kt0 = (int)((int64_t)nk_total * split / k_splits);
  const int nk = (int)((int64_t)nk_total * (split + 1) / k_splits);
  using gptr_t = const __attribute__((address_space(1))) void*;
  using lptr_t = __attribute__((address_space(3))) void*;
#define DLI_GG_STAGE(kt_, buf_)                                                                                   \
  {                                                                                                               \
    char* dst_ = lds + (buf_) * STAGE + wave * 1024;                  /* wave-uniform; + lane·16 by hardware */   \
    _Pragma("unroll") for (int i = 0; i < 4; ++i) {                                                               \
      __builtin_amdgcn_global_load_lds((gptr_t)(a_src[i] + (kt_) * BK), (lptr_t)(dst_ + i * 4096), 16, 0, 0);     \
      __builtin_amdgcn_global_load_lds((gptr_t)(b_src[i] + (kt_) * BK), (lptr_t)(dst_ + BM * BK * 2 + i * 4096), 16, 0, 0); \
    }                                                                                                             \
  }
  DLI_GG_STAGE(kt0, 0);
  for (int kt = kt0; kt < nk; ++kt) {
    const int buf = (kt - kt0) & 1;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // my share of K-step kt has landed …
    __syncthreads();                                           // … everyone's has, and everyone is done with kt-1
    if (kt + 1 < nk) DLI_GG_STAGE(kt + 1, buf ^ 1);            // next K-step streams in under the MFMAs
    const char* ldsA = lds + buf * STAGE;
    const char* ldsB = ldsA + BM * BK * 2;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8 fa[4], fb[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) fa[m] = *reinterpret_cast<const bf16x8*>(ldsA + lds_off(wm * 64 + m * 16 + col, ks * 4 + g));
#pragma unroll
      for (int n = 0; n < 4; ++n) fb[n] = *reinterpret_cast<const bf16x8*>(ldsB + lds_off(wn * 64 + n * 16 + col, ks * 4 + g));
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n) acc[m][n] = mfma16(fb[n], fa[m], acc[m][n]);
      // operands swapped on purpose: D[row = weight column n (4g+r)][col = token row m (lane&15)], i.e. each
      // lane holds 4 *consecutive output columns* of one token row → 8-byte row-contiguous stores
    }
  }

#undef DLI_GG_STAGE

  // ---- epilogue.  acc[m][n][r]: token row = wm*64 + m*16 + col, output column = wn*64 + n*16 + 4g + r
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int prow = tile * BM + wm * 64 + m * 16 + col;
    const int sid = sorted_ids[prow];
    if (EPI == EPI_SWIGLU) {
      // wave columns: n = 0,1 gate (32 cols), n = 2,3 the matching up columns
      uint16_t* dst = out + (int64_t)prow * out_stride + n0 + wn * 32 + 4 * g;
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        bf16x4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float gate = acc[m][n][r], up = acc[m][n + 2][r];
          o[r] = (short)f2bf(gated_act(gate, up, act_limit));
        }
        *reinterpret_cast<bf16x4*>(dst + n * 16) = o;           // padding rows hold finite junk, never read back
      }
    } else if (EPI == EPI_RELU2) {
      uint16_t* dst = out + (int64_t)prow * out_stride + n0 + wn * 64 + 4 * g;
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        bf16x4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float a = fmaxf(acc[m][n][r], 0.f);
          o[r] = (short)f2bf(a * a);
        }
        *reinterpret_cast<bf16x4*>(dst + n * 16) = o;
      }
    } else if (EPI == EPI_SCATTER_SPLITK) {
      if (sid >= 0) {
        const float w = topk_w[sid];
        float* dst = reinterpret_cast<float*>(out_) + split * slab_elems + (int64_t)sid * out_stride + n0 + wn * 64 + 4 * g;
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          f32x4 o;
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = acc[m][n][r] * w;
          *reinterpret_cast<f32x4*>(dst + n * 16) = o;
        }
      }
    } else if (sid >= 0) {
      const float w = topk_w[sid];
      uint16_t* dst = out + (int64_t)sid * out_stride + n0 + wn * 64 + 4 * g;
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        bf16x4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = (short)f2bf(acc[m][n][r] * w);
        *reinterpret_cast<bf16x4*>(dst + n * 16) = o;
      }
    }
  }
}

// ------------------------------------------------------------------------------------------ un-permute
// SLABS == 0: y is bf16 [T·k, H].  SLABS > 0 (runtime count in n_slabs): y is fp32 [n_slabs][T·k, H] split-K partials.
template <bool F32>
__global__ __launch_bounds__(256) void moe_sum_kernel(const void* __restrict__ y_, const int* __restrict__ ids,
                                                      int expert_offset, int E_local, int top_k, int H, int n_slabs,
                                                      int64_t slab_elems, uint16_t* __restrict__ out) {
  const int t = blockIdx.x;
  for (int v = threadIdx.x; v < H / 8; v += blockDim.x) {
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int s = 0; s < top_k; ++s) {
      const int e = ids[t * top_k + s] - expert_offset;
      if (e < 0 || e >= E_local) continue;
      const int64_t row = ((int64_t)t * top_k + s) * H + v * 8;
      if (F32) {
        const float* y = reinterpret_cast<const float*>(y_);
        for (int k = 0; k < n_slabs; ++k) {                 // fixed order: bitwise reproducible
          const f32x4 a = *reinterpret_cast<const f32x4*>(y + k * slab_elems + row);
          const f32x4 b = *reinterpret_cast<const f32x4*>(y + k * slab_elems + row + 4);
#pragma unroll
          for (int j = 0; j < 4; ++j) { acc[j] += a[j]; acc[4 + j] += b[j]; }
        }
      } else {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(reinterpret_cast<const uint16_t*>(y_) + row);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] += bf2f((uint16_t)a[j]);
      }
    }
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = (short)f2bf(acc[j]);
    *reinterpret_cast<bf16x8*>(out + (int64_t)t * H + v * 8) = o;
  }
}

// The same behind a down projection on 256 × 256 tiles: y bf16 or fp32 rows (F32) of the tiles in whole rounds; the sums of a cut tile (meta[2], meta[3]) are
// those of its slices, [slice][tile][256][256] fp32.
template <bool F32>
__global__ __launch_bounds__(256) void moe_sum_cut_kernel(const void* __restrict__ y_, const float* __restrict__ slabs, const int* __restrict__ pos_of,
                                                          const int* __restrict__ meta, const int* __restrict__ ids, int expert_offset, int E_local,
                                                          int top_k, int H, uint16_t* __restrict__ out) {
  const int t = blockIdx.x, n_tiles = meta[0], plain = meta[2], slices = meta[3], n_col = H >> 8, rest = n_tiles * n_col - plain;
  for (int v = threadIdx.x; v < H / 8; v += blockDim.x) {
    // this column block's tiles in the order in which the kernel deals them: groups of 8 column blocks, row tile, column block
    const int cb = v >> 5, first = cb & ~7, width = min(8, n_col - first), lin0 = first * n_tiles + cb - first - plain;
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int s = 0; s < top_k; ++s) {
      const int pair = t * top_k + s, e = ids[pair] - expert_offset;
      if (e < 0 || e >= E_local) continue;
      const int row = pos_of[pair], lin = lin0 + (row >> 8) * width;
      const bool cut = slices > 1 && lin >= 0;
      if (F32 || cut) {
        const float* y = cut ? slabs + (int64_t)lin * 65536 + (row & 255) * 256 + (v & 31) * 8 : reinterpret_cast<const float*>(y_) + (int64_t)pair * H + v * 8;
        for (int k = 0; k < (cut ? slices : 1); ++k, y += (int64_t)rest * 65536) {        // fixed order: bitwise reproducible
          const f32x4 a = *reinterpret_cast<const f32x4*>(y), b = *reinterpret_cast<const f32x4*>(y + 4);
#pragma unroll
          for (int j = 0; j < 4; ++j) { acc[j] += a[j]; acc[4 + j] += b[j]; }
        }
      } else {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(reinterpret_cast<const uint16_t*>(y_) + (int64_t)pair * H + v * 8);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] += bf2f((uint16_t)a[j]);
      }
    }
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = (short)f2bf(acc[j]);
    *reinterpret_cast<bf16x8*>(out + (int64_t)t * H + v * 8) = o;
  }
}

// ------------------------------------------------------------------------------------------ launchers
void launch_moe_route(const void* logits, int T, int E, int K, int* ids, float* weights, hipStream_t stream) {
  if (T == 0) return;
  hipLaunchKernelGGL(moe_route_kernel, dim3((T + 3) / 4), dim3(256), 0, stream, (const uint16_t*)logits, T, E, K, ids, weights);
}

void launch_moe_align(const int* ids, int n, int expert_offset, int E_local, int* sorted_ids, int* tile_expert, int* meta,
                      int capacity_rows, int tile_rows, hipStream_t stream, int n_col_blocks, int nk, int* pos_of) {
  hipLaunchKernelGGL(moe_align_kernel, dim3(1), dim3(1024), 0, stream, ids, n, expert_offset, E_local, sorted_ids, tile_expert,
                     meta, capacity_rows, tile_rows, n_col_blocks, nk, pos_of);
}

void launch_grouped_gemm(int epilogue, const void* A, int64_t a_stride, const void* W, int64_t w_expert_stride,
                         const int* sorted_ids, const int* tile_expert, const int* meta, const float* topk_w, int top_k,
                         void* out, int64_t out_stride, int K, int N_out, int max_tiles, int k_splits, int64_t slab_elems,
                         hipStream_t stream, float act_limit) {
  if (max_tiles == 0) return;
  const int n_col_blocks = N_out / (epilogue == EPI_SWIGLU ? BN / 2 : BN);
  const int n_virtual = n_col_blocks * k_splits;
  const int supers = (max_tiles + 7) / 8 * ((n_virtual + 7) / 8);
  dim3 grid((supers + 7) / 8 * 8 * 64);                                      // surplus blocks exit on meta[0]
#define DLI_GG(EPI)                                                                                                       \
  hipLaunchKernelGGL(grouped_gemm_kernel<EPI>, grid, dim3(256), 0, stream, (const uint16_t*)A, a_stride, (const uint16_t*)W, \
                     w_expert_stride, sorted_ids, tile_expert, meta, topk_w, top_k, out, out_stride, K, N_out, n_col_blocks, \
                     k_splits, slab_elems, act_limit)
  if (epilogue == EPI_SWIGLU) DLI_GG(EPI_SWIGLU);
  else if (epilogue == EPI_RELU2) DLI_GG(EPI_RELU2);
  else if (epilogue == EPI_SCATTER) DLI_GG(EPI_SCATTER);
  else DLI_GG(EPI_SCATTER_SPLITK);
#undef DLI_GG
}

void launch_moe_sum(const void* y, bool y_fp32, int n_slabs, int64_t slab_elems, const int* ids, int expert_offset, int E_local,
                    int top_k, int T, int H, void* out, hipStream_t stream) {
  if (T == 0) return;
  if (y_fp32)
    hipLaunchKernelGGL(moe_sum_kernel<true>, dim3(T), dim3(256), 0, stream, y, ids, expert_offset, E_local, top_k, H, n_slabs,
                       slab_elems, (uint16_t*)out);
  else
    hipLaunchKernelGGL(moe_sum_kernel<false>, dim3(T), dim3(256), 0, stream, y, ids, expert_offset, E_local, top_k, H, 1,
                       slab_elems, (uint16_t*)out);
}

void launch_moe_sum_cut(const void* y, bool y_fp32, const float* slabs, const int* pos_of, const int* meta, const int* ids, int expert_offset, int E_local,
                        int top_k, int T, int H, void* out, hipStream_t stream) {
  if (T == 0) return;
  hipLaunchKernelGGL((y_fp32 ? moe_sum_cut_kernel<true> : moe_sum_cut_kernel<false>), dim3(T), dim3(256), 0, stream, y, slabs, pos_of, meta, ids,
                     expert_offset, E_local, top_k, H, (uint16_t*)out);
}

}  // namespace dli

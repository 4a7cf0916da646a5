// K4 / K5: paged attention for gfx950 — single-query decode (split-KV) and chunked-prefill
// (varlen, causal, paged prefix) — on v_mfma_f32_16x16x32_bf16.
//
// Both kernels use the *transposed* formulation so that nothing ever moves between lanes:
//
//   Sᵀ[token, qcol] = K[token, :] · Qᵀ[:, qcol]      A = K page rows (tokens), B = Qᵀ
//   Oᵀ[d, qcol]    += Vᵀ[d, token] · Pᵀ[token, qcol]  A = Vᵀ page rows (d),    B = Pᵀ
//
// A lane (qcol = lane & 15, g = lane >> 4) therefore owns one query column for the whole kernel: its
// Sᵀ accumulators are 4 tokens of that column, the online-softmax state (m, l) is per lane, and the
// exponentiated accumulators of two 16-token tiles are — after a bf16 pack — exactly the B fragment
// of the P·V MFMA, because the V page stores its 32 tokens in that register order
// (ops/kv_layout.py).  K and V fragments are 16-byte loads straight from the page to VGPRs: every
// wave-level load is one contiguous 1 KiB, each byte of the cache is read once per consumer wave,
// so decode needs no LDS staging (memory-bound GEMV-like regime: every wave walks different pages).
// Prefill tiles share their pages between four waves and stage them through LDS (see below).
//
// qcol meaning:  decode  → query head inside the GQA group (G <= 16, padded columns are zero)
//                prefill → query token inside a 16-token tile, one (head, tile) "column group" per
//                          accumulator set, two column groups per wave.
//
// KV8: pages hold OCP e4m3 (K chunks are 64 wide, see kv_layout); values are widened to bf16 in
// registers, the per-tensor scales are folded into the softmax scale (K) and the epilogue (V).
#include <algorithm>
#include <cstdlib>

#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace dli {

constexpr int HD = 128;                 // head dim
constexpr int PAGE_ELEMS = HD * 32;     // elements per (page, kv head)
constexpr float NEG_BIG = -1.0e30f;


// ---- fragment loads ------------------------------------------------------------------------------
// K fragment for row tile rt (tokens 16rt..16rt+15) and k-step c (0..3) of lane (col, g).
template <bool KV8>
struct KLoader {
  // bf16: page [4][32 tok][32]:  element offset ((c*32 + rt*16 + col)*32 + 8g)
  // fp8 : page [2][32 tok][64]:  byte offset ((c2*32 + rt*16 + col)*64 + 16g) holds k-steps 2c2, 2c2+1
  // NT: streaming (non-temporal) loads — decode reads every K/V byte exactly once per step
  template <bool NT = false>
  static __device__ __forceinline__ void load(const void* page, int col, int g, bf16x8 (&kf)[2][4]) {
    if constexpr (!KV8) {
      const uint16_t* p = reinterpret_cast<const uint16_t*>(page) + col * 32 + g * 8;
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const bf16x8* src = reinterpret_cast<const bf16x8*>(p + (c * 32 + rt * 16) * 32);
          kf[rt][c] = NT ? __builtin_nontemporal_load(src) : *src;
        }
    } else {
      const uint8_t* p = reinterpret_cast<const uint8_t*>(page) + col * 64 + g * 16;
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int c2 = 0; c2 < 2; ++c2) {
          const u32x4* src = reinterpret_cast<const u32x4*>(p + (c2 * 32 + rt * 16) * 64);
          const u32x4 raw = NT ? __builtin_nontemporal_load(src) : *src;
          const uint32_t w[4] = {raw[0], raw[1], raw[2], raw[3]};
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            bf16x8 f;
            fp8x4_to_bf16(w[2 * h], f, 0);
            fp8x4_to_bf16(w[2 * h + 1], f, 4);
            kf[rt][2 * c2 + h] = f;
          }
        }
    }
  }
  // Matching d index of element j of the B (Qᵀ) fragment for k-step c of lane group g.
  static __device__ __forceinline__ int q_d0(int c, int g) {
    if constexpr (!KV8) return 32 * c + 8 * g;
    else return 64 * (c >> 1) + 16 * g + 8 * (c & 1);
  }
};

// V fragment for d tile n (rows 16n..16n+15) of lane (col, g): slots 8g..8g+7 of row d = 16n + col.
template <bool KV8, bool NT = false>
__device__ __forceinline__ bf16x8 load_v(const void* page, int n, int col, int g) {
  if constexpr (!KV8) {
    const bf16x8* src = reinterpret_cast<const bf16x8*>(reinterpret_cast<const uint16_t*>(page) + (16 * n + col) * 32 + 8 * g);
    return NT ? __builtin_nontemporal_load(src) : *src;
  } else {
    const u32x2* src = reinterpret_cast<const u32x2*>(reinterpret_cast<const uint8_t*>(page) + (16 * n + col) * 32 + 8 * g);
    const u32x2 raw = NT ? __builtin_nontemporal_load(src) : *src;
    bf16x8 f;
    fp8x4_to_bf16(raw[0], f, 0);
    fp8x4_to_bf16(raw[1], f, 4);
    return f;
  }
}

// Reductions over the 4 lanes (l, l^16, l^32, l^48) that share a query column, with the gfx950 row-swap VALU
// instructions instead of LDS-crossbar shuffles.  v_permlane16_swap(x, x) returns (rows 0,0,2,2 / rows 1,1,3,3) of
// x, v_permlane32_swap(x, x) returns (upper half twice / lower half twice): in every lane one of the two results
// is the lane's own value and the other its partner's, so max3 / a plain sum of the pair needs no select.
__device__ __forceinline__ float group_max(float v) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(v, fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1])));
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(v, fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1])));
}
__device__ __forceinline__ float group_sum(float v) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// One 32-token page against one query-column set: Sᵀ → online softmax → Pᵀ fragment.
// `limit`: tokens with index > limit are masked (limit = L-1 for decode, query position for prefill).
// The scale is applied inside the exponent (one fma per element: exp2(s·scale − m)); the running maximum m is
// kept in scaled units.
template <bool MASK>
__device__ __forceinline__ bf16x8 softmax_step(f32x4 (&s)[2], int tok0, int limit, float scale_log2, float& m,
                                               float& lsum, float& alpha) {
  float raw = NEG_BIG;
#pragma unroll
  for (int rt = 0; rt < 2; ++rt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float v = s[rt][r];
      if (MASK) v = (tok0 + rt * 16 + r <= limit) ? v : NEG_BIG;
      s[rt][r] = v;
      raw = fmaxf(raw, v);
    }
  const float mx = group_max(fmaxf(m, raw * scale_log2));
  alpha = fast_exp2(m - mx);
  m = mx;
  bf16x8 pb;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const f32x4 sc = {scale_log2, scale_log2, scale_log2, scale_log2}, nm = {-mx, -mx, -mx, -mx};
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const f32x4 e = __builtin_elementwise_fma(s[rt], sc, nm);            // v_pk_fma_f32: two elements per instruction
    f32x4 p;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      p[r] = fast_exp2(e[r]);
      if (MASK) p[r] = (tok0 + rt * 16 + r <= limit) ? p[r] : 0.f;
      pb[rt * 4 + r] = (short)f2bf(p[r]);
    }
    acc += p;                                                            // v_pk_add_f32
  }
  const float ps = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  lsum = lsum * alpha + ps;
  return pb;
}

// ==================================================================================================
// Decode: NW waves per workgroup; wave w takes pages w, w + NW, … of the workgroup's page range of one (sequence, kv head).
// The kv head is the fastest grid index: the 8 heads of a sequence (contiguous 64 KB per page) are read at the same
// time by neighbouring workgroups, and a long sequence's work is spread over 8 workgroups that start together instead
// of 8 that start num_seqs ids apart: +3–4 % on mixed-length batches (profiles/kernels_decode_r2aa.txt).
//
// Two ways to say which pages a workgroup reads:
//   WL = true   work list, grid (Hkv, items): `work[item] = {sequence, first page, end page, partial slot}` built by the
//               host per step (ops.build_decode_work) — page ranges of about equal size whatever the sequence's length,
//               so a 2048-token row and a 40-token row no longer get the same split count, longest range first, so the tail of
//               the launch is made of short ones (B = 160 of 128 … 2048 tokens, 721 MB: 122 µs in row order, 110 sorted).  slot < 0: the range is the whole sequence, the result goes straight to `out`.  The
//               number of valid items is read from DEVICE memory (`counts[0]`; extra workgroups exit), which is what
//               lets a hipGraph with a fixed grid serve any batch.
//   WL = false  uniform splits, grid (Hkv, num_seqs, num_splits): every sequence is cut into `num_splits` ranges.
// Partial results: `part_o[(p·Hq + head)·128 + d]`, `part_ml[(p·Hq + head)·2 + {m, l}]` with p = slot (WL) or
// seq·num_splits + split; decode_reduce_kernel combines them per sequence.
// ==================================================================================================
// item `item` of key head kvh (WL = false: sequence `item`, split `split`) by the NW waves whose threads are tid = 0 …; smem: decode_lds(NW, G) bytes of theirs.
// All waves of the workgroup pass its one barrier (or have ended).
template <bool KV8, bool WL, int NW, bool NT>
__device__ __forceinline__ void decode_item(
    int tid, int kvh, int item, int split, float* smem, const uint16_t* __restrict__ q, int64_t q_stride, const void* __restrict__ k_cache,
    const void* __restrict__ v_cache, const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ seq_lens,
    uint16_t* __restrict__ out, int64_t out_stride, float* __restrict__ part_o, float* __restrict__ part_ml, int Hq, int Hkv, int num_splits,
    float scale_log2, float v_scale, const float* __restrict__ kv_scales, const int4* __restrict__ work, const int* __restrict__ counts) {
  int seq, b_begin, b_end, part;                           // part < 0: write `out` directly
  if constexpr (WL) {
    if (item >= counts[0]) return;
    const int4 w = work[item];
    seq = w.x, b_begin = w.y, b_end = w.z, part = w.w;
  } else {
    seq = item;
    part = num_splits == 1 ? -1 : seq * num_splits + split;
  }
  if (KV8 && kv_scales != nullptr) {                       // calibrated per-(layer, kv head) fp8 scales: [k | v][Hkv]
    scale_log2 *= kv_scales[kvh];
    v_scale = kv_scales[Hkv + kvh];
  }
  const int G = Hq / Hkv;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // scalar: page loop, block-table reads and page bases in SGPRs
  const int col = lane & 15, g = lane >> 4;
  const int L = seq_lens[seq];
  const int nblk = (L + 31) >> 5;
  if constexpr (!WL) {
    const int per = (nblk + num_splits - 1) / num_splits;
    b_begin = split * per;
    b_end = min(nblk, b_begin + per);
  } else {
    b_end = min(b_end, nblk);
  }
  constexpr int ESZ = KV8 ? 1 : 2;

  bf16x8 qf[4];
  {
    const bool ok = col < G;
    const uint16_t* qp = q + (int64_t)seq * q_stride + (kvh * G + (ok ? col : 0)) * HD;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      bf16x8 v = *reinterpret_cast<const bf16x8*>(qp + KLoader<KV8>::q_d0(c, g));
      qf[c] = ok ? v : bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }

  f32x4 o[8];
#pragma unroll
  for (int n = 0; n < 8; ++n) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = NEG_BIG, lsum = 0.f;

  const int* bt = block_tables + (int64_t)seq * max_blocks;
  const char* kc = reinterpret_cast<const char*>(k_cache);
  const char* vc = reinterpret_cast<const char*>(v_cache);

  // the block-table entry of the NEXT page of this wave is fetched one iteration ahead: the entry → page address → 16
  // fragment loads chain is otherwise paid in full at the top of every iteration
  int blk_next = b_begin + wave < b_end ? bt[b_begin + wave] : 0;
  for (int b = b_begin + wave; b < b_end; b += NW) {
    const int blk_cur = blk_next;
    if (b + NW < b_end) blk_next = bt[b + NW];
    const int64_t page = ((int64_t)blk_cur * Hkv + kvh) * (PAGE_ELEMS * ESZ);
    bf16x8 kf[2][4];
    KLoader<KV8>::template load<NT>(kc + page, col, g, kf);
    bf16x8 vf[8];
#pragma unroll
    for (int n = 0; n < 8; ++n) vf[n] = load_v<KV8, NT>(vc + page, n, col, g);

    f32x4 s[2];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      s[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 4; ++c) s[rt] = mfma16(kf[rt][c], qf[c], s[rt]);
    }
    float alpha;
    bf16x8 pb;
    const int tok0 = b * 32 + 4 * g;
    if (b == nblk - 1) pb = softmax_step<true>(s, tok0, L - 1, scale_log2, m, lsum, alpha);
    else pb = softmax_step<false>(s, tok0, L - 1, scale_log2, m, lsum, alpha);
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      o[n] *= alpha;
      o[n] = mfma16(vf[n], pb, o[n]);
    }
  }
  lsum = group_sum(lsum);

  // ---- merge the waves through LDS: [wave][G][128 + 4] fp32 + [wave][G] (m, l).  Rows are padded by one 16-byte
  // slot: the G active lanes of a ds_write_b128 lane group hold the same d range of G different rows, and with
  // 512-byte rows they would all start on bank 0 (4-way conflict: 0.46 conflict cycles per LDS cycle in round 1).
  constexpr int HDP = HD + 4;
  float* sm_o = smem;
  float* sm_m = smem + NW * G * HDP;
  float* sm_l = sm_m + NW * G;
  if (col < G) {
    float* dst = sm_o + (wave * G + col) * HDP + 4 * g;
#pragma unroll
    for (int n = 0; n < 8; ++n) *reinterpret_cast<f32x4*>(dst + 16 * n) = o[n];
    if (g == 0) { sm_m[wave * G + col] = m; sm_l[wave * G + col] = lsum; }
  }
  __syncthreads();
  for (int idx = tid; idx < G * HD; idx += NW * 64) {
    const int head = idx >> 7, d = idx & 127;
    float M = NEG_BIG;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, sm_m[w * G + head]);
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = fast_exp2(sm_m[w * G + head] - M);
      num += f * sm_o[(w * G + head) * HDP + d];
      den += f * sm_l[w * G + head];
    }
    const int qh = kvh * G + head;
    if (part < 0) {
      const float r = den > 0.f ? v_scale / den : 0.f;
      out[(int64_t)seq * out_stride + qh * HD + d] = f2bf(num * r);
    } else {
      const int64_t slot = (int64_t)part * Hq + qh;
      part_o[slot * HD + d] = num;
      if (d == 0) { part_ml[slot * 2] = M; part_ml[slot * 2 + 1] = den; }
    }
  }
}

template <bool KV8, bool WL, int NW, bool NT = false>
__global__ __launch_bounds__(NW * 64) void paged_decode_kernel(
    const uint16_t* __restrict__ q, int64_t q_stride, const void* __restrict__ k_cache, const void* __restrict__ v_cache,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ seq_lens, uint16_t* __restrict__ out,
    int64_t out_stride, float* __restrict__ part_o, float* __restrict__ part_ml, int Hq, int Hkv, int num_splits,
    float scale_log2, float v_scale, const float* __restrict__ kv_scales, const int4* __restrict__ work,
    const int* __restrict__ counts) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  decode_item<KV8, WL, NW, NT>(threadIdx.x, blockIdx.x, blockIdx.y, blockIdx.z, smem, q, q_stride, k_cache, v_cache, block_tables, max_blocks, seq_lens, out,
                               out_stride, part_o, part_ml, Hq, Hkv, num_splits, scale_log2, v_scale, kv_scales, work, counts);
}

// Combine the partials of one (sequence, query head): 128 threads, one per d.  Uniform splits: grid (num_seqs, Hq),
// partials seq·num_splits … ; work list: grid (reduce entries, Hq), `red[i] = {sequence, first partial, count}` and the
// number of valid entries in `counts[1]` (device memory, like the decode kernel's item count).
__global__ __launch_bounds__(128) void decode_reduce_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                            uint16_t* __restrict__ out, int64_t out_stride, int Hq,
                                                            int num_splits, float v_scale, const float* __restrict__ kv_scales,
                                                            int Hkv, const int4* __restrict__ red, const int* __restrict__ counts) {
  int seq = blockIdx.x, first = (int)blockIdx.x * num_splits, n = num_splits;
  if (red != nullptr) {
    if ((int)blockIdx.x >= counts[1]) return;
    const int4 r = red[blockIdx.x];
    seq = r.x, first = r.y, n = r.z;
  }
  const int qh = blockIdx.y, d = threadIdx.x, lane = threadIdx.x & 63;
  if (kv_scales != nullptr) v_scale = kv_scales[Hkv + qh / (Hq / Hkv)];
  // 64 partials at a time, a lane each: their (m, l) arrive together and the rows' loads do not wait for one another.  (One after the
  // other — a load's latency per partial, twice — five partials took 4.5 µs.)  The rows come 8 at a time, 32 where there are many: behind one row of 16000 tokens
  // of one key head, in 126 ranges, the whole call 19.3 → 15.6 µs (beside a prompt's chunk of 400 tokens, which cannot hide it, 48.2 → 45.5); up to 16
  // ranges 24 loads too many cost up to 0.4.
  float M = NEG_BIG, num = 0.f, den = 0.f;
  for (int s0 = 0; s0 < n; s0 += 64) {
    const int k = min(n - s0, 64);
    const int64_t slot0 = (int64_t)(first + s0) * Hq + qh;
    const bool in = lane < k;
    const f32x2 ml = in ? *reinterpret_cast<const f32x2*>(part_ml + (slot0 + (int64_t)lane * Hq) * 2) : f32x2{NEG_BIG, 0.f};
    const float Mn = fmaxf(M, wave_max(ml[0])), old = fast_exp2(M - Mn);
    const float f = in ? fast_exp2(ml[0] - Mn) : 0.f;
    den = den * old + wave_sum(f * ml[1]);
    num *= old;
    M = Mn;
    auto add = [&](auto rows, int s) __attribute__((always_inline)) {
      constexpr int N = decltype(rows)::value;
      float x[N];
#pragma unroll
      for (int j = 0; j < N; ++j) x[j] = part_o[(slot0 + (int64_t)min(s + j, k - 1) * Hq) * HD + d];
#pragma unroll
      for (int j = 0; j < N; ++j) num += s + j < k ? __shfl(f, s + j, 64) * x[j] : 0.f;
    };
    if (k <= 16)
      for (int s = 0; s < k; s += 8) add(std::integral_constant<int, 8>{}, s);
    else
      for (int s = 0; s < k; s += 32) add(std::integral_constant<int, 32>{}, s);
  }
  const float r = den > 0.f ? v_scale / den : 0.f;
  out[(int64_t)seq * out_stride + qh * HD + d] = f2bf(num * r);
}

// ==================================================================================================
// Prefill: one workgroup of 4 waves per (tile, kv head).  A tile is TQ = 16·(8/G) consecutive query tokens of one sequence; its
// 8 column groups (head, 16-token sub-tile) are spread two per wave = 32 query columns per wave.  All K/V — paged
// prefix and the chunk itself — come from the cache (rope_and_cache has already written the chunk).
//
// Staging.  Unlike decode, all four waves of a tile walk the SAME pages, so K and V pages go through LDS: the block
// copies each 32-token page (K + V, 16 KB bf16 / 8 KB fp8) once by LDS-DMA (global_load_lds, 16 bytes per lane, no
// VGPRs) into a ring, and every wave reads its fragments with ds_read_b128.  A turn (one barrier) is one page of three stages, two pages ahead of
// the math, or with two groups, whose one workgroup a compute unit has the registers for it, two pages of two stages: two score
// chains side by side, and one question for both whether a maximum rises.  The page keeps its global layout in LDS except that the four 16-byte
// slots of every 64-byte row are permuted by the row (slot ^ h[(row >> 2) & 3], h = {0,2,3,1}; the DMA's LDS image is
// lane-linear, so the permutation sits on the SOURCE address): the 16 lanes the hardware serves together for a
// ds_read_b128 — {0–3, 12–15, 20–27} etc. — then touch 16 different slots of the 256-byte bank row.
//
// GROUPS = 2 (few tiles): a workgroup has two such sets of four waves; group g takes turns g, g + 2, … in a ring of its own, and at the end the
// groups' maxima, sums and accumulators meet in LDS.
// Two pages a turn: e4m3 with two groups.  µs, one page / two: 2 × 1024 behind 1024 41.7 / 35.5, one of 2048 behind 1500 with 8/1 heads 92.2 / 75.7, 64 behind
// 1900 54.7 / 45.8 (with 16-byte reads of the pages, which alone give 0.95: 8-byte ones of rows of 32 bytes met in 4 of 16 bank groups).  One group,
// where three workgroups share a compute unit, keeps one page (two leave two of them: e4m3, five prompts of up to 1333, 55.0 / 56.5; with 8-byte
// reads 61.4).  bf16 keeps one too: with two groups and one maximum for both, two pages are 4 % faster but round more weights (error against 64
// bits 0.00290 → 0.00291); with a maximum each they are not measured.
//
// Math on v_mfma_f32_32x32x16_bf16: a wave's 32 query columns are ONE MFMA column set.  Lane (c = lane & 31,
// hi = lane >> 5) owns column c:
//   Sᵀ(32 tok × 32 col)  = 8 MFMAs over d (k-step j: d = 16 j + 8 hi …); the lane's 16 accumulators are tokens
//                          (r & 3) + 8 (r >> 2) + 4 hi of the page;
//   P fragments          : slot jj·2 + hi (16 bytes) of a V page row holds the tokens of accumulators 4 jj … 4 jj + 3 and 8 + 4 jj …
//                          11 + 4 jj (v_slot, ops/kv_layout.py — the layout serves both MFMA shapes): exp2 and a bf16 pack of
//                          those are the B fragment of k-step jj, one ds_read_b128 of the slot its A fragment;
//   Oᵀ(128 d × 32 col)   = 4 d-tiles × 2 k-steps = 8 MFMAs.
// A wave's page is ≈ 75 vector instructions beside the 16 products (and 64 where a maximum rises; 205 with the
// halves of two V slots mixed into a fragment); one wave alone needs ≈ 0.7 µs for it, a serial chain of fragment reads, products,
// exponentials and the issue of its share of the next page's DMA.  Whole steps, 32/8 heads: fresh prompts of up to 1333 tokens (4100 in all)
// 56.4 → 55.2 µs, one of 4000 159 → 151 (0.99 PFLOP/s), two of 2048 87.9 → 85.4.
// ==================================================================================================
__device__ __forceinline__ int slot_swizzle(int row) { return (0x78 >> (2 * ((row >> 2) & 3))) & 3; }

// One page of a 32-column set.  Largest visible score of the lane's 16 (masked ones become NEG_BIG) …
template <bool MASK>
__device__ __forceinline__ float page_max32(f32x16& s, int tok0, int limit) {
  float raw = NEG_BIG;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    if (MASK) s[r] = (tok0 + (r & 3) + 8 * (r >> 2) <= limit) ? s[r] : NEG_BIG;
    raw = fmaxf(raw, s[r]);
  }
  return raw;
}
// … and scores → weights 2^(s · scale − m) as the two B fragments of P·V; returns the lane's sum.  pb[jj] holds accumulators 4 jj … 4 jj + 3
// and 8 + 4 jj … 11 + 4 jj: the tokens of 16-byte slot 2 jj + hi of a V page row.
template <bool MASK>
__device__ __forceinline__ float page_weights32(const f32x16& s, int tok0, int limit, float scale_log2, float m, bf16x8 (&pb)[2]) {
  float ps = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    float p = fast_exp2(__builtin_fmaf(s[r], scale_log2, -m));
    if (MASK) p = (tok0 + (r & 3) + 8 * (r >> 2) <= limit) ? p : 0.f;
    ps += p;
    pb[(r >> 2) & 1][(r & 3) + 4 * (r >> 3)] = (short)f2bf(p);
  }
  return ps;
}

// 16 bytes of an e4m3 V row are slots 2 hi and 2 hi + 1, not hi and 2 + hi: the weights of slots 1 and 2 change places
__device__ __forceinline__ void swap_slots(bf16x8 (&w)[2]) {
  u32x4 w0 = __builtin_bit_cast(u32x4, w[0]), w1 = __builtin_bit_cast(u32x4, w[1]);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    auto x = __builtin_amdgcn_permlane32_swap(w0[e], w1[e], false, false);
    w0[e] = x[0];
    w1[e] = x[1];
  }
  w[0] = __builtin_bit_cast(bf16x8, w0);
  w[1] = __builtin_bit_cast(bf16x8, w1);
}

// row d = 32 n + c32 of a staged V page: the A fragments of the two k-steps (off0, off1: this lane's offsets in n = 0; e4m3: one)
template <bool KV8>
__device__ __forceinline__ void value_fragments(const char* vb, int n, int off0, int off1, bf16x8& v0, bf16x8& v1) {
  if constexpr (!KV8) {
    v0 = *reinterpret_cast<const bf16x8*>(vb + n * 2048 + off0);
    v1 = *reinterpret_cast<const bf16x8*>(vb + n * 2048 + off1);
  } else {
    const u32x4 raw = *reinterpret_cast<const u32x4*>(vb + n * 1024 + off0);
    fp8x4_to_bf16(raw[0], v0, 0);
    fp8x4_to_bf16(raw[1], v0, 4);
    fp8x4_to_bf16(raw[2], v1, 0);
    fp8x4_to_bf16(raw[3], v1, 4);
  }
}

static constexpr int PREFILL_UNITS = 256;                      // workgroups of two groups that run at once: one a compute unit
template <bool KV8, int GROUPS, int NPG> struct PrefillShape {
  static constexpr int PAGE_BYTES = PAGE_ELEMS * (KV8 ? 1 : 2);
  static constexpr int STAGE = NPG * 2 * PAGE_BYTES;        // K and V of a turn's pages
  static constexpr int NSTAGE = NPG == 1 ? 3 : 2;
  static constexpr int RING = NSTAGE * STAGE;
  static constexpr int SWAP = GROUPS == 2 ? 4 * 2 * 8192 : 0;      // what two groups exchange at the end
  static constexpr int LDS = GROUPS * RING > SWAP ? GROUPS * RING : SWAP;
};
// workgroup `block` of a launch over num_tiles · Hkv tiles; smem_all: PrefillShape::LDS bytes
template <bool KV8, int GROUPS, int NPG>
__device__ __forceinline__ void prefill_tile(
    int block, char* smem_all, const uint16_t* __restrict__ q, int64_t q_stride, const void* __restrict__ k_cache, const void* __restrict__ v_cache,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ seq_lens,
    const int* __restrict__ query_start_loc, const int* __restrict__ tile_seq, const int* __restrict__ tile_q0,
    uint16_t* __restrict__ out, int64_t out_stride, int Hq, int Hkv, int num_tiles, float scale_log2, float v_scale,
    const float* __restrict__ kv_scales, int units) {
  using Shape = PrefillShape<KV8, GROUPS, NPG>;
  constexpr int PAGE_BYTES = Shape::PAGE_BYTES, STAGE = Shape::STAGE, NSTAGE = Shape::NSTAGE, RING = Shape::RING;
  constexpr int NCH = PAGE_BYTES / (16 * 256);
  constexpr int FLIGHT = 2 * NCH;                           // (three stages) DMA instructions of a wave for a turn

  // Block → (kv head, tile): the kv head is the fastest index.  Workgroups are dealt round-robin over the 8 XCDs (private L2s), so with 8
  // kv heads XCD x serves head x — a sequence's pages of that head are fetched into one L2 instead of eight —, with 2 or 4 every XCD
  // serves one head too, and every XCD gets the same mix of long and short tiles (a contiguous eighth of one head's tiles, longest
  // first, would leave most XCDs waiting for the first).
  const int G = Hq / Hkv;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);   // scalar: LDS-DMA destinations and the wave's page bounds in SGPRs
  const int wave = wave_all & 3, grp = GROUPS == 2 ? wave_all >> 2 : 0;
  char* smem = smem_all + grp * RING;
  const int c32 = lane & 31, hi = lane >> 5;
  // Two groups and more tiles than `units` workgroups: what is left over, the shortest tiles, goes to the second groups of the last workgroups, whose
  // two groups then do a tile each; the longest tiles keep both.
  const int items = num_tiles * Hkv, over = GROUPS == 2 ? max(items - units, 0) : 0;
  if (block >= items - over) return;
  const bool alone = GROUPS == 2 && block >= units - over;
  const int id = block + (alone ? grp * over : 0);
  const int kvh = id % Hkv, rank = id / Hkv;
  const int tile_id = num_tiles - 1 - rank;
  if (KV8 && kv_scales != nullptr) {
    scale_log2 *= kv_scales[kvh];
    v_scale = kv_scales[Hkv + kvh];
  }
  const int seq = tile_seq[tile_id], q0 = tile_q0[tile_id];
  const int qs = query_start_loc[seq];
  const int n_new = query_start_loc[seq + 1] - qs;
  const int L = seq_lens[seq];
  const int ctx = L - n_new;

  // this lane's column: column group cg = 2·wave + (c32 >> 4) is (head cg % G, 16-token sub-tile cg / G)
  const int cg = 2 * wave + (c32 >> 4);
  const int head = cg % G;
  const int qtok = q0 + (cg / G) * 16 + (c32 & 15);
  const bool valid = qtok < n_new;
  const int qpos = ctx + min(qtok, n_new - 1);
  int first_tok = 1 << 30, last_pos = -1;      // wave-uniform bounds over both column groups
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int t0 = q0 + ((2 * wave + i) / G) * 16;
    if (t0 < n_new) {
      first_tok = min(first_tok, ctx + t0);
      last_pos = max(last_pos, ctx + min(t0 + 15, n_new - 1));
    }
  }
  const int my_nblk = last_pos < 0 ? 0 : (last_pos >> 5) + 1;
  const int tile_tokens = 16 * (8 / G);
  const int nblk = ((ctx + min(q0 + tile_tokens, n_new) - 1) >> 5) + 1;
  // A tile of a few pages is done by one group alone, the other ends here (a barrier waits for the waves that are left): meeting at the end
  // costs as much as a turn of four pages less saves (prompts of 64 tokens, µs, two groups / one / now 8.25 / 7.28 / 7.4, of 160 10.4 / 9.7 / 9.8,
  // of 256 12.0 / 12.3 / 12.2).
  const bool both = GROUPS == 2 && !alone && nblk > 7;
  if (GROUPS == 2 && !both && !alone && grp == 1) return;
  const int nturn = (nblk + NPG - 1) / NPG;
  int turns = both ? (nturn + 1) >> 1 : nturn;
  const int step = both ? 2 : 1, start = both ? grp : 0;
  __shared__ int turns_of[2];
  if (alone && lane == 0 && wave == 0) turns_of[grp] = turns;

  // Qᵀ fragments: k-step j covers d = 16 j + 8 hi … + 7; with e4m3 pages, whose 16-byte slots hold two k-steps, d = 32 (j / 2) + 16 hi + 8 (j % 2) … + 7
  bf16x8 qf[8];
  {
    const uint16_t* qp = q + (int64_t)(qs + min(qtok, n_new - 1)) * q_stride + (kvh * G + head) * HD;
#pragma unroll
    for (int j = 0; j < 8; ++j) qf[j] = *reinterpret_cast<const bf16x8*>(qp + (KV8 ? 32 * (j >> 1) + 16 * hi + 8 * (j & 1) : 16 * j + 8 * hi));
  }

  f32x16 o[4];
#pragma unroll
  for (int n = 0; n < 4; ++n)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[n][r] = 0.f;
  float m = NEG_BIG, lsum = 0.f;

  const int* bt = block_tables + (int64_t)seq * max_blocks;
  const char* kc = reinterpret_cast<const char*>(k_cache);
  const char* vc = reinterpret_cast<const char*>(v_cache);

  int src_k[NCH], src_v[NCH];
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int ci = (tid & 255) + 256 * i, row = ci >> 2, slot = ci & 3;
    src_k[i] = (row * 4 + (slot ^ slot_swizzle(row))) * 16;
    src_v[i] = KV8 ? ci * 16 : src_k[i];
  }
  using gptr_t = const __attribute__((address_space(1))) void*;
  using lptr_t = __attribute__((address_space(3))) void*;
  auto stage_page = [&](int b, char* to) {
    const int64_t page = ((int64_t)bt[b] * Hkv + kvh) * PAGE_BYTES;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      char* dst = to + (wave + 4 * i) * 1024;
      __builtin_amdgcn_global_load_lds((gptr_t)(kc + page + src_k[i]), (lptr_t)dst, 16, 0, 0);
      __builtin_amdgcn_global_load_lds((gptr_t)(vc + page + src_v[i]), (lptr_t)(dst + PAGE_BYTES), 16, 0, 0);
    }
  };
  auto stage = [&](int turn, int at) {
#pragma unroll
    for (int p = 0; p < NPG; ++p)
      if (p == 0 || NPG * turn + p < nblk) stage_page(NPG * turn + p, smem + at * STAGE + p * 2 * PAGE_BYTES);
  };
  // SPREAD (two groups): the pieces of the turn that is fetched are asked for behind the first score products, whose fragments are read before them, and its
  // block table entries a turn before.  At the start of a turn, where all waves have just passed the barrier, the pieces queue up for the unit's one path to memory while
  // the matrix cores are idle, and a scalar load that is waited for where it is made stops the wave for its latency.  Whole calls with rotation and cache
  // write, µs, at the start / spread: bf16, 32/8 heads, one prompt of 1000 tokens 41.4 / 39.7, of 2000 80.4 / 76.4, 8/1 heads 58.8 / 51.5, of 3500 95.9 / 83.7;
  // e4m3, 32/8 heads, 2000 77.6 / 76.7, 8/1 heads 55.8 / 53.9, of 3500 90.5 / 86.2.
  // One group, whose unit has three workgroups at different places, loses 1 to 4 %.
  constexpr bool SPREAD = GROUPS == 2;
  int entry[NPG];
  auto look_up = [&](int turn) {
#pragma unroll
    for (int p = 0; p < NPG; ++p) entry[p] = bt[min(NPG * turn + p, nblk - 1)];
  };
  // quarter `part` of a turn's pieces
  auto stage_part = [&](int turn, int at, int part) __attribute__((always_inline)) {
    constexpr int PIECES = 2 * NCH;                         // a wave's DMA instructions for a page
#pragma unroll
    for (int i = NPG * PIECES * part / 4; i < NPG * PIECES * (part + 1) / 4; ++i) {
      if (i >= PIECES && NPG * turn + 1 >= nblk) break;
      const int64_t page = ((int64_t)entry[i / PIECES] * Hkv + kvh) * PAGE_BYTES;
      char* dst = smem + at * STAGE + i / PIECES * 2 * PAGE_BYTES + (wave + 4 * (i % PIECES >> 1)) * 1024;
      if (i & 1) __builtin_amdgcn_global_load_lds((gptr_t)(vc + page + src_v[i % PIECES >> 1]), (lptr_t)(dst + PAGE_BYTES), 16, 0, 0);
      else __builtin_amdgcn_global_load_lds((gptr_t)(kc + page + src_k[i % PIECES >> 1]), (lptr_t)dst, 16, 0, 0);
    }
  };
  // Lane offsets inside a staged page.  Rows of 64 bytes (K: token rows of a d chunk; bf16 V: d rows) carry the slot
  // swizzle of their row; it depends on (row >> 2) & 3 only, and every row this lane reads is c32 + a multiple of 32.
  const int swz = slot_swizzle(c32);
  int k_off[2];                                   // logical slot 2 p + hi
#pragma unroll
  for (int p = 0; p < 2; ++p) k_off[p] = c32 * 64 + (((2 * p + hi) ^ swz) << 4);
  const int v_off0 = c32 * 64 + ((hi ^ swz) << 4), v_off1 = c32 * 64 + (((2 + hi) ^ swz) << 4);
  const int v8_off = c32 * 32 + 16 * hi;

  // NP pages from b on, staged at `kb`: scores, maxima, weights, P·V; between(0 … 3) behind the first four pairs of products
  auto pages = [&](auto np, int b, const char* kb, auto&& between) __attribute__((always_inline)) {
    constexpr int NP = decltype(np)::value;
    f32x16 s[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[p][r] = 0.f;
    if constexpr (!SPREAD && !KV8) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int p = 0; p < NP; ++p)
          s[p] = mfma32(*reinterpret_cast<const bf16x8*>(kb + p * 2 * PAGE_BYTES + (j >> 1) * 2048 + k_off[j & 1]), qf[j], s[p]);
    } else if constexpr (!KV8) {
      bf16x8 kf[NP][8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int p = 0; p < NP; ++p) kf[p][j] = *reinterpret_cast<const bf16x8*>(kb + p * 2 * PAGE_BYTES + (j >> 1) * 2048 + k_off[j & 1]);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
#pragma unroll
        for (int p = 0; p < NP; ++p) s[p] = mfma32(kf[p][j], qf[j], s[p]);
        if (j < 4) between(j);
      }
    } else if constexpr (!SPREAD) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          const u32x4 raw = *reinterpret_cast<const u32x4*>(kb + p * 2 * PAGE_BYTES + (j >> 1) * 2048 + k_off[j & 1]);
          bf16x8 k0, k1;
          fp8x4_to_bf16(raw[0], k0, 0);
          fp8x4_to_bf16(raw[1], k0, 4);
          fp8x4_to_bf16(raw[2], k1, 0);
          fp8x4_to_bf16(raw[3], k1, 4);
          s[p] = mfma32(k0, qf[2 * j], s[p]);
          s[p] = mfma32(k1, qf[2 * j + 1], s[p]);
        }
    } else {
      u32x4 raw[NP][4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int p = 0; p < NP; ++p) raw[p][j] = *reinterpret_cast<const u32x4*>(kb + p * 2 * PAGE_BYTES + (j >> 1) * 2048 + k_off[j & 1]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          bf16x8 k0, k1;
          fp8x4_to_bf16(raw[p][j][0], k0, 0);
          fp8x4_to_bf16(raw[p][j][1], k0, 4);
          fp8x4_to_bf16(raw[p][j][2], k1, 0);
          fp8x4_to_bf16(raw[p][j][3], k1, 4);
          s[p] = mfma32(k0, qf[2 * j], s[p]);
          s[p] = mfma32(k1, qf[2 * j + 1], s[p]);
        }
        between(j);
      }
    }
    const int tok0 = b * 32 + 4 * hi;
    // The maximum moves with every page that raises it in some lane, so a column's largest weight is 1, exact in bf16.  (A maximum that lags by up to
    // 2^8 saves these 64 products on most pages, 3 – 10 % of a launch, but rounds the largest weight like all others: relative error
    // against 64 bits 0.00266 → 0.00272, e4m3 pages 0.00731 → 0.00734.)
    if constexpr (NP == 1) {
      const bool edge = b * 32 + 31 > first_tok;
      float mx = edge ? page_max32<true>(s[0], tok0, qpos) : page_max32<false>(s[0], tok0, qpos);
      mx *= scale_log2;
      auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
      if (__any(mx > m)) {
        asm volatile("" ::: "memory");
        const float mn = fmaxf(m, mx), alpha = fast_exp2(m - mn);
        m = mn;
        lsum *= alpha;
#pragma unroll
        for (int n = 0; n < 4; ++n) o[n] *= alpha;
      }
      bf16x8 pb[2];
      lsum += edge ? page_weights32<true>(s[0], tok0, qpos, scale_log2, m, pb) : page_weights32<false>(s[0], tok0, qpos, scale_log2, m, pb);
      if constexpr (KV8) swap_slots(pb);
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        bf16x8 v0, v1;
        value_fragments<KV8>(kb + PAGE_BYTES, n, KV8 ? v8_off : v_off0, v_off1, v0, v1);
        o[n] = mfma32(v0, pb[0], o[n]);
        o[n] = mfma32(v1, pb[1], o[n]);
      }
    } else {
      // both maxima, then both pages' weights, each to its own maximum; only where one of them rises are the accumulators asked twice.  (One
      // maximum for both rounds the first page's largest weights: 0.007210 → 0.007213 for a mixed step, larger in 43 of 48 calls, and takes 1.00 to 1.03 of the time.)
      bool edge[2];
      float mx[2];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        edge[p] = (b + p) * 32 + 31 > first_tok;
        const float x = (edge[p] ? page_max32<true>(s[p], tok0 + 32 * p, qpos) : page_max32<false>(s[p], tok0 + 32 * p, qpos)) * scale_log2;
        auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
        mx[p] = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
      }
      bf16x8 pb[2][2];
      auto weights = [&](int p, float top) __attribute__((always_inline)) {
        const float ps = edge[p] ? page_weights32<true>(s[p], tok0 + 32 * p, qpos, scale_log2, top, pb[p]) : page_weights32<false>(s[p], tok0 + 32 * p, qpos, scale_log2, top, pb[p]);
        if constexpr (KV8) swap_slots(pb[p]);
        return ps;
      };
      auto rescale = [&](float alpha) __attribute__((always_inline)) {
        asm volatile("" ::: "memory");
        lsum *= alpha;
#pragma unroll
        for (int n = 0; n < 4; ++n) o[n] *= alpha;
      };
      auto add_values = [&](int p) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          bf16x8 v0, v1;
          value_fragments<KV8>(kb + p * 2 * PAGE_BYTES + PAGE_BYTES, n, KV8 ? v8_off : v_off0, v_off1, v0, v1);
          o[n] = mfma32(v0, pb[p][0], o[n]);
          o[n] = mfma32(v1, pb[p][1], o[n]);
        }
      };
      const float m0 = fmaxf(m, mx[0]), m1 = fmaxf(m0, mx[1]);
      const float ps0 = weights(0, m0), ps1 = weights(1, m1);
      if (__any(m1 > m)) {
        rescale(fast_exp2(m - m0));
        lsum += ps0;
        add_values(0);
        rescale(fast_exp2(m0 - m1));
        add_values(1);
      } else {
        lsum += ps0;
        add_values(0);
        add_values(1);
      }
      lsum += ps1;
      m = m1;
    }
  };

  // group g takes turns g, g + 2, … (of a tile of its own: all) in a ring of its own; both pass the same barriers
  if (start < nturn) stage(start, 0);
  if (NSTAGE == 3 && start + step < nturn) {
    stage(start + step, 1);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FLIGHT) : "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  if (SPREAD) look_up(start + (NSTAGE - 1) * step);
  __syncthreads();
  if (alone) turns = max(turns_of[0], turns_of[1]);
  int st = 0;
  for (int t = 0; t < turns; ++t) {
    const int turn = step * t + start;
    const int later = turn + (NSTAGE - 1) * step, to = st == 0 ? NSTAGE - 1 : st - 1;
    const bool ahead = later < nturn;
    auto between = [&](int part) __attribute__((always_inline)) {
      if (SPREAD && ahead) stage_part(later, to, part);
    };
    if (!SPREAD && ahead) stage(later, to);
    const char* kb = smem + st * STAGE;
    if (NPG == 2 && 2 * turn + 1 < my_nblk) pages(std::integral_constant<int, 2>{}, 2 * turn, kb, between);
    else if (NPG * turn < my_nblk) pages(std::integral_constant<int, 1>{}, NPG * turn, kb, between);
    else
#pragma unroll
      for (int part = 0; part < 4; ++part) between(part);
    if (SPREAD && ahead) look_up(later + step);
    if (NSTAGE == 3 && ahead) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FLIGHT) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    st = st == NSTAGE - 1 ? 0 : st + 1;
  }

  if constexpr (GROUPS == 2) {
    if (both) {
      // the two groups of a column set swap halves of their sums: group 0 finishes d tiles 0 and 1, group 1 tiles 2 and 3
      __shared__ float ml[2][4][2][64];
      float* X = reinterpret_cast<float*>(smem_all) + wave * 2 * 2048;              // [wave][from group][32][64]
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) X[grp * 2048 + (n * 16 + r) * 64 + lane] = grp ? o[n][r] : o[n + 2][r];
      ml[grp][wave][0][lane] = m;
      ml[grp][wave][1][lane] = lsum;
      __syncthreads();
      const float m2 = ml[grp ^ 1][wave][0][lane], M = fmaxf(m, m2), f1 = fast_exp2(m - M), f2 = fast_exp2(m2 - M);
      float l = lsum * f1 + ml[grp ^ 1][wave][1][lane] * f2;
      {
        auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
        l = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
      }
      if (valid) {
        const float rcp = l > 0.f ? v_scale / l : 0.f;
        const float r1 = f1 * rcp, r2 = f2 * rcp;
        uint16_t* op = out + (int64_t)(qs + qtok) * out_stride + (kvh * G + head) * HD + 4 * hi + grp * 64;
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
          for (int r4 = 0; r4 < 4; ++r4) {
            bf16x4 w;
#pragma unroll
            for (int e = 0; e < 4; ++e)
              w[e] = (short)f2bf((grp ? o[n + 2][4 * r4 + e] : o[n][4 * r4 + e]) * r1 + X[(grp ^ 1) * 2048 + (n * 16 + 4 * r4 + e) * 64 + lane] * r2);
            *reinterpret_cast<bf16x4*>(op + 32 * n + 8 * r4) = w;
          }
      }
      return;
    }
  }
  {
    auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(lsum), __float_as_uint(lsum), false, false);
    const float l = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
    if (valid) {
      const float rcp = l > 0.f ? v_scale / l : 0.f;
      uint16_t* op = out + (int64_t)(qs + qtok) * out_stride + (kvh * G + head) * HD + 4 * hi;
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
          bf16x4 w;
#pragma unroll
          for (int e = 0; e < 4; ++e) w[e] = (short)f2bf(o[n][4 * r4 + e] * rcp);
          *reinterpret_cast<bf16x4*>(op + 32 * n + 8 * r4) = w;
        }
    }
  }
}

template <bool KV8, int GROUPS, int NPG>
__global__ __launch_bounds__(256 * GROUPS, 2) void paged_prefill_kernel(
    const uint16_t* __restrict__ q, int64_t q_stride, const void* __restrict__ k_cache, const void* __restrict__ v_cache,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ seq_lens,
    const int* __restrict__ query_start_loc, const int* __restrict__ tile_seq, const int* __restrict__ tile_q0,
    uint16_t* __restrict__ out, int64_t out_stride, int Hq, int Hkv, int num_tiles, float scale_log2, float v_scale,
    const float* __restrict__ kv_scales, const int* __restrict__ counts, int units) {
  __shared__ __attribute__((aligned(16))) char smem[PrefillShape<KV8, GROUPS, NPG>::LDS];
  // inside a hipGraph the grid is an upper bound and the step's tile count lives in device memory (counts[2])
  if (counts != nullptr) num_tiles = counts[2];
  prefill_tile<KV8, GROUPS, NPG>(blockIdx.x, smem, q, q_stride, k_cache, v_cache, block_tables, max_blocks, seq_lens, query_start_loc, tile_seq,
                                 tile_q0, out, out_stride, Hq, Hkv, num_tiles, scale_log2, v_scale, kv_scales, units);
}

// Mixed steps: decode rows and prompt tiles in one launch, workgroups of four waves each.  Prompt tiles are bound by their chain of pages and the vector
// instructions, decode rows by the cache's bytes, so a compute unit that holds both does one while the other waits; one after the other, 96 e4m3 rows of
// up to 1500 tokens and two chunks of up to 1024 behind up to 1024 (32/8 heads) take 67 µs, here 49, and in bf16 99 → 65.  (Two streams or two branches of a
// graph reach part of it: their launches compete for the units as they come, a captured branch costs 5 µs where the step is small, an event on an eager
// stream 10 and 30 to 55 of the host.)
// Three workgroups share a unit (145 registers, 48 KB of LDS).  Octets of workgroups, one for each XCD so that a head's pages stay in one L2:
//   * more than 512 tiles: every third octet is one of decode rows, as long as there are both, then what is left.  So many tiles would fill all units and
//     leave the decode rows for the end (96 bf16 rows, one fresh prompt of 3500 tokens, 880 tiles: prompts first 152 µs, every second 185, every third 138,
//     every fourth 152; e4m3 rows, four of 1000 behind 500, 672 tiles 68 / 78 / 58 / 65);
//   * up to 512: all prompts first, whose longest chain the launch has to wait for anyway, where they leave a third of the units' room (e4m3, 504 tiles:
//     85 / 115 / 94 / 91; 200 tiles 50 / 47 / 49 / 48).
// A captured launch deals the step's own tiles and rows, which the device knows, not the bounds of its grid: by the bounds, 256 tiles among 2304 had decode rows
// between them, which left units with two of the longest tiles beside units without any (e4m3, 16 rows and 1000 tokens behind 6000: branches 245 µs, dealt
// by bounds 258, by what there is 205).
// GROUPS = 2: tiles by two page groups and decode items by as many waves as in their own launch (both give the same bits), a workgroup a compute unit.
template <bool KV8, bool WL, int GROUPS, bool NT>
__global__ __launch_bounds__(256 * GROUPS, GROUPS == 1 ? 3 : 2) void paged_mixed_kernel(
    const uint16_t* __restrict__ q, int64_t q_stride, const void* __restrict__ k_cache, const void* __restrict__ v_cache,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ seq_lens, const int* __restrict__ query_start_loc,
    const int* __restrict__ tile_seq, const int* __restrict__ tile_q0, uint16_t* __restrict__ out, int64_t out_stride,
    float* __restrict__ part_o, float* __restrict__ part_ml, int Hq, int Hkv, int num_tiles, int items, int num_splits, float scale_log2, float v_scale,
    const float* __restrict__ kv_scales, const int4* __restrict__ work, const int* __restrict__ counts, int on_device) {
  constexpr int NPG = GROUPS == 2 && KV8 ? 2 : 1, NW = GROUPS == 2 && !KV8 ? 8 : 4, IPW = 4 * GROUPS / NW;      // IPW: decode items a workgroup
  __shared__ __attribute__((aligned(16))) char smem[PrefillShape<KV8, GROUPS, NPG>::LDS];      // (a decode item of up to 8 heads a group takes 17 KB of it, 34 by eight waves)
  if (on_device) {                                          // the launched numbers are bounds
    num_tiles = min(num_tiles, counts[2]);
    if (WL) items = min(items, counts[0]);
  }
  const int period = num_tiles * Hkv > 2 * PREFILL_UNITS ? 3 : 0;
  const int octets = (num_tiles * Hkv + 7) >> 3, rows = ((items + IPW - 1) / IPW * Hkv + 7) >> 3;
  const int octet = (int)blockIdx.x >> 3, in = (int)blockIdx.x & 7;
  const int turns = period > 1 ? min(rows, octets / (period - 1)) : 0;
  int tile = octet - turns, row = -1;                       // behind the turns: the other tiles, then the other rows
  if (octet < turns * period) {
    const int turn = octet / period, at = octet - turn * period;
    if (at == period - 1) row = turn;
    else tile = octet - turn;
  } else if (tile >= octets) {
    row = octet - octets;
  }
  if (row < 0) {
    prefill_tile<KV8, GROUPS, NPG>(8 * tile + in, smem, q, q_stride, k_cache, v_cache, block_tables, max_blocks, seq_lens, query_start_loc, tile_seq,
                                   tile_q0, out, out_stride, Hq, Hkv, num_tiles, scale_log2, v_scale, kv_scales, 0x7fffffff);
    return;
  }
  const int sub = IPW == 2 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8) : 0;
  const int id = 8 * row + in, group = id / Hkv, kvh = id - group * Hkv, item = group * IPW + sub;
  if (item >= items) return;                                // the last octet, the last item's neighbour
  const int seq = WL ? item : item / num_splits, split = WL ? 0 : item - seq * num_splits;
  decode_item<KV8, WL, NW, NT>((int)threadIdx.x - 256 * sub, kvh, seq, split, reinterpret_cast<float*>(smem + sub * (int)(sizeof(smem) / 2)), q, q_stride,
                                 k_cache, v_cache, block_tables, max_blocks, seq_lens, out, out_stride, part_o, part_ml, Hq, Hkv, num_splits,
                                 scale_log2, v_scale, kv_scales, work, counts);
}

// ---- launchers -------------------------------------------------------------------------------------
// Decode reads every K/V byte exactly once per step: the loads are NON-TEMPORAL (streaming cache policy), so the pages do not
// displace what the GEMMs keep in L2 / the infinity cache and are themselves not written into them: 5.95 → 6.60 TB/s on the
// trace's length mix at B = 1024 (profiles/ab_decode_nt_r3.jsonl).  DLI_DECODE_NT=0: plain loads (A/B knob).
static const bool g_decode_nt = std::getenv("DLI_DECODE_NT") == nullptr || std::atoi(std::getenv("DLI_DECODE_NT")) != 0;

// Waves of a decode workgroup, the same for both launches, so that a row that is one range gets the same bits from either.
// bf16: eight halve a whole row's serial pages; e4m3 pages take half the bytes a wave and the registers of the
// widening: four.  Sorted lists, 32/8 heads, µs, 4 against 8 waves — bf16, rows of up to 1500 tokens: B = 100 55.9 / 52.6; e4m3:
// B = 100 30.0 / 32.6, 160 60.1 / 60.9, 300 104.6 / 112.4.  Rows cut into ranges of four pages and more, where
// half of eight waves may have none, bf16: B = 1 of 620 tokens 7.9 / 7.6, 8 8.6 / 8.4, 1 of 2048 9.1 / 8.9, 8 13.3 / 14.3, 48 41.1 / 38.7.
// Many workgroups keep four: the compute units are full anyway, and of a short row's eight waves half have no page.  Rows of up to 40 / 100 / 200 /
// 1000 tokens, four against eight — B = 128 (1024 workgroups) 9.2 / 9.4, 11.0 / 10.8, 14.4 / 14.6, 45.0 / 44.6; B = 160 of up to
// 2048 111.8 / 109.5, but of up to 40 10.0 / 11.5; B = 256 14.2 / 16.5, 17.6 / 19.6,
// 24.6 / 25.1, 86.2 / 86.4; B = 512 26.8 / 31.8, 31.1 / 35.6, 44.9 / 46.4, 175 / 176.
// Groups of more than 8 heads keep four: eight waves' merge buffers would pass 64 KB of LDS.
static int decode_waves(bool kv_fp8, int G, int64_t workgroups) { return kv_fp8 || G > 8 || workgroups > 1024 ? 4 : 8; }
static size_t decode_lds(int waves, int G) { return (size_t)(waves * G * (HD + 4) + 2 * waves * G) * sizeof(float); }

void launch_paged_decode(const void* q, int64_t q_stride, const void* k_cache, const void* v_cache,
                         const int* block_tables, int max_blocks, const int* seq_lens, void* out, int64_t out_stride,
                         float* part_o, float* part_ml, int num_seqs, int Hq, int Hkv, int num_splits, float scale,
                         bool kv_fp8, float k_scale, float v_scale, const float* kv_scales, hipStream_t stream) {
  if (num_seqs == 0) return;
  const int G = Hq / Hkv;
  if (kv_scales != nullptr) k_scale = v_scale = 1.f;        // the kernels read the per-head values themselves
  const float scale_log2 = scale * 1.4426950408889634f * (kv_fp8 ? k_scale : 1.f);
  dim3 grid(Hkv, num_seqs, num_splits);
#define DLI_DECODE_GO(KV8_, NW_, NT_)                                                                                         \
  hipLaunchKernelGGL((paged_decode_kernel<KV8_, false, NW_, NT_>), grid, dim3(NW_ * 64), decode_lds(NW_, G), stream, (const uint16_t*)q, \
                     q_stride, k_cache, v_cache, block_tables, max_blocks, seq_lens, (uint16_t*)out, out_stride, part_o, part_ml, Hq, Hkv, \
                     num_splits, scale_log2, KV8_ ? v_scale : 1.f, KV8_ ? kv_scales : nullptr, nullptr, nullptr)
  if (kv_fp8) { if (g_decode_nt) DLI_DECODE_GO(true, 4, true); else DLI_DECODE_GO(true, 4, false); }
  else if (decode_waves(kv_fp8, G, (int64_t)Hkv * num_seqs * num_splits) == 4) { if (g_decode_nt) DLI_DECODE_GO(false, 4, true); else DLI_DECODE_GO(false, 4, false); }
  else { if (g_decode_nt) DLI_DECODE_GO(false, 8, true); else DLI_DECODE_GO(false, 8, false); }
#undef DLI_DECODE_GO
  if (num_splits > 1)
    hipLaunchKernelGGL(decode_reduce_kernel, dim3(num_seqs, Hq), dim3(128), 0, stream, part_o, part_ml, (uint16_t*)out,
                       out_stride, Hq, num_splits, kv_fp8 ? v_scale : 1.f, kv_fp8 ? kv_scales : nullptr, Hkv, nullptr, nullptr);
}

// Work-list decode: `items` / `reds` are the LAUNCHED grid extents (an upper bound inside a hipGraph); the valid counts
// are counts[0] / counts[1] on the device.
void launch_paged_decode_worklist(const void* q, int64_t q_stride, const void* k_cache, const void* v_cache,
                                  const int* block_tables, int max_blocks, const int* seq_lens, void* out,
                                  int64_t out_stride, float* part_o, float* part_ml, const int* work, const int* red,
                                  const int* counts, int items, int reds, int Hq, int Hkv, float scale, bool kv_fp8,
                                  float k_scale, float v_scale, const float* kv_scales, hipStream_t stream) {
  if (items <= 0) return;
  const int G = Hq / Hkv;
  if (kv_scales != nullptr) k_scale = v_scale = 1.f;
  const float scale_log2 = scale * 1.4426950408889634f * (kv_fp8 ? k_scale : 1.f);
  dim3 grid(Hkv, items);
#define DLI_DECODE_GO(KV8_, NW_, NT_)                                                                                         \
  hipLaunchKernelGGL((paged_decode_kernel<KV8_, true, NW_, NT_>), grid, dim3(NW_ * 64), decode_lds(NW_, G), stream, (const uint16_t*)q, \
                     q_stride, k_cache, v_cache, block_tables, max_blocks, seq_lens, (uint16_t*)out, out_stride, part_o, part_ml, Hq,  \
                     Hkv, 1, scale_log2, KV8_ ? v_scale : 1.f, KV8_ ? kv_scales : nullptr, (const int4*)work, counts)
  if (kv_fp8) { if (g_decode_nt) DLI_DECODE_GO(true, 4, true); else DLI_DECODE_GO(true, 4, false); }
  else if (decode_waves(kv_fp8, G, (int64_t)Hkv * items) == 4) { if (g_decode_nt) DLI_DECODE_GO(false, 4, true); else DLI_DECODE_GO(false, 4, false); }
  else { if (g_decode_nt) DLI_DECODE_GO(false, 8, true); else DLI_DECODE_GO(false, 8, false); }
#undef DLI_DECODE_GO
  if (reds > 0)
    hipLaunchKernelGGL(decode_reduce_kernel, dim3(reds, Hq), dim3(128), 0, stream, part_o, part_ml, (uint16_t*)out,
                       out_stride, Hq, 1, kv_fp8 ? v_scale : 1.f, kv_fp8 ? kv_scales : nullptr, Hkv, (const int4*)red, counts);
}

// Two groups where a compute unit gets one workgroup: a tile's pages are a serial chain of 0.7 µs each, and what the chip has no second tile for, a
// second half of the same tile can fill.  Causal tiles of 32/8 heads, µs, one / two groups: prompts of 1000 tokens (256 workgroups) 34.1 / 29.6, of 2000
// with 8/1 heads (125) 58.2 / 45.8, 8 × 128 tokens behind 1000 (256) 40.9 / 34.5, 32 × 16 behind 300 15.5 / 15.1.
// A unit holds one workgroup of two groups (100 KB of LDS; e4m3 68 KB, but its registers leave room for one too), and three of one.  Past 256 tiles:
//   * the shortest share workgroups, a group each (SHARED).  Both pass the same barriers, so they wait for their loads and products at the same time and
//     take 1.25 of what they take in workgroups of their own; the longest take 0.8.  It pays where the shared ones are the shorter ones: 2 × 600 tokens
//     (304 tiles) 24.1 / 20.6, 4 × 300 (320) 15.8 / 14.9, one of 1100 behind 500 (280) 51.2 / 39.4, but 3 × 400 behind 1000 (312) 50.2 / 54.8, 2 × 1024
//     (512, all shared) 38.6 / 45.1.  e4m3, whose two groups take two pages a turn: 2 × 600 behind 600 42.8 / 41.2, 1100 behind 2000 (280) 100 / 93.8,
//     4 × 1500 behind 500 with 8/1 heads (376) 62.8 / 61.9.
//   * or the rest comes in a second round (ROUNDS), whose workgroups all start with 5 µs of latencies: 16 × 100 tokens (512) 13.0 / 16.6, 9 × 128 behind
//     1000 (288) 49.5 / 57.8.  It pays only if that is made of short tiles: one prompt of 2000 (504) 65.1 / 58.0.  With 5 µs + 0.0285 µs a token for
//     one group, 5.5 + 0.0225 for two, and the first tile of the second round at `second` tokens of context, that is what the last line says.
// The lines were fitted on 190 steps of equal prompts before two groups spread their fetches, which takes a token of theirs from 0.0225 to 0.0207 µs.  At 47
// sizes timed since (profiles/prefill_page_groups.txt) the form taken is the fastest or within 3 % for equal prompts, but for one of 2000 behind 500
// (1.06) and, 8/1 heads, of several long ones that would rather have a second round than share (1.06 to 1.09).  `mean` speaks of equal prompts: of uneven
// ones, a long one beside short ones is kept at one group where two would take 0.78.
// longest: tokens of context (new ones included) of the longest sequence, sequences: with new tokens; 0: not known, as for a captured launch of bounds.
int prefill_page_groups(int num_tiles, int Hkv, int G, int longest, int sequences, bool kv_fp8) {
  constexpr int ONE = 1, ROUNDS = 2, SHARED = 3;
  const int blocks = num_tiles * Hkv, tile_tokens = 16 * (8 / G);
  if (blocks <= PREFILL_UNITS) return longest == 0 || longest > 224 ? ROUNDS : ONE;
  if (blocks > 2 * PREFILL_UNITS || longest <= 224 || sequences <= 0) return ONE;
  const float mean = std::min((float)longest, (float)num_tiles * tile_tokens / sequences);
  const float shared = longest - mean * (2 * PREFILL_UNITS - blocks) / blocks;        // context of the longest tile that shares
  if (shared < (kv_fp8 ? 0.75f : 0.7f) * longest) return SHARED;
  const float second = longest - mean + mean * (blocks - PREFILL_UNITS) / blocks;
  return second < 0.63f * longest - 180.f ? ROUNDS : ONE;
}

void launch_paged_prefill(const void* q, int64_t q_stride, const void* k_cache, const void* v_cache,
                          const int* block_tables, int max_blocks, const int* seq_lens, const int* query_start_loc,
                          const int* tile_seq, const int* tile_q0, int num_tiles, void* out, int64_t out_stride, int Hq,
                          int Hkv, float scale, bool kv_fp8, float k_scale, float v_scale, const float* kv_scales,
                          const int* counts, int longest, int sequences, hipStream_t stream) {
  if (num_tiles == 0) return;
  if (kv_scales != nullptr) k_scale = v_scale = 1.f;
  const float scale_log2 = scale * 1.4426950408889634f * (kv_fp8 ? k_scale : 1.f);
  const int form = prefill_page_groups(num_tiles, Hkv, Hq / Hkv, longest, sequences, kv_fp8), groups = form == 1 ? 1 : 2;
  const int units = form == 3 ? PREFILL_UNITS : num_tiles * Hkv;
  const dim3 grid(std::min(num_tiles * Hkv, units));
#define DLI_PREFILL_GO(KV8_, G_, N_)                                                                                              \
  hipLaunchKernelGGL((paged_prefill_kernel<KV8_, G_, N_>), grid, dim3(256 * G_), 0, stream, (const uint16_t*)q, q_stride, k_cache, v_cache, \
                     block_tables, max_blocks, seq_lens, query_start_loc, tile_seq, tile_q0, (uint16_t*)out, out_stride, Hq, Hkv, num_tiles, \
                     scale_log2, KV8_ ? v_scale : 1.f, KV8_ ? kv_scales : nullptr, counts, units)
  if (kv_fp8) { if (groups == 2) DLI_PREFILL_GO(true, 2, 2); else DLI_PREFILL_GO(true, 1, 1); }
  else { if (groups == 2) DLI_PREFILL_GO(false, 2, 1); else DLI_PREFILL_GO(false, 1, 1); }
#undef DLI_PREFILL_GO
}

// Page groups of a mixed step's tiles (paged_mixed_kernel), 0: launches of their own.  rows: decode rows; longest, sequences as in prefill_page_groups.
// The rule compares what the forms should take, in µs:
//   * the longest tile's chain, with one and two groups as measured with 8/1 heads at 250 to 3500 tokens;
//   * the decode rows by themselves: 5, and their pages' bytes at 5.5 TB/s.  `longest` may be a prompt's, so the rows are taken for half of it, 800 tokens at most;
//   * one launch of one group: its chain and 0.4 of the rows' time, or what the rows take;
//   * one of two groups, a workgroup a unit: its chain, 0.15 of the rows' time and what the units without a tile leave of them (such a unit reads 2.2 of its
//     share), or 1.15 of the rows' time.
// Past 256 tiles, where their own launch may have two groups, one launch of one group pays if it hides rows of some length.
// Measured, after each other / one group / two:
//   8/1 heads, one prompt of 2000 behind 500 (125 tiles): 16 bf16 rows of up to 1500 64.0 / 75.9 / 59.6, e4m3 65.8 / 80.6 / 61.4, 400 bf16 89.2 / 86.8 / 60.7;
//   64/8, one of 500 behind 1500 (256), bf16: 16 rows 68.7 / 67.9 / 60.3, 96 104 / 82.9 / 103;
//   64/8, one of 400 behind 500 (200), e4m3: 48 rows 49.5 / 40.8 / 39.3, 96 58.3 / 40.2 / 49.1 (two are taken);
//   32/8, two of up to 1024 behind up to 1024 (296), e4m3: 16 rows 49.4 / 50.6 / 41.1, 96 66.9 / 49.8 / 60.7.
// Long rows are taken for short ones, and a long row's context for the chain of a short chunk's tiles.  That costs no step more than launches of its own
// would (336 steps with rows of 4000 to 16000 tokens: 0.83 of them on average, at most 1.03), but it is not the best form: 64 rows of up to 16000 beside 1000
// behind 6000 (256 tiles), where two groups are taken, bf16 532 / 418 / 498, e4m3 362 / 245 / 355; beside 40 behind 3000, e4m3 278 / 209 / 214.
// (More: profiles/mixed_steps_one_launch.txt.)
int mixed_page_groups(int num_tiles, int Hkv, int G, int longest, int sequences, int rows, bool kv_fp8) {
  const int blocks = num_tiles * Hkv;
  const bool two = prefill_page_groups(num_tiles, Hkv, G, longest, sequences, kv_fp8) != 1;
  if (longest == 0) return two ? 2 : 1;                       // (up to 256 tiles: at most 1.05 of launches of their own)
  const float one_us = 5.f + (kv_fp8 ? 0.03f : 0.0277f) * longest;
  const float two_us = longest > 224 ? 5.5f + 0.0207f * longest : one_us;      // short tiles are done by one group in either form
  const float rows_us = 5.f + (float)rows * std::min(longest / 2, 800) * Hkv * (kv_fp8 ? 256.f : 512.f) / 5.5e6f;
  if (blocks > PREFILL_UNITS) return two && rows_us < one_us / 2.2f ? 0 : 1;
  const float idle = (float)(PREFILL_UNITS - blocks) / PREFILL_UNITS;
  const float with_two = std::max(two_us + 0.15f * rows_us + std::max(0.f, rows_us - 2.2f * idle * two_us), 1.15f * rows_us);
  return with_two < std::max(one_us + 0.4f * rows_us, rows_us + 4.f) ? 2 : 1;
}

// Decode rows as launch_paged_decode_worklist (work != nullptr: `items`, `reds`) or as launch_paged_decode (`num_seqs`, `num_splits`) takes them, prompt
// tiles as launch_paged_prefill does.
void launch_paged_mixed(const void* q, int64_t q_stride, const void* k_cache, const void* v_cache, const int* block_tables, int max_blocks,
                        const int* seq_lens, const int* query_start_loc, const int* tile_seq, const int* tile_q0, int num_tiles, void* out,
                        int64_t out_stride, float* part_o, float* part_ml, const int* work, const int* red, const int* counts, int items, int reds,
                        int num_seqs, int num_splits, int Hq, int Hkv, float scale, bool kv_fp8, float k_scale, float v_scale, const float* kv_scales,
                        bool tiles_on_device, int longest, int sequences, hipStream_t stream) {
  const bool wl = work != nullptr;
  if (!wl) items = num_seqs * num_splits;
  int groups = std::max(1, mixed_page_groups(num_tiles, Hkv, Hq / Hkv, longest, sequences, num_seqs, kv_fp8));
  if (groups == 2 && !kv_fp8 && decode_waves(false, Hq / Hkv, (int64_t)Hkv * items) != 8) groups = 1;
  const int rows = groups == 2 && kv_fp8 ? (items + 1) / 2 : items;
  const int64_t octets = ((int64_t)num_tiles * Hkv + 7) / 8 + ((int64_t)rows * Hkv + 7) / 8;
  if (octets == 0) return;
  if (kv_scales != nullptr) k_scale = v_scale = 1.f;
  const float scale_log2 = scale * 1.4426950408889634f * (kv_fp8 ? k_scale : 1.f);
#define DLI_MIXED_GO(KV8_, WL_, G_, NT_)                                                                                                 \
  hipLaunchKernelGGL((paged_mixed_kernel<KV8_, WL_, G_, NT_>), dim3((unsigned)(8 * octets)), dim3(256 * G_), 0, stream, (const uint16_t*)q, q_stride,  \
                     k_cache, v_cache, block_tables, max_blocks, seq_lens, query_start_loc, tile_seq, tile_q0, (uint16_t*)out, out_stride, part_o, part_ml, \
                     Hq, Hkv, num_tiles, items, wl ? 1 : num_splits, scale_log2, KV8_ ? v_scale : 1.f, KV8_ ? kv_scales : nullptr, (const int4*)work,  \
                     counts, tiles_on_device ? 1 : 0)
#define DLI_MIXED_NT(KV8_, WL_, G_) do { if (g_decode_nt) DLI_MIXED_GO(KV8_, WL_, G_, true); else DLI_MIXED_GO(KV8_, WL_, G_, false); } while (0)
#define DLI_MIXED_WL(KV8_, G_) do { if (wl) DLI_MIXED_NT(KV8_, true, G_); else DLI_MIXED_NT(KV8_, false, G_); } while (0)
  if (groups == 2) { if (kv_fp8) DLI_MIXED_WL(true, 2); else DLI_MIXED_WL(false, 2); }
  else { if (kv_fp8) DLI_MIXED_WL(true, 1); else DLI_MIXED_WL(false, 1); }
#undef DLI_MIXED_WL
#undef DLI_MIXED_NT
#undef DLI_MIXED_GO
  if (wl ? reds > 0 : num_splits > 1)
    hipLaunchKernelGGL(decode_reduce_kernel, dim3(wl ? reds : num_seqs, Hq), dim3(128), 0, stream, part_o, part_ml, (uint16_t*)out,
                       out_stride, Hq, wl ? 1 : num_splits, kv_fp8 ? v_scale : 1.f, kv_fp8 ? kv_scales : nullptr, Hkv,
                       wl ? (const int4*)red : nullptr, wl ? counts : nullptr);
}

}  // namespace dli

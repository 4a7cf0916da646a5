// K2: NeoX rotate-half RoPE on q and k fused with the paged-KV write.
//
// Work items are 8-element (16-byte) chunks: a q/k item owns
// the pair (x[d0:d0+8], x[d0+64:d0+72]) of one head, so both halves of the rotation are produced by
// the same thread; cos/sin come from a host-built fp32 table (no device trig).  Rotated k goes back
// into the qkv buffer (the prefill kernel reads everything from the cache, but the in-place result
// keeps the op's semantics testable) and into the K page as one 16-byte store per chunk; v goes into
// the transposed, slot-permuted V page (layout: ops/kv_layout.py).
//
// KV8 = true stores the cache as OCP e4m3 with per-tensor scales (value / scale, saturating).
#include <algorithm>

#include "common.h"
#include "kernels.h"

namespace dli {

constexpr int D = 128;

__device__ __forceinline__ int v_slot(int t) { return ((t & 15) >> 2) * 8 + (t >> 4) * 4 + (t & 3); }

// q/k of one token: thread = (chunk j of the half-row, head hg; hg + step, … where a workgroup has fewer threads than that); lanes j = 0..7 of a
// head cover 128 contiguous bytes, the 8 heads of a wave 8 such lines: every load and store is whole cache lines.
template <bool KV8>
__device__ __forceinline__ void turn_heads(uint16_t* row, int pos, const float* cos_sin, int slot, void* k_cache_, int Hq, int Hkv,
                                           float k_inv_scale_, const float* kv_scales, int hg, int step) {
  const int j = threadIdx.x & 7;
  f32x4 c0, c1, s0, s1;
  if (cos_sin != nullptr) {
    const float* cs = cos_sin + (int64_t)pos * D + j * 8;
    c0 = *reinterpret_cast<const f32x4*>(cs);
    c1 = *reinterpret_cast<const f32x4*>(cs + 4);
    s0 = *reinterpret_cast<const f32x4*>(cs + 64);
    s1 = *reinterpret_cast<const f32x4*>(cs + 68);
  }
  for (int head = hg; head < Hq + Hkv; head += step) {
    uint16_t* p = row + head * D + j * 8;
    bf16x8 a = *reinterpret_cast<const bf16x8*>(p);
    bf16x8 b = *reinterpret_cast<const bf16x8*>(p + 64);
    if (cos_sin != nullptr) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float c = e < 4 ? c0[e] : c1[e - 4], sn = e < 4 ? s0[e] : s1[e - 4];
        const float x1 = bf2f((uint16_t)a[e]), x2 = bf2f((uint16_t)b[e]);
        a[e] = (short)f2bf(x1 * c - x2 * sn);
        b[e] = (short)f2bf(x2 * c + x1 * sn);
      }
      *reinterpret_cast<bf16x8*>(p) = a;
      *reinterpret_cast<bf16x8*>(p + 64) = b;
    }
    if (head >= Hq && slot >= 0) {             // k head → K page
      const int h = head - Hq, blk = slot >> 5, tok = slot & 31;
      const int64_t page = (int64_t)blk * Hkv + h;
      if (!KV8) {
        uint16_t* kc = reinterpret_cast<uint16_t*>(k_cache_) + page * (D * 32);
        const int d0 = j * 8, d1 = 64 + j * 8;   // chunk c = d/32, offset d%32
        *reinterpret_cast<bf16x8*>(kc + ((d0 >> 5) * 32 + tok) * 32 + (d0 & 31)) = a;
        *reinterpret_cast<bf16x8*>(kc + ((d1 >> 5) * 32 + tok) * 32 + (d1 & 31)) = b;
      } else {
        uint8_t* kc = reinterpret_cast<uint8_t*>(k_cache_) + page * (D * 32);
        const float k_inv_scale = kv_scales != nullptr ? fast_rcp(kv_scales[h]) : k_inv_scale_;
        uint64_t pa = 0, pb = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          pa |= (uint64_t)f_to_fp8(bf2f((uint16_t)a[e]) * k_inv_scale) << (8 * e);
          pb |= (uint64_t)f_to_fp8(bf2f((uint16_t)b[e]) * k_inv_scale) << (8 * e);
        }
        // chunk c = d/64: first half is chunk 0, second half chunk 1
        *reinterpret_cast<uint64_t*>(kc + (0 * 32 + tok) * 64 + j * 8) = pa;
        *reinterpret_cast<uint64_t*>(kc + (1 * 32 + tok) * 64 + j * 8) = pb;
      }
    }
  }
}

// eight v entries (d0 …) of one head for N tokens that sit in neighbouring slots from `slot` on (N = 4: slot a multiple of 4)
template <bool KV8, int N>
__device__ __forceinline__ void put_values(const uint16_t* v, int64_t row_stride, int slot, int h, int d0, int Hkv, void* v_cache_,
                                           float v_inv_scale_, const float* kv_scales) {
  bf16x8 x[N];
#pragma unroll
  for (int i = 0; i < N; ++i) x[i] = *reinterpret_cast<const bf16x8*>(v + i * row_stride + h * D + d0);
  const int64_t at = ((int64_t)(slot >> 5) * Hkv + h) * (D * 32) + d0 * 32 + v_slot(slot & 31);
  if (!KV8) {
    uint16_t* vc = reinterpret_cast<uint16_t*>(v_cache_) + at;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if constexpr (N == 4) *reinterpret_cast<bf16x4*>(vc + e * 32) = bf16x4{x[0][e], x[1][e], x[2][e], x[3][e]};
      else vc[e * 32] = (uint16_t)x[0][e];
    }
  } else {
    uint8_t* vc = reinterpret_cast<uint8_t*>(v_cache_) + at;
    const float v_inv_scale = kv_scales != nullptr ? fast_rcp(kv_scales[Hkv + h]) : v_inv_scale_;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      uint32_t w = 0;
#pragma unroll
      for (int i = 0; i < N; ++i) w |= (uint32_t)f_to_fp8(bf2f((uint16_t)x[i][e]) * v_inv_scale) << (8 * i);
      if constexpr (N == 4) *reinterpret_cast<uint32_t*>(vc + e * 32) = w;
      else vc[e * 32] = (uint8_t)w;
    }
  }
}

// v_groups == 0 (few tokens: pure latency): workgroup t does everything of token t.  Otherwise workgroups 0 … 8·ceil(v_groups / 8) − 1
// write the v entries of VT tokens each and the others turn the q and k of `per` tokens.  Many small workgroups are what the in-place rotation
// needs: with four tokens and their v in one, whose loads, stores and loads again wait for each other, 4100 tokens of 32 + 8
// heads in five prompts (109 MB) took 33 µs; now 22 (VT = 8: 24.5, 16: 26.5), 740 tokens of twenty 9.6 → 6.6.  A workgroup has a thread for every
// chunk of its tokens' heads (up to 1024), so that nobody has a second head to wait for and few are idle: with 256 threads for any number of
// heads 8 + 1 heads of 4096 tokens took 7.4 µs (four tokens a workgroup 6.2; now 6.3), one token of 32 + 8 3.7 → 3.4.  Rows that arrive from memory, one prompt of
// 4096 tokens, four tokens a workgroup / 256 threads / now: 32 + 8 heads 29.9 / 30.9 / 29.8, 64 + 8 44.3 / 44.4 / 41.9, 2047 tokens 17.0 / 18.0 / 17.4.
// (Two or four tokens a thread: 5 and 20 % slower.)
//   v: tokens 4k…4k+3 of a page occupy 4 ADJACENT slots of every d row (v_slot), so a prefill chunk — whose tokens sit in consecutive
// cache slots — is written with one 8-byte store per (d row, 4 tokens) instead of four 2-byte ones.  The groups of four go by SLOTS: the second
// prompt of a step starts at any row of the batch (groups of four batch rows left most prompts to 2-byte stores: 21 µs for 16 MB of v).  A
// 64-byte row of a V page is completed by eight such stores: XCD x takes the x-th eighth of the tokens, so they meet in one L2 instead of
// leaving as partial lines of eight.
constexpr int VT = 4;
template <bool KV8>
__global__ __launch_bounds__(1024) void rope_cache_kernel(uint16_t* __restrict__ qkv, int64_t row_stride,
                                                         const int* __restrict__ positions,
                                                         const float* __restrict__ cos_sin,  // [max_pos, D] or null
                                                         const int* __restrict__ slot_mapping,
                                                         void* __restrict__ k_cache, void* __restrict__ v_cache,
                                                         int T, int Hq, int Hkv, float k_inv_scale, float v_inv_scale,
                                                         const float* __restrict__ kv_scales,   // [k | v][Hkv] or null
                                                         int v_groups, int per) {
  const int v_blocks = (v_groups + 7) & ~7;
  const uint16_t* v0 = qkv + (int64_t)(Hq + Hkv) * D;
  const int vi_count = Hkv * (D / 8);
  if ((int)blockIdx.x < v_blocks) {
    const int grp = (int)(blockIdx.x & 7) * (v_blocks >> 3) + (int)(blockIdx.x >> 3);
    const int t0 = grp * VT;
    for (int it = threadIdx.x; it < VT * vi_count; it += blockDim.x) {
      const int t = t0 + it / vi_count, vi = it % vi_count, h = vi >> 4, d0 = (vi & 15) * 8;
      if (t >= T) break;
      // one token of every run of up to four neighbouring slots inside a group writes for all of them
      const int slot = slot_mapping[t], before = t > 0 ? slot_mapping[t - 1] : -2;
      int next[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) next[i] = t + 1 + i < T ? slot_mapping[t + 1 + i] : -1;
      if (slot < 0 || ((slot & 3) != 0 && before == slot - 1)) continue;
      int n = 1;
#pragma unroll
      for (int i = 0; i < 3; ++i) n += n == i + 1 && ((slot + n) & 3) != 0 && next[i] == slot + n ? 1 : 0;
      const uint16_t* v = v0 + t * row_stride;
      if (n == 4) {
        put_values<KV8, 4>(v, row_stride, slot, h, d0, Hkv, v_cache, v_inv_scale, kv_scales);
      } else {
        for (int i = 0; i < n; ++i) put_values<KV8, 1>(v + i * row_stride, row_stride, slot + i, h, d0, Hkv, v_cache, v_inv_scale, kv_scales);
      }
    }
    return;
  }
  const int heads = Hq + Hkv, hg = threadIdx.x >> 3, in = per == 1 ? 0 : hg / heads;
  const int t = ((int)blockIdx.x - v_blocks) * per + in;
  if (t >= T || in >= per) return;
  const int slot = slot_mapping[t];
  turn_heads<KV8>(qkv + t * row_stride, positions[t], cos_sin, slot, k_cache, Hq, Hkv, k_inv_scale, kv_scales, hg - in * heads,
                  per == 1 ? blockDim.x >> 3 : heads);
  if (v_groups == 0 && slot >= 0)
    for (int vi = threadIdx.x; vi < vi_count; vi += blockDim.x)
      put_values<KV8, 1>(v0 + t * row_stride, row_stride, slot, vi >> 4, (vi & 15) * 8, Hkv, v_cache, v_inv_scale, kv_scales);
}

void launch_rope_and_cache(void* qkv, int64_t row_stride, const int* positions, const float* cos_sin,
                           const int* slot_mapping, void* k_cache, void* v_cache, int T, int Hq, int Hkv,
                           bool kv_fp8, float k_scale, float v_scale, const float* kv_scales, hipStream_t stream) {
  if (T == 0) return;
  const int v_groups = T <= 128 ? 0 : (T + VT - 1) / VT;
  const int chunks = (Hq + Hkv) * 8, per = v_groups == 0 ? 1 : std::max(1, 256 / chunks);
  const int threads = std::min(1024, (per * chunks + 63) / 64 * 64);
  const dim3 grid((v_groups + 7) / 8 * 8 + (T + per - 1) / per);
#define DLI_ROPE(KV8_, ks_, vs_)                                                                                        \
  hipLaunchKernelGGL((rope_cache_kernel<KV8_>), grid, dim3(threads), 0, stream, (uint16_t*)qkv, row_stride, positions, cos_sin, slot_mapping, \
                     k_cache, v_cache, T, Hq, Hkv, ks_, vs_, kv_fp8 ? kv_scales : nullptr, v_groups, per)
  if (kv_fp8) DLI_ROPE(true, 1.f / k_scale, 1.f / v_scale);
  else DLI_ROPE(false, 1.f, 1.f);
#undef DLI_ROPE
}

// K9 helper: device-side page copy for copy-on-write (pairs = [n, 2] int32: src, dst page ids).
__global__ void copy_pages_kernel(uint8_t* __restrict__ cache, const int* __restrict__ pairs, int64_t page_bytes) {
  const int64_t src = pairs[2 * blockIdx.x], dst = pairs[2 * blockIdx.x + 1];
  const uint4* s = reinterpret_cast<const uint4*>(cache + src * page_bytes);
  uint4* d = reinterpret_cast<uint4*>(cache + dst * page_bytes);
  for (int64_t i = threadIdx.x; i < page_bytes / 16; i += blockDim.x) d[i] = s[i];
}

void launch_copy_pages(void* cache, const int* pairs, int n_pairs, int64_t page_bytes, hipStream_t stream) {
  if (n_pairs == 0) return;
  hipLaunchKernelGGL(copy_pages_kernel, dim3(n_pairs), dim3(256), 0, stream, (uint8_t*)cache, pairs, page_bytes);
}

}  // namespace dli

// K6: temperature / top-k / top-p / multinomial sampling, sort-free.
//
//   * temperature == 0          → arg-max (lowest index on ties).
//   * top_k == 0 && top_p >= 1  → Gumbel-max draw  argmax_i(x_i / T + g_i) (shift invariant, so neither the row max nor the
//                                  softmax sum is needed).
//   * otherwise                 → a cut-off on the logit instead of a sort, then the Gumbel-max draw over what reaches it.
//
// Serving path (bf16 rows of up to 131072 logits, 16-byte aligned): sample_cut_kernel finds the cut-off key of the rows that need
// one, sample_draw_kernel draws with a row's slices spread over the chip; rows of up to 8192 logits are done by sample_whole_kernel alone.
// Other rows (fp32, unaligned, longer) take
// sample_kernel: one 1024-thread workgroup per row, cut-off by a 4-pass radix descent (8 bits per pass, 256-bin LDS histogram of
// *counts* for top-k, of *probability mass* for top-p).
// Gumbel noise comes from Philox4x32-10 keyed by the request seed, counter = (element/4, step), so a
// request's draw is independent of the batch it happens to share; a `noise` tensor can be supplied
// instead (tests: bit-exact comparison against the torch reference with the same uniforms).
// Ties at the cut-off key are all kept (the torch reference keeps as many as needed) — only
// observable when several tokens share the exact same logit at the nucleus boundary.
#include "common.h"
#include "kernels.h"

namespace dli {

constexpr int SNT = 1024;

__device__ __forceinline__ uint32_t okey(float f) {   // monotone float → uint
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ uint32_t mulhilo(uint32_t a, uint32_t b, uint32_t& hi) {
  const uint64_t p = (uint64_t)a * b;
  hi = (uint32_t)(p >> 32);
  return (uint32_t)p;
}
__device__ __forceinline__ uint4 philox4x32_10(uint4 ctr, uint2 key) {
#pragma unroll
  for (int i = 0; i < 10; ++i) {
    uint32_t hi0, hi1;
    const uint32_t lo0 = mulhilo(0xD2511F53u, ctr.x, hi0);
    const uint32_t lo1 = mulhilo(0xCD9E8D57u, ctr.z, hi1);
    ctr = make_uint4(hi1 ^ ctr.y ^ key.x, lo1, hi0 ^ ctr.w ^ key.y, lo0);
    key.x += 0x9E3779B9u;
    key.y += 0xBB67AE85u;
  }
  return ctr;
}
__device__ __forceinline__ float u01(uint32_t r) { return ((r >> 8) + 0.5f) * (1.0f / 16777216.0f); }   // (0,1)
// Logarithm of a normal number whose logarithm is finite.  It gives the bits of __logf, which also scales subnormal numbers and lets infinities by: 6
// instructions, not 14.  ln 2 in two floats, and the order of the products, are those that this compiler emits for __logf (read from this file's
// assembly): y·hi + (y·lo + what y·hi lost), the first product unrounded as well, so that its rounding counts twice there and here.  -log(-log(u)) of all
// 2^24 numbers that u01 gives has the same bits either way.
__device__ __forceinline__ float log_normal(float x) {
  const float hi = __uint_as_float(0x3F317217u), lo = __uint_as_float(0x3377D1CFu), y = __builtin_amdgcn_logf(x);
  return __builtin_fmaf(y, hi, __builtin_fmaf(y, lo, __builtin_fmaf(y, hi, -(y * hi))));
}
// Gumbel noise of 32 random bits, for every kernel here: paths that pick the same token need the same bits.  u01 gives 2^-25 … 1, so -log(u) is 0 or at
// least 2^-24.
__device__ __forceinline__ float gumbel_of(uint32_t r) {
  const float t = -log_normal(u01(r));
  return t == 0.f ? __builtin_inff() : -log_normal(t);
}
// of a caller's number, which may be any
__device__ __forceinline__ float gumbel_at(float u) { return -__logf(-__logf(u)); }

struct ArgMax {
  float v;
  int i;
};

// A row of NaN logits never beats the initial candidate and leaves its out-of-range index behind: the next step would
// use it as an embedding row (a GPU fault).  Such a row yields token 0 instead; the NaN itself is the caller's bug.
__device__ __forceinline__ int valid_token(int i, int V) { return (unsigned)i < (unsigned)V ? i : 0; }
__device__ __forceinline__ ArgMax amax(ArgMax a, ArgMax b) {
  return (b.v > a.v || (b.v == a.v && b.i < a.i)) ? b : a;
}
__device__ ArgMax block_argmax(ArgMax a, float* sv, int* si) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    ArgMax b{__shfl_xor(a.v, o, 64), __shfl_xor(a.i, o, 64)};
    a = amax(a, b);
  }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { sv[w] = a.v; si[w] = a.i; }
  __syncthreads();
  ArgMax r{sv[0], si[0]};
  for (int k = 1; k < SNT / 64; ++k) r = amax(r, ArgMax{sv[k], si[k]});
  __syncthreads();
  return r;
}
__device__ float block_max(float v, float* sv) {
  v = wave_max(v);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) sv[w] = v;
  __syncthreads();
  float r = sv[0];
  for (int k = 1; k < SNT / 64; ++k) r = fmaxf(r, sv[k]);
  __syncthreads();
  return r;
}

template <typename T>
__device__ __forceinline__ float ld(const T* p, int i);
template <>
__device__ __forceinline__ float ld<uint16_t>(const uint16_t* p, int i) { return bf2f(p[i]); }
template <>
__device__ __forceinline__ float ld<float>(const float* p, int i) { return p[i]; }

// Radix descent.  MASS = false: find the key of the k-th largest element (target = k, weights 1).
// MASS = true : find the largest key K with  mass(key >= K) >= target   (weights exp2(z - zmax)).
// Only elements with key >= floor_key take part.  Returns the cut-off key.
template <typename T, bool MASS>
__device__ uint32_t radix_cut(const T* row, int V, float inv_t_log2, float zmax, float target, uint32_t floor_key,
                              float* hist, uint32_t* s_pick, float* s_rem) {
  uint32_t prefix = 0, prefix_mask = 0;
  float remaining = target;
  for (int shift = 24; shift >= 0; shift -= 8) {
    for (int i = threadIdx.x; i < 256; i += SNT) hist[i] = 0.f;
    __syncthreads();
    for (int i = threadIdx.x; i < V; i += SNT) {
      const float z = ld<T>(row, i) * inv_t_log2;
      const uint32_t k = okey(z);
      if (k >= floor_key && (k & prefix_mask) == prefix)
        atomicAdd(&hist[(k >> shift) & 255], MASS ? fast_exp2(z - zmax) : 1.f);
    }
    __syncthreads();
    if (threadIdx.x == 0) {   // walk the bins from the top until the running total reaches the target
      float acc = 0.f;
      int bin = 255;
      for (; bin > 0; --bin) {
        if (acc + hist[bin] >= remaining) break;
        acc += hist[bin];
      }
      *s_pick = (uint32_t)bin;
      *s_rem = remaining - acc;
    }
    __syncthreads();
    prefix |= (*s_pick) << shift;
    prefix_mask |= 255u << shift;
    remaining = *s_rem;
    __syncthreads();
  }
  return prefix;
}

template <typename T>
__global__ __launch_bounds__(SNT) void sample_kernel(const T* __restrict__ logits, int64_t row_stride, int V,
                                                     const float* __restrict__ temperature, const float* __restrict__ top_p,
                                                     const int* __restrict__ top_k, const int64_t* __restrict__ seeds,
                                                     const int64_t* __restrict__ steps, const float* __restrict__ noise,
                                                     int64_t* __restrict__ out) {
  __shared__ float sv[SNT / 64];
  __shared__ int si[SNT / 64];
  __shared__ float hist[256];
  __shared__ uint32_t s_pick;
  __shared__ float s_rem;

  const int b = blockIdx.x;
  const T* row = logits + (int64_t)b * row_stride;
  const float temp = temperature[b];

  if (temp <= 0.f) {
    ArgMax a{-3.0e38f, 0x7fffffff};
    for (int i = threadIdx.x; i < V; i += SNT) a = amax(a, ArgMax{ld<T>(row, i), i});
    a = block_argmax(a, sv, si);
    if (threadIdx.x == 0) out[b] = valid_token(a.i, V);
    return;
  }

  const float inv_t_log2 = 1.4426950408889634f / temp;    // z = x / T in log2 units
  const float p = top_p[b];
  int k = top_k[b];
  if (k <= 0 || k > V) k = V;
  uint32_t floor_key = 0;

  if (k < V || p < 1.f) {
    float zmax = -3.0e38f;
    for (int i = threadIdx.x; i < V; i += SNT) zmax = fmaxf(zmax, ld<T>(row, i) * inv_t_log2);
    zmax = block_max(zmax, sv);
    if (k < V) floor_key = radix_cut<T, false>(row, V, inv_t_log2, zmax, (float)k, 0u, hist, &s_pick, &s_rem);
    if (p < 1.f) {
      float tot = 0.f;                                     // mass of what survived top-k
      for (int i = threadIdx.x; i < V; i += SNT) {
        const float z = ld<T>(row, i) * inv_t_log2;
        if (okey(z) >= floor_key) tot += fast_exp2(z - zmax);
      }
      tot = wave_sum(tot);
      if ((threadIdx.x & 63) == 0) sv[threadIdx.x >> 6] = tot;
      __syncthreads();
      tot = 0.f;
      for (int w = 0; w < SNT / 64; ++w) tot += sv[w];
      __syncthreads();
      floor_key = radix_cut<T, true>(row, V, inv_t_log2, zmax, p * tot, floor_key, hist, &s_pick, &s_rem);
    }
  }

  const uint64_t seed = (uint64_t)seeds[b];
  const uint64_t step = (uint64_t)steps[b];
  const uint2 key = make_uint2((uint32_t)seed, (uint32_t)(seed >> 32));
  ArgMax a{-3.0e38f, 0x7fffffff};
  const float ln2 = 0.6931471805599453f;
  for (int i4 = threadIdx.x; i4 * 4 < V; i4 += SNT) {
    uint4 r = make_uint4(0, 0, 0, 0);
    if (noise == nullptr) r = philox4x32_10(make_uint4((uint32_t)i4, (uint32_t)step, (uint32_t)(step >> 32), 0x5A17u), key);
    const uint32_t rr[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = i4 * 4 + e;
      if (i < V) {
        const float z = ld<T>(row, i) * inv_t_log2;
        if (okey(z) >= floor_key) {
          a = amax(a, ArgMax{z * ln2 + (noise != nullptr ? gumbel_at(noise[(int64_t)b * V + i]) : gumbel_of(rr[e])), i});
        }
      }
    }
  }
  a = block_argmax(a, sv, si);
  if (threadIdx.x == 0) out[b] = valid_token(a.i, V);
}

// ---------------------------------------------------------------------------------------------------------------
// bf16 serving path (logits come out of the LM-head GEMM in bf16, V ≤ 131072, V % 8 == 0).
//
// A draw without a cut-off is bound by Philox (≈ 45 µs of integer multiplies when one compute unit does a 128k row) and a cut-off by
// the LDS atomics of its histogram, so neither fits one kernel of a workgroup per row, which leaves most of the chip idle at
// decode batch sizes: B = 57, V = 128256 with a quarter each of greedy, plain, top-p and top-k rows took 239 µs that way.
// ---------------------------------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t okey16(uint32_t h) { return (h & 0x8000u) ? (~h & 0xFFFFu) : (h | 0x8000u); }
__device__ __forceinline__ uint32_t half_of(const uint4& c, int e) {   // e-th bf16 (0..7) of a chunk, compile-time e
  const uint32_t w = e < 2 ? c.x : e < 4 ? c.y : e < 6 ? c.z : c.w;
  return (e & 1) ? (w >> 16) : (w & 0xFFFFu);
}

// The row of a cut-off lives in registers — thread t holds 16-byte chunks t, t+1024, … (8 logits each, packed).
// Every pass re-derives keys and weights from the packed row.  Without this fence the compiler keeps the 128 unpacked
// keys of a thread alive from one pass to the next (CSE) and spills; the empty asm makes the registers opaque.
template <int NCH>
__device__ __forceinline__ void opaque(uint4 (&regs)[NCH]) {
#pragma unroll
  for (int c = 0; c < NCH; ++c) asm volatile("" : "+v"(regs[c].x), "+v"(regs[c].y), "+v"(regs[c].z), "+v"(regs[c].w));
}

// descending walk over 256 bins by one wave: first bin where the running total reaches `remaining`
__device__ __forceinline__ void pick_bin(const float* hist, float remaining, uint32_t* s_pick, float* s_rem) {
  const int lane = threadIdx.x;                       // called by threads 0..63
  float h[4], local = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) { h[j] = hist[255 - 4 * lane - j]; local += h[j]; }
  float incl = local;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float up = __shfl_up(incl, o, 64);
    if (lane >= o) incl += up;
  }
  const uint64_t hit = __ballot(incl >= remaining);
  const int first = hit ? __ffsll((long long)hit) - 1 : 63;
  if (lane == first) {
    float acc = incl - local;
    int j = 0;
    for (; j < 3; ++j) {
      if (acc + h[j] >= remaining) break;
      acc += h[j];
    }
    if (!hit) { j = 3; acc = incl - h[3]; }           // total < remaining (rounding): lowest bin, like the serial walk
    *s_pick = (uint32_t)(255 - 4 * lane - j);
    *s_rem = remaining - acc;
  }
}

// Exact for any row, two 8-bit passes over the 16-bit keys; the fallback of cut_by_counts.  A thread adds runs of equal bins to the
// LDS histogram with one atomic.
template <int NCH, bool MASS>
__device__ __forceinline__ uint32_t radix_cut16(uint4 (&regs)[NCH], float inv_t_log2, float zmax, float target, uint32_t floor_key,
                                float* hist, uint32_t* s_pick, float* s_rem) {
  uint32_t prefix = 0;
  float remaining = target;
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int shift = pass == 0 ? 8 : 0;
    for (int i = threadIdx.x; i < 256; i += SNT) hist[i] = 0.f;
    __syncthreads();
    opaque(regs);
    int cur_bin = -1;
    float cur = 0.f;
#pragma clang loop unroll(full)
    for (int c = 0; c < NCH; ++c) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t h = half_of(regs[c], e);
        const uint32_t k = okey16(h);
        const bool take = k >= floor_key && (pass == 0 || (k >> 8) == (prefix >> 8));
        if (take) {
          const float w = MASS ? fast_exp2(bf2f((uint16_t)h) * inv_t_log2 - zmax) : 1.f;
          const int bin = (int)((k >> shift) & 255u);
          if (bin == cur_bin) {
            cur += w;
          } else {
            if (cur_bin >= 0) atomicAdd(&hist[cur_bin], cur);
            cur_bin = bin;
            cur = w;
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);      // one chunk at a time: keeps the 64 row registers the only long-lived ones
    }
    if (cur_bin >= 0) atomicAdd(&hist[cur_bin], cur);
    __syncthreads();
    if (threadIdx.x < 64) pick_bin(hist, remaining, s_pick, s_rem);
    __syncthreads();
    prefix |= (*s_pick) << shift;
    remaining = *s_rem;
    __syncthreads();
  }
  return prefix;
}

// ---- cut-off by counting.  One pass adds the logits of the row to a histogram of COUNTS with a bin per bf16 value: magnitudes from
// the largest that matters down 32 octaves (MBINS = 32 · 128 mantissa steps) for either sign, smaller ones share the bin at zero.  What
// matters: the row's largest VALUE, and below it whatever has a weight in fp32 (2^-128); logits farther down (masked tokens: −inf, the
// type's lowest value, −1e9) stay outside the bins: as bins they would push the row's ordinary logits into the shared one, and half a row
// of equal masks meets in one word (57 rows of 128256, half masked with the lowest value: 246 µs then, 37 now).  Logits
// spread over hundreds of such bins, so the LDS atomics hardly collide (bins of the upper 8 key bits put a softmax-shaped row
// into five or six), and a bin's probability mass is count · exp2(z − zmax): top-k and top-p read the same histogram, each sum in a
// fixed order.  The logits of the shared bin count as ± its bound there: at most 2^-32 of max(|zmax|, 128 − zmax), i.e. a relative error of
// 1e-7 where their weights are not zero beside the largest.  A cut-off inside the shared bin, or a row with +inf or NaN, is left to
// radix_cut16; one outside the bins too, unless all logits there are equal.  The atomics and the row's
// arrival at one compute unit bound it: 20 µs a launch at V = 128256 up to 256 filtered rows (radix descents of the whole row: 235).
// Position d runs from the largest value down: positive magnitude index c at MBINS − 1 − c, negative at MBINS + c.
constexpr int MBINS = 4096;
constexpr int BINS_PER_THREAD = 2 * MBINS / SNT;
static_assert(BINS_PER_THREAD == 8, "scan_cut reads a thread's bins as two 16-byte words");
// position of the logit in half `odd` of a word: MBINS + i for a negative one, MBINS - 1 - i = MBINS + ~i for another, i = max(magnitude - lo, 0).  Five
// instructions a logit with the address; rotated positions and maxima of values, one logit at a time, took twice as many (V = 128256: a launch 22.5 → 20 µs).
template <int ODD> __device__ __forceinline__ int bin_of(uint32_t word, int lo) {
  const uint32_t mag = __builtin_amdgcn_ubfe(word, 16 * ODD, 15);
  const int i = (int)__builtin_elementwise_sub_sat(mag, (uint32_t)lo);
  const int neg = __builtin_amdgcn_sbfe((int)word, 16 * ODD + 15, 1);                // -1: negative
  return MBINS + ~(i ^ neg);
}

struct CutScratch {
  float wave_tot[SNT / 64];
  int first;
  int pick;
};

// position of the first bin where the running weight of the bins up to position d_last reaches `target` (FRACTION: that share of
// their total), or −1
template <bool MASS, bool FRACTION>
__device__ __forceinline__ int scan_cut(const uint32_t* counts, int lo, float inv_t_log2, float zmax, float target, int d_last,
                                        CutScratch* s) {
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  float w[BINS_PER_THREAD], local = 0.f;
  const uint4 c0 = reinterpret_cast<const uint4*>(counts)[2 * t], c1 = reinterpret_cast<const uint4*>(counts)[2 * t + 1];
  const uint32_t cnt[BINS_PER_THREAD] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
#pragma unroll
  for (int j = 0; j < BINS_PER_THREAD; ++j) {
    const int d = t * BINS_PER_THREAD + j;
    const uint32_t n = d <= d_last ? cnt[j] : 0u;
    const int c = d < MBINS ? MBINS - 1 - d : d - MBINS;
    const float x = bf2f((uint16_t)(c + lo)) * (d < MBINS ? inv_t_log2 : -inv_t_log2);
    w[j] = n == 0u ? 0.f : MASS ? (float)n * fast_exp2(x - zmax) : (float)n;
    local += w[j];
  }
  float incl = local;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float up = __shfl_up(incl, o, 64);
    if (lane >= o) incl += up;
  }
  if (lane == 63) s->wave_tot[wave] = incl;
  if (t == 0) { s->first = SNT; s->pick = -1; }
  __syncthreads();
  float before = 0.f, total = 0.f;
#pragma unroll
  for (int k = 0; k < SNT / 64; ++k) {
    const float x = s->wave_tot[k];
    before += k < wave ? x : 0.f;
    total += x;
  }
  const float want = FRACTION ? target * total : target;
  const bool reached = before + incl >= want && local > 0.f;
  const uint64_t hit = __ballot(reached);
  if (hit != 0 && lane == 0) atomicMin(&s->first, wave * 64 + __ffsll((long long)hit) - 1);
  __syncthreads();
  if (t == s->first) {
    float acc = before + (incl - local);
    int pick = -1;
#pragma unroll
    for (int j = 0; j < BINS_PER_THREAD; ++j) {
      if (w[j] > 0.f && (pick < 0 || acc < want)) pick = t * BINS_PER_THREAD + j;   // `want` was not reached in front of it
      acc += w[j];
    }
    s->pick = pick;
  }
  __syncthreads();
  const int r = s->pick;
  __syncthreads();
  return r;
}

// per row of the launch: what the draw needs to know, and the words its slices meet in (a cache line each: the atomics of eight rows on
// one line wait for each other)
struct alignas(128) SampleRow {
  unsigned long long best;     // (ordered value, ~index) of the best candidate so far
  uint32_t cut;                // smallest 16-bit key that takes part
  uint32_t done;               // slices that have delivered
};

// a row's logits into its bins; those outside (FAR): `far_any`, `far_all` are equal where they have one value only
template <int NCH, bool FAR>
__device__ __forceinline__ void count_logits(uint4 (&regs)[NCH], int nchunks, int top, int lo, uint32_t* counts, uint32_t& far_any,
                                             uint32_t& far_all) {
#pragma clang loop unroll(full)
  for (int c = 0; c < NCH; ++c) {
    if (c * SNT + (int)threadIdx.x < nchunks) {
      const uint32_t words[4] = {regs[c].x, regs[c].y, regs[c].z, regs[c].w};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t word = words[e >> 1];
        const int d = e & 1 ? bin_of<1>(word, lo) : bin_of<0>(word, lo);
        if (FAR) {
          const int m = (int)((e & 1 ? word >> 16 : word) & 0x7FFFu);
          if (m > top) {
            far_any |= (uint32_t)m;
            far_all &= (uint32_t)m;
            continue;
          }
        }
        atomicAdd(&counts[d], 1u);
      }
    }
    __builtin_amdgcn_sched_barrier(0);        // one chunk at a time: keeps the row registers the only long-lived ones
  }
}

struct CutShared {
  alignas(16) uint32_t counts[2 * MBINS];
  float sv[SNT / 64];
  CutScratch cs;
  uint32_t pick;
  float rem;
};
static_assert(alignof(CutShared) % 16 == 0, "scan_cut reads the counts 16 bytes at a time");

// what a row asks for; k is set to V where there is no top-k
__device__ __forceinline__ bool needs_cut(float temp, float p, int& k, int V) {
  if (k <= 0 || k > V) k = V;
  return temp > 0.f && (k < V || p < 1.f);
}

template <int NCH>
__device__ __forceinline__ void load_row(uint4 (&regs)[NCH], const uint16_t* logits, int nchunks) {
  const uint4* row = reinterpret_cast<const uint4*>(logits);
#pragma clang loop unroll(full)
  for (int c = 0; c < NCH; ++c) {
    const int idx = c * SNT + threadIdx.x;
    regs[c] = idx < nchunks ? row[idx] : make_uint4(0xFF80FF80u, 0xFF80FF80u, 0xFF80FF80u, 0xFF80FF80u);   // -inf padding
  }
}

// smallest 16-bit key that takes part
template <int NCH>
__device__ __forceinline__ uint32_t row_cut(uint4 (&regs)[NCH], int nchunks, int V, float temp, float p, int k, CutShared& sh) {
  uint32_t* counts = sh.counts;
  float* sv = sh.sv;
  for (int i = threadIdx.x; i < 2 * MBINS; i += SNT) counts[i] = 0u;

  const float inv_t_log2 = 1.4426950408889634f / temp;    // z = x / T in log2 units
  // Largest value and largest magnitude, two logits an instruction: as signed 16-bit numbers positive logits are in order and above all negative
  // ones, and negative ones are in reverse order.
  typedef short s16x2 __attribute__((ext_vector_type(2)));
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  s16x2 hi2 = {-32768, -32768}, lo2 = {32767, 32767};
  u16x2 mag2 = {0, 0};
#pragma clang loop unroll(full)
  for (int c = 0; c < NCH; ++c) {
    if (c * SNT + (int)threadIdx.x < nchunks) {
      const uint32_t words[4] = {regs[c].x, regs[c].y, regs[c].z, regs[c].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const s16x2 w = __builtin_bit_cast(s16x2, words[e]);
        hi2 = __builtin_elementwise_max(hi2, w);
        lo2 = __builtin_elementwise_min(lo2, w);
        mag2 = __builtin_elementwise_max(mag2, __builtin_bit_cast(u16x2, words[e] & 0x7FFF7FFFu));
      }
    }
  }
  const int hi = (int)block_max((float)max(hi2[0], hi2[1]), sv), low = -(int)block_max(-(float)min(lo2[0], lo2[1]), sv);
  const int mag = (int)block_max((float)max(mag2[0], mag2[1]), sv);         // (whole numbers of 16 bits are exact in fp32)
  float vmax = bf2f((uint16_t)(hi >= 0 ? hi : low));
  if (mag > 0x7F80) {                                       // NaN among them: the largest of the others
    vmax = -3.0e38f;
#pragma clang loop unroll(full)
    for (int c = 0; c < NCH; ++c) {
#pragma unroll
      for (int e = 0; e < 8; ++e) vmax = fmaxf(vmax, bf2f((uint16_t)half_of(regs[c], e)));
    }
    vmax = block_max(vmax, sv);
  }
  vmax = fmaxf(vmax, -3.0e38f);
  const float zmax = vmax * inv_t_log2;
  uint32_t floor_key = 0;                                   // 16-bit key of the raw bf16 logit (x → x/T is monotone)
  bool exact = mag <= 0x7F80 && vmax > -3.0e38f && vmax < 3.4e38f;      // no NaN; a finite maximum
  if (exact) {
    // weights end 128 octaves, 128 · ln 2 · T, below the maximum
    const float span = fmaxf(fabsf(vmax), 88.722839f * temp - vmax);
    const int top = min(min(mag, (int)((__float_as_uint(span) + 0xFFFFu) >> 16)), 0x7F7F), lo = max(top - (MBINS - 1), 0);
    uint32_t far_any = 0, far_all = 0x7FFFu;
    opaque(regs);
    // (a row without logits outside the bins pays no condition per logit: a call of 57 rows of 128256 35.1 against 37.6 µs)
    if (mag > top) count_logits<NCH, true>(regs, nchunks, top, lo, counts, far_any, far_all);
    else count_logits<NCH, false>(regs, nchunks, top, lo, counts, far_any, far_all);
    __syncthreads();
    int d = 2 * MBINS - 1;
    if (k < V) {
      d = scan_cut<false, false>(counts, lo, inv_t_log2, zmax, (float)k, d, &sh.cs);
      if (d < 0) {                                          // among the logits outside the bins, all of them negative: one value?
        const float far_max = block_max((float)far_any, sv), far_min = -block_max(far_any != 0u ? -(float)far_all : -32768.f, sv);
        exact = far_max == far_min;
        floor_key = 0x7FFFu - (uint32_t)far_max;
        d = 2 * MBINS - 1;
      } else {
        exact = !(lo > 0 && (d == MBINS - 1 || d == MBINS));
        floor_key = d < MBINS ? 0x8000u | (uint32_t)(MBINS - 1 - d + lo) : 0x7FFFu - (uint32_t)(d - MBINS + lo);
      }
    }
    if (exact && p < 1.f) {
      d = scan_cut<true, true>(counts, lo, inv_t_log2, zmax, p, d, &sh.cs);
      exact = d >= 0 && !(lo > 0 && (d == MBINS - 1 || d == MBINS));
      floor_key = d < MBINS ? 0x8000u | (uint32_t)(MBINS - 1 - d + lo) : 0x7FFFu - (uint32_t)(d - MBINS + lo);
    }
  }
  if (!exact) {
    floor_key = 0;
    float* hist = reinterpret_cast<float*>(counts);
    if (k < V) floor_key = radix_cut16<NCH, false>(regs, inv_t_log2, zmax, (float)k, 0u, hist, &sh.pick, &sh.rem);
    if (p < 1.f) {
      float tot = 0.f;                                     // mass of what survived top-k
      opaque(regs);
#pragma clang loop unroll(full)
      for (int c = 0; c < NCH; ++c) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t h = half_of(regs[c], e);
          if (okey16(h) >= floor_key) tot += fast_exp2(bf2f((uint16_t)h) * inv_t_log2 - zmax);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      tot = wave_sum(tot);
      if ((threadIdx.x & 63) == 0) sv[threadIdx.x >> 6] = tot;
      __syncthreads();
      tot = 0.f;
      for (int w = 0; w < SNT / 64; ++w) tot += sv[w];
      __syncthreads();
      floor_key = radix_cut16<NCH, true>(regs, inv_t_log2, zmax, p * tot, floor_key, hist, &sh.pick, &sh.rem);
    }
  }
  return floor_key;
}

// ---- draw.  The Philox counter of element i is i/4 exactly as in sample_kernel: all paths draw the same token.
struct DrawArgs {
  const int64_t *seeds, *steps;
  const float* noise;
};
__device__ __forceinline__ ArgMax no_candidate() { return ArgMax{-3.0e38f, 0x7fffffff}; }
// a thread meets its logits in order of index, so an equal one never wins
__device__ __forceinline__ void take(ArgMax& a, float v, int i) {
  if (v > a.v) a = ArgMax{v, i};
}
__device__ __forceinline__ void greedy_chunk(const uint4& x, int chunk, ArgMax& a) {
#pragma unroll
  for (int e = 0; e < 8; ++e) take(a, bf2f((uint16_t)half_of(x, e)), chunk * 8 + e);
}
// Groups of four logits, a Philox block each.  CUT: only what reaches floor_key draws.
template <bool CUT>
__device__ __forceinline__ void draw_chunk(const uint4& x, int chunk, float inv_t_log2, uint32_t floor_key, uint2 key, uint64_t step,
                                           const float* noise_row, ArgMax& a) {
  const float ln2 = 0.6931471805599453f;
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    if (CUT) {
      bool any = false;
#pragma unroll
      for (int e = 0; e < 4; ++e) any = any || okey16(half_of(x, half * 4 + e)) >= floor_key;
      if (!any) continue;                                  // behind a cut-off most groups of four draw nothing
    }
    const int i4 = chunk * 2 + half;
    uint4 r = make_uint4(0, 0, 0, 0);
    if (!CUT || noise_row == nullptr) r = philox4x32_10(make_uint4((uint32_t)i4, (uint32_t)step, (uint32_t)(step >> 32), 0x5A17u), key);
    const uint32_t rr[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t h = half_of(x, half * 4 + e);
      const float z = bf2f((uint16_t)h) * inv_t_log2 * ln2;
      if (!CUT) {
        take(a, z + gumbel_of(rr[e]), i4 * 4 + e);
      } else if (okey16(h) >= floor_key) {
        take(a, z + (noise_row != nullptr ? gumbel_at(noise_row[i4 * 4 + e]) : gumbel_of(rr[e])), i4 * 4 + e);
      }
    }
  }
}
// a thread's best of chunks first, first + stride, …
template <int NC>
__device__ __forceinline__ ArgMax best_of(uint4 (&regs)[NC], int first, int stride, int nchunks, int V, float temp, uint32_t floor_key, int b,
                                          const DrawArgs& draw) {
  ArgMax a = no_candidate();
  if (temp <= 0.f) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if (first + c * stride < nchunks) greedy_chunk(regs[c], first + c * stride, a);
    return a;
  }
  const uint64_t seed = (uint64_t)draw.seeds[b], step = (uint64_t)draw.steps[b];
  const uint2 key = make_uint2((uint32_t)seed, (uint32_t)(seed >> 32));
  const float inv_t_log2 = 1.4426950408889634f / temp;
  const float* noise_row = draw.noise != nullptr ? draw.noise + (int64_t)b * V : nullptr;
  if (floor_key == 0 && noise_row == nullptr) {
    // Every logit draws: no keys and short logarithms (bound by the vector instructions: µs a call, before → now: rows of 128256 1 8.5 → 7.6,
    // 57 18.9 → 15.2, 256 54.9 → 41.5; of 32000 100 12.3 → 10.3).  Behind a cut-off few do: __logf in a branch of its own (without branches 57 rows 30 → 33).
#pragma unroll
    for (int c = 0; c < NC; ++c)
      if (first + c * stride < nchunks) draw_chunk<false>(regs[c], first + c * stride, inv_t_log2, 0u, key, step, nullptr, a);
    return a;
  }
#pragma unroll
  for (int c = 0; c < NC; ++c)
    if (first + c * stride < nchunks) draw_chunk<true>(regs[c], first + c * stride, inv_t_log2, floor_key, key, step, noise_row, a);
  return a;
}
// Rows of up to 8192 logits: a workgroup each, from the logits to the token in one launch.  V = 2048, one row, µs, two launches / one: greedy 6.5 / 4.6,
// plain 8.1 / 5.7, top-p 11.2 / 8.9.  (Rows of 32000 logits would take 17 µs for a plain draw, 8.8 in slices; 512 of them 34 and 31.5.)
__global__ __launch_bounds__(SNT) void sample_whole_kernel(const uint16_t* __restrict__ logits, int64_t row_stride, int V,
                                                           const float* __restrict__ temperature, const float* __restrict__ top_p,
                                                           const int* __restrict__ top_k, DrawArgs draw, int64_t* __restrict__ out) {
  __shared__ CutShared sh;
  __shared__ int si[SNT / 64];
  const int b = blockIdx.x, nchunks = V >> 3;
  const float temp = temperature[b], p = top_p[b];
  int k = top_k[b];
  uint4 regs[1];
  load_row<1>(regs, logits + (int64_t)b * row_stride, nchunks);
  uint32_t floor_key = 0;
  if (needs_cut(temp, p, k, V)) floor_key = row_cut<1>(regs, nchunks, V, temp, p, k, sh);
  const ArgMax a = block_argmax(best_of<1>(regs, threadIdx.x, SNT, nchunks, V, temp, floor_key, b, draw), sh.sv, si);
  if (threadIdx.x == 0) out[b] = valid_token(a.i, V);
}

// Longer rows take two launches, the first of which only clears the words of a row without cut-off.  (That is 1 µs of a greedy row of 32000 logits, 6.7
// instead of the 5.7 of a workgroup a row, which takes 12.1 instead of 7.2 for 128256.  Slices of these rows in the first launch, with no
// words to clear, have the cut-off's registers and LDS and so one workgroup a compute unit: 57 greedy rows of 128256 17 instead of 10.8.)
template <int NCH>
__global__ __launch_bounds__(SNT) void sample_cut_kernel(const uint16_t* __restrict__ logits, int64_t row_stride, int V,
                                                         const float* __restrict__ temperature, const float* __restrict__ top_p,
                                                         const int* __restrict__ top_k, SampleRow* __restrict__ rows) {
  __shared__ CutShared sh;
  const int b = blockIdx.x, nchunks = V >> 3;
  const float temp = temperature[b], p = top_p[b];
  int k = top_k[b];
  uint32_t cut = 0;
  if (needs_cut(temp, p, k, V)) {
    uint4 regs[NCH];
    load_row<NCH>(regs, logits + (int64_t)b * row_stride, nchunks);
    cut = row_cut<NCH>(regs, nchunks, V, temp, p, k, sh);
  }
  if (threadIdx.x == 0) rows[b] = SampleRow{0ull, cut, 0u};
}

// Grid (slices, B): a 256-thread workgroup takes 256 · NC chunks of 8 logits.  Its best candidate goes into the row's
// 64-bit maximum (value in the order-preserving 32 bits, then the lowest index); the slice that delivers last reads the result.
// V = 128256, a quarter of the rows without cut-off: 10.5 µs at B = 57.  (Slices of 4096 logits from 2048 workgroups on: greedy rows 57 9.6 → 7.9, but
// rows behind a cut-off 80 33 → 38, whose Philox blocks then follow one another.)
constexpr int DNT = 256;
template <int NC>
__global__ __launch_bounds__(DNT) void sample_draw_kernel(const uint16_t* __restrict__ logits, int64_t row_stride, int V,
                                                          const float* __restrict__ temperature, DrawArgs draw, SampleRow* __restrict__ rows,
                                                          int64_t* __restrict__ out) {
  __shared__ ArgMax sa[DNT / 64];
  const int b = blockIdx.y;
  const uint4* row = reinterpret_cast<const uint4*>(logits + (int64_t)b * row_stride);
  const int nchunks = V >> 3, first = blockIdx.x * (DNT * NC) + threadIdx.x;
  uint4 regs[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) regs[c] = first + c * DNT < nchunks ? row[first + c * DNT] : make_uint4(0, 0, 0, 0);
  const float temp = temperature[b];
  ArgMax a = best_of<NC>(regs, first, DNT, nchunks, V, temp, temp <= 0.f ? 0u : rows[b].cut, b, draw);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) a = amax(a, ArgMax{__shfl_xor(a.v, o, 64), __shfl_xor(a.i, o, 64)});
  if ((threadIdx.x & 63) == 0) sa[threadIdx.x >> 6] = a;
  __syncthreads();
  if (threadIdx.x != 0) return;
#pragma unroll
  for (int w = 1; w < DNT / 64; ++w) a = amax(a, sa[w]);
  SampleRow* r = rows + b;
  // The two words are only ever touched by atomics at the memory side, so the order "maximum, then count" is all it takes, and the wait
  // for the maximum's old value gives it.  (A release / acquire count writes back and empties the die's L2 once per workgroup: 340 µs
  // instead of 67 at B = 512, V = 128256.)
  if ((unsigned)a.i < (unsigned)V) {                       // a slice without a candidate delivers none; + 0: −0 ties with +0
    const unsigned long long old = __hip_atomic_fetch_max(&r->best, (unsigned long long)okey(a.v + 0.f) << 32 | (uint32_t)~a.i,
                                                          __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("" ::"v"((uint32_t)old), "v"((uint32_t)(old >> 32)) : "memory");
  }
  const uint32_t before = __hip_atomic_fetch_add(&r->done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (before == gridDim.x - 1) {
    const unsigned long long best = __hip_atomic_fetch_max(&r->best, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    out[b] = best == 0ull ? 0 : valid_token((int)~(uint32_t)best, V);
  }
}

bool sample_by_slices(bool logits_fp32, const void* logits, int64_t row_stride, int B, int V) {
  return !logits_fp32 && V % 8 == 0 && V > 0 && V <= 16 * SNT * 8 && row_stride % 8 == 0 && reinterpret_cast<uintptr_t>(logits) % 16 == 0 &&
         B <= 65535;
}

static bool sample_whole(int V) { return V <= SNT * 8; }
size_t sample_workspace_bytes(int B, int V) { return sample_whole(V) ? 0 : (size_t)B * sizeof(SampleRow); }

// `ws`: sample_workspace_bytes where sample_by_slices says so (contents do not matter), else not read.
void launch_sample(const void* logits, bool logits_fp32, int64_t row_stride, int B, int V, const float* temperature,
                   const float* top_p, const int* top_k, const int64_t* seeds, const int64_t* steps, const float* noise,
                   int64_t* out, void* ws, hipStream_t stream) {
  if (B == 0) return;
  if (!sample_by_slices(logits_fp32, logits, row_stride, B, V)) {
    if (logits_fp32)
      hipLaunchKernelGGL(sample_kernel<float>, dim3(B), dim3(SNT), 0, stream, (const float*)logits, row_stride, V,
                         temperature, top_p, top_k, seeds, steps, noise, out);
    else
      hipLaunchKernelGGL(sample_kernel<uint16_t>, dim3(B), dim3(SNT), 0, stream, (const uint16_t*)logits, row_stride, V,
                         temperature, top_p, top_k, seeds, steps, noise, out);
    return;
  }
  const uint16_t* x = (const uint16_t*)logits;
  const DrawArgs draw{seeds, steps, noise};
  if (sample_whole(V)) {
    hipLaunchKernelGGL(sample_whole_kernel, dim3(B), dim3(SNT), 0, stream, x, row_stride, V, temperature, top_p, top_k, draw, out);
    return;
  }
  SampleRow* rows = (SampleRow*)ws;
  if (V <= 4 * SNT * 8)
    hipLaunchKernelGGL(sample_cut_kernel<4>, dim3(B), dim3(SNT), 0, stream, x, row_stride, V, temperature, top_p, top_k, rows);
  else
    hipLaunchKernelGGL(sample_cut_kernel<16>, dim3(B), dim3(SNT), 0, stream, x, row_stride, V, temperature, top_p, top_k, rows);
  // slices of 8192 logits where they keep all compute units busy several times over (half the atomics), of 2048 below: B = 57 18 → 16 µs
  const int wide = (V / 8 + DNT * 4 - 1) / (DNT * 4);
  if ((int64_t)wide * B >= 2048)
    hipLaunchKernelGGL(sample_draw_kernel<4>, dim3(wide, B), dim3(DNT), 0, stream, x, row_stride, V, temperature, draw, rows, out);
  else
    hipLaunchKernelGGL(sample_draw_kernel<1>, dim3((V / 8 + DNT - 1) / DNT, B), dim3(DNT), 0, stream, x, row_stride, V, temperature, draw, rows, out);
}

// Pipelined stepping: a decode row whose input id was sampled by the step still in flight reads it from the
// sampler's device output (``src`` = row there, -1 = the host already staged the id).
__global__ void gather_sampled_kernel(int* __restrict__ input, const int* __restrict__ src,
                                      const int64_t* __restrict__ sampled, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    const int s = src[i];
    if (s >= 0) input[i] = (int)sampled[s];
  }
}

void launch_gather_sampled(int* input, const int* src, const int64_t* sampled, int n, hipStream_t stream) {
  if (n <= 0) return;
  hipLaunchKernelGGL(gather_sampled_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, input, src, sampled, n);
}

}  // namespace dli

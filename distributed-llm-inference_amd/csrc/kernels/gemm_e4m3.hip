// W8A8 product on the e4m3 matrix cores: y[m, n] = bf16(Σ_k x[m, k] · w[n, k] · x_scale[m] · w_scale[n]).
//
// The K loop is gemm_core.h's; at most one workgroup per compute unit runs 256 × 256 tiles, then 128 × 256 ones.  What bounds it: the matrix
// cores at the clock that the card holds under them.  Results leave through LDS, 256 contiguous bytes of a row at a time, with the next tile's
// first steps already on their way (one tile per workgroup, 8-byte stores from the accumulators: 191 µs instead of 173 for the first line's 2000
// rows).  The kernel takes all 512 registers and spills four 8-byte row offsets; store() reloads each and waits for everything in flight with it.
// Measured (µs; library product in brackets):
//   28672 × 4096 weights   M = 512 50 (63)   1024 94 (118)   2000 173 (230)   4096 329 (402, 2.92 against 2.40 PFLOP/s)
//   4096 × 14336           M = 1600 89 (94)   2000 95 (110)   4096 151 (178, 3.18 against 2.71 PFLOP/s)
//   8192 × 3584            M = 700 28 (30)   1024 31 (37)   2000 47 (57)   4096 89 (105)
#include <algorithm>

#include "common.h"
#include "gemm_core.h"
#include "kernels.h"

namespace dli {

namespace ge4 {

using namespace gcore;

constexpr int TURN = stage_bytes<8>;                         // LDS behind the step buffers: 4 KB of each wave, 16 rows × 128 columns bf16
constexpr int SCALES = TURN + 4 * 4096;                      // [4 tiles][256 row scales, 256 column scales]
constexpr int LDS_BYTES = SCALES + 4 * 2048;

// byte offset, inside the operand that starts at it, of lane `lane`'s 16 bytes of row r (swizzled as the LDS image is).  Rows of a weight
// tile lie up to 255 · K bytes apart, K up to 2^24: beyond the signed range.
constexpr __host__ __device__ uint32_t chunk_offset(int r, int K, int lane) { return (uint32_t)r * (uint32_t)K + (uint32_t)(((lane & 7) ^ (r & 7)) << 4); }
static_assert(chunk_offset(255, (1 << 24) - 256, 0) == 255u * ((1u << 24) - 256u) + 112u, "the last row of a tile at the largest K");

struct Args {
  const uint8_t* X;
  int64_t x_stride;
  const uint8_t* W;
  const float *xs, *ws;
  uint16_t* out;
  int64_t out_stride;
  int M, K, col_blocks, pairs, whole, halves;
};

// The first `whole` places of the order of 256-row tiles run as such; the other places, and the last 128 rows where the number of
// 128-row tiles is odd, run as 128-row tiles behind them.
template <int MB>
struct Tiles {
  const Args& p;
  char* lds;
  Places places;
  int count;
  __device__ __forceinline__ Tiles(const Args& p_, char* lds_) : p(p_), lds(lds_), places(MB == 8 ? p_.whole : p_.halves, MB != 8), count(places.count) {}
  __device__ __forceinline__ void where(int i, int& row0, int& n0) const {
    int row, col;
    const int lin = places.at(i);
    if constexpr (MB == 8) {
      tile_of(lin, p.pairs, p.col_blocks, row, col);
      row0 = row * 256;
    } else {
      const int cut = 2 * (p.pairs * p.col_blocks - p.whole);
      if (lin < cut) {
        tile_of(p.whole + (lin >> 1), p.pairs, p.col_blocks, row, col);
        row0 = row * 256 + (lin & 1) * 128;
      } else {
        row0 = p.pairs * 256;
        col = lin - cut;
      }
    }
    n0 = col * TN;
  }
  __device__ __forceinline__ void sources(int i, int lane, int wave, const char*& A, const char*& W, uint32_t (&a_src)[2][MB / 2],
                                          uint32_t (&w_src)[2][4]) const {
    int row0, n0;
    where(i, row0, n0);
    A = reinterpret_cast<const char*>(p.X);
    W = reinterpret_cast<const char*>(p.W) + (int64_t)n0 * p.K;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int j = 0; j < MB / 2; ++j) {
        const int r = a_piece_row<MB>(h, wave * (MB / 2) + j) + (lane >> 3);
        a_src[h][j] = (uint32_t)(min(row0 + r, p.M - 1) * p.x_stride + (((lane & 7) ^ (r & 7)) << 4));   // rows past M repeat the last
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = b_piece_row(h, wave * 4 + j) + (lane >> 3);
        w_src[h][j] = chunk_offset(r, p.K, lane);
      }
    }
    char* s = lds + SCALES + (i & 3) * 2048;
    if (wave * 64 < tile_rows<MB>)
      __builtin_amdgcn_global_load_lds((gptr_t)(p.xs + min(row0 + wave * 64 + lane, p.M - 1)), (lptr_t)(s + wave * 256), 4, 0, 0);
    __builtin_amdgcn_global_load_lds((gptr_t)(p.ws + n0 + wave * 64 + lane), (lptr_t)(s + 1024 + wave * 256), 4, 0, 0);
  }
  // 16 rows at a time through LDS: a store instruction writes 256 bytes of each of four rows (from the accumulators 32 of each of 16)
  __device__ __forceinline__ bool store(int i, int lane, int wave, f32x4 (&acc)[MB][8]) const {
    int row0, n0;
    where(i, row0, n0);
    const int wr = wave >> 1, wc = wave & 1, col = lane & 15, g = lane >> 4;
    const float* s = reinterpret_cast<const float*>(lds + SCALES + (i & 3) * 2048);
    char* turn = lds + TURN + wave * 4096;
    f32x4 sw[8];
#pragma unroll
    for (int n = 0; n < 8; ++n) sw[n] = *reinterpret_cast<const f32x4*>(s + 256 + wc * 128 + n * 16 + 4 * g);
    const int left = p.M - row0 - wr * (MB * 16);            // rows of this wave that there are
    uint16_t* dst = p.out + (int64_t)(row0 + wr * (MB * 16)) * p.out_stride + n0 + wc * 128 + col * 8;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const float sx = s[wr * (MB * 16) + m * 16 + col];
#pragma unroll
      for (int n = 0; n < 8; ++n) {
        bf16x4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = (short)f2bf(acc[m][n][r] * sx * sw[n][r]);
        *reinterpret_cast<bf16x4*>(turn + col * 256 + (((n * 2 + (g >> 1)) ^ col) << 4) + (g & 1) * 8) = o;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = q * 4 + g;
        const u32x4 v = *reinterpret_cast<const u32x4*>(turn + r * 256 + ((col ^ r) << 4));
        if (m * 16 + r < left) *reinterpret_cast<u32x4*>(dst + (int64_t)(m * 16 + r) * p.out_stride) = v;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    return row0 + tile_rows<MB> <= p.M;
  }
};

__global__ __launch_bounds__(256, 1) void gemm_e4m3_kernel(Args p) {
  __shared__ __attribute__((aligned(1024))) char lds[LDS_BYTES];
  Tiles<8> whole(p, lds);
  stream_tiles<8>(lds, whole, p.K / STEP_BYTES);
  Tiles<4> halves(p, lds);
  stream_tiles<4>(lds, halves, p.K / STEP_BYTES);
}

}  // namespace ge4

// Of the 256-row tiles, those beyond the last whole round of one per compute unit are cut in two where that is shorter.  A 128-row tile takes
// 0.58 of a 256-row one (4096 × 4096 × 14336 as one round of the latter 150 µs, 2000 rows as one round of the former 87).
constexpr int NUM_CU = 256;
constexpr double HALF = 0.58;
struct Plan {
  int whole, halves, grid;
  double rounds;                                             // of the workgroup that has most, in 256-row tiles
  Plan(int whole_, int halves_) : whole(whole_), halves(halves_), rounds(0) {
    grid = std::min(NUM_CU, (whole + 7) / 8 * 8 + (halves + 7) / 8 * 8);         // enough of them on every XCD
    // As gcore::Places deals them: an XCD's 256-row tiles in turn from its first workgroup on, its 128-row tiles from the last one back.  What the
    // turns leave over meets in one workgroup where there is more of it than workgroups.
    const int groups = grid >> 3;
    for (int x = 0; x < 8 && groups > 0; ++x) {
      auto mine = [&](int total) { const int per = (total + 7) >> 3; return std::max(0, std::min(per, total - x * per)); };
      const int w = mine(whole), h = mine(halves), w_over = w % groups, h_over = h % groups;
      const double over = w_over + h_over > groups ? 1 + HALF : w_over ? 1 : h_over ? HALF : 0;
      rounds = std::max(rounds, w / groups + HALF * (h / groups) + over);
    }
  }
};
static Plan plan(int M, int col_blocks) {
  const int units = (M + 127) / 128, odd = (units & 1) * col_blocks, total = units / 2 * col_blocks, rest = total % NUM_CU;
  const Plan keep(total, odd), cut(total - rest, 2 * rest + odd);
  return keep.rounds <= cut.rounds ? keep : cut;
}

// multiplied part of what the chip could multiply in the time that launch_gemm_e4m3 takes by its plan
double gemm_e4m3_fill(int64_t M, int64_t N) {
  return (double)M * N / (256.0 * gcore::TN * NUM_CU * plan((int)M, (int)(N / gcore::TN)).rounds);
}

// (256-row tiles, 128-row tiles, workgroups, rounds)
std::tuple<int64_t, int64_t, int64_t, double> gemm_e4m3_plan(int64_t M, int64_t N) {
  const Plan p = plan((int)M, (int)(N / gcore::TN));
  return {p.whole, p.halves, p.grid, p.rounds};
}

// x [M, K] (rows 16-byte aligned), w [N, K] contiguous, K % 256 == 0, N % 256 == 0, both operands below 4 GiB
void launch_gemm_e4m3(const void* x, int64_t x_stride, const void* w, const float* x_scale, const float* w_scale, void* out,
                      int64_t out_stride, int M, int N, int K, hipStream_t stream) {
  const int col_blocks = N / gcore::TN, units = (M + 127) / 128, pairs = units / 2;
  const Plan p = plan(M, col_blocks);
  hipLaunchKernelGGL(ge4::gemm_e4m3_kernel, dim3(p.grid), dim3(256), 0, stream,
                     ge4::Args{(const uint8_t*)x, x_stride, (const uint8_t*)w, x_scale, w_scale, (uint16_t*)out, out_stride, M, K,
                               col_blocks, pairs, p.whole, p.halves});
}

}  // namespace dli

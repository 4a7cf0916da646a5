// K loop of the large e4m3 products: a workgroup of four waves multiplies a 256 × 256 (or 128 × 256) tile, each wave 128 × 128 (64 × 128)
// of it, C[rows, n] = A[rows, :] · W[n, :]ᵀ, sums in fp32.  (The same loop on bf16 operands, twice the instructions of half the length,
// took 312 µs for 4096 × 4096 × 14336 where the eight-wave tile of gemm256.hip takes 305: both run at the clock that the card's power allows.)
//
//   * A K-step is 128 bytes of every row, 2048 cycles of the matrix cores for a 256² tile.
//   * One wave per SIMD and the largest wave tile its registers hold (256 accumulators + 128 fragment registers of 512): a step reads
//     128 KB of fragments from LDS, where eight waves of 128 × 64 read 192 KB — beside the 64 KB the DMA writes, that alone fills the LDS
//     port for as long as the matrix cores need.
//   * Matrix instructions are issued in program order and take 32 cycles each; what else the wave has to issue
//     (fragment reads of the NEXT quadrant, LDS-DMA of the step after next) stands between them, one at a time, so nothing waits.
//   * Both operands go global → LDS by LDS-DMA, two step buffers.  The LDS image is lane-linear: slot p of row r holds 16-byte chunk
//     p ^ (r & 7), applied on the source address and on the read; ds_read_b128 then has no bank conflicts.
//   * A step is four quadrants (a0 bf) (a0 bo) (a1 bo) (a1 bf); the next step starts with bo.  Fragments are read one quadrant ahead:
//     bo, a1, next a0, next bo.  Every half-tile is re-filled for the step two ahead after the first barrier behind its last read, and
//     read after the barrier that follows its counted wait: two barriers a step, six quadrants (1.3 µs) for a DMA to land.
//   * D[weight row][token row] (operands swapped): a lane holds four consecutive output columns of one row.
#pragma once
#include "common.h"

namespace dli {
namespace gcore {

constexpr int STEP_BYTES = 128;                              // bytes of K per row and step
constexpr int TN = 256;                                      // weight rows of a tile
template <int MB> constexpr int tile_rows = 32 * MB;         // MB: 16-row blocks of a wave (8: 256-row tiles, 4: 128-row tiles)
template <int MB> constexpr int stage_bytes = 2 * (tile_rows<MB> + TN) * STEP_BYTES;

typedef __attribute__((ext_vector_type(8))) int i32x8;
using gptr_t = const __attribute__((address_space(1))) void*;
using lptr_t = __attribute__((address_space(3))) void*;

__device__ __forceinline__ int lds_off(int r, int c) { return r * STEP_BYTES + ((c ^ (r & 7)) << 4); }

// first row (inside the operand tile) of DMA piece `piece` (8 rows of 128 bytes) of half `h`: a half is the h-th half of both waves' rows
template <int MB> __device__ __forceinline__ int a_piece_row(int h, int piece) {
  return (piece / MB) * (MB * 16) + h * (MB * 8) + (piece % MB) * 8;
}
__device__ __forceinline__ int b_piece_row(int h, int piece) { return (piece >> 3) * 128 + h * 64 + (piece & 7) * 8; }

// One matrix instruction.  Written out because its sum has to stay in the accumulator register it came from: the builtin leaves source
// and target apart, and with 256 + 128 registers taken the allocator then moved accumulators about in the loop and spilled 70.  The
// compiler does not see a matrix instruction here, so the waits are ours: two cycles behind a write of an operand by a vector instruction
// (the s_nop; the matrix pipe is busy longer), and before anything but another product reads a sum (behind the K loop).
// A lane's 32 bytes are chunks g and 4 + g of its row (both operands alike: any order of k will do).
__device__ __forceinline__ void mma(const u32x4 (&w)[2], const u32x4 (&a)[2], f32x4& c) {
  const i32x8 wv = __builtin_bit_cast(i32x8, __builtin_shufflevector(w[0], w[1], 0, 1, 2, 3, 4, 5, 6, 7));
  const i32x8 av = __builtin_bit_cast(i32x8, __builtin_shufflevector(a[0], a[1], 0, 1, 2, 3, 4, 5, 6, 7));
  asm volatile("s_nop 1\n\tv_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0" : "+a"(c) : "v"(wv), "v"(av));
}

// Runs `tiles.count` tiles of nk K-steps each (an even number: the buffers change places), one stream of steps: behind a tile's last step the DMA goes on with the next tile's
// first, so only the first tile of a workgroup waits for memory; a tile's results are stored with the next one's steps on their way, and their
// instructions are counted in its first waits (a store() that waits for memory itself drains these steps: its loss, not an error).
//   tiles.sources(i, lane, wave, A, W, a_src, w_src): bases of tile i's operands (wave-uniform) and this lane's byte offsets at k = 0 for
//     DMA piece wave · (pieces per wave) + j of half h; may fetch into LDS what store(i) needs (landed by then, ring of four tiles)
//   tiles.store(i, lane, wave, acc): acc[m][n]: rows wr·16·MB + m·16 + (lane & 15), columns wc·128 + n·16 + 4 (lane >> 4) + r;
//     true: it issued exactly MB · 4 vector memory instructions (whole tiles), else any number
template <int MB, class Tiles>
__device__ __forceinline__ void stream_tiles(char* lds, Tiles& tiles, int nk) {
  constexpr int A_TILE = tile_rows<MB> * STEP_BYTES, W_TILE = TN * STEP_BYTES;
  constexpr int HB = MB / 2;                                 // row blocks of a quadrant
  constexpr int NMMA = HB * 4;                               // matrix instructions of a quadrant
  constexpr int FLIGHT = MB + 8;                             // DMA instructions of a wave in a step
  constexpr int STORES = MB * 4;
  if (tiles.count <= 0) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave >> 1, wc = wave & 1, col = lane & 15, g = lane >> 4;
  const char* a_rd[2] = {lds + lds_off(wr * (MB * 16) + col, g), lds + lds_off(wr * (MB * 16) + col, 4 + g)};
  const char* w_rd[2] = {lds + 2 * A_TILE + lds_off(wc * 128 + col, g), lds + 2 * A_TILE + lds_off(wc * 128 + col, 4 + g)};
  u32x4 fa[2][HB][2], fw[2][4][2];
  f32x4 acc[MB][8];

  // what is fetched: step f_k of tile f_tile (behind the last tile its last step again, which nothing reads)
  int f_tile = 0, f_k = 0;
  const char *A, *W;
  uint32_t a_src[2][HB], w_src[2][4];
  tiles.sources(0, lane, wave, A, W, a_src, w_src);
  auto advance = [&]() __attribute__((always_inline)) {
    if (++f_k < nk) return;
    f_k = nk - 1;
    if (f_tile + 1 < tiles.count) {
      f_k = 0;
      tiles.sources(++f_tile, lane, wave, A, W, a_src, w_src);
    }
  };
  auto dma_a = [&](int buf, int h, int j) __attribute__((always_inline)) {
    __builtin_amdgcn_global_load_lds((gptr_t)(A + (int64_t)f_k * STEP_BYTES + a_src[h][j]),
                                     (lptr_t)(lds + buf * A_TILE + a_piece_row<MB>(h, wave * HB + j) * STEP_BYTES), 16, 0, 0);
  };
  auto dma_w = [&](int buf, int h, int j) __attribute__((always_inline)) {
    __builtin_amdgcn_global_load_lds((gptr_t)(W + (int64_t)f_k * STEP_BYTES + w_src[h][j]),
                                     (lptr_t)(lds + 2 * A_TILE + buf * W_TILE + b_piece_row(h, wave * 4 + j) * STEP_BYTES), 16, 0, 0);
  };
  auto rd_a = [&](int buf, int h, int i) __attribute__((always_inline)) {
    fa[h][i >> 1][i & 1] = *reinterpret_cast<const u32x4*>(a_rd[i & 1] + buf * A_TILE + (h * HB + (i >> 1)) * 16 * STEP_BYTES);
  };
  auto rd_w = [&](int buf, int h, int i) __attribute__((always_inline)) {
    fw[h][i >> 1][i & 1] = *reinterpret_cast<const u32x4*>(w_rd[i & 1] + buf * W_TILE + (h * 4 + (i >> 1)) * 16 * STEP_BYTES);
  };
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int n = 0; n < 8; ++n) {
        acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
        asm volatile("" : "+a"(acc[m][n]));                  // here, not right before the first product: see mma()
      }
  };
  // barriers behind a store whose instructions are still counted: they are younger than what the barrier waits for
  int relaxed = 0;
  // quadrant (row half MH, column half NH): after matrix instruction i one fragment read (n_rd of them, from the front) or one DMA
  // instruction (n_dma, evenly over the quadrant's second half)
#define GC_QUAD(MH, NH, n_rd, RD, n_dma, DMA)                                                                      \
  _Pragma("unroll") for (int i = 0; i < NMMA; ++i) {                                                               \
    const int m = i >> 2, n = i & 3;                                                                               \
    mma(fw[NH][n], fa[MH][m], acc[(MH) * HB + m][(NH) * 4 + n]);                                                   \
    constexpr int first = NMMA / 2, rd_gap = first / (n_rd) > 0 ? first / (n_rd) : 1, dma_gap = first / (n_dma);   \
    if (i % rd_gap == 0 && i / rd_gap < (n_rd)) { const int x = i / rd_gap; RD; }                                  \
    if (i >= first && (i - first) % dma_gap == 0 && (i - first) / dma_gap < (n_dma)) { const int x = (i - first) / dma_gap; DMA; } \
    __builtin_amdgcn_sched_barrier(0);                                                                             \
  }
#define GC_BARRIER()                                                                                               \
  {                                                                                                                \
    if (relaxed > 0) {                                                                                             \
      --relaxed;                                                                                                   \
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(FLIGHT + STORES) : "memory");                            \
    } else {                                                                                                       \
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(FLIGHT) : "memory");                                     \
    }                                                                                                              \
    __builtin_amdgcn_s_barrier();                                                                                  \
    asm volatile("" ::: "memory");                                                                                 \
    __builtin_amdgcn_sched_barrier(0);                                                                             \
  }
#define GC_STEP(BUF)                                                                                               \
  {                                                                                                                \
    constexpr int f_ = (BUF), o_ = 1 - (BUF);                                                                      \
    GC_BARRIER()                                                                                                   \
    GC_QUAD(0, f_, 8, rd_w(BUF, o_, x), HB, dma_a(BUF, 0, x))                                                      \
    GC_QUAD(0, o_, MB, rd_a(BUF, 1, x), 4, dma_w(BUF, f_, x))                                                      \
    GC_BARRIER()                                                                                                   \
    GC_QUAD(1, o_, MB, rd_a((BUF) ^ 1, 0, x), 4, dma_w(BUF, o_, x))                                                \
    GC_QUAD(1, f_, 8, rd_w((BUF) ^ 1, o_, x), HB, dma_a(BUF, 1, x))                                                \
    advance();                                                                                                     \
  }
  // steps 0 and 1, in the order in which the loop issues: a0 bf | bo a1
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int j = 0; j < HB; ++j) dma_a(s, 0, j);
#pragma unroll
    for (int j = 0; j < 4; ++j) dma_w(s, s, j);
#pragma unroll
    for (int j = 0; j < 4; ++j) dma_w(s, 1 - s, j);
#pragma unroll
    for (int j = 0; j < HB; ++j) dma_a(s, 1, j);
    advance();
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FLIGHT) : "memory");                  // step 0 has landed
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < MB; ++i) rd_a(0, 0, i);
#pragma unroll
  for (int i = 0; i < 8; ++i) rd_w(0, 0, i);

  int tile = 0;
  do {
    clear();
    int k = nk;
    do {
      GC_STEP(0)
      GC_STEP(1)
    } while ((k -= 2) > 0);
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");       // the last sums are written 16 passes after their instruction
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int n = 0; n < 8; ++n) asm volatile("" : "+a"(acc[m][n]));            // read behind this line only
    if (tiles.store(tile, lane, wave, acc)) {
      relaxed = 3;
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      relaxed = 0;
    }
  } while (++tile < tiles.count);
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");                    // nothing lands in LDS behind this function
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#undef GC_QUAD
#undef GC_BARRIER
#undef GC_STEP
}

// x-th eighth of `total` places for XCD x (the hardware deals workgroups round-robin): place of a workgroup's j-th tile, and how many it
// has.  `back`: the last workgroups of an XCD take the first places.
struct Places {
  int first, count;
  __device__ __forceinline__ Places(int total, bool back) {
    const int per = (total + 7) >> 3, x = blockIdx.x & 7, groups = gridDim.x >> 3;
    const int i = back ? groups - 1 - (int)(blockIdx.x >> 3) : (int)(blockIdx.x >> 3);
    const int mine = min(per, total - x * per) - i;
    first = x * per + i;
    count = mine > 0 ? (mine + groups - 1) / groups : 0;
  }
  __device__ __forceinline__ int at(int j) const { return first + j * (int)(gridDim.x >> 3); }
};

// place of a tile → (row tile, column block): groups of 8 column blocks, row tile, column in the group: the 32 tiles that an XCD has at a
// time are 4 row tiles × 8 column blocks
__device__ __forceinline__ void tile_of(int lin, int row_tiles, int col_blocks, int& row, int& col) {
  const int grp = lin / (8 * row_tiles), within = lin - grp * (8 * row_tiles), gw = min(8, col_blocks - grp * 8);
  row = within / gw;
  col = grp * 8 + (within - row * gw);
}

}  // namespace gcore
}  // namespace dli

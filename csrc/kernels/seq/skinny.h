// Products of a few rows with a weight matrix on the matrix cores (decode steps): what the dense layers
// (skinny_linear.hip) and the experts (expert_ffn.hip) share.
//
// Such a product reads every weight once and does next to nothing with it, so its time is the latency of one load
// plus the weights over the bandwidth. A workgroup of 8 waves owns 16 columns (NT tiles of them, or HALF a tile) and splits K over its
// waves, 64 k at a time; the waves' sums meet in LDS. At 2048 columns that is 128 workgroups, or 256 of half tiles.
//
// What a compute unit takes in (its weights, and the rows again for every workgroup) bounds the larger M, and how a load
// spreads its addresses decides how much that is. The matrix cores want 16 rows side by side over the lanes; a load that
// follows them jumps to another row from lane to lane, and the addresses of its 64 lanes are looked up one by one: 34 KB per us
// and CU, however many loads are in flight. So the rows go through LDS: global_load_lds takes 8 lanes side by side along a row
// (whole 128-byte lines, four lanes per look-up) and the operands are read from there, without registers for loads in
// flight: 60 - 80 KB per us. Each wave copies into a part of LDS that is its own, DEPTH pieces of 64 k ahead, and waits for
// its own copies alone. us, cold weights, loads in operand order -> this (the vendor's GEMM), 1 / 16 / 48 rows:
//   1024 x 1024   3.4 -> 2.6 (5.7)    4.2 -> 2.8 (5.8)    6.5 -> 3.8 (8.0)     (columns x k)
//   2048 x 2048   5.0 -> 4.0 (11.0)   6.4 -> 4.3 (11.0)   10.5 -> 7.0 (11.1)   (half tiles but for 48 rows)
//   2048 x 6144   9.3 -> 6.7 (11.2)   13.6 -> 8.4 (11.4)  24.7 -> 14.0 (16.8)  (half tiles)
//   32000 x 2048  25.2 -> 25.0 (32.3) 33.7 -> 27.5 (32.7) 60 -> 33.3, two tiles per workgroup (37.4)
// Deeper copies of whole tiles (3 or 5 pieces) changed nothing at one workgroup per CU and cost up to a fifth where they leave room for fewer; so do two
// pieces but for up to 16 rows and more than a piece per wave. Half tiles, one workgroup per CU, run two for any rows, three for up to 8 rows of more
// than 4096 k, in 32 bits what whole tiles do (skinny_linear.hip).
// 32-bit operands (F32) are the same rows of twice as many 16-bit halves: a step is 64 bytes of a row, 16 numbers, and four
// products of 4 k each; the four numbers of a lane are k 4 g + e on both sides, so nothing else differs.
#pragma once
#include "lds_copy.h"
#include "seq_common.h"

namespace hipserve {

constexpr int kSkWaves = 8, kSkThreads = 64 * kSkWaves, kSkLd = 20;   // kSkLd: row stride of the sums in LDS (floats)

template <int N> HS_DEVICE void wait_copies() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// One wave's part of W[NT tiles of 16 columns] . x[XG groups of 8 rows]. K in 16-bit halves, K % 8 == 0.
// A piece (64 k) in LDS: [NT tiles][16 rows][128 bytes] of W, then [XG][8 rows][128 bytes] of x; the 16-byte part q of row r sits
// at part q ^ (r / 2 % 8), so that the 16 rows of an operand use all banks evenly: a lane copies the part that belongs at its place.
// HALF: the last tile is its first 8 columns.
template <int XG, int NT, int DEPTH, bool F32 = false, bool HALF = false> struct Skinny {
  static constexpr int WG = 2 * NT - HALF;   // groups of 8 rows of W
  static constexpr int ST = (XG + 1) / 2, kCopies = WG + XG, kPiece = kCopies * 1024;
  // the last tile's missing 8 rows, where XG is odd, are read past the piece
  static constexpr int kRing = kSkWaves * DEPTH * kPiece + (XG & 1) * 1024, kSums = kSkWaves * 16 * ST * kSkLd * 4;
  static constexpr int kLds = kRing > kSums ? kRing : kSums;
  static_assert(kLds <= 160 * 1024 && kCopies * (DEPTH - 1) < 64, "LDS; copies that a wait can count");

  static HS_DEVICE int part(int lane, int row) { return (lane & 7) ^ (row >> 1 & 7); }   // of a row, for a lane's copy

  // acc[nt][st] += the products; lane (c, g) = (lane % 16, lane / 16) ends with columns 4 g .. + 3 of row 16 st + c. w[nt]: first row
  // of the tile; w_row[i] / x_row[j]: byte offsets of the lane's row (lane / 8 of the 8) in the half tile i (of 2 NT) from w[i / 2] and in
  // the group j of x from `x`. Every row is one that exists: what rows past the last one give is not used.
  // started(): what a kernel loads besides, once the first copies are on their way.
  template <typename F>
  static HS_DEVICE void accumulate(f32x4 (&acc)[NT][ST], const unsigned char* const (&w)[NT], const unsigned (&w_row)[WG],
                                   const unsigned char* x, const unsigned (&x_row)[XG], int K, unsigned char* smem,
                                   int lane, int wave, F&& started) {
    const int c = lane & 15, g = lane >> 4, r8 = lane >> 3;
    unsigned char* ring = smem + wave * DEPTH * kPiece;
    const unsigned lds0 = lds_at(ring);
    const int pieces = (K + 63) >> 6, n = (pieces - wave + kSkWaves - 1) >> 3;   // (kSkWaves is 1 << 3) this wave's: wave, wave + 8, ...
    // the lane's bytes past the piece's first k of the first row: full pieces differ by uniform numbers
    unsigned w_at[WG], x_at[XG];
#pragma unroll
    for (int j = 0; j < WG; ++j) w_at[j] = w_row[j] + 16 * part(lane, 8 * (j & 1) + r8);
#pragma unroll
    for (int j = 0; j < XG; ++j) x_at[j] = x_row[j] + 16 * part(lane, 8 * (j & 1) + r8);
    auto copy = [&](int i) {
      const int k0 = 64 * (wave + kSkWaves * i);
      const unsigned to = lds0 + i % DEPTH * kPiece;
      if (k0 + 64 <= K) {
#pragma unroll
        for (int j = 0; j < XG; ++j) copy_1k(x + 2 * k0, x_at[j], to + (WG + j) * 1024);
#pragma unroll
        for (int j = 0; j < WG; ++j) copy_1k(w[j / 2] + 2 * k0, w_at[j], to + j * 1024);
        return;
      }
#pragma unroll
      for (int j = 0; j < XG; ++j)   // what lies past K is not used
        copy_1k(x, x_row[j] + 2 * min(k0 + 8 * part(lane, 8 * (j & 1) + r8), K - 8), to + (WG + j) * 1024);
#pragma unroll
      for (int j = 0; j < WG; ++j)
        copy_1k(w[j / 2], w_row[j] + 2 * min(k0 + 8 * part(lane, 8 * (j & 1) + r8), K - 8), to + j * 1024);
    };
    int at[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) at[s] = c * 128 + (((4 * s + g) ^ (c >> 1)) << 4);
    int half_of[2];   // HALF: both halves of the last tile are the same eight rows
#pragma unroll
    for (int s = 0; s < 2; ++s) half_of[s] = (c & 7) * 128 + (((4 * s + g) ^ ((c & 7) >> 1)) << 4);
#pragma unroll
    for (int i = 0; i < DEPTH; ++i)
      if (i < n) copy(i);
    started();   // its loads are younger: the waits below cover some of them too early at most
    for (int i = 0; i < n; ++i) {
      if (i + DEPTH <= n) wait_copies<kCopies * (DEPTH - 1)>();
      else wait_copies<0>();
      const unsigned char* t = ring + i % DEPTH * kPiece;
      u16x8 a[2][NT], b[2][ST];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) a[s][nt] = *reinterpret_cast<const u16x8*>(t + nt * 2048 + (HALF && nt == NT - 1 ? half_of[s] : at[s]));
#pragma unroll
        for (int st = 0; st < ST; ++st) b[s][st] = *reinterpret_cast<const u16x8*>(t + WG * 1024 + st * 2048 + at[s]);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the piece is read
      if (i + DEPTH < n) copy(i + DEPTH);
      if (64 * (wave + kSkWaves * i) + 64 > K) {   // what lies past K is 0 on both sides
        const u16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          if (64 * (wave + kSkWaves * i) + 32 * s + 8 * g < K) continue;
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) a[s][nt] = zero;
#pragma unroll
          for (int st = 0; st < ST; ++st) b[s][st] = zero;
        }
      }
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int st = 0; st < ST; ++st) {
            if constexpr (F32) {
              const f32x4 fa = __builtin_bit_cast(f32x4, a[s][nt]), fb = __builtin_bit_cast(f32x4, b[s][st]);
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[nt][st] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[e], fb[e], acc[nt][st], 0, 0, 0);
            } else {
              acc[nt][st] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[s][nt]),
                                                                    __builtin_bit_cast(bf16x8, b[s][st]), acc[nt][st], 0, 0, 0);
            }
          }
    }
  }

  static HS_DEVICE void accumulate(f32x4 (&acc)[NT][ST], const unsigned char* const (&w)[NT], const unsigned (&w_row)[WG],
                                   const unsigned char* x, const unsigned (&x_row)[XG], int K, unsigned char* smem,
                                   int lane, int wave) {
    accumulate(acc, w, w_row, x, x_row, K, smem, lane, wave, [] {});
  }

  // Sums the waves' parts: v[nt][i] = element (row, column) = (e / kCols, e % kCols), e = threadIdx.x + kSkThreads * i, of
  // the [16 ST, kCols] result of column tile nt (threads past it get nothing).
  static constexpr int kCols = HALF && NT == 1 ? 8 : 16, kElems = (16 * ST * kCols + kSkThreads - 1) / kSkThreads;
  static HS_DEVICE void reduce(float (&v)[NT][kElems], const f32x4 (&acc)[NT][ST], unsigned char* smem) {
    float* red = reinterpret_cast<float*>(smem);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, g = lane >> 4;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      __syncthreads();   // the pieces, or the previous tile's sums, are read
#pragma unroll
      for (int st = 0; st < ST; ++st)
        *reinterpret_cast<f32x4*>(red + ((wave * ST + st) * 16 + c) * kSkLd + 4 * g) = acc[nt][st];
      __syncthreads();
#pragma unroll
      for (int i = 0; i < kElems; ++i) {
        const int e = tid + kSkThreads * i;
        float s = 0.f;
        if (e < 16 * kCols * ST) {
#pragma unroll
          for (int w = 0; w < kSkWaves; ++w) s += red[(w * ST * 16 + e / kCols) * kSkLd + e % kCols];
        }
        v[nt][i] = s;
      }
    }
  }
};

}  // namespace hipserve

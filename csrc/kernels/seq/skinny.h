// Products of a few rows with a weight matrix on the matrix cores (decode steps): what the dense layers
// (skinny_linear.hip) and the experts (expert_ffn.hip) share.
//
// Such a product reads every weight once and does next to nothing with it, so its time is the latency of one load
// plus the weights over the bandwidth. A workgroup of 8 waves owns 16 columns (NT tiles of them) and splits K over its
// waves: every wave issues the loads of its KU steps of 32 k before the first product, and the waves' sums meet in LDS.
// 16 columns per workgroup give 128 workgroups at 2048 columns. A compute unit takes in about 34 KB per us this way, so
// the rows' own bytes (16 columns of weights serve M rows) bound the larger M: 2048 x 2048, cold weights: 1 row 4.7 us,
// 16 rows 6.2, 32 rows 8.0, 48 rows 10.2 (the vendor's GEMM: 11.0 - 11.2); 32000 x 2048, 1 row: 26 us = 5.0 TB/s (34).
// 32-bit operands (F32) are the same rows of twice as many 16-bit halves: a step is 64 bytes of a row, 16 numbers, and four
// products of 4 k each; the four numbers of a lane are k 4 g + e on both sides, so nothing else differs. 3 rows, cold
// weights, 3072 x 1024: 5.9 us (the vendor's GEMM: 11.3); 32000 x 1024: 29 us = 4.5 TB/s (34).
#pragma once
#include "seq_common.h"

namespace hipserve {

constexpr int kSkWaves = 8, kSkThreads = 64 * kSkWaves, kSkLd = 20;   // kSkLd: row stride of the sums in LDS (floats)

// Two k steps of 16 rows as MFMA operands: lane (c, g) wants k 8 g .. + 7 of row c of both steps (64 bytes of a row each).
// The loads instead take whole 128-byte lines: lane (c, g) reads the part g + 4 (c / 8) of row c % 8 and of row c % 8 + 8
// (whole lines measured 4 - 14 % faster than 64 bytes of 16 rows), and the lanes c, c ^ 8 then exchange what belongs to the other's row (a rotation by 8 within 16 lanes).
HS_DEVICE void swap_steps(u16x8& s0, u16x8& s1, bool low) {
  const u32x4 a = __builtin_bit_cast(u32x4, s0), b = __builtin_bit_cast(u32x4, s1);
  u32x4 x, y;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const unsigned give = low ? b[i] : a[i];
    const unsigned got = (unsigned)__builtin_amdgcn_update_dpp(0, (int)give, 0x128, 0xf, 0xf, true);
    x[i] = low ? a[i] : got;
    y[i] = low ? got : b[i];
  }
  s0 = __builtin_bit_cast(u16x8, x);
  s1 = __builtin_bit_cast(u16x8, y);
}

// acc[nt][st] += the wave's part of W[16 columns of tile nt] . x[16 rows of tile st]; lane (c, g) = (lane % 16, lane / 16)
// ends with columns 4 g .. + 3 of row c. K in 16-bit halves. wr / xr: two row addresses per tile (c % 8 and c % 8 + 8), advanced by
// 8 g8, g8 = g + 4 (c / 8); low = c < 8. K % 8 == 0, KU even.
template <int ST, int NT, int KU, bool F32 = false>
HS_DEVICE void skinny_accumulate(f32x4 (&acc)[NT][ST], const unsigned short* const (&wr)[NT][2],
                                 const unsigned short* const (&xr)[ST][2], const bool (&live)[ST][2], int K, int g8,
                                 bool low, int wave) {
  const u16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int k0 = wave * 32 * KU; k0 < K; k0 += kSkWaves * 32 * KU) {
    u16x8 a[KU][NT], b[KU][ST];
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      const int k = k0 + 64 * (u / 2);
      const bool in = k + 8 * g8 < K;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) a[u][nt] = in ? *reinterpret_cast<const u16x8*>(wr[nt][u & 1] + k) : zero;
#pragma unroll
      for (int st = 0; st < ST; ++st) b[u][st] = (in && live[st][u & 1]) ? *reinterpret_cast<const u16x8*>(xr[st][u & 1] + k) : zero;
    }
#pragma unroll
    for (int u = 0; u < KU; u += 2) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) swap_steps(a[u][nt], a[u + 1][nt], low);
#pragma unroll
      for (int st = 0; st < ST; ++st) swap_steps(b[u][st], b[u + 1][st], low);
    }
#pragma unroll
    for (int u = 0; u < KU; ++u)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int st = 0; st < ST; ++st) {
          if constexpr (F32) {
            const f32x4 fa = __builtin_bit_cast(f32x4, a[u][nt]), fb = __builtin_bit_cast(f32x4, b[u][st]);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[nt][st] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[e], fb[e], acc[nt][st], 0, 0, 0);
          } else {
            acc[nt][st] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[u][nt]),
                                                                  __builtin_bit_cast(bf16x8, b[u][st]), acc[nt][st], 0, 0, 0);
          }
        }
  }
}

// Sums the waves' parts: v[nt][i] = element (row, column) = (e / 16, e % 16), e = threadIdx.x + kSkThreads * i, of
// the [16 ST, 16] result of column tile nt (threads past 256 ST get nothing). red: kSkWaves * 16 ST * kSkLd floats.
template <int ST, int NT>
HS_DEVICE void skinny_reduce(float (&v)[NT][(ST + 1) / 2], const f32x4 (&acc)[NT][ST], float* red) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, g = lane >> 4;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    if (nt > 0) __syncthreads();   // the previous tile's sums are read
#pragma unroll
    for (int st = 0; st < ST; ++st)
      *reinterpret_cast<f32x4*>(red + ((wave * ST + st) * 16 + c) * kSkLd + 4 * g) = acc[nt][st];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < (ST + 1) / 2; ++i) {
      const int e = tid + kSkThreads * i;
      float s = 0.f;
      if (e < 256 * ST) {
#pragma unroll
        for (int w = 0; w < kSkWaves; ++w) s += red[(w * ST * 16 + (e >> 4)) * kSkLd + (e & 15)];
      }
      v[nt][i] = s;
    }
  }
}

}  // namespace hipserve

// A workgroup's part of a product of a few rows, for the launches of such products (skinny_linear.hip) and those that hold the experts' besides
// (expert_beside.hip).
#pragma once
#include <type_traits>

#include "hipserve/seq_kernels.h"
#include "skinny.h"

namespace hipserve {
namespace {

HS_DEVICE float skinny_act(float z, int act, float c0, float c1) {
  if (act == 0) return tanhf(z);
  if (act == 1) return z > 0.f ? c0 * z * z + 0.5f * z : c1 * (expm1f(z) - z) + 0.5f * z;
  if (act == 2) { z = fmaxf(z, 0.f); return z * z; }
  if (act == 5) return tanhf(z / c0) * c0;
  return z;
}

// Sum over the lanes of a row's columns; every one of them gets it.
template <int COLS> HS_DEVICE float cols_sum(float v) {
  if constexpr (COLS == 16) return row_sum(v);
  v = dpp_step<0xB1, 0xf, false>(v);      // quad_perm [1, 0, 3, 2]
  v = dpp_step<0x4E, 0xf, false>(v);      // quad_perm [2, 3, 0, 1]
  return dpp_step<0x141, 0xf, false>(v);  // row_half_mirror
}

enum { kPlain, kNormed, kUpdate };   // SkinnyNorm: none; rows without their norm's factor; a result that goes into the residual stream
struct NoNorm {};
// The kernel's arguments: the parameters are what its first loads need, the rest is loaded once the copies are on their way (seq_common.h), and
// nothing is asked for after the product any more. us of four products in a captured loop (square, 3 x wider, back, 1.5 x wider), cold weights,
// 1 and 16 rows: width 1024 15.1 -> 13.6, 17.4 -> 16.0, width 2048 24.4 -> 22.8, 29.4 -> 27.8.
template <int NORM> struct SkinnyRest {
  long x_bs, out_ld, out_bs, out_zs;
  int act, act_from;
  float c0, c1, cols, eps;
  void* out;
  float* squares;      // kUpdate
  const void* bias;
};
template <int NORM> struct SkinnyArgs {
  const void *x, *w, *p, *q;
  int x_ld, M, N, K, i;
  SkinnyRest<NORM> rest;
};

// XG: groups of 8 rows; NT: 16-column tiles (GLU: the gate's and the up projection's of the same 16 output columns).
// F32: 32-bit operands, x, w, their strides and K in 16-bit halves (skinny.h). Workgroups z take `part` of K each (a multiple of 64) and write
// their sums out_zs elements apart (the bias in the first).
// p, q, i: kPlain - , bias, part; kNormed squares, bias, blocks; kUpdate residual, weight, blocks (K in one part for both).
// HALF: the last of the NT tiles is half of one; one of its own is 8 columns of squares, too.
template <int XG, int NT, int DEPTH, bool GLU, typename TO, bool F32, int NORM, bool HALF>
HS_DEVICE void skinny_block(int bx, int by, int bz, const unsigned short* __restrict__ x, const unsigned short* __restrict__ w, void* p, const void* q,
                            int x_ld, int M, int N, int K, int ni, int rest_at, unsigned char* smem) {
  static_assert(!GLU || NT == 2, "a gate tile and an up tile");
  static_assert(!HALF || NT == 1 || NORM != kUpdate, "squares of whole tiles");
  using SK = Skinny<XG, NT, DEPTH, F32, HALF>;
  constexpr int ST = SK::ST, kCols = SK::kCols, kTileCols = GLU ? 16 : 8 * SK::WG;   // of a workgroup
  using TB = std::conditional_t<F32, float, unsigned short>;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int No = GLU ? N / 2 : N;
  const int n0 = bx * kTileCols;
  const int k0 = NORM == kPlain ? bz * ni : 0, k1 = NORM == kPlain ? min(K, k0 + ni) : K;
  if (NORM == kPlain && by != 0) {
    x += (long)by * late_args<SkinnyRest<NORM>>(rest_at)->x_bs;
    w += (long)by * N * K;
  }
  const unsigned char* wt[NT];
  unsigned w_row[SK::WG];
  unsigned x_row[XG];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int first = GLU ? n0 : min(n0 + 16 * nt, N - 1);   // of the tile's columns
    wt[nt] = reinterpret_cast<const unsigned char*>(w + ((long)(GLU ? nt * No : 0) + first) * K + k0);
#pragma unroll
    for (int h = 0; h < (HALF && nt == NT - 1 ? 1 : 2); ++h) w_row[2 * nt + h] = (unsigned)min(8 * h + (lane >> 3), No - 1 - first) * (unsigned)(2 * K);
  }
#pragma unroll
  for (int j = 0; j < XG; ++j) x_row[j] = (unsigned)min(8 * j + (lane >> 3), M - 1) * (unsigned)(2 * x_ld);
  f32x4 acc[NT][ST];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int st = 0; st < ST; ++st) acc[nt][st] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int IT = SK::kElems, SQ = kCols == 8 ? 8 : 4;   // kCols threads x SQ loads x 4 sums: 256 of them, rows of up to 4096 at 16 columns each
  [[maybe_unused]] f32x4 sq[IT][SQ];
  [[maybe_unused]] float res[IT][NT], wgt[NT];
  [[maybe_unused]] TB bs[NT];
  // for the epilogue, ahead of the copies: without branches, behind which the copies would be waited for, and first, since loads return in
  // order and a wait for the copies would be one for these too
  const int c = tid % kCols;
  const bool biased = NORM != kUpdate && q != nullptr && bz == 0;
  const TB* bias = static_cast<const TB*>(biased ? q : x);
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    [[maybe_unused]] const long m = min((tid + kSkThreads * i) / kCols, M - 1);
    if constexpr (NORM == kNormed) {
#pragma unroll
      for (int j = 0; j < SQ; ++j) sq[i][j] = *reinterpret_cast<const f32x4*>(static_cast<const float*>(p) + m * ni + min(4 * kCols * j + 4 * c, ni - 4));
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int n = (GLU ? nt * No : 0) + min(n0 + (GLU ? 0 : 16 * nt) + c, No - 1);
      if constexpr (NORM == kUpdate) res[i][nt] = static_cast<const float*>(p)[m * N + n];
      if (i == 0) {
        if constexpr (NORM == kUpdate) wgt[nt] = static_cast<const float*>(q)[n];
        else bs[nt] = bias[biased ? n : 0];
      }
    }
  }
  int act = 0, act_from = 0;
  float c0 = 0.f, c1 = 0.f, cols = 1.f, eps = 0.f;
  long out_ld = 0;
  TO* out = nullptr;
  [[maybe_unused]] float* squares = nullptr;
  [[maybe_unused]] const TB* late_bias = nullptr;
  SK::accumulate(acc, wt, w_row, reinterpret_cast<const unsigned char*>(x + k0), x_row, k1 - k0, smem, lane, wave, [&] {
    const auto rest = late_args<SkinnyRest<NORM>>(rest_at);
    out = static_cast<TO*>(rest->out);
    out_ld = NORM == kPlain ? rest->out_ld : GLU ? No : N;
    if constexpr (NORM == kPlain) out += (long)by * rest->out_bs + (long)bz * rest->out_zs;
    if constexpr (NORM == kUpdate) squares = rest->squares;
    act = rest->act;
    act_from = rest->act_from;
    c0 = rest->c0;
    c1 = rest->c1;
    cols = rest->cols;
    eps = rest->eps;
    asm volatile("" ::"s"(act), "s"(act_from), "s"(c0), "s"(c1), "s"(cols), "s"(eps), "s"(out), "s"(out_ld), "s"(squares));
    if constexpr (NORM == kUpdate) {
      late_bias = static_cast<const TB*>(rest->bias);
      if (late_bias != nullptr) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) bs[nt] = late_bias[n0 + 16 * nt + c];
      }
    }
  });
  float v[NT][IT];
  SK::reduce(v, acc, smem);
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int e = tid + kSkThreads * i, m = e / kCols;
    if (m >= M) continue;   // a row's lanes together
    if constexpr (NORM == kUpdate) {   // N is a multiple of the workgroup's columns
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int n = n0 + 16 * nt + e % kCols;
        const float r = res[i][nt] + (v[nt][i] + (late_bias != nullptr ? ldf<TB>(&bs[nt], 0) : 0.f));
        static_cast<float*>(p)[(long)m * N + n] = r;
        stf<TO>(out, m * out_ld + n, r * wgt[nt]);
        const float s = cols_sum<kCols>(r * r);
        if (e % kCols == 0) squares[(long)m * ni + n / kCols] = s;
      }
      continue;
    }
    if constexpr (NORM == kNormed) {
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < SQ; ++j)
        if (4 * kCols * j + 4 * c < ni) s += (sq[i][j][0] + sq[i][j][1]) + (sq[i][j][2] + sq[i][j][3]);
      const float inv = 1.f / sqrtf(cols_sum<kCols>(s) / cols + eps);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) v[nt][i] *= inv;
    }
    if constexpr (GLU) {
      const int n = n0 + (e & 15);
      if (n >= No) continue;
      const float gv = v[0][i] + (biased ? ldf<TB>(&bs[0], 0) : 0.f);
      const float uv = v[1][i] + (biased ? ldf<TB>(&bs[1], 0) : 0.f);
      stf<TO>(out, m * out_ld + n, act == 4 ? clamped_glu_f(gv, uv, c0) : gv * sigmoid_f(gv) * uv);
    } else {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int n = n0 + 16 * nt + e % kCols;
        if (n >= N || (HALF && NT > 1 && nt == NT - 1 && e % kCols >= 8)) continue;
        const float z = v[nt][i] + (biased ? ldf<TB>(&bs[nt], 0) : 0.f);
        stf<TO>(out, m * out_ld + n, skinny_act(z, n >= act_from ? act : -1, c0, c1));
      }
    }
  }
}

// launch.run<XG, NT, DEPTH, F32, HALF>() for a kUpdate product of up to 32 rows, K in halves: one rule for its launches. The number of its squares' blocks says
// whether its workgroups are to take 8 columns. Two pieces ahead for one tile, but for more than 16 rows of 32 bits: a decode step of 20 rows (width
// 1024) 122.4 us with two, 124.2 with one, in 32 bits 167.1 and 166.0, of 32 rows 128.4 and 130.0, 173.7 and 170.0.
template <bool F32, typename L> bool run_update(const L& launch, int M, int N, int K, int blocks) {
  if (blocks == N / 8) {
    if (M <= 8) return K > 4096 ? launch.template run<1, 1, 3, F32, true>() : launch.template run<1, 1, 2, F32, true>();
    return M <= 16 ? launch.template run<2, 1, 2, F32, true>() : launch.template run<4, 1, 2, F32, true>();
  }
  const int nt = skinny_tiles(M, (N + 15) / 16, K);   // 4 above 16 rows alone; N is a multiple of 64
  if (nt == 4) return launch.template run<4, 4, 1, F32, false>();
  if (nt == 2)
    return M <= 8 ? launch.template run<1, 2, 1, F32, false>() : M <= 16 ? launch.template run<2, 2, 1, F32, false>() : launch.template run<4, 2, 1, F32, false>();
  return M <= 8 ? launch.template run<1, 1, 2, F32, false>() : M <= 16 ? launch.template run<2, 1, 2, F32, false>()
       : launch.template run<4, 1, F32 ? 1 : 2, F32, false>();
}

}  // namespace
}  // namespace hipserve

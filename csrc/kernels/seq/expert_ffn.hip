// Expert GEMMs of the mixtures of experts over moe_align tiles: out[slot, :] = act(W[e] . x[row(slot)])
// where a tile is `tile` consecutive expert-sorted slots of one expert (tile_expert[t]; -1 = unused, and a
// value >= E, a bucket of pairs whose expert has no weights, is skipped too),
// row(slot) = slots[slot] / gather_k (the token row of the pair; first GEMM) or the slot itself
// (second GEMM) and act = none (0), squared ReLU (1) or a SiLU gate (2): W[e] = [gate rows; up rows], N / 2 each,
// and out[slot, c] = silu(gate_c . x) * (up_c . x) has N / 2 columns (a thread / lane holds a column's pair); act 3:
// the same with g sigmoid(1.702 g) (u + 1), both clamped at `limit`. row_scale: every product of a pair's row is
// multiplied by row_scale[pair] first (the pair's weight on its input: the products are linear in it). Any N and K: edges are bounds-checked. A workgroup
// computes a [32 slots x 64 columns] block, x and W staged through LDS in K-chunks of 32, fp32
// accumulation; bf16 and fp32 element types.
#include <algorithm>

#include "expert_rows.h"
#include "hipserve/seq_kernels.h"

namespace hipserve {
namespace {

constexpr int kTM = 32, kTN = 64, kTK = 32;

template <typename T>
__global__ __launch_bounds__(256) void expert_gemm_kernel(T* __restrict__ out, const T* __restrict__ x, long x_ld,
                                                          const T* __restrict__ w, const int* __restrict__ slots,
                                                          const int* __restrict__ tile_expert, int tile, int gather_k,
                                                          int N, int K, int act, int E,
                                                          const float* __restrict__ row_scale, float limit) {
  __shared__ float xscale[kTM];
  __shared__ float xs[kTM][kTK + 1], ws[kTN][kTK + 1];
  __shared__ long xrow[kTM];
  const int e = tile_expert[(blockIdx.y * kTM) / tile];
  if (e < 0 || e >= E) return;
  const int tid = threadIdx.x;
  const bool glu = act >= 2;
  const int No = glu ? N / 2 : N;   // output columns
  // gated: the block's 64 weight rows are 32 gate rows and the 32 up rows of the same output columns
  const int slot0 = blockIdx.y * kTM, n0 = blockIdx.x * (glu ? kTN / 2 : kTN);
  if (tid < kTM) {
    const int p = slots[slot0 + tid];
    xscale[tid] = (row_scale != nullptr && p >= 0) ? row_scale[p] : 1.f;
    xrow[tid] = p < 0 ? -1 : (gather_k > 0 ? (long)(p / gather_k) : (long)(slot0 + tid)) * x_ld;
  }
  const T* we = w + (long)e * N * K;
  const int tx = tid & 15, ty = tid >> 4;  // 4 columns x 2 slots per thread
  float acc[2][4] = {};
  for (int k0 = 0; k0 < K; k0 += kTK) {
    __syncthreads();
    for (int idx = tid; idx < kTM * kTK; idx += 256) {
      const int r = idx / kTK, k = idx % kTK;
      const long xr = xrow[r];
      xs[r][k] = (xr >= 0 && k0 + k < K) ? ldf<T>(x, xr + k0 + k) : 0.f;
    }
    for (int idx = tid; idx < kTN * kTK; idx += 256) {
      const int c = idx / kTK, k = idx % kTK;
      const int col = glu ? n0 + (c & 31) : n0 + c;              // output column
      const long wrow = glu && c >= 32 ? (long)No + col : col;   // its weight row (the up row for c >= 32)
      ws[c][k] = (col < No && k0 + k < K) ? ldf<T>(we, wrow * K + k0 + k) : 0.f;
    }
    __syncthreads();
#pragma unroll 8
    for (int k = 0; k < kTK; ++k) {
      const float a0 = xs[ty * 2][k], a1 = xs[ty * 2 + 1][k];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float b = ws[tx + 16 * j][k];
        acc[0][j] = __builtin_fmaf(a0, b, acc[0][j]);
        acc[1][j] = __builtin_fmaf(a1, b, acc[1][j]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = ty * 2 + i;
    if (xrow[r] < 0) continue;
    const float f = xscale[r];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] *= f;
    if (glu) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {   // columns tx, tx + 16: gates in acc[.][j], ups in acc[.][j + 2]
        const int c = n0 + tx + 16 * j;
        const float gv = acc[i][j], uv = acc[i][j + 2];
        if (c < No)
          stf<T>(out, (long)(slot0 + r) * No + c, act == 3 ? clamped_glu_f(gv, uv, limit) : gv * sigmoid_f(gv) * uv);
      }
      continue;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = n0 + tx + 16 * j;
      if (c >= N) continue;
      float v = acc[i][j];
      if (act == 1) { v = fmaxf(v, 0.f); v *= v; }
      stf<T>(out, (long)(slot0 + r) * N + c, v);
    }
  }
}

// bf16 on the matrix cores: a workgroup (4 waves) computes [16 ST slots x 128 columns]; wave w owns
// columns 32 w .. 32 w + 31. Operands go from global memory straight into the MFMA registers (16 bytes
// per lane and step: 8 consecutive k of one W row / one x row); W rows are read once per slot tile, the
// x rows of the tile are shared by the four waves through L1. Needs K % 8 == 0, N % 8 == 0.
template <int ST>
__global__ __launch_bounds__(256) void expert_gemm_mfma_kernel(
    unsigned short* __restrict__ out, const unsigned short* __restrict__ x, long x_ld,
    const unsigned short* __restrict__ w, const int* __restrict__ slots, const int* __restrict__ tile_expert,
    int gather_k, int N, int K, int act, int E, const float* __restrict__ row_scale, float limit) {
  const int e = tile_expert[blockIdx.y];
  if (e < 0 || e >= E) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int slot0 = blockIdx.y * 16 * ST;
  const bool glu = act >= 2;
  const int No = glu ? N / 2 : N;
  // gated: the wave's two 16-column tiles are the gate rows and the up rows of the SAME 16 output columns
  const int n0 = glu ? blockIdx.x * 64 + 16 * wave : blockIdx.x * 128 + 32 * wave;
  if (n0 >= No) return;
  const unsigned short* xr[ST];
  bool live[ST];
  float xscale[ST];
#pragma unroll
  for (int st = 0; st < ST; ++st) {
    const int slot = slot0 + 16 * st + c;
    const int p = slots[slot];
    xscale[st] = (row_scale != nullptr && p >= 0) ? row_scale[p] : 1.f;
    live[st] = p >= 0;
    xr[st] = x + (p < 0 ? 0 : (gather_k > 0 ? (long)(p / gather_k) : (long)slot)) * x_ld + 8 * g;
  }
  const unsigned short* wr[2];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt)
    wr[nt] = w + ((long)e * N + (glu ? nt * No + min(n0 + c, No - 1) : min(n0 + 16 * nt + c, N - 1))) * K + 8 * g;
  f32x4 acc[2][ST];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt)
#pragma unroll
    for (int st = 0; st < ST; ++st) acc[nt][st] = f32x4{0.f, 0.f, 0.f, 0.f};
  const u16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  constexpr int kU = 4;  // k steps whose operand loads are in flight together
  for (int k0 = 0; k0 < K; k0 += 32 * kU) {
    u16x8 a[kU][2], b[kU][ST];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int k = k0 + 32 * u;
      const bool in = k + 8 * g < K;
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) a[u][nt] = in ? *reinterpret_cast<const u16x8*>(wr[nt] + k) : zero;
#pragma unroll
      for (int st = 0; st < ST; ++st) b[u][st] = (in && live[st]) ? *reinterpret_cast<const u16x8*>(xr[st] + k) : zero;
    }
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int st = 0; st < ST; ++st)
          acc[nt][st] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[u][nt]),
                                                                __builtin_bit_cast(bf16x8, b[u][st]), acc[nt][st], 0, 0, 0);
  }
  // lane (c, g): columns n0 + 16 nt + 4 g .. + 3 of slot 16 st + c
#pragma unroll
  for (int st = 0; st < ST; ++st) {
    if (!live[st]) continue;
    const long slot = slot0 + 16 * st + c;
    acc[0][st] *= xscale[st];
    acc[1][st] *= xscale[st];
    if (glu) {
      const int n = n0 + 4 * g;
      if (n >= No) continue;  // No % 4 == 0: the four columns are inside together
      u16x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float gv = acc[0][st][j], uv = acc[1][st][j];
        o[j] = f32_to_bf16(act == 3 ? clamped_glu_f(gv, uv, limit) : gv * sigmoid_f(gv) * uv);
      }
      *reinterpret_cast<u16x4*>(out + slot * No + n) = o;
      continue;
    }
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const int n = n0 + 16 * nt + 4 * g;
      if (n >= N) continue;  // N % 8 == 0: the four columns are inside together
      u16x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float v = acc[nt][st][j];
        if (act == 1) { v = fmaxf(v, 0.f); v *= v; }
        o[j] = f32_to_bf16(v);
      }
      *reinterpret_cast<u16x4*>(out + slot * N + n) = o;
    }
  }
}

// bf16, tiles of 128 slots (prompts of some dozen to a few thousand rows): a workgroup of four waves computes a tile's live rows (32, 64, 96 or 128 of them)
// x 64 columns, a wave 16 columns of all rows. Rows and weights are copied to LDS as in skinny.h, stages of 64 k, two ahead, one barrier each. What
// bounds it is what a compute unit takes in, 40 - 50 KB per us: an expert's weights once per 128 rows instead of once per 32, its rows once per
// 64 columns instead of once per 16. 72 KB of LDS, so that two workgroups fit a compute unit: with three or five stages ahead and one workgroup 54 and 55 us
// where this takes 43 (16 experts, 4000 pairs, 1024 x 2048), nowhere less than 2 % faster. us of both products by tiles of 32 (expert_rows; packed weights) ->
// this, 16 experts of 1024 x 2048: 200 pairs 32.8 -> 28.9, 600 47.6 -> 31.6, 1400 76 -> 39, 4000 167 (96) -> 82; 8 of 2048 x 4096: 600 pairs 128 -> 69, 2000 303
// -> 145 (2000 pairs; packed 165); 8 of 512 x 1024: 1400 24.1 (24.4) -> 19.7, 4000 59 (55) -> 27.6.
constexpr int kMidRows = 128, kMidCols = 64, kMidStages = 3, kMidLds = kMidStages * (kMidRows + kMidCols) * 128;
template <int RT>
HS_DEVICE void expert_mid(unsigned short* __restrict__ out, const unsigned short* __restrict__ x, unsigned x_ld, const unsigned char* __restrict__ we,
                          const int (&mine)[2], int slot0, int n0, int gather_k, int gather_shift, int N, int K, int act, unsigned char* smem) {
  constexpr int D = kMidStages, kX = RT * 2048, kStage = kX + kMidCols * 128, XC = RT / 2, kCopies = XC + 2;   // XC: copies of a wave's rows per stage
  static_assert(RT % 2 == 0 && kCopies * (D - 2) < 64, "copies that a wait can count");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4, r8 = lane >> 3;
  const unsigned lds0 = lds_at(smem);
  unsigned x_at[XC], w_at[2];
  auto part = [&](int row) { return 16u * ((lane & 7) ^ (row >> 1 & 7)); };
  auto pair_of = [&](int r) {   // every lane asks
    const int a = __shfl(mine[0], r & 63, 64), b = __shfl(mine[1], r & 63, 64);
    return r < 64 ? a : b;
  };
#pragma unroll
  for (int j = 0; j < XC; ++j) {
    const int r = 8 * (wave * XC + j) + r8, p = pair_of(r);
    const int from = gather_shift >= 0 ? p >> gather_shift : gather_k > 0 ? p / gather_k : slot0 + r;
    x_at[j] = (unsigned)(p < 0 ? 0 : from) * x_ld * 2 + part(r);   // no pair: any row
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = 8 * (2 * wave + j) + r8;
    w_at[j] = (unsigned)min(r, N - 1 - n0) * (unsigned)K * 2 + part(r);
  }
  const unsigned char* xb = reinterpret_cast<const unsigned char*>(x);
  const int nst = K >> 6;
  auto copy = [&](int st) {
    const unsigned to = lds0 + st % D * kStage;
    const long k = 128L * st;
#pragma unroll
    for (int j = 0; j < XC; ++j) copy_1k(xb + k, x_at[j], to + (wave * XC + j) * 1024);
#pragma unroll
    for (int j = 0; j < 2; ++j) copy_1k(we + k, w_at[j], to + kX + (2 * wave + j) * 1024);
  };
  f32x4 acc[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < D - 1; ++i)
    if (i < nst) copy(i);
  int at[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) at[s] = c * 128 + (((4 * s + g) ^ (c >> 1)) << 4);
  for (int st = 0; st < nst; ++st) {
    // the stage's copies are there, every wave's; and every wave has read the stage before, whose place the next copies take
    if (st + D - 1 <= nst) barrier_copies<kCopies * (D - 2)>();
    else barrier_copies<0>();
    if (st + D - 1 < nst) copy(st + D - 1);
    const unsigned char* t = smem + st % D * kStage;
    u16x8 a[2], b[2][RT];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      a[s] = *reinterpret_cast<const u16x8*>(t + kX + wave * 2048 + at[s]);
#pragma unroll
      for (int i = 0; i < RT; ++i) b[s][i] = *reinterpret_cast<const u16x8*>(t + i * 2048 + at[s]);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < RT; ++i)
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[s]), __builtin_bit_cast(bf16x8, b[s][i]), acc[i], 0, 0, 0);
  }
  // lane (c, g): columns n0 + 16 wave + 4 g .. + 3 of slot 16 i + c
  const int n = n0 + 16 * wave + 4 * g;
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int r = 16 * i + c, p = pair_of(r);
    if (p < 0 || n >= N) continue;   // N % 8 == 0: the four columns are inside together
    u16x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float v = acc[i][j];
      if (act == 1) { v = fmaxf(v, 0.f); v *= v; }
      o[j] = f32_to_bf16(v);
    }
    *reinterpret_cast<u16x4*>(out + (long)(slot0 + r) * N + n) = o;
  }
}

__global__ __launch_bounds__(256) void expert_gemm_mid_kernel(
    const int* __restrict__ slots, const int* __restrict__ tile_expert, const unsigned short* __restrict__ x, const unsigned short* __restrict__ w,
    int x_ld, int N, int K, int E, int gather_k, int gather_shift, unsigned short* __restrict__ out, int act) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63, slot0 = blockIdx.y * kMidRows, n0 = blockIdx.x * kMidCols;
  const int e = tile_expert[blockIdx.y], mine[2] = {slots[slot0 + lane], slots[slot0 + 64 + lane]};
  const unsigned long low = __ballot(mine[0] >= 0), high = __ballot(mine[1] >= 0);
  const int rows = high != 0 ? 128 - __clzll(high) : 64 - (low != 0 ? __clzll(low) : 64);   // up to the last one: a table may have slots without a pair before it
  if (e < 0 || e >= E) return;
  const unsigned char* we = reinterpret_cast<const unsigned char*>(w + ((long)e * N + n0) * K);
#define HS_EM(RT) expert_mid<RT>(out, x, x_ld, we, mine, slot0, n0, gather_k, gather_shift, N, K, act, smem)
  if (rows <= 32) HS_EM(2);
  else if (rows <= 64) HS_EM(4);
  else if (rows <= 96) HS_EM(6);
  else HS_EM(8);
#undef HS_EM
}

template <int NT, bool GLU>
__global__ __launch_bounds__(kSkThreads) void expert_gemm_skinny_kernel(
    const int* __restrict__ slots, const int* __restrict__ tile_expert, const unsigned short* __restrict__ x, const unsigned short* __restrict__ w,
    int x_ld, int N, int K, int E, int gather_k, int gather_shift, const ExpertRest) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  expert_block<NT, GLU>(blockIdx.x, blockIdx.y, slots, tile_expert, x, w, x_ld, N, K, E, gather_k, gather_shift, offsetof(ExpertArgs, rest), smem);
}

}  // namespace

// Which of the two kernels serves `ntiles` launched tiles of 32 slots that hold so many pairs: the one for few rows, but for thousands of workgroups of
// 512 k and fewer, whose start costs more than their products, and where thousands of workgroups find no pair (0.37 us per 1000; only a launch of the
// whole capacity has so many). 244 sizes of 4 to 256 experts, k 512 - 4096, 1 to 255 pairs per expert, gated and not, cold weights: 0.4 % longer than the
// faster one on average, at most 15 %, with the whole capacity launched 0.4 and 17 %. us, tile kernel / this one: 16 experts, 2048 x 1024: 32, 128 and 4080
// pairs 17.5 / 12.8, 18.0 / 16.0, 131 / 93; 8 experts, 4096 x 2048, 16 pairs 35.1 / 27.5; 64 experts, 2048 x 704, 128 and 16320 pairs 37.6 / 31.7, 344 /
// 287; 128 experts, 2048 x 768, 64 pairs 40.2 / 31.1; but 32 experts, 1000 x 520, 4096 pairs 36 / 45, 256 experts, 2048 x 512, 512 and 65280 pairs 91 / 107, 987 /
// 1086, and with all of 125 tiles launched for 4 pairs, 128 experts, 4096 x 1024, 14 / 27. Two tiles of 16 columns per workgroup are hardly ever
// faster (16 experts, 2048 x 1024, 82 pairs: 19.1, 1400 pairs: 51).
bool expert_rows_pay(long ntiles, long pairs, long cols, long K) {
  const long per_tile = (cols + 15) / 16;
  return (K >= 640 || per_tile * ntiles <= 8192) && per_tile * (ntiles - pairs) <= 8192;
}

bool expert_rows_ok(const ExpertRows& ex) {
  return ex.ntiles > 0 && ex.act <= 1 && ex.K % 8 == 0 && ex.N % 8 == 0 && ex.x_ld % 8 == 0 && ex.K < (1 << 24) && 2L * ex.cap * ex.x_ld < (1L << 32) && (uintptr_t)ex.x % 16 == 0 &&
         (uintptr_t)ex.w % 16 == 0 && expert_rows_pay(ex.ntiles, ex.pairs, ex.N, ex.K);
}

void launch_expert_gemm(void* out, const void* x, long x_ld, const void* w, const int* slots, const int* tile_expert,
                        int ntiles_cap, int ntiles, int tile, int gather_k, int N, int K, int act, int E, const float* row_scale,
                        float limit, int pairs, bool f32, hipStream_t s) {
  if (ntiles_cap <= 0) return;
  // the capacity covers a partly filled tile per expert
  pairs = pairs > 0 ? pairs : std::max(1, ntiles_cap * tile - E * (tile - 1));
  const int No = act >= 2 ? N / 2 : N;
  if (!f32 && tile == kMidRows && act <= 1 && row_scale == nullptr && K % 64 == 0 && N % 8 == 0 && x_ld % 8 == 0 && K < (1 << 24) &&
      2L * ntiles_cap * tile * x_ld < (1L << 32) && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0) {
    const dim3 mg((N + kMidCols - 1) / kMidCols, ntiles);
    const int shift = gather_k > 0 && (gather_k & (gather_k - 1)) == 0 ? __builtin_ctz(gather_k) : -1;
    if (allow_lds(&expert_gemm_mid_kernel, kMidLds)) {
      expert_gemm_mid_kernel<<<mg, 256, kMidLds, s>>>(slots, tile_expert, (const unsigned short*)x, (const unsigned short*)w, (int)x_ld, N, K, E, gather_k,
                                                      shift, (unsigned short*)out, act);
      return;
    }
  }
  if (!f32 && K % 8 == 0 && No % 8 == 0 && x_ld % 8 == 0 && (tile == 32 || tile == 64)) {
    dim3 mg(act >= 2 ? (No + 63) / 64 : (N + 127) / 128, ntiles);
    auto o = (unsigned short*)out;
    auto xi = (const unsigned short*)x, wi = (const unsigned short*)w;
    if (tile == 32 && K < (1 << 24) && 2L * ntiles_cap * tile * x_ld < (1L << 32) && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0 &&
        expert_rows_pay(ntiles, pairs, No, K)) {
      const dim3 sg((No + 15) / 16, ntiles);
      const int shift = gather_k > 0 && (gather_k & (gather_k - 1)) == 0 ? __builtin_ctz(gather_k) : -1;
      if (act >= 2)
        expert_gemm_skinny_kernel<2, true><<<sg, kSkThreads, expert_lds<2>(), s>>>(slots, tile_expert, xi, wi, (int)x_ld, N, K, E, gather_k, shift,
                                                                                  ExpertRest{o, row_scale, act, limit});
      else
        expert_gemm_skinny_kernel<1, false><<<sg, kSkThreads, expert_lds<1>(), s>>>(slots, tile_expert, xi, wi, (int)x_ld, N, K, E, gather_k, shift,
                                                                                   ExpertRest{o, row_scale, act, limit});
      return;
    }
    if (tile == 32) expert_gemm_mfma_kernel<2><<<mg, 256, 0, s>>>(o, xi, x_ld, wi, slots, tile_expert, gather_k, N, K, act, E, row_scale, limit);
    else expert_gemm_mfma_kernel<4><<<mg, 256, 0, s>>>(o, xi, x_ld, wi, slots, tile_expert, gather_k, N, K, act, E, row_scale, limit);
    return;
  }
  dim3 grid(act >= 2 ? (No + kTN / 2 - 1) / (kTN / 2) : (N + kTN - 1) / kTN, (long)ntiles * tile / kTM);
  if (f32)
    expert_gemm_kernel<float><<<grid, 256, 0, s>>>((float*)out, (const float*)x, x_ld, (const float*)w, slots,
                                                   tile_expert, tile, gather_k, N, K, act, E, row_scale, limit);
  else
    expert_gemm_kernel<unsigned short><<<grid, 256, 0, s>>>((unsigned short*)out, (const unsigned short*)x, x_ld,
                                                            (const unsigned short*)w, slots, tile_expert, tile,
                                                            gather_k, N, K, act, E, row_scale, limit);
}

}  // namespace hipserve

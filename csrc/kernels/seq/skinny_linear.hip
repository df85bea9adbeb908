// out[b, m, :] = act(x[b, m, :] . W[b]^T + bias) for up to 64 rows m (decode steps and short prompts): bf16 or 32-bit
// operands, 32-bit accumulation, a result of the operands' type or in 32 bits, row and batch strides of their own for x and out.
// act: 0 tanh, 1 xIELU, 2 squared ReLU, 3 SiLU gate, 4 clamped gate (3, 4: W = [gate rows; up rows], half as many
// columns in out), 5 soft cap, -1 none; they see the unrounded product.
#include "skinny.h"

#include <type_traits>

#include "hipserve/seq_kernels.h"

namespace hipserve {
namespace {

HS_DEVICE float skinny_act(float z, int act, float c0, float c1) {
  if (act == 0) return tanhf(z);
  if (act == 1) return z > 0.f ? c0 * z * z + 0.5f * z : c1 * (expm1f(z) - z) + 0.5f * z;
  if (act == 2) { z = fmaxf(z, 0.f); return z * z; }
  if (act == 5) return tanhf(z / c0) * c0;
  return z;
}

// ST: 16-row tiles; NT: 16-column tiles (GLU: the gate's and the up projection's of the same 16 output columns);
// KU: k steps of 32 whose loads a wave has in flight.
// F32: 32-bit operands, x, w, their strides and K in 16-bit halves (skinny.h).
template <int ST, int NT, int KU, bool GLU, typename TO, bool F32>
__global__ __launch_bounds__(kSkThreads) void skinny_linear_kernel(
    TO* __restrict__ out, long out_ld, long out_bs, const unsigned short* __restrict__ x, long x_ld, long x_bs,
    const unsigned short* __restrict__ w, const void* __restrict__ bias_, int M, int N, int K, int act, float c0, float c1) {
  static_assert(!GLU || NT == 2, "a gate tile and an up tile");
  using TB = std::conditional_t<F32, float, unsigned short>;
  const TB* bias = static_cast<const TB*>(bias_);
  __shared__ __attribute__((aligned(16))) float red[kSkWaves * 16 * ST * kSkLd];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, g = lane >> 4;
  const int No = GLU ? N / 2 : N;
  const int n0 = blockIdx.x * (GLU ? 16 : 16 * NT);
  x += (long)blockIdx.y * x_bs;
  w += (long)blockIdx.y * N * K;
  const bool low = c < 8;
  const int g8 = g + 4 * (c >> 3);
  const unsigned short* wr[NT][2];
  const unsigned short* xr[ST][2];
  bool live[ST][2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int cc = (c & 7) + 8 * h;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      wr[nt][h] = w + (long)(GLU ? nt * No + min(n0 + cc, No - 1) : min(n0 + 16 * nt + cc, N - 1)) * K + 8 * g8;
#pragma unroll
    for (int st = 0; st < ST; ++st) {
      live[st][h] = 16 * st + cc < M;
      xr[st][h] = x + (live[st][h] ? 16 * st + cc : 0) * x_ld + 8 * g8;
    }
  }
  f32x4 acc[NT][ST];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int st = 0; st < ST; ++st) acc[nt][st] = f32x4{0.f, 0.f, 0.f, 0.f};
  skinny_accumulate<ST, NT, KU, F32>(acc, wr, xr, live, K, g8, low, wave);
  float v[NT][(ST + 1) / 2];
  skinny_reduce<ST, NT>(v, acc, red);
  out += (long)blockIdx.y * out_bs;
#pragma unroll
  for (int i = 0; i < (ST + 1) / 2; ++i) {
    const int e = tid + kSkThreads * i, m = e >> 4;
    if (m >= M) continue;
    if constexpr (GLU) {
      const int n = n0 + (e & 15);
      if (n >= No) continue;
      const float gv = v[0][i] + (bias != nullptr ? ldf<TB>(bias, n) : 0.f);
      const float uv = v[1][i] + (bias != nullptr ? ldf<TB>(bias, No + n) : 0.f);
      stf<TO>(out, m * out_ld + n, act == 4 ? clamped_glu_f(gv, uv, c0) : gv * sigmoid_f(gv) * uv);
    } else {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int n = n0 + 16 * nt + (e & 15);
        if (n >= N) continue;
        const float z = v[nt][i] + (bias != nullptr ? ldf<TB>(bias, n) : 0.f);
        stf<TO>(out, m * out_ld + n, skinny_act(z, act, c0, c1));
      }
    }
  }
}

template <int ST, int NT, int KU, bool GLU>
void launch_one(void* out, bool out_f32, long out_ld, long out_bs, const void* x, long x_ld, long x_bs, const void* w,
                const void* bias, bool f32, int batch, int M, int N, int K, int act, float c0, float c1, hipStream_t s) {
  const int cols = GLU ? N / 2 : N, per = GLU ? 16 : 16 * NT;
  const dim3 grid((cols + per - 1) / per, batch);
  auto xi = (const unsigned short*)x, wi = (const unsigned short*)w;
  if (f32)
    skinny_linear_kernel<ST, NT, KU, GLU, float, true><<<grid, kSkThreads, 0, s>>>((float*)out, out_ld, out_bs, xi, x_ld, x_bs, wi,
                                                                                  bias, M, N, K, act, c0, c1);
  else if (out_f32)
    skinny_linear_kernel<ST, NT, KU, GLU, float, false><<<grid, kSkThreads, 0, s>>>((float*)out, out_ld, out_bs, xi, x_ld, x_bs, wi,
                                                                                   bias, M, N, K, act, c0, c1);
  else
    skinny_linear_kernel<ST, NT, KU, GLU, unsigned short, false><<<grid, kSkThreads, 0, s>>>(
        (unsigned short*)out, out_ld, out_bs, xi, x_ld, x_bs, wi, bias, M, N, K, act, c0, c1);
}

}  // namespace

void launch_skinny_linear(void* out, bool out_f32, long out_ld, long out_bs, const void* x, long x_ld, long x_bs,
                          const void* w, const void* bias, bool f32, int batch, int M, int N, int K, int act, float c0, float c1,
                          hipStream_t s) {
  if (batch <= 0 || M <= 0 || N <= 0) return;
  if (f32) { x_ld *= 2; x_bs *= 2; K *= 2; }   // in halves
#define HS_SK(ST, NT, KU, GLU) \
  launch_one<ST, NT, KU, GLU>(out, out_f32, out_ld, out_bs, x, x_ld, x_bs, w, bias, f32, batch, M, N, K, act, c0, c1, s)
  // the loads in flight per wave cover K in one go where the registers allow it: KU steps of 32 k on 8 waves
  if (act == 3 || act == 4) {
    if (M <= 16) HS_SK(1, 2, 4, true);
    else if (M <= 32) HS_SK(2, 2, 4, true);
    else HS_SK(4, 2, 4, true);
  } else if (K <= 512) {
    if (M <= 16) HS_SK(1, 1, 2, false);
    else if (M <= 32) HS_SK(2, 1, 2, false);
    else HS_SK(4, 1, 2, false);
  } else if (M <= 4 && K > 1024) {
    HS_SK(1, 1, 8, false);
  } else {
    if (M <= 16) HS_SK(1, 1, 4, false);
    else if (M <= 32) HS_SK(2, 1, 4, false);
    else HS_SK(4, 1, 2, false);
  }
#undef HS_SK
}

}  // namespace hipserve

// A workgroup's part of the generalized delta rule's decode step (delta_rule_step.hip), for its own launch and for one that holds window attention besides
// (window_delta_step.hip).
#pragma once
#include "seq_common.h"

namespace hipserve {
namespace {

constexpr int kD = 64;

// w2 (LOW): [heads * 64, rank], rank a multiple of 32; the row's bottleneck lies behind the five parts of `proj`. Else wl is the product.
// The sequence's numbers and the arguments that are no parameters of the first 14 words are asked for in one batch: 1 and
// 16 rows of 32 heads with the bottleneck 3.75 -> 3.67, 6.62 -> 6.30 us in a loop.
struct DeltaRuleRest {
  void* out;
  long out_ld;
  const float *w0, *norm_w;
  float eps, out_scale;
};
constexpr int kDeltaThreads = 256, kDeltaLds = (4 + 4 * 5 + 2 * 4) * kD * 4;
template <typename T, bool LOW>
HS_DEVICE void delta_rule_step_block(int h, int s, const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx, const int* __restrict__ seq_state,
                                     const T* __restrict__ proj, float* __restrict__ S, const void* __restrict__ low, int heads, int rank,
                                     const float* __restrict__ a_b, long ld, const DeltaRuleRest& rest, float* lds) {
  auto chan = reinterpret_cast<float(*)[5][kD]>(lds);                  // [wave] w, a, u, k, r
  auto sums = reinterpret_cast<float(*)[4][kD]>(lds + 4 * 5 * kD);     // x, o: [wave]
  [[maybe_unused]] auto decay = reinterpret_cast<float(*)[kD]>(lds + (4 * 5 + 2 * 4) * kD);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long t = seq_cu[s], after = seq_cu[s + 1];
  const int ctx = seq_ctx[s], slot = seq_state[s];
  const float *__restrict__ const w0 = rest.w0, *__restrict__ const norm_w = rest.norm_w;
  const float eps = rest.eps, out_scale = rest.out_scale;
  T* __restrict__ const out = static_cast<T*>(rest.out);
  const long out_ld = rest.out_ld;
  [[maybe_unused]] const T* __restrict__ const w2 = static_cast<const T*>(low);           // LOW
  [[maybe_unused]] const float* __restrict__ const wl = static_cast<const float*>(low);   // not LOW
  asm volatile("" ::"s"(t), "s"(after), "s"(ctx), "s"(slot), "s"(a_b), "s"(ld), "s"(w0), "s"(norm_w), "s"(eps), "s"(out_scale), "s"(out), "s"(out_ld));
  if (after <= t) return;
  const int N = heads * kD, c = h * kD + lane, v0 = 4 * (tid & 15), k0 = 4 * (tid >> 4);
  const T* row = proj + t * ld;
  float* Sp = S + (((long)slot * heads + h) * kD + k0) * kD + v0;
  const bool carried = ctx > 1;
  f32x4 st[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) st[i] = carried ? *reinterpret_cast<const f32x4*>(Sp + i * kD) : f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 val;
#pragma unroll
  for (int e = 0; e < 4; ++e) val[e] = ldf<T>(row, 2 * N + h * kD + v0 + e);
  const float k = ldf<T>(row, N + c), r = ldf<T>(row, c), a = ldf<T>(row, 3 * N + c), gate = ldf<T>(row, 4 * N + c);
  const float w0_c = w0[c], a_b_c = a_b[c], norm_c = norm_w[c];
  float d = 0.f;
  if constexpr (LOW) {
    const int part = rank / 4, j0 = __builtin_amdgcn_readfirstlane(wave) * part;
    const T *wr = w2 + (long)c * rank + j0, *lr = row + 5 * N + j0;
    for (int j = 0; j < part; j += 8) {
      float a8[8], b8[8];
      Row<T, 8>::ld(wr + j, a8);
      Row<T, 8>::ld(lr + j, b8);
#pragma unroll
      for (int e = 0; e < 8; ++e) d = __builtin_fmaf(a8[e], b8[e], d);
    }
    decay[wave][lane] = d;
    __syncthreads();
    d = (decay[0][lane] + decay[1][lane]) + (decay[2][lane] + decay[3][lane]);
  } else {
    d = wl[t * N + c];
  }
  const float u = k / sqrtf(wave_sum(k * k) + 1e-6f);
  float(*mine)[kD] = chan[wave];
  mine[0][lane] = expf(-0.60653065971263342f * sigmoid_f(d + w0_c));
  mine[1][lane] = sigmoid_f(a + a_b_c) * u;
  mine[2][lane] = u;
  mine[3][lane] = k;
  mine[4][lane] = r;
  __builtin_amdgcn_wave_barrier();   // the wave reads what the wave wrote
  auto rows = [&](int j) { return *reinterpret_cast<const f32x4*>(&mine[j][k0]); };
  // sum over the wave's 16 rows, then over the waves
  auto total = [&](f32x4 p, float(*to)[kD]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      p[e] += __shfl_xor(p[e], 16, 64);
      p[e] += __shfl_xor(p[e], 32, 64);
    }
    if (lane < 16) *reinterpret_cast<f32x4*>(&to[wave][v0]) = p;
    __syncthreads();
  };
  const f32x4 uu = rows(2);
  total(uu[0] * st[0] + uu[1] * st[1] + (uu[2] * st[2] + uu[3] * st[3]), sums[0]);
  f32x4 x = *reinterpret_cast<const f32x4*>(&sums[0][0][v0]);
#pragma unroll
  for (int w = 1; w < 4; ++w) x += *reinterpret_cast<const f32x4*>(&sums[0][w][v0]);
  const f32x4 w = rows(0), au = rows(1), kk = rows(3), rr = rows(4);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    st[i] = w[i] * st[i] - au[i] * x + kk[i] * val;
    *reinterpret_cast<f32x4*>(Sp + i * kD) = st[i];
  }
  total(rr[0] * st[0] + rr[1] * st[1] + (rr[2] * st[2] + rr[3] * st[3]), sums[1]);
  if (wave != 0) return;
  const float o = (sums[1][0][lane] + sums[1][1][lane]) + (sums[1][2][lane] + sums[1][3][lane]);
  const float inv = out_scale / sqrtf(wave_sum(o * o) / (float)kD + eps);
  stf<T>(out, t * out_ld + c, o * inv * norm_c * sigmoid_f(gate));
}

}  // namespace
}  // namespace hipserve

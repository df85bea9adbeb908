// A channel's part of the update of the convolution's inputs that a sequence keeps (delta_scan.hip), for its own launch and for one that holds a product
// besides (update_conv.hip).
#pragma once
#include "seq_common.h"

namespace hipserve {
namespace {

// The last taps - 1 conv inputs of every sequence into its slot (after the prepare kernel has read the old ones).
constexpr int kMaxHist = 15;
// HIST inputs are kept per channel (0: taps - 1, up to kMaxHist). All loads side by side, of rows that exist, and the sequence's numbers in one batch: one
// row of four taps beside the step before it (below).
template <typename T, int HIST>
HS_DEVICE void conv_update_block(int s, int c, const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx, const int* __restrict__ seq_state,
                                 const T* __restrict__ proj, float* __restrict__ conv_state, int C, int taps, long ld) {
  constexpr int N = HIST > 0 ? HIST : kMaxHist;
  const int r0 = seq_cu[s], r1 = seq_cu[s + 1], ctx = seq_ctx[s], slot = seq_state[s], hist = HIST > 0 ? HIST : taps - 1;
  asm volatile("" ::"s"(r0), "s"(r1), "s"(ctx), "s"(slot), "s"(ld));
  const int n = r1 - r0;
  if (c >= C || n <= 0 || hist <= 0) return;
  const bool carried = ctx - n > 0;
  float* cs = conv_state + (long)slot * hist * C + c;
  const T* rows = proj + (long)r0 * ld + c;
  float old[N], now[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {   // new input i is row n - hist + i of the step, or (negative) one of the old ones
    if (i >= hist) continue;
    const int j = n - hist + i;
    now[i] = ldf<T>(rows, (long)max(j, 0) * ld);
    old[i] = cs[(long)min(max(hist + j, 0), hist - 1) * C];
  }
#pragma unroll
  for (int i = 0; i < N; ++i)
    if (i < hist) cs[(long)i * C] = n - hist + i >= 0 ? now[i] : carried ? old[i] : 0.f;
}

}  // namespace
}  // namespace hipserve

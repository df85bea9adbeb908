// The generalized delta rule (delta_scan.hip) of a step in which every sequence has one row, heads of 64: preparation,
// recurrence, norm and gate in one launch, a workgroup per (sequence, head).
//   S' = diag(w) S - a x^T + k v^T,  x = S^T u;  out = o / rms(o) * norm * sigmoid(gate) * scale,  o = S'^T r
// What bounds it: the chain row -> u -> x -> S' -> o -> out, and the state's 16 KB in and out. A thread holds 4 x 4 elements of
// the state, loaded by 16 bytes side by side; every wave prepares the 64 channels for itself (a lane each), so two
// barriers, for the sums over the rows, are all. As three launches (five row vectors written as fp32 and read back, the state
// read by 4-byte columns, one wave per head for the norm): 16 sequences x 32 heads in bf16 27.7 us, this 6.7
// (one sequence x 16 heads 13.0, 4.5). The decays' bottleneck (its product w2 . low, 64 of its rows per head) can come with it: each wave sums
// a quarter of the rank for all channels, 8 KB of weights beside the state's 16. One sequence, in a captured step: 2.4 + 4.3 -> 4.7 us.
#include "delta_rule_step.h"
#include "hipserve/seq_kernels.h"

namespace hipserve {
namespace {

template <typename T, bool LOW>
__global__ __launch_bounds__(kDeltaThreads) void delta_rule_step_kernel(
    const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx, const int* __restrict__ seq_state, const T* __restrict__ proj,
    float* __restrict__ S, const void* __restrict__ low, int heads, int rank, const float* __restrict__ a_b, long ld, const DeltaRuleRest rest) {
  __shared__ __attribute__((aligned(16))) float lds[kDeltaLds / 4];
  delta_rule_step_block<T, LOW>(blockIdx.x, blockIdx.y, seq_cu, seq_ctx, seq_state, proj, S, low, heads, rank, a_b, ld, rest, lds);
}

}  // namespace

bool delta_rule_step_ok(int dim) { return dim == kD; }

void launch_delta_rule_step(void* out, long out_ld, float* S, const void* proj, long ld, const float* wl, const float* a_b,
                            const float* w0, const float* norm_w, const int* seq_cu, const int* seq_ctx, const int* seq_state,
                            int nseq, int heads, float eps, float out_scale, const void* w2, int rank, bool f32, hipStream_t s) {
  if (nseq <= 0) return;
  const dim3 grid(heads, nseq);
#define HS_DRS(T, LOW)                                                                                                             \
  delta_rule_step_kernel<T, LOW><<<grid, 256, 0, s>>>(seq_cu, seq_ctx, seq_state, (const T*)proj, S, LOW ? w2 : (const void*)wl, heads, rank, a_b, ld, \
                                                      DeltaRuleRest{out, out_ld, w0, norm_w, eps, out_scale})
  if (f32) { if (w2 != nullptr) HS_DRS(float, true); else HS_DRS(float, false); }
  else if (w2 != nullptr) HS_DRS(unsigned short, true);
  else HS_DRS(unsigned short, false);
#undef HS_DRS
}

}  // namespace hipserve

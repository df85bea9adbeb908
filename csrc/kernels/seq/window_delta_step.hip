// Window attention and the generalized delta rule of a decode step in one launch: the halves of a parallel mixer, which are independent of each other. Either
// is a chain of loads that depend on each other and of instructions that a wave issues in turn, on a few of the compute units; apart they are one chain behind
// the other with a launch (1.6 us when empty) between. A workgroup runs what its own launch would, with the same results; the attention's come first, as they
// take longest, and all have the threads and the LDS of the larger of the two: waves that a workgroup has no use for end at once (a barrier waits for those of
// its workgroup that are left). us of both, apart -> in one launch, in a captured step: one row of 8 heads over 2 of 128 and 16 of 64, 45 keys 13.0 -> 9.1, 16 rows of
// 16 over 4 and 32, 230 keys 17.7 -> 12.2; a step of width 1024 of one row 116 -> 111.5, of width 2048 of 16 rows 232 -> 226, in 32 bits, 3 rows, 300 keys, 8 us less.
#include "delta_rule_step.h"
#include "window_decode.h"

namespace hipserve {
namespace {

template <typename T> struct DeltaArgs {
  const int *seq_cu, *seq_ctx, *seq_state;
  const T* proj;
  float* S;
  const T* w2;
  int heads, rank, nseq;
  const float* a_b;
  long ld;
  DeltaRuleRest rest;
};

template <typename T, int D, int MODE>
__global__ __launch_bounds__(512) void window_delta_step_kernel(
    const T* __restrict__ proj, const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx, const int* __restrict__ seq_bt,
    const long* __restrict__ positions, const long* __restrict__ slots, int bt_width, unsigned sizes, const WindowRest<T, true> rest,
    const DeltaArgs<T> delta) {
  extern __shared__ __attribute__((aligned(16))) float both_lds[];
  int b = blockIdx.x;
  const int window_wgs = sizes & 0xffff, T_rows = sizes >> 16;   // one word: more would not reach the kernel in registers
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // a wave that its workgroup has no use for ends here: the barriers are the others'
  if (b < window_wgs) {
    if (wave >= rest.waves) return;
    const int rows = rest.seq1 - rest.seq0, per = rows * rest.kv_heads * rest.hchunks;
    const int z = __builtin_amdgcn_readfirstlane((unsigned)b / (unsigned)per);
    b -= z * per;
    const int y = __builtin_amdgcn_readfirstlane((unsigned)b / (unsigned)rows);
    window_decode_block<T, D, false, MODE>(b - y * rows, y, z, proj, seq_cu, seq_ctx, seq_bt, positions, slots, bt_width, T_rows, rest, both_lds);
    return;
  }
  if (wave >= kDeltaThreads / 64) return;
  b -= window_wgs;
  const int s = __builtin_amdgcn_readfirstlane((unsigned)b / (unsigned)delta.heads);
  delta_rule_step_block<T, true>(b - s * delta.heads, s, delta.seq_cu, delta.seq_ctx, delta.seq_state, delta.proj, delta.S, delta.w2, delta.heads, delta.rank,
                                 delta.a_b, delta.ld, delta.rest, both_lds);
}

template <typename T, int D>
bool launch(T* out, long out_ld, const T* proj, long proj_ld, const T* cache, int block_size, const int* seq_cu, const int* seq_ctx, const int* seq_bt,
            int bt_width, int rows, int heads, int kv_heads, int gate_off, float scale, int window, bool sink, float out_scale, int nparts, int part_keys, float* ws_acc,
            float* ws_ml, int keep, float softcap, const float* sink_w, bool channel_gate, int chunk, const WindowPrep& prep, const DeltaStep& d, hipStream_t s) {
  const WindowLaunch<T, D, true> l(out, out_ld, proj_ld, cache, block_size, 0, rows, heads, kv_heads, gate_off, scale, window, sink, out_scale, nparts, part_keys,
                                   ws_acc, ws_ml, keep, softcap, sink_w, channel_gate, chunk, &prep);
  const long wgs = (long)l.grid.x * l.grid.y * l.grid.z;
  if (wgs > 0xffff || prep.rows > 0xffff) return false;
  const DeltaArgs<T> delta{seq_cu, seq_ctx, d.seq_state, (const T*)d.proj, d.S, (const T*)d.w2, d.heads, d.rank, rows, d.a_b, d.ld,
                           DeltaRuleRest{d.out, d.out_ld, d.w0, d.norm_w, d.eps, d.out_scale}};
  auto go = [&](auto* kernel) {
    kernel<<<wgs + (long)d.heads * rows, std::max(64 * l.waves, kDeltaThreads), std::max(l.smem, (size_t)kDeltaLds), s>>>(
        proj, seq_cu, seq_ctx, seq_bt, prep.positions, prep.slots, bt_width, (unsigned)prep.rows << 16 | (unsigned)wgs, l.rest, delta);
  };
  if (prep.norm_mode == 1) go(&window_delta_step_kernel<T, D, 1>);
  else if (prep.norm_mode == 2) go(&window_delta_step_kernel<T, D, 2>);
  else go(&window_delta_step_kernel<T, D, 0>);
  if (nparts > 1)
    launch_window_decode_reduce(out, out_ld, ws_acc, ws_ml, proj, proj_ld, gate_off, nparts, heads, rows, 0, D, out_scale, channel_gate, sizeof(T) == 4, s);
  return true;
}

}  // namespace

bool launch_window_delta_step(void* out, long out_ld, const void* proj, long proj_ld, const void* cache, int block_size, const int* seq_cu,
                              const int* seq_ctx, const int* seq_bt, int bt_width, int rows, int heads, int kv_heads, int dim, int gate_off, float scale,
                              int window, bool sink, float out_scale, int nparts, int part_keys, float* ws_acc, float* ws_ml, int keep, float softcap,
                              const float* sink_w, bool channel_gate, int chunk, bool f32, const WindowPrep& prep, const DeltaStep& delta, hipStream_t s) {
  if (rows <= 0 || prep.rows <= 0) return true;
#define HS_WDS(T, D)                                                                                                                       \
  return launch<T, D>((T*)out, out_ld, (const T*)proj, proj_ld, (const T*)cache, block_size, seq_cu, seq_ctx, seq_bt, bt_width, rows, heads, kv_heads, gate_off, \
               scale, window, sink, out_scale, nparts, part_keys, ws_acc, ws_ml, keep, softcap, sink_w, channel_gate, chunk, prep, delta, s)
  if (f32) { if (dim == 64) HS_WDS(float, 64); HS_WDS(float, 128); }
  if (dim == 64) HS_WDS(unsigned short, 64);
  HS_WDS(unsigned short, 128);
#undef HS_WDS
}

}  // namespace hipserve

// Window attention of decode rows (a workgroup per row, one map per head; same cache, masks, sink and gates as
// window_attention.hip), bf16 and fp32, heads of 64, 128 (and in bf16 256) dims.
//
// A workgroup owns up to 16 query heads of one key / value head and a run of keys. Its waves take tiles of 32 keys (fp32: 16)
// in turn, each with its own running (max, sum) and accumulators, and meet once, at the end. Nothing is shared between the
// waves, so nothing goes through LDS before that: every operand is loaded as the matrix instruction wants it.
//   scores S^T = K . Q^T: a lane's part of a key row is 16 consecutive bytes of it;
//   output O^T = V^T . P^T: the k slots of the instruction stand for the keys whose weights a lane already holds (4 g + i of
//   each 16), and the instruction's rows for the dims that 16 consecutive bytes of a value row hold, every E-th of a block
//   of 16 E: a lane loads whole 16-byte parts of its keys' rows, and in bf16 two byte permutations per pair of keys and pair
//   of dims put the keys of one dim side by side.
// fp32 prompts take the same kernel with several tokens in the 16 rows and a mask per score: the waves (eight, seven at
// 128 dims) share no tile, but the 32-bit products are slow enough that reading the keys once per 16 rows costs less than they do.
// What bounds it: the chain table -> cache -> scores -> output of one tile, then (many sequences) memory. All loads of a
// tile are issued at once and no wave waits for another's. A workgroup that stages every tile for four waves of which one has
// rows (a group of 4 heads) waits for two barriers and a transposing store per 32 keys: one sequence of 100 keys, 8 heads
// over 2 of 128 dims, in bf16 11.5 us, this 5.8; 16 sequences of 900 keys, 16 heads over 4: 17.4, 13.3 (with the merge); 64
// sequences of 1024 keys, 32 heads over 8: 78.6, 48.4 (5.5 TB/s). In fp32 the kernel of window_attention.hip, one wave per
// head and no split over keys: 16 sequences 528 us, this 19.
#include "window_decode.h"

namespace hipserve {
namespace {

// The parameters before `rest` reach the kernel in scalar registers.
template <typename T, int D, bool MULTI, int MODE = 3>
__global__ __launch_bounds__(512) void window_decode_kernel(
    const T* __restrict__ proj, const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx, const int* __restrict__ seq_bt,
    const long* __restrict__ positions, const long* __restrict__ slots, int bt_width, int T_rows, const WindowRest<T, (MODE < 3)> rest) {
  extern __shared__ float lds[];
  window_decode_block<T, D, MULTI, MODE>(blockIdx.x, blockIdx.y, blockIdx.z, proj, seq_cu, seq_ctx, seq_bt, positions, slots, bt_width, T_rows, rest, lds);
}

// out[row_base + r, head] = sum_p acc_p e^(m_p - M) / sum_p l_p e^(m_p - M) * sigmoid(gate) * out_scale
template <typename T>
__global__ __launch_bounds__(128) void window_decode_reduce_kernel(
    T* __restrict__ out, long out_ld, const float* __restrict__ ws_acc, const float* __restrict__ ws_ml,
    const T* __restrict__ proj, long proj_ld, int gate_off, int nparts, int heads, int ws_rows, int row_base, int vdim,
    float out_scale, bool channel_gate) {
  using S = Softmax<T>;
  __shared__ float sc[kMaxRuns];  // each run's weight e^(m_p - M) / L * gate * scale, 0 for empty runs
  const int r = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const long trow = row_base + r;
  if (tid < 64) {  // one wave: run p on lane p
    const long w = ((long)min(tid, nparts - 1) * heads + h) * ws_rows + r;
    const float m = tid < nparts ? ws_ml[2 * w] : -INFINITY;
    const float l = tid < nparts ? ws_ml[2 * w + 1] : 0.f;
    const float M = wave_max(m);
    const float e = m == -INFINITY ? 0.f : S::exp(m - M);
    const float L = wave_sum(l * e);
    float f = out_scale;
    if (gate_off >= 0 && !channel_gate) f *= sigmoid_f(ldf<T>(proj, trow * proj_ld + gate_off + h));
    sc[tid] = L == 0.f ? 0.f : e * f / L;
  }
  __syncthreads();
  for (int d = tid; d < vdim; d += 128) {
    float o = 0.f;
    for (int p = 0; p < nparts; ++p) o += ws_acc[(((long)p * heads + h) * ws_rows + r) * vdim + d] * sc[p];
    if (channel_gate) o *= sigmoid_f(ldf<T>(proj, trow * proj_ld + gate_off + (long)h * vdim + d));
    stf<T>(out, trow * out_ld + (long)h * vdim + d, o);
  }
}

template <typename T, int D>
void launch(T* out, long out_ld, const T* proj, long proj_ld, const T* cache, int block_size, const int* seq_cu,
            const int* seq_ctx, const int* seq_bt, int bt_width, int seq0, int rows, int row_base, int heads, int kv_heads,
            int gate_off, float scale, int window, bool sink, float out_scale, int nparts, int part_keys, float* ws_acc,
            float* ws_ml, int keep, float softcap, const float* sink_w, bool channel_gate, int chunk, const WindowPrep* prep,
            hipStream_t s) {
#define HS_WL(PREP) \
  WindowLaunch<T, D, PREP>(out, out_ld, proj_ld, cache, block_size, seq0, rows, heads, kv_heads, gate_off, scale, window, sink, out_scale, nparts, part_keys, \
                           ws_acc, ws_ml, keep, softcap, sink_w, channel_gate, chunk, prep)
  auto go = [&](auto* kernel, const auto& l) {
    const WindowPrep none{};
    const WindowPrep& pr = prep != nullptr ? *prep : none;
    kernel<<<l.grid, 64 * l.waves, l.smem, s>>>(proj, seq_cu, seq_ctx, seq_bt, pr.positions, pr.slots, bt_width, pr.rows, l.rest);
  };
  if (prep == nullptr) go(&window_decode_kernel<T, D, false>, HS_WL(false));
  if constexpr (D <= 128) {
    if (prep != nullptr) {
      const auto l = HS_WL(true);
      if (prep->norm_mode == 1) go(&window_decode_kernel<T, D, false, 1>, l);
      else if (prep->norm_mode == 2) go(&window_decode_kernel<T, D, false, 2>, l);
      else go(&window_decode_kernel<T, D, false, 0>, l);
    }
  }
#undef HS_WL
  if (nparts > 1)
    launch_window_decode_reduce(out, out_ld, ws_acc, ws_ml, proj, proj_ld, gate_off, nparts, heads, rows, row_base, D, out_scale, channel_gate,
                                sizeof(T) == 4, s);
}

template <int D>
void launch_prompts(float* out, long out_ld, const float* proj, long proj_ld, const float* cache, int block_size, const int* seq_cu,
                    const int* seq_ctx, const int* seq_bt, int bt_width, int seq0, int seq1, int rows_bound, int heads, int kv_heads,
                    int gate_off, float scale, int window, bool sink, float out_scale, int keep, float softcap, const float* sink_w,
                    bool channel_gate, int chunk, hipStream_t s) {
  const int group = heads / kv_heads, hc = std::min(group, 16), hchunks = (group + hc - 1) / hc, tq = 16 / hc;
  const int wave_floats = 16 * D + 32, nw = std::min(8, (1 << 14) / wave_floats);
  WindowRest<float, false> rest{};
  rest.out = out; rest.out_ld = out_ld; rest.proj_ld = proj_ld; rest.cache = cache; rest.sink_w = sink_w; rest.block_shift = __builtin_ctz(block_size);
  rest.seq0 = seq0; rest.seq1 = seq1; rest.tq = tq; rest.hc = hc; rest.hchunks = hchunks; rest.heads = heads; rest.kv_heads = kv_heads;
  rest.group = group; rest.gate_off = gate_off; rest.window = window; rest.keep = keep; rest.chunk = chunk; rest.scale = scale;
  rest.out_scale = out_scale; rest.softcap = softcap; rest.sink = sink; rest.channel_gate = channel_gate; rest.waves = nw; rest.nparts = 1;
  window_decode_kernel<float, D, true><<<dim3(rows_bound / tq + (seq1 - seq0), kv_heads * hchunks, 1), 64 * nw,
                                         (size_t)nw * wave_floats * sizeof(float), s>>>(proj, seq_cu, seq_ctx, seq_bt, nullptr, nullptr, bt_width, 0, rest);
}

}  // namespace

void launch_window_attention_prompts_f32(float* out, long out_ld, const float* proj, long proj_ld, const float* cache, int block_size,
                                         const int* seq_cu, const int* seq_ctx, const int* seq_bt, int bt_width, int seq0, int seq1,
                                         int rows_bound, int heads, int kv_heads, int dim, int gate_off, float scale, int window,
                                         bool sink, float out_scale, int keep, float softcap, const float* sink_w, bool channel_gate,
                                         int chunk, hipStream_t s) {
  if (seq1 <= seq0 || rows_bound <= 0) return;
  auto go = dim == 64 ? launch_prompts<64> : launch_prompts<128>;
  go(out, out_ld, proj, proj_ld, cache, block_size, seq_cu, seq_ctx, seq_bt, bt_width, seq0, seq1, rows_bound, heads, kv_heads, gate_off,
     scale, window, sink, out_scale, keep, softcap, sink_w, channel_gate, chunk, s);
}

bool window_attention_decode_ok(int dim, int vdim, int block_size, bool f32) {
  return dim == vdim && (dim == 64 || dim == 128 || (dim == 256 && !f32)) && (block_size & (block_size - 1)) == 0;
}

void launch_window_decode_reduce(void* out, long out_ld, const float* ws_acc, const float* ws_ml, const void* proj, long proj_ld, int gate_off, int nparts,
                                 int heads, int rows, int row_base, int vdim, float out_scale, bool channel_gate, bool f32, hipStream_t s) {
  const dim3 grid(rows, heads);
  if (f32)
    window_decode_reduce_kernel<float><<<grid, 128, 0, s>>>((float*)out, out_ld, ws_acc, ws_ml, (const float*)proj, proj_ld, gate_off, nparts, heads, rows,
                                                            row_base, vdim, out_scale, channel_gate);
  else
    window_decode_reduce_kernel<unsigned short><<<grid, 128, 0, s>>>((unsigned short*)out, out_ld, ws_acc, ws_ml, (const unsigned short*)proj, proj_ld,
                                                                     gate_off, nparts, heads, rows, row_base, vdim, out_scale, channel_gate);
}

void launch_window_attention_decode(void* out, long out_ld, const void* proj, long proj_ld, const void* cache, int block_size,
                                    const int* seq_cu, const int* seq_ctx, const int* seq_bt, int bt_width, int seq0, int rows,
                                    int row_base, int heads, int kv_heads, int dim, int gate_off, float scale, int window,
                                    bool sink, float out_scale, int nparts, int part_keys, float* ws_acc, float* ws_ml, int keep,
                                    float softcap, const float* sink_w, bool channel_gate, int chunk, bool f32, const WindowPrep* prep,
                                    hipStream_t s) {
  if (rows <= 0 || (prep != nullptr && prep->rows <= 0)) return;
#define HS_WD(T, D)                                                                                                        \
  launch<T, D>((T*)out, out_ld, (const T*)proj, proj_ld, (const T*)cache, block_size, seq_cu, seq_ctx, seq_bt, bt_width, seq0, \
               rows, row_base, heads, kv_heads, gate_off, scale, window, sink, out_scale, nparts, part_keys, ws_acc, ws_ml,   \
               keep, softcap, sink_w, channel_gate, chunk, prep, s)
  if (f32) { if (dim == 64) HS_WD(float, 64); else HS_WD(float, 128); }
  else if (dim == 64) HS_WD(unsigned short, 64);
  else if (dim == 128) HS_WD(unsigned short, 128);
  else HS_WD(unsigned short, 256);
#undef HS_WD
}

}  // namespace hipserve

// minGRU scan. proj rows = [z | x | g] pre-activations (width each). Per sequence and channel,
//   z = sigmoid(zp + b_z), u = xp + b_x, c = u + 0.5 (u >= 0) or sigmoid(u),
//   S_t = (1 - z_t) S_{t-1} + z_t c_t,   y_t = S_t * silu(g_t),
// all in fp32, from the sequence's state slot (zero when the step starts at position 0) and back
// into it. A workgroup owns 64 channels of one sequence. Its waves hold 16 consecutive rows each: a wave folds its rows into
// (A, B) with S_out = A S_in + B, the waves' pairs are chained through LDS, and the rows are replayed from their true S_in.
// 1 - z and z c stay in registers in between: the arithmetic (three sigmoids per element, 60 instructions in all) and, in 32 bits, the
// bytes bound it. Nothing is computed twice, rows are addressed by buffers whose bounds stand for the last block's missing rows
// and the columns past the width, and the next block's rows are loaded while this one's are folded and replayed. 8192 rows (4 prompts)
// x 4096 in bf16: with 64-bit addresses, a branch per element and loads at the head of the block (110 instructions) 95 us, now 71 (float32 112, 115:
// 4.7 TB/s); 7 prompts, 8100 rows x 8192 223 -> 176 (241 -> 231), 700 rows x 4096 29.7 -> 23.3. Waves that fold and then replay one long
// segment each, reading z and x again: 171 us. Two launches over segments of 64 rows (fold, replay; 4 channels per
// thread) fill the card whatever the sequences are, but compute z and c twice: 188. z and x loaded in turns: 74.
//
// Decode steps (mingru_step): one row per sequence needs no folding; 4 channels per thread, 9.1 -> 5.0 us for 41 sequences. Up to 64 of
// them run in the epilogue of the product that makes z, x and g (mingru_product): a workgroup has all three of its 16 channels,
// unrounded, and the states arrive beside its weights. Width 4096, K 2048, in a captured step: one row 11.6 + 4.4
// -> 12.0 us, 48 rows 16.0 + 4.7 -> 15.4. The copies need no arguments that have to be loaded, and the rows' sequences come through the scalar unit:
// 1, 16, 48, 64 rows 12.4 -> 11.5, 12.5 -> 11.8, 15.4 -> 14.6, 16.8 -> 15.7 (in a loop), width 2048, K 1024 5.0 -> 4.4, 5.2 -> 4.5, 7.4 -> 6.8, 8.3 -> 7.5.
#include "expert_rows.h"

#include <type_traits>

namespace hipserve {
namespace {

constexpr int kMaxWaves = 16, kRows = 16;   // waves of a workgroup; rows that a wave holds at a time

struct Gru {
  float keep, zc;   // S <- keep S + zc, keep = 1 - z
  HS_DEVICE Gru() {}
  HS_DEVICE Gru(float zp, float xp, float bz, float bx) {
    const float z = sigmoid_f(zp + bz);
    keep = 1.f - z;
    const float u = xp + bx;
    float e;
    const float r = sigmoid_of_abs(u, e);
    zc = z * (u >= 0.f ? u + 0.5f : e * r);
  }
};

// A number of a row as it is in memory, a register each: packed in pairs, they would be waited for where they are loaded.
template <typename T>
HS_DEVICE unsigned ld_raw(__amdgpu_buffer_rsrc_t from, unsigned at) {
  if constexpr (sizeof(T) == 4) return __builtin_amdgcn_raw_buffer_load_b32(from, at, 0, 0);
  else return __builtin_amdgcn_raw_buffer_load_b16(from, at, 0, 0);
}
template <typename T>
HS_DEVICE float of_raw(unsigned x) { return __builtin_bit_cast(float, sizeof(T) == 4 ? x : x << 16); }

// MANY: more than one block of nw * kRows rows. A block alone has no next one whose loads would go out for nothing, and needs half of the registers: with them all,
// many short sequences in 32 bits waited for each other (400 of 20 rows x 8192 282 us, without 225; 300 of 16 166 and 138).
template <typename T, bool MANY>
__global__ __launch_bounds__(64 * kMaxWaves) void mingru_scan_kernel(
    T* __restrict__ y, float* __restrict__ state, const T* __restrict__ proj, const float* __restrict__ b_z,
    const float* __restrict__ b_x, const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx,
    const int* __restrict__ seq_state, int width) {
  __shared__ float2 fold[2][kMaxWaves][64];
  const int s = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
  const int c = blockIdx.y * 64 + lane;
  const int r0 = seq_cu[s], n = seq_cu[s + 1] - r0;
  if (n <= 0) return;
  const bool live = c < width;
  const int cc = live ? c : 0;
  const float bz = b_z[cc], bx = b_x[cc];
  const long ld = 3L * width, slot = (long)seq_state[s] * width + cc;
  const unsigned at0 = live ? c * sizeof(T) : 0x80000000u;   // outside every row
  // every wave reads the carried state before the first barrier; the slot is rewritten only after the last, by the wave that
  // replays the last row (the chained pairs round once more: 5.3e-8 from 64 bits instead of 5.0e-8 after 2048 rows)
  float last = 0.f;
  bool holds = false;
  float S = (seq_ctx[s] - n > 0) ? state[slot] : 0.f;
  // The wave's rows of the next block are loaded while this one is replayed; rows that do not exist are outside the buffers.
  auto rows_of = [&](int b0) { return min(kRows, n - b0 - wave * kRows); };
  unsigned zp[kRows], xp[kRows], gp[kRows];
  auto load = [&](unsigned* to, int b0, int which) {
    const int rows = rows_of(b0);
    const auto from = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(proj) + (long)(r0 + b0 + wave * kRows) * ld + (long)which * width, 0,
                                                        rows > 0 ? ((rows - 1) * 3 + 1) * width * (int)sizeof(T) : 0, 0x00020000);
    unsigned at = at0;
#pragma unroll
    for (int i = 0; i < kRows; ++i, at += 3 * width * sizeof(T)) to[i] = ld_raw<T>(from, at);
  };
  load(zp, 0, 0);
  load(xp, 0, 1);
  load(gp, 0, 2);
#pragma nounroll
  for (int b0 = 0, buf = 0; b0 < n; b0 += nw * kRows, buf ^= 1) {
    const int rows = rows_of(b0);   // of this wave; none or fewer in the last block
    Gru g[kRows];
    float A = 1.f, B = 0.f;
    if (rows > 0) {
#pragma unroll
      for (int i = 0; i < kRows; ++i) g[i] = Gru(of_raw<T>(zp[i]), of_raw<T>(xp[i]), bz, bx);
      if (rows < kRows) {
        asm volatile("");   // a branch, not selects
#pragma unroll
        for (int i = 0; i < kRows; ++i)
          if (i >= rows) { g[i].keep = 1.f; g[i].zc = 0.f; }
      }
#pragma unroll
      for (int i = 0; i < kRows; ++i) {
        A *= g[i].keep;
        B = g[i].keep * B + g[i].zc;
      }
    }
    if constexpr (MANY) {
      load(zp, b0 + nw * kRows, 0);
      load(xp, b0 + nw * kRows, 1);
    }
    fold[buf][wave][lane] = float2{A, B};
    __syncthreads();
    float mine = S;
#pragma unroll 4
    for (int k = 0; k < nw; ++k) {
      if (k == wave) mine = S;
      const float2 f = fold[buf][k][lane];
      S = f.x * S + f.y;
    }
    if (rows > 0) {
      const auto to = __builtin_amdgcn_make_buffer_rsrc(y + (long)(r0 + b0 + wave * kRows) * width, 0, rows * width * (int)sizeof(T), 0x00020000);
      unsigned at = at0;
#pragma unroll
      for (int i = 0; i < kRows; ++i, at += width * sizeof(T)) {
        mine = g[i].keep * mine + g[i].zc;
        const float gate = of_raw<T>(gp[i]), out = mine * (gate * sigmoid_f(gate));
        if constexpr (sizeof(T) == 4) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, out), to, at, 0, 0);
        else __builtin_amdgcn_raw_buffer_store_b16(f32_to_bf16(out), to, at, 0, 0);
      }
      if (b0 + wave * kRows + rows == n) { last = mine; holds = true; }
    }
    if constexpr (!MANY) break;
    load(gp, b0 + nw * kRows, 2);
  }
  if (live && holds) state[slot] = last;
}

constexpr int kV = 4, kCh = 256 * kV;   // decode steps: channels per thread and per workgroup

template <typename T>
__global__ __launch_bounds__(256) void mingru_step_kernel(T* __restrict__ y, float* __restrict__ state,
                                                          const T* __restrict__ proj, const float* __restrict__ b_z,
                                                          const float* __restrict__ b_x, const int* __restrict__ seq_cu,
                                                          const int* __restrict__ seq_ctx, const int* __restrict__ seq_state,
                                                          int width) {
  const int s = blockIdx.x, c = (blockIdx.y * 256 + threadIdx.x) * kV;
  if (c >= width) return;
  const long row = seq_cu[s];
  if (seq_cu[s + 1] <= row) return;
  float* st = state + (long)seq_state[s] * width + c;
  const T* p = proj + row * 3 * width + c;
  float zp[kV], xp[kV], gp[kV], bz[kV], bx[kV], S[kV] = {}, o[kV];
  Row<T, kV>::ld(p, zp);
  Row<T, kV>::ld(p + width, xp);
  Row<T, kV>::ld(p + 2 * width, gp);
  Row<float, kV>::ld(b_z + c, bz);
  Row<float, kV>::ld(b_x + c, bx);
  if (seq_ctx[s] > 1) Row<float, kV>::ld(st, S);
#pragma unroll
  for (int v = 0; v < kV; ++v) {
    const Gru g(zp[v], xp[v], bz[v], bx[v]);
    S[v] = g.keep * S[v] + g.zc;
    o[v] = S[v] * (gp[v] * sigmoid_f(gp[v]));
  }
  Row<T, kV>::st(y + row * width + c, o);
  Row<float, kV>::st(st, S);
}

struct MinGruSeqs { const int *cu = nullptr, *ctx = nullptr, *state = nullptr; };
struct MinGruRest {
  void* y;
  float* state;
  const float *b_z, *b_x;
  int nseq;
  MinGruSeqs seqs;   // where the kernel has no parameters of them
};
struct MinGruArgs {
  const void *x, *w, *seq_cu, *seq_ctx, *seq_state;
  int x_ld, M, width, K;
  MinGruRest rest;
};

// y, state of the rows x [M, K], one per sequence, and w = [z rows; x rows; g rows]. F32: x, w, x_ld and K in 16-bit halves (skinny.h).
// A MinGruRest lies at byte rest_at of the kernel's arguments.
// HALF: 8 channels per workgroup (mingru_half): the z and x rows are the halves of one tile, the g rows half of another, and a channel's x meets its z from 8
// lanes further. Twice the workgroups, eight rows of weights per load and tile, and two pieces ahead beside the experts, too; the sums are the same. us, cold
// weights, 16 channels -> 8: one row, 2048 x 2048 8.2 -> 7.5, 4096 x 2048 12.0 -> 10.9, with the experts of a row beside 13.2 -> 12.4, 6144 x 2048 18.3 ->
// 15.8, 8192 x 4096 38.8 -> 37.3, with experts 44.5 -> 41.7; 16 rows, 2048 x 2048 9.5 -> 8.6.
template <int XG, int DEPTH, bool F32, bool HALF, bool LATE>
HS_DEVICE void mingru_block(int wg, const unsigned short* __restrict__ x, const unsigned short* __restrict__ w, const MinGruSeqs& seqs, int x_ld, int M,
                            int width, int K, int rest_at, unsigned char* smem) {
  using SK = std::conditional_t<HALF, Skinny<XG, 2, DEPTH, F32, true>, Skinny<XG, 3, DEPTH, F32>>;
  using T = std::conditional_t<F32, float, unsigned short>;
  constexpr int ST = SK::ST, IT = (ST + 1) / 2, NT = HALF ? 2 : 3, kChannels = HALF ? 8 : 16;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = wg * kChannels, c = min(n0 + (tid & (kChannels - 1)), width - 1);
  const unsigned char* wt[NT];
  unsigned w_row[SK::WG], x_row[XG];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    wt[nt] = reinterpret_cast<const unsigned char*>(w + ((long)(HALF ? 2 * nt : nt) * width + n0) * K);
#pragma unroll
    for (int h = 0; h < (HALF && nt == 1 ? 1 : 2); ++h)
      w_row[2 * nt + h] = (unsigned)(HALF ? h * width + min(lane >> 3, width - 1 - n0) : min(8 * h + (lane >> 3), width - 1 - n0)) * (unsigned)K * 2;
  }
#pragma unroll
  for (int j = 0; j < XG; ++j) x_row[j] = (unsigned)min(8 * j + (lane >> 3), M - 1) * (unsigned)x_ld * 2;
  f32x4 acc[NT][ST];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int st = 0; st < ST; ++st) acc[nt][st] = f32x4{0.f, 0.f, 0.f, 0.f};
  T* y = nullptr;
  float* state = nullptr;
  float bz, bx, S[IT];
  long at[IT];   // the channel's place in the row's state, -1: the row has no sequence
  bool fresh[IT];
  SK::accumulate(acc, wt, w_row, reinterpret_cast<const unsigned char*>(x), x_row, K, smem, lane, wave, [&] {
    const auto rest = late_args<MinGruRest>(rest_at);
    const int nseq = rest->nseq;
    // Nothing writes these while the kernel runs, and as constants they are read by the scalar unit, whichever way the pointers come; as loads behind the copies'
    // inline assembly they would be the vector unit's, which wait for the copies.
    using Numbers = const __attribute__((address_space(4))) int*;
    auto numbers = [](const int* p) { return (Numbers)(unsigned long)p; };
    const Numbers seq_cu = numbers(LATE ? rest->seqs.cu : seqs.cu), seq_ctx = numbers(LATE ? rest->seqs.ctx : seqs.ctx),
                  seq_state = numbers(LATE ? rest->seqs.state : seqs.state);
    y = static_cast<T*>(rest->y);
    state = rest->state;
    bz = rest->b_z[c];
    bx = rest->b_x[c];
    // A wave's four rows' sequences
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      int slot = -1, ctx = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int m = 4 * wave + 32 * i + k;
        if (m >= M) continue;
        int s = min(m, nseq - 1), ctx_k = seq_ctx[s], slot_k = seq_state[s];
        const int first = seq_cu[s], end = seq_cu[s + 1];
        if ((first ^ m) | (end ^ (m + 1))) {   // sequences without a row lie between
          for (s = 0; s < nseq && !(seq_cu[s] <= m && m < seq_cu[s + 1]);) ++s;
          ctx_k = s < nseq ? seq_ctx[s] : 0;
          slot_k = s < nseq ? seq_state[s] : -1;
        }
        if (lane >> 4 == k) { slot = slot_k; ctx = ctx_k; }
      }
      at[i] = slot < 0 ? -1 : (long)slot * width + c;
      fresh[i] = ctx <= 1;
      S[i] = state[at[i] < 0 ? c : at[i]];
    }
  });
  float v[NT][IT];
  SK::reduce(v, acc, smem);
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int m = (tid + kSkThreads * i) >> 4;
    const float xv = HALF ? __shfl_xor(v[0][i], 8, 64) : v[1][i], gv = v[NT - 1][i];
    if (m >= M || n0 + (tid & 15) >= width || at[i] < 0 || (HALF && (tid & 8))) continue;
    const Gru g(v[0][i], xv, bz, bx);
    const float o = fmaf(g.keep, fresh[i] ? 0.f : S[i], g.zc);   // as the scan has it, in both kernels
    stf<T>(y, (long)m * width + c, o * (gv * sigmoid_f(gv)));
    state[at[i]] = o;
  }
}

template <int XG, int DEPTH, bool F32, bool HALF>
__global__ __launch_bounds__(kSkThreads) void mingru_product_kernel(
    const unsigned short* __restrict__ x, const unsigned short* __restrict__ w, const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx,
    const int* __restrict__ seq_state, int x_ld, int M, int width, int K, const MinGruRest) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  mingru_block<XG, DEPTH, F32, HALF, false>(blockIdx.x, x, w, MinGruSeqs{seq_cu, seq_ctx, seq_state}, x_ld, M, width, K, offsetof(MinGruArgs, rest), smem);
}

struct MinGruBesideArgs {
  const void *x, *w, *slots, *tile_expert;
  int x_ld, M, width, K, split;
  MinGruRest rest;
  ExpertBeside experts;
};

// The same with the experts' product of tiles with few rows besides (expert_beside.hip): workgroups from `split` on. With 16 channels one piece ahead, so that
// two workgroups fit a compute unit.
template <int XG, int DEPTH, bool HALF>
__global__ __launch_bounds__(kSkThreads) void mingru_product_experts_kernel(
    const unsigned short* __restrict__ x, const unsigned short* __restrict__ w, const int* __restrict__ slots, const int* __restrict__ tile_expert,
    int x_ld, int M, int width, int K, int split, const MinGruRest, const ExpertBeside) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int b = blockIdx.x;
  if (b >= split) expert_beside(b - split, slots, tile_expert, offsetof(MinGruBesideArgs, experts), smem);
  else mingru_block<XG, DEPTH, false, HALF, true>(b, x, w, MinGruSeqs{}, x_ld, M, width, K, offsetof(MinGruBesideArgs, rest), smem);
}

template <int XG, int DEPTH, bool HALF, bool F32>
bool launch_product(void* y, float* state, const void* x, long x_ld, const void* w, const float* b_z, const float* b_x, const int* seq_cu,
                    const int* seq_ctx, const int* seq_state, int nseq, int M, int width, int K, hipStream_t s) {
  constexpr int lds = HALF ? Skinny<XG, 2, DEPTH, F32, true>::kLds : Skinny<XG, 3, DEPTH>::kLds, per = HALF ? 8 : 16;
  static const bool ok = allow_lds(&mingru_product_kernel<XG, DEPTH, F32, HALF>, lds);
  if (!ok) return false;
  mingru_product_kernel<XG, DEPTH, F32, HALF><<<(width + per - 1) / per, kSkThreads, lds, s>>>(
      (const unsigned short*)x, (const unsigned short*)w, seq_cu, seq_ctx, seq_state, (int)x_ld, M, width, K, MinGruRest{y, state, b_z, b_x, nseq, {}});
  return true;
}

template <int XG, int DEPTH, bool HALF>
bool launch_beside(void* y, float* state, const void* x, long x_ld, const void* w, const float* b_z, const float* b_x, const int* seq_cu,
                   const int* seq_ctx, const int* seq_state, int nseq, int M, int width, int K, const ExpertRows& ex, hipStream_t s) {
  constexpr int own = HALF ? Skinny<XG, 2, DEPTH, false, true>::kLds : Skinny<XG, 3, DEPTH>::kLds, lds = own > expert_lds<1>() ? own : expert_lds<1>();
  constexpr int per = HALF ? 8 : 16;
  static const bool ok = allow_lds(&mingru_product_experts_kernel<XG, DEPTH, HALF>, lds);
  if (!ok) return false;
  const int split = (width + per - 1) / per;
  const ExpertBeside experts = expert_beside_args(ex);
  // Two workgroups fit a compute unit and not three: thousands of experts' workgroups of a short k lose more than the launch (two_per_unit_pay, expert_beside.hip), the
  // sooner the shorter minGRU's own are. us apart -> in one, experts of 4096 x 1024: 16 of them, 16 rows, width 2048, k 1024 27.7 -> 29.9, 32 rows, 4096, k 2048 39.2 ->
  // 41.0; 8 of them, 9 rows, 2048, k 1024 19.0 -> 19.8. Of 832 sizes of 1 - 32 rows three that go together take 1.1 - 1.4 % longer than apart, and all 12 % less on average.
  if (ex.K < 2048 && (long)experts.per_tile * ex.ntiles > (HALF ? 2200 : 4000)) return false;
  mingru_product_experts_kernel<XG, DEPTH, HALF><<<split + experts.per_tile * ex.ntiles, kSkThreads, lds, s>>>(
      (const unsigned short*)x, (const unsigned short*)w, ex.slots, ex.tile_expert, (int)x_ld, M, width, K, split,
      MinGruRest{y, state, b_z, b_x, nseq, {seq_cu, seq_ctx, seq_state}}, experts);
  return true;
}

// Steps of one row per sequence: widths that are multiples of 4, everything at multiples of 16 bytes.
template <typename T>
void launch(T* y, float* state, const T* proj, const float* b_z, const float* b_x, const int* seq_cu, const int* seq_ctx,
            const int* seq_state, int nseq, int width, int max_q, hipStream_t s) {
  uintptr_t at = 0;
  for (const void* p : {(const void*)y, (const void*)state, (const void*)proj, (const void*)b_z, (const void*)b_x})
    at |= reinterpret_cast<uintptr_t>(p);
  if (max_q == 1 && width % kV == 0 && at % 16 == 0) {
    mingru_step_kernel<T><<<dim3(nseq, (width + kCh - 1) / kCh), 256, 0, s>>>(y, state, proj, b_z, b_x, seq_cu, seq_ctx, seq_state, width);
    return;
  }
  const int nw = min(kMaxWaves, (max_q + kRows - 1) / kRows);
  auto kernel = max_q <= nw * kRows ? &mingru_scan_kernel<T, false> : &mingru_scan_kernel<T, true>;
  kernel<<<dim3(nseq, (width + 63) / 64), 64 * nw, 0, s>>>(y, state, proj, b_z, b_x, seq_cu, seq_ctx, seq_state, width);
}

}  // namespace

// Whether workgroups take 8 channels (mingru_block): where 16 leave half of the compute units idle, and, for up to 4 rows, where either has the units full and k
// is long; not between the two, where 16 are one round and 8 nearly two (3000 x 2048, one row 9.7 -> 9.9 us), nor for more rows, which are read twice as often
// then (8192 x 4096, 16 rows 39.2 -> 42.2; with experts beside 4096 x 2048, 8 rows 20.3 -> 21.3). Offsets within a workgroup's rows have 32 bits.
static bool mingru_half(int M, int width, int K) {
  if (M > 16 || 4L * (width + 8) * K >= (1L << 32)) return false;
  return width <= 2048 ? width > 1024 && K >= 1024 : M <= 4 && width >= 4096 && K >= 2048;
}

bool launch_mingru_product(void* y, float* state, const void* x, long x_ld, const void* w, const float* b_z, const float* b_x,
                           const int* seq_cu, const int* seq_ctx, const int* seq_state, int nseq, int M, int width, int K, bool f32,
                           hipStream_t s) {
  if (M <= 0 || nseq <= 0 || width <= 0) return true;
  if (f32) { x_ld *= 2; K *= 2; }   // in halves
#define HS_MH(XG, DEPTH, HALF, F32) launch_product<XG, DEPTH, HALF, F32>(y, state, x, x_ld, w, b_z, b_x, seq_cu, seq_ctx, seq_state, nseq, M, width, K, s)
#define HS_MG(XG, DEPTH) (f32 ? HS_MH(XG, DEPTH, false, true) : HS_MH(XG, DEPTH, false, false))
  if (!f32 && mingru_half(M, width, K)) return M <= 8 ? HS_MH(1, 2, true, false) : HS_MH(2, 2, true, false);
  return M <= 8 ? HS_MG(1, 2) : M <= 16 ? HS_MG(2, 2) : M <= 32 ? HS_MG(4, 1) : M <= 48 ? HS_MG(6, 1) : HS_MG(8, 1);
#undef HS_MG
#undef HS_MH
}

bool launch_mingru_product_experts(void* y, float* state, const void* x, long x_ld, const void* w, const float* b_z, const float* b_x,
                                   const int* seq_cu, const int* seq_ctx, const int* seq_state, int nseq, int M, int width, int K,
                                   const ExpertRows& ex, hipStream_t s) {
  if (M <= 0 || nseq <= 0 || width <= 0 || M > 32 || !expert_rows_ok(ex)) return false;   // more rows: 96 KB, the experts would have a compute unit's LDS to themselves each
#define HS_MG(XG, DEPTH, HALF) launch_beside<XG, DEPTH, HALF>(y, state, x, x_ld, w, b_z, b_x, seq_cu, seq_ctx, seq_state, nseq, M, width, K, ex, s)
  if (mingru_half(M, width, K)) return M <= 8 ? HS_MG(1, 2, true) : HS_MG(2, 2, true);
  return M <= 8 ? HS_MG(1, 1, false) : M <= 16 ? HS_MG(2, 1, false) : HS_MG(4, 1, false);
#undef HS_MG
}

void launch_mingru_scan(void* y, float* state, const void* proj, const float* b_z, const float* b_x,
                        const int* seq_cu, const int* seq_ctx, const int* seq_state, int nseq, int width, int max_q,
                        bool f32, hipStream_t s) {
  if (nseq <= 0 || max_q <= 0) return;
  if (f32)
    launch((float*)y, state, (const float*)proj, b_z, b_x, seq_cu, seq_ctx, seq_state, nseq, width, max_q, s);
  else
    launch((unsigned short*)y, state, (const unsigned short*)proj, b_z, b_x, seq_cu, seq_ctx, seq_state, nseq, width, max_q, s);
}

}  // namespace hipserve

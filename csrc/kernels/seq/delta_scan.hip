// Delta-rule recurrences over per-sequence state slots, fp32 state [slots, heads, key dim, value dim].
//
// gated delta rule (per head, one decay g and one write strength beta per token):
//   S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q
// the same with a decay g per key channel (the rows of S), from a bottleneck
// generalized delta rule (per head, decay w and removal rate a per key channel, unit key u):
//   S <- diag(w) S - (a * u)(u^T S) + k v^T  (both terms read the old S);  o = S^T r
//
// linear attention with a decay per key channel (per head, bonus u for the current token):
//   o = (S + diag(u) k v^T)^T r;  S <- diag(w) S + k v^T
//
// All scans keep a COLUMN of the state (all key channels of one value channel) in the registers
// of the 16 lanes of a DPP row, dim / 16 key channels each, so a product with the state is a few
// multiply-adds per lane and a four-step DPP sum; the per-token vectors shared by all columns (k, q / w, a u,
// u, k, r) are staged through LDS a few tokens at a time. A step that starts at position 0 starts from a zero state.
//
// The prepare kernels compute what enters the recurrences in fp32: the short causal convolution
// (+ SiLU) from the step's rows and the sequence's last taps - 1 inputs, unit vectors, sigmoid /
// softplus / exp of the decays and rates. head_norm_gate finishes both: per-head RMS norm of the
// read-out, weight, SiLU or sigmoid gate, optional scale.
//
// Long prompt portions of the gated rule run in chunks on the matrix cores instead (delta_chunk.hip).
//
// Steps in which every sequence brings one row run the whole gated rule of a (sequence, head) in one workgroup
// (gated_delta_step).
#include "conv_update.h"
#include "seq_common.h"
#include "hipserve/seq_kernels.h"

namespace hipserve {
namespace {

HS_DEVICE float softplus_f(float x) { return x > 20.f ? x : log1pf(expf(x)); }

HS_DEVICE int find_seq(const int* __restrict__ seq_cu, int nseq, int row) {
  for (int s = 0; s < nseq; ++s)
    if (row < seq_cu[s + 1]) return row >= seq_cu[s] ? s : -1;
  return -1;
}

// What enters the gated rule, as fp32 rows. One wave per item and `run` rows (prep_run); the items of a row are
//   the query heads: unit(silu(conv q)) dim^-1/2,  the key heads: unit(silu(conv k))      -> qk[t] = [q | k]
//   the value channels in parts of 256: silu(conv v)                                       -> vv[t]
//   the heads' decays: exp(-exp(a_log) softplus(. + dt_bias)), one per head or (CH) per head and key channel
//   (dec [T, heads * dim])                                                                 -> gg[t]
//   beta: sigmoid                                                                          -> bb[t]
// Lane l owns channels l, l + 64, ... of its item and keeps their last TAPS - 1 inputs in registers while it walks
// the rows (TAPS 0: any number of taps, inputs read again per row).
constexpr int kPrepCh = 4;   // kPrepCh * 64: most channels of an item

// Rows that a wave of gated_delta_prepare walks, one after the other: 16, or, of steps that leave the card room, 2 - 8: a row takes
// about 1 us, the TAPS - 1 rows read again cost bytes. The whole rule in us with 2 / 4 / 8 / 16 rows (workgroups with 16): 33 rows of 8 heads of 128 (9)
// 24.8 / 26.5 / 29.9 / 36.8; 3 prompts of 300 (171) 46.7 / 47.7 / 52.4 / 62.8; 16 of 200 (600) 96 / 91 / 94 / 103; 4 of 2048 (1536) 217 / 204 / 200 /
// 212; of 16 heads (2560) 407 / 383 / 368 / 368.
int prep_run(int T, int groups) {
  int run = 2;
  while (run < 16 && (long)((T + run - 1) / run) * groups > 3600) run *= 2;
  return run;
}

template <typename T, int TAPS, bool CH>
__global__ __launch_bounds__(256) void gated_delta_prepare_kernel(
    float* __restrict__ qk, float* __restrict__ vv, float* __restrict__ gg, float* __restrict__ bb,
    const T* __restrict__ proj, long ld, const float* __restrict__ dec, const float* __restrict__ conv_state,
    const float* __restrict__ conv_w, const float* __restrict__ a_log, const float* __restrict__ dt_bias,
    const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx, const int* __restrict__ seq_state, int nseq, int T_,
    int heads, int kv_heads, int dim, int vdim, int taps_, int off_a, int off_b, int run) {
  const int lane = threadIdx.x & 63;
  const int nqk = kv_heads * dim, nv = heads * vdim, C = 2 * nqk + nv;
  const int vparts = (nv + 64 * kPrepCh - 1) / (64 * kPrepCh), dparts = CH ? heads : 1;
  int item = blockIdx.y * 4 + (threadIdx.x >> 6);
  const int t0 = blockIdx.x * run, t1 = min(t0 + run, T_);
  if (item >= 2 * kv_heads + vparts) {
    item -= 2 * kv_heads + vparts;
    if (item < dparts) {
      if constexpr (CH) {
        const float ea = expf(a_log[item]);
        for (int t = t0; t < t1; ++t)
          for (int e = lane; e < dim; e += 64) {
            const long i = (long)item * dim + e;
            gg[(long)t * heads * dim + i] = expf(-ea * softplus_f(dec[(long)t * heads * dim + i] + dt_bias[i]));
          }
      } else {
        for (int t = t0; t < t1; ++t)
          for (int h = lane; h < heads; h += 64)
            gg[(long)t * heads + h] = expf(-expf(a_log[h]) * softplus_f(ldf<T>(proj, (long)t * ld + off_a + h) + dt_bias[h]));
      }
    } else if (item == dparts) {
      for (int t = t0; t < t1; ++t)
        for (int h = lane; h < heads; h += 64) bb[(long)t * heads + h] = sigmoid_f(ldf<T>(proj, (long)t * ld + off_b + h));
    }
    return;
  }
  const bool value = item >= 2 * kv_heads;
  const int c0 = value ? 2 * nqk + (item - 2 * kv_heads) * 64 * kPrepCh : item * dim;   // the item's first channel
  const int nc = value ? min(64 * kPrepCh, C - c0) : dim;
  const int taps = TAPS > 0 ? TAPS : taps_, hist = taps - 1;
  constexpr int kW = TAPS > 0 ? TAPS : 1, kX = TAPS > 1 ? TAPS - 1 : 1;
  float w[kPrepCh][kW], x[kPrepCh][kX];
  if constexpr (TAPS > 0) {
#pragma unroll
    for (int i = 0; i < kPrepCh; ++i)
#pragma unroll
      for (int j = 0; j < TAPS; ++j) w[i][j] = lane + 64 * i < nc ? conv_w[(long)(c0 + lane + 64 * i) * TAPS + j] : 0.f;
  }
  int s = find_seq(seq_cu, nseq, t0), r0 = 0, end = 0;
  const float* cs = nullptr;
  bool carried = false, fresh = true;
  if (s < 0) return;
  end = seq_cu[s + 1];
  float nxt[kPrepCh];   // the next row's inputs, loaded a row ahead
#pragma unroll
  for (int i = 0; i < kPrepCh; ++i) nxt[i] = lane + 64 * i < nc ? ldf<T>(proj, (long)t0 * ld + c0 + lane + 64 * i) : 0.f;
  for (int t = t0; t < t1; ++t) {
    float row[kPrepCh];
#pragma unroll
    for (int i = 0; i < kPrepCh; ++i) {
      row[i] = nxt[i];
      if (t + 1 < t1 && lane + 64 * i < nc) nxt[i] = ldf<T>(proj, (long)(t + 1) * ld + c0 + lane + 64 * i);
    }
    while (t >= end) {   // the next sequence that has rows
      if (++s >= nseq) return;
      end = seq_cu[s + 1];
      fresh = true;
    }
    // the input `back` rows before row t: an earlier row of the step, or one of the sequence's kept inputs, or zero
    auto before = [&](int c, int back) {
      const int r = t - back;
      if (r >= r0) return ldf<T>(proj, (long)r * ld + c);
      return carried ? cs[(long)(hist + r - r0) * C + c] : 0.f;
    };
    if (fresh) {
      r0 = seq_cu[s];
      carried = seq_ctx[s] - (end - r0) > 0;
      cs = conv_state + (long)seq_state[s] * max(hist, 1) * C;
      fresh = false;
      if constexpr (TAPS > 1) {
#pragma unroll
        for (int i = 0; i < kPrepCh; ++i)
#pragma unroll
          for (int j = 0; j < TAPS - 1; ++j) x[i][j] = lane + 64 * i < nc ? before(c0 + lane + 64 * i, TAPS - 1 - j) : 0.f;
      }
    }
    float y[kPrepCh];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < kPrepCh; ++i) {
      y[i] = 0.f;
      if (64 * i >= nc) continue;
      const int c = c0 + lane + 64 * i;
      if (lane + 64 * i < nc) {
        const float cur = row[i];
        float a = 0.f;
        if constexpr (TAPS > 0) {
#pragma unroll
          for (int j = 0; j < TAPS - 1; ++j) a = __builtin_fmaf(w[i][j], x[i][j], a);
          a = __builtin_fmaf(w[i][TAPS - 1], cur, a);
#pragma unroll
          for (int j = 0; j + 1 < TAPS - 1; ++j) x[i][j] = x[i][j + 1];
          if constexpr (TAPS > 1) x[i][TAPS - 2] = cur;
        } else {
          for (int j = 0; j < taps; ++j)
            a = __builtin_fmaf(conv_w[(long)c * taps + j], j == hist ? cur : before(c, hist - j), a);
        }
        y[i] = a * sigmoid_f(a);
        ss = __builtin_fmaf(y[i], y[i], ss);
      }
    }
    float f = 1.f;
    if (!value) {
      f = 1.f / sqrtf(wave_sum(ss) + 1e-6f);
      if (item < kv_heads) f *= 1.f / sqrtf((float)dim);
    }
    float* dst = value ? vv + (long)t * nv + (c0 - 2 * nqk) : qk + (long)t * 2 * nqk + c0;
#pragma unroll
    for (int i = 0; i < kPrepCh; ++i)
      if (lane + 64 * i < nc) dst[lane + 64 * i] = y[i] * f;
  }
}

template <typename T, int HIST>
__global__ __launch_bounds__(256) void conv_state_update_kernel(
    const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx, const int* __restrict__ seq_state, const T* __restrict__ proj,
    float* __restrict__ conv_state, int C, int taps, long ld) {
  conv_update_block<T, HIST>(blockIdx.x, blockIdx.y * 256 + threadIdx.x, seq_cu, seq_ctx, seq_state, proj, conv_state, C, taps, ld);
}

constexpr int kTB = 8;     // tokens staged at a time
constexpr int kSeg = 16;   // lanes that share a state column (one DPP row)
constexpr int kScanThreads = 256;
constexpr int kCols = kScanThreads / kSeg;  // state columns per workgroup, one per lane row (two: half the waves, each twice as long; slower)

HS_DEVICE __amdgpu_buffer_rsrc_t rows_at(const float* p, int bytes) {   // `bytes` of rows, in scalar registers
  const unsigned long at = reinterpret_cast<uintptr_t>(p);
  const unsigned long lo = (unsigned)__builtin_amdgcn_readfirstlane((int)at), hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(at >> 32));
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(hi << 32 | lo), 0, __builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}

constexpr unsigned kNone = 0x80000000u;   // outside every buffer: reads as zero, is not stored

HS_DEVICE float ld_at(__amdgpu_buffer_rsrc_t from, unsigned at) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(from, at, 0, 0)); }

// grid (heads, ceil(vdim / kCols), sequences), four waves: the step's first sequences (its prompt portions, the
// long ones) are dispatched first and spread over the CUs before the one-token sequences fill in. A state column (one value channel) is held by the 16
// lanes of a DPP row, DS key channels each (dim <= 16 DS; the padding rows stay zero): a product with the
// state is DS multiply-adds per lane and four DPP steps, so the chain from one token to the next is short. The instructions that a wave issues
// in turn bound it, so a full batch of tokens tests nothing and what does not exist is outside the buffers instead of behind branches. The whole rule in
// 32 bits, 3 prompts of 300 rows, 8 heads of 128: 124 -> 90 us, one of 700 237 -> 175 (the generalized one, 16 heads of 64: 102 -> 70, 209 -> 132).
// AHEAD: a token's vectors are read while the one before is computed. Its second set of them is 2 - 5 DS registers, so wider rows go without it (and,
// past 8 channels a lane, without the second copy of the tokens): the generalized rule with it 209 and 388 registers at 8 and 16 channels, without 122
// and 168, two and three waves per SIMD more. 200 sequences of 10 rows with / without, us: 16 heads of 128 406 / 334, 8 of 200 995 / 593; this rule with a
// decay per channel, 8 of 200, 793 / 489, 8 of 256 with one 617 / 515. One prompt of 300 of 8 heads of 128 gives 86 / 93 back.
// CH: a decay per key channel, staged beside q and k.
template <int DS, bool CH>
__global__ __launch_bounds__(kScanThreads) void gated_delta_scan_kernel(
    float* __restrict__ o, float* __restrict__ S, const float* __restrict__ qk, const float* __restrict__ vv,
    const float* __restrict__ gg, const float* __restrict__ bb, const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx,
    const int* __restrict__ seq_state, int heads, int kv_heads, int dim, int vdim) {
  constexpr bool AHEAD = DS <= 4;
  constexpr int DP = kSeg * DS;
  __shared__ __attribute__((aligned(16))) float sq[kTB][DP], sk[kTB][DP], sg[CH ? kTB : 1][CH ? DP : 1];
  __shared__ float sb[kTB][2];   // beta, and the head's decay without CH
  const int s = blockIdx.z, h = blockIdx.x, zb = blockIdx.y, tid = threadIdx.x;
  const int r0 = seq_cu[s], n = seq_cu[s + 1] - r0;
  if (n <= 0) return;
  const int seg = tid & (kSeg - 1), k0 = seg * DS;
  const int v0 = zb * kCols + tid / kSeg;   // this lane row's column
  const int kh = h / (heads / kv_heads), nqk = kv_heads * dim, nv = heads * vdim;
  float* Sp = S + (((long)seq_state[s] * heads + h) * dim) * vdim;
  const bool carried = seq_ctx[s] - n > 0;
  const auto kept = rows_at(Sp, carried ? dim * vdim * 4 : 0);
  float st[DS];
#pragma unroll
  for (int i = 0; i < DS; ++i) st[i] = ld_at(kept, v0 < vdim ? ((k0 + i) * vdim + v0) * 4u : kNone);
  // the next batch of tokens is loaded into registers while this batch is computed
  constexpr int kLd = (kTB * DP + kScanThreads - 1) / kScanThreads;
  float rq[kLd], rk[kLd], rg[CH ? kLd : 1], rv[kTB], rb = 0.f;
  const unsigned v_at = v0 < vdim ? (h * vdim + v0) * 4u : kNone, b_at = tid < 2 * kTB ? ((tid >> 1) * heads + h) * 4u : kNone;
  auto fetch = [&](int t0) {
    const int nt = min(kTB, n - t0);
    const long r = r0 + t0;
    const auto fq = rows_at(qk + r * 2 * nqk, nt * 2 * nqk * 4), fk = rows_at(qk + r * 2 * nqk + nqk, (nt * 2 - 1) * nqk * 4), fv = rows_at(vv + r * nv, nt * nv * 4),
               fb = rows_at(bb + r * heads, nt * heads * 4), fg = rows_at(gg + r * heads * (CH ? dim : 1), nt * heads * (CH ? dim : 1) * 4);
#pragma unroll
    for (int it = 0; it < kLd; ++it) {
      const int i = it * kScanThreads + tid;
      const int tt = i / DP, k = i % DP;
      const unsigned at = k < dim ? (tt * 2 * nqk + kh * dim + k) * 4u : kNone;
      rq[it] = ld_at(fq, at);
      rk[it] = ld_at(fk, at);
      if constexpr (CH) rg[it] = ld_at(fg, k < dim ? ((tt * heads + h) * dim + k) * 4u : kNone);
    }
    rb = ld_at(fb, b_at);
    if constexpr (!CH) {
      const float g = ld_at(fg, b_at);
      rb = tid & 1 ? g : rb;
    }
#pragma unroll
    for (int tt = 0; tt < kTB; ++tt) rv[tt] = ld_at(fv, v_at + tt * nv * 4);
  };
  // the read-outs, by the first lane of a row; every other lane's are outside as well
  const unsigned out_at = seg == 0 ? v_at : kNone;
  fetch(0);
  for (int t0 = 0; t0 < n; t0 += kTB) {
    const int nt = min(kTB, n - t0);
    __syncthreads();
#pragma unroll
    for (int it = 0; it < kLd; ++it) {
      const int i = it * kScanThreads + tid;
      if (i < kTB * DP) {
        sq[i / DP][i % DP] = rq[it];
        sk[i / DP][i % DP] = rk[it];
        if constexpr (CH) sg[i / DP][i % DP] = rg[it];
      }
    }
    if (tid < 2 * kTB) sb[tid >> 1][tid & 1] = rb;
    float val[kTB];
#pragma unroll
    for (int tt = 0; tt < kTB; ++tt) val[tt] = rv[tt];
    __syncthreads();
    if (t0 + kTB < n) fetch(t0 + kTB);
    const auto to = rows_at(o + (long)(r0 + t0) * nv, nt * nv * 4);
    struct Token {
      float beta, g, kk[DS], qq[DS], gd[CH ? DS : 1];
    } x[AHEAD ? 2 : 1];
    auto read = [&](Token& x, int tt) {
      x.beta = sb[tt][0];
      x.g = sb[tt][1];
#pragma unroll
      for (int i = 0; i < DS; ++i) {
        x.kk[i] = sk[tt][k0 + i];
        x.qq[i] = sq[tt][k0 + i];
        if constexpr (CH) x.gd[i] = sg[tt][k0 + i];
      }
    };
    auto token = [&](int tt) {
      if (!AHEAD) read(x[0], tt);
      else if (tt + 1 < kTB) read(x[(tt + 1) & 1], tt + 1);
      if (AHEAD) __builtin_amdgcn_sched_barrier(0);   // those loads stay here
      const auto& [beta, g, kk, qq, gd] = x[AHEAD ? tt & 1 : 0];
      float pred = 0.f, pred2 = 0.f;
#pragma unroll
      for (int i = 0; i < DS; ++i) {
        st[i] *= CH ? gd[CH ? i : 0] : g;
        if (i & 1) pred2 = __builtin_fmaf(st[i], kk[i], pred2);
        else pred = __builtin_fmaf(st[i], kk[i], pred);
      }
      const float u = beta * (val[tt] - row_sum(pred + pred2));
      float out = 0.f, out2 = 0.f;
#pragma unroll
      for (int i = 0; i < DS; ++i) {
        st[i] = __builtin_fmaf(kk[i], u, st[i]);
        if (i & 1) out2 = __builtin_fmaf(st[i], qq[i], out2);
        else out = __builtin_fmaf(st[i], qq[i], out);
      }
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, row_sum(out + out2)), to, out_at + tt * nv * 4, 0, 0);
    };
    if (AHEAD) read(x[0], 0);
    if (DS <= 8 && nt == kTB) {   // no tests between the tokens
#pragma unroll
      for (int tt = 0; tt < kTB; ++tt) token(tt);
    } else {
#pragma unroll
      for (int tt = 0; tt < kTB; ++tt)
        if (tt < nt) token(tt);
    }
  }
#pragma unroll
  for (int i = 0; i < DS; ++i)
    if (v0 < vdim && k0 + i < dim) Sp[(long)(k0 + i) * vdim + v0] = st[i];
}

// proj rows = [r | k | v | a | g | ...] (N = heads * dim each), wl = decay pre-activation (fp32 [T, N]).
// pre[t] = [w = exp(-e^-1/2 sigmoid(wl + w0)) | a u | u | k | r | v] with a = sigmoid(a + a_b), u = unit(k) per head.
template <typename T>
__global__ __launch_bounds__(256) void delta_rule_prepare_kernel(
    float* __restrict__ pre, const T* __restrict__ proj, long ld, const float* __restrict__ wl,
    const float* __restrict__ a_b, const float* __restrict__ w0, int heads, int dim) {
  const long t = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int N = heads * dim;
  const T* row = proj + t * ld;
  for (int h = wave; h < heads; h += 4) {
    float a = 0.f;
    for (int e = lane; e < dim; e += 64) { const float v = ldf<T>(row, N + h * dim + e); a += v * v; }
    const float inv = 1.f / sqrtf(wave_sum(a) + 1e-6f);
    for (int e = lane; e < dim; e += 64) {
      const int c = h * dim + e;
      const float u = ldf<T>(row, N + c) * inv;
      pre[t * 6 * N + c] = expf(-0.60653065971263342f * sigmoid_f(wl[t * N + c] + w0[c]));
      pre[t * 6 * N + N + c] = sigmoid_f(ldf<T>(row, 3 * N + c) + a_b[c]) * u;
      pre[t * 6 * N + 2 * N + c] = u;
      pre[t * 6 * N + 3 * N + c] = ldf<T>(row, N + c);       // k, r, v as fp32: the scan reads one buffer
      pre[t * 6 * N + 4 * N + c] = ldf<T>(row, c);
      pre[t * 6 * N + 5 * N + c] = ldf<T>(row, 2 * N + c);
    }
  }
}

// As gated_delta_scan_kernel. Rows past a partial batch are not asked for where a row is wide: they hold up a step of one token each (200 sequences of 8
// heads of 200: 302 us with them, 252 without), and are never read back from LDS.
template <typename T, int DS>
__global__ __launch_bounds__(kScanThreads) void delta_rule_scan_kernel(
    float* __restrict__ o, float* __restrict__ S, const float* __restrict__ pre, const T* __restrict__ proj, long ld,
    const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx, const int* __restrict__ seq_state, int heads,
    int dim) {
  constexpr bool AHEAD = DS <= 4;
  constexpr int DP = kSeg * DS, TB = kTB;
  __shared__ __attribute__((aligned(16))) float sv[TB][5][DP];  // w, a u, u, k, r (zero past dim), all from `pre`
  const int s = blockIdx.z, h = blockIdx.x, zb = blockIdx.y, tid = threadIdx.x;
  const int r0 = seq_cu[s], n = seq_cu[s + 1] - r0;
  if (n <= 0) return;
  const int seg = tid & (kSeg - 1), k0 = seg * DS;
  const int v0 = zb * kCols + tid / kSeg;   // this lane row's column
  const int N = heads * dim;
  float* Sp = S + (((long)seq_state[s] * heads + h) * dim) * dim;
  const bool carried = seq_ctx[s] - n > 0;
  const auto kept = rows_at(Sp, carried ? dim * dim * 4 : 0);
  float st[DS];
#pragma unroll
  for (int i = 0; i < DS; ++i) st[i] = ld_at(kept, v0 < dim ? ((k0 + i) * dim + v0) * 4u : kNone);
  // the next batch of tokens is loaded into registers while this batch is computed
  constexpr int kLd = (TB * DP + kScanThreads - 1) / kScanThreads;
  float rg[5][kLd] = {}, rv[TB] = {};
  const unsigned v_at = v0 < dim ? (h * dim + v0) * 4u : kNone;
  const unsigned k_at = tid % DP < dim ? (tid / DP * 6 * N + h * dim + tid % DP) * 4u : kNone;
  auto fetch = [&](int t0) {
    const int nt = min(TB, n - t0);
    const float* p = pre + (long)(r0 + t0) * 6 * N;
    unsigned at = k_at, v = v_at;
    if (DS > 8) asm volatile("" : "+v"(at), "+v"(v));   // the rows' offsets are added up here, not kept over the batches
    auto rows = [&](auto full) {
#pragma unroll
      for (int j = 0; j < 5; ++j) {
        const auto from = rows_at(p + j * N, (nt * 6 - j) * N * 4);
#pragma unroll
        for (int it = 0; it < kLd; ++it)
          if (full || it * kScanThreads < nt * DP) rg[j][it] = ld_at(from, at + it * (kScanThreads / DP) * 6 * N * 4);
      }
      const auto fv = rows_at(p + 5 * N, (nt * 6 - 5) * N * 4);
#pragma unroll
      for (int tt = 0; tt < TB; ++tt)
        if (full || tt < nt) rv[tt] = ld_at(fv, v + tt * 6 * N * 4);
    };
    if (AHEAD || nt == TB) rows(std::true_type{});
    else rows(std::false_type{});
  };
  fetch(0);
  for (int t0 = 0; t0 < n; t0 += TB) {
    const int nt = min(TB, n - t0);
    __syncthreads();
#pragma unroll
    for (int it = 0; it < kLd; ++it) {
      const int i = it * kScanThreads + tid;
      if (i < TB * DP) {
#pragma unroll
        for (int j = 0; j < 5; ++j) sv[i / DP][j][i % DP] = rg[j][it];
      }
    }
    float val[TB];
#pragma unroll
    for (int tt = 0; tt < TB; ++tt) val[tt] = rv[tt];
    __syncthreads();
    if (t0 + TB < n) fetch(t0 + TB);
    const auto to = rows_at(o + (long)(r0 + t0) * N, nt * N * 4);
    unsigned out_at = seg == 0 ? v_at : kNone;
    if (DS > 8) asm volatile("" : "+v"(out_at));
    struct Token {
      float w[DS], au[DS], uu[DS], kk[DS], rr[DS];
    } x[AHEAD ? 2 : 1];
    auto read = [&](Token& x, int tt) {
#pragma unroll
      for (int i = 0; i < DS; ++i) {
        x.w[i] = sv[tt][0][k0 + i]; x.au[i] = sv[tt][1][k0 + i]; x.uu[i] = sv[tt][2][k0 + i];
        x.kk[i] = sv[tt][3][k0 + i]; x.rr[i] = sv[tt][4][k0 + i];
      }
    };
    auto token = [&](int tt) {
      if (!AHEAD) read(x[0], tt);
      else if (tt + 1 < TB) read(x[(tt + 1) & 1], tt + 1);
      if (AHEAD) __builtin_amdgcn_sched_barrier(0);
      const auto& [w, au, uu, kk, rr] = x[AHEAD ? tt & 1 : 0];
      float us = 0.f, us2 = 0.f;
#pragma unroll
      for (int i = 0; i < DS; ++i) {
        if (i & 1) us2 = __builtin_fmaf(uu[i], st[i], us2);
        else us = __builtin_fmaf(uu[i], st[i], us);
      }
      us = row_sum(us + us2);
      float out = 0.f, out2 = 0.f;
#pragma unroll
      for (int i = 0; i < DS; ++i) {
        st[i] = w[i] * st[i] - au[i] * us + kk[i] * val[tt];
        if (i & 1) out2 = __builtin_fmaf(st[i], rr[i], out2);
        else out = __builtin_fmaf(st[i], rr[i], out);
      }
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, row_sum(out + out2)), to, out_at + tt * N * 4, 0, 0);
    };
    if (AHEAD) read(x[0], 0);
    if (DS <= 8 && nt == TB) {
#pragma unroll
      for (int tt = 0; tt < TB; ++tt) token(tt);
    } else {
#pragma unroll
      for (int tt = 0; tt < TB; ++tt)
        if (tt < nt) token(tt);
    }
  }
#pragma unroll
  for (int i = 0; i < DS; ++i)
    if (v0 < dim && k0 + i < dim) Sp[(long)(k0 + i) * dim + v0] = st[i];
}

// out[b, t] = x[t] + (x[t - 1] - x[t]) * mu[b] for nb blends of the 32-bit rows x; the row before a sequence's
// first row of the step comes from its slot of `state` (zeros at position 0). The thread that reads the slot (the
// first row's) also writes the step's last row into it, after its read, so no other thread touches that element.
template <typename T>
__global__ __launch_bounds__(256) void token_shift_kernel(
    T* __restrict__ out, const float* __restrict__ x, float* __restrict__ state, const float* __restrict__ mu,
    const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx, const int* __restrict__ seq_state, int nseq, int T_,
    int H, int nb) {
  const int t = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  const int s = find_seq(seq_cu, nseq, t);
  if (s < 0 || c >= H) return;
  const int r0 = seq_cu[s], n = seq_cu[s + 1] - r0;
  const float cur = x[(long)t * H + c];
  float prev;
  if (t > r0) {
    prev = x[(long)(t - 1) * H + c];
  } else {
    float* slot = state + (long)seq_state[s] * H + c;
    prev = seq_ctx[s] - n > 0 ? *slot : 0.f;
    *slot = x[(long)(r0 + n - 1) * H + c];
  }
  const float d = prev - cur;
  for (int b = 0; b < nb; ++b) stf<T>(out, ((long)b * T_ + t) * H + c, __builtin_fmaf(d, mu[(long)b * H + c], cur));
}

// proj [4, T, N] = r, k, v, gate pre-activation (N = heads * dim), wl = decay pre-activation (fp32 [T, N]).
// pre[t] = [w = exp(-exp(wl + w0)) | k | r | v] as fp32, bonus[t, h] = sum_c r u k over the head's channels.
template <typename T>
__global__ __launch_bounds__(256) void wkv_prepare_kernel(
    float* __restrict__ pre, float* __restrict__ bonus, const T* __restrict__ proj, long T_,
    const float* __restrict__ wl, const float* __restrict__ w0, const float* __restrict__ u, int heads, int dim) {
  const long t = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long N = (long)heads * dim;
  const T* pr = proj + t * N;
  const T* pk = proj + (T_ + t) * N;
  const T* pv = proj + (2 * T_ + t) * N;
  for (int h = wave; h < heads; h += 4) {
    float b = 0.f;
    for (int e = lane; e < dim; e += 64) {
      const int c = h * dim + e;
      const float r = ldf<T>(pr, c), k = ldf<T>(pk, c);
      pre[t * 4 * N + c] = expf(-expf(wl[t * N + c] + w0[c]));
      pre[t * 4 * N + N + c] = k;
      pre[t * 4 * N + 2 * N + c] = r;
      pre[t * 4 * N + 3 * N + c] = ldf<T>(pv, c);
      b = __builtin_fmaf(r * u[c], k, b);
    }
    b = wave_sum(b);
    if (lane == 0) bonus[t * heads + h] = b;
  }
}

// Same layout as the delta-rule scans: a state column per 16-lane DPP row, DS key channels per lane. Per token
// the read-out uses the state BEFORE the update, so the only chain from token to token is one multiply-add per
// state element; the read-outs' row sums are independent of it.
template <int DS, int TBK, int CV, int NT>
__global__ __launch_bounds__(NT) void wkv_scan_kernel(
    float* __restrict__ o, float* __restrict__ S, const float* __restrict__ pre, const float* __restrict__ bonus,
    const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx, const int* __restrict__ seq_state, int heads,
    int dim) {
  constexpr int DP = kSeg * DS, TB = TBK;
  constexpr int kColsW = NT / kSeg * CV;  // state columns per workgroup
  __shared__ __attribute__((aligned(16))) float sv[TB][3][DP];  // w, k, r (zero past dim)
  __shared__ float sb[TB];
  const int s = blockIdx.z, h = blockIdx.x, zb = blockIdx.y, tid = threadIdx.x;
  const int r0 = seq_cu[s], n = seq_cu[s + 1] - r0;
  if (n <= 0) return;
  const int seg = tid & (kSeg - 1), k0 = seg * DS;
  const int v0 = zb * kColsW + (tid / kSeg) * CV;   // this lane row's first column
  const int N = heads * dim;
  float* Sp = S + (((long)seq_state[s] * heads + h) * dim) * dim;
  const bool carried = seq_ctx[s] - n > 0;
  float st[CV][DS];
#pragma unroll
  for (int cv = 0; cv < CV; ++cv)
#pragma unroll
    for (int i = 0; i < DS; ++i)
      st[cv][i] = (carried && v0 + cv < dim && k0 + i < dim) ? Sp[(long)(k0 + i) * dim + v0 + cv] : 0.f;
  constexpr int kLd = (TB * DP + NT - 1) / NT;
  float rg[3][kLd], rv[TB][CV], rb = 0.f;
  auto fetch = [&](int t0) {
    const int nt = min(TB, n - t0);
#pragma unroll
    for (int it = 0; it < kLd; ++it) {
      const int i = it * NT + tid;
      const int tt = i / DP, k = i % DP;
      const long row = r0 + t0 + tt;
      const int c = h * dim + k;
      const bool in = tt < nt && k < dim;
#pragma unroll
      for (int j = 0; j < 3; ++j) rg[j][it] = in ? pre[row * 4 * N + j * N + c] : 0.f;
    }
    if (tid < nt) rb = bonus[(long)(r0 + t0 + tid) * heads + h];
#pragma unroll
    for (int tt = 0; tt < TB; ++tt)
#pragma unroll
      for (int cv = 0; cv < CV; ++cv)
        rv[tt][cv] = (tt < nt && v0 + cv < dim) ? pre[(long)(r0 + t0 + tt) * 4 * N + 3 * N + h * dim + v0 + cv] : 0.f;
  };
  float* po = o + (long)r0 * N + h * dim + v0 + seg;
  fetch(0);
  for (int t0 = 0; t0 < n; t0 += TB) {
    const int nt = min(TB, n - t0);
    __syncthreads();
#pragma unroll
    for (int it = 0; it < kLd; ++it) {
      const int i = it * NT + tid;
      if (i < TB * DP) {
#pragma unroll
        for (int j = 0; j < 3; ++j) sv[i / DP][j][i % DP] = rg[j][it];
      }
    }
    if (tid < TB) sb[tid] = rb;
    float val[TB][CV];
#pragma unroll
    for (int tt = 0; tt < TB; ++tt)
#pragma unroll
      for (int cv = 0; cv < CV; ++cv) val[tt][cv] = rv[tt][cv];
    __syncthreads();
    if (t0 + TB < n) fetch(t0 + TB);
#pragma unroll
    for (int tt = 0; tt < TB; ++tt) {
      if (tt < nt) {
        float w[DS], kk[DS], rr[DS];
#pragma unroll
        for (int i = 0; i < DS; ++i) { w[i] = sv[tt][0][k0 + i]; kk[i] = sv[tt][1][k0 + i]; rr[i] = sv[tt][2][k0 + i]; }
        const float b = sb[tt];
        float outs[CV];
#pragma unroll
        for (int cv = 0; cv < CV; ++cv) {
          float out = 0.f, out2 = 0.f;
#pragma unroll
          for (int i = 0; i < DS; ++i) {
            if (i & 1) out2 = __builtin_fmaf(st[cv][i], rr[i], out2);
            else out = __builtin_fmaf(st[cv][i], rr[i], out);
            st[cv][i] = __builtin_fmaf(w[i], st[cv][i], kk[i] * val[tt][cv]);
          }
          outs[cv] = __builtin_fmaf(val[tt][cv], b, row_sum(out + out2));
        }
        if (seg < CV && v0 + seg < dim) po[(long)(t0 + tt) * N] = seg == 0 ? outs[0] : outs[CV - 1];
      }
    }
  }
#pragma unroll
  for (int cv = 0; cv < CV; ++cv)
#pragma unroll
    for (int i = 0; i < DS; ++i)
      if (v0 + cv < dim && k0 + i < dim) Sp[(long)(k0 + i) * dim + v0 + cv] = st[cv][i];
}

// Decode rows (one row per sequence): the whole linear-attention step of one (sequence, head) in one workgroup:
// decay bottleneck up-projection wl = w2 . tanh(low) (the tanh rounded to the activation type, as the batched path
// stores it), decay, bonus, read-out from the state before its update, state update, per-head RMS norm, weight and
// SiLU gate. Thread v owns state column v (dim <= blockDim): it walks the key channels, so state reads and writes
// are coalesced across the threads.
template <typename T>
__global__ __launch_bounds__(256) void wkv_step_kernel(
    T* __restrict__ out, float* __restrict__ S, const T* __restrict__ proj, long T_, const T* __restrict__ low,
    const T* __restrict__ w2, int rank, const float* __restrict__ w0, const float* __restrict__ u,
    const float* __restrict__ norm_w, const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx,
    const int* __restrict__ seq_state, int heads, int dim, float eps) {
  extern __shared__ float sm[];   // [rank] tanh(low), then w, k, r [dim] each
  __shared__ float red[16];
  float* tl = sm;
  float* sw = sm + rank;
  float* sk = sw + dim;
  float* sr = sk + dim;
  const int h = blockIdx.x, s = blockIdx.y, tid = threadIdx.x;
  const int t = seq_cu[s];
  if (seq_cu[s + 1] - t != 1) return;   // sequences without a row in this step
  const long N = (long)heads * dim;
  for (int j = tid; j < rank; j += 256) {
    float v = tanhf(ldf<T>(low, (long)t * rank + j));
    if constexpr (sizeof(T) == 2) v = bf16_to_f32(f32_to_bf16(v));
    tl[j] = v;
  }
  __syncthreads();
  float val = 0.f, gate = 0.f, b = 0.f;
  if (tid < dim) {
    const long c = (long)h * dim + tid;
    float a = 0.f;
    for (int j = 0; j < rank; ++j) a = __builtin_fmaf(ldf<T>(w2, c * rank + j), tl[j], a);
    const float r = ldf<T>(proj, t * N + c), k = ldf<T>(proj, (T_ + t) * N + c);
    sw[tid] = expf(-expf(a + w0[c]));
    sk[tid] = k;
    sr[tid] = r;
    val = ldf<T>(proj, (2 * T_ + t) * N + c);
    gate = ldf<T>(proj, (3 * T_ + t) * N + c);
    b = r * u[c] * k;
  }
  b = block_sum(b, red);   // also orders the writes of sw / sk / sr before the reads below
  float o = 0.f;
  if (tid < dim) {
    float* Sp = S + (((long)seq_state[s] * heads + h) * dim) * dim + tid;
    const bool carried = seq_ctx[s] - 1 > 0;
    o = val * b;
#pragma unroll 8
    for (int k = 0; k < dim; ++k) {
      const float st = carried ? Sp[(long)k * dim] : 0.f;
      o = __builtin_fmaf(st, sr[k], o);
      Sp[(long)k * dim] = __builtin_fmaf(sw[k], st, sk[k] * val);
    }
  }
  const float ss = block_sum(tid < dim ? o * o : 0.f, red);
  if (tid < dim) {
    const long c = (long)h * dim + tid;
    stf<T>(out, t * N + c, o / sqrtf(ss / (float)dim + eps) * norm_w[c] * gate * sigmoid_f(gate));
  }
}

// Decode rows (one row per sequence): the whole gated rule of one (sequence, head) in one workgroup: convolution, unit
// query and key, decays and output gate (CH: with their bottlenecks' up-projections), recurrence, norm, gate. The
// state is read and written once: with VEC 4 and at most kStepIt rows per thread it waits in registers (loaded
// before anything else), else it is read once more from the caches. Per element of the OLD state the two sums
//   pred_v = sum_k g_k k_k S_kv,  read_v = sum_k g_k q_k S_kv
// give u_v = beta (v - pred_v) and o_v = read_v + (q . k) u_v, the read-out of the new state S' = g S + k u^T.
// Thread (r, w) owns columns VEC w .. of rows r, r + R, ...
constexpr int kStepThreads = 512, kStepIt = 8, kStepRank = 1024;

// sum_j w[j] x[j] over a bottleneck, shared by the 16 lanes of a DPP row (every lane gets it); x in LDS
template <typename T>
HS_DEVICE float low_dot(const T* __restrict__ w, const float* x, int n, int seg, bool vec) {
  float a = 0.f, b = 0.f;
  if (vec) {
    for (int j = 8 * seg; j < n; j += 128) {
      float v[8];
      Row<T, 8>::ld(w + j, v);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a = __builtin_fmaf(v[i], x[j + i], a);
        b = __builtin_fmaf(v[4 + i], x[j + 4 + i], b);
      }
    }
  } else {
    for (int j = seg; j < n; j += 16) a = __builtin_fmaf(ldf<T>(w, j), x[j], a);
  }
  return row_sum(a + b);
}

// The same from weights that were loaded before x was there: lane seg holds w[8 seg .. 8 seg + 7] (n <= 128).
HS_DEVICE float low_dot8(const u16x8 w, const float* x, int n, int seg) {
  float a = 0.f;
  if (8 * seg < n) {
#pragma unroll
    for (int i = 0; i < 8; ++i) a = __builtin_fmaf(bf16_to_f32(w[i]), x[8 * seg + i], a);
  }
  return row_sum(a);
}

// EARLY (bf16, ranks of a multiple of 8 up to 128, head sizes up to 128): the up-projections' weights are loaded with the state.
// DIM: both head sizes, where the compiler shall know them (0: any). With them, the numbers of a sequence and the arguments in one batch and no division: us with the
// update of the convolution's inputs, heads of 128, 1 and 16 rows of 8 heads 9.0 -> 7.4, 11.3 -> 9.7, of 16 heads 9.0 -> 7.7, 16.0 -> 13.6, of 32 heads 10.1 -> 8.4, 22.3 -> 19.9.
template <typename T, bool CH, int VEC, bool EARLY, int DIM = 0>
__global__ __launch_bounds__(kStepThreads) void gated_delta_step_kernel(
    const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx, const int* __restrict__ seq_state, const T* __restrict__ proj,
    float* __restrict__ state, float* __restrict__ conv_state, const float* __restrict__ conv_w, const GatedDelta p, int group, bool own_conv, bool vec_a,
    bool vec_g) {
  static_assert(!EARLY || (CH && sizeof(T) == 2), "early weights are bf16 bottlenecks");
  constexpr int kEarly = EARLY ? 128 / (kStepThreads / kSeg) : 1;   // rows of each up-projection per lane row
  __shared__ float low[CH ? kStepRank : 1];                                 // [decay bottleneck | gate bottleneck]
  __shared__ float xs[3 * 256];                                             // silu(conv): q | k | v
  __shared__ float sg[256], su[256], sgate[256];                            // decays, u, the gate before its activation
  __shared__ float red[2][4 * kStepThreads];                                // partial sums [r][column]: pred, read
  __shared__ float sc[16], sn[4];
  const int h = blockIdx.x, s = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // the sequence's numbers and the arguments in one batch
  const int t = seq_cu[s], after = seq_cu[s + 1], ctx = seq_ctx[s], slot = seq_state[s];
  const long ld = p.ld;
  const int heads = p.heads, taps = p.taps, off_a = p.off_a, off_g = p.off_g, off_b = p.off_b, kv_heads = p.kv_heads;
  const float *dt_bias = p.dt_bias, *a_log = p.a_log, *norm_w = p.norm_w;
  asm volatile("" ::"s"(t), "s"(after), "s"(ctx), "s"(slot), "s"(ld), "s"(heads), "s"(kv_heads), "s"(group), "s"(taps), "s"(off_a), "s"(off_g), "s"(off_b),
               "s"(dt_bias), "s"(a_log), "s"(norm_w), "s"(p.y), "s"(p.y_ld), "s"(p.eps));
  if (after - t != 1) return;   // sequences without a row in this step
  const int dim = DIM > 0 ? DIM : p.dim, vdim = DIM > 0 ? DIM : p.vdim, hist = taps - 1;
  const int nqk = kv_heads * dim, C = 2 * nqk + heads * vdim, kh = group == 1 ? h : h / group;
  const bool carried = ctx - 1 > 0;
  const T* row = proj + (long)t * ld;
  float* Sp = state + ((long)slot * heads + h) * dim * vdim;
  const int W = vdim / VEC, R = kStepThreads / W, r = tid / W, w = tid - r * W;
  const bool active = r < R;
  const bool kept = VEC == 4 && dim <= R * kStepIt;
  // All that is small before the state: loads come back in order, and the chain (convolution, unit vectors, decays) runs while the state's
  // 64 KB arrive. One launch of 16 sequences x 16 heads 13.3 -> 11.8 us, of one x 8 9.2 -> 8.0 (each tap waited
  // for the one before it, all of them for the state, and gates and weights were asked for where they are used).
  constexpr int kTaps = 4;
  const int channels = 2 * dim + vdim;
  const bool quick = taps <= kTaps && channels <= kStepThreads;
  float* cs = conv_state + (long)slot * max(hist, 1) * C;
  auto channel_of = [&](int i) {
    return i < dim ? kh * dim + i : i < 2 * dim ? nqk + kh * dim + i - dim : 2 * nqk + h * vdim + i - 2 * dim;
  };
  float now = 0.f, old[kTaps - 1], cwt[kTaps];
  const float beta_in = ldf<T>(row, off_b + h), weight = tid < vdim ? norm_w[tid] : 0.f;   // vdim <= 256
  float decay_in = 0.f, bias_in = 0.f, rate = 0.f, gate_in = 0.f;
  if constexpr (!CH) {
    decay_in = ldf<T>(row, off_a + h);
    bias_in = dt_bias[h];
    rate = a_log[h];
    if (tid < vdim) gate_in = ldf<T>(row, off_g + h * vdim + tid);
  }
  if (quick) {
    const int c = channel_of(min(tid, channels - 1));
    now = ldf<T>(row, c);
#pragma unroll
    for (int j = 0; j < kTaps; ++j) {
      cwt[j] = j < taps ? conv_w[(long)c * taps + j] : 0.f;
      if (j < kTaps - 1) old[j] = carried && j < hist ? cs[(long)j * C + c] : 0.f;
    }
  }
  f32x4 st[VEC == 4 ? kStepIt : 1];
  if constexpr (VEC == 4) {
    if (kept) {
#pragma unroll
      for (int i = 0; i < kStepIt; ++i) {
        const int k = r + i * R;
        st[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (active && k < dim && carried) st[i] = *reinterpret_cast<const f32x4*>(Sp + (long)k * vdim + 4 * w);
      }
    }
  }
  const int seg = tid & (kSeg - 1);
  u16x8 wa[kEarly], wg[kEarly];
  if constexpr (EARLY) {
#pragma unroll
    for (int i = 0; i < kEarly; ++i) {
      const int e = tid / kSeg + i * (kStepThreads / kSeg);
      wa[i] = wg[i] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
      if (e < dim && 8 * seg < p.ra) wa[i] = *reinterpret_cast<const u16x8*>((const T*)p.a2 + ((long)h * dim + e) * p.ra + 8 * seg);
      if (e < vdim && 8 * seg < p.rg) wg[i] = *reinterpret_cast<const u16x8*>((const T*)p.g2 + ((long)h * vdim + e) * p.rg + 8 * seg);
    }
  }
  if constexpr (CH) {
    for (int j = tid; j < p.ra + p.rg; j += kStepThreads)
      low[j] = j < p.ra ? ldf<T>(row, off_a + j) : ldf<T>(row, off_g + j - p.ra);
  }
  // the convolution of the head's channels; with heads of their own queries and keys the kept inputs move on here
  if (quick && tid < channels) {
    const int c = channel_of(tid);
    float a = 0.f, last = 0.f;
#pragma unroll
    for (int j = 0; j < kTaps - 1; ++j) {
      if (j < hist) a = __builtin_fmaf(cwt[j], old[j], a);
      last = j + 1 == hist ? cwt[j + 1] : hist == 0 ? cwt[0] : last;
      if (own_conv && j > 0 && j < hist) cs[(long)(j - 1) * C + c] = old[j];
    }
    if (own_conv && hist > 0) cs[(long)(hist - 1) * C + c] = now;
    a = __builtin_fmaf(last, now, a);
    xs[tid] = a * sigmoid_f(a);
  }
  for (int i = quick ? channels : tid; i < channels; i += kStepThreads) {
    const int c = channel_of(i);
    const float cur = ldf<T>(row, c);
    const float* cw = conv_w + (long)c * taps;
    float a = 0.f;
    for (int j = 0; j < hist; ++j) {
      const float x = carried ? cs[(long)j * C + c] : 0.f;
      a = __builtin_fmaf(cw[j], x, a);
      if (own_conv && j > 0) cs[(long)(j - 1) * C + c] = x;
    }
    if (own_conv && hist > 0) cs[(long)(hist - 1) * C + c] = cur;
    a = __builtin_fmaf(cw[hist], cur, a);
    xs[i] = a * sigmoid_f(a);
  }
  __syncthreads();
  // unit query and key and their product (waves 0 - 2), decays
  if (wave < 3) {
    float a = 0.f;
    for (int e = lane; e < dim; e += 64) a = __builtin_fmaf(xs[(wave == 1 ? dim : 0) + e], xs[(wave == 0 ? 0 : dim) + e], a);
    a = wave_sum(a);
    if (lane == 0) sn[wave] = a;   // q . q, k . k, q . k
  }
  if constexpr (CH) {
    const float ea = expf(a_log[h]);
    if constexpr (EARLY) {
#pragma unroll
      for (int i = 0; i < kEarly; ++i) {
        const int e = tid / kSeg + i * (kStepThreads / kSeg);
        const float a = low_dot8(wa[i], low, p.ra, seg), b = low_dot8(wg[i], low + p.ra, p.rg, seg);
        if (seg == 0 && e < dim) sg[e] = expf(-ea * softplus_f(a + dt_bias[(long)h * dim + e]));
        if (seg == 0 && e < vdim) sgate[e] = b;
      }
    } else {
      for (int e = tid / kSeg; e < dim; e += kStepThreads / kSeg) {
        const long i = (long)h * dim + e;
        const float a = low_dot<T>((const T*)p.a2 + i * p.ra, low, p.ra, seg, vec_a);
        if (seg == 0) sg[e] = expf(-ea * softplus_f(a + dt_bias[i]));
      }
      for (int e = tid / kSeg; e < vdim; e += kStepThreads / kSeg) {
        const float a = low_dot<T>((const T*)p.g2 + ((long)h * vdim + e) * p.rg, low + p.ra, p.rg, seg, vec_g);
        if (seg == 0) sgate[e] = a;
      }
    }
  } else {
    const float g = expf(-expf(rate) * softplus_f(decay_in + bias_in));
    if (tid < dim) sg[tid] = g;   // dim, vdim <= 256
    if (tid < vdim) sgate[tid] = gate_in;
  }
  __syncthreads();
  const float fq = 1.f / sqrtf(sn[0] + 1e-6f) / sqrtf((float)dim), fk = 1.f / sqrtf(sn[1] + 1e-6f);
  const float qk = sn[2] * fq * fk;
  const float* xq = xs;
  const float* xk = xs + dim;
  float pr[VEC], rd[VEC];
#pragma unroll
  for (int i = 0; i < VEC; ++i) pr[i] = rd[i] = 0.f;
  if (active && carried) {
    if (kept) {
      if constexpr (VEC == 4) {
#pragma unroll
        for (int i = 0; i < kStepIt; ++i) {
          const int k = r + i * R;
          if (k < dim) {
            const float g = sg[k], gk = g * xk[k], gq = g * xq[k];
#pragma unroll
            for (int e = 0; e < 4; ++e) { pr[e] = __builtin_fmaf(gk, st[i][e], pr[e]); rd[e] = __builtin_fmaf(gq, st[i][e], rd[e]); }
          }
        }
      }
    } else {
      for (int k = r; k < dim; k += R) {
        const float g = sg[k], gk = g * xk[k], gq = g * xq[k];
        float v[VEC];
        Row<float, VEC>::ld(Sp + (long)k * vdim + VEC * w, v);
#pragma unroll
        for (int e = 0; e < VEC; ++e) { pr[e] = __builtin_fmaf(gk, v[e], pr[e]); rd[e] = __builtin_fmaf(gq, v[e], rd[e]); }
      }
    }
  }
  if (active) {
#pragma unroll
    for (int e = 0; e < VEC; ++e) { red[0][r * vdim + VEC * w + e] = pr[e]; red[1][r * vdim + VEC * w + e] = rd[e]; }
  }
  __syncthreads();
  float o = 0.f;
  if (tid < vdim) {
    float a = 0.f, b = 0.f;
    for (int i = 0; i < R; ++i) { a += red[0][i * vdim + tid]; b += red[1][i * vdim + tid]; }
    const float u = sigmoid_f(beta_in) * (xs[2 * dim + tid] - fk * a);
    su[tid] = u;
    o = fq * b + qk * u;
  }
  const float ss = block_sum(tid < vdim ? o * o : 0.f, sc);   // also orders the writes of su before the reads below
  if (tid < vdim) {
    const float gp = sgate[tid], gv = sigmoid_f(gp) * (p.silu ? gp : 1.f);
    stf<T>((T*)p.y, (long)t * p.y_ld + (long)h * vdim + tid, o / sqrtf(ss / (float)vdim + p.eps) * weight * gv);
  }
  if (!active) return;
  float u[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) u[e] = fk * su[VEC * w + e];
  if (kept) {
    if constexpr (VEC == 4) {
#pragma unroll
      for (int i = 0; i < kStepIt; ++i) {
        const int k = r + i * R;
        if (k < dim) {
          const float g = sg[k], kk = xk[k];
          f32x4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = __builtin_fmaf(kk, u[e], g * st[i][e]);
          *reinterpret_cast<f32x4*>(Sp + (long)k * vdim + 4 * w) = v;
        }
      }
    }
  } else {
    for (int k = r; k < dim; k += R) {
      const float g = sg[k], kk = xk[k];
      float v[VEC];
#pragma unroll
      for (int e = 0; e < VEC; ++e) v[e] = 0.f;
      if (carried) Row<float, VEC>::ld(Sp + (long)k * vdim + VEC * w, v);
#pragma unroll
      for (int e = 0; e < VEC; ++e) v[e] = __builtin_fmaf(kk, u[e], g * v[e]);
      Row<float, VEC>::st(Sp + (long)k * vdim + VEC * w, v);
    }
  }
}

// One wave per (token, head): out = o / rms(o) * w[head * w_stride + e] * act(gate) * scale.
template <typename T>
__global__ __launch_bounds__(256) void head_norm_gate_kernel(
    T* __restrict__ out, long out_ld, const float* __restrict__ o, const T* __restrict__ proj, long ld, int gate_off,
    const float* __restrict__ w, int w_stride, int rows, int heads, int vdim, float eps, bool silu, float scale) {
  const long idx = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (idx >= (long)rows * heads) return;
  const long t = idx / heads;
  const int h = idx % heads;
  const float* src = o + (t * heads + h) * vdim;
  float a = 0.f;
  for (int e = lane; e < vdim; e += 64) { const float x = src[e]; a += x * x; }
  const float inv = scale / sqrtf(wave_sum(a) / (float)vdim + eps);
  const T* gate = proj + t * ld + gate_off + (long)h * vdim;
  for (int e = lane; e < vdim; e += 64) {
    const float gp = ldf<T>(gate, e);
    const float gv = silu ? gp * sigmoid_f(gp) : sigmoid_f(gp);
    stf<T>(out, t * out_ld + (long)h * vdim + e, src[e] * inv * w[h * w_stride + e] * gv);
  }
}

// The same for value sizes of 8, 16, ... 512 and rows at multiples of 16 bytes: 8 channels per thread, the threads of a head
// within a wave. Memory bounds it: 8192 rows x 16 heads of 128 in bf16 with 4- and 2-byte accesses 70 us, this 38 (3.5 TB/s).
template <typename T>
__global__ __launch_bounds__(256) void head_norm_gate_vec_kernel(
    T* __restrict__ out, long out_ld, const float* __restrict__ o, const T* __restrict__ proj, long ld, int gate_off,
    const float* __restrict__ w, int w_stride, long items, int heads, int vdim, float eps, bool silu, float scale) {
  const long idx = (long)blockIdx.x * 256 + threadIdx.x, it = min(idx, items - 1);
  const int per = vdim / 8, e = (int)(it & (per - 1)) * 8;
  const long hh = it >> __builtin_ctz(per), t = hh / heads;
  const int h = (int)(hh - t * heads);
  float x[8], g[8], f[8];
  Row<float, 8>::ld(o + hh * vdim + e, x);
  Row<T, 8>::ld(proj + t * ld + gate_off + (long)h * vdim + e, g);
  Row<float, 8>::ld(w + (long)h * w_stride + e, f);
  float a = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) a += x[i] * x[i];
  for (int d = 1; d < per; d <<= 1) a += __shfl_xor(a, d, 64);
  if (idx >= items) return;
  const float inv = scale / sqrtf(a / (float)vdim + eps);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float s = sigmoid_f(g[i]);
    x[i] = x[i] * inv * f[i] * (silu ? g[i] * s : s);
  }
  Row<T, 8>::st(out + t * out_ld + (long)h * vdim + e, x);
}

template <typename T>
void head_norm_gate(void* out, long out_ld, const float* o, const void* proj, long ld, int gate_off, const float* w,
                    int w_stride, int rows, int heads, int vdim, float eps, bool silu, float scale, hipStream_t s) {
  const long n = (long)rows * heads;
  uintptr_t at = out_ld * sizeof(T) | ld * sizeof(T) | gate_off * sizeof(T) | w_stride * sizeof(float);
  for (const void* p : {(const void*)out, (const void*)o, (const void*)proj, (const void*)w}) at |= reinterpret_cast<uintptr_t>(p);
  if (vdim >= 8 && vdim <= 512 && (vdim & (vdim - 1)) == 0 && at % 16 == 0 && n > 0) {
    const long items = n * (vdim / 8);
    head_norm_gate_vec_kernel<T><<<(unsigned)((items + 255) / 256), 256, 0, s>>>((T*)out, out_ld, o, (const T*)proj, ld, gate_off, w,
                                                                                 w_stride, items, heads, vdim, eps, silu, scale);
    return;
  }
  head_norm_gate_kernel<T><<<(unsigned)((n + 3) / 4), 256, 0, s>>>((T*)out, out_ld, o, (const T*)proj, ld, gate_off, w,
                                                                   w_stride, rows, heads, vdim, eps, silu, scale);
}

int ds_of(int dim) { return dim <= 16 ? 1 : dim <= 32 ? 2 : dim <= 64 ? 4 : dim <= 128 ? 8 : 16; }

}  // namespace

int delta_max_dim() { return 256; }
int delta_max_taps() { return kMaxHist + 1; }

int gated_delta_step_max_rank() { return kStepRank; }

namespace {

template <typename T>
void conv_state_update(const GatedDelta& p, hipStream_t s) {
  const int C = 2 * p.kv_heads * p.dim + p.heads * p.vdim;
  auto fn = p.taps == 4 ? &conv_state_update_kernel<T, 3> : &conv_state_update_kernel<T, 0>;
  fn<<<dim3(p.nseq, (C + 255) / 256), 256, 0, s>>>(p.seq_cu, p.seq_ctx, p.seq_state, (const T*)p.proj, p.conv_state, C, p.taps, p.ld);
}

template <typename T, bool CH>
void gated_delta(const GatedDelta& p, float* scratch, hipStream_t s) {
  const int nqk = p.kv_heads * p.dim, nv = p.heads * p.vdim, ng = CH ? p.heads * p.dim : p.heads;
  const long T_ = p.T;
  float* qk = scratch;            // [T, 2 nqk]
  float* gg = qk + T_ * 2 * nqk;  // [T, ng]
  float* vv = gg + T_ * ng;       // [T, nv]
  float* bb = vv + T_ * nv;       // [T, heads]
  float* o = bb + T_ * p.heads;   // [T, nv]
  const int items = 2 * p.kv_heads + (nv + 64 * kPrepCh - 1) / (64 * kPrepCh) + (CH ? p.heads : 1) + 1;
  const int run = prep_run(p.T, (items + 3) / 4);
  dim3 pgrid((p.T + run - 1) / run, (items + 3) / 4);
#define HS_GP(N)                                                                                                       \
  gated_delta_prepare_kernel<T, N, CH><<<pgrid, 256, 0, s>>>(qk, vv, gg, bb, (const T*)p.proj, p.ld, p.decay,           \
                                                             p.conv_state, p.conv_w, p.a_log, p.dt_bias, p.seq_cu,      \
                                                             p.seq_ctx, p.seq_state, p.nseq, p.T, p.heads, p.kv_heads,  \
                                                             p.dim, p.vdim, p.taps, p.off_a, p.off_b, run)
  if (p.taps == 4) HS_GP(4); else if (p.taps == 3) HS_GP(3); else if (p.taps == 2) HS_GP(2); else HS_GP(0);
#undef HS_GP
  conv_state_update<T>(p, s);
  if (p.chunks != nullptr) {
    launch_delta_chunk(o, p.S, p.chunks, qk, vv, gg, bb, p.seq_cu, p.seq_ctx, p.seq_state, p.nseq, p.T, p.heads, p.kv_heads,
                       p.dim, p.vdim, CH, s);
  } else {
    dim3 grid(p.heads, (p.vdim + kCols - 1) / kCols, p.nseq);
    switch (ds_of(p.dim)) {
#define HS_GD(D)                                                                                                     \
  case D:                                                                                                            \
    gated_delta_scan_kernel<D, CH><<<grid, kScanThreads, 0, s>>>(o, p.S, qk, vv, gg, bb, p.seq_cu, p.seq_ctx,          \
                                                                 p.seq_state, p.heads, p.kv_heads, p.dim, p.vdim);    \
    break;
      HS_GD(1) HS_GD(2) HS_GD(4) HS_GD(8) HS_GD(16)
#undef HS_GD
    }
  }
  const bool own = p.gate != nullptr;   // the gate's rows: the bottleneck's result, or columns of the projection
  head_norm_gate<T>(p.y, p.y_ld, o, own ? p.gate : p.proj, own ? nv : p.ld, own ? 0 : p.off_g, p.norm_w, 0, p.T, p.heads,
                    p.vdim, p.eps, p.silu, 1.f, s);
}

template <typename T, bool CH>
void gated_delta_step(const GatedDelta& p, hipStream_t s) {
  const bool own_conv = p.heads == p.kv_heads;
  auto ok = [](const void* q, int n) { return n % 8 == 0 && reinterpret_cast<uintptr_t>(q) % 16 == 0; };
  const bool va = ok(p.a2, p.ra), vg = ok(p.g2, p.rg);
  const int group = p.heads / p.kv_heads;
  auto go = [&](auto* kernel) {
    kernel<<<dim3(p.heads, p.nseq), kStepThreads, 0, s>>>(p.seq_cu, p.seq_ctx, p.seq_state, (const T*)p.proj, p.S, p.conv_state, p.conv_w, p, group, own_conv,
                                                         va, vg);
  };
  bool early = false;
  if constexpr (CH && sizeof(T) == 2) {
    early = va && vg && p.ra <= 128 && p.rg <= 128 && p.dim <= 128 && p.vdim <= 128 && p.vdim % 4 == 0;
    if (early) go(&gated_delta_step_kernel<T, CH, 4, true>);
  }
  if (early) {
  } else if (!CH && p.dim == 128 && p.vdim == 128) {   // the head size of this package's own configurations (both sides: at the kernel)
    if constexpr (!CH) go(&gated_delta_step_kernel<T, CH, 4, false, 128>);
  } else if (p.vdim % 4 == 0) {
    go(&gated_delta_step_kernel<T, CH, 4, false>);
  } else {
    go(&gated_delta_step_kernel<T, CH, 1, false>);
  }
  if (!own_conv && p.update_conv) conv_state_update<T>(p, s);   // its readers are other workgroups too: after all of them
}

}  // namespace

void launch_gated_delta(const GatedDelta& p, float* scratch, bool f32, hipStream_t s) {
  if (p.nseq <= 0 || p.T <= 0) return;
  if (f32) { if (p.channel) gated_delta<float, true>(p, scratch, s); else gated_delta<float, false>(p, scratch, s); }
  else if (p.channel) gated_delta<unsigned short, true>(p, scratch, s);
  else gated_delta<unsigned short, false>(p, scratch, s);
}

void launch_gated_delta_step(const GatedDelta& p, bool f32, hipStream_t s) {
  if (p.nseq <= 0 || p.T <= 0) return;
  if (f32) { if (p.channel) gated_delta_step<float, true>(p, s); else gated_delta_step<float, false>(p, s); }
  else if (p.channel) gated_delta_step<unsigned short, true>(p, s);
  else gated_delta_step<unsigned short, false>(p, s);
}

void launch_conv_update(const ConvUpdate& c, int nseq, bool f32, hipStream_t s) {
  if (nseq <= 0) return;
  GatedDelta p{};
  p.seq_cu = c.seq_cu; p.seq_ctx = c.seq_ctx; p.seq_state = c.seq_state; p.proj = c.proj; p.conv_state = c.conv_state; p.ld = c.ld; p.nseq = nseq;
  p.taps = c.taps; p.heads = 1; p.vdim = c.C;   // so many channels
  if (f32) conv_state_update<float>(p, s); else conv_state_update<unsigned short>(p, s);
}

void launch_delta_rule(void* out, long out_ld, float* S, const void* proj, long ld, const float* wl, const float* a_b,
                       const float* w0, const float* norm_w, const int* seq_cu, const int* seq_ctx,
                       const int* seq_state, int nseq, int T, float* scratch, int heads, int dim, float eps,
                       float out_scale, bool f32, float* chunks, hipStream_t s) {
  if (nseq <= 0 || T <= 0) return;
  const int N = heads * dim;
  if (chunks != nullptr) {
    launch_delta_rule_chunk(scratch, S, chunks, proj, ld, wl, a_b, w0, seq_cu, seq_ctx, seq_state, nseq, T, heads, s);
    head_norm_gate<unsigned short>(out, out_ld, scratch, proj, ld, 4 * N, norm_w, dim, T, heads, dim, eps, false, out_scale, s);
    return;
  }
  float* pre = scratch;               // [T, 6 N]
  float* o = pre + (long)T * 6 * N;   // [T, N]
  dim3 grid(heads, (dim + kCols - 1) / kCols, nseq);
  if (f32) {
    delta_rule_prepare_kernel<float><<<T, 256, 0, s>>>(pre, (const float*)proj, ld, wl, a_b, w0, heads, dim);
    switch (ds_of(dim)) {
#define HS_DR(D)                                                                                                  \
  case D:                                                                                                         \
    delta_rule_scan_kernel<float, D><<<grid, kScanThreads, 0, s>>>(o, S, pre, (const float*)proj, ld, seq_cu, seq_ctx,      \
                                                         seq_state, heads, dim);                                  \
    break;
      HS_DR(1) HS_DR(2) HS_DR(4) HS_DR(8) HS_DR(16)
#undef HS_DR
    }
    head_norm_gate<float>(out, out_ld, o, proj, ld, 4 * N, norm_w, dim, T, heads, dim, eps, false, out_scale, s);
  } else {
    delta_rule_prepare_kernel<unsigned short><<<T, 256, 0, s>>>(pre, (const unsigned short*)proj, ld, wl, a_b, w0,
                                                                heads, dim);
    switch (ds_of(dim)) {
#define HS_DR(D)                                                                                                   \
  case D:                                                                                                          \
    delta_rule_scan_kernel<unsigned short, D><<<grid, kScanThreads, 0, s>>>(o, S, pre, (const unsigned short*)proj, ld, seq_cu, \
                                                                  seq_ctx, seq_state, heads, dim);                 \
    break;
      HS_DR(1) HS_DR(2) HS_DR(4) HS_DR(8) HS_DR(16)
#undef HS_DR
    }
    head_norm_gate<unsigned short>(out, out_ld, o, proj, ld, 4 * N, norm_w, dim, T, heads, dim, eps, false, out_scale,
                                   s);
  }
}

void launch_token_shift(void* out, const float* x, float* state, const float* mu, const int* seq_cu,
                        const int* seq_ctx, const int* seq_state, int nseq, int T, int H, int nb, bool f32,
                        hipStream_t s) {
  if (nseq <= 0 || T <= 0) return;
  dim3 grid(T, (H + 255) / 256);
  if (f32) token_shift_kernel<float><<<grid, 256, 0, s>>>((float*)out, x, state, mu, seq_cu, seq_ctx, seq_state, nseq, T, H, nb);
  else token_shift_kernel<unsigned short><<<grid, 256, 0, s>>>((unsigned short*)out, x, state, mu, seq_cu, seq_ctx,
                                                              seq_state, nseq, T, H, nb);
}

void launch_wkv(void* out, float* S, const void* proj, const float* wl, const float* w0, const float* u,
                const float* norm_w, const int* seq_cu, const int* seq_ctx, const int* seq_state, int nseq, int T,
                float* scratch, int heads, int dim, float eps, bool f32, hipStream_t s) {
  if (nseq <= 0 || T <= 0) return;
  const long N = (long)heads * dim;
  float* pre = scratch;                   // [T, 4 N]
  float* bonus = pre + (long)T * 4 * N;   // [T, heads]
  float* o = bonus + (long)T * heads;     // [T, N]
  if (f32) wkv_prepare_kernel<float><<<T, 256, 0, s>>>(pre, bonus, (const float*)proj, T, wl, w0, u, heads, dim);
  else wkv_prepare_kernel<unsigned short><<<T, 256, 0, s>>>(pre, bonus, (const unsigned short*)proj, T, wl, w0, u, heads, dim);
  // prompt portions (many rows per sequence): 16 tokens per staged batch and 32 state columns per workgroup
  // (measured 7 % faster than 8 / 16 on 2048-row sequences); decode rows keep the small workgroup
  const bool wide = T >= 64 * nseq;
  const int cols = (wide ? 512 : kScanThreads) / kSeg;
  dim3 grid(heads, (dim + cols - 1) / cols, nseq);
#define HS_WKV(D, TB, NT) wkv_scan_kernel<D, TB, 1, NT><<<grid, NT, 0, s>>>(o, S, pre, bonus, seq_cu, seq_ctx, seq_state, heads, dim)
  switch (ds_of(dim)) {
#define HS_WK(D)                                                            \
  case D:                                                                   \
    if (wide) HS_WKV(D, 16, 512); else HS_WKV(D, kTB, kScanThreads);        \
    break;
    HS_WK(1) HS_WK(2) HS_WK(4) HS_WK(8) HS_WK(16)
#undef HS_WK
  }
#undef HS_WKV
  // the gate's pre-activation is the fourth projection: rows of N from proj + 3 T N
  if (f32)
    head_norm_gate<float>(out, N, o, (const float*)proj + 3 * (long)T * N, N, 0, norm_w, dim, T, heads, dim, eps, true, 1.f, s);
  else
    head_norm_gate<unsigned short>(out, N, o, (const unsigned short*)proj + 3 * (long)T * N, N, 0, norm_w, dim, T, heads,
                                   dim, eps, true, 1.f, s);
}

void launch_wkv_step(void* out, float* S, const void* proj, long T, const void* low, const void* w2, int rank,
                     const float* w0, const float* u, const float* norm_w, const int* seq_cu, const int* seq_ctx,
                     const int* seq_state, int nseq, int heads, int dim, float eps, bool f32, hipStream_t s) {
  if (nseq <= 0 || T <= 0) return;
  dim3 grid(heads, nseq);
  const size_t smem = (size_t)(rank + 3 * dim) * sizeof(float);
  if (f32)
    wkv_step_kernel<float><<<grid, 256, smem, s>>>((float*)out, S, (const float*)proj, T, (const float*)low,
                                                   (const float*)w2, rank, w0, u, norm_w, seq_cu, seq_ctx, seq_state,
                                                   heads, dim, eps);
  else
    wkv_step_kernel<unsigned short><<<grid, 256, smem, s>>>(
        (unsigned short*)out, S, (const unsigned short*)proj, T, (const unsigned short*)low, (const unsigned short*)w2,
        rank, w0, u, norm_w, seq_cu, seq_ctx, seq_state, heads, dim, eps);
}

}  // namespace hipserve

// A workgroup's part of window attention of decode rows (window_attention_decode.hip), for its own launch and for one that holds a delta rule's step besides
// (window_delta_step.hip).
#pragma once
#include <algorithm>
#include <type_traits>

#include "hipserve/seq_kernels.h"
#include "seq_common.h"

namespace hipserve {
namespace {

constexpr int kMaxRuns = 64;
constexpr float kLog2e = 1.44269504088896341f;

// Scores and their exponentials: bf16 in the log2 domain; fp32 in the natural one, exp(d) with the rounding error of d log2(e)
// carried as in sigmoid_f.
template <typename T> struct Softmax;
template <> struct Softmax<unsigned short> {
  static constexpr float kUnit = kLog2e;
  static HS_DEVICE float exp(float d) { return __builtin_amdgcn_exp2f(d); }
  static HS_DEVICE float tanh(float x) { return tanh_fast(x); }
};
template <> struct Softmax<float> {
  static constexpr float kUnit = 1.f;
  static HS_DEVICE float exp(float d) {   // d <= 0
    if (!(d >= -104.f)) return d < -104.f ? 0.f : d;
    const float t = d * 1.44269502f, lo = fmaf(d, 1.92596299e-8f, fmaf(d, 1.44269502f, -t)), e = __builtin_amdgcn_exp2f(t);
    return fmaf(e, lo * 0.693147182f, e);
  }
  static HS_DEVICE float tanh(float x) { return tanhf(x); }
};

template <bool MAX>
HS_DEVICE float over_rows(float x) {   // over the lanes c, c + 16, c + 32, c + 48
  const unsigned u = __builtin_bit_cast(unsigned, x);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const float a0 = __builtin_bit_cast(float, (unsigned)a[0]), a1 = __builtin_bit_cast(float, (unsigned)a[1]);
  const unsigned w = __builtin_bit_cast(unsigned, MAX ? fmaxf(a0, a1) : a0 + a1);
  const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  const float b0 = __builtin_bit_cast(float, (unsigned)b[0]), b1 = __builtin_bit_cast(float, (unsigned)b[1]);
  return MAX ? fmaxf(b0, b1) : b0 + b1;
}

using u32x4 = __attribute__((ext_vector_type(4))) unsigned;

struct NoPrep {};

// N elements of a row as they lie in memory (4 or 8).
template <typename T, int N> struct Raw {
  using V = __attribute__((ext_vector_type(N * sizeof(T) >= 16 ? 4 : 2))) unsigned;
  static constexpr int PER = sizeof(V) / sizeof(T);
  V w[N / PER];
  HS_DEVICE void ld(const T* p) {
#pragma unroll
    for (int i = 0; i < N / PER; ++i) w[i] = reinterpret_cast<const V*>(p)[i];
  }
  HS_DEVICE void get(float* f) const {
#pragma unroll
    for (int e = 0; e < N; ++e) {
      const unsigned u = sizeof(T) == 4 ? w[e / PER][e % PER] : (e & 1) ? w[0][e / 2] & 0xffff0000u : w[0][e / 2 % 4] << 16;
      f[e] = __builtin_bit_cast(float, u);
    }
  }
};

// attn_prepare_vec_kernel's work for one workgroup of a decode step: its query heads, and the new key and value of their
// key / value head, from the projection row into LDS (`heads` [nh][D], then key [D], value [D]), the latter two into the cache
// row as well where `keep_row` says so. What is normed over the whole projection (MODE 1) is summed by every workgroup of the row: 5 KB
// for 16 + 4 heads of 128 in bf16, while the keys' addresses are on their way. `places` asks for the first tile's places, `early` for the tile.
// Loads return in order and nothing here branches between them: the angles' frequencies, the places, the row, then, once the places are there,
// the tile, which is on its way while the row is worked on. MODE: WindowPrep's norm_mode, 0 for 3 too.
template <typename T, int D, int MODE, typename F, typename G>
HS_DEVICE void prepare_row(const WindowPrep& pr, int waves, const T* __restrict__ row, long at, long slot, int head0, int nh, int kvh, int heads,
                           int kv_heads, bool keep_row, T* hs, float* angles, F&& places, G&& early) {
  __shared__ float red[2][8];
  constexpr int PER = D / 8, NS = sizeof(T) == 4 ? 4 : 8;   // NS: loads of the sums in flight beside the tile's, within the registers
  const int tid = threadIdx.x, nt = 64 * waves, lane = tid & 63, wave = tid >> 6;
  const int nq = heads * D, nk = pr.own_kv ? kv_heads * D : 0, rot = pr.nfreq / 4, items = (nh + (pr.own_kv ? 2 : 0)) * PER;
  const int chunks = (nq + nk) / 8;
  int o0 = 0, o1 = 0;
  auto place = [&](int it) {   // of an item: two 4-dim chunks of a head, as rotated pairs have them
    const int h = it / PER, j = it % PER;
    const bool pair = j < rot && h <= nh;
    o0 = pair ? 4 * j : h <= nh ? 2 * pr.nfreq + 8 * (j - rot) : 8 * j;
    o1 = o0 + (pair ? pr.nfreq : 4);
    return row + (h < nh ? (head0 + h) * D : h == nh ? nq + kvh * D : nq + nk + kvh * D);
  };
  Raw<T, 4> lo{}, hi{};
  Raw<T, 8> sum[NS];
  f32x4 wl, wh;
  using Weights = const __attribute__((address_space(1))) f32x4*;
  using Weight = const __attribute__((address_space(1))) float*;
  auto qn = reinterpret_cast<Weight>(reinterpret_cast<unsigned long>(pr.q_norm));
  auto kn = reinterpret_cast<Weight>(reinterpret_cast<unsigned long>(pr.own_kv ? pr.k_norm : pr.q_norm));
  if constexpr (MODE != 0) asm volatile("" : "+s"(qn), "+s"(kn));   // two pointers to choose from, not a place in the arguments
  auto weights = [&](int it) {   // place(it) is the last one; the new value has none, and takes any
    const int h = it / PER;
    const auto w = (h < nh ? qn : kn) + (MODE == 2 ? 0 : h < nh ? (head0 + h) * D : kvh * D);
    wl = *reinterpret_cast<Weights>(w + o0);
    wh = *reinterpret_cast<Weights>(w + o1);
  };
  const float freq = *(pr.nfreq > 0 ? pr.inv_freq + min(lane, pr.nfreq - 1) : reinterpret_cast<const float*>(row));
  places();
  {
    const int it = min(tid, items - 1);
    const T* src = place(it);
    lo.ld(src + o0);
    hi.ld(src + o1);
    if constexpr (MODE != 0) weights(it);
  }
  if constexpr (MODE == 1) {
#pragma unroll
    for (int b = 0; b < NS; ++b) sum[b].ld(row + 8L * min(tid + b * nt, chunks - 1));
  }
  early();
  if (tid >= nt - 64 && lane < pr.nfreq) {   // at most 64 frequencies, by the last wave, which has the fewest items
    float sn, cs;
    sincosf((float)at * freq, &sn, &cs);
    angles[lane] = cs * pr.amp;
    angles[pr.nfreq + lane] = sn * pr.amp;
  }
  float a = 0.f, b = 0.f;
  if constexpr (MODE == 1) {
    auto add = [&](int i0) {
#pragma unroll
      for (int n = 0; n < NS; ++n) {
        const int i = tid + i0 + n * nt;
        float x[8], v[4] = {};
        sum[n].get(x);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e & 3] += x[e] * x[e];
        const float t = i < chunks ? (v[0] + v[1]) + (v[2] + v[3]) : 0.f;
        a += 8 * i < nq ? t : 0.f;
        b += 8 * i < nq ? 0.f : t;
      }
    };
    add(0);   // apart from the others, whose loads would have this one wait for the tile
    for (int i0 = NS * nt; i0 < chunks; i0 += NS * nt) {
#pragma unroll
      for (int n = 0; n < NS; ++n) sum[n].ld(row + 8L * min(tid + i0 + n * nt, chunks - 1));
      add(i0);
    }
    a = wave_sum(a);
    b = wave_sum(b);
    if (lane == 0) { red[0][wave] = a; red[1][wave] = b; }
  }
  float x[4], y[4], ss = 0.f;   // an item's elements and the sum of its head's squares
  auto take = [&](int it) {   // place(it) is the last one
    const int h = it / PER, j = it % PER;
    lo.get(x);
    hi.get(y);
    if (pr.norm_mode >= 2 || pr.v_norm) {
      const float grow = pr.norm_mode == 3 && j < rot && h <= nh ? pr.amp : 1.f;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) { const float p = x[e] * grow, q = y[e] * grow; v[e] = p * p + q * q; }
      ss = (v[0] + v[1]) + (v[2] + v[3]);
      static_assert(PER == 8 || PER == 16, "a head's lanes are a lane row or half of one");
      ss = dpp_step<0xB1, 0xf, false>(ss);                              // quad_perm [1, 0, 3, 2]
      ss = dpp_step<0x4E, 0xf, false>(ss);                              // quad_perm [2, 3, 0, 1]
      ss = dpp_step<0x141, 0xf, false>(ss);                             // row_half_mirror
      if constexpr (PER == 16) ss = dpp_step<0x140, 0xf, false>(ss);    // row_mirror
    }
  };
  if ((tid & ~63) < items) take(min(tid, items - 1));   // whole waves: a head's sum is over its lanes
  __syncthreads();
  float iq = 1.f, ik = 1.f;
  if constexpr (MODE == 1) {
    a = b = 0.f;
#pragma unroll
    for (int w = 0; w < 8; ++w) {   // one wait for all of them
      const float u = red[0][w], t = red[1][w];
      a += w < nt / 64 ? u : 0.f;
      b += w < nt / 64 ? t : 0.f;
    }
    iq = 1.f / sqrtf(a / (float)nq + pr.eps);
    ik = 1.f / sqrtf(b / (float)max(nk, 1) + pr.eps);
  }
  const float temp = pr.temp_every > 0 ? 1.f + pr.temp_coef * logf((float)((at + 1) / pr.temp_every) + 1.f) : 1.f;
  T* dst = reinterpret_cast<T*>(pr.cache) + slot * (2L * kv_heads * D) + kvh * D;
  auto item = [&](int it) {
    if (it >= items) return;
    const int h = it / PER, j = it % PER;
    const bool qk = h <= nh, isq = h < nh;
    float f = isq ? iq : qk ? ik : 1.f;
    if (qk ? pr.norm_mode >= 2 : pr.v_norm) f = 1.f / sqrtf(ss / (float)D + pr.eps);
    if (isq) f *= temp;
#pragma unroll
    for (int e = 0; e < 4; ++e) { x[e] *= f; y[e] *= f; }
    if (MODE != 0 && qk) {
#pragma unroll
      for (int e = 0; e < 4; ++e) { x[e] *= wl[e]; y[e] *= wh[e]; }
    }
    if (qk && j < rot) {
      float cs[4], sn[4];
      Row<float, 4>::ld(angles + 4 * j, cs);
      Row<float, 4>::ld(angles + pr.nfreq + 4 * j, sn);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float p = x[e], q = y[e];
        x[e] = p * cs[e] - q * sn[e];
        y[e] = q * cs[e] + p * sn[e];
      }
    }
    Row<T, 4>::st(hs + h * D + o0, x);
    Row<T, 4>::st(hs + h * D + o1, y);
    if (!isq && keep_row) {
      T* to = dst + (qk ? 0 : kv_heads * D);
      Row<T, 4>::st(to + o0, x);
      Row<T, 4>::st(to + o1, y);
    }
  };
  if ((tid & ~63) < items) item(tid);
  for (int it = tid + nt; (it & ~63) < items; it += nt) {
    const T* src = place(min(it, items - 1));
    lo.ld(src + o0);
    hi.ld(src + o1);
    if constexpr (MODE != 0) weights(min(it, items - 1));
    take(min(it, items - 1));
    item(it);
  }
  __syncthreads();
}

// MULTI: prompt portions, tq tokens x hc heads in the 16 rows, tiles of tokens in blockIdx.x; one run.
// PREP: the projection rows come as the product leaves them (one row per sequence), and the new key and value of a row reach its
// own tile through LDS. What bounds a short step is the number of instructions that one wave issues in turn, some 5 cycles each, more than
// memory: the scalars that places and lengths need are asked for in one batch with the arguments, a row's elements are spread over more lanes, the angles
// are the last wave's, and the waves' results are read side by side at the end. us behind a copy of the row, before / with these, keys not in the L2:
// one row of 8 heads over 2, 45 keys 5.9 / 5.1 (normed over the projection 6.9 / 6.2), 16 rows of 16 over 4, 230 keys 9.2 / 8.2, 16 rows of 32 over 8,
// 1000 keys 25.9 / 23.5; fp32, 4 rows of 8 over 2, 300 keys 12.4 / 11.9.
template <typename T, bool PREP> struct WindowRest {
  T* out;
  long out_ld, proj_ld;
  const T* cache;
  float *ws_acc, *ws_ml;
  const float* sink_w;
  int block_shift, seq0, seq1, tq, hc, hchunks, heads, kv_heads, group, gate_off, window, part_keys, keep, chunk, waves, nparts;
  float scale, out_scale, softcap;
  bool sink, channel_gate;
  std::conditional_t<PREP, WindowPrep, NoPrep> prep;
};

// MODE: 3 without the preparation, else prepare_row's. (bx, by, bz): row or tile of rows, key head (and chunk of its queries), run. `lds`: [waves][rows][D],
// [waves][16][2], then what is prepared.
template <typename T, int D, bool MULTI, int MODE>
HS_DEVICE void window_decode_block(int bx, int by, int bz, const T* __restrict__ proj, const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx,
                                   const int* __restrict__ seq_bt, const long* __restrict__ positions, const long* __restrict__ slots, int bt_width,
                                   int T_rows, const WindowRest<T, (MODE < 3)>& rest, float* lds) {
  constexpr bool PREP = MODE < 3;
  constexpr bool F32 = sizeof(T) == 4;
  constexpr int SUB = F32 ? 1 : 2, KT = 16 * SUB;          // 16-key tiles and keys of a wave's tile
  constexpr int QN = F32 ? D / 16 : D / 32;                // 16-byte parts of a row per lane
  // Chains of an fp32 score. Decode rows take two: their outputs are at 0.57 - 0.71 of the error against 64 bits that the kernel without
  // matrix cores has, with one chain 0.96 - 1.02 (over draws of 77 - 2000 keys), in the same time; four: 0.42 - 0.59 and 4 - 9 %
  // slower. Prompts are at 0.97 - 1.0 with one, and two cost them 12 %.
  constexpr int CH = MULTI ? 1 : 2;
  constexpr int E = F32 || D == 64 ? 4 : 8, NB = D / (16 * E);   // dims of a value row per load; loads per row
  using S = Softmax<T>;
  T* __restrict__ const out = rest.out;
  const T* __restrict__ const cache = rest.cache;
  float *__restrict__ const ws_acc = rest.ws_acc, *__restrict__ const ws_ml = rest.ws_ml;
  const float* __restrict__ const sink_w = rest.sink_w;
  const long out_ld = rest.out_ld, proj_ld = rest.proj_ld;
  const int block_shift = rest.block_shift, tq = rest.tq, hc = rest.hc, hchunks = rest.hchunks, heads = rest.heads, kv_heads = rest.kv_heads;
  const int group = rest.group, gate_off = rest.gate_off, window = rest.window, part_keys = rest.part_keys, keep = rest.keep, chunk = rest.chunk;
  const float scale = rest.scale, out_scale = rest.out_scale, softcap = rest.softcap;
  const bool sink = rest.sink, channel_gate = rest.channel_gate;
  int s, tok0, seq_r0, n, ctx;
  [[maybe_unused]] long at = 0, new_slot = -1;
  if constexpr (PREP) {
    // asked for together, with the arguments, as if every sequence had a row, as they have in nearly every step
    const int x = bx, row = min(x, T_rows - 1);
    int cu1 = seq_cu[x + 1];
    seq_r0 = seq_cu[x];
    ctx = seq_ctx[x];
    at = positions[row];
    new_slot = slots[row];
    s = x;
    tok0 = 0;
    n = 1;
    asm volatile("" ::"s"(rest.prep.q_norm), "s"(rest.prep.k_norm), "s"(rest.prep.inv_freq), "s"(rest.prep.nfreq), "s"(rest.prep.norm_mode),
                 "s"(rest.prep.amp), "s"(rest.prep.eps), "s"(proj_ld), "s"(cache), "s"(heads), "s"(kv_heads), "s"(group), "s"(gate_off), "s"(window),
                 "s"(part_keys), "s"(keep), "s"(chunk), "s"(rest.waves), "s"(rest.nparts), "s"(block_shift), "s"(hc), "s"(hchunks));
    if (seq_r0 != x || cu1 != x + 1) {
      if (!find_row(seq_cu, 0, rest.seq1, x, s, tok0)) return;
      seq_r0 = seq_cu[s];
      n = seq_cu[s + 1] - seq_r0;
      ctx = seq_ctx[s];
      at = positions[seq_r0 + tok0];
      new_slot = slots[seq_r0 + tok0];
    }
  } else {
    if (!(MULTI ? find_row_tile(seq_cu, rest.seq0, rest.seq1, tq, bx, s, tok0) : find_row(seq_cu, rest.seq0, rest.seq1, bx, s, tok0))) return;
    seq_r0 = seq_cu[s];
    n = seq_cu[s + 1] - seq_r0;
    ctx = seq_ctx[s];
  }
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = rest.waves, nparts = rest.nparts;   // (not from the launch's sizes: one more load)
  const int kvh = hchunks == 1 ? by : by / hchunks, h0 = hchunks == 1 ? 0 : by % hchunks * hc;
  const int nh = min(hc, group - h0), head0 = kvh * group + h0;
  const int ntok = MULTI ? min(tq, n - tok0) : 1, p_first = ctx - n + tok0, p = p_first + ntok - 1;
  const int lo_all = first_key(max(p_first, 0), window, chunk);
  // this lane's row
  const int rt = MULTI ? c / hc : 0, rh = MULTI ? c % hc : c;
  const bool act = rt < ntok && rh < nh;
  const int head = head0 + (act ? rh : 0), spos = p_first + rt, s_lo = first_key(max(spos, 0), window, chunk);
  const long r0 = seq_r0 + tok0 + (act ? rt : 0);
  const int nk = (window > 0 && keep > 0) ? min(keep, lo_all) : 0;   // kept keys below the window
  const int total = nk + p - lo_all + 1;
  const int lo = bz * part_keys, hi = nparts > 1 ? min(total, lo + part_keys) - 1 : total - 1;
  const int* bt = seq_bt + (long)s * bt_width;
  // The u-th visible key (past the run's end: its last) is row key_of(u) of the sequence, which lies in block bt[key_of(u) >> block_shift].
  const int last = max(hi, 0), in_block = (1 << block_shift) - 1;
  auto key_of = [&](int u) {
    u = min(u, last);
    return u < nk ? u : u - nk + lo_all;
  };
  // Global addresses by their type: of pointers that come from either of two places below the compiler forgets it, and flat loads wait for
  // each other and for LDS (bf16, 64 rows of 32 heads over 8, 1000 keys 54 -> 58 us, before / with those).
  using Row1 = const __attribute__((address_space(1))) T*;
  const Row1 keys = reinterpret_cast<Row1>(reinterpret_cast<unsigned long>(cache));
  auto row_of = [&](int block, int key) {
    return keys + (unsigned long)(unsigned)((block << block_shift) + (key & in_block)) * (unsigned)(2 * kv_heads * D);
  };
  using Keys = u32x4[SUB][QN];
  // as they lie in memory: 16-bit elements of their own are taken apart, and waited for, where they are loaded
  using Part = __attribute__((ext_vector_type(E * sizeof(T) / 4))) unsigned;
  using Values = Part[4 * SUB][NB];
  // A decode row's 16 keys side by side lie in at most two blocks, which are the same in every lane, unless blocks are smaller or keys are kept:
  // ten rows per lane, each with a load and a 64-bit address of its own, were a quarter of a short step's time. us with those two / each lane's own: steps with
  // their preparation in bf16, 1000 keys, 41 rows of 40 heads of 128 over 2 22.7 / 24.7, 64 of 32 of 64 over 4 19.5 / 21.2; decode rows beside prompts in 32
  // bits, 64 of 32 of 128 over 8, 500 keys 53 / 65, of 64 over 4, 1000 keys 29.8 / 34.1; but in bf16, where nothing else is between them, 64 of 32 of 128
  // over 8, 1000 keys 58 / 54, 16 of 256 over 4, 500 keys 31.5 / 29.6.
  const bool near = !MULTI && nk == 0 && block_shift >= 4;
  typedef int i32x2 __attribute__((ext_vector_type(2)));
  using Blocks = i32x2[SUB];
  auto blocks_of = [&](int u0, Blocks& block) {
#pragma unroll
    for (int a = 0; a < SUB; ++a) block[a] = i32x2{bt[key_of(u0 + 16 * a) >> block_shift], bt[key_of(u0 + 16 * a + 15) >> block_shift]};
  };
  using Rows = Row1[5 * SUB];
  auto rows_of = [&](int u0, Rows& src, auto&& block) {   // block(a, key): of a key of the 16 from u0 + 16 a on
    auto row = [&](int a, int u) {
      const int key = key_of(u);
      return row_of(block(a, key), key);
    };
#pragma unroll
    for (int a = 0; a < SUB; ++a) src[a] = row(a, u0 + 16 * a + c) + kvh * D;
#pragma unroll
    for (int i = 0; i < 4 * SUB; ++i) src[SUB + i] = row(i >> 2, u0 + 16 * (i >> 2) + 4 * g + (i & 3)) + (kv_heads + kvh) * D + E * c;
  };
  auto looked_up = [&](int, int key) { return bt[key >> block_shift]; };
  auto rows_of_blocks = [&](int u0, Rows& src, const Blocks& block) {
    rows_of(u0, src, [&](int a, int key) { return key >> block_shift == key_of(u0 + 16 * a) >> block_shift ? block[a][0] : block[a][1]; });
  };
  auto load = [&](const Rows& src, Keys& k, Values& v) {
#pragma unroll
    for (int a = 0; a < SUB; ++a)
#pragma unroll
      for (int i = 0; i < QN; ++i) k[a][i] = reinterpret_cast<const __attribute__((address_space(1))) u32x4*>(src[a])[4 * i + g];
#pragma unroll
    for (int i = 0; i < 4 * SUB; ++i)
#pragma unroll
      for (int b = 0; b < NB; ++b) v[i][b] = *reinterpret_cast<const __attribute__((address_space(1))) Part*>(src[SUB + i] + 16 * E * b);
  };
  const int first = lo + wave * KT;
  constexpr bool EARLY = PREP && D * sizeof(T) <= 256;      // the first tile fits the registers beside the preparation
  T* hs = reinterpret_cast<T*>(lds + nw * (hc * D + 32));   // PREP: the prepared heads, key and value
  bool fresh = false;                                       // the run ends with the row's own key
  [[maybe_unused]] Keys k0;
  [[maybe_unused]] Values v0;
  [[maybe_unused]] Blocks block0;
  [[maybe_unused]] T gate0{};   // of the thread's first results
  if constexpr (PREP) {
    const long slot = rest.prep.own_kv ? new_slot : -1;
    const T* row = proj + r0 * proj_ld;
    fresh = slot >= 0 && hi >= lo && hi == total - 1;
    prepare_row<T, D, MODE>(rest.prep, nw, row, at, slot, head0, nh, kvh, heads, kv_heads, fresh && h0 == 0, hs, reinterpret_cast<float*>(hs + (hc + 2) * D), [&] {
      if (EARLY) blocks_of(first, block0);
      gate0 = row[gate_off >= 0 && !channel_gate ? gate_off + head0 + min(tid / (D / 4), nh - 1) : 0];
    }, [&] {
      if constexpr (EARLY) {
        Rows src;
        if (near) rows_of_blocks(first, src, block0);
        else {
          rows_of(first, src, looked_up);
          __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): the paths meet with none of these look-ups open, for which the other would wait
        }
        load(src, k0, v0);
      }
    });
  }
  u32x4 q[QN];
#pragma unroll
  for (int i = 0; i < QN; ++i) {
    q[i] = u32x4{0, 0, 0, 0};
    if (act) q[i] = reinterpret_cast<const u32x4*>(PREP ? hs + rh * D : proj + r0 * proj_ld + (long)head * D)[4 * i + g];
  }
  f32x4 acc[NB][E];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int j = 0; j < E; ++j) acc[b][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const bool sunk = sink && bz == 0 && wave == 0;
  float m = sunk ? (sink_w != nullptr ? sink_w[head] * S::kUnit : 0.f) : -INFINITY, l = sunk ? 1.f : 0.f;
  const float unit = scale * S::kUnit, cap = softcap * S::kUnit, icap = softcap > 0.f ? scale / softcap : 0.f;

  for (int u0 = first; u0 <= hi; u0 += nw * KT) {
    Keys kl;
    Values vl;
    Keys& k = EARLY ? k0 : kl;
    Values& v = EARLY ? v0 : vl;
    if (!EARLY || u0 != first) {
      Rows src;
      if ((F32 || PREP) && near) {
        Blocks block;
        blocks_of(u0, block);
        rows_of_blocks(u0, src, block);
      } else {
        rows_of(u0, src, looked_up);
      }
      load(src, k, v);
    }
    if (PREP && fresh && hi - u0 < KT) {   // the cache row is being written: its key and value are in LDS
      const T* key = hs + nh * D;
#pragma unroll
      for (int a = 0; a < SUB; ++a)
        if (u0 + 16 * a + c == hi)
#pragma unroll
          for (int i = 0; i < QN; ++i) k[a][i] = reinterpret_cast<const u32x4*>(key)[4 * i + g];
#pragma unroll
      for (int i = 0; i < 4 * SUB; ++i)
        if (u0 + 16 * (i >> 2) + 4 * g + (i & 3) == hi)
#pragma unroll
          for (int b = 0; b < NB; ++b) v[i][b] = *reinterpret_cast<const Part*>(key + D + E * c + 16 * E * b);
    }
    f32x4 sc[SUB];
#pragma unroll
    for (int a = 0; a < SUB; ++a) {
      sc[a] = f32x4{0.f, 0.f, 0.f, 0.f};
      f32x4 part[CH] = {};
#pragma unroll
      for (int i = 0; i < QN; ++i) {
        if constexpr (F32) {
          const f32x4 kf = __builtin_bit_cast(f32x4, k[a][i]), qf = __builtin_bit_cast(f32x4, q[i]);
#pragma unroll
          for (int e = 0; e < 4; ++e) part[e % CH] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[e], qf[e], part[e % CH], 0, 0, 0);
        } else {
          sc[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, k[a][i]), __builtin_bit_cast(bf16x8, q[i]),
                                                          sc[a], 0, 0, 0);
        }
      }
      if constexpr (F32) sc[a] = CH == 2 ? part[0] + part[CH - 1] : part[0];
    }
    // lane (c, g): row c against keys 16 a + 4 g + i
    const bool whole = u0 + KT - 1 <= hi;   // a decode row sees every key of the run
    auto hidden = [&](int u) {
      const int j = u < nk ? u : u - nk + lo_all;
      return u > hi || (MULTI && (j > spos || (j < s_lo && j >= keep)));
    };
    const bool open = MULTI ? __all(whole && u0 >= nk && u0 + KT - 1 - nk + lo_all <= spos && u0 - nk + lo_all >= s_lo) : whole;
    float mx = -INFINITY;
#pragma unroll
    for (int a = 0; a < SUB; ++a)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float x = softcap > 0.f ? cap * S::tanh(sc[a][i] * icap) : sc[a][i] * unit;
        if (!open && hidden(u0 + 16 * a + 4 * g + i)) x = -INFINITY;
        sc[a][i] = x;
        mx = fmaxf(mx, x);
      }
    const float mn = fmaxf(m, over_rows<true>(mx)), al = mn > -INFINITY ? S::exp(m - mn) : 1.f;
    float sum = 0.f, w[4 * SUB];
    u16x8 pk;
#pragma unroll
    for (int i = 0; i < 4 * SUB; ++i) {
      w[i] = mn > -INFINITY ? S::exp(sc[i >> 2][i & 3] - mn) : 0.f;
      if constexpr (!F32) {
        pk[i] = f32_to_bf16(w[i]);       // rounded to bf16: what is multiplied, and what is summed
        w[i] = bf16_to_f32(pk[i]);
      }
      sum += w[i];
    }
    l = l * al + over_rows<false>(sum);
    m = mn;
    if (!whole) {   // a weight of 0 does not hide an infinity behind the run's end
#pragma unroll
      for (int i = 0; i < 4 * SUB; ++i)
        if (u0 + 16 * (i >> 2) + 4 * g + (i & 3) > hi)
#pragma unroll
          for (int b = 0; b < NB; ++b) v[i][b] = Part{};
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
      for (int j = 0; j < E; ++j) acc[b][j] *= al;
      if constexpr (F32) {
#pragma unroll
        for (int j = 0; j < E; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[b][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, (unsigned)v[i][b][j]), w[i], acc[b][j], 0, 0, 0);
      } else {
#pragma unroll
        for (int j = 0; j < E; ++j) {
          u32x4 a;
#pragma unroll
          for (int r = 0; r < 4; ++r)   // keys 2 r and 2 r + 1 of dim j
            a[r] = __builtin_amdgcn_perm(v[2 * r + 1][b][j / 2], v[2 * r][b][j / 2], j & 1 ? 0x07060302u : 0x05040100u);
          acc[b][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, pk),
                                                              acc[b][j], 0, 0, 0);
        }
      }
    }
  }
  // lane (c, g): row c, dims 16 E b + E (4 g + i) + j
  const int nr = MULTI ? 16 : nh;   // rows
  float* ml = lds + nw * nr * D;
  auto put = [&](auto&& of) {
    if (c >= nr) return;
    float* dst = lds + ((long)wave * nr + c) * D;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < E; j += 4)
          *reinterpret_cast<f32x4*>(dst + 16 * E * b + E * (4 * g + i) + j) =
              f32x4{of(acc[b][j][i]), of(acc[b][j + 1][i]), of(acc[b][j + 2][i]), of(acc[b][j + 3][i])};
    if (g == 0) *reinterpret_cast<float2*>(ml + 2 * (c * nw + wave)) = float2{m, l};
  };
  // A wave that sees none of a row's keys leaves zeros: a hidden key's weight of 0 does not hide an infinity or a NaN among its values. (Apart
  // from the others' stores: zeros in the accumulators before one store would be moves of all of them in every step, 0.1 - 0.3 us.)
  const bool none = m == -INFINITY;
  if (__any(none)) put([&](float x) { return none ? 0.f : x; });
  else put([](float x) { return x; });
  __syncthreads();
  for (int it = tid; it < nr * (D / 4); it += 64 * nw) {
    const int h = it / (D / 4), d = it % (D / 4) * 4, ht = MULTI ? h / hc : 0, hh = MULTI ? h % hc : h;
    if (MULTI && (ht >= ntok || hh >= nh)) continue;
    float2 mw[8];
    f32x4 part[8];
#pragma unroll
    for (int w = 0; w < 8; ++w) {   // at most eight waves: what there is of them is asked for at once
      mw[w] = *reinterpret_cast<const float2*>(ml + 2 * (h * nw + min(w, nw - 1)));
      part[w] = *reinterpret_cast<const f32x4*>(lds + ((long)min(w, nw - 1) * nr + h) * D + d);
    }
    float M = mw[0].x, L = 0.f;
#pragma unroll
    for (int w = 1; w < 8; ++w) M = fmaxf(M, mw[w].x);
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 8; ++w) {
      if (w >= nw) break;
      const float f = mw[w].x == -INFINITY ? 0.f : S::exp(mw[w].x - M);   // no key: its sums and outputs are 0 (above)
      L += mw[w].y * f;
      o += part[w] * f;
    }
    const int hd = head0 + hh;
    const long row = seq_r0 + tok0 + ht;
    if (nparts > 1) {
      const long wrow = ((long)bz * heads + hd) * (rest.seq1 - rest.seq0) + bx;
      *reinterpret_cast<f32x4*>(ws_acc + wrow * D + d) = o;
      if (d == 0) { ws_ml[2 * wrow] = M; ws_ml[2 * wrow + 1] = L; }
      continue;
    }
    float f = out_scale;
    if (gate_off >= 0 && !channel_gate) f *= sigmoid_f(PREP && it == tid ? ldf<T>(&gate0, 0) : ldf<T>(proj, row * proj_ld + gate_off + hd));
    f = L == 0.f ? 0.f : f / L;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float cg = channel_gate ? sigmoid_f(ldf<T>(proj, row * proj_ld + gate_off + (long)hd * D + d + e)) : 1.f;
      stf<T>(out, row * out_ld + (long)hd * D + d + e, o[e] * f * cg);
    }
  }
}

// What a launch of decode rows takes: its arguments, its grid, its waves' threads and its LDS.
template <typename T, int D, bool PREP> struct WindowLaunch {
  WindowRest<T, PREP> rest{};
  dim3 grid;
  int waves;
  size_t smem;
  WindowLaunch(T* out, long out_ld, long proj_ld, const T* cache, int block_size, int seq0, int rows, int heads, int kv_heads, int gate_off, float scale,
               int window, bool sink, float out_scale, int nparts, int part_keys, float* ws_acc, float* ws_ml, int keep, float softcap, const float* sink_w,
               bool channel_gate, int chunk, const WindowPrep* prep) {
    const int group = heads / kv_heads, hc = std::min(group, 16), hchunks = (group + hc - 1) / hc;
    // a wave per tile of the run, as many as their accumulators and sums (and the prepared heads and angles) fit 64 KB of LDS
    const int kt = sizeof(T) == 4 ? 16 : 32, wave_floats = hc * D + 32;
    const int prepared = PREP ? ((hc + 2) * D * (int)sizeof(T) + 3) / 4 + 2 * prep->nfreq : 0, room = (1 << 14) - 16 - prepared;
    waves = std::max(1, std::min({8, (part_keys + kt - 1) / kt, room / wave_floats}));
    smem = ((size_t)waves * wave_floats + prepared) * sizeof(float);
    grid = dim3(rows, kv_heads * hchunks, nparts);
    rest.out = out; rest.out_ld = out_ld; rest.proj_ld = proj_ld; rest.cache = cache; rest.ws_acc = ws_acc; rest.ws_ml = ws_ml; rest.sink_w = sink_w;
    rest.block_shift = __builtin_ctz(block_size); rest.seq0 = seq0; rest.seq1 = seq0 + rows; rest.tq = 1; rest.hc = hc; rest.hchunks = hchunks;
    rest.heads = heads; rest.kv_heads = kv_heads; rest.group = group; rest.gate_off = gate_off; rest.window = window; rest.part_keys = part_keys;
    rest.keep = keep; rest.chunk = chunk; rest.scale = scale; rest.out_scale = out_scale; rest.softcap = softcap; rest.sink = sink;
    rest.channel_gate = channel_gate; rest.waves = waves; rest.nparts = nparts;
    if constexpr (PREP) rest.prep = *prep;
  }
};

}  // namespace
}  // namespace hipserve

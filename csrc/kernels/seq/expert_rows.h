// Expert GEMMs of tiles with few live slots: a workgroup's part, for their own launch (expert_ffn.hip) and for launches that hold a
// dense product besides (skinny_linear.hip, mingru.hip).
#pragma once
#include "hipserve/seq_kernels.h"
#include "skinny.h"

namespace hipserve {
namespace {

struct ExpertRest {
  unsigned short* out;
  const float* row_scale;
  int act;
  float limit;
};
struct ExpertArgs {
  const void *slots, *tile_expert, *x, *w;
  int x_ld, N, K, E, gather_k, gather_shift;
  ExpertRest rest;
};

// bf16, tiles with few live slots (decode steps): 16 columns per workgroup, K split over its waves (skinny.h). XG groups of 8 slots:
// moe_align fills a tile from its first slot on, so one is enough for most. mine: the pair in the tile's slot lane % 32: asked for once, together with
// the tile's expert. What bounds it is the memory, and for a few rows the start of its workgroups: one row of 16 experts, two of them hit, 1024 x 2048
// and 2048 x 1024 4.0 -> 3.7 and 3.9 -> 3.6 us with two of 16 tiles launched and without loads of arguments ahead of the copies.
template <int XG, int NT, int DEPTH, bool GLU>
HS_DEVICE void expert_rows(const unsigned short* __restrict__ x, unsigned x_ld, const unsigned char* const (&wt)[NT], const unsigned (&w_row)[2 * NT],
                           int mine, int slot0, int n0, int No, int gather_k, int gather_shift, int K, int rest_at, unsigned char* smem) {
  using SK = Skinny<XG, NT, DEPTH>;
  constexpr int ST = SK::ST;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned x_row[XG];
#pragma unroll
  for (int j = 0; j < XG; ++j) {
    const int r = 8 * j + (lane >> 3), p = __shfl(mine, r, 64);
    const int from = gather_shift >= 0 ? p >> gather_shift : gather_k > 0 ? p / gather_k : slot0 + r;
    x_row[j] = (unsigned)(p < 0 ? 0 : from) * x_ld * 2;   // no pair: any row
  }
  f32x4 acc[NT][ST];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int st = 0; st < ST; ++st) acc[nt][st] = f32x4{0.f, 0.f, 0.f, 0.f};
  unsigned short* out = nullptr;
  const float* row_scale = nullptr;
  int act = 0;
  float limit = 0.f;
  SK::accumulate(acc, wt, w_row, reinterpret_cast<const unsigned char*>(x), x_row, K, smem, lane, wave, [&] {
    const auto rest = late_args<ExpertRest>(rest_at);
    out = rest->out;
    row_scale = rest->row_scale;
    act = rest->act;
    limit = rest->limit;
    asm volatile("" ::"s"(out), "s"(row_scale), "s"(act), "s"(limit));
  });
  float v[NT][(ST + 1) / 2];
  SK::reduce(v, acc, smem);
  const int slot = slot0 + (tid >> 4), p = __shfl(mine, tid >> 4 & 31, 64);   // an element of the [8 XG, 16] result per thread
  if (tid >= 128 * XG || p < 0) return;
  const float f = row_scale != nullptr ? row_scale[p] : 1.f;
#pragma unroll
  for (int nt = 0; nt < (GLU ? 1 : NT); ++nt) {
    const int n = n0 + 16 * nt + (tid & 15);
    if (n >= No) continue;
    float r = v[nt][0] * f;
    if constexpr (GLU) {
      const float u = v[1][0] * f;
      r = act == 3 ? clamped_glu_f(r, u, limit) : r * sigmoid_f(r) * u;
    } else if (act == 1) {
      r = fmaxf(r, 0.f);
      r *= r;
    }
    out[(long)slot * No + n] = f32_to_bf16(r);
  }
}

// Of the widest of the three below: 50 KB, with two tiles (gated) 64 KB, for two workgroups per compute unit at the least: nearly all of them
// are empty where the experts are many, and find that out side by side. Gated ones therefore copy one piece ahead for 8 slots too: two
// (81 KB) took 16 % longer on average (128 experts, 1536 x 2048, 2 of them hit: 9.6 -> 7.5 us, 51 of them 70 -> 60).
template <int NT> constexpr int expert_lds() {
  constexpr int a = Skinny<1, NT, NT == 1 ? 2 : 1>::kLds, b = Skinny<2, NT, 1>::kLds, c = Skinny<4, NT, 1>::kLds;
  constexpr int most = a > b ? (a > c ? a : c) : (b > c ? b : c);
  static_assert(most <= 64 * 1024, "what a launch may ask for as it is");
  return most;
}

// Columns 16 NT bx .. of tile `by`; the arguments that the epilogue needs are an ExpertRest at byte rest_at of the kernel's.
template <int NT, bool GLU>
HS_DEVICE void expert_block(int bx, int by, const int* __restrict__ slots, const int* __restrict__ tile_expert, const unsigned short* __restrict__ x,
                            const unsigned short* __restrict__ w, int x_ld, int N, int K, int E, int gather_k, int gather_shift, int rest_at,
                            unsigned char* smem) {
  const int lane = threadIdx.x & 63, slot0 = by * 32;
  const int e = tile_expert[by], mine = slots[slot0 + (lane & 31)];   // both loads in flight
  const unsigned long live = __ballot(mine >= 0);
  if (e < 0 || e >= E) return;
  const int No = GLU ? N / 2 : N, n0 = bx * (GLU ? 16 : 16 * NT);
  const unsigned char* wt[NT];
  unsigned w_row[2 * NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int first = GLU ? n0 : min(n0 + 16 * nt, N - 1);   // of the tile's columns
    wt[nt] = reinterpret_cast<const unsigned char*>(w + ((long)e * N + (GLU ? nt * No : 0) + first) * K);
#pragma unroll
    for (int h = 0; h < 2; ++h) w_row[2 * nt + h] = (unsigned)min(8 * h + (lane >> 3), No - 1 - first) * (unsigned)K * 2;
  }
#define HS_ER(XG, DEPTH) expert_rows<XG, NT, DEPTH, GLU>(x, x_ld, wt, w_row, mine, slot0, n0, No, gather_k, gather_shift, K, rest_at, smem)
  if (live >> 16 & 0xffff) HS_ER(4, 1);
  else if (live >> 8 & 0xff) HS_ER(2, 1);
  else HS_ER(1, GLU ? 1 : 2);
#undef HS_ER
}

// The experts' part of a launch that holds another product besides: what a workgroup needs behind the tables, in one batch with their loads.
struct ExpertBeside {
  const unsigned short *x, *w;
  int x_ld, N, K, E, gather_k, gather_shift, per_tile;
  ExpertRest rest;
};

// Workgroup `b` of the experts'; ExpertBeside at byte `at` of the kernel's arguments.
HS_DEVICE void expert_beside(int b, const int* __restrict__ slots, const int* __restrict__ tile_expert, int at, unsigned char* smem) {
  const auto a = late_args<ExpertBeside>(at);
  const int tile = __builtin_amdgcn_readfirstlane((unsigned)b / (unsigned)a->per_tile);
  expert_block<1, false>(b - tile * a->per_tile, tile, slots, tile_expert, a->x, a->w, a->x_ld, a->N, a->K, a->E, a->gather_k, a->gather_shift,
                         at + offsetof(ExpertBeside, rest), smem);
}

inline ExpertBeside expert_beside_args(const ExpertRows& ex) {
  const int shift = ex.gather_k > 0 && (ex.gather_k & (ex.gather_k - 1)) == 0 ? __builtin_ctz(ex.gather_k) : -1;
  return {(const unsigned short*)ex.x, (const unsigned short*)ex.w, (int)ex.x_ld, ex.N, ex.K, ex.E, ex.gather_k, shift, (ex.N + 15) / 16,
          {(unsigned short*)ex.out, nullptr, ex.act, 0.f}};
}

}  // namespace
}  // namespace hipserve

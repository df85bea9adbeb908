// A dense product of a few rows and the experts' product of the same step in one launch, where neither reads what the other writes (a parallel block:
// the mixer's products and the experts' both start from the block's norm). A launch of its own costs each at least 1.6 us, which is what empty ones
// in a captured graph take, and about 1 us more until its first loads are back, while the other product would keep the memory busy. The dense
// product's workgroups come first, since they are fewer and longer. The sums are the bits of the two launches; a dense workgroup may take other columns and
// copy fewer pieces ahead than in a launch of its own (skinny_cols and skinny_wide are not asked here).
//
// What bounds it is the memory once the two overlap, and the LDS of the larger workgroup, which all get: with one workgroup per compute unit (more than 80
// KB) the experts lose more than the launch costs, so dense workgroups of more than 16 rows copy one piece ahead. us apart -> in one launch, in a captured
// loop, cold weights, 16 experts of 2048 x 1024 (1 row: two of them hit, 16: 14, 48: all) beside the products of latent attention and minGRU, 1, 16, 48 rows:
// 1616 x 2048 6.8 -> 4.5, 17.2 -> 14.1, 21.2 -> 18.3; 2048 x 2048 6.9 -> 4.6, 17.0 -> 14.3, (19.9 -> 20.0); minGRU's 3 x 4096 x 2048 16.0 -> 13.7, 25.6 -> 22.6,
// (29.9 -> 30.6); 2048 x 4096 8.4 -> 5.9, 18.8 -> 16.1, (21.9 -> 23.6); those in brackets are left apart.
//
// The same order between dependent products (workgroups of the next one copy their weights, then wait for a count of the previous one's) was measured, too: a wait for 256
// workgroups of another XCD takes 7 - 20 us, a launch 1.6.
#include "expert_rows.h"
#include "skinny_block.h"

namespace hipserve {
namespace {

struct BesideArgs {
  const void *x, *w, *slots, *tile_expert;
  int x_ld, M, N, K, ni, split;
  SkinnyRest<kPlain> rest;
  ExpertBeside experts;
};

// Workgroups from `split` on are the experts'.
template <int XG, int NT, int DEPTH, typename TO, bool HALF>
__global__ __launch_bounds__(kSkThreads) void skinny_linear_experts_kernel(
    const unsigned short* __restrict__ x, const unsigned short* __restrict__ w, const int* __restrict__ slots, const int* __restrict__ tile_expert,
    int x_ld, int M, int N, int K, int ni, int split, const SkinnyRest<kPlain>, const ExpertBeside) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  int b = blockIdx.x;
  if (b >= split) {
    expert_beside(b - split, slots, tile_expert, offsetof(BesideArgs, experts), smem);
    return;
  }
  constexpr int per = HALF ? 8 : 16 * NT;
  int part = 0;
  for (const int wgs = (N + per - 1) / per; b >= wgs; ++part) b -= wgs;
  skinny_block<XG, NT, DEPTH, false, TO, false, kPlain, HALF>(b, 0, part, x, w, nullptr, nullptr, x_ld, M, N, K, ni, offsetof(BesideArgs, rest), smem);
}

// Whether the two are faster together where a compute unit has room for two of these workgroups and not for three, which is what the experts have on their
// own: not where thousands of theirs are of a short k, whose start is what they take, nor where the dense ones are many. us apart -> in one launch, 40 rows: 16 experts
// of 4096 x 1024 beside 8192 x 2048 35.8 -> 41.0, 64 of 1024 x 512 22.8 -> 25.7; 16 of 2048 x 1024 beside 4096 x 2048 22.0 -> 22.8, of 1024 x 1024 16.0 -> 15.6. Of 1306
// sizes (1 - 64 rows, 2 M - 32 M dense weights, experts of k 512 - 4096) 488 are left apart for these bounds; of the others one takes more than 1 % longer than apart
// (33 rows, 2.8 %), and all take 17 % less on average; without the bounds 307 do, up to 15 %. With room for three, all were faster together.
// Nor where more than 1.6 rounds of 33 rows and more go onto dense workgroups of one tile, as all here are, which two tiles are for otherwise (skinny_tiles): of 17774
// sizes these are 214, which took 2.9 % less together on average and up to 9.5 % more (56 rows, 16 experts of 2560 x 512 beside 8000 x 2560 24.0 -> 26.3); of the
// others 23 take more than 1 % more, up to 5 %.
bool two_per_unit_pay(const ExpertRows& ex, long wgs, int M, int K, int parts, int split) {
  if (M > 32 && parts == 1 && split >= 416 && K > 2048) return false;
  return ex.K >= 2048 || wgs <= 512 || (wgs <= 1536 && K <= 2048 && split <= 384) || (wgs <= 2560 && split <= 160);
}

template <int XG, int NT, int DEPTH, typename TO, bool HALF = false>
bool launch_beside(void* out, long out_ld, long out_zs, int parts, const void* x, long x_ld, const void* w, int M, int N, int K,
                   const ExpertRows& ex, hipStream_t s) {
  constexpr int dense = Skinny<XG, NT, DEPTH, false, HALF>::kLds, lds = dense > expert_lds<1>() ? dense : expert_lds<1>(), per = HALF ? 8 : 16 * NT;
  static const bool ok = allow_lds(&skinny_linear_experts_kernel<XG, NT, DEPTH, TO, HALF>, lds);
  if (!ok) return false;
  const int split = (N + per - 1) / per * parts;
  const ExpertBeside experts = expert_beside_args(ex);
  if (3 * lds > 160 * 1024 && !two_per_unit_pay(ex, experts.per_tile * ex.ntiles, M, K, parts, split)) return false;
  skinny_linear_experts_kernel<XG, NT, DEPTH, TO, HALF><<<split + experts.per_tile * ex.ntiles, kSkThreads, lds, s>>>(
      (const unsigned short*)x, (const unsigned short*)w, ex.slots, ex.tile_expert, (int)x_ld, M, N, K, ((K + 63) / 64 + parts - 1) / parts * 64, split,
      SkinnyRest<kPlain>{0, out_ld, 0, out_zs, -1, 0, 0.f, 0.f, 1.f, 0.f, out, nullptr, nullptr}, experts);
  return true;
}

}  // namespace

bool launch_skinny_linear_experts(void* out, bool out_f32, long out_ld, long out_zs, int parts, const void* x, long x_ld, const void* w, int M, int N,
                                  int K, const ExpertRows& ex, hipStream_t s) {
  if (M <= 0 || N <= 0 || !expert_rows_ok(ex)) return false;
  const int xg = (M + 7) / 8;
  const long tiles = ((long)N + 15) / 16 * parts;
  auto go = [&](auto f32, auto f16) { return (out_f32 ? f32 : f16)(out, out_ld, out_zs, parts, x, x_ld, w, M, N, K, ex, s); };
#define HS_SB(XG, NT, DEPTH, HALF) go(&launch_beside<XG, NT, DEPTH, float, HALF>, &launch_beside<XG, NT, DEPTH, unsigned short, HALF>)
  if (skinny_half(M, tiles, K / parts)) {
    if (xg <= 1) return K / parts > 4096 ? HS_SB(1, 1, 3, true) : HS_SB(1, 1, 2, true);
    return xg <= 2 ? HS_SB(2, 1, 2, true) : xg <= 4 ? HS_SB(4, 1, 1, true) : xg <= 6 ? HS_SB(6, 1, 1, true) : HS_SB(8, 1, 1, true);
  }
  const int nt = skinny_tiles(M, tiles, K / parts);
  if (nt == 4) return false;   // thousands of columns for many rows: nothing beside them is left to win
  if (nt == 2 && xg <= 4) return xg <= 2 ? HS_SB(2, 2, 1, false) : HS_SB(4, 2, 1, false);
  return xg <= 1 ? HS_SB(1, 1, 2, false) : xg <= 2 ? HS_SB(2, 1, 1, false) : xg <= 4 ? HS_SB(4, 1, 1, false)
       : xg <= 6 ? HS_SB(6, 1, 1, false) : HS_SB(8, 1, 1, false);
#undef HS_SB
}

}  // namespace hipserve

// out[b, m, :] = act(x[b, m, :] . W[b]^T + bias) for up to 64 rows m (decode steps and short prompts): bf16 or 32-bit
// operands, 32-bit accumulation, a result of the operands' type or in 32 bits, row and batch strides of their own for x and out.
// parts > 1: as many 32-bit results, each the sum over a part of K, for a next kernel to add up (the residual update).
// act: 0 tanh, 1 xIELU, 2 squared ReLU, 3 SiLU gate, 4 clamped gate (3, 4: W = [gate rows; up rows], half as many
// columns in out), 5 soft cap, -1 none; they see the unrounded product. act_from: the first column that it applies to (not for gates).
//
// Norms between such products cost a launch of their own, 2.5 - 4 us of a decode step each, nearly all of it latency. A product whose
// result goes into the residual stream therefore can take the update with it (SkinnyNorm with a residual): it adds its result to the
// 32-bit stream, writes the rows times the next norm's weights, and leaves the sums of squares of its 16 or 8 columns; the products that
// read these rows (SkinnyNorm without one) sum the squares and scale their results, of which a norm's factor per row is part
// as well. The rows are rounded once either way, and the update sees the unrounded product. Six norms less in a decode step of Fikizen: one
// row, width 1024, 2450 -> 2328 us (17 steps), 16 rows, width 2048, 9271 -> 8957 (33 steps); both products take about 0.3 us longer.
#include "skinny_block.h"

#include <algorithm>
#include <cmath>

#include "hipserve/seq_kernels.h"

namespace hipserve {
namespace {

template <int XG, int NT, int DEPTH, bool GLU, typename TO, bool F32, int NORM, bool HALF>
__global__ __launch_bounds__(kSkThreads) void skinny_linear_kernel(
    const unsigned short* __restrict__ x, const unsigned short* __restrict__ w, void* p, const void* q, int x_ld, int M, int N, int K, int ni,
    const SkinnyRest<NORM>) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  skinny_block<XG, NT, DEPTH, GLU, TO, F32, NORM, HALF>(blockIdx.x, blockIdx.y, blockIdx.z, x, w, p, q, x_ld, M, N, K, ni,
                                                         offsetof(SkinnyArgs<NORM>, rest), smem);
}

template <int XG, int NT, int DEPTH, bool GLU, typename TO, bool F32, int NORM = kPlain, bool HALF = false>
bool launch_kernel(dim3 grid, void* out, long out_ld, long out_bs, long out_zs, const void* x, long x_ld, long x_bs, const void* w, const void* bias,
                   int M, int N, int K, int act, int act_from, float c0, float c1, hipStream_t s,
                   const std::conditional_t<NORM != kPlain, SkinnyNorm, NoNorm>& norm = {}) {
  constexpr int lds = Skinny<XG, NT, DEPTH, F32, HALF>::kLds;
  static const bool ok = allow_lds(&skinny_linear_kernel<XG, NT, DEPTH, GLU, TO, F32, NORM, HALF>, lds);
  if (!ok) return false;
  SkinnyRest<NORM> rest{x_bs, out_ld, out_bs, out_zs, act, act_from, c0, c1, 1.f, 0.f, out, nullptr, bias};
  void* p = nullptr;
  const void* q = bias;
  int i = ((K + 63) / 64 + (int)grid.z - 1) / (int)grid.z * 64;
  if constexpr (NORM != kPlain) {
    rest.cols = norm.cols;
    rest.eps = norm.eps;
    i = norm.blocks;
    p = norm.squares;
    if constexpr (NORM == kUpdate) {
      p = norm.residual;
      q = norm.weight;
      rest.squares = norm.squares;
    }
  }
  skinny_linear_kernel<XG, NT, DEPTH, GLU, TO, F32, NORM, HALF><<<grid, kSkThreads, lds, s>>>((const unsigned short*)x, (const unsigned short*)w, p, q,
                                                                                        (int)x_ld, M, N, K, i, rest);
  return true;
}

// DEPTH32: of 32-bit operands.
template <int XG, int NT, int DEPTH, bool GLU, bool HALF = false, int DEPTH32 = DEPTH>
bool launch_one(void* out, bool out_f32, long out_ld, long out_bs, long out_zs, int parts, const void* x, long x_ld, long x_bs,
                const void* w, const void* bias, bool f32, int batch, int M, int N, int K, int act, int act_from, float c0, float c1, hipStream_t s) {
  const int cols = GLU ? N / 2 : N, per = GLU ? 16 : 16 * NT - 8 * HALF;
  const dim3 grid((cols + per - 1) / per, batch, parts);
#define HS_SK(TO, F32) launch_kernel<XG, NT, F32 ? DEPTH32 : DEPTH, GLU, TO, F32, kPlain, HALF>(grid, out, out_ld, out_bs, out_zs, x, x_ld, x_bs, w, bias, M, N, K, act, act_from, c0, c1, s)
  return f32 ? HS_SK(float, true) : out_f32 ? HS_SK(float, false) : HS_SK(unsigned short, false);
#undef HS_SK
}

// The same for 16-bit operands alone.
template <int XG, int NT, int DEPTH, bool HALF>
bool launch_16(void* out, bool out_f32, long out_ld, const void* x, long x_ld, const void* w, const void* bias, int M, int N, int K, int act, int act_from,
               float c0, float c1, hipStream_t s) {
  constexpr int per = 16 * NT - 8 * HALF;
#define HS_SK(TO) launch_kernel<XG, NT, DEPTH, false, TO, false, kPlain, HALF>(dim3((N + per - 1) / per), out, out_ld, 0, 0, x, x_ld, 0, w, bias, M, N, K, act, act_from, c0, c1, s)
  return out_f32 ? HS_SK(float) : HS_SK(unsigned short);
#undef HS_SK
}

// us of a launch (K in halves, over `parts`): a latency, the results, and the time the weights take at 5.2 TB/s, or, where that is more, at 9 TB/s and with it
// what the busiest compute unit takes in (80 KB per us), its sums in LDS and its products of 32-bit operands. 9 % off on average over 5127 sizes (1 -
// 64 rows, 64 - 65536 columns, k 128 - 12288, plain and gated, 32 bits).
// per: columns of a workgroup.
double skinny_time_of(int M, long cols, double K, int per, int parts, bool f32, double out_bytes) {
  const long wgs = (cols + per - 1) / per * parts, rounds = (wgs + 255) / 256;
  const double bytes = 2.0 * cols * K, rows = (M + 7) / 8 * 8, k = K / parts, st = (per + 15) / 16 * ((M + 15) / 16);
  const double each = 2.0 * k * (per + rows) / 80e3 + st * (0.09 + (f32 ? 8.5e-5 * k : 0));
  return 2.16 + std::max(bytes / 5.2e6, bytes / 9e6 + rounds * each) + 0.7e-6 * out_bytes;
}

}  // namespace

// How many tiles of 16 columns a workgroup takes. One, unless their workgroups are more than the compute units (or a few of them hold
// many k each): then two or four share what they copy of the rows; up to 16 rows there is too little of that. Cold weights, us with 1 / 2 / 4
// tiles: 6144 x 4096, 16 rows 14.5 / 15.1 / 21, 48 rows 20.9 / 18.7 / 26; 16384 x 2048, 16 rows 17.0 / 15.5 / 15.5, 24 rows 18.3 / 16.4 /
// 16.2, 48 rows 22.6 / 19.4 / 18.8; 32000 x 512, 24 rows 10.4 / 10.0 / 11.9; 16384 x 4096, 64 rows 41.6 / 35.9 / 29.3.
int skinny_tiles(int M, long tiles, int K) {
  if (tiles <= 256) return 1;
  if (M <= 16) return M > 8 && tiles <= 512 && K >= 8192 ? 2 : 1;
  if (tiles <= 512) return K >= 1024 ? 2 : 1;
  if (M > 48) return K >= 1024 ? 4 : 1;
  return K >= 4096 ? 4 : 2;
}

// Whether a workgroup takes half a tile, 8 columns: where whole ones leave half of the compute units idle, and K (in halves) is long enough for what
// a workgroup takes in to matter. Two pieces ahead (three for up to 8 rows of more than 4096). The sums are the same. Cold weights, us, whole ->
// half: 2048 x 2048 with 1, 16, 24 rows 3.6 -> 3.4, 3.8 -> 3.65, 4.25 -> 3.85; 2048 x 6144 with 1, 16, 48 rows 7.3 -> 6.4, 10.1 -> 8.25, 16.2 ->
// 14.0; 1024 x 3072 with 1, 16, 48 rows 3.6 -> 3.6, 4.2 -> 3.9, 6.4 -> 5.9; in 32 bits, 16 rows, 2048 x 2048 7.2 -> 6.3, 1024 x 3072 9.0 -> 7.6. 2048
// x 1024 with 1, 16 rows 2.85 -> 2.95, 2.95 -> 3.0; 2048 x 2048 with 48 rows 5.2 -> 5.35. 1024 x 3072 with one row: no gain, and the sums of squares of an
// update are twice as many (a decode step of width 1024 116 -> 118).
bool skinny_half(int M, long tiles, int K) {
  return tiles <= 128 && (M <= 8 && tiles <= 64 ? K > 4096 : K > 1024) && (M <= 32 || tiles <= 104 || K > 2048);
}

// Columns of a workgroup where whole tiles by the rules above would be rounds of workgroups over the compute units of which the last is far from full: 24, 40, 48 or 56,
// which are one round, or two. 0: by the rules above. 16-bit operands of 9 - 48 rows. What a compute unit takes in, its columns' weights and the rows once per
// workgroup, is what bounds these sizes, and a started round costs as much as a full one. Cold weights, us, by the rules above -> here, 16, 24, 48
// rows: 6144 x 2048 7.7 -> 7.0, 8.0 -> 7.5, 9.9 -> 9.2, 5120 x 4096 12.4 -> 10.2, 13.1 -> 11.2, 15.8 -> 14.4 (24 columns); 10240 x 3072 15.1 -> 13.0, 18.0 ->
// 13.6, 22.7 -> 16.8 (40); 12288 x 4096, 24, 48 rows 22.5 -> 21.1, 25.5 -> 23.6 (48); 13376 x 3072 18.8 -> 16.6, 19.8 -> 17.4, 24.0 -> 20.7 (56); 20480 x 2048, 24
// rows 19.6 -> 18.4 (40, two rounds). A short k is latency, and wider workgroups sum more tiles: 4104 x 1024, 16 rows 4.1 -> 4.6; 8200 x 2048, 16 rows 9.2 -> 9.2;
// 13376 x 2048, 24 rows 14.1 -> 14.3; 20480 x 2048, 48 rows 23.3 -> 24.4: these stay. Nor for 9 - 12 rows where the others are taken for 16: fewer rows are less
// to share, above all where those of the weights lie 4096 bytes apart (9, 12, 16 rows: 11264 x 3328 15.6 -> 16.3, 16.1 -> 16.1, 17.3 -> 16.3; 11264 x 6144 26.8 -> 30.6, 28.2 -> 30.7, 30.4 ->
// 30.7; 28672 x 3072 30.5 -> 32.1, 31.9 -> 32.1, 34.5 -> 32.0). Of 2770 sizes (9 - 48 rows, 4104 - 32000 columns, k 512 - 10240) 1480 are taken, which take 10 % less
// on average and at most 2 % more.
int skinny_cols(int M, long cols, int K) {
  const long tiles = (cols + 15) / 16;
  if (M <= 8 || M > 48 || tiles <= 256 || tiles > 1792) return 0;
  if (tiles <= 384) return K >= (M > 16 ? 1024 : 2048) ? 24 : 0;
  if (tiles <= 512) return 0;
  if (tiles <= 768) {
    if (M <= 16 && (K < 3072 || tiles > (M <= 12 ? 672 : 704) || ((M <= 12 || tiles > 640) && K % 2048 == 0))) return 0;
    return K >= 1024 && !(tiles <= 544 && K < 2048) ? tiles <= 640 ? 40 : 48 : 0;
  }
  if (tiles <= 896) return K >= 3072 && K < (M <= 16 ? 4096 : 1 << 30) ? 56 : 0;
  if (tiles <= 1024) return 0;
  if (tiles <= 1280) return M > 16 && K >= (M > 32 ? 3072 : 1024) ? 40 : 0;
  return tiles > 1536 && M > 12 && K >= 3072 && K < (M <= 16 ? 4096 : 1 << 30) ? 56 : 0;
}

// Of up to 8 rows and more workgroups than compute units: how many pieces a workgroup of one whole tile copies ahead where three are best (0: by the rules of
// the launch), and whether half tiles are better still.
// Three are for weights whose rows lie a multiple of 4096 bytes apart, once the units have a workgroup and a half each, and in 16 bits for k of 2560 and more and two each.
// Half tiles are for up to 4 rows and weights whose rows lie a power of two of bytes apart, 4096 or 16384 and more, where whole tiles' loads of 16 rows meet on
// fewer channels. (8192 apart they take 2 - 10 % longer, for which there is no reason but the measurement; at other multiples of 4096 they gain 2 % on average and lose
// up to 7; rows a little off such places are as fast in whole tiles.) 105 sizes of 5632 - 32000 columns, k 2048, 8192 and 16384, 1 - 4 rows: 10 % less than whole tiles on
// average, one 3.6 % more. Not for rows without their norm's factor (normed): a workgroup sums all of their squares, for half the columns (k 1024 - 4096: 5 - 50 %
// longer than whole tiles, 32000 x 2048 15 %).
// Cold weights, us, one row, one or two pieces / three / half tiles: 8192 x 2048 9.2 / 8.2 / 7.5, 12288 x 2048 12.3 / 11.2 / 10.1, 32000 x 2048 25.8 / 23.9 / 22.1, 32000 x
// 1984 21.7 / 22.1 / 21.4, 32000 x 2112 22.8 / 23.0 / 22.7, 12288 x 2112 10.4 / 10.9 / 10.8, 12288 x 2560 12.1 / 12.2 / 12.0, 8192 x 4096 14.2 / 13.2 / 13.9, 12288 x 4096 19.3 / 18.5 /
// 19.4, 8192 x 8192 28.8 / 27.1 / 24.0, 12288 x 8192 39.4 / 38.5 / 34.1; 8 rows, 32000 x 2048 26.3 / 25.0 / 24.7; in 32 bits, 32000 x 1024 26.2 / 24.5 / 26.5, 12288 x 1152 11.3 / 12.1 /
// 13.8. As they were: 5152 x 2048 6.5 (half tiles 6.4), 8192 x 3072 10.0 (10.3).
SkinnyWide skinny_wide(int M, long tiles, int K, bool f32, bool normed) {
  if (M > 8 || K < 2048) return {0, false};
  const bool apart = (K & (K - 1)) == 0 && K % 8192 != 4096;
  if (M <= 4 && !f32 && !normed && apart && tiles > 352) return {K > 4096 ? 3 : 2, true};
  return {K % 2048 == 0 ? (tiles > 384 ? 3 : 0) : !f32 && K >= 2560 && tiles > 512 ? 3 : 0, false};
}

double skinny_time(int M, long cols, int k, bool glu, bool f32, int parts) {
  const int K = f32 ? 2 * k : k;
  const double out = (double)M * (glu ? cols / 2 : cols) * (f32 ? 4 : 2);
  const long tiles = (cols + 15) / 16 * parts;
  // (not of two rounds of 56 columns: what this time is compared with for such sizes is an estimate of the vendor's that is up to a fifth too long: 40 rows,
  // 25600 x 3072, vendor 32.5 us, ours 37.7, estimates 40.7 and, with 56 columns, 38.0; 24 rows 30.8 and 32.8; but 48 rows 47.1 and 39.1)
  const int own = !glu && !f32 && parts == 1 && cols <= 1280 * 16 ? skinny_cols(M, cols, K) : 0;
  const int per = glu ? 32 : own > 0 ? own : skinny_half(M, tiles, K / parts) ? 8 : 16 * skinny_tiles(M, tiles, K / parts);
  return skinny_time_of(M, cols, K, per, parts, f32, out);
}

double mingru_product_time(int M, int width, int k, bool f32) {   // a workgroup's three tiles (mingru.hip)
  return skinny_time_of(M, 3L * width, f32 ? 2 * k : k, 48, 1, f32, (double)M * width * (f32 ? 4 : 2));
}

bool launch_skinny_linear(void* out, bool out_f32, long out_ld, long out_bs, long out_zs, int parts, const void* x, long x_ld, long x_bs,
                          const void* w, const void* bias, bool f32, int batch, int M, int N, int K, int act, int act_from, float c0, float c1,
                          hipStream_t s) {
  if (batch <= 0 || M <= 0 || N <= 0) return true;
  if (f32) { x_ld *= 2; x_bs *= 2; K *= 2; }   // in halves
#define HS_SK(XG, NT, DEPTH, ...)   launch_one<XG, NT, DEPTH, __VA_ARGS__>(out, out_f32, out_ld, out_bs, out_zs, parts, x, x_ld, x_bs, w, bias, f32, batch, M, N, K, act, act_from, c0, c1, s)
  const int xg = (M + 7) / 8;
  if (act == 3 || act == 4)
    return xg <= 1 ? HS_SK(1, 2, 1, true) : xg <= 2 ? HS_SK(2, 2, 1, true) : xg <= 4 ? HS_SK(4, 2, 1, true)
         : xg <= 6 ? HS_SK(6, 2, 1, true) : HS_SK(8, 2, 1, true);
  const long tiles = ((long)N * batch + 15) / 16 * parts;
  if (skinny_half(M, tiles, K / parts)) {
    // 32 bits, whose products of a piece take longer than its copies, have what whole tiles have: two for up to 16 rows, up to 24 where the weights are
    // 12 MB, else one. With two or three / so (whole tiles), us: 64 columns of k 4096, one row 8.2 / 7.7 (7.8), 64 rows 20.3 / 19.2 (19.4); 16 columns
    // of k 8192, 20 rows 20.6 / 18.7 (19.0). 20 rows of 2048 columns of k 3072 10.4 with two, 11.0 with one.
    if (xg <= 1) return K / parts > 4096 ? HS_SK(1, 1, 3, false, true, 2) : HS_SK(1, 1, 2, false, true);
    if (xg == 3) return tiles * K / parts >= 393216 ? HS_SK(3, 1, 2, false, true) : HS_SK(3, 1, 2, false, true, 1);
    return xg <= 2 ? HS_SK(2, 1, 2, false, true) : xg <= 4 ? HS_SK(4, 1, 2, false, true, 1) : xg <= 6 ? HS_SK(6, 1, 2, false, true, 1)
         : HS_SK(8, 1, 2, false, true, 1);
  }
  if (const int cols = batch == 1 && parts == 1 && !f32 ? skinny_cols(M, N, K) : 0) {
#define HS_S16(XG, NT, HALF) launch_16<XG, NT, 1, HALF>(out, out_f32, out_ld, x, x_ld, w, bias, M, N, K, act, act_from, c0, c1, s)
#define HS_SG(NT, HALF) (xg <= 2 ? HS_S16(2, NT, HALF) : xg <= 4 ? HS_S16(4, NT, HALF) : HS_S16(6, NT, HALF))
    return cols == 24 ? HS_SG(2, true) : cols == 40 ? HS_SG(3, true) : cols == 48 ? HS_SG(3, false) : HS_SG(4, true);
#undef HS_SG
#undef HS_S16
  }
  if (const auto wide = batch == 1 && parts == 1 ? skinny_wide(M, tiles, K, f32, false) : SkinnyWide{}; wide.ahead > 0)
    return !wide.half ? HS_SK(1, 1, 3, false) : wide.ahead > 2 ? HS_SK(1, 1, 3, false, true, 2) : HS_SK(1, 1, 2, false, true);
  const int nt = skinny_tiles(M, tiles, K / parts);
  // One piece ahead: two are faster (up to 40 %) where a wave waits for its few copies, up to 16 rows and more than a piece per wave (more than
  // two where a compute unit holds several workgroups: 12288 x 1024, 16 rows 9 % slower; 3072 x 1024, one row 4 % faster), and slower
  // where they leave room for fewer workgroups (33 - 64 rows, 16384 x 256: 19 -> 13 us; 32 heads of 512 x 128, one row 4.1 -> 3.4).
  if (nt == 4) return xg <= 4 ? HS_SK(4, 4, 1, false) : xg <= 6 ? HS_SK(6, 4, 1, false) : HS_SK(8, 4, 1, false);
  if (nt == 2) return xg <= 2 ? HS_SK(2, 2, 1, false) : xg <= 4 ? HS_SK(4, 2, 1, false) : xg <= 6 ? HS_SK(6, 2, 1, false) : HS_SK(8, 2, 1, false);
  const bool ahead = xg <= 2 && K / parts > (tiles <= 256 ? 512 : 1024) && !(xg == 1 && tiles > 256 && tiles <= 512);
  if (ahead) return xg <= 1 ? HS_SK(1, 1, 2, false) : HS_SK(2, 1, 2, false);
  return xg <= 1 ? HS_SK(1, 1, 1, false) : xg <= 2 ? HS_SK(2, 1, 1, false) : xg <= 3 ? HS_SK(3, 1, 1, false)
       : xg <= 4 ? HS_SK(4, 1, 1, false) : xg <= 6 ? HS_SK(6, 1, 1, false) : HS_SK(8, 1, 1, false);
#undef HS_SK
}

// The products of rows without their norm's factor (kNormed), K in halves.
static bool launch_normed(void* out, bool out_f32, const SkinnyNorm& norm, const void* x, long x_ld, const void* w, const void* bias,
                          bool f32, int M, int N, int K, int act, int act_from, float c0, float c1, hipStream_t s) {
  const bool glu = act == 3 || act == 4;
  const long No = glu ? N / 2 : N;
#define HS_SN(XG, NT, DEPTH, GLU, TO, F32, HALF)                                                                                              \
  launch_kernel<XG, NT, DEPTH, GLU, TO, F32, kNormed, HALF>(dim3((No + (GLU ? 16 : 16 * NT - 8 * HALF) - 1) / (GLU ? 16 : 16 * NT - 8 * HALF)), out, No, \
                                                            0, 0, x, x_ld, 0, w, bias, M, N, K, act, act_from, c0, c1, s, norm)
#define HS_SX(NT, D, GLU, TO, F32) \
  (M <= 8 ? HS_SN(1, NT, D, GLU, TO, F32, false) : M <= 16 ? HS_SN(2, NT, D, GLU, TO, F32, false) : HS_SN(4, NT, F32 ? 1 : D, GLU, TO, F32, false))
#define HS_SH(TO, F32)                                                                                                              \
  (M <= 8 ? K > 4096 ? HS_SN(1, 1, 3, false, TO, F32, true) : HS_SN(1, 1, 2, false, TO, F32, true)                                  \
          : M <= 16 ? HS_SN(2, 1, 2, false, TO, F32, true) : HS_SN(4, 1, 2, false, TO, F32, true))
#define HS_ST(NT, D, GLU) (f32 ? HS_SX(NT, D, GLU, float, true) : out_f32 ? HS_SX(NT, D, GLU, float, false) : HS_SX(NT, D, GLU, unsigned short, false))
#define HS_S4() \
  (f32 ? HS_SN(4, 4, 1, false, float, true, false) : out_f32 ? HS_SN(4, 4, 1, false, float, false, false) : HS_SN(4, 4, 1, false, unsigned short, false, false))
  if (glu) return HS_ST(2, 1, true);
  if (skinny_half(M, (N + 15) / 16, K)) return f32 ? HS_SH(float, true) : out_f32 ? HS_SH(float, false) : HS_SH(unsigned short, false);
  if (const int cols = f32 ? 0 : skinny_cols(M, N, K)) {
#define HS_SG(NT, HALF, TO) (M <= 16 ? HS_SN(2, NT, 1, false, TO, false, HALF) : HS_SN(4, NT, 1, false, TO, false, HALF))
#define HS_SO(NT, HALF) (out_f32 ? HS_SG(NT, HALF, float) : HS_SG(NT, HALF, unsigned short))
    return cols == 24 ? HS_SO(2, true) : cols == 40 ? HS_SO(3, true) : cols == 48 ? HS_SO(3, false) : HS_SO(4, true);
#undef HS_SO
#undef HS_SG
  }
  if (skinny_wide(M, (N + 15) / 16, K, f32, true).ahead == 3)
    return f32 ? HS_SN(1, 1, 3, false, float, true, false) : out_f32 ? HS_SN(1, 1, 3, false, float, false, false)
         : HS_SN(1, 1, 3, false, unsigned short, false, false);
  // Pieces ahead for one tile: as run_update has them.
  const int nt = skinny_tiles(M, (N + 15) / 16, K);   // 4 above 16 rows alone
  return nt == 4 ? HS_S4() : nt == 2 ? HS_ST(2, 1, false) : HS_ST(1, 2, false);
#undef HS_S4
#undef HS_SH
#undef HS_ST
#undef HS_SX
#undef HS_SN
}

namespace {

// A residual update's launch: rows of the operands' type.
struct UpdateLaunch {
  void* out;
  const SkinnyNorm& norm;
  const void *x, *w, *bias;
  long x_ld;
  int M, N, K;
  hipStream_t s;
  template <int XG, int NT, int DEPTH, bool F32, bool HALF> bool run() const {
    constexpr int per = 16 * NT - 8 * HALF;
    return launch_kernel<XG, NT, DEPTH, false, std::conditional_t<F32, float, unsigned short>, F32, kUpdate, HALF>(
        dim3((N + per - 1) / per), out, N, 0, 0, x, x_ld, 0, w, bias, M, N, K, -1, 0, 0.f, 0.f, s, norm);
  }
};

}  // namespace

bool launch_skinny_linear_normed(void* out, bool out_f32, const SkinnyNorm& norm, const void* x, long x_ld, const void* w, const void* bias,
                                 bool f32, int M, int N, int K, int act, int act_from, float c0, float c1, hipStream_t s) {
  if (M <= 0 || N <= 0) return true;
  if (f32) { x_ld *= 2; K *= 2; }   // in halves
  if (norm.residual == nullptr) return launch_normed(out, out_f32, norm, x, x_ld, w, bias, f32, M, N, K, act, act_from, c0, c1, s);
  const UpdateLaunch l{out, norm, x, w, bias, x_ld, M, N, K, s};
  return f32 ? run_update<true>(l, M, N, K, norm.blocks) : run_update<false>(l, M, N, K, norm.blocks);
}

}  // namespace hipserve

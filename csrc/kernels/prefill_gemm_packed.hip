// Prefill GEMM over the decode kernels' packed weight layout (one weight layout for prefill and
// decode, hand-written MFMA on the prefill hot path):
//
//   C[M, N] = X[M, K] . W[N, K]^T      bf16 in, fp32 accumulate, epilogue fused
//
// W is read from pack_decode_weight's copy (decode_gemm.hip),
// [ceil(N/128)][K/256][8 row groups][8 k-slots][64 lanes][8 bf16]: every 1 KiB
// (row group, k-slot) piece is exactly the first operand of one
// v_mfma_f32_16x16x32_bf16 for a wave (lane l: row 16 rg + (l & 15), k 32 s + 8 (l >> 4)).
// Weight fragments therefore go global -> VGPR with ONE coalesced buffer_load_dwordx4
// each and never touch LDS. Only X is staged through LDS. Per 32-deep K step a wave issues
// 8 LDS fragment reads + XP/2 staging writes, against 16 reads (+ 8 writes) when both
// operands are staged — LDS issue was what held the previous kernels at ~55 % MFMA
// busy (profiles/r3_pgemm_pmc.md).
//
// Geometry: 256 threads = 4 waves, one per SIMD (512 registers each), every wave a
// 128 (m) x 128 (n) output block = ONE packed weight tile: 64 accumulator tiles
// acc[rg][i] (rg: 16-row weight group, i: 16-row X group) = 256 fp32 per lane.
// WM x WN waves per workgroup: WM = 1 -> 128 x 512 (X staged once for four weight
// tiles), WM = 2 -> 256 x 256 (two waves stream the same weight tile, the second read
// is an L1 / L2 hit).
//
// Pipeline, per 64-deep K stage st (two 32-deep slots, 64 MFMAs per wave each):
//   slot 2st   : MFMA(wa, xa) row group by row group; after a group's 8 MFMAs its
//                weight register is reloaded with slot 2st + 2; the X fragments of slot
//                2st + 1 (xb) are read from LDS stage st; stage st + 1 (registers,
//                loaded two slots ago) is written to the other LDS buffer and stage
//                st + 2 is loaded from global; ONE barrier closes the slot.
//   slot 2st+1 : MFMA(wb, xb); wb reloaded with slot 2st + 3; xa <- LDS stage st + 1.
// Weight and X global loads are two slots (~2,000 MFMA cycles) ahead of their use. Loads
// past the end re-read the last slot / stage (clamped offsets: no branches in the loop,
// so the compiler's vmcnt waits stay exact). Rows past M read as zero (buffer range).
//
// Epilogues (lane holds C[m][n .. n+3], m = m0 + 128 wm + 16 i + (l & 15),
// n = 128 t + 16 rg + 4 (l >> 4)):
//   PW_EPI_STORE  C = bf16(acc) (+ bias[n])
//   PW_EPI_ADD    C (the residual, in place) = bf16(bf16(acc) + C)
//   PW_EPI_GLU    W packed with glu=true (each tile: 64 gate rows then their 64 up
//                 rows): gate rg and up rg + 4 sit in the same lane, so
//                 act[m, 64 t + 16 rg + 4 (l >> 4) + j] = silu(gate) * up in registers
//   PW_EPI_GEGLU  as GLU with tanh-GELU (Gemma)
//   PW_EPI_RELU2  C = bf16(max(acc, 0)^2): the table-routed experts' squared ReLU
//   PW_EPI_CGLU   as GLU with the clamped gate g sigmoid(1.702 g) (u + 1) and a scale per gathered row
#include "hipserve/common.h"
#include "hipserve/kernels.h"

#include <algorithm>

namespace hipserve {

constexpr int PW_T = 256;

// Persistent tile walk: G workgroups (one per CU), workgroup b takes tiles
// L = it * G + r (r = b remapped so an XCD's workgroups hold consecutive r), and a
// logical tile L -> (tm, tn) walks groups of PW_GM m-tiles n-major: the ~32 workgroups an
// XCD runs at once cover 8 m-tiles x 4 n-tiles and share both operands in its L2.
constexpr int PW_GM = kTileGroup;
HS_DEVICE void pw_tile(int L, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int grp = L / (PW_GM * tiles_n), first = grp * PW_GM;
  const int gsz = min(PW_GM, tiles_m - first);
  const int r = L - first * tiles_n;
  tm = first + r % gsz;
  tn = r / gsz;
}

// The m-tile that is taken tm-th: its place, its expert, its rows. One load either way: it stands before every tile's first one.
// readfirstlane: a load through a generic pointer counts as divergent, which put the weight descriptor in VGPRs and wrapped every weight load of
// the main loop in a waterfall loop (197 VALU instructions per loop body vs 0)
struct PwPlace { int place, expert, rows; };
HS_DEVICE PwPlace pw_place(const PwGroup& grp, int tm, int tile_rows) {
  const int* from = grp.order != nullptr ? grp.order : grp.tile_expert;
  const int v = __builtin_amdgcn_readfirstlane(from[tm]);
  if (grp.order == nullptr) return {tm, v, tile_rows};
  return {v >> 16, v >> 8 & 255, (v & 255) + 1};
}

// Whether none of the last `left` tiles has more than 64 rows. Their m-tiles are those of the group that the first of them lies in, without the ones whose last
// column of tiles is taken before, and all behind it; a lane asks for each.
HS_DEVICE bool pw_rest_short(int left, int tiles_m, int tiles_n, const PwGroup& grp) {
  const int whole = tiles_m * tiles_n - left, first = whole / (PW_GM * tiles_n) * PW_GM;
  const int from = first + max(whole - first * tiles_n - (tiles_n - 1) * min(PW_GM, tiles_m - first), 0);
  for (int tm = from; tm < tiles_m; tm += 64) {
    const int at = tm + (int)(threadIdx.x & 63);
    if (__ballot(at < tiles_m && (grp.order[min(at, tiles_m - 1)] & 255) >= 64) != 0) return false;
  }
  return true;
}

// What whole rounds of `ncu` tiles leave over, and how it is taken: as one more round (24 us per 1024 of K), by quarters (pw_tail, 9 + 12.5 us per 1024) or by
// columns (pw_few: each round of theirs 3 us and, per 1024, 3 us for up to 32 rows, 5 for 64, 8 for 128, beside the latency of the first). In an order that has
// the tiles of the fewest rows last: one round of columns or two always, three if all are short or K is too short for quarters. us of a round / quarters /
// columns, two rounds: 16 experts of 2048 x 1024, 24 tiles of up to 59 rows 69 / 58 / 49, 8 of 4096 x 2048, 32 of up to 66 123 / 93 / 88, 16 of 1536 x 3072, 32 of
// up to 126 176 / 127 / 125; three: 32 of 1536 x 1536, 38 of up to 63 100 / 77 / 69, 8 of 2048 x 4096, 36 of up to 126 (as they lie) 184 / 145 / 154. 131 such
// sizes: this takes 1.2 % longer than the best of these and both orders, a choice by the rows of the first of the tiles 2.9 %.
enum PwRest { kRestRound, kRestQuarters, kRestColumns };
HS_DEVICE PwRest pw_rest(int left, int tiles_m, int tiles_n, int ncu, int K, const PwGroup& grp) {
  if (left == 0) return kRestRound;
  const int rounds = (16 * left + ncu - 1) / ncu;
  const bool ordered = grp.order != nullptr;
  if (rounds <= 1 || (rounds == 2 && (ordered || K < 1536))) return kRestColumns;
  if (rounds == 3 && ordered && (K < 1536 || pw_rest_short(left, tiles_m, tiles_n, grp))) return kRestColumns;
  return 4 * left <= ncu && K >= 1536 ? kRestQuarters : kRestRound;
}

HS_DEVICE void pw_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// MFMA on an AGPR accumulator as inline asm: with the builtin, hipcc moved the 256
// accumulators between AGPRs inside the loop (about 200 v_accvgpr moves
// per 128 MFMAs). asm MFMAs are invisible to the hazard recognizer: the epilogue covers the
// MFMA -> VALU read of the accumulators by hand.
HS_DEVICE void pw_mfma(f32x4& acc, const u32x4& w, const u32x4& x) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(w), "v"(x));
}

// per-tile operand streams of one wave: its weight tile and the workgroup's X rows
struct PwTile {
  __amdgpu_buffer_rsrc_t w, x;
  int m0, t;
  int xo[8];  // kGather: this thread's byte offsets of its X rows (row p * 32 + (tid >> 3))
};

template <int WM, bool kGroup, bool kGather = false>
HS_DEVICE PwTile pw_make(int L, int tiles_m, int tiles_n, int wn, const unsigned short* X, long ldx,
                         const unsigned short* Wp, int M, int ntiles, int KS, const PwGroup& grp) {
  constexpr int WN = 4 / WM, BM = 128 * WM;
  int tm, tn;
  pw_tile(L, tiles_m, tiles_n, tm, tn);
  PwTile T;
  if constexpr (kGroup) {
    const PwPlace p = pw_place(grp, tm, BM);
    tm = p.place;
    Wp += (long)p.expert * grp.estride;
  }
  T.m0 = tm * BM;
  T.t = tn * WN + wn;
  const int tl = min(T.t, ntiles - 1);  // waves past the last weight tile compute a copy, store nothing
  T.w = __builtin_amdgcn_make_buffer_rsrc((void*)(Wp + (long)tl * KS * 32768), 0, KS * 65536, 0x00020000);
  if constexpr (kGather) {  // token rows through the slot table; padding slots read past the end = zero
    const int bytes = (int)((long)grp.x_rows * ldx * 2);
    T.x = __builtin_amdgcn_make_buffer_rsrc((void*)X, 0, bytes, 0x00020000);
    const int tid = threadIdx.x;
#pragma unroll
    for (int p = 0; p < BM / 32; ++p) {
      const int row = T.m0 + p * 32 + (tid >> 3);
      const int s = row < M ? grp.gather_slots[row] : -1;
      T.xo[p] = (s >= 0 ? (s / grp.gather_k) * (int)ldx * 2 : bytes) + (tid & 7) * 16;
    }
  } else {
    // rows >= M fall outside the buffer range and read as zero
    T.x = __builtin_amdgcn_make_buffer_rsrc((void*)(X + (long)T.m0 * ldx), 0,
                                            (int)((long)min(BM, M - T.m0) * ldx * 2), 0x00020000);
  }
  return T;
}

// Stores a wave's 128 x 128 block, weight tile t: this lane's columns 16 rg + 4 fq .. + 3 of rows mb + 16 i. own >= 0: the row groups
// own and own + 4 alone (a gate and its up projection lie four groups apart).
template <int EPI, int NI = 8, int STEP = 16>   // rows mb + STEP * i, i < NI
HS_DEVICE void pw_epilogue(f32x4 (&acc)[8][NI], int own, int t, int mb, int fq, int ntiles, unsigned short* __restrict__ C, long ldc,
                           int M, int N, const unsigned short* __restrict__ bias, const PwGroup& grp) {
  if (t >= ntiles) return;
  if constexpr (EPI == PW_EPI_GLU || EPI == PW_EPI_GEGLU || EPI == PW_EPI_CGLU) {
    const int I = N >> 1;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int m = mb + STEP * i;
      if (m >= M) continue;
      float rs = 1.f;
      if constexpr (EPI == PW_EPI_CGLU) {
        const int p = grp.gather_slots[m];
        if (grp.row_scale != nullptr && p >= 0) rs = grp.row_scale[p];
      }
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        if (own >= 0 && rg != own) continue;
        const int c = t * 64 + rg * 16 + 4 * fq;
        unsigned short o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if constexpr (EPI == PW_EPI_CGLU) {
            const float g = fminf(acc[rg][i][j] * rs, grp.limit);
            const float u = fminf(fmaxf(acc[rg + 4][i][j] * rs, -grp.limit), grp.limit);
            o[j] = f32_to_bf16(g / (1.f + __expf(-1.702f * g)) * (u + 1.f));
            continue;
          }
          const unsigned short g = f32_to_bf16(acc[rg][i][j]), u = f32_to_bf16(acc[rg + 4][i][j]);
          o[j] = EPI == PW_EPI_GEGLU ? gelu_mul1(g, u) : silu_mul1(g, u);
        }
        if (c < I)
          *reinterpret_cast<uint2*>(C + (long)m * ldc + c) =
              uint2{(unsigned)o[0] | ((unsigned)o[1] << 16), (unsigned)o[2] | ((unsigned)o[3] << 16)};
      }
    }
  } else {
#pragma unroll
    for (int rg = 0; rg < 8; ++rg) {
      if (own >= 0 && (rg & 3) != own) continue;
      const int n = t * 128 + rg * 16 + 4 * fq;
      if (n >= N) continue;
      float bv[4] = {0.f, 0.f, 0.f, 0.f};
      if (bias != nullptr)
#pragma unroll
        for (int j = 0; j < 4; ++j) bv[j] = n + j < N ? bf16_to_f32(bias[n + j]) : 0.f;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int m = mb + STEP * i;
        if (m >= M) continue;
        uint2* dst = reinterpret_cast<uint2*>(C + (long)m * ldc + n);
        float o[4];
        if constexpr (EPI == PW_EPI_ADD) {  // C is the residual: C = bf16(bf16(acc) + C)
          const uint2 rv = *dst;
          const unsigned short rr[4] = {(unsigned short)(rv.x & 0xffff), (unsigned short)(rv.x >> 16),
                                        (unsigned short)(rv.y & 0xffff), (unsigned short)(rv.y >> 16)};
#pragma unroll
          for (int j = 0; j < 4; ++j) o[j] = bf16_to_f32(f32_to_bf16(acc[rg][i][j])) + bf16_to_f32(rr[j]);
        } else {  // bias added to the fp32 accumulator, one rounding
#pragma unroll
          for (int j = 0; j < 4; ++j) o[j] = acc[rg][i][j] + bv[j];
          if constexpr (EPI == PW_EPI_RELU2) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const float r = fmaxf(o[j], 0.f);
              o[j] = r * r;
            }
          }
        }
        *dst = uint2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
      }
    }
  }
}

// The tiles that whole rounds leave over (WM = 1, grouped): 272 tiles on 256 compute units took two rounds, the second on 16 of them.
// A workgroup takes one 128 x 128 weight tile of such a tile, each of its waves a quarter of K with X rows of its own in LDS (no
// barriers; loads a 64-deep stage ahead), and the waves' sums meet in LDS, in the order of K. A stage is bound by what a compute unit
// takes in (X and weights 1 : 1 instead of 1 : 4: 40 KB per us), so that a quarter costs about 9 + 12.5 us per 1024 of K where
// the round that it replaces costs 24 us per 1024, as it has the memory to itself: nothing is gained below K = 1536 (1024: 24 -> 22 us),
// and two rounds of quarters never pay; few tiles go by columns instead (pw_rest). Whole rounds alone -> with quarters, 8 experts: 1024 x 2048, 260 tiles 102 -> 80 us; 2048 x 4096, 520
// tiles 290 -> 247; 4096 x 2048, 560 tiles 160 -> 141. The quarters follow in the launch of the whole rounds: one of its own, which has to come
// whatever the device's counts are, cost 2 - 3 us of products that leave nothing over (1024 x 2048, 400 tiles: 114, 117 with it, 114 now).
constexpr int PW_TAIL_LDS = 4 * 2 * 128 * 128;   // [wave][2][128 rows of 128 bytes], then the sums [owner][other][8 KB]
template <int EPI, bool kGather>
HS_DEVICE void pw_tail(unsigned char* lds, int r, const unsigned short* __restrict__ X, long ldx, const unsigned short* __restrict__ Wp,
                       unsigned short* __restrict__ C, long ldc, int M, int N, int K, int tiles_m, int tiles_n, const PwGroup& grp,
                       int whole) {
  constexpr int BUF = 128 * 128, XP = 16;   // a wave's stage: 128 rows of 128 bytes, 8 rows a load
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ntiles = (N + 127) >> 7, KS = K >> 8;
  const int units = 4 * (tiles_m * tiles_n - whole);
  const int nst = K >> 8, q0 = wave * 2 * nst;   // the wave's stages, its first 32-deep slot
  const int fr = lane & 15, fq = lane >> 4, sw = (fr >> 1) & 7;
  const int foff = wave * 2 * BUF + fr * 128;
  const int ch[2] = {(fq ^ sw) * 16, ((4 + fq) ^ sw) * 16};
  // staging: lane -> rows 8 p + lane / 8, 16-byte chunk c of row r at chunk c ^ ((r >> 1) & 7): r / 2 % 8 = 4 (p % 2) + lane / 16
  const int xd = wave * 2 * BUF + (lane >> 3) * 128;
  const int xdo[2] = {xd + (((lane & 7) ^ (lane >> 4)) * 16), xd + (((lane & 7) ^ (4 + (lane >> 4))) * 16)};
  for (int u = r; u < units; u += gridDim.x) {
    int tm, tn;
    pw_tile(whole + (u >> 2), tiles_m, tiles_n, tm, tn);
    const PwPlace p = pw_place(grp, tm, 128);
    const int m0 = p.place * 128, t = 4 * tn + (u & 3);
    if (t >= ntiles) continue;
    const unsigned short* wp = Wp + (long)p.expert * grp.estride + (long)t * KS * 32768;
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void*)wp, 0, KS * 65536, 0x00020000);
    // rows that do not exist lie past the buffer and read as zero (pw_make)
    const int bytes = kGather ? (int)((long)grp.x_rows * ldx * 2) : (int)((long)min(128, M - m0) * ldx * 2);
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)(kGather ? X : X + (long)m0 * ldx), 0, bytes, 0x00020000);
    int xo[XP];
#pragma unroll
    for (int p = 0; p < XP; ++p) {
      const int r = 8 * p + (lane >> 3);
      if constexpr (kGather) {
        const int s = m0 + r < M ? grp.gather_slots[m0 + r] : -1;
        xo[p] = (s >= 0 ? (s / grp.gather_k) * (int)ldx * 2 : bytes) + (lane & 7) * 16;
      } else {
        xo[p] = r * (int)ldx * 2 + (lane & 7) * 16;
      }
    }
    u32x4 xst[XP], w[2][8], xa[8], xb[8];
    f32x4 acc[8][8];
    auto wload = [&](int q, int rg) -> u32x4 {   // slot q of the wave's
      q += q0;
      return __builtin_amdgcn_raw_buffer_load_b128(wr, lane * 16, (q >> 3) * 65536 + rg * 8192 + (q & 7) * 1024, 0);
    };
    auto xload = [&](int st) {
#pragma unroll
      for (int p = 0; p < XP; ++p) xst[p] = __builtin_amdgcn_raw_buffer_load_b128(xr, xo[p], q0 * 64 + st * 128, 0);
    };
    auto xstore = [&](int buf) {
#pragma unroll
      for (int p = 0; p < XP; ++p) *reinterpret_cast<u32x4*>(lds + buf * BUF + p * 1024 + xdo[p & 1]) = xst[p];
    };
    auto xfrag = [&](int buf, int h, int i) -> u32x4 {
      return *reinterpret_cast<const u32x4*>(lds + buf * BUF + foff + i * 2048 + ch[h]);
    };
    xload(0);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int rg = 0; rg < 8; ++rg) w[j][rg] = wload(j, rg);
#pragma unroll
    for (int rg = 0; rg < 8; ++rg)
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[rg][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    xstore(0);
    xload(min(1, nst - 1));
#pragma unroll
    for (int i = 0; i < 8; ++i) xa[i] = xfrag(0, 0, i);
    for (int st = 0; st < nst; ++st) {
      const int buf = st & 1, nq = 2 * min(st + 1, nst - 1);
#pragma unroll
      for (int rg = 0; rg < 8; ++rg) {
#pragma unroll
        for (int i = 0; i < 8; ++i) pw_mfma(acc[rg][i], w[0][rg], xa[i]);
        w[0][rg] = wload(nq, rg);
        xb[rg] = xfrag(buf, 1, rg);
        if (rg == 2) xstore(buf ^ 1);
        if (rg == 3) xload(min(st + 2, nst - 1));
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int rg = 0; rg < 8; ++rg) {
#pragma unroll
        for (int i = 0; i < 8; ++i) pw_mfma(acc[rg][i], w[1][rg], xb[i]);
        w[1][rg] = wload(nq + 1, rg);
        xa[rg] = xfrag(buf ^ 1, 0, rg);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");  // last MFMA -> VALU reads
    // wave w ends with the row groups w and w + 4: the others' parts through LDS, half of the rows at a time, added in the order of K
    f32x4* sums = reinterpret_cast<f32x4*>(lds);   // [owner][wave][2][4][64 lanes]
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      __syncthreads();
#pragma unroll
      for (int rg = 0; rg < 8; ++rg)
#pragma unroll
        for (int i = 0; i < 4; ++i) sums[((((rg & 3) * 4 + wave) * 2 + (rg >> 2)) * 4 + i) * 64 + lane] = acc[rg][4 * half + i];
      __syncthreads();
#pragma unroll
      for (int rg = 0; rg < 8; ++rg) {
        if ((rg & 3) != wave) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          f32x4 a = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int o = 0; o < 4; ++o) a += sums[(((wave * 4 + o) * 2 + (rg >> 2)) * 4 + i) * 64 + lane];
          acc[rg][4 * half + i] = a;
        }
      }
    }
    pw_epilogue<EPI>(acc, wave, t, m0 + fr, fq, ntiles, C, ldc, M, N, nullptr, grp);
    __syncthreads();   // the sums are read before the next unit's rows come
  }
}

// The same by columns: a workgroup takes 32 columns (row groups own and own + 4 of a weight tile), its waves a quarter of K each with rows of their own in LDS,
// and of the rows the 16 RI that there are. Four times as many workgroups as by quarters, each of which takes in 8 KB per 64-deep stage and 32 rows (40 of
// 128) for 128; what bounds it is the latency of a unit's first loads (its place, its slots, its rows) and then the intake, some 40 KB per us. With
// the order that leaves the tiles of few rows for last (order_tiles), one round of columns is 11 - 15 us, of quarters 25 - 35, a whole round 24 per 1024
// of K. Up and down of 16384 pairs, whole rounds and quarters -> with these: 16 experts of 1024 x 2048 84.7 -> 76.0, 89.8 -> 77.2 us, 8 of 2048 x 4096 243 ->
// 222, 256 -> 248; 12000 pairs, down, 190 -> 181; 2048 pairs of 512 x 1024 31 -> 22.
template <int EPI, bool kGather, int RI>
HS_DEVICE void pw_few_unit(unsigned char* lds, const unsigned short* __restrict__ X, long ldx, const unsigned short* __restrict__ wp,
                           unsigned short* __restrict__ C, long ldc, int M, int N, int K, int t, int own, int m0, int rows, const PwGroup& grp) {
  constexpr int BUF = 128 * 128, XP = 2 * RI, PD = RI == 2 ? 4 : 2;   // PD: stages in flight
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ntiles = (N + 127) >> 7, KS = K >> 8;
  const int nst = K >> 8, q0 = wave * 2 * nst;
  const int fr = lane & 15, fq = lane >> 4, sw = (fr >> 1) & 7;
  const int foff = wave * 2 * BUF + fr * 128;
  const int ch[2] = {(fq ^ sw) * 16, ((4 + fq) ^ sw) * 16};
  const int xd = wave * 2 * BUF + (lane >> 3) * 128;
  const int xdo[2] = {xd + (((lane & 7) ^ (lane >> 4)) * 16), xd + (((lane & 7) ^ (4 + (lane >> 4))) * 16)};
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void*)wp, 0, KS * 65536, 0x00020000);
  // rows that do not exist lie past the buffer and read as zero (pw_make)
  const int bytes = kGather ? (int)((long)grp.x_rows * ldx * 2) : (int)((long)min(rows, M - m0) * ldx * 2);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)(kGather ? X : X + (long)m0 * ldx), 0, bytes, 0x00020000);
  int xo[XP];
#pragma unroll
  for (int p = 0; p < XP; ++p) {
    const int r = 8 * p + (lane >> 3);
    if constexpr (kGather) {
      const int s = m0 + r < M ? grp.gather_slots[m0 + r] : -1;
      xo[p] = (s >= 0 ? (s / grp.gather_k) * (int)ldx * 2 : bytes) + (lane & 7) * 16;
    } else {
      xo[p] = r * (int)ldx * 2 + (lane & 7) * 16;
    }
  }
  u32x4 xst[PD][XP], w[PD][2][2];   // [stage][half][row group]
  f32x4 acc[2][RI];
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int i = 0; i < RI; ++i) acc[g][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto wload = [&](int st, u32x4 (&to)[2][2]) {
    const int q = q0 + 2 * st;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int g = 0; g < 2; ++g)
        to[h][g] = __builtin_amdgcn_raw_buffer_load_b128(wr, lane * 16, ((q + h) >> 3) * 65536 + (own + 4 * g) * 8192 + ((q + h) & 7) * 1024, 0);
  };
  auto xload = [&](int st, u32x4 (&to)[XP]) {
#pragma unroll
    for (int p = 0; p < XP; ++p) to[p] = __builtin_amdgcn_raw_buffer_load_b128(xr, xo[p], q0 * 64 + st * 128, 0);
  };
#pragma unroll
  for (int j = 0; j < PD; ++j) {
    xload(min(j, nst - 1), xst[j]);
    wload(min(j, nst - 1), w[j]);
  }
  for (int s0 = 0; s0 < nst; s0 += PD) {
#pragma unroll
    for (int j = 0; j < PD; ++j) {
      if (s0 + j >= nst) break;
      const int next = min(s0 + j + PD, nst - 1);
#pragma unroll
      for (int p = 0; p < XP; ++p) *reinterpret_cast<u32x4*>(lds + (j & 1) * BUF + p * 1024 + xdo[p & 1]) = xst[j][p];
      xload(next, xst[j]);
      u32x4 x[2][RI];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < RI; ++i) x[h][i] = *reinterpret_cast<const u32x4*>(lds + (j & 1) * BUF + foff + i * 2048 + ch[h]);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
          for (int i = 0; i < RI; ++i)
            acc[g][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[j][h][g]), __builtin_bit_cast(bf16x8, x[h][i]), acc[g][i], 0, 0, 0);
      wload(next, w[j]);
    }
  }
  // wave v ends with the row groups of X v, v + 4, ..: the others' parts through LDS, added in the order of K
  f32x4* sums = reinterpret_cast<f32x4*>(lds);   // [wave][2][RI][64 lanes]
  __syncthreads();
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int i = 0; i < RI; ++i) sums[((wave * 2 + g) * RI + i) * 64 + lane] = acc[g][i];
  __syncthreads();
  constexpr int NI = (RI + 3) / 4;
  f32x4 all[8][NI];
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      f32x4 a = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int o = 0; o < 4; ++o) a += sums[((o * 2 + g) * RI + min(wave + 4 * i, RI - 1)) * 64 + lane];
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) all[4 * g + rg][i] = a;
    }
  if (wave < RI) pw_epilogue<EPI, NI, 64>(all, own, t, m0 + 16 * wave + fr, fq, ntiles, C, ldc, M, N, nullptr, grp);
  __syncthreads();   // the sums are read before the next unit's rows come
}

template <int EPI, bool kGather>
HS_DEVICE void pw_few(unsigned char* lds, int r, const unsigned short* __restrict__ X, long ldx, const unsigned short* __restrict__ Wp,
                      unsigned short* __restrict__ C, long ldc, int M, int N, int K, int tiles_m, int tiles_n, const PwGroup& grp, int whole) {
  const int ntiles = (N + 127) >> 7, units = 16 * (tiles_m * tiles_n - whole);
  for (int u = r; u < units; u += gridDim.x) {
    int tm, tn;
    pw_tile(whole + (u >> 4), tiles_m, tiles_n, tm, tn);
    const PwPlace p = pw_place(grp, tm, 128);
    const int t = 4 * tn + (u >> 2 & 3);
    if (t >= ntiles) continue;
    const unsigned short* wp = Wp + (long)p.expert * grp.estride + (long)t * (K >> 8) * 32768;
#define PW_FEW(RI) pw_few_unit<EPI, kGather, RI>(lds, X, ldx, wp, C, ldc, M, N, K, t, u & 3, p.place * 128, p.rows, grp)
    if (p.rows <= 32) PW_FEW(2);
    else if (p.rows <= 64) PW_FEW(4);
    else PW_FEW(8);
#undef PW_FEW
  }
}

// The tiles r, r + G, .. < total of a workgroup.
template <int WM, int EPI, bool kGroup, int RW, bool LDLY, bool kGather>
HS_DEVICE void pw_tiles(unsigned char* lds, int r, int G, int total, const unsigned short* __restrict__ X, long ldx,
                        const unsigned short* __restrict__ Wp, unsigned short* __restrict__ C, long ldc, int M, int N, int K,
                        int tiles_m, int tiles_n, const unsigned short* __restrict__ bias, const PwGroup& grp) {
  constexpr int WN = 4 / WM, BM = 128 * WM, STAGE = BM * 128, XP = BM / 32;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave - (wave / WN) * WN;
  const int ntiles = (N + 127) >> 7;
  const int KS = K >> 8, nq = K >> 5, nst = K >> 6;
  if (r >= total) return;

  // cur: the tile whose MFMAs run; nxt: the one the loads past cur's end stream in, so
  // the pipeline runs on across the tile boundary (only the epilogue sits between)
  PwTile cur = pw_make<WM, kGroup, kGather>(r, tiles_m, tiles_n, wn, X, ldx, Wp, M, ntiles, KS, grp);
  PwTile nxt = r + G < total ? pw_make<WM, kGroup, kGather>(r + G, tiles_m, tiles_n, wn, X, ldx, Wp, M, ntiles, KS, grp) : cur;

  const int wvo = lane * 16;
  auto wload = [&](int q, int rg) -> u32x4 {  // 32-deep slot q of cur (q >= nq: of nxt), row group rg
    const bool n = q >= nq;
    q = n ? q - nq : q;
    return __builtin_amdgcn_raw_buffer_load_b128(n ? nxt.w : cur.w, wvo, (q >> 3) * 65536 + rg * 8192 + (q & 7) * 1024,
                                                 0);
  };
  // X staging: thread -> rows 32 p + (tid >> 3), 16-byte chunk tid & 7 of the 128-byte
  // (64-deep) row
  int xvo[XP];
#pragma unroll
  for (int p = 0; p < XP; ++p) xvo[p] = (p * 32 + (tid >> 3)) * (int)ldx * 2 + (tid & 7) * 16;
  // LDS image [BM rows][128 B]: 16-byte chunk c of row r at chunk c ^ ((r >> 1) & 7), which
  // spreads each ds_read_b128 lane group (rows 0-3 / 12-15 of one chunk, 4-11 of the
  // next) over all 16 slots of a 256-byte bank row; (r >> 1) & 7 is the same for rows
  // r and r + 32 p
  const int xdo = (tid >> 3) * 128 + (((tid & 7) ^ ((tid >> 4) & 7)) * 16);
  // RW weight register sets (one per 32-deep slot in flight: a set's next slot is
  // loaded right after its MFMAs, RW slots ahead) and XS = RW / 2 X staging sets (stage
  // s + 1 + XS is loaded into the set stage s + 1 was just written to LDS from)
  constexpr int XS = RW / 2;
  u32x4 xst[XS][XP];
  auto xload = [&](int st, u32x4 (&xs)[XP]) {  // 64-deep stage st of cur (st >= nst: of nxt)
    const bool n = st >= nst;
    st = n ? st - nst : st;
#pragma unroll
    for (int p = 0; p < XP; ++p)
      xs[p] = __builtin_amdgcn_raw_buffer_load_b128(n ? nxt.x : cur.x, kGather ? (n ? nxt.xo[p] : cur.xo[p]) : xvo[p],
                                                    st * 128, 0);
  };
  auto xstore = [&](int buf, const u32x4 (&xs)[XP]) {
#pragma unroll
    for (int p = 0; p < XP; ++p) *reinterpret_cast<u32x4*>(lds + buf * STAGE + p * 4096 + xdo) = xs[p];
  };
  const int fr = lane & 15, fq = lane >> 4, sw = (fr >> 1) & 7;
  const int foff = (wm * 128 + fr) * 128;
  const int ch[2] = {(fq ^ sw) * 16, ((4 + fq) ^ sw) * 16};
  auto xfrag = [&](int buf, int h, int i) -> u32x4 {
    return *reinterpret_cast<const u32x4*>(lds + buf * STAGE + foff + i * 2048 + ch[h]);
  };

  f32x4 acc[8][8];
  u32x4 w[RW][8], xa[8], xb[8];
  int wvoj[RW];
#pragma unroll
  for (int j = 0; j < RW; ++j) wvoj[j] = wvo + j * 1024;

  // prologue (first tile only): stage 0 in LDS, stages 1 .. XS in registers, weight
  // slots 0 .. RW - 1 in flight; later tiles find theirs loaded by the previous tile's
  // last slots
  xload(0, xst[0]);
  xstore(0, xst[0]);
#pragma unroll
  for (int s = 1; s <= XS; ++s) xload(s, xst[s % XS]);
#pragma unroll
  for (int j = 0; j < RW; ++j)
#pragma unroll
    for (int rg = 0; rg < 8; ++rg) w[j][rg] = wload(j, rg);
  pw_barrier();
#pragma unroll
  for (int i = 0; i < 8; ++i) xa[i] = xfrag(0, 0, i);

  // one 32-deep slot: J (compile time) = slot index inside the RW-slot loop body. The
  // weight loads of one loop body all stream the same tile (nq % RW == 0): their buffer
  // resource and K offset are chosen once per body (wrs, wk), so a load costs one scalar
  // add — per-load selects cost ~6 SALU each and delayed the next MFMA group
  auto slot = [&](auto jc, int s0, const __amdgpu_buffer_rsrc_t& wrs, int wk) {
    constexpr int J = decltype(jc)::value, H = J & 1;
    const int s = s0 + J / 2, buf = s & 1;
    constexpr int XI = (J / 2 + 1) % XS;  // staging set of stage s + 1 (s0 is a multiple of XS)
#pragma unroll
    for (int rg = 0; rg < 8; ++rg) {
#pragma unroll
      for (int i = 0; i < 8; ++i) pw_mfma(acc[rg][i], w[J][rg], H ? xb[i] : xa[i]);
      // slot J's 1 KiB offset rides in a per-slot VGPR offset: 8 scalar adds per body, not 32.
      // LDLY: reload a group's weight register one group later, so the load is not issued
      // right behind the MFMAs still reading that register
      if constexpr (LDLY) {
        if (rg > 0) w[J][rg - 1] = __builtin_amdgcn_raw_buffer_load_b128(wrs, wvoj[J], wk + (rg - 1) * 8192, 0);
        if (rg == 7) w[J][7] = __builtin_amdgcn_raw_buffer_load_b128(wrs, wvoj[J], wk + 7 * 8192, 0);
      } else {
        w[J][rg] = __builtin_amdgcn_raw_buffer_load_b128(wrs, wvoj[J], wk + rg * 8192, 0);
      }
      if constexpr (H == 0) {
        xb[rg] = xfrag(buf, 1, rg);
        if (rg == 2) xstore(buf ^ 1, xst[XI]);     // stage s + 1 (loaded XS stages ago)
        if (rg == 3) xload(s + 1 + XS, xst[XI]);
      } else {
        xa[rg] = xfrag(buf ^ 1, 0, rg);            // stage s + 1, visible since the barrier
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (H == 0) pw_barrier();  // stage s + 1 visible; every read of stage s - 1 done
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;

  for (int L = r;;) {
#pragma unroll
    for (int rg = 0; rg < 8; ++rg)
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[rg][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int q0 = 0; q0 < nq; q0 += RW) {  // nq % 8 == 0; a tile starts in LDS buffer 0
      const int s0 = q0 >> 1;
      const bool wn = q0 + RW >= nq;  // this body's weight loads stream the next tile
      const int wq = wn ? q0 + RW - nq : q0 + RW;
      const __amdgpu_buffer_rsrc_t wrs = wn ? nxt.w : cur.w;
      const int wk = (wq >> 3) * 65536 + (wq & 7) * 1024;  // (wq & 7) + J <= 7
      slot(I0(), s0, wrs, wk);
      slot(I1(), s0, wrs, wk);
      if constexpr (RW == 4) {
        slot(I2(), s0, wrs, wk);
        slot(I3(), s0, wrs, wk);
      }
    }

    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");  // last MFMA -> VALU reads
    pw_epilogue<EPI>(acc, -1, cur.t, cur.m0 + wm * 128 + fr, fq, ntiles, C, ldc, M, N, bias, grp);
    L += G;
    if (L >= total) break;
    cur = nxt;
    if (L + G < total) nxt = pw_make<WM, kGroup, kGather>(L + G, tiles_m, tiles_n, wn, X, ldx, Wp, M, ntiles, KS, grp);
  }
}

// kGroup (MoE prefill experts): X rows are expert-sorted slots in BM-row tiles
// (moe_align with tile BM, moe_gather); m-tile tm multiplies expert grp.tile_expert[tm]'s
// packed weight (Wp + e * estride) and only the first *grp.num_tiles m-tiles (the
// device-side count: no host round trip, graph-capturable) are walked. TAIL: whole rounds of
// `ncu` tiles, then what they leave over (pw_rest).
template <int WM, int EPI, bool kGroup, int RW, bool LDLY = false, bool kGather = false, bool TAIL = false>
__global__ __launch_bounds__(PW_T) __attribute__((amdgpu_waves_per_eu(1, 1))) void pgw_kernel(
    const unsigned short* __restrict__ X, long ldx, const unsigned short* __restrict__ Wp,
    unsigned short* __restrict__ C, long ldc, int M, int N, int K, int tiles_m, int tiles_n,
    const unsigned short* __restrict__ bias, PwGroup grp, int ncu) {
  static_assert(!TAIL || (WM == 1 && kGroup), "pw_tail");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[TAIL ? PW_TAIL_LDS : 2 * 128 * WM * 128];
  // TAIL: of the grid, as many as there can be whole tiles for, which the XCDs share evenly that way
  const int G = TAIL ? min((int)gridDim.x, tiles_m * tiles_n) : gridDim.x;
  if constexpr (kGroup) tiles_m = min(tiles_m, __builtin_amdgcn_readfirstlane(*grp.num_tiles));
  int total = tiles_m * tiles_n;
  [[maybe_unused]] PwRest rest = kRestRound;
  if constexpr (TAIL) {
    const int left = total % ncu;
    rest = pw_rest(left, tiles_m, tiles_n, ncu, K, grp);
    if (rest != kRestRound) total -= left;
  }
  const int r = (int)blockIdx.x < G ? xcd_remap(blockIdx.x, G) : total;
  pw_tiles<WM, EPI, kGroup, RW, LDLY, kGather>(lds, r, G, total, X, ldx, Wp, C, ldc, M, N, K, tiles_m, tiles_n, bias, grp);
  if constexpr (TAIL) {
    __syncthreads();   // the last tile's rows are read
    const int u = xcd_remap(blockIdx.x, gridDim.x);
    if (rest == kRestColumns) pw_few<EPI, kGather>(lds, u, X, ldx, Wp, C, ldc, M, N, K, tiles_m, tiles_n, grp, total);
    else if (rest == kRestQuarters) pw_tail<EPI, kGather>(lds, u, X, ldx, Wp, C, ldc, M, N, K, tiles_m, tiles_n, grp, total);
  }
}

bool launch_prefill_gemm_packed(int epi, void* C, long ldc, const void* X, long ldx, const void* Wp, int M, int N,
                                int K, const void* bias, int wm, int grid_req, hipStream_t s, const PwGroup* group,
                                int rw) {
  const PwGroup grp = group != nullptr ? *group : PwGroup{nullptr, nullptr, 0};
  const bool grouped = group != nullptr;
  const bool gather = grouped && grp.gather_slots != nullptr;
  if (grouped && (bias != nullptr || epi == PW_EPI_ADD)) return false;
  // (the gather form always runs rw = 4, PW_LAUNCH1: any rw knob value is accepted)
  if (gather && (grp.gather_k < 1 || (long)grp.x_rows * ldx * 2 >= (1L << 31) - 4096)) return false;
  if (M < 1 || N < 1 || K < 256 || K % 256 || (wm != 1 && wm != 2) || (rw != 2 && rw != 4 && rw != 5)) return false;
  const bool glu = epi == PW_EPI_GLU || epi == PW_EPI_GEGLU || epi == PW_EPI_CGLU;
  if (epi == PW_EPI_CGLU && !gather) return false;
  if (glu && (N % 128 || bias != nullptr)) return false;
  if (epi == PW_EPI_ADD && bias != nullptr) return false;
  // 32-bit buffer offsets: the weight stream of one tile and one workgroup's X rows
  if ((long)(K / 256) * 65536 >= (1L << 31) || (long)128 * wm * ldx * 2 >= (1L << 31)) return false;
  const int BM = 128 * wm, WN = 4 / wm;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = ((N + 127) / 128 + WN - 1) / WN;
  // persistent: one workgroup per CU (grid <= 0) unless the caller asks for a grid
  static int ncu = 0;
  if (ncu == 0) {
    int dev = 0;
    (void)hipGetDevice(&dev);
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || ncu < 1) ncu = 256;
  }
  const int total = tiles_m * tiles_n;
  const dim3 grid(min(total, grid_req > 0 ? grid_req : ncu));
  auto* x = static_cast<const unsigned short*>(X);
  auto* w = static_cast<const unsigned short*>(Wp);
  auto* c = static_cast<unsigned short*>(C);
  auto* b = static_cast<const unsigned short*>(bias);
#define PW_LAUNCH1(WM_, E_, RW_)                                                                               \
  do {                                                                                                         \
    if (gather)                                                                                                \
      pgw_kernel<WM_, E_, true, 4, false, true><<<grid, PW_T, 0, s>>>(x, ldx, w, c, ldc, M, N, K, tiles_m, tiles_n, b, grp, ncu); \
    else if (grouped)                                                                                          \
      pgw_kernel<WM_, E_, true, RW_><<<grid, PW_T, 0, s>>>(x, ldx, w, c, ldc, M, N, K, tiles_m, tiles_n, b, grp, ncu);  \
    else                                                                                                       \
      pgw_kernel<WM_, E_, false, RW_><<<grid, PW_T, 0, s>>>(x, ldx, w, c, ldc, M, N, K, tiles_m, tiles_n, b, grp, ncu); \
  } while (0)
#define PW_LAUNCH(WM_, E_)                                                                                   \
  do {                                                                                                       \
    if (rw == 4)                                                                                             \
      PW_LAUNCH1(WM_, E_, 4);                                                                                \
    else if (rw == 2)                                                                                        \
      PW_LAUNCH1(WM_, E_, 2);                                                                                \
    else if (grouped)                                                                                        \
      pgw_kernel<WM_, E_, true, 4, true><<<grid, PW_T, 0, s>>>(x, ldx, w, c, ldc, M, N, K, tiles_m, tiles_n, b, grp, ncu);  \
    else                                                                                                     \
      pgw_kernel<WM_, E_, false, 4, true><<<grid, PW_T, 0, s>>>(x, ldx, w, c, ldc, M, N, K, tiles_m, tiles_n, b, grp, ncu); \
  } while (0)
  if (grouped && wm == 1 && grid_req <= 0) {
    const dim3 tg(std::min(16L * total, (long)ncu));   // fewer tiles than compute units may come in parts
#define PW_TAIL(E_)                                                                                                                  \
  do {                                                                                                                               \
    if (gather) pgw_kernel<1, E_, true, 4, false, true, true><<<tg, PW_T, 0, s>>>(x, ldx, w, c, ldc, M, N, K, tiles_m, tiles_n, b, grp, ncu); \
    else if constexpr (E_ != PW_EPI_CGLU)                                                                                             \
      pgw_kernel<1, E_, true, 4, false, false, true><<<tg, PW_T, 0, s>>>(x, ldx, w, c, ldc, M, N, K, tiles_m, tiles_n, b, grp, ncu);   \
    return true;                                                                                                                     \
  } while (0)
    switch (epi) {
      case PW_EPI_STORE: PW_TAIL(PW_EPI_STORE);
      case PW_EPI_GLU: PW_TAIL(PW_EPI_GLU);
      case PW_EPI_GEGLU: PW_TAIL(PW_EPI_GEGLU);
      case PW_EPI_RELU2: PW_TAIL(PW_EPI_RELU2);
      case PW_EPI_CGLU: PW_TAIL(PW_EPI_CGLU);
      default: return false;
    }
#undef PW_TAIL
  }
  if (epi == PW_EPI_CGLU) {   // instantiated in the gather form only
    if (wm == 1)
      pgw_kernel<1, PW_EPI_CGLU, true, 4, false, true><<<grid, PW_T, 0, s>>>(x, ldx, w, c, ldc, M, N, K, tiles_m, tiles_n, b, grp, ncu);
    else
      pgw_kernel<2, PW_EPI_CGLU, true, 4, false, true><<<grid, PW_T, 0, s>>>(x, ldx, w, c, ldc, M, N, K, tiles_m, tiles_n, b, grp, ncu);
    return true;
  }
#define PW_EPIS(WM_)                                          \
  switch (epi) {                                              \
    case PW_EPI_STORE: PW_LAUNCH(WM_, PW_EPI_STORE); return true; \
    case PW_EPI_ADD: PW_LAUNCH(WM_, PW_EPI_ADD); return true;     \
    case PW_EPI_GLU: PW_LAUNCH(WM_, PW_EPI_GLU); return true;     \
    case PW_EPI_GEGLU: PW_LAUNCH(WM_, PW_EPI_GEGLU); return true; \
    case PW_EPI_RELU2: PW_LAUNCH(WM_, PW_EPI_RELU2); return true; \
    default: return false;                                    \
  }
  if (wm == 1) {
    PW_EPIS(1)
  }
  PW_EPIS(2)
#undef PW_EPIS
#undef PW_LAUNCH
#undef PW_LAUNCH1
}

}  // namespace hipserve

// Latent attention on the matrix cores for cache rows of 128, 256 or 512 latent dims and 64 rotary ones (bf16): the
// products of latent_attention_mfma.hip with the cache rows copied straight into LDS.
//
// That kernel loads a 32-key tile into registers, stores it to LDS and only then multiplies: a tile waits for its page
// lookup and for its rows (about 3 us) before 0.5 us of products, its operand reads wait one by one (no registers left),
// and the V operand of P . V is gathered from LDS two bytes at a time. Here
//   * global_load_lds brings the rows into one of four LDS buffers, a tile ahead of the scores;
//   * a buffer holds [32][latent dims] and [32][64 rotary dims]; the 16-byte chunks of a row are XOR-swizzled by the key, by
//     choosing which chunk a lane copies, so that neither the row-wise operand reads of S = K . Q^T nor the transposing
//     reads below meet in a bank, without padding;
//   * the V^T operand comes from ds_read_tr16_b64: within 16 lanes, lane l gets element l % 4 of the 8 bytes that lane
//     4 j + l / 4 addresses, j = 0 .. 3. Lane (c, g) addresses key 16 h + 4 g + c / 4, dims 4 (c % 4) .. + 3 and so
//     receives keys 16 h + 4 g + 0 .. 3 of dim c: half of an MFMA operand in the key order of P;
//   * waves 0 - 3 (one per SIMD) compute the scores and softmax of 16 rows each, waves 4 - 7 the P . V of the previous tile,
//     DV / 4 latent dims each for all 64 rows: the softmax of one tile runs beside the products of another, neither half
//     holds the other's registers (queries 72, outputs 128 per lane), and a tile costs one barrier;
//   * the queries' rotary part is rotated when the operands are loaded (its halves meet in one lane), no pass of its own.
//   * maxima are taken of the raw products, sums come from a product with ones, and the accumulators (128 per lane) are
//     rescaled only where a row's maximum grows. (Not rarer: the largest weight is 1 then, which bf16 holds exactly. A maximum that
//     follows only when a score is larger by 2^8 saves 20 us below, and the outputs' error against 64 bits grows by up to
//     a tenth, 1.81e-3 -> 1.98e-3 with their own rounding.)
// 8192 rows (4 prompts) x 16 heads, 512 + 64 dims, window 1024: 980 -> 363 us (620 TFLOP/s). Without the rescaling (341 us, 690 k
// cycles) a SIMD's matrix unit is busy 220 k cycles, the vector unit 125 k, the LDS 180 k; the rest waits for operands and at
// the one barrier per tile. Eight-way swizzles (operand rows met two to a bank) took 45 us more, scores without the next tile's
// operand reads beside them a fifth more.
// latent_dma_decode_kernel serves decode rows: a workgroup takes 16 heads of one row and a run of keys, 64 of them
// at a time; its waves split the keys for S and the latent dims for P . V. One row of 724 keys, 16 heads, with the merge: 46 -> 10 us.
#include "lds_copy.h"
#include "seq_common.h"
#include "hipserve/seq_kernels.h"

namespace hipserve {
namespace {

constexpr int kKeys = 32, kRot = 64, kPLd = 40;   // kPLd: row stride of P in elements (16-byte rows, padded)
constexpr float kLog2e = 1.44269504088896341f;

// K tile rows in LDS: [KEYS][DV] then [KEYS][64]; 16-byte chunk ch of key k sits at chunk ch ^ swizzle(k) (rotary part:
// ch ^ rot_swizzle(k), rows of 128 bytes, two fill the banks): the 16 keys of an operand use 16 different chunks of 256 bytes,
// the 8 keys of a transposing read 8 different pairs.
// (An operand's lanes are served in groups of keys 0 - 3, 12 - 15 with chunk x and 4 - 11 with chunk x ^ 1: bit 3 goes into bit 2 too.)
HS_DEVICE int swizzle(int k) { return ((k ^ (k >> 1 & 4)) & 7) << 1 | (k >> 3 & 1); }
HS_DEVICE int rot_swizzle(int k) { return k >> 1 & 7; }
template <int DV, int KEYS> struct Tile {
  static constexpr int kMain = KEYS * DV * 2, kBytes = kMain + KEYS * kRot * 2;
  static HS_DEVICE int main_at(int k, int ch) { return k * DV * 2 + ((ch ^ swizzle(k)) << 4); }
  static HS_DEVICE int rot_at(int k, int ch) { return kMain + k * kRot * 2 + ((ch ^ rot_swizzle(k)) << 4); }
  // The wave copies keys 8 w .. 8 w + 7 of the tile; `row` = element offset of key `lane` % KEYS's cache row.
  static HS_DEVICE void copy(unsigned lds, const unsigned short* cache, long row, int w, int lane) {
    constexpr int kPer = 512 / DV, kChunks = DV / 8;   // keys and 16-byte chunks of a key in one 1 KB copy
#pragma unroll
    for (int i = 0; i < 8 / kPer; ++i) {
      if constexpr (kPer == 1) {   // one key, the same for all lanes
        const int k = 8 * w + i;
        const unsigned lo = __builtin_amdgcn_readlane((int)row, k), hi = __builtin_amdgcn_readlane((int)(row >> 32), k);
        copy_1k(reinterpret_cast<const unsigned char*>(cache + (long)((unsigned long)hi << 32 | lo)), 16 * (lane ^ swizzle(k)), lds + k * DV * 2);
        continue;
      }
      const int k = 8 * w + i * kPer + lane / kChunks, ch = (lane % kChunks) ^ swizzle(k);
      const unsigned short* src = cache + __shfl(row, k, 64) + 8 * ch;
      copy_1k(src, lds + (8 * w + i * kPer) * DV * 2);
    }
    const int k = 8 * w + lane / 8, ch = (lane & 7) ^ rot_swizzle(k);
    const unsigned short* src = cache + __shfl(row, k, 64) + DV + 8 * ch;
    copy_1k(src, lds + kMain + 8 * w * kRot * 2);
  }
  // The lane's places in a tile: the swizzle touches four bits of the chunk, so four (keys) and up to eight (values)
  // offsets serve all operands, with constants added.
  static constexpr int NPW = DV / 64, JB = NPW < 8 ? NPW : 8;   // 16-dim value tiles per wave
  struct Places { int key[4], rot[2], val[JB]; };
  static HS_DEVICE Places places(int wave, int c, int g) {
    Places p;
#pragma unroll
    for (int i = 0; i < 4; ++i) p.key[i] = main_at(c, 4 * i + g);
#pragma unroll
    for (int i = 0; i < 2; ++i) p.rot[i] = rot_at(c, 4 * i + g);
#pragma unroll
    for (int j = 0; j < JB; ++j)
      p.val[j] = main_at(4 * g + (c >> 2), 2 * (wave * NPW + j) + ((c & 3) >> 1)) + 8 * (c & 1);
    return p;
  }
  // MFMA operand of 32-dim step ks of key rows k0 + c (k0 a multiple of 16): dims 32 ks + 8 g .. + 7
  static HS_DEVICE bf16x8 key_operand(const unsigned char* lds, const Places& p, int k0, int ks) {
    const int at = ks < DV / 32 ? p.key[ks & 3] + (ks >> 2) * 256 + k0 * DV * 2 : p.rot[ks & 1] + k0 * kRot * 2;
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u16x8*>(lds + at));
  }
  // MFMA operand of the wave's value tile j against keys k0 .. k0 + 31 (k0 a multiple of 32): lane (c, g) holds dim c,
  // keys k0 + 16 (e / 4) + 4 g + e % 4
  static HS_DEVICE bf16x8 value_operand(unsigned char* lds, const Places& p, int k0, int j) {
    s16x4 h[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
      h[i] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_s16x4)(lds + p.val[j] + (k0 + 16 * i) * DV * 2));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(h[0], h[1], 0, 1, 2, 3, 4, 5, 6, 7));
  }
};

// Query operands of one (token, head) row: the latent part from qc, the last 64 dims from qc too, or rotated here from
// the projection's rotary part (q_rot: its 64 numbers; entry i pairs with i + 32, angle pos * inv_freq[i]). angle(i, sn, cs): of entry i, after
// asked(), which runs behind the loads.
template <int DV, typename F, typename G>
HS_DEVICE void load_query(bf16x8 (&qf)[DV / 32 + 2], bool act, const unsigned short* qc, const unsigned short* q_rot, int g, G&& asked, F&& angle) {
  constexpr int KL = DV / 32;
  const u16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int ks = 0; ks < KL; ++ks)
    qf[ks] = __builtin_bit_cast(bf16x8, act ? *reinterpret_cast<const u16x8*>(qc + 32 * ks + 8 * g) : zero);
  u16x8 a = zero, b = zero;
  if (act) {
    const unsigned short* src = q_rot != nullptr ? q_rot : qc + DV;
    a = *reinterpret_cast<const u16x8*>(src + 8 * g);
    b = *reinterpret_cast<const u16x8*>(src + 32 + 8 * g);
  }
  asked();
  if (q_rot != nullptr && act) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float sn, cs;
      angle(8 * g + e, sn, cs);
      const float u = bf16_to_f32(a[e]), w = bf16_to_f32(b[e]);
      a[e] = f32_to_bf16(u * cs - w * sn);
      b[e] = f32_to_bf16(w * cs + u * sn);
    }
  }
  qf[KL] = __builtin_bit_cast(bf16x8, a);
  qf[KL + 1] = __builtin_bit_cast(bf16x8, b);
}

// 64 (token, head) rows of consecutive tokens of one sequence. Between two barriers waves 0 - 3 multiply tile i with the
// queries and make P of it (the next tile's operands on their way from LDS meanwhile), waves 4 - 7 add tile i - 1 to the
// outputs, and all copy tile i + 2 into the buffer that tile i - 2 has left.
template <int DV>
__global__ __launch_bounds__(512, 2) void latent_dma_prefill_kernel(
    unsigned short* __restrict__ o_lat, const unsigned short* __restrict__ qc, const unsigned short* __restrict__ q,
    const long* __restrict__ positions, const float* __restrict__ inv_freq, const unsigned short* __restrict__ proj,
    long proj_ld, const unsigned short* __restrict__ cache, int block_shift, const int* __restrict__ seq_cu,
    const int* __restrict__ seq_ctx, const int* __restrict__ seq_bt, int bt_width, int seq0, int seq1, int tq, int hc,
    int T_rows, int heads, int dim, int gate_off, float scale, int window) {
  using KT = Tile<DV, kKeys>;
  constexpr int KS = DV / 32 + 2, NPW = KT::NPW, Dk = DV + kRot;
  constexpr int kMainCopies = DV / 128;   // a wave's share of a tile: 4 keys of the latent part, 1 KB per copy
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  unsigned short* p_lds = reinterpret_cast<unsigned short*>(smem + 4 * KT::kBytes);   // [2][64][kPLd], MFMA k order
  float* alpha = reinterpret_cast<float*>(p_lds + 2 * 64 * kPLd);                     // [2][64]
  float* l_lds = alpha + 2 * 64;                                                      // [64] (epilogue)
  int s, tok0;
  if (!find_row_tile(seq_cu, seq0, seq1, tq, blockIdx.x, s, tok0)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int r0 = seq_cu[s], n = seq_cu[s + 1] - r0, ctx = seq_ctx[s];
  const int ntok = min(tq, n - tok0);
  const int h0 = blockIdx.y * hc, nh = min(hc, heads - h0);
  const int p_first = ctx - n + tok0, hi = p_first + ntok - 1;
  // tiles start at multiples of 32: a wave's 4 keys (8 of the rotary part) lie on one page, looked up by the scalar unit
  const int lo0 = window > 0 ? max(0, p_first - window + 1) : 0, lo = lo0 & ~(kKeys - 1);
  const int ntiles = (hi - lo) / kKeys + 1;
  const int* bt = seq_bt + (long)s * bt_width;
  const int mask = (1 << block_shift) - 1;
  // the first of the keys 4 wave .. + 3 of tile t that exists, and its page; keys past the last one are the last one again
  auto page_of = [&](int t, int k) { return bt[min(lo + t * kKeys + k, hi) >> block_shift]; };
  constexpr int kPer = 512 / DV, kChunks = DV / 8;   // keys and 16-byte chunks of a key per copy
  unsigned off_main[kMainCopies], off_rot;           // the lane's bytes past the row of the tile's first key (of its page)
#pragma unroll
  for (int i = 0; i < kMainCopies; ++i) {
    const int k = 4 * wave + i * kPer + lane / kChunks;
    off_main[i] = ((k & mask) * Dk + 8 * ((lane % kChunks) ^ swizzle(k))) * 2;
  }
  {
    const int k = 8 * (wave & 3) + lane / 8;
    off_rot = ((k & mask) * Dk + DV + 8 * ((lane & 7) ^ rot_swizzle(k))) * 2;
  }
  const unsigned lds0 = lds_at(smem);
  auto copy = [&](int t, int page, int page_rot) {
    const unsigned lds = lds0 + (t & 3) * KT::kBytes;
    const int j0 = lo + t * kKeys;
    if (j0 + kKeys - 1 <= hi) {   // all keys exist: the addresses differ from tile to tile by uniform numbers
      const unsigned char* base = reinterpret_cast<const unsigned char*>(cache + (((long)page << block_shift) + (j0 & mask)) * Dk);
#pragma unroll
      for (int i = 0; i < kMainCopies; ++i) copy_1k(base, off_main[i], lds + (4 * wave + i * kPer) * DV * 2);
      if (wave < 4)
        copy_1k(reinterpret_cast<const unsigned char*>(cache + (((long)page_rot << block_shift) + (j0 & mask)) * Dk), off_rot,
                lds + KT::kMain + 8 * wave * kRot * 2);
      return;
    }
#pragma unroll
    for (int i = 0; i < kMainCopies; ++i) {
      const int k = 4 * wave + i * kPer + lane / kChunks, ch = (lane % kChunks) ^ swizzle(k);
      const unsigned short* src = cache + (((long)page << block_shift) + (min(j0 + k, hi) & mask)) * Dk + 8 * ch;
      copy_1k(src, lds + (4 * wave + i * kPer) * DV * 2);
    }
    if (wave < 4) {
      const int k = 8 * wave + lane / 8, ch = (lane & 7) ^ rot_swizzle(k);
      const unsigned short* src = cache + (((long)page_rot << block_shift) + (min(j0 + k, hi) & mask)) * Dk + DV + 8 * ch;
      copy_1k(src, lds + KT::kMain + 8 * wave * kRot * 2);
    }
  };
  const int krot = 8 * (wave & 3);
  copy(0, page_of(0, 4 * wave), page_of(0, krot));
  if (ntiles > 1) copy(1, page_of(1, 4 * wave), page_of(1, krot));
  int page = page_of(2, 4 * wave), page_rot = page_of(2, krot);   // clamped: always an existing page
  auto copy_next = [&](int t) {   // tile t, whose pages are at hand
    if (t >= ntiles) return;
    copy(t, page, page_rot);
    page = page_of(t + 1, 4 * wave);
    page_rot = page_of(t + 1, krot);
  };
  const typename KT::Places at = KT::places(wave & 3, c, g);
  if (wave < 4) {
    const int sr = 16 * wave + c, srt = sr / hc, srh = sr % hc;
    const bool sact = srt < ntok && srh < nh;
    const long strow = r0 + tok0 + (sact ? srt : 0);
    const int shead = h0 + (sact ? srh : 0);
    const int spos = p_first + srt;
    const int s_lo = window > 0 ? max(0, spos - window + 1) : 0;
    bf16x8 qf[KS];
    load_query<DV>(qf, sact, qc + ((long)shead * T_rows + strow) * Dk,
                   q != nullptr ? q + strow * heads * (dim + kRot) + (long)shead * (dim + kRot) + dim : nullptr,
                   g, [] {}, [&, pos = (float)positions[strow]](int i, float& sn, float& cs) { sincosf(pos * inv_freq[i], &sn, &cs); });
    float m_run = -INFINITY;   // what the weights are relative to, log2 domain
    f32x4 lsum = {0.f, 0.f, 0.f, 0.f};   // sums of the weights that are multiplied, the same number in all four
    const u32x4 ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
    const float scale2 = scale * kLog2e;
    constexpr int kBatch = 6, kBatches = (KS + kBatch - 1) / kBatch;   // steps whose operands are read together
    bf16x8 ka[2][kBatch][2];
    f32x4 sc[2];
    auto read_keys = [&](int i, int b) {
      const unsigned char* kt = smem + (i & 3) * KT::kBytes;
#pragma unroll
      for (int u = 0; u < kBatch; ++u)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          if (b * kBatch + u < KS) ka[b & 1][u][nt] = KT::key_operand(kt, at, 16 * nt, b * kBatch + u);
    };
    auto multiply = [&](int i) {   // batches 0 and 1 of tile i are read
      sc[0] = sc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < kBatches; ++b) {
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
#pragma unroll
          for (int nt = 0; nt < 2; ++nt)
            if (b * kBatch + u < KS)
              sc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[b & 1][u][nt], qf[b * kBatch + u], sc[nt], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (b + 2 < kBatches) read_keys(i, b + 2);
      }
    };
    barrier_all();
    copy_next(2);
    read_keys(0, 0);
    if constexpr (kBatches > 1) read_keys(0, 1);
    multiply(0);
    for (int i = 1; i <= ntiles; ++i) {
      if (i < ntiles) {
        read_keys(i, 0);
        if constexpr (kBatches > 1) read_keys(i, 1);
      }
      __builtin_amdgcn_sched_barrier(0);
      // masked online softmax (log2 domain) of tile i - 1, row sr: lane (c, g) holds keys 16 nt + 4 g + e
      const int j0 = lo + (i - 1) * kKeys;
      float v[8], mx = -INFINITY;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = sc[e >> 2][e & 3];
      if (!__all(sact && j0 + kKeys - 1 <= spos && j0 >= s_lo)) {   // not every row of the wave sees the whole tile
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int j = j0 + 16 * (e >> 2) + 4 * g + (e & 3);
          if (!sact || j > spos || j < s_lo) v[e] = -INFINITY;
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) mx = fmaxf(mx, v[e]);
      mx = max_of_rows(mx) * scale2;
      float al = 1.f;
      if (__any(mx > m_run)) {
        const float mn = fmaxf(m_run, mx);
        al = mn > -INFINITY ? __builtin_amdgcn_exp2f(m_run - mn) : 1.f;  // m_run = -inf: 0
        m_run = mn;
        lsum *= al;
      }
      const float off = m_run > -INFINITY ? m_run : 0.f;   // no key seen yet: every weight is exp2(-inf) = 0
      u32x4 pk;
#pragma unroll
      for (int e = 0; e < 8; e += 2)   // rounded: what is multiplied, and its sum
        pk[e / 2] = pack2(__builtin_amdgcn_exp2f(fmaf(v[e], scale2, -off)), __builtin_amdgcn_exp2f(fmaf(v[e + 1], scale2, -off)));
      const int pb = (i - 1) & 1;
      *reinterpret_cast<u32x4*>(p_lds + (pb * 64 + sr) * kPLd + 8 * g) = pk;
      if (g == 0) alpha[pb * 64 + sr] = al;
      lsum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ones), __builtin_bit_cast(bf16x8, pk), lsum, 0, 0, 0);
      barrier_all();
      copy_next(i + 2);
      if (i < ntiles) multiply(i);
    }
    if (g == 0) {   // gate / softmax sum of the row
      float f = 0.f;
      if (sact && lsum[0] > 0.f) {
        f = 1.f / lsum[0];
        if (gate_off >= 0) f *= sigmoid_f(bf16_to_f32(proj[strow * proj_ld + gate_off + shead]));
      }
      l_lds[sr] = f;
    }
    barrier_lds();
    return;
  }
  f32x4 acc[4][NPW];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int j = 0; j < NPW; ++j) acc[mt][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  barrier_all();
  copy_next(2);
  for (int i = 1; i <= ntiles; ++i) {
    barrier_all();
    copy_next(i + 2);
    unsigned char* kt = smem + ((i - 1) & 3) * KT::kBytes;
    const unsigned short* pt = p_lds + ((i - 1) & 1) * 64 * kPLd;
    bf16x8 pb[4], va[NPW];
    float al[4];
    bool rescale = false;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      pb[mt] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u16x8*>(pt + (16 * mt + c) * kPLd + 8 * g));
      al[mt] = alpha[((i - 1) & 1) * 64 + 16 * mt + c];
      rescale |= al[mt] != 1.f;
    }
#pragma unroll
    for (int j = 0; j < NPW; ++j) va[j] = KT::value_operand(kt, at, 0, j);
    if (i == 1 && lo < lo0) clear_below(va, lo, lo0, g);
    __builtin_amdgcn_sched_barrier(0);
    if (__any(rescale)) {
#pragma unroll
      for (int j = 0; j < NPW; ++j)
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) acc[mt][j] *= al[mt];
    }
#pragma unroll
    for (int j = 0; j < NPW; ++j)
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) acc[mt][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[j], pb[mt], acc[mt][j], 0, 0, 0);
  }
  barrier_lds();
  // lane (c, g) holds latent dims 16 nt + 4 g .. + 3 of row 16 mt + c
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    const int r = 16 * mt + c, rt = r / hc, rh = r % hc;
    if (rt >= ntok || rh >= nh) continue;
    const float f = l_lds[r];
    unsigned short* dst = o_lat + ((long)(h0 + rh) * T_rows + r0 + tok0 + rt) * DV + 16 * NPW * (wave - 4) + 4 * g;
#pragma unroll
    for (int j = 0; j < NPW; ++j) {
      u16x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = f32_to_bf16(acc[mt][j][e] * f);
      *reinterpret_cast<u16x4*>(dst + 16 * j) = o;
    }
  }
}

// 16 heads of the portion's row blockIdx.x against the run blockIdx.z of part_keys keys, 64 at a time: for portions of a row per
// sequence, as decode rows are, and for runs. Wave w: scores of keys 16 w .., P . V of the latent dims DV / 4 w ... With
// runs the unnormalised outputs and (max, sum) go to ws_acc / ws_ml.
// What bounds it where the keys are few: the instructions of one wave in turn. The scalars that places and lengths need are asked for in one batch
// with the arguments, the row's 32 angles are made once, a lane each, and a copy takes its key's row from a scalar
// register, the scores are two chains. us with the merge of runs (latent_attention_mfma.hip), 16 heads, before / this: one row of 64 keys 8.4 / 6.9, of 256 11.1 /
// 9.3, of 1024 11.4 / 9.7, 13 rows of 1300 15.6 / 14.2, 48 rows of 182 12.4 / 10.6.
struct LatentDecodeRest {
  unsigned short* o_lat;
  const unsigned short *qc, *q, *proj;
  const float* inv_freq;
  float *ws_acc, *ws_ml;
  long proj_ld;
  int T_rows, heads, dim, gate_off, window, part_keys, row_base, ws_rows, nparts;
  float scale;
};

template <int DV>
__global__ __launch_bounds__(256, 2) void latent_dma_decode_kernel(
    const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx, const int* __restrict__ seq_bt, const long* __restrict__ positions,
    const unsigned short* __restrict__ cache, int seq0, int seq1, int bt_width, int block_shift, const LatentDecodeRest rest) {
  constexpr int kTile = 64, kPd = kTile + 8;   // kPd: row stride of P in elements
  using KT = Tile<DV, kTile>;
  constexpr int KS = DV / 32 + 2, NPW = DV / 64, Dk = DV + kRot;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ float2 angles[kRot / 2];
  unsigned short* p_lds = reinterpret_cast<unsigned short*>(smem + KT::kBytes);   // [16][kPd], MFMA k order
  float* mw = reinterpret_cast<float*>(p_lds + 16 * kPd);                         // [4][16] the waves' maxima
  float* lw = mw + 64;                                                            // [4][16] the waves' sums
  const int x = blockIdx.x;
  int s = min(seq0 + x, seq1 - 1), tok0 = 0;
  int first = seq_cu[seq0], r0 = seq_cu[s], r1 = seq_cu[s + 1], ctx = seq_ctx[s];
  unsigned short* __restrict__ const o_lat = rest.o_lat;
  const unsigned short *__restrict__ const qc = rest.qc, *__restrict__ const q = rest.q, *__restrict__ const proj = rest.proj;
  const float* __restrict__ const inv_freq = rest.inv_freq;
  float *__restrict__ const ws_acc = rest.ws_acc, *__restrict__ const ws_ml = rest.ws_ml;
  const int T_rows = rest.T_rows, heads = rest.heads, dim = rest.dim, gate_off = rest.gate_off, window = rest.window, part_keys = rest.part_keys;
  const long proj_ld = rest.proj_ld;
  const float scale = rest.scale;
  const bool partial = rest.nparts > 1;
  asm volatile("" ::"s"(qc), "s"(q), "s"(inv_freq), "s"(ws_ml), "s"(T_rows), "s"(heads), "s"(dim), "s"(window), "s"(part_keys), "s"(rest.row_base),
               "s"(rest.ws_rows), "s"(rest.nparts));
  if (seq0 + x >= seq1 || r0 - first != x || r1 - r0 != 1) {   // not one row per sequence up to here
    if (!find_row(seq_cu, seq0, seq1, x, s, tok0)) return;
    r0 = seq_cu[s];
    r1 = seq_cu[s + 1];
    ctx = seq_ctx[s];
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4;
  const int head = blockIdx.y * 16 + c;
  const bool act = head < heads;
  const int pos = ctx - (r1 - r0) + tok0;
  const long trow = r0 + tok0;
  const int lo = (window > 0 ? max(0, pos - window + 1) : 0) + blockIdx.z * part_keys;
  const int hi = partial ? min(pos, lo + part_keys - 1) : pos;
  const long wrow = ((long)blockIdx.z * heads + (act ? head : 0)) * rest.ws_rows + (trow - rest.row_base);
  const int d0 = 16 * NPW * wave + 4 * g;   // the lane's latent dims of the output: 16 j + d0 .. + 3
  if (lo > hi) {   // an empty run, whose weight in the merge is 0, or a row that sees no key
    if (partial && act && wave == 0 && g == 0) { ws_ml[2 * wrow] = -INFINITY; ws_ml[2 * wrow + 1] = 0.f; }
    if (!partial && act)
#pragma unroll
      for (int j = 0; j < NPW; ++j) *reinterpret_cast<u16x4*>(o_lat + ((long)head * T_rows + trow) * DV + d0 + 16 * j) = u16x4{0, 0, 0, 0};
    return;
  }
  const int* bt = seq_bt + (long)s * bt_width;
  const int mask = (1 << block_shift) - 1;
  auto row_of = [&](int j0) {
    const int j = min(j0 + lane, hi);
    return (long)((unsigned long)(unsigned)((bt[j >> block_shift] << block_shift) + (j & mask)) * Dk);
  };
  const unsigned lds0 = lds_at(smem);
  auto copy = [&](int j0) {
    const long row = row_of(j0);
    KT::copy(lds0, cache, row, 2 * wave, lane);
    KT::copy(lds0, cache, row, 2 * wave + 1, lane);
  };
  const bool rotate = q != nullptr;
  const float at_pos = (float)positions[trow], freq = rotate ? inv_freq[lane & (kRot / 2 - 1)] : 0.f;
  copy(lo);
  bf16x8 qf[KS];
  load_query<DV>(qf, act, qc + ((long)(act ? head : 0) * T_rows + trow) * Dk,
                 rotate ? q + trow * heads * (dim + kRot) + (long)(act ? head : 0) * (dim + kRot) + dim : nullptr, g,
                 [&] {
                   if (!rotate) return;
                   if (tid < kRot / 2) {
                     float sn, cs;
                     sincosf(at_pos * freq, &sn, &cs);
                     angles[tid] = float2{sn, cs};
                   }
                   barrier_lds();
                 },
                 [&](int i, float& sn, float& cs) { const float2 a = angles[i]; sn = a.x; cs = a.y; });
  f32x4 acc[NPW];
#pragma unroll
  for (int j = 0; j < NPW; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;   // of row c, the same in every wave
  const float scale2 = scale * kLog2e;
  const typename KT::Places at = KT::places(wave, c, g);
  for (int j0 = lo; j0 <= hi; j0 += kTile) {
    barrier_all();
    f32x4 half[2] = {};   // two chains
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      half[ks & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(KT::key_operand(smem, at, 16 * wave, ks), qf[ks], half[ks & 1], 0, 0, 0);
    const f32x4 sc = half[0] + half[1];
    float v[4], mx = -INFINITY;   // keys 16 wave + 4 g + i
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = act && j0 + 16 * wave + 4 * g + i <= hi ? sc[i] * scale2 : -INFINITY;
      mx = fmaxf(mx, v[i]);
    }
    mx = max_of_rows(mx);
    if (g == 0) mw[16 * wave + c] = mx;
    barrier_lds();
    const float mn = fmaxf(fmaxf(fmaxf(mw[c], mw[16 + c]), fmaxf(mw[32 + c], mw[48 + c])), m_run);
    float sum = 0.f;
    u16x4 pk;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      pk[i] = f32_to_bf16(mn > -INFINITY ? __builtin_amdgcn_exp2f(v[i] - mn) : 0.f);
      sum += bf16_to_f32(pk[i]);
    }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    // key 32 kk + 16 h + 4 g + i sits at column 32 kk + 8 g + 4 h + i (kk = wave / 2, h = wave % 2)
    *reinterpret_cast<u16x4*>(p_lds + c * kPd + 32 * (wave >> 1) + 8 * g + 4 * (wave & 1)) = pk;
    if (g == 0) lw[16 * wave + c] = sum;
    const float al = mn > -INFINITY ? __builtin_amdgcn_exp2f(m_run - mn) : 1.f;
    m_run = mn;
    barrier_lds();
    l_run = l_run * al + (lw[c] + lw[16 + c]) + (lw[32 + c] + lw[48 + c]);
#pragma unroll
    for (int j = 0; j < NPW; ++j) acc[j] *= al;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const bf16x8 pb = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u16x8*>(p_lds + c * kPd + 32 * kk + 8 * g));
#pragma unroll
      for (int j = 0; j < NPW; ++j)
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(KT::value_operand(smem, at, 32 * kk, j), pb, acc[j], 0, 0, 0);
    }
    if (j0 + kTile <= hi) {
      barrier_lds();   // the tile is read
      copy(j0 + kTile);
    }
  }
  if (!act) return;
  if (partial) {
    if (wave == 0 && g == 0) { ws_ml[2 * wrow] = m_run / kLog2e; ws_ml[2 * wrow + 1] = l_run; }
#pragma unroll
    for (int j = 0; j < NPW; ++j) *reinterpret_cast<f32x4*>(ws_acc + wrow * DV + d0 + 16 * j) = acc[j];
    return;
  }
  float f = l_run > 0.f ? 1.f / l_run : 0.f;
  if (gate_off >= 0) f *= sigmoid_f(bf16_to_f32(proj[trow * proj_ld + gate_off + head]));
  unsigned short* dst = o_lat + ((long)head * T_rows + trow) * DV + d0;
#pragma unroll
  for (int j = 0; j < NPW; ++j) {
    u16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = f32_to_bf16(acc[j][e] * f);
    *reinterpret_cast<u16x4*>(dst + 16 * j) = o;
  }
}

template <int DV>
bool launch_dma(void* o_lat, const void* qc, const void* q, const long* positions, const float* inv_freq, const void* proj,
                long proj_ld, const void* cache, int block_shift, const int* seq_cu, const int* seq_ctx, const int* seq_bt,
                int bt_width, int seq0, int seq1, int rows_bound, int T, int heads, int dim, int gate_off, float scale,
                int window, int nparts, int part_keys, float* ws_acc, float* ws_ml, int row_base, hipStream_t s) {
  auto o = (unsigned short*)o_lat;
  auto a = (const unsigned short*)qc, b = (const unsigned short*)q, p = (const unsigned short*)proj, k = (const unsigned short*)cache;
  if (nparts > 1 || rows_bound == seq1 - seq0) {   // either kernel takes any rows: a workgroup per row where they are single ones
    constexpr size_t smem = Tile<DV, 64>::kBytes + 16 * (64 + 8) * 2 + 128 * 4;
    static_assert(smem <= 80 * 1024, "two workgroups per CU");
    static const bool ok = allow_lds(&latent_dma_decode_kernel<DV>, smem);
    if (!ok) return false;
    latent_dma_decode_kernel<DV><<<dim3(rows_bound, (heads + 15) / 16, nparts), 256, smem, s>>>(
        seq_cu, seq_ctx, seq_bt, positions, k, seq0, seq1, bt_width, block_shift,
        LatentDecodeRest{o, a, b, p, inv_freq, ws_acc, ws_ml, proj_ld, T, heads, dim, gate_off, window, part_keys, row_base, rows_bound, nparts, scale});
    return true;
  }
  constexpr size_t smem = 4 * Tile<DV, kKeys>::kBytes + 2 * 64 * kPLd * 2 + 3 * 64 * 4;
  static_assert(smem <= 160 * 1024, "LDS");
  static const bool ok = allow_lds(&latent_dma_prefill_kernel<DV>, smem);
  if (!ok) return false;
  const int hc = min(heads, 64), tq = 64 / hc;
  latent_dma_prefill_kernel<DV><<<dim3(rows_bound / tq + (seq1 - seq0), (heads + hc - 1) / hc), 512, smem, s>>>(
      o, a, b, positions, inv_freq, p, proj_ld, k, block_shift, seq_cu, seq_ctx, seq_bt, bt_width, seq0, seq1, tq, hc, T, heads, dim,
      gate_off, scale, window);
  return true;
}

}  // namespace

bool latent_attention_dma_ok(int kv_rank, int rot_dim) {
  return rot_dim == kRot && (kv_rank == 128 || kv_rank == 256 || kv_rank == 512);
}

bool launch_latent_attention_dma(void* o_lat, const void* qc, const void* q, const long* positions, const float* inv_freq,
                                 const void* proj, long proj_ld, const void* cache, int block_size, const int* seq_cu,
                                 const int* seq_ctx, const int* seq_bt, int bt_width, int seq0, int seq1, int rows_bound, int T,
                                 int heads, int dim, int kv_rank, int gate_off, float scale, int window, int nparts,
                                 int part_keys, float* ws_acc, float* ws_ml, int row_base, hipStream_t s) {
  if (seq1 <= seq0 || rows_bound <= 0) return true;
  const int block_shift = __builtin_ctz(block_size);   // a power of two
#define HS_LD(DV)                                                                                                        \
  launch_dma<DV>(o_lat, qc, q, positions, inv_freq, proj, proj_ld, cache, block_shift, seq_cu, seq_ctx, seq_bt, bt_width, \
                 seq0, seq1, rows_bound, T, heads, dim, gate_off, scale, window, nparts, part_keys, ws_acc,     \
                 ws_ml, row_base, s)
  return kv_rank == 128 ? HS_LD(128) : kv_rank == 256 ? HS_LD(256) : HS_LD(512);
#undef HS_LD
}

}  // namespace hipserve

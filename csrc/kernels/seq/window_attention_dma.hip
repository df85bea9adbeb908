// Window attention of prompt portions in bf16 for heads of 64 or 128 dims (keys and values alike) without kept first keys:
// the products of window_attention_mfma.hip with the cache rows copied straight into LDS.
//
// That kernel loads a 32-key tile into registers, stores the values to LDS transposed, two bytes at a time, and waits at two
// barriers per tile: a tile costs far more than its products and its softmax. Here
//   * global_load_lds brings the rows into one of four LDS buffers, three tiles ahead; a wave copies 8 keys and 8 values of
//     each tile, whose page the scalar unit looks up (tiles start at multiples of 32);
//   * the V^T operand comes from ds_read_tr16_b64 (latent_attention_dma.hip says how), so a tile needs one barrier;
//   * softmax costs the vector unit little more than an fma, an exponential and half a conversion per score: maxima are taken
//     of the raw products and go round by row swaps, sums come from a product with ones, and the accumulators are rescaled
//     only where a row's maximum grows. (Not rarer: the largest weight is 1 then, which bf16 holds exactly. A maximum that follows
//     only when a score is larger by 2^8 saves 8 us below, and the outputs' error against 64 bits grows by up to a tenth, 1.80e-3 ->
//     1.97e-3 with their own rounding);
//   * the workgroups of one key / value head follow each other on the same XCD, whose L2 holds its rows, and the late
//     tokens of the step, which see the most keys, go first.
// 8192 rows (4 prompts) x 16 heads over 4 of 128, window 1024: 185 -> 110 us (470 TFLOP/s). Without the rescaling (104 us) the vector
// unit is busy 40 % of the time, the matrix cores 27 %; waves wait at the barrier and for operands a third of their time, and a
// fifth of the wave slots is empty at the ends. On the way, without it: 152 with a branch per score for the score cap, 124 with the softmax of
// window_attention_mfma.hip, 110 with row-wise operands two to a bank, 107 with tests of LDS pointers at each copy; three
// workgroups per CU (three buffers, 168 registers) spill: 131.
#include "lds_copy.h"
#include "seq_common.h"
#include "hipserve/seq_kernels.h"

namespace hipserve {
namespace {

constexpr int kKeys = 32, kStages = 4, kThreads = 256;
constexpr float kLog2e = 1.44269504088896341f;

// 16-byte chunk ch of key (value) row k sits at chunk ch ^ key_swizzle (value_swizzle) of it: the 16 rows of a key operand use
// 16 different chunks of 256 bytes, the 8 rows of a transposing read 8 different pairs (rows of 128 bytes: two fill 256).
template <int D> HS_DEVICE int key_swizzle(int k) { return D == 128 ? k & 15 : k >> 1 & 7; }
template <int D> HS_DEVICE int value_swizzle(int k) { return (D == 128 ? k & 7 : k >> 1 & 3) << 1; }

// MT: 16-row tiles per wave; 64 MT (token, head) rows of one key / value head per workgroup.
template <int D, int MT>
__global__ __launch_bounds__(kThreads, 2) void window_dma_prefill_kernel(
    unsigned short* __restrict__ out, long out_ld, const unsigned short* __restrict__ proj, long proj_ld,
    const unsigned short* __restrict__ cache, int block_shift, const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx,
    const int* __restrict__ seq_bt, int bt_width, int seq0, int seq1, int tiles, int tq, int hc, int hchunks, int heads,
    int kv_heads, int gate_off, float scale, int window, bool sink, float out_scale, float softcap,
    const float* __restrict__ sink_w, bool channel_gate, int chunk) {
  constexpr int KS = D / 32, NV = D / 16, kRow = D * 2, kHalf = kKeys * kRow, kStage = 2 * kHalf;
  constexpr int kPer = 1024 / kRow, kCopies = 8 / kPer, kChunks = D / 8;   // rows per copy; copies of 8 rows; chunks per row
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];     // [stage][keys | values][32][D]
  const int ny = kv_heads * hchunks, hy = blockIdx.x % ny;
  int s, tok0;
  if (!find_row_tile(seq_cu, seq0, seq1, tq, tiles - 1 - (int)(blockIdx.x / ny), s, tok0)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4;
  const int group = heads / kv_heads, kvh = hy / hchunks, h0 = (hy % hchunks) * hc, nh = min(hc, group - h0);
  const int r0 = seq_cu[s], n = seq_cu[s + 1] - r0, ctx = seq_ctx[s], ntok = min(tq, n - tok0);
  const int p_first = ctx - n + tok0, hi = p_first + ntok - 1;
  const int lo0 = first_key(p_first, window, chunk), lo = lo0 & ~(kKeys - 1), ntiles = (hi - lo) / kKeys + 1;
  const long Dc = 2L * kv_heads * D;
  const int* bt = seq_bt + (long)s * bt_width;
  const int mask = (1 << block_shift) - 1;
  auto page_of = [&](int t) { return bt[min(lo + t * kKeys + 8 * wave, hi) >> block_shift]; };   // of the wave's 8 keys
  unsigned koff[kCopies], voff[kCopies];   // the lane's bytes past the row of the tile's first key (of its page)
#pragma unroll
  for (int i = 0; i < kCopies; ++i) {
    const int k = 8 * wave + i * kPer + lane / kChunks;
    koff[i] = ((unsigned)(k & mask) * Dc + 8 * ((lane % kChunks) ^ key_swizzle<D>(k))) * 2;
    voff[i] = ((unsigned)(k & mask) * Dc + kv_heads * D + 8 * ((lane % kChunks) ^ value_swizzle<D>(k))) * 2;
  }
  const unsigned lds0 = lds_at(smem) + 8 * wave * kRow;
  const unsigned short* const keys0 = cache + (long)kvh * D;
  const unsigned row_bytes = (unsigned)Dc * 2;
  auto copy = [&](int t, int page) {
    const unsigned to = lds0 + (t % kStages) * kStage;
    const int j0 = lo + t * kKeys;
    if (j0 + kKeys - 1 <= hi) {   // all keys exist: the addresses differ from tile to tile by uniform numbers
      const unsigned char* keys = reinterpret_cast<const unsigned char*>(keys0) +
                                  (unsigned long)(((unsigned)page << block_shift) + (unsigned)(j0 & mask)) * row_bytes;
#pragma unroll
      for (int i = 0; i < kCopies; ++i) {
        copy_1k(keys, koff[i], to + i * 1024);
        copy_1k(keys, voff[i], to + kHalf + i * 1024);
      }
      return;
    }
    const unsigned short* keys = keys0 + ((long)page << block_shift) * Dc;
    const unsigned short* vals = keys + (long)kv_heads * D;
#pragma unroll
    for (int i = 0; i < kCopies; ++i) {   // keys past the last one are the last one again
      const int k = 8 * wave + i * kPer + lane / kChunks;
      const long at = (long)(min(j0 + k, hi) & mask) * Dc;
      copy_1k(keys + at + 8 * ((lane % kChunks) ^ key_swizzle<D>(k)), to + i * 1024);
      copy_1k(vals + at + 8 * ((lane % kChunks) ^ value_swizzle<D>(k)), to + kHalf + i * 1024);
    }
  };
  // pages of tiles 0 .. 2 and, one tile before its copy, of the next: clamped, so always an existing page
  const int page0 = page_of(0), page1 = page_of(1), page2 = page_of(2);
  copy(0, page0);
  if (ntiles > 1) copy(1, page1);
  if (ntiles > 2) copy(2, page2);
  int page = page_of(3);

  // this lane's rows: row sr = token sr / hc, head sr % hc of the group
  bool sact[MT];
  int head[MT], spos[MT], s_lo[MT];
  long trow[MT];
  bf16x8 qf[MT][KS];
  f32x4 acc[MT][NV];
  f32x4 lsum[MT];    // sums of the weights that are multiplied, the same number in all four
  float m_run[MT];   // what the weights are relative to, log2 domain
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int sr = 16 * (wave * MT + mt) + c, srt = sr / hc, srh = sr % hc;
    sact[mt] = srt < ntok && srh < nh;
    head[mt] = kvh * group + h0 + (sact[mt] ? srh : 0);
    trow[mt] = r0 + tok0 + (sact[mt] ? srt : 0);
    spos[mt] = sact[mt] ? p_first + srt : -1;   // a row that does not exist sees no key
    s_lo[mt] = first_key(p_first + srt, window, chunk);
    const unsigned short* src = proj + trow[mt] * proj_ld + (long)head[mt] * D + 8 * g;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[mt][ks] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u16x8*>(src + 32 * ks));
#pragma unroll
    for (int j = 0; j < NV; ++j) acc[mt][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    m_run[mt] = sink ? (sink_w != nullptr ? sink_w[head[mt]] * kLog2e : 0.f) : -INFINITY;
    const float l0 = sink ? 1.f : 0.f;
    lsum[mt] = f32x4{l0, l0, l0, l0};
  }
  const float unit = softcap > 0.f ? 1.f : scale * kLog2e, cap2 = softcap * kLog2e, icap = softcap > 0.f ? scale / softcap : 0.f;
  const u32x4 ones_u = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
  const bf16x8 ones = __builtin_bit_cast(bf16x8, ones_u);
  int kat[KS], vat[NV];   // the lane's places in a tile
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) kat[ks] = c * kRow + (((4 * ks + g) ^ key_swizzle<D>(c)) << 4);
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int k = 4 * g + (c >> 2);
    vat[j] = kHalf + k * kRow + (((2 * j + ((c & 3) >> 1)) ^ value_swizzle<D>(k)) << 4) + 8 * (c & 1);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): the queries; the copies in flight below are this loop's own
  for (int i = 0; i < ntiles; ++i) {
    if (i + 2 < ntiles) barrier_copies<4 * kCopies>();   // two tiles may be in flight
    else if (i + 1 < ntiles) barrier_copies<2 * kCopies>();
    else barrier_copies<0>();
    if (i + 3 < ntiles) {   // into the buffer of tile i - 1, which every wave has left
      copy(i + 3, page);
      page = page_of(i + 4);
    }
    unsigned char* tile = smem + (i % kStages) * kStage;
    const int j0 = lo + i * kKeys;
    f32x4 sc[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) sc[mt][0] = sc[mt][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        const bf16x8 a = __builtin_bit_cast(
            bf16x8, *reinterpret_cast<const u16x8*>(tile + kat[ks] + 16 * nt * kRow));
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) sc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qf[mt][ks], sc[mt][nt], 0, 0, 0);
      }
    bf16x8 va[NV];   // read while softmax runs
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      s16x4 h[2];
#pragma unroll
      for (int i2 = 0; i2 < 2; ++i2) h[i2] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(tile + vat[j] + 16 * i2 * kRow));
      va[j] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(h[0], h[1], 0, 1, 2, 3, 4, 5, 6, 7));
    }
    if (i == 0 && lo < lo0) clear_below(va, lo, lo0, g);
    __builtin_amdgcn_sched_barrier(0);
    bf16x8 pb[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      // lane (c, g): keys 16 nt + 4 g + e; times `unit`: log2 domain
      float v[8], mx = -INFINITY;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = sc[mt][e >> 2][e & 3];
      if (softcap > 0.f) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = cap2 * tanh_fast(v[e] * icap);
      }
      if (!__all(j0 + kKeys - 1 <= spos[mt] && j0 >= s_lo[mt])) {   // most tiles of a long window are seen whole
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int j = j0 + 16 * (e >> 2) + 4 * g + (e & 3);
          if (j > spos[mt] || j < s_lo[mt]) v[e] = -INFINITY;
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) mx = fmaxf(mx, v[e]);
      mx = max_of_rows(mx) * unit;
      if (__any(mx > m_run[mt])) {
        const float mn = fmaxf(m_run[mt], mx), al = mn > -INFINITY ? __builtin_amdgcn_exp2f(m_run[mt] - mn) : 1.f;
        m_run[mt] = mn;
        lsum[mt] *= al;
#pragma unroll
        for (int j = 0; j < NV; ++j) acc[mt][j] *= al;
      }
      const float base = m_run[mt] > -INFINITY ? m_run[mt] : 0.f;   // no key seen yet: every weight is exp2(-inf) = 0
      u32x4 pk;
#pragma unroll
      for (int e = 0; e < 8; e += 2)
        pk[e / 2] = pack2(__builtin_amdgcn_exp2f(fmaf(v[e], unit, -base)), __builtin_amdgcn_exp2f(fmaf(v[e + 1], unit, -base)));
      pb[mt] = __builtin_bit_cast(bf16x8, pk);
      lsum[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb[mt], lsum[mt], 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[j], pb[mt], acc[mt][j], 0, 0, 0);
  }
  // lane (c, g) holds value dims 16 j + 4 g .. + 3 of its rows
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    if (!sact[mt]) continue;
    const float l = lsum[mt][0];
    float f = out_scale;
    if (gate_off >= 0 && !channel_gate) f *= sigmoid_f(bf16_to_f32(proj[trow[mt] * proj_ld + gate_off + head[mt]]));
    f = l == 0.f ? 0.f : f / l;
    const unsigned short* cg = proj + trow[mt] * proj_ld + gate_off + (long)head[mt] * D;   // channel_gate
    unsigned short* dst = out + trow[mt] * out_ld + (long)head[mt] * D;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int d = 16 * j + 4 * g;
      u16x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        o[e] = f32_to_bf16(acc[mt][j][e] * f * (channel_gate ? sigmoid_f(bf16_to_f32(cg[d + e])) : 1.f));
      *reinterpret_cast<u16x4*>(dst + d) = o;
    }
  }
}

template <int D, int MT>
void launch(unsigned short* out, long out_ld, const unsigned short* proj, long proj_ld, const unsigned short* cache, int block_size,
            const int* seq_cu, const int* seq_ctx, const int* seq_bt, int bt_width, int seq0, int seq1, int rows_bound, int heads,
            int kv_heads, int gate_off, float scale, int window, bool sink, float out_scale, float softcap, const float* sink_w,
            bool channel_gate, int chunk, hipStream_t s) {
  const int group = heads / kv_heads, rows = 64 * MT, hc = std::min(group, rows), hchunks = (group + hc - 1) / hc, tq = rows / hc;
  const int tiles = rows_bound / tq + (seq1 - seq0);
  constexpr int smem = kStages * 2 * kKeys * D * 2;
  window_dma_prefill_kernel<D, MT><<<(unsigned)(tiles * kv_heads * hchunks), kThreads, smem, s>>>(
      out, out_ld, proj, proj_ld, cache, __builtin_ctz(block_size), seq_cu, seq_ctx, seq_bt, bt_width, seq0, seq1, tiles, tq, hc,
      hchunks, heads, kv_heads, gate_off, scale, window, sink, out_scale, softcap, sink_w, channel_gate, chunk);
}

}  // namespace

bool window_attention_dma_ok(int dim, int vdim, int block_size, int heads, int kv_heads, const void* proj, long proj_ld,
                             const void* cache) {
  return dim == vdim && (dim == 64 || dim == 128) && block_size >= 16 && (block_size & (block_size - 1)) == 0 &&
         proj_ld % 8 == 0 && reinterpret_cast<uintptr_t>(proj) % 16 == 0 && reinterpret_cast<uintptr_t>(cache) % 16 == 0 &&
         (long)block_size * 4 * kv_heads * dim < (1L << 31);   // a lane's offset on a page is 32 bits
}

void launch_window_attention_dma(void* out, long out_ld, const void* proj, long proj_ld, const void* cache, int block_size,
                                 const int* seq_cu, const int* seq_ctx, const int* seq_bt, int bt_width, int seq0, int seq1,
                                 int rows_bound, int heads, int kv_heads, int dim, int gate_off, float scale, int window, bool sink,
                                 float out_scale, bool wide, float softcap, const float* sink_w, bool channel_gate, int chunk,
                                 hipStream_t s) {
  if (seq1 <= seq0 || rows_bound <= 0) return;
#define HS_WP(D, MT)                                                                                                              \
  launch<D, MT>((unsigned short*)out, out_ld, (const unsigned short*)proj, proj_ld, (const unsigned short*)cache, block_size, seq_cu, \
                seq_ctx, seq_bt, bt_width, seq0, seq1, rows_bound, heads, kv_heads, gate_off, scale, window, sink, out_scale, softcap, \
                sink_w, channel_gate, chunk, s)
  if (dim == 64) { if (wide) HS_WP(64, 2); else HS_WP(64, 1); }
  else if (wide) HS_WP(128, 2);
  else HS_WP(128, 1);
#undef HS_WP
}

}  // namespace hipserve

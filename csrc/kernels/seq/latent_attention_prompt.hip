// Latent attention of prompt steps in bf16 with the keys and values of every head formed once (128 + 64 rotary key dims, 128
// value dims): the visible cache rows of the step's sequences are laid side by side (latent_gather_kernel), one product makes
// [keys of all heads | values of all heads] of them, and latent_prompt_kernel attends to those.
//
// The kernels that attend to the latents themselves multiply 576 + 512 dims per key and head, this one 192 + 128; the product
// that makes the keys and values costs what taking W_uk into the queries and W_uv out of the outputs costs there, once per cache
// row instead of once per token. So it pays where a step brings about as many rows as it sees keys: prompts, not decode rows.
//
// The kernel is that of window_attention_dma.hip for one head per workgroup: tiles of 32 keys go straight into one of four LDS
// buffers (20 KB: keys, values, rotary parts), three tiles ahead; one barrier per tile; V^T by transposing reads. What differs:
// the key rows lie side by side, so that tiles start at the first key a workgroup's rows see and no page is looked up; a wave
// leaves out the tiles that its own rows do not see (of 128 rows x 1024 keys every tenth).
// 8192 rows (4 prompts of 2048) x 16 heads, window 1024: 363 -> 131 us (490 TFLOP/s of the products with visible keys; the LDS is read
// about as long as the matrix units work: 20 KB per 32 rows and tile), the mixer with its products 680 -> 349 us; 41 prompts of 150
// 388 -> 274. Errors of the mixer's output against 64 bits, both ways: 7.0e-3 - 7.4e-3.
#include "lds_copy.h"
#include "seq_common.h"
#include "hipserve/seq_kernels.h"

namespace hipserve {
namespace {

constexpr int kD = 128, kRot = 64, kQ = kD + kRot, kKeys = 32, kStages = 4, kThreads = 256;
constexpr int kRow = kD * 2, kHalf = kKeys * kRow, kStage = 2 * kHalf + kKeys * kRot * 2;
constexpr float kLog2e = 1.44269504088896341f;

// 16-byte chunk ch of key / value / rotary row k sits at chunk ch ^ swizzle of it (window_attention_dma.hip, latent_attention_dma.hip).
HS_DEVICE int key_swizzle(int k) { return k & 15; }
HS_DEVICE int value_swizzle(int k) { return (k & 7) << 1; }
HS_DEVICE int rot_swizzle(int k) { return k >> 1 & 7; }

// The values of keys outside lo .. hi as zeros (the order of clear_below).
template <int N> HS_DEVICE void clear_outside(bf16x8 (&va)[N], int j0, int lo, int hi, int g) {
  u32x4 keep;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int j = j0 + 16 * (r >> 1) + 4 * g + 2 * (r & 1);
    keep[r] = (j >= lo && j <= hi ? 0x0000ffffu : 0u) | (j + 1 >= lo && j + 1 <= hi ? 0xffff0000u : 0u);
  }
#pragma unroll
  for (int i = 0; i < N; ++i) va[i] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, va[i]) & keep);
}

// Keys that a sequence's rows of the step see: from first_key of its first row to its last position.
HS_DEVICE int seen_keys(int n, int ctx, int window) { return n > 0 ? ctx - first_key(ctx - n, window, 0) : 0; }

// lat[off[s] + i] = cache row of key i that sequence s sees; off[s]: sums of the sequences' counts. A wave takes `per` rows.
__global__ __launch_bounds__(256) void latent_gather_kernel(unsigned short* __restrict__ lat, int* __restrict__ off,
                                                            const unsigned short* __restrict__ cache, int block_shift, int dim,
                                                            const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx,
                                                            const int* __restrict__ seq_bt, int bt_width, int nseq, int rows,
                                                            int per, int window) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r0 = (blockIdx.x * 4 + wave) * per, r1 = min(r0 + per, rows);
  const int mask = (1 << block_shift) - 1, chunks = dim / 8;
  int base = 0;
  for (int i0 = 0; i0 < nseq; i0 += 64) {
    const int i = i0 + lane;
    int cnt = 0, kb = 0;
    if (i < nseq) {
      const int n = seq_cu[i + 1] - seq_cu[i], ctx = seq_ctx[i];
      cnt = seen_keys(n, ctx, window);
      kb = ctx - cnt;
    }
    int end = cnt;   // inclusive sum over the lanes
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(end, o, 64);
      if (lane >= o) end += v;
    }
    const int start = base + end - cnt;
    if (blockIdx.x == 0 && wave == 0 && i < nseq) {
      off[i] = start;
      if (i + 1 == nseq) off[nseq] = start + cnt;
    }
    for (unsigned long long mine = __ballot(cnt > 0 && start < r1 && start + cnt > r0); mine != 0; mine &= mine - 1) {
      const int l = __builtin_ctzll(mine);
      const int s0 = __builtin_amdgcn_readlane(start, l), c0 = __builtin_amdgcn_readlane(cnt, l), k0 = __builtin_amdgcn_readlane(kb, l);
      const int* bt = seq_bt + (long)(i0 + l) * bt_width;
      const int first = max(r0, s0), total = (min(r1, s0 + c0) - first) * chunks;
      for (int e = lane; e < total; e += 64) {
        const int r = first + e / chunks, ch = e % chunks, j = k0 + r - s0;
        const unsigned short* src = cache + (((long)bt[j >> block_shift] << block_shift) + (j & mask)) * dim;
        *reinterpret_cast<u16x8*>(lat + (long)r * dim + 8 * ch) = *reinterpret_cast<const u16x8*>(src + 8 * ch);
      }
    }
    base += __builtin_amdgcn_readlane(end, 63);
  }
}

// MT: 16-token tiles per wave; 64 MT tokens of one head per workgroup.
template <int MT>
__global__ __launch_bounds__(kThreads, 2) void latent_prompt_kernel(
    unsigned short* __restrict__ out, const unsigned short* __restrict__ q, const unsigned short* __restrict__ kv,
    const unsigned short* __restrict__ lat, int lat_ld, int rot_at, const int* __restrict__ off, int rows,
    const int* __restrict__ seq_cu, const int* __restrict__ seq_ctx, int nseq, int tiles,
    const long* __restrict__ positions, const float* __restrict__ inv_freq, const unsigned short* __restrict__ proj, long proj_ld, int heads, int gate_off, bool channel_gate, float scale, int window) {
  constexpr int KL = kD / 32, KS = kQ / 32, NV = kD / 16, kTq = 64 * MT;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // [stage][keys | values | rotary parts][32]
  const int head = blockIdx.x % heads;
  int s, tok0;
  if (!find_row_tile(seq_cu, 0, nseq, kTq, tiles - 1 - (int)(blockIdx.x / heads), s, tok0)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4;
  const int r0 = seq_cu[s], n = seq_cu[s + 1] - r0, ctx = seq_ctx[s], ntok = min(kTq, n - tok0);
  const int p_first = ctx - n + tok0, hi = p_first + ntok - 1;
  const int lo = first_key(p_first, window, 0), ntiles = (hi - lo) / kKeys + 1;
  const int first = off[s] + lo - first_key(ctx - n, window, 0);   // row of key lo
  if (first < 0 || first + (hi - lo) >= rows) return;   // never, where rows is at least the sequences' sum
  const long kv_ld = 2L * heads * kD;
  // the wave's own tokens: keys it sees
  const int w_tok = 16 * MT * wave, w_any = w_tok < ntok;
  const int w_lo = first_key(p_first + w_tok, window, 0), w_hi = min(p_first + w_tok + 16 * MT - 1, hi);

  unsigned koff[2], voff[2];   // the lane's bytes past the tile's first row
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int k = 8 * wave + 4 * i + (lane >> 4);
    koff[i] = (unsigned)k * (unsigned)kv_ld * 2 + 16 * ((lane & 15) ^ key_swizzle(k));
    voff[i] = (unsigned)k * (unsigned)kv_ld * 2 + heads * kD * 2 + 16 * ((lane & 15) ^ value_swizzle(k));
  }
  const int kr = 8 * wave + (lane >> 3);
  const unsigned roff = (unsigned)(kr * lat_ld + rot_at) * 2 + 16 * ((lane & 7) ^ rot_swizzle(kr));
  const unsigned lds0 = lds_at(smem);
  const unsigned char* const kv0 = reinterpret_cast<const unsigned char*>(kv + first * kv_ld + head * kD);
  const unsigned char* const lat0 = reinterpret_cast<const unsigned char*>(lat + (long)first * lat_ld);
  auto copy = [&](int t) {
    const unsigned to = lds0 + (t % kStages) * kStage;
    const unsigned char *keys = kv0 + (long)t * kKeys * kv_ld * 2, *rot = lat0 + (long)t * kKeys * lat_ld * 2;
    if (lo + t * kKeys + kKeys - 1 <= hi) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        copy_1k(keys, koff[i], to + (8 * wave + 4 * i) * kRow);
        copy_1k(keys, voff[i], to + kHalf + (8 * wave + 4 * i) * kRow);
      }
      copy_1k(rot, roff, to + 2 * kHalf + 8 * wave * kRot * 2);
      return;
    }
    const int last = hi - lo - t * kKeys;   // keys past the last one are the last one again
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int k = 8 * wave + 4 * i + (lane >> 4);
      const unsigned back = (unsigned)(k - min(k, last)) * (unsigned)kv_ld * 2;
      copy_1k(keys, koff[i] - back, to + (8 * wave + 4 * i) * kRow);
      copy_1k(keys, voff[i] - back, to + kHalf + (8 * wave + 4 * i) * kRow);
    }
    copy_1k(rot, roff - (unsigned)(kr - min(kr, last)) * (unsigned)lat_ld * 2, to + 2 * kHalf + 8 * wave * kRot * 2);
  };
  copy(0);
  if (ntiles > 1) copy(1);
  if (ntiles > 2) copy(2);

  bool sact[MT];
  int spos[MT], s_lo[MT];
  long trow[MT];
  bf16x8 qf[MT][KS];
  f32x4 acc[MT][NV];
  f32x4 lsum[MT];    // sums of the weights that are multiplied, the same number in all four
  float m_run[MT];   // what the weights are relative to, log2 domain
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int tok = w_tok + 16 * mt + c;
    sact[mt] = tok < ntok;
    trow[mt] = r0 + tok0 + (sact[mt] ? tok : 0);
    spos[mt] = sact[mt] ? p_first + tok : -1;   // a row that does not exist sees no key
    s_lo[mt] = first_key(p_first + tok, window, 0);
    const unsigned short* src = q + (trow[mt] * heads + head) * kQ + 8 * g;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[mt][ks] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u16x8*>(src + 32 * ks));
    // the last 64 dims: entry i pairs with i + 32, angle position * inv_freq[i]
    u16x8 a = __builtin_bit_cast(u16x8, qf[mt][KL]), b = __builtin_bit_cast(u16x8, qf[mt][KL + 1]);
    const float pos = (float)positions[trow[mt]];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float sn, cs;
      sincosf(pos * inv_freq[8 * g + e], &sn, &cs);
      const float u = bf16_to_f32(a[e]), w = bf16_to_f32(b[e]);
      a[e] = f32_to_bf16(u * cs - w * sn);
      b[e] = f32_to_bf16(w * cs + u * sn);
    }
    qf[mt][KL] = __builtin_bit_cast(bf16x8, a);
    qf[mt][KL + 1] = __builtin_bit_cast(bf16x8, b);
#pragma unroll
    for (int j = 0; j < NV; ++j) acc[mt][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    m_run[mt] = -INFINITY;
    lsum[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const float unit = scale * kLog2e;
  const u32x4 ones_u = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
  const bf16x8 ones = __builtin_bit_cast(bf16x8, ones_u);
  int kat[KS], vat[NV];   // the lane's places in a tile
#pragma unroll
  for (int ks = 0; ks < KL; ++ks) kat[ks] = c * kRow + (((4 * ks + g) ^ key_swizzle(c)) << 4);
#pragma unroll
  for (int ks = KL; ks < KS; ++ks) kat[ks] = 2 * kHalf + c * kRot * 2 + (((4 * (ks - KL) + g) ^ rot_swizzle(c)) << 4);
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int k = 4 * g + (c >> 2);
    vat[j] = kHalf + k * kRow + (((2 * j + ((c & 3) >> 1)) ^ value_swizzle(k)) << 4) + 8 * (c & 1);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): the queries; the copies in flight below are this loop's own
  for (int i = 0; i < ntiles; ++i) {
    if (i + 2 < ntiles) barrier_copies<10>();   // two tiles may be in flight, five copies each
    else if (i + 1 < ntiles) barrier_copies<5>();
    else barrier_copies<0>();
    if (i + 3 < ntiles) copy(i + 3);   // into the buffer of tile i - 1, which every wave has left
    const int j0 = lo + i * kKeys;
    if (!w_any || j0 > w_hi || j0 + kKeys - 1 < w_lo) continue;   // the wave's rows see nothing of the tile
    unsigned char* tile = smem + (i % kStages) * kStage;
    f32x4 sc[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) sc[mt][0] = sc[mt][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        const bf16x8 a = __builtin_bit_cast(
            bf16x8, *reinterpret_cast<const u16x8*>(tile + kat[ks] + 16 * nt * (ks < KL ? kRow : kRot * 2)));
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
    if (j0 < w_lo || j0 + kKeys - 1 > w_hi) clear_outside(va, j0, w_lo, w_hi, g);   // a weight of 0 does not hide an infinity or a NaN
    __builtin_amdgcn_sched_barrier(0);
    bf16x8 pb[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      // lane (c, g): keys 16 nt + 4 g + e; times `unit`: log2 domain
      float v[8], mx = -INFINITY;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = sc[mt][e >> 2][e & 3];
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
    float f = l == 0.f ? 0.f : 1.f / l;
    const unsigned short* gates = proj + trow[mt] * proj_ld + gate_off;
    if (gate_off >= 0 && !channel_gate) f *= sigmoid_f(bf16_to_f32(gates[head]));
    unsigned short* dst = out + (trow[mt] * heads + head) * kD;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int d = 16 * j + 4 * g;
      u16x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        o[e] = f32_to_bf16(acc[mt][j][e] * f * (channel_gate ? sigmoid_f(bf16_to_f32(gates[head * kD + d + e])) : 1.f));
      *reinterpret_cast<u16x4*>(dst + d) = o;
    }
  }
}

}  // namespace

void launch_latent_gather(void* lat, int* off, const void* cache, int block_size, int dim, const int* seq_cu, const int* seq_ctx,
                          const int* seq_bt, int bt_width, int nseq, int rows, int window, hipStream_t s) {
  if (nseq <= 0 || rows <= 0) return;
  const int per = rows >= 4096 ? 4 : 1;
  latent_gather_kernel<<<(rows + 4 * per - 1) / (4 * per), 256, 0, s>>>(
      (unsigned short*)lat, off, (const unsigned short*)cache, __builtin_ctz(block_size), dim, seq_cu, seq_ctx, seq_bt, bt_width, nseq,
      rows, per, window);
}

bool latent_prompt_ok(int dim, int rot_dim, int vdim) { return dim == kD && rot_dim == kRot && vdim == kD; }

bool launch_latent_prompt(void* out, const void* q, const void* kv, const void* lat, int lat_ld, int rot_at, const int* off, int rows,
                          const int* seq_cu, const int* seq_ctx, int nseq, int T, const long* positions, const float* inv_freq,
                          const void* proj, long proj_ld, int heads, int gate_off, bool channel_gate, float scale, int window, hipStream_t s) {
  if (nseq <= 0 || T <= 0) return true;
  constexpr int smem = kStages * kStage;
  static_assert(smem <= 80 * 1024, "two workgroups per CU");
  auto go = [&](auto* kernel, int mt) {
    const int tiles = T / (64 * mt) + nseq;
    kernel<<<(unsigned)(tiles * heads), kThreads, smem, s>>>(
        (unsigned short*)out, (const unsigned short*)q, (const unsigned short*)kv, (const unsigned short*)lat, lat_ld, rot_at, off, rows,
        seq_cu, seq_ctx, nseq, tiles, positions, inv_freq, (const unsigned short*)proj, proj_ld, heads, gate_off, channel_gate, scale, window);
  };
  static const bool ok = allow_lds(&latent_prompt_kernel<1>, smem) && allow_lds(&latent_prompt_kernel<2>, smem);
  if (!ok) return false;
  // half as many rows per wave where 128 per workgroup would leave compute units idle
  if ((long)T * heads >= 512L * 128) go(&latent_prompt_kernel<2>, 2);
  else go(&latent_prompt_kernel<1>, 1);
  return true;
}

}  // namespace hipserve

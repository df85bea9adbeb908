// The gated delta rule of prompt portions in chunks of 16 tokens, fp32 throughout (fp32 matrix cores):
//   S_t = diag(g_t) S_{t-1} + k_t u_t^T,  u_t = beta_t (v_t - (diag(g_t) S_{t-1})^T k_t),  o_t = S_t^T q_t
// with a decay g per key channel or per head. With G_i the product of a chunk's decays up to token i and S the
// state before the chunk,
//   u_i + beta_i sum_{j<i} A_ij u_j = beta_i (v_i - S^T (G_i k_i)),   A_ij = k_i^T diag(G_i / G_j) k_j
//   o_i = S^T (G_i q_i) + sum_{j<=i} P_ij u_j,                         P_ij = q_i^T diag(G_i / G_j) k_j
//   S' = diag(G_15) S + sum_j (G_15 / G_j k_j) u_j^T
// so a chunk costs a few small matrix products instead of 16 dependent passes over the state. The ratios G_i / G_j are
// formed as products of the decays between the two tokens (never as a quotient), so strong decays only underflow.
//
// delta_chunk_prepare (a decay per channel), delta_chunk_prepare_head: everything that does not need the state, one workgroup per (head, chunk): A, P, the inverse
// M = (1 + diag(beta) A)^-1 diag(beta) by forward substitution, and W = -M (G k), U0 = M v, G q, G_15 / G k, G_15.
// delta_chunk_scan: one workgroup per (sequence, head, 16 or 32 value channels) walks the chunks: U = U0 + W S,
// o = (G q) S + P U, S = G_15 S + (G_15 / G k)^T U on mfma_f32_16x16x4f32. The state stays in registers in the
// accumulators' layout, which is also the second operand's: lane (n, g) of a 16-row tile holds rows 4 g + r of column n,
// and k step r of a product takes rows {4 g + r}.
#include "seq_common.h"
#include "hipserve/seq_kernels.h"

namespace hipserve {
namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int kC = 16;   // tokens per chunk

// Chunk `id` of the step: its sequence and first token there; false past the last one.
HS_DEVICE bool find_chunk(const int* __restrict__ seq_cu, int nseq, int id, int& s, int& t0) {
  for (s = 0; s < nseq; ++s) {
    const int nc = (seq_cu[s + 1] - seq_cu[s] + kC - 1) / kC;
    if (id < nc) {
      t0 = id * kC;
      return true;
    }
    id -= nc;
  }
  return false;
}

// Buffers per (chunk, head): W, GQ [16][DP], KT [DP][16], GE [DP], UT [VP][16], P [16][16]. The first four lie as the scan's lanes take
// them, a tile of 16 x 16 as 64 times four numbers (`in_tiles`): a load of 1 KB side by side is looked up in a quarter of the steps that
// 64 lanes take which jump from row to row. 8192 rows (4 prompts) x 16 heads, all kernels of the rule: 424 -> 401 us, 16 prompts of 200:
// 209 -> 198 (the same in delta_rule_chunk.hip, which loads less: 374 -> 372, not worth its longer places).
struct ChunkBuf {
  float *W, *GQ, *KT, *GE, *UT, *P;
};
HS_DEVICE ChunkBuf chunk_buf(float* base, long item, int DP, int VP) {
  float* p = base + item * (3L * kC * DP + DP + (long)kC * VP + kC * kC);
  ChunkBuf b;
  b.W = p;
  b.GQ = b.W + kC * DP;
  b.KT = b.GQ + kC * DP;
  b.GE = b.KT + kC * DP;
  b.UT = b.GE + DP;
  b.P = b.UT + kC * VP;
  return b;
}

// Where (a, b) of an operand lies whose lane (a % 16, g) holds b = 16 t + 4 g .. + 3 of the tile t (W, GQ: token, channel), or, with a and b
// swapped, (channel, token): tiles go along the channels.
HS_DEVICE int in_tiles(int token, int channel) {
  return ((channel >> 4) * 64 + (channel >> 2 & 3) * 16 + token) * 4 + (channel & 3);
}
HS_DEVICE int in_tiles_t(int channel, int token) {
  return ((channel >> 4) * 64 + (token >> 2) * 16 + (channel & 15)) * 4 + (token & 3);
}

// A decay per key channel. 16 DPP rows of 16 lanes: row i is token i; lane `seg` of a row owns channels 16 VD j + VD seg + e (DS in all).
template <int DS>
__global__ __launch_bounds__(256) void delta_chunk_prepare_kernel(
    float* __restrict__ base, const float* __restrict__ qk, const float* __restrict__ vv, const float* __restrict__ gg,
    const float* __restrict__ bb, const int* __restrict__ seq_cu, int nseq, int heads, int kv_heads, int dim, int vdim,
    int VP) {
  constexpr int DP = 16 * DS, VD = DS < 4 ? DS : 4, NJ = DS / VD;
  __shared__ __attribute__((aligned(16))) float sk[kC][DP], sg[kC][DP];
  __shared__ __attribute__((aligned(16))) float sMt[kC][kC];   // [j][i]
  __shared__ float sA[kC][kC + 1], sP[kC][kC + 1], sb[kC];
  int s, t0;
  if (!find_chunk(seq_cu, nseq, blockIdx.y, s, t0)) return;
  const int h = blockIdx.x, tid = threadIdx.x, row = tid >> 4, seg = tid & 15;
  const int r0 = seq_cu[s] + t0, nt = min(kC, seq_cu[s + 1] - r0);
  const int nqk = kv_heads * dim, nv = heads * vdim, kh = h / (heads / kv_heads);
  const ChunkBuf out = chunk_buf(base, (long)blockIdx.y * heads + h, DP, VP);
  float vcol[kC];   // this thread's value channel (tid < vdim), all tokens: loaded early, used at the end
#pragma unroll
  for (int j = 0; j < kC; ++j) vcol[j] = (tid < vdim && j < nt) ? vv[(long)(r0 + j) * nv + h * vdim + tid] : 0.f;
  float xk[NJ][VD], xq[NJ][VD], g0[NJ][VD];
  const bool in = row < nt;
  const long t = r0 + (in ? row : 0);
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int c = 16 * VD * j + VD * seg;
    const float* pq = qk + t * 2 * nqk + kh * dim + c;
    const float* pg = gg + (t * heads + h) * dim + c;
    if (VD == 4 && dim % 4 == 0) {   // four channels are inside together, rows are 16-byte aligned
      f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = a, g = {1.f, 1.f, 1.f, 1.f};
      if (in && c < dim) {
        a = *reinterpret_cast<const f32x4*>(pq + nqk);
        b = *reinterpret_cast<const f32x4*>(pq);
        g = *reinterpret_cast<const f32x4*>(pg);
      }
#pragma unroll
      for (int e = 0; e < VD; ++e) { xk[j][e] = a[e]; xq[j][e] = b[e]; g0[j][e] = g[e]; }
    } else {
#pragma unroll
      for (int e = 0; e < VD; ++e) {
        const bool ok = in && c + e < dim;
        xk[j][e] = ok ? pq[nqk + e] : 0.f;
        xq[j][e] = ok ? pq[e] : 0.f;
        g0[j][e] = ok ? pg[e] : 1.f;
      }
    }
    Row<float, VD>::st(&sk[row][c], xk[j]);
    Row<float, VD>::st(&sg[row][c], g0[j]);
  }
  if (seg == 0) sb[row] = in ? bb[t * heads + h] : 0.f;
  for (int i = tid; i < kC * (kC + 1); i += 256) { (&sA[0][0])[i] = 0.f; (&sP[0][0])[i] = 0.f; }
  __syncthreads();
  float yk[NJ][VD], ge[NJ][VD];
  float p = 0.f;
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int e = 0; e < VD; ++e) {
      yk[j][e] = xk[j][e];
      ge[j][e] = g0[j][e];
      p = __builtin_fmaf(xq[j][e], xk[j][e], p);
    }
  p = row_sum(p);
  if (seg == 0) sP[row][row] = p;
  // back through the earlier tokens: xk, xq = k_i, q_i times the decays of tokens m + 1 .. i
  for (int m = row - 1; m >= 0; --m) {
    float a = 0.f;
    p = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      float g[VD], k[VD];
      Row<float, VD>::ld(&sg[m + 1][16 * VD * j + VD * seg], g);
      Row<float, VD>::ld(&sk[m][16 * VD * j + VD * seg], k);
#pragma unroll
      for (int e = 0; e < VD; ++e) {
        xk[j][e] *= g[e];
        xq[j][e] *= g[e];
        a = __builtin_fmaf(xk[j][e], k[e], a);
        p = __builtin_fmaf(xq[j][e], k[e], p);
      }
    }
    a = row_sum(a);   // the 16 lanes of a row take the same trips
    p = row_sum(p);
    if (seg == 0) { sA[row][m] = a; sP[row][m] = p; }
  }
  // forward: yk = k_i times the decays of the later tokens; row 0 also forms the product of all of them
  for (int m = row + 1; m < kC; ++m) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      float g[VD];
      Row<float, VD>::ld(&sg[m][16 * VD * j + VD * seg], g);
#pragma unroll
      for (int e = 0; e < VD; ++e) { yk[j][e] *= g[e]; ge[j][e] *= g[e]; }
    }
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int c = 16 * VD * j + VD * seg;
    float g[VD];
    Row<float, VD>::ld(&sg[0][c], g);
#pragma unroll
    for (int e = 0; e < VD; ++e) { xk[j][e] *= g[e]; xq[j][e] *= g[e]; }   // G_i k_i, G_i q_i
    Row<float, VD>::st(out.GQ + in_tiles(row, c), xq[j]);
    if (row == 0) Row<float, VD>::st(out.GE + c, ge[j]);
  }
  __syncthreads();   // sk, sg are read, sA is written
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    Row<float, VD>::st(&sg[row][16 * VD * j + VD * seg], xk[j]);
    Row<float, VD>::st(&sk[row][16 * VD * j + VD * seg], yk[j]);
  }
  if (tid < kC) {   // column tid of M: (1 + diag(beta) A) x = beta e
    float x[kC];
#pragma unroll
    for (int i = 0; i < kC; ++i) {
      float r = 0.f;
#pragma unroll
      for (int j = 0; j < i; ++j) r = __builtin_fmaf(sA[i][j], x[j], r);
      x[i] = sb[i] * ((i == tid ? 1.f : 0.f) - r);
      sMt[tid][i] = x[i];
    }
  }
  out.P[64 * (seg & 3) + 16 * (seg >> 2) + row] = sP[row][seg];   // by k step and lane of the scan
  __syncthreads();
  // W = M (G k)
  float w[NJ][VD];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int e = 0; e < VD; ++e) w[j][e] = 0.f;
  for (int m = 0; m <= row; ++m) {
    const float f = sMt[m][row];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      float k[VD];
      Row<float, VD>::ld(&sg[m][16 * VD * j + VD * seg], k);
#pragma unroll
      for (int e = 0; e < VD; ++e) w[j][e] = __builtin_fmaf(f, k[e], w[j][e]);
    }
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
#pragma unroll
    for (int e = 0; e < VD; ++e) w[j][e] = -w[j][e];
    Row<float, VD>::st(out.W + in_tiles(row, 16 * VD * j + VD * seg), w[j]);
  }
  // G_15 / G k, transposed
  for (int i = tid; i < DP * (kC / 4); i += 256) {
    const int c = i >> 2, q = 4 * (i & 3);
    *reinterpret_cast<f32x4*>(out.KT + in_tiles_t(c, q)) = f32x4{sk[q][c], sk[q + 1][c], sk[q + 2][c], sk[q + 3][c]};
  }
  // U0 = M v, transposed, a value channel per thread
  for (int v = tid; v < VP; v += 256) {
    float u[kC];
#pragma unroll
    for (int i = 0; i < kC; ++i) u[i] = 0.f;
#pragma unroll
    for (int j = 0; j < kC; ++j) {
      const float x = v == tid ? vcol[j] : (v < vdim && j < nt ? vv[(long)(r0 + j) * nv + h * vdim + v] : 0.f);
#pragma unroll
      for (int i = j; i < kC; ++i) u[i] = __builtin_fmaf(sMt[j][i], x, u[i]);
    }
#pragma unroll
    for (int q = 0; q < kC; q += 4)
      *reinterpret_cast<f32x4*>(out.UT + in_tiles_t(v, q)) = f32x4{u[q], u[q + 1], u[q + 2], u[q + 3]};
  }
}

// The same for a decay per head, where all that the channels differ in are products of matrices: the pairs k_i k_j and q_i k_j on the
// matrix cores, a quarter of the channels per wave, times the decays between the two tokens; W and U0 with M as an operand, whose results lie as
// the scan's lanes take them. What bounds it are the bytes, 34 KB written per head and chunk: 8192 rows (4 prompts) x 16 heads of 128 x 128 with a
// walk through the tokens per row, as above, 126 us, now 90; 16 prompts of 200 56 -> 39. Errors against 64 bits beside the token by token scan's, over
// 100 - 700 tokens, weak and strong decays: states 0.82 - 1.33 of them (0.87 - 1.34 before), outputs 0.96 - 1.28 (1.11 - 1.40): the pairs of
// queries and keys and the products of decays are formed in 64 bits and rounded once (in 32 bits, four chains per wave, 0.99 - 1.43 and 5 us less).
template <int DS>
__global__ __launch_bounds__(256) void delta_chunk_prepare_head_kernel(
    float* __restrict__ base, const float* __restrict__ qk, const float* __restrict__ vv, const float* __restrict__ gg,
    const float* __restrict__ bb, const int* __restrict__ seq_cu, int nseq, int heads, int kv_heads, int dim, int vdim, int VP) {
  constexpr int DP = 16 * DS, LD = DP + 4, NK = DS < 4 ? DS : 4, KS = DP / 4 / NK;   // waves that share the channels; k steps of each
  __shared__ __attribute__((aligned(16))) float sk[kC][LD], sq[kC][LD];
  __shared__ __attribute__((aligned(16))) f32x4 part[NK][64];
  __shared__ __attribute__((aligned(16))) f64x4 partq[NK][64];
  __shared__ float sA[kC][kC + 1], sM[kC][kC + 4], sMG[kC][kC + 4];
  __shared__ float sg[kC], sb[kC], sG[kC], sE[kC];   // decays, rates, products up to a token and after it
  int s, t0;
  if (!find_chunk(seq_cu, nseq, blockIdx.y, s, t0)) return;
  const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4;
  const int r0 = seq_cu[s] + t0, nt = min(kC, seq_cu[s + 1] - r0);
  const int nqk = kv_heads * dim, nv = heads * vdim, kh = h / (heads / kv_heads);
  const ChunkBuf out = chunk_buf(base, (long)blockIdx.y * heads + h, DP, VP);
  // a value tile's second operand: four tokens of a channel
  auto values = [&](int t, f32x4& v) {
    const int ch = 16 * t + c;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = vv[(long)(r0 + min(4 * r + g, nt - 1)) * nv + h * vdim + min(ch, vdim - 1)];
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = 4 * r + g < nt && ch < vdim ? v[r] : 0.f;
  };
  f32x4 v0 = {0.f, 0.f, 0.f, 0.f}, v1 = v0;   // of the wave's first two tiles, loaded early
  if (16 * wave < VP) values(wave, v0);
  if (16 * (wave + 4) < VP) values(wave + 4, v1);
  const bool vec = dim % 4 == 0;
  for (int i = tid; i < kC * DP / 4; i += 256) {
    const int row = i / (DP / 4), ch = i % (DP / 4) * 4;
    f32x4 k = {0.f, 0.f, 0.f, 0.f}, q = k;
    if (row < nt && ch < dim) {
      const float* p = qk + (long)(r0 + row) * 2 * nqk + kh * dim + ch;
      if (vec) {
        q = *reinterpret_cast<const f32x4*>(p);
        k = *reinterpret_cast<const f32x4*>(p + nqk);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (ch + e < dim) { q[e] = p[e]; k[e] = p[nqk + e]; }
      }
    }
    *reinterpret_cast<f32x4*>(&sk[row][ch]) = k;
    *reinterpret_cast<f32x4*>(&sq[row][ch]) = q;
  }
  if (tid < kC) {
    const long at = (long)(r0 + min(tid, nt - 1)) * heads + h;
    const float d = gg[at], beta = bb[at];
    sg[tid] = tid < nt ? d : 1.f;
    sb[tid] = tid < nt ? beta : 0.f;
  }
  __syncthreads();
  if (wave < NK) {   // lane (c, g): rows 4 g + r of column c, in 64 bits rows 4 r + g
    f32x4 a[4] = {};
    f64x4 p = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int st = 0; st < KS; ++st) {
      const int ch = 4 * (wave * KS + st) + g;
      const float k = sk[c][ch], q = sq[c][ch];
      a[st & 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(k, k, a[st & 3], 0, 0, 0);
      p = __builtin_amdgcn_mfma_f64_16x16x4f64((double)q, (double)k, p, 0, 0, 0);
    }
    part[wave][lane] = (a[0] + a[1]) + (a[2] + a[3]);
    partq[wave][lane] = p;
  }
  // the products of the decays between two tokens, never a quotient; row i, column j
  const int i = tid >> 4, j = tid & 15;
  double exact = 1.0;   // rounded once: a factor that all channels share
#pragma unroll
  for (int m = kC - 1; m > 0; --m) exact *= m <= i && m > j ? (double)sg[m] : 1.0;
  const float ratio = (float)exact;
  if (j == 0) sG[i] = (float)(exact * (double)sg[0]);
  if (i == kC - 1) sE[j] = ratio;
  __syncthreads();
  {
    float a = 0.f;
    double p = 0.0;
#pragma unroll
    for (int w = 0; w < NK; ++w) {
      a += reinterpret_cast<const float*>(&part[w][(i >> 2) * 16 + j])[i & 3];
      p += reinterpret_cast<const double*>(&partq[w][(i & 3) * 16 + j])[i >> 2];
    }
    sA[i][j] = j < i ? a * ratio : 0.f;
    out.P[64 * (j & 3) + 16 * (j >> 2) + i] = j <= i ? (float)(p * exact) : 0.f;   // by k step and lane of the scan
  }
  __syncthreads();
  if (tid < kC) {   // column tid of M: (1 + diag(beta) A) x = beta e
    float x[kC];
    const float G = sG[tid];
#pragma unroll
    for (int i = 0; i < kC; ++i) {
      float r = 0.f;
#pragma unroll
      for (int j = 0; j < i; ++j) r = __builtin_fmaf(sA[i][j], x[j], r);
      x[i] = sb[i] * ((i == tid ? 1.f : 0.f) - r);
      sM[i][tid] = x[i];
      sMG[i][tid] = -x[i] * G;
    }
  } else if (tid >= 64) {   // G q, G_15 / G k as they lie in tiles, by the other waves
    for (int t = wave - 1; t < DS; t += 3) {
      f32x4 q = *reinterpret_cast<const f32x4*>(&sq[c][16 * t + 4 * g]), k;
      q *= sG[c];
#pragma unroll
      for (int r = 0; r < 4; ++r) k[r] = sk[4 * g + r][16 * t + c] * sE[4 * g + r];
      *reinterpret_cast<f32x4*>(out.GQ + (t * 64 + lane) * 4) = q;
      *reinterpret_cast<f32x4*>(out.KT + (t * 64 + lane) * 4) = k;
    }
    for (int ch = tid - 64; ch < DP; ch += 192) out.GE[ch] = sG[kC - 1];
  }
  __syncthreads();
  float mg[4], m[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    mg[r] = sMG[c][4 * r + g];
    m[r] = sM[c][4 * r + g];
  }
  for (int t = wave; t < DS; t += 4) {
    f32x4 w = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) w = __builtin_amdgcn_mfma_f32_16x16x4f32(sk[4 * r + g][16 * t + c], mg[r], w, 0, 0, 0);
    *reinterpret_cast<f32x4*>(out.W + (t * 64 + lane) * 4) = w;
  }
  for (int t = wave; 16 * t < VP; t += 4) {
    f32x4 v, u = {0.f, 0.f, 0.f, 0.f};
    if (t == wave) v = v0;
    else if (t == wave + 4) v = v1;
    else values(t, v);
#pragma unroll
    for (int r = 0; r < 4; ++r) u = __builtin_amdgcn_mfma_f32_16x16x4f32(m[r], v[r], u, 0, 0, 0);
    *reinterpret_cast<f32x4*>(out.UT + (t * 64 + lane) * 4) = u;
  }
}

// NW waves with TPW 16-row state tiles each, NC tiles of 16 value channels per workgroup. U0 is loaded by one wave per tile, every wave does
// its share of the k steps of P U, and the outputs are summed with the next chunk's exchange. What bounds it is the chain from chunk to
// chunk: a wave's matrix instructions (50 of 32 cycles at 128 x 128 and two tiles, 0.67 us) and the exchange of W S through LDS, which
// goes round while (G q) S runs; loads go out among the products, two chunks ahead (four: 184 us for 169). Prompts x tokens, 16 heads of
// 128 x 128: 4 x 2048 197 -> 167 us, 6 x 1300 243 -> 169, 16 x 200 92 -> 59. One tile per workgroup where two leave CUs idle, and of smaller heads
// always: 1 x 300 30 -> 16 us (two tiles: 25), 2 x 600 57 -> 30, 4 x 2048 of 64 x 64 128 -> 76 (103), of 32 x 32 122 -> 57 (87). A tile's U0 is
// added in the same wave either way, so that the bits do not depend on it.
// W S and P U are summed from 0, and U0 and (G q) S added to the sums: as the start of the sums they would make every product round
// at their size (512 tokens, mean decay 0.47, against 64 bits: state 6.0e-8, with U0 as the start 1.1e-7; outputs 8.6e-8, 1.4e-7).
constexpr int kAhead = 2;   // chunks in flight
template <int TPW, int NW, int NC>
__global__ __launch_bounds__(64 * NW, 2) void delta_chunk_scan_kernel(
    float* __restrict__ o, float* __restrict__ S, float* __restrict__ base, const int* __restrict__ seq_cu,
    const int* __restrict__ seq_ctx, const int* __restrict__ seq_state, int heads, int dim, int vdim, int VP) {
  constexpr int DP = 16 * TPW * NW, KPW = 4 / NW, RPW = 4 * NC / NW;   // k steps of P U and rows of the read-out per wave
  static_assert(NW % NC == 0 && 4 * NC % NW == 0, "a wave per tile for U0, whole rows per wave");
  static_assert(kAhead % 2 == 0, "a place of the ring has one parity");
  __shared__ __attribute__((aligned(16))) f32x4 sums[2][2][NC][NW][64];   // [chunk parity][U | the last chunk's o][tile][wave][lane]
  const int s = blockIdx.z, h = blockIdx.x, v0 = 16 * NC * blockIdx.y;
  const int r0 = seq_cu[s], n = seq_cu[s + 1] - r0;
  if (n <= 0) return;
  int first = 0;   // the sequence's first chunk in the step
  for (int i = 0; i < s; ++i) first += (seq_cu[i + 1] - seq_cu[i] + kC - 1) / kC;
  const int nc = (n + kC - 1) / kC;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, g = lane >> 4;
  const unsigned starts = NC == 1 ? blockIdx.y & 1 : 0;   // U0 of an even tile is added to the first wave's sums, of an odd one to the second's
  const bool odd = threadIdx.x & 64, high = threadIdx.x & 128;   // the wave's bits as lane masks: selects, not branches
  const int nv = heads * vdim, mine = wave % NC, row0 = (wave / NC) * RPW;
  const bool carried = seq_ctx[s] - n > 0;
  float* Sp = S + ((long)seq_state[s] * heads + h) * dim * vdim;
  f32x4 st[NC][TPW] = {};
  // Operands, each loaded kAhead chunks ahead as soon as its registers are free. Loads and stores of the loop are
  // unconditional (past the end the last chunk is loaded again, rows and columns that do not exist are outside the
  // store's bounds), so that the wait for an operand never has to cover the younger loads behind it.
  struct Ops {
    f32x4 W[TPW], Q[TPW], K[TPW], E[TPW], U;
    float p[KPW];
  } ops[kAhead];
  const unsigned kE = 3 * kC * DP * 4, kU = kE + DP * 4, kP = kU + kC * VP * 4, bytes = kP + kC * kC * 4;   // where GE, UT, P start
  const unsigned w_at = (wave * TPW * 64 + lane) * 16, e_at = kE + (16 * wave * TPW + 4 * g) * 4,
                 u_at = kU + (min(v0 / 16 + mine, VP / 16 - 1) * 64 + lane) * 16, p_at = kP + (64 * wave * KPW + lane) * 4;
  const char* next = reinterpret_cast<const char*>(base) + ((long)first * heads + h) * bytes;   // the next chunk to be loaded
  int left = nc - 1;
  auto from = [&] { return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(next), 0, bytes, 0x00020000); };
  auto get = [&](unsigned at) { return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(from(), at, 0, 0)); };
  auto fetch = [&](Ops& x, int part) {
    if (part == 0) {
#pragma unroll
      for (int i = 0; i < TPW; ++i) x.W[i] = get(w_at + 1024 * i);
      x.U = get(u_at);
    } else if (part == 1) {
#pragma unroll
      for (int i = 0; i < TPW; ++i) {
        x.Q[i] = get(kC * DP * 4 + w_at + 1024 * i);
        x.E[i] = get(e_at + 64 * i);
      }
    } else {
#pragma unroll
      for (int i = 0; i < TPW; ++i) x.K[i] = get(2 * kC * DP * 4 + w_at + 1024 * i);
#pragma unroll
      for (int i = 0; i < KPW; ++i) x.p[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(from(), p_at + 256 * i, 0, 0));
      next += left > 0 ? (long)heads * bytes : 0;
      --left;
    }
  };
  auto step_of = [&](const f32x4& v, int i) {   // the wave's i-th k step
    if constexpr (NW == 1) return v[i];
    else if constexpr (NW == 2) return odd ? v[2 + i] : v[i];
    else return high ? (odd ? v[3] : v[2]) : odd ? v[1] : v[0];
  };
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 os[NC] = {};
  const unsigned out_at = v0 + 16 * mine + c < vdim ? ((4 * g + row0) * nv + h * vdim + v0 + 16 * mine + c) * 4 : 0x80000000u;
  // sum of the waves' parts, pairs first
  auto sum_of = [&](const f32x4* p) {
    if constexpr (NW == 1) return p[0];
    else if constexpr (NW == 2) return p[0] + p[64];
    else return (p[0] + p[64]) + (p[128] + p[192]);
  };
  auto read_out = [&](int ci, int buf) {   // the outputs of chunk ci from the sums in sums[buf]
    const auto to = __builtin_amdgcn_make_buffer_rsrc(o + (long)(r0 + ci * kC) * nv, 0, (min(kC, n - ci * kC) & ~(ci >> 31)) * nv * 4, 0x00020000);
#pragma unroll
    for (int e = 0; e < RPW; ++e) {
      float y = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) y += reinterpret_cast<const float*>(&sums[buf][1][mine][w][lane])[row0 + e];
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, y), to, out_at + 4 * e * nv, 0, 0);
    }
  };
  auto step = [&](Ops& x, int ci, int buf) {
    f32x4 us[NC], qs[NC], u[NC];
#pragma unroll
    for (int t = 0; t < NC; ++t) us[t] = qs[t] = zero;
#pragma unroll
    for (int b = 0; b < TPW; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int t = 0; t < NC; ++t) us[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.W[b][r], st[t][b][r], us[t], 0, 0, 0);
#pragma unroll
    for (int t = 0; t < NC; ++t) sums[buf][1][t][wave][lane] = os[t];
    __builtin_amdgcn_sched_barrier(0);
    auto queries = [&](int b, int r) {
#pragma unroll
      for (int t = 0; t < NC; ++t) qs[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.Q[b][r], st[t][b][r], qs[t], 0, 0, 0);
    };
    queries(0, 0);
    queries(0, 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < NC; ++t) sums[buf][0][t][wave][lane] = us[t] + (NW == 1 || (!high && odd == (starts + t)) ? x.U : zero);
    fetch(x, 0);
    __builtin_amdgcn_sched_barrier(0);
    queries(0, 2);
    queries(0, 3);
#pragma unroll
    for (int b = 1; b < TPW; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) queries(b, r);
#pragma unroll
    for (int t = 0; t < NC; ++t)
#pragma unroll
      for (int b = 0; b < TPW; ++b) st[t][b] *= x.E[b];
    fetch(x, 1);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();   // the other parity's rows are read before a wave comes here again
#pragma unroll
    for (int t = 0; t < NC; ++t) u[t] = sum_of(&sums[buf][0][t][0][lane]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int b = 0; b < TPW; ++b)
#pragma unroll
        for (int t = 0; t < NC; ++t) st[t][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.K[b][r], u[t][r], st[t][b], 0, 0, 0);
#pragma unroll
    for (int t = 0; t < NC; ++t) {
      os[t] = zero;
#pragma unroll
      for (int i = 0; i < KPW; ++i) os[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.p[i], step_of(u[t], i), os[t], 0, 0, 0);
      os[t] += qs[t];
    }
    fetch(x, 2);
    read_out(ci - 1, buf);
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int i = 0; i < kAhead; ++i)
    for (int part = 0; part < 3; ++part) fetch(ops[i], part);
  // The carried state, rows and columns that do not exist as zeros of a place that does: a branch for each element came with a wait for the one
  // before (200 sequences of one row x 16 heads in a step, all kernels of the rule, 792 -> 638 us; 50 of 64 rows 287 -> 258).
  if (carried) {
#pragma unroll
    for (int t = 0; t < NC; ++t)
#pragma unroll
      for (int b = 0; b < TPW; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          st[t][b][r] = Sp[(long)min(16 * (wave * TPW + b) + 4 * g + r, dim - 1) * vdim + min(v0 + 16 * t + c, vdim - 1)];
#pragma unroll
    for (int t = 0; t < NC; ++t)
#pragma unroll
      for (int b = 0; b < TPW; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          st[t][b][r] = 16 * (wave * TPW + b) + 4 * g + r < dim && v0 + 16 * t + c < vdim ? st[t][b][r] : 0.f;
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): the loop's own waits then count the loop's loads only
  int ci = 0;
#pragma nounroll
  for (; ci + kAhead <= nc; ci += kAhead) {   // no exit in between: a wait would cover the loads of the shortest way round
#pragma unroll
    for (int i = 0; i < kAhead; ++i) step(ops[i], ci + i, i & 1);
  }
#pragma unroll
  for (int i = 0; i < kAhead - 1; ++i)
    if (ci + i < nc) step(ops[i], ci + i, i & 1);
#pragma unroll
  for (int t = 0; t < NC; ++t) sums[nc & 1][1][t][wave][lane] = os[t];
  __syncthreads();
  read_out(nc - 1, nc & 1);
#pragma unroll
  for (int t = 0; t < NC; ++t)
#pragma unroll
    for (int b = 0; b < TPW; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = 16 * (wave * TPW + b) + 4 * g + r;
        if (k < dim && v0 + 16 * t + c < vdim) Sp[(long)k * vdim + v0 + 16 * t + c] = st[t][b][r];
      }
}

int padded(int dim) { return dim <= 16 ? 16 : dim <= 32 ? 32 : dim <= 64 ? 64 : 128; }

}  // namespace

int delta_chunk_max_dim() { return 128; }
int delta_chunk_bound(int T, int nseq) { return T / kC + nseq; }

long delta_chunk_floats(int T, int nseq, int heads, int dim, int vdim) {
  const long DP = padded(dim), VP = (vdim + 15) / 16 * 16;
  return delta_chunk_bound(T, nseq) * (long)heads * (3 * kC * DP + DP + kC * VP + kC * kC);
}

void launch_delta_chunk(float* o, float* S, float* buf, const float* qk, const float* vv, const float* gg,
                        const float* bb, const int* seq_cu, const int* seq_ctx, const int* seq_state, int nseq, int T,
                        int heads, int kv_heads, int dim, int vdim, bool channel, hipStream_t s) {
  const int VP = (vdim + 15) / 16 * 16;
  dim3 pgrid(heads, delta_chunk_bound(T, nseq));
#define HS_DC(DS, TPW, NW, NC)                                                                                             \
  do {                                                                                                                 \
    if (channel)                                                                                                       \
      delta_chunk_prepare_kernel<DS><<<pgrid, 256, 0, s>>>(buf, qk, vv, gg, bb, seq_cu, nseq, heads, kv_heads, dim,  \
                                                                 vdim, VP);                                            \
    else                                                                                                               \
      delta_chunk_prepare_head_kernel<DS><<<pgrid, 256, 0, s>>>(buf, qk, vv, gg, bb, seq_cu, nseq, heads, kv_heads, dim, vdim, VP); \
    delta_chunk_scan_kernel<TPW, NW, NC><<<dim3(heads, (VP + 16 * NC - 1) / (16 * NC), nseq), 64 * NW, 0, s>>>(            \
        o, S, buf, seq_cu, seq_ctx, seq_state, heads, dim, vdim, VP);                                                      \
  } while (0)
  switch (padded(dim)) {
    case 16: HS_DC(1, 1, 1, 1); break;
    case 32: HS_DC(2, 1, 2, 1); break;
    case 64: HS_DC(4, 1, 4, 1); break;
    default:
      if (heads * ((VP + 31) / 32) * nseq < 256) HS_DC(8, 2, 4, 1);
      else HS_DC(8, 2, 4, 2);   // two tiles per workgroup where such workgroups are one per CU
  }
#undef HS_DC
}

}  // namespace hipserve

// The generalized delta rule of prompt portions in chunks of 16 tokens, heads of 64, fp32 throughout (fp32 matrix cores):
//   S_t = diag(w_t) S_{t-1} - a_t x_t^T + k_t v_t^T,  x_t = S_{t-1}^T u_t,  o_t = S_t^T r_t
// (delta_scan.hip: w = exp(-e^-1/2 sigmoid(decay)), u = unit(k), a = sigmoid(a) u). With D_ij the product of the decays of
// tokens i .. j, S the state before the chunk and strictly lower A_ij = u_i^T D_(j+1)(i-1) a_j, B_ij with k_j for a_j,
//   X = (1 + A)^-1 (D_0(i-1) u_i S + B V)
//   O = D_0i r_i S - Pa X + Pk V,   Pa_ij = r_i^T D_(j+1)i a_j (j <= i), Pk_ij with k_j
//   S' = D_0,15 S - (D_(j+1),15 a_j)^T X + (D_(j+1),15 k_j)^T V
// so that 16 dependent passes over the state become a few products. A decay is at least exp(-e^-1/2) = 0.545, a chunk's product
// at least 6e-5: the inner ratios are quotients of products from the chunk's start, and the matrix cores form all pairs.
//
// delta_rule_chunk_prepare: all that does not need the state, one workgroup per (head, chunk), straight from the projection.
// delta_rule_chunk_scan: one workgroup per (sequence, head, 16 or 32 value channels) walks the chunks as in delta_chunk.hip, with
// U = -X: U = U0 + W S (W = -(1 + A)^-1 U), O = R S + Pa U + Pk V, S = E S + KA U + KK V.
// A product over the chunk would carry a NaN or an infinity of one token's inputs to the tokens before it (0 times it), so such
// inputs take part as zeros, and where a chunk has some the scan ends with a walk that writes NaN: to the outputs of a token whose r
// is not finite (F), and to the outputs and the state of a column from the token on (B) whose value is not finite, or, all columns,
// whose k is not finite or a pre-activation of which is NaN (infinite ones saturate).
// What bounds it: the prepared operands (6816 floats per head and chunk) are written and read once, and the scan's products.
// 8192 rows (4 prompts) x 32 heads: rows prepared one by one and scanned token by token (five row vectors through LDS for
// every 4 state elements of a lane) took 126 + 700 us; this 171 + 144 (188 before the products of the
// decays were a channel per lane of one wave, three swaps and seven selects for each).
// Errors against 64 bits, over 32 .. 2048 tokens, fresh and carried states, strong and weak decays: state 5.8e-8 - 6.4e-8 (token by
// token 6.3e-8 - 7.0e-8), outputs before their norm 7.2e-8 - 7.9e-8 (9.2e-8 - 9.8e-8). What it takes: decays and their products
// in 64 bits, rounded once into the operands (else 7.9e-8 for the state); Pa and Pk summed in 64 bits and the larger part of an output added
// last (else 1.3e-7); tokens that go from the oldest to the newest into the state (else 1.3e-7).
#include "seq_common.h"
#include "hipserve/seq_kernels.h"

namespace hipserve {
namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int kC = 16, kD = 64, kLd = kD + 4;   // tokens per chunk; key and value channels of a head; LDS row

// Buffers per (chunk, head): W, R [16][64], KA, KK [64][16], U0, V [64][16], E [64], Pa, Pk [16][16], F [16], B [64], any [1]
struct Buf {
  float *W, *R, *KA, *KK, *U, *V, *E, *Pa, *Pk, *F, *B, *any;
};
constexpr long kBuf = 6L * kC * kD + 2 * kD + 2 * kC * kC + kC + 16;
HS_DEVICE Buf buf_of(float* base, long item) {
  float* p = base + item * kBuf;
  constexpr int m = kC * kD;
  return Buf{p,         p + m,          p + 2 * m,           p + 3 * m, p + 4 * m, p + 5 * m, p + 6 * m, p + 6 * m + kD,
             p + 6 * m + kD + kC * kC, p + 6 * m + kD + 2 * kC * kC, p + 6 * m + kD + 2 * kC * kC + kC,
             p + 6 * m + 2 * kD + 2 * kC * kC + kC};
}

// Where a token stands in the buffers' rows and columns: a lane's four values 4 g + r are the tokens 4 r + g, so that the k steps
// r of a sum over the tokens take the oldest four first. Their decayed parts are small, and the sum rounds to the size it
// has by then, as token by token.
HS_DEVICE int place(int t) { return 4 * (t & 3) + (t >> 2); }

// exp(-e^-1/2 s) for s in 0 .. 1, a token's decay, in 64 bits: rounded to 32 bits, the decays would cost the state as much as the
// recurrence's own roundings. Taylor polynomial of exp around the middle, up to x^7: |x| <= e^-1/2 / 2 leaves 2e-9.
HS_DEVICE double decay_of(float s) {
  constexpr double c[7] = {1.0, 1.0, 1.0 / 2, 1.0 / 6, 1.0 / 24, 1.0 / 120, 1.0 / 720};
  const double x = __builtin_fma((double)s, -0.6065306597126334, 0.3032653298563167);
  double p = 1.0 / 5040.0;
#pragma unroll
  for (int i = 6; i >= 0; --i) p = __builtin_fma(p, x, c[i]);
  return p * 0.738403149974731;   // exp(-e^-1/2 / 2)
}

HS_DEVICE f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
HS_DEVICE f32x4 mfma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

__global__ __launch_bounds__(256) void delta_rule_chunk_prepare_kernel(
    float* __restrict__ base, const unsigned short* __restrict__ proj, long ld, const float* __restrict__ wl,
    const float* __restrict__ a_b, const float* __restrict__ w0, const int* __restrict__ seq_cu, int nseq, int heads) {
  __shared__ __attribute__((aligned(16))) float su[kC][kLd], sr[kC][kLd], sa[kC][kLd], sk[kC][kLd], sv[kC][kLd];
  // The products of the decays before and after a token, then, where those are, KA and KK, and A, B and M: 39 KB for four workgroups per CU.
  constexpr int kBytes = kC * kD * 8, kAt = 2 * kC * kLd * 4;
  __shared__ __attribute__((aligned(16))) unsigned char pool[kAt + kBytes];
  static_assert(kAt >= kBytes && 3 * kC * 20 * 4 <= kBytes, "two regions");
  auto sbefore = reinterpret_cast<double(*)[kD]>(pool), safter = reinterpret_cast<double(*)[kD]>(pool + kAt);
  auto sx = reinterpret_cast<float(*)[kLd]>(pool), sy = sx + kC;   // KA, KK
  auto sA = reinterpret_cast<float(*)[20]>(pool + kAt), sB = sA + kC, sM = sB + kC;
  __shared__ float sf[2][kC];   // NaN: what reaches every column of a token's, its r, is not finite
  __shared__ int sv_bad[kD];    // a column's first value that is not finite
  int s, t0;
  if (!find_row_tile(seq_cu, 0, nseq, kC, blockIdx.y, s, t0)) return;
  const int h = blockIdx.x, tid = threadIdx.x, row = tid >> 4, ch = 4 * (tid & 15), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r0 = seq_cu[s] + t0, nt = min(kC, seq_cu[s + 1] - r0), N = heads * kD;
  const Buf out = buf_of(base, (long)blockIdx.y * heads + h);
  const bool in = row < nt;
  if (tid < kD) sv_bad[tid] = kC;
  f32x4 ka, kk;
  {
    const long t = r0 + (in ? row : 0);
    const int c = h * kD + ch;
    float r[4], k[4], v[4], a[4], w[4], ab[4], wb[4], u[4];
    const unsigned short* p = proj + t * ld + c;
    Row<unsigned short, 4>::ld(p, r);
    Row<unsigned short, 4>::ld(p + N, k);
    Row<unsigned short, 4>::ld(p + 2 * N, v);
    Row<unsigned short, 4>::ld(p + 3 * N, a);
    Row<float, 4>::ld(wl + t * N + c, w);
    Row<float, 4>::ld(a_b + c, ab);
    Row<float, 4>::ld(w0 + c, wb);
    float ss = 0.f, f = 0.f, fr = 0.f;
    double dec[4];
    bool lost[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      ss += k[e] * k[e];
      a[e] = sigmoid_f(a[e] + ab[e]);
      dec[e] = decay_of(sigmoid_f(w[e] + wb[e]));
      f += (k[e] - k[e]) + (a[e] - a[e]) + (float)(dec[e] - dec[e]);   // 0 or NaN
      fr += r[e] - r[e];
      lost[e] = in && !(v[e] - v[e] == 0.f);
    }
    f = in ? row_sum(f) : 0.f;
    fr = in ? row_sum(fr) : 0.f;
    if (ch == 0) { sf[0][row] = f; sf[1][row] = fr; }
    const bool use = in && f == 0.f;
    const float inv = 1.f / sqrtf(row_sum(ss) + 1e-6f);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      u[e] = use ? k[e] * inv : 0.f;
      a[e] = use ? a[e] * u[e] : 0.f;
      if (!use) { dec[e] = 1.0; k[e] = 0.f; }
      if (!use || lost[e]) v[e] = 0.f;
      if (!use || fr != 0.f) r[e] = 0.f;
    }
    // the products of the decays of the chunk's earlier and later tokens, a channel per lane of a wave that has little else to do
#pragma unroll
    for (int e = 0; e < 4; ++e) sbefore[row][ch + e] = dec[e];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (lost[e]) atomicMin(&sv_bad[ch + e], row);
    if (wave == 1) {
      double d[kC], p = 1.0;
#pragma unroll
      for (int i = 0; i < kC; ++i) d[i] = sbefore[i][lane];
#pragma unroll
      for (int i = 0; i < kC; ++i) {
        sbefore[i][lane] = p;
        p *= d[i];
      }
      p = 1.0;
#pragma unroll
      for (int i = kC - 1; i >= 0; --i) {
        safter[i][lane] = p;
        p *= d[i];
      }
    }
    __syncthreads();
    double before[4], after[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      before[e] = sbefore[row][ch + e];
      after[e] = safter[row][ch + e];
    }
    f32x4 upto, U, R, A, K, V;
#pragma unroll
    for (int e = 0; e < 4; ++e) {   // each rounded once
      const double d = before[e] * dec[e], seed = (double)__builtin_amdgcn_rcpf((float)d);
      const double inv = seed * __builtin_fma(-d, seed, 2.0);
      upto[e] = (float)d;
      U[e] = (float)(u[e] * before[e]);
      R[e] = (float)(r[e] * d);
      A[e] = (float)(a[e] * inv);
      K[e] = (float)(k[e] * inv);
      V[e] = v[e];
      ka[e] = (float)(a[e] * after[e]);
      kk[e] = (float)(k[e] * after[e]);
    }
    *reinterpret_cast<f32x4*>(&su[row][ch]) = U;
    *reinterpret_cast<f32x4*>(&sr[row][ch]) = R;
    *reinterpret_cast<f32x4*>(&sa[row][ch]) = A;
    *reinterpret_cast<f32x4*>(&sk[row][ch]) = K;
    *reinterpret_cast<f32x4*>(&sv[row][ch]) = V;
    *reinterpret_cast<f32x4*>(out.R + place(row) * kD + ch) = R;
    if (row == kC - 1) *reinterpret_cast<f32x4*>(out.E + ch) = upto;
    __syncthreads();   // the products are read
    *reinterpret_cast<f32x4*>(&sx[row][ch]) = ka;
    *reinterpret_cast<f32x4*>(&sy[row][ch]) = kk;
  }
  if (wave == 1) {
    const unsigned long all = __ballot(lane < kC && sf[0][lane & 15] != 0.f), rs = __ballot(lane < kC && sf[1][lane & 15] != 0.f);
    const int first = min(sv_bad[lane], all ? __builtin_ctzll(all) : kC);
    out.B[lane] = (float)first;
    const bool any = __any(first < kC) || rs != 0;
    if (lane < kC) out.F[lane] = sf[1][lane];
    if (lane == 0) *out.any = any ? 1.f : 0.f;
  }
  // all pairs of tokens: wave 0 A, 1 B in four chains, 2 Pa, 3 Pk in 64 bits (in 32, the outputs' largest error; A and B in 64
  // bits too: 18 us more and no smaller an error); lane (c, g) gets rows 4 g + r of column c, in 64 bits rows 4 r + g
  const int c = lane & 15, g = lane >> 4;
  {
    const float(*x)[kLd] = wave < 2 ? su : sr;
    const float(*y)[kLd] = wave & 1 ? sk : sa;
    f32x4 xa[4], ya[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      xa[q] = ld4(&x[c][16 * q + 4 * g]);
      ya[q] = ld4(&y[c][16 * q + 4 * g]);
    }
    if (wave < 2) {
      f32x4 d[4] = {};
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) d[e] = mfma(xa[q][e], ya[q][e], d[e]);
      const f32x4 t = (d[0] + d[1]) + (d[2] + d[3]);
#pragma unroll
      for (int r = 0; r < 4; ++r) (wave == 0 ? sA : sB)[4 * g + r][c] = c < 4 * g + r ? t[r] : 0.f;
    } else {
      f64x4 d = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) d = __builtin_amdgcn_mfma_f64_16x16x4f64((double)xa[q][e], (double)ya[q][e], d, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r)   // by k step and lane of the scan
        (wave == 2 ? out.Pa : out.Pk)[64 * (c >> 2) + 16 * (c & 3) + place(4 * r + g)] = c <= 4 * r + g ? (float)d[r] : 0.f;
    }
  }
  __syncthreads();
  if (wave == 0) {
    if (lane < kC) {   // column `lane` of M = (1 + A)^-1
      float x[kC];
#pragma unroll
      for (int i = 0; i < kC; ++i) {
        float r = i == lane ? 1.f : 0.f;
#pragma unroll
        for (int j = 0; j < i; ++j) r = __builtin_fmaf(-sA[i][j], x[j], r);
        x[i] = r;
        sM[i][lane] = r;
      }
    }
  } else {
    for (int i = tid - 64; i < 2 * kD * 4; i += 192) {   // KA, KK transposed
      const int k = i >> 2 & (kD - 1), q = i & 3;
      const float(*x)[kLd] = i < kD * 4 ? sx : sy;
      *reinterpret_cast<f32x4*>((i < kD * 4 ? out.KA : out.KK) + k * kC + 4 * q) = f32x4{x[q][k], x[q + 4][k], x[q + 8][k], x[q + 12][k]};
    }
  }
  __syncthreads();
  // W = M U, and U0 = -(M B) V with (M B)^T = B^T M^T, whose accumulators are the next product's first operand
  const int col = 16 * wave + c;
  const f32x4 m = ld4(&sM[place(c)][4 * g]);
  f32x4 wv = {0.f, 0.f, 0.f, 0.f}, mb = wv, u0 = wv, v;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    wv = mfma(m[r], su[4 * g + r][col], wv);
    mb = mfma(sB[4 * g + r][place(c)], m[r], mb);
    v[r] = sv[4 * r + g][col];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) u0 = mfma(-mb[r], v[r], u0);
#pragma unroll
  for (int r = 0; r < 4; ++r) out.W[(4 * g + r) * kD + col] = -wv[r];
  *reinterpret_cast<f32x4*>(out.U + col * kC + 4 * g) = u0;
  *reinterpret_cast<f32x4*>(out.V + col * kC + 4 * g) = v;
}

// Four waves with 16 state rows each, kTiles tiles of 16 value channels. Nothing but the wave's own rows is loaded: of U0 (the start of
// a tile's sums) and V each one tile per wave, which goes round with the sums; each wave does one of the four k steps of Pa U and Pk V, and
// the outputs are summed with the next chunk's exchange. What bounds it is the chain from chunk to chunk: 36 matrix instructions of
// a wave's own (0.5 us), the exchange of W S through LDS, and the loads' way into the CU. So W S comes first and goes round
// while R S and KK V run, V is exchanged a chunk early, loads go out among the products, and two chunks ahead are enough (four: 256
// registers and 146 us). 4 prompts of 2048 x 32 heads: 186 -> 144 us, 6 of 1300: 225 -> 142, 16 of 200: 83 -> 53.
// One tile per workgroup where two leave CUs idle: 1 prompt of 300 26 -> 15 us (two tiles: 21), 2 of 600 50 -> 27, 4 of 2048 166. A tile's
// sums start in the same wave either way, so that the bits do not depend on it.
constexpr int kNW = 4, kAhead = 2;   // kAhead: chunks in flight
template <int kTiles>
__global__ __launch_bounds__(64 * kNW, 2) void delta_rule_chunk_scan_kernel(
    float* __restrict__ o, float* __restrict__ S, float* __restrict__ base, const int* __restrict__ seq_cu,
    const int* __restrict__ seq_ctx, const int* __restrict__ seq_state, int heads) {
  static_assert(kNW == 4 && kTiles <= 2, "U0 and V: a wave per tile each");
  static_assert(kAhead % 2 == 0, "a place of the ring has one parity");
  __shared__ __attribute__((aligned(16))) f32x4 sums[2][2][kTiles][kNW][64];   // [chunk parity][U | the last chunk's O]
  __shared__ __attribute__((aligned(16))) f32x4 vals[2][kNW][64];              // [chunk parity] U0, V
  const int s = blockIdx.z, h = blockIdx.x;
  const int r0 = seq_cu[s], n = seq_cu[s + 1] - r0;
  if (n <= 0) return;
  int first = 0;   // the sequence's first chunk in the step
  for (int i = 0; i < s; ++i) first += (seq_cu[i + 1] - seq_cu[i] + kC - 1) / kC;
  const int nc = (n + kC - 1) / kC;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, g = lane >> 4;
  const bool odd = threadIdx.x & 64, high = threadIdx.x & 128;   // the wave's bits as lane masks: selects, not branches
  const int N = heads * kD, k0 = 16 * wave, col0 = 16 * kTiles * blockIdx.y, half = wave >> 1;
  const int mine = kTiles == 2 ? wave & 1 : 0, row0 = kTiles == 2 ? 2 * half : wave;
  const unsigned starts = kTiles == 2 ? 0 : blockIdx.y & 1;   // a tile's sums start with U0 in wave (column / 16) % 2
  const bool carried = seq_ctx[s] - n > 0;
  float* Sp = S + ((long)seq_state[s] * heads + h) * kD * kD + col0 + c;
  f32x4 st[kTiles] = {};
  if (carried)
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) st[t][r] = Sp[(k0 + 4 * g + r) * kD + 16 * t];
  // Operands, each loaded kAhead chunks ahead as soon as its registers are free. The loop's loads and stores are unconditional
  // (past the end the last chunk again, rows that do not exist outside the store's bounds), so that the wait for an operand never
  // covers the younger loads behind it.
  struct Ops {
    f32x4 W, R, KA, KK, E, X;
    float pa, pk;
  } ops[kAhead];
  constexpr unsigned kM = kC * kD * sizeof(float), kE = 6 * kM, kP = kE + kD * 4;   // bytes of an operand, where E and Pa start
  const unsigned rows = (c * kD + k0 + 4 * g) * 4, cols = ((k0 + c) * kC + 4 * g) * 4, states = kE + (k0 + 4 * g) * 4,
                 vals_at = (4 + half) * kM + ((col0 + 16 * mine + c) * kC + 4 * g) * 4, pair = kP + (64 * wave + lane) * 4;
  const long stride = heads * kBuf * (long)sizeof(float);
  const char* chunks = reinterpret_cast<const char*>(base + ((long)first * heads + h) * kBuf);
  const char* next = chunks;   // the next chunk to be loaded
  int left = nc - 1;
  auto from = [&] { return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(next), 0, kBuf * (int)sizeof(float), 0x00020000); };
  auto get = [&](unsigned at) { return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(from(), at, 0, 0)); };
  auto one = [&](unsigned at) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(from(), at, 0, 0)); };
  auto fetch = [&](Ops& x, int part) {
    if (part == 0) { x.W = get(rows); x.X = get(vals_at); }
    if (part == 1) { x.R = get(kM + rows); x.E = get(states); }
    if (part == 2) x.KK = get(3 * kM + cols);
    if (part == 3) {
      x.KA = get(2 * kM + cols);
      x.pa = one(pair);
      x.pk = one(kC * kC * 4 + pair);
      next += left > 0 ? stride : 0;
      --left;
    }
  };
  auto of_wave = [&](const f32x4& v) { return high ? (odd ? v[3] : v[2]) : odd ? v[1] : v[0]; };
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 os[kTiles] = {}, v[kTiles];
  float vr[kTiles];   // the wave's k step of v
  // the outputs of chunk ci from the sums in sums[buf]: every wave kTiles rows of four
  const unsigned out_at = ((4 * row0 + g) * N + h * kD + col0 + 16 * mine + c) * 4;
  auto read_out = [&](int ci, int buf) {
    float x[kNW][kTiles];
#pragma unroll
    for (int w = 0; w < kNW; ++w)
#pragma unroll
      for (int e = 0; e < kTiles; ++e) x[w][e] = reinterpret_cast<const float*>(&sums[buf][1][mine][w][lane])[row0 + e];
    const auto to = __builtin_amdgcn_make_buffer_rsrc(o + (long)(r0 + ci * kC) * N, 0, (min(kC, n - ci * kC) & ~(ci >> 31)) * N * 4, 0x00020000);
#pragma unroll
    for (int e = 0; e < kTiles; ++e)
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, (x[0][e] + x[1][e]) + (x[2][e] + x[3][e])), to, out_at + 16 * e * N, 0, 0);
  };
  auto step = [&](Ops& x, const Ops& y, int ci, int buf) {
    f32x4 us[kTiles], u[kTiles], rs[kTiles] = {}, sa[kTiles] = {};
    float pv[kTiles];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) pv[t] = vr[t];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) us[t] = !high && odd == (starts + t) ? x.X : zero;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int t = 0; t < kTiles; ++t) us[t] = mfma(x.W[r], st[t][r], us[t]);
#pragma unroll
    for (int t = 0; t < kTiles; ++t) sums[buf][1][t][wave][lane] = os[t];
    vals[buf ^ 1][wave][lane] = y.X;   // the next chunk's
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int t = 0; t < kTiles; ++t) rs[t] = mfma(x.R[r], st[t][r], rs[t]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < kTiles; ++t) sums[buf][0][t][wave][lane] = us[t];
    fetch(x, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 2; r < 4; ++r)
#pragma unroll
      for (int t = 0; t < kTiles; ++t) rs[t] = mfma(x.R[r], st[t][r], rs[t]);
#pragma unroll
    for (int t = 0; t < kTiles; ++t) st[t] *= x.E;
    fetch(x, 1);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int t = 0; t < kTiles; ++t) st[t] = mfma(x.KK[r], v[t][r], st[t]);
    fetch(x, 2);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();   // the other parity's rows are read before a wave comes here again
    f32x4 part[kTiles][kNW];
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
      for (int w = 0; w < kNW; ++w) part[t][w] = sums[buf][0][t][w][lane];
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
      u[t] = part[t][0];
#pragma unroll
      for (int w = 1; w < kNW; ++w) u[t] += part[t][w];
    }
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
      v[t] = vals[buf ^ 1][2 + t][lane];
      vr[t] = reinterpret_cast<const float*>(&vals[buf ^ 1][2 + t][lane])[wave];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int t = 0; t < kTiles; ++t) sa[t] = mfma(x.KA[r], u[t][r], sa[t]);
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
      os[t] = mfma(x.pa, of_wave(u[t]), rs[t]);   // the larger part last: its roundings are the outputs'
      os[t] = mfma(x.pk, pv[t], os[t]);
    }
    fetch(x, 3);
    read_out(ci - 1, buf);
#pragma unroll
    for (int t = 0; t < kTiles; ++t) st[t] += sa[t];
    __builtin_amdgcn_sched_barrier(0);
  };
  // 1 if a token's inputs were not finite
  float any = 0.f;
  for (int ci = threadIdx.x; ci < nc; ci += 64 * kNW) any = fmaxf(any, *reinterpret_cast<const float*>(chunks + ci * stride + kP + (2 * kC * kC + kC + kD) * 4));
#pragma unroll
  for (int i = 0; i < kAhead; ++i) for (int part = 0; part < 4; ++part) fetch(ops[i], part);
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): the loop's own waits then count the loop's loads only
  vals[0][wave][lane] = ops[0].X;
  __syncthreads();
#pragma unroll
  for (int t = 0; t < kTiles; ++t) {
    v[t] = vals[0][2 + t][lane];
    vr[t] = reinterpret_cast<const float*>(&vals[0][2 + t][lane])[wave];
  }
  int ci = 0;
#pragma nounroll
  for (; ci + kAhead <= nc; ci += kAhead) {   // no exit in between: a wait would cover the loads of the shortest way round
#pragma unroll
    for (int i = 0; i < kAhead; ++i) step(ops[i], ops[(i + 1) % kAhead], ci + i, i & 1);
  }
#pragma unroll
  for (int i = 0; i < kAhead - 1; ++i)
    if (ci + i < nc) step(ops[i], ops[i + 1], ci + i, i & 1);
#pragma unroll
  for (int t = 0; t < kTiles; ++t) sums[nc & 1][1][t][wave][lane] = os[t];
  any = __syncthreads_or(any != 0.f);
  read_out(nc - 1, nc & 1);
#pragma unroll
  for (int t = 0; t < kTiles; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) Sp[(long)(k0 + 4 * g + r) * kD + 16 * t] = st[t][r];
  if (any == 0.f) return;
  __syncthreads();   // the outputs and the state are written
  const float nan = __builtin_nanf("");
  const int tid = threadIdx.x, col = col0 + tid % (16 * kTiles), part = tid / (16 * kTiles), parts = 64 * kNW / (16 * kTiles);
  bool lost = false;
  for (int ci = 0; ci < nc; ++ci) {
    const Buf b = buf_of(base, (long)(first + ci) * heads + h);
    const float from = b.B[col];
    for (int i = part; i < min(kC, n - ci * kC); i += parts)
      if (lost || i >= from || b.F[i] != 0.f) o[(long)(r0 + ci * kC + i) * N + h * kD + col] = nan;
    lost |= from < kC;
  }
  if (lost)
    for (int k = part; k < kD; k += parts) S[((long)seq_state[s] * heads + h) * kD * kD + (long)k * kD + col] = nan;
}

}  // namespace

bool delta_rule_chunk_ok(int heads, int dim, const void* proj, long ld) {
  return dim == kD && ld % 4 == 0 && reinterpret_cast<uintptr_t>(proj) % 8 == 0;
}
long delta_rule_chunk_floats(int T, int nseq, int heads) { return (T / kC + nseq) * (long)heads * kBuf; }

void launch_delta_rule_chunk(float* o, float* S, float* buf, const void* proj, long ld, const float* wl, const float* a_b,
                             const float* w0, const int* seq_cu, const int* seq_ctx, const int* seq_state, int nseq, int T,
                             int heads, hipStream_t s) {
  delta_rule_chunk_prepare_kernel<<<dim3(heads, T / kC + nseq), 256, 0, s>>>(buf, (const unsigned short*)proj, ld, wl, a_b, w0,
                                                                             seq_cu, nseq, heads);
  const bool few = heads * (kD / 32) * nseq < 256;   // two tiles per workgroup where such workgroups are one per CU
  (few ? delta_rule_chunk_scan_kernel<1> : delta_rule_chunk_scan_kernel<2>)<<<dim3(heads, kD / (few ? 16 : 32), nseq), 64 * kNW, 0, s>>>(
      o, S, buf, seq_cu, seq_ctx, seq_state, heads);
}

}  // namespace hipserve

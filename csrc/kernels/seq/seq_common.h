#pragma once
#include "hipserve/common.h"

namespace hipserve {

template <typename T> HS_DEVICE float ldf(const T* p, long i);
template <> HS_DEVICE float ldf<unsigned short>(const unsigned short* p, long i) { return bf16_to_f32(p[i]); }
template <> HS_DEVICE float ldf<float>(const float* p, long i) { return p[i]; }
template <typename T> HS_DEVICE void stf(T* p, long i, float v);
template <> HS_DEVICE void stf<unsigned short>(unsigned short* p, long i, float v) { p[i] = f32_to_bf16(v); }
template <> HS_DEVICE void stf<float>(float* p, long i, float v) { p[i] = v; }

// Kernel arguments from byte `at` of the argument block on, loaded where this stands and not before: the compiler loads arguments
// at the kernel's entry and waits for them there, which takes 0.26 us of a small launch (a second, dependent load of them 0.34). The ones that the first loads need come first and reach
// the kernel in scalar registers (the build's flags ask for it).
template <typename T> using LateArgs = const __attribute__((address_space(4))) T*;
template <typename T> HS_DEVICE LateArgs<T> late_args(int at) {
  unsigned long p = reinterpret_cast<unsigned long>(__builtin_amdgcn_kernarg_segment_ptr()) + at;
  asm volatile("" : "+s"(p));
  return reinterpret_cast<LateArgs<T>>(p);
}

// V consecutive elements of a row as fp32 (V > 1: the address is aligned to V elements)
template <typename T, int V> struct Row;
template <> struct Row<float, 1> {
  static HS_DEVICE void ld(const float* p, float (&v)[1]) { v[0] = *p; }
  static HS_DEVICE void st(float* p, const float (&v)[1]) { *p = v[0]; }
};
template <> struct Row<float, 2> {
  static HS_DEVICE void ld(const float* p, float (&v)[2]) { const float2 a = *reinterpret_cast<const float2*>(p); v[0] = a.x; v[1] = a.y; }
  static HS_DEVICE void st(float* p, const float (&v)[2]) { *reinterpret_cast<float2*>(p) = float2{v[0], v[1]}; }
};
template <> struct Row<float, 4> {
  static HS_DEVICE void ld(const float* p, float (&v)[4]) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = a[i];
  }
  static HS_DEVICE void st(float* p, const float (&v)[4]) { *reinterpret_cast<f32x4*>(p) = f32x4{v[0], v[1], v[2], v[3]}; }
};
template <> struct Row<unsigned short, 1> {
  static HS_DEVICE void ld(const unsigned short* p, float (&v)[1]) { v[0] = bf16_to_f32(*p); }
  static HS_DEVICE void st(unsigned short* p, const float (&v)[1]) { *p = f32_to_bf16(v[0]); }
};
template <> struct Row<unsigned short, 4> {
  static HS_DEVICE void ld(const unsigned short* p, float (&v)[4]) {
    const u16x4 a = *reinterpret_cast<const u16x4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = bf16_to_f32(a[i]);
  }
  static HS_DEVICE void st(unsigned short* p, const float (&v)[4]) {
    u16x4 a;
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = f32_to_bf16(v[i]);
    *reinterpret_cast<u16x4*>(p) = a;
  }
};
template <> struct Row<float, 8> {
  static HS_DEVICE void ld(const float* p, float (&v)[8]) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) { v[i] = a[i]; v[4 + i] = b[i]; }
  }
  static HS_DEVICE void st(float* p, const float (&v)[8]) {
    *reinterpret_cast<f32x4*>(p) = f32x4{v[0], v[1], v[2], v[3]};
    *reinterpret_cast<f32x4*>(p + 4) = f32x4{v[4], v[5], v[6], v[7]};
  }
};
template <> struct Row<unsigned short, 8> {
  static HS_DEVICE void ld(const unsigned short* p, float (&v)[8]) {
    const u16x8 a = *reinterpret_cast<const u16x8*>(p);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = bf16_to_f32(a[i]);
  }
  static HS_DEVICE void st(unsigned short* p, const float (&v)[8]) {
    u16x8 a;
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = f32_to_bf16(v[i]);
    *reinterpret_cast<u16x8*>(p) = a;
  }
};

// exp(-|x|) and 1 / (1 + exp(-|x|)), which neither overflow nor need the scaled division: e is the hardware's exp2 of the rounded
// product t = -|x| log2(e) times exp of what the rounding left, -(|x| + t ln 2), and the hardware's reciprocal r of 1 + e takes one
// Newton step from 1 - r - e r (1 - r is exact from r = 1/2 on, which r falls below by its last bit at most).
HS_DEVICE float sigmoid_of_abs(float x, float& e) {
  const float a = __builtin_elementwise_minimum(fabsf(x), 104.f);   // exp(-104) is 0 in 32 bits; NaN stays
  const float t = a * -1.44269502f;
  const float lost = fmaf(t, -1.90465432e-9f, fmaf(t, 0.693147182f, a));
  e = __builtin_amdgcn_exp2f(t);
  e = fmaf(-lost, e, e);
  const float r = __builtin_amdgcn_rcpf(1.f + e);
  return fmaf(fmaf(-e, r, 1.f - r), r, r);
}
// 1 / (1 + exp(-x)) in 14 instructions, 18 where the Newton step carried what 1 + e lost and the product's rounding was found beside
// log2(e). Relative error against 64 bits in units of 2^-24, of either (every 8th number, octave by octave the same), rms over x in [-16, 16]: 0.59
// (largest 3.35, below -16 3.45); of 1.f / (1.f + expf(-x)) 2.95 (12.7).
HS_DEVICE float sigmoid_f(float x) {
  float e;
  const float r = sigmoid_of_abs(x, e);
  return x < 0.f ? e * r : r;
}

HS_DEVICE float tanh_fast(float x) {  // 1 - 2 / (e^2x + 1); saturates cleanly at both ends
  return 1.f - 2.f * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(x * 2.88539008177792681f) + 1.f);
}

// Sum over the 16 lanes of a DPP row; every lane of the row gets it.
HS_DEVICE float row_sum(float v) {
  v = dpp_step<0xB1, 0xf, false>(v);   // quad_perm [1, 0, 3, 2]
  v = dpp_step<0x4E, 0xf, false>(v);   // quad_perm [2, 3, 0, 1]
  v = dpp_step<0x141, 0xf, false>(v);  // row_half_mirror
  return dpp_step<0x140, 0xf, false>(v);  // row_mirror
}

// Workgroup `wg` of those that cut every sequence seq0 .. seq1 - 1 of a step into tiles of tq rows: its sequence and first row
// (the same in every lane); false past the last one. A lane per sequence: a walk over them would wait for every row count.
HS_DEVICE bool find_row_tile(const int* __restrict__ seq_cu, int seq0, int seq1, int tq, int wg, int& s, int& tok0) {
  const int lane = threadIdx.x & 63;
  int base = 0;
  for (int i0 = seq0; i0 < seq1; i0 += 64) {
    const int i = i0 + lane;
    const int nt = i < seq1 ? (seq_cu[i + 1] - seq_cu[i] + tq - 1) / tq : 0;
    int end = nt;   // inclusive sum over the lanes
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(end, o, 64);
      if (lane >= o) end += v;
    }
    const unsigned long long mine = __ballot(wg >= base + end - nt && wg < base + end);
    if (mine != 0) {
      const int l = __builtin_ctzll(mine);
      s = i0 + l;
      tok0 = (wg - base - (__builtin_amdgcn_readlane(end, l) - __builtin_amdgcn_readlane(nt, l))) * tq;
      return true;
    }
    base += __builtin_amdgcn_readlane(end, 63);
  }
  return false;
}

// Row `wg` of the sequences seq0 .. seq1 - 1: its sequence and its place there; false past the last row. Decode rows, one per
// sequence, need no search.
HS_DEVICE bool find_row(const int* __restrict__ seq_cu, int seq0, int seq1, int wg, int& s, int& tok0) {
  s = seq0 + wg;
  tok0 = 0;
  if (s < seq1 && seq_cu[s] - seq_cu[seq0] == wg && seq_cu[s + 1] - seq_cu[s] == 1) return true;
  return find_row_tile(seq_cu, seq0, seq1, 1, wg, s, tok0);
}

// First key (behind the kept ones) that position pos sees: its window's, its chunk's, or the sequence's first.
HS_DEVICE int first_key(int pos, int window, int chunk) {
  return chunk > 0 ? pos - pos % chunk : window > 0 ? max(0, pos - window + 1) : 0;
}

// g sigmoid(1.702 g) (u + 1) of g = min(gate, limit), u = clamp(up, -limit, limit)
HS_DEVICE float clamped_glu_f(float g, float u, float limit) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g * sigmoid_f(1.702f * g) * (u + 1.f);
}

}  // namespace hipserve

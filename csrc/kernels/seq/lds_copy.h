// Copies from memory straight into LDS, for kernels that multiply cache rows from there (latent_attention_dma.hip,
// window_attention_dma.hip).
#pragma once
#include "seq_common.h"

namespace hipserve {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4* lds_s16x4;

// All LDS and vector memory operations issued so far are done, then every wave of the workgroup is here.
HS_DEVICE void barrier_all() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// 1 KB from the lanes' addresses to LDS, 16 bytes per lane side by side, asynchronously. Written out because the compiler
// would otherwise wait for every copy in flight before the next transposing read; the waits are the callers' barrier_all.
// A copy takes its place in LDS from m0 and must not follow a scalar write of m0 directly: one wait state, which the
// compiler does not add inside an asm block.
HS_DEVICE void copy_1k(const unsigned short* src, unsigned lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(__builtin_amdgcn_readfirstlane(lds)), "v"(src) : "m0", "memory");
}
// The same from a uniform base and the lanes' byte offsets.
HS_DEVICE void copy_1k(const unsigned char* base, unsigned off, unsigned lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(lds)), "v"(off), "s"(base) : "m0", "memory");
}
// Where a pointer into LDS points, for copy_1k: once, since turning a generic pointer into an offset costs a test.
HS_DEVICE unsigned lds_at(const unsigned char* p) {
  return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) unsigned char*)p;
}
// The same for LDS operations alone: copies into LDS may still be in flight.
HS_DEVICE void barrier_lds() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Largest of the values of the lanes c, c + 16, c + 32, c + 48, in all of them (row and half swaps of the vector unit).
HS_DEVICE float max_of_rows(float x) {
  const unsigned u = __builtin_bit_cast(unsigned, x);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const float y = fmaxf(__builtin_bit_cast(float, (unsigned)a[0]), __builtin_bit_cast(float, (unsigned)a[1]));
  const unsigned w = __builtin_bit_cast(unsigned, y);
  const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  return fmaxf(__builtin_bit_cast(float, (unsigned)b[0]), __builtin_bit_cast(float, (unsigned)b[1]));
}

// Waits until no more than N of the wave's copies are in flight (they land in order), then for every wave of the workgroup.
template <int N> HS_DEVICE void barrier_copies() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// The parts of a value operand (lane (c, g): keys j0 + 16 (e / 4) + 4 g + e % 4) that belong to keys before `lo`, as zeros: a weight of
// 0 does not hide an infinity or a NaN.
template <int N> HS_DEVICE void clear_below(bf16x8 (&va)[N], int j0, int lo, int g) {
  u32x4 keep;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int j = j0 + 16 * (r >> 1) + 4 * g + 2 * (r & 1);
    keep[r] = (j >= lo ? 0x0000ffffu : 0u) | (j + 1 >= lo ? 0xffff0000u : 0u);
  }
#pragma unroll
  for (int i = 0; i < N; ++i) va[i] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, va[i]) & keep);
}

HS_DEVICE unsigned pack2(float a, float b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{a, b}), bf16x2));
}

template <typename F>
inline bool allow_lds(F* fn, size_t bytes) {   // more dynamic LDS than the default limit, once per kernel
  return bytes <= 64 * 1024 ||
         hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) == hipSuccess;
}

}  // namespace hipserve

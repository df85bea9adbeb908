// Residual update + grouped RMSNorm of the layer-list decoders, one workgroup per token row:
//   r = residual + ls1 * mix (ls1 null: 1) + ls2 * (1/top) * sum_j y[pair_slot[t*top + j]] + extra     (fp32, written back)
//   out = r / sqrt(mean over the element's group of r^2 + eps) * w
// The row is split into `groups` equal consecutive parts with their own mean square. The MoE
// combine (rows of the expert-sorted y picked through pair_slot) and the embedding re-added at
// the start of a loop pass (`extra`) ride along, so one launch sits between two layers. With a
// table the row starts as the embedding of its id instead of the residual. `mix` may be 32-bit sums over parts of a product's K
// (mix_parts of [T, H]), which are added up first: a product of a few rows then fills the chip with workgroups of a part each.
#include "seq_common.h"
#include "hipserve/seq_kernels.h"

namespace hipserve {
namespace {

constexpr int kNT = 256;

// Rows whose length and group length are multiples of V: the row stays in registers (N vectors of V elements per
// thread) between the update and the norm, and every load but the expert rows' is issued before the first use. A
// prompt step is bound by memory, a decode step (a workgroup or two per XCD) by the latency of its loads: the element
// loop below waits for them once per 256 elements and again for the squares. 8192 rows x 2048, bf16: 59.5 -> 41.0 us
// (4.9 TB/s), with two expert rows 113 -> 55 us; 1 row: 5.8 -> 3.2 us, with two expert rows 8.2 -> 3.8 us (an empty kernel: 3.1).
// PARTS: `mix` comes in 32-bit parts; a kernel of its own, since a decode step's launches wait for their code as well (one row of 2048
// with two expert rows in a captured step 4.1 us, 4.8 with the parts' code in it).
template <typename T, int V, int N, bool PARTS>
__global__ __launch_bounds__(kNT) void scaled_add_group_rmsnorm_vec_kernel(
    T* __restrict__ out, float* __restrict__ residual, const float* __restrict__ w, int H, int groups, float eps,
    const void* __restrict__ mix_, int mix_parts, const float* __restrict__ ls1, const T* __restrict__ y,
    const int* __restrict__ pair_slot, int top, const float* __restrict__ ls2, const T* __restrict__ extra, const T* __restrict__ table,
    const long* __restrict__ ids, long table_rows) {
  extern __shared__ float sm[];  // groups > 1: [H / V] sums of squares, then [groups] inverse rms
  __shared__ float red[16];
  const long t = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const T* mix = PARTS ? nullptr : static_cast<const T*>(mix_);
  const float* part = PARTS ? static_cast<const float*>(mix_) + t * H : nullptr;
  float* r = residual + t * H;
  long id = 0;
  if (table != nullptr) id = ids[t];
  const bool known = id >= 0 && id < table_rows;   // an id outside the table gives a row of NaN, as no row is read
  float v[N][V], wv[N][V];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int e = (tid + i * kNT) * V;
    if (e < H) {
      if (table == nullptr) Row<float, V>::ld(r + e, v[i]);
      else if (known) Row<T, V>::ld(table + id * H + e, v[i]);
      Row<float, V>::ld(w + e, wv[i]);
    }
    if (e >= H || (table != nullptr && !known))
#pragma unroll
      for (int k = 0; k < V; ++k) v[i][k] = e < H ? __builtin_nanf("") : 0.f;
  }
  if (mix != nullptr) {
    float a[N][V], b[N][V];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int e = (tid + i * kNT) * V;
      if (e < H) {
        Row<T, V>::ld(mix + t * H + e, a[i]);
        if (ls1 != nullptr) Row<float, V>::ld(ls1 + e, b[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
      if ((tid + i * kNT) * V < H)
#pragma unroll
        for (int k = 0; k < V; ++k) v[i][k] += ls1 != nullptr ? a[i][k] * b[i][k] : a[i][k];
  }
  if constexpr (PARTS) {
    // loads before the first use again: up to kAhead parts, the last one in place of those that do not exist
    constexpr int kAhead = N <= 2 ? 4 : 2;
    const long rows = (long)gridDim.x * H;   // elements of a part
    float f[N][V], a[kAhead][N][V], b[N][V];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int e = (tid + i * kNT) * V;
#pragma unroll
      for (int k = 0; k < V; ++k) f[i][k] = 0.f;
      if (e < H) {
#pragma unroll
        for (int j = 0; j < kAhead; ++j) Row<float, V>::ld(part + min(j, mix_parts - 1) * rows + e, a[j][i]);
        if (ls1 != nullptr) Row<float, V>::ld(ls1 + e, b[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
      if ((tid + i * kNT) * V < H)
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
#pragma unroll
          for (int k = 0; k < V; ++k) f[i][k] += j < mix_parts ? a[j][i][k] : 0.f;
    for (int j = kAhead; j < mix_parts; ++j)
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int e = (tid + i * kNT) * V;
        if (e < H) {
          Row<float, V>::ld(part + j * rows + e, a[0][i]);
#pragma unroll
          for (int k = 0; k < V; ++k) f[i][k] += a[0][i][k];
        }
      }
#pragma unroll
    for (int i = 0; i < N; ++i)
      if ((tid + i * kNT) * V < H)
#pragma unroll
        for (int k = 0; k < V; ++k) v[i][k] += ls1 != nullptr ? f[i][k] * b[i][k] : f[i][k];
  }
  if (y != nullptr) {
    float f[N][V], a[N][V], b[N][V];
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int k = 0; k < V; ++k) f[i][k] = 0.f;
    for (int j = 0; j < top; j += 2) {   // two expert rows in flight
      const bool two = j + 1 < top;
      const T* y0 = y + (long)pair_slot[t * top + j] * H;
      const T* y1 = two ? y + (long)pair_slot[t * top + j + 1] * H : y0;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int e = (tid + i * kNT) * V;
        if (e < H) {
          Row<T, V>::ld(y0 + e, a[i]);
          Row<T, V>::ld(y1 + e, b[i]);
        }
      }
#pragma unroll
      for (int i = 0; i < N; ++i)
        if ((tid + i * kNT) * V < H)
#pragma unroll
          for (int k = 0; k < V; ++k) {
            f[i][k] += a[i][k];
            if (two) f[i][k] += b[i][k];
          }
    }
    const float wtop = 1.f / (float)top;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int e = (tid + i * kNT) * V;
      if (e < H) {
        Row<float, V>::ld(ls2 + e, b[i]);
#pragma unroll
        for (int k = 0; k < V; ++k) v[i][k] += f[i][k] * wtop * b[i][k];
      }
    }
  }
  if (extra != nullptr) {
    float a[V];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int e = (tid + i * kNT) * V;
      if (e < H) {
        Row<T, V>::ld(extra + t * H + e, a);
#pragma unroll
        for (int k = 0; k < V; ++k) v[i][k] += a[k];
      }
    }
  }
  const bool changed = table != nullptr || mix_ != nullptr || y != nullptr || extra != nullptr;
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int e = (tid + i * kNT) * V;
    float q = 0.f;
    if (e < H) {
      if (changed) Row<float, V>::st(r + e, v[i]);
#pragma unroll
      for (int k = 0; k < V; ++k) q += v[i][k] * v[i][k];
      if (groups > 1) sm[e / V] = q;
    }
    ss += q;
  }
  const int gs = H / groups;
  float inv1 = 0.f;
  float* ginv = sm + H / V;
  if (groups == 1) {
    inv1 = 1.f / sqrtf(block_sum(ss, red) / (float)H + eps);
  } else {
    __syncthreads();
    for (int g = wave; g < groups; g += kNT / 64) {  // one wave sums a group, in a fixed order
      float a = 0.f;
      for (int e = lane; e < gs / V; e += 64) a += sm[g * (gs / V) + e];
      a = wave_sum(a);
      if (lane == 0) ginv[g] = 1.f / sqrtf(a / (float)gs + eps);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int e = (tid + i * kNT) * V;
    if (e < H) {
      const float inv = groups == 1 ? inv1 : ginv[e / gs];
#pragma unroll
      for (int k = 0; k < V; ++k) v[i][k] = v[i][k] * inv * wv[i][k];
      Row<T, V>::st(out + t * H + e, v[i]);
    }
  }
}

// The same for sizes that the compiler knows: rows of WAVES * 256, 4 elements per thread, groups of whole waves, TOP expert rows. A decode step's
// rows are bound by the instructions that a wave issues in turn, of which there are half as many, a prompt's by memory; arguments that are
// there at the start, every load before the first use, one barrier. us in a captured loop, rows not in the L2, bf16, the kernel above / this, 1, 48,
// 512, 8192 rows: 2048, two expert rows 3.1 / 2.2, 4.3 / 2.8, 6.5 / 5.1, 58.9 / 55.0, with four parts 3.8 / 2.4, 5.2 / 3.3, 9.8 / 8.4, 98.2 / 95.9;
// 4096, a row alone 3.0 / 2.6, 4.0 / 3.1, 8.6 / 7.7, 80.6 / 75.3; 1024, a row alone 2.3 / 2.0, 2.5 / 2.1, 3.9 / 3.2, 20.7 / 18.3.
enum { kMixRow, kMixTwoParts, kMixFourParts, kFromTable };   // where the rows' addend (or the rows) come from

struct KnownNormRest {
  void* out;
  int parts, rows, per;   // of mix; 1 << per waves share a group
  float icols, eps;       // 1 / columns of a group (a power of two)
  long table_rows;
};
struct KnownNormArgs {
  const void *residual, *mix, *y, *pair_slot, *w, *ls1, *ls2;
  KnownNormRest rest;
};

template <typename T, int WAVES, int KIND, int TOP>
__global__ __launch_bounds__(64 * WAVES) void scaled_add_group_rmsnorm_known_kernel(
    float* residual, const void* __restrict__ mix, const T* __restrict__ y, const int* __restrict__ pair_slot, const float* __restrict__ w,
    const float* __restrict__ ls1, const float* __restrict__ ls2, const KnownNormRest) {
  __shared__ float sums[WAVES];
  constexpr int H = 256 * WAVES, P = KIND == kMixFourParts ? 4 : 2;
  const int t = blockIdx.x, tid = threadIdx.x, e = 4 * tid, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const auto rest = late_args<KnownNormRest>(offsetof(KnownNormArgs, rest));
  float* r = residual + (long)t * H + e;
  float v[4], a[4], wv[4], l1[4], l2[4], part[P][4], ye[TOP > 0 ? TOP : 1][4];
  int slot[TOP > 0 ? TOP : 1];
#pragma unroll
  for (int j = 0; j < TOP; ++j) slot[j] = pair_slot[t * TOP + j];
  [[maybe_unused]] bool known = true;
  if constexpr (KIND == kFromTable) {   // y: the table, pair_slot: the ids (an id outside the table gives a row of NaN, as no row is read)
    const long id = reinterpret_cast<const long*>(pair_slot)[t];
    known = id >= 0 && id < rest->table_rows;
    Row<T, 4>::ld((known ? y + id * H : reinterpret_cast<const T*>(w)) + e, v);
  } else {
    Row<float, 4>::ld(r, v);
  }
  if constexpr (KIND == kMixRow) Row<T, 4>::ld(static_cast<const T*>(mix) + (long)t * H + e, a);
  Row<float, 4>::ld(w + e, wv);
  if constexpr (KIND != kFromTable) Row<float, 4>::ld((ls1 != nullptr ? ls1 : w) + e, l1);
  if constexpr (TOP > 0) Row<float, 4>::ld(ls2 + e, l2);
#pragma unroll
  for (int j = 0; j < TOP; ++j) Row<T, 4>::ld(y + (long)slot[j] * H + e, ye[j]);
  const int parts = rest->parts;
  if constexpr (KIND == kMixTwoParts || KIND == kMixFourParts) {   // the last part in place of one that does not exist
#pragma unroll
    for (int j = 0; j < P; ++j) Row<float, 4>::ld(static_cast<const float*>(mix) + ((long)min(j, parts - 1) * rest->rows + t) * H + e, part[j]);
  }
  T* out = static_cast<T*>(rest->out);
  const int per = rest->per;
  const float icols = rest->icols, eps = rest->eps;
  asm volatile("" ::"s"(out), "s"(per), "s"(icols), "s"(eps));
  float q = 0.f;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if constexpr (KIND == kFromTable) {
      if (!known) v[k] = __builtin_nanf("");
    } else {
      float m = 0.f;
      if constexpr (KIND == kMixRow) m = a[k];
      else {
#pragma unroll
        for (int j = 0; j < P; ++j) m += j < parts ? part[j][k] : 0.f;
      }
      v[k] += ls1 != nullptr ? m * l1[k] : m;
    }
    if constexpr (TOP > 0) {
      float f = 0.f;
#pragma unroll
      for (int j = 0; j < TOP; ++j) f += ye[j][k];
      v[k] += f * (1.f / (float)TOP) * l2[k];
    }
    q += v[k] * v[k];
  }
  Row<float, 4>::st(r, v);
  q = wave_sum(q);
  if ((tid & 63) == 0) sums[wave] = q;
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < WAVES; ++i) s += i >> per == wave >> per ? sums[i] : 0.f;
  const float inv = 1.f / sqrtf(s * icols + eps);
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = v[k] * inv * wv[k];
  Row<T, 4>::st(out + (long)t * H + e, v);
}

// Any length and grouping, element by element.
template <typename T>
__global__ __launch_bounds__(kNT) void scaled_add_group_rmsnorm_kernel(
    T* __restrict__ out, float* __restrict__ residual, const float* __restrict__ w, int H, int groups, float eps,
    const void* __restrict__ mix_, int mix_parts, const float* __restrict__ ls1, const T* __restrict__ y,
    const int* __restrict__ pair_slot, int top, const float* __restrict__ ls2, const T* __restrict__ extra,
    const T* __restrict__ table, const long* __restrict__ ids, long table_rows) {
  extern __shared__ float sm[];  // [H] squares, then [groups] inverse rms
  float* sq = sm;
  float* ginv = sm + H;
  const long t = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  float* r = residual + t * H;
  const float wtop = top > 0 ? 1.f / (float)top : 0.f;
  const long id = table != nullptr ? ids[t] : 0;
  const bool known = id >= 0 && id < table_rows;
  for (int e = tid; e < H; e += kNT) {
    float v = table == nullptr ? r[e] : known ? ldf<T>(table, id * H + e) : __builtin_nanf("");
    if (mix_ != nullptr) {
      float m = mix_parts == 0 ? ldf<T>(static_cast<const T*>(mix_), t * H + e) : 0.f;
      for (int j = 0; j < mix_parts; ++j) m += static_cast<const float*>(mix_)[((long)j * gridDim.x + t) * H + e];
      v += ls1 != nullptr ? m * ls1[e] : m;
    }
    if (y != nullptr) {
      float f = 0.f;
      for (int j = 0; j < top; ++j) f += ldf<T>(y, (long)pair_slot[t * top + j] * H + e);
      v += f * wtop * ls2[e];
    }
    if (extra != nullptr) v += ldf<T>(extra, t * H + e);
    r[e] = v;
    sq[e] = v * v;
  }
  __syncthreads();
  const int gs = H / groups;
  for (int g = wave; g < groups; g += kNT / 64) {  // one wave sums a group, in a fixed order
    float a = 0.f;
    for (int e = lane; e < gs; e += 64) a += sq[g * gs + e];
    a = wave_sum(a);
    if (lane == 0) ginv[g] = 1.f / sqrtf(a / (float)gs + eps);
  }
  __syncthreads();
  for (int e = tid; e < H; e += kNT) stf<T>(out, t * H + e, r[e] * ginv[e / gs] * w[e]);
}

// Residual update with the norm on the sublayer's OUTPUT, one workgroup per token row:
//   y = addend row, or the mixture's output
//       shared + sum_j wts[t, j] * (ids[t, j] < E ? ye[pair_slot[t * top + j]] : h[t])      (fp32)
//   residual += y / sqrt(mean(y^2) + eps) * w        (fp32, written back);  out = residual in T
template <typename T>
__global__ __launch_bounds__(kNT) void add_normed_kernel(
    T* __restrict__ out, float* __restrict__ residual, const float* __restrict__ w, int H, float eps,
    const T* __restrict__ y, const T* __restrict__ ye, const int* __restrict__ pair_slot, const int* __restrict__ ids,
    const float* __restrict__ wts, int top, int E, const T* __restrict__ h, const T* __restrict__ shared) {
  extern __shared__ float sm[];  // [H] the addend
  __shared__ float red[16];
  const long t = blockIdx.x;
  const int tid = threadIdx.x;
  float sq = 0.f;
  float wsum_id = 0.f;  // weight of the token's identity experts
  if (y == nullptr)
    for (int j = 0; j < top; ++j)
      if (ids[t * top + j] >= E) wsum_id += wts[t * top + j];
  for (int e = tid; e < H; e += kNT) {
    float v;
    if (y != nullptr) {
      v = ldf<T>(y, t * H + e);
    } else {
      v = shared != nullptr ? ldf<T>(shared, t * H + e) : 0.f;
      for (int j = 0; j < top; ++j)
        if (ids[t * top + j] < E) v = __builtin_fmaf(wts[t * top + j], ldf<T>(ye, (long)pair_slot[t * top + j] * H + e), v);
      if (wsum_id != 0.f) v = __builtin_fmaf(wsum_id, ldf<T>(h, t * H + e), v);
    }
    sm[e] = v;
    sq += v * v;
  }
  sq = block_sum(sq, red);
  const float inv = 1.f / sqrtf(sq / (float)H + eps);
  float* r = residual + t * H;
  for (int e = tid; e < H; e += kNT) {
    const float v = r[e] + sm[e] * inv * w[e];
    r[e] = v;
    stf<T>(out, t * H + e, v);
  }
}

}  // namespace

void launch_add_normed(void* out, float* residual, const float* w, int T, int H, float eps, const void* y,
                       const void* ye, const int* pair_slot, const int* ids, const float* wts, int top, int E,
                       const void* h, const void* shared, bool f32, hipStream_t s) {
  if (T <= 0) return;
  const size_t smem = (size_t)H * sizeof(float);
  if (f32)
    add_normed_kernel<float><<<T, kNT, smem, s>>>((float*)out, residual, w, H, eps, (const float*)y, (const float*)ye,
                                                  pair_slot, ids, wts, top, E, (const float*)h, (const float*)shared);
  else
    add_normed_kernel<unsigned short><<<T, kNT, smem, s>>>(
        (unsigned short*)out, residual, w, H, eps, (const unsigned short*)y, (const unsigned short*)ye, pair_slot, ids,
        wts, top, E, (const unsigned short*)h, (const unsigned short*)shared);
}

namespace {

template <typename T>
void launch_group_norm(T* out, float* residual, const float* w, int T_, int H, int groups, float eps, const void* mix,
                       int mix_parts, const float* ls1, const T* y, const int* pair_slot, int top, const float* ls2, const T* extra,
                       const T* table, const long* ids, long table_rows, hipStream_t s) {
  uintptr_t at = 0;
  for (const void* p : {(const void*)out, (const void*)residual, (const void*)w, (const void*)mix, (const void*)ls1,
                        (const void*)y, (const void*)ls2, (const void*)extra, (const void*)table})
    at |= reinterpret_cast<uintptr_t>(p);
  // 4, 8 and 16 waves, two expert rows or none: the widths and the choices per token of this package's own layer-list configurations, 1024, 2048 and 4096
  // (both sides: at the kernel). Powers of two, so that a wave's group is a shift and 1 / columns exact; other sizes take the kernels below. So do more than
  // 2000 rows of 4096 16-bit elements from a table, whose 16 waves leave too few rows under way: 4096, 8192, 16384 rows 24.8 / 24.2, 58.3 / 55.0, 132 / 116 us
  // (known / below; 2000 rows 14.9 / 14.9, 1000 9.1 - 9.3 / 9.4 - 9.6).
  const int waves = H / 256;
  const bool long_table = table != nullptr && waves == 16 && sizeof(T) == 2 && T_ > 2000;
  if (!long_table && at % 16 == 0 && extra == nullptr && H % 256 == 0 && (waves == 4 || waves == 8 || waves == 16) && groups > 0 &&
      waves % groups == 0 && (y == nullptr || (top == 2 && ls2 != nullptr)) && (table != nullptr ? mix == nullptr && y == nullptr : mix != nullptr) &&
      mix_parts <= 4) {
    const KnownNormRest rest{out, mix_parts, T_, __builtin_ctz(waves / groups), (float)groups / (float)H, eps, table_rows};
    auto go = [&](auto* kernel) {
      if (table != nullptr) kernel<<<T_, 64 * waves, 0, s>>>(residual, nullptr, table, reinterpret_cast<const int*>(ids), w, ls1, ls2, rest);
      else kernel<<<T_, 64 * waves, 0, s>>>(residual, mix, y, pair_slot, w, ls1, ls2, rest);
    };
#define HS_GS(W, KIND) (y != nullptr ? go(&scaled_add_group_rmsnorm_known_kernel<T, W, KIND, 2>) : go(&scaled_add_group_rmsnorm_known_kernel<T, W, KIND, 0>))
#define HS_GW(W) (table != nullptr ? go(&scaled_add_group_rmsnorm_known_kernel<T, W, kFromTable, 0>) \
                  : mix_parts == 0 ? HS_GS(W, kMixRow) : mix_parts <= 2 ? HS_GS(W, kMixTwoParts) : HS_GS(W, kMixFourParts))
    if (waves == 4) HS_GW(4);
    else if (waves == 8) HS_GW(8);
    else HS_GW(16);
#undef HS_GW
#undef HS_GS
    return;
  }
  // 8 elements per thread and step, or 4 for rows that would leave half of the threads idle
  const int V = H <= 4 * kNT ? 4 : 8;
  if (at % 16 == 0 && H % V == 0 && (H / groups) % V == 0 && H <= 8 * 8 * kNT) {
    const size_t smem = groups > 1 ? (size_t)(H / V + groups) * sizeof(float) : 0;
#define HS_GN(V, N) (mix_parts > 0 ? HS_GP(V, N, true) : HS_GP(V, N, false))
#define HS_GP(V, N, PARTS)                                                                                           \
  scaled_add_group_rmsnorm_vec_kernel<T, V, N, PARTS><<<T_, kNT, smem, s>>>(out, residual, w, H, groups, eps, mix, mix_parts, ls1, y, \
                                                                     pair_slot, top, ls2, extra, table, ids, table_rows)
    if (V == 4) HS_GN(4, 1);
    else if (H <= 8 * kNT) HS_GN(8, 1);
    else if (H <= 16 * kNT) HS_GN(8, 2);
    else if (H <= 32 * kNT) HS_GN(8, 4);
    else HS_GN(8, 8);
#undef HS_GN
#undef HS_GP
    return;
  }
  scaled_add_group_rmsnorm_kernel<T><<<T_, kNT, (size_t)(H + groups) * sizeof(float), s>>>(
      out, residual, w, H, groups, eps, mix, mix_parts, ls1, y, pair_slot, top, ls2, extra, table, ids, table_rows);
}

}  // namespace

void launch_scaled_add_group_rmsnorm(void* out, float* residual, const float* w, int T, int H, int groups, float eps,
                                     const void* mix, int mix_parts, const float* ls1, const void* y, const int* pair_slot, int top,
                                     const float* ls2, const void* extra, const void* table, const long* ids,
                                     long table_rows, bool f32, hipStream_t s) {
  if (T <= 0) return;
  if (f32)
    launch_group_norm<float>((float*)out, residual, w, T, H, groups, eps, mix, mix_parts, ls1, (const float*)y,
                             pair_slot, top, ls2, (const float*)extra, (const float*)table, ids, table_rows, s);
  else
    launch_group_norm<unsigned short>((unsigned short*)out, residual, w, T, H, groups, eps, mix, mix_parts,
                                      ls1, (const unsigned short*)y, pair_slot, top, ls2, (const unsigned short*)extra,
                                      (const unsigned short*)table, ids, table_rows, s);
}

}  // namespace hipserve

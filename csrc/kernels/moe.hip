// Mixture-of-experts kernels for Mixtral-style sparse MLPs on
// gfx950. Graph-capturable: every grid is sized from static upper bounds and the
// data-dependent parts (tile count, expert of a tile) are read on the device.
//
//   moe_topk_softmax  router logits -> top-k experts + renormalised weights
//                     (one wave per token, experts on lanes, wave64 reductions)
//   moe_align         token/expert pairs sorted by expert into 16-row tiles,
//                     padding slots = -1 (one 1024-thread workgroup, LDS counts)
//   moe_gemm          per tile: out[slot] = x[row(slot)] . W_e^T on MFMA, rows
//                     gathered through the slot list (token rows for w13, slot rows
//                     for w2); each expert's weights stream once per 16-row tile
//   moe_combine       y rows of a token's k pairs, weighted sum -> hidden state
#include "hipserve/common.h"
#include "hipserve/kernels.h"

namespace hipserve {

template <typename T>
HS_DEVICE float ld_f(const T* p, long i);
template <>
HS_DEVICE float ld_f<unsigned short>(const unsigned short* p, long i) { return bf16_to_f32(p[i]); }
template <>
HS_DEVICE float ld_f<float>(const float* p, long i) { return p[i]; }

// One wave per token, expert e on lane e % 64, slot e / 64 (E <= 128). renorm:
// weights / sum over the selected k (Mixtral, Qwen3-MoE norm_topk_prob); else the
// plain softmax probabilities of the selected experts.
// S > 0: ``logits`` are the router decode GEMM's fp32 split-K partials [S, T, E]; each
// logit is their in-order sum rounded to bf16, as splitk_reduce would have written it
// (bit-identical to reduce + this kernel, one launch fewer per MoE layer).
template <typename T>
__global__ __launch_bounds__(256) void moe_topk_softmax_kernel(const T* __restrict__ logits, float* __restrict__ w,
                                                               int* __restrict__ ids, int Tn, int E, int k,
                                                               int renorm, int S = 0) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (t >= Tn) return;
  float v[2], p[2];
  int rank[2] = {-1, -1};
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int e = lane + 64 * s;
    if constexpr (sizeof(T) == 4) {
      if (S > 0) {  // 8 slices' loads in flight at a time, summed in slice order
        float acc = 0.f;
        const int ec = e < E ? e : 0;
        for (int j0 = 0; j0 < S; j0 += 8) {
          float pv[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) pv[i] = j0 + i < S ? ld_f<T>(logits, ((long)(j0 + i) * Tn + t) * E + ec) : 0.f;
#pragma unroll
          for (int i = 0; i < 8; ++i)
            if (j0 + i < S) acc += pv[i];
        }
        v[s] = e < E ? bf16_to_f32(f32_to_bf16(acc)) : -INFINITY;
        continue;
      }
    }
    v[s] = e < E ? ld_f<T>(logits, (long)t * E + e) : -INFINITY;
  }
  const float mx = wave_max(fmaxf(v[0], v[1]));
  float ex[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) ex[s] = (lane + 64 * s) < E ? __expf(v[s] - mx) : 0.f;
  const float sum = wave_sum(ex[0] + ex[1]);
#pragma unroll
  for (int s = 0; s < 2; ++s) p[s] = ex[s] / sum;
  float sel_sum = 0.f;
  for (int j = 0; j < k; ++j) {
    // argmax over (lane, slot), ties -> lower expert id: the wave max of the unselected
    // probabilities, then the lowest lane holding it (slot 0 = experts 0-63 first)
    const float c0 = rank[0] < 0 && lane < E ? p[0] : -1.f;
    const float c1 = rank[1] < 0 && lane + 64 < E ? p[1] : -1.f;
    const float bv = wave_max(fmaxf(c0, c1));  // DPP reduction (common.h), wave-uniform
    const unsigned long long b0 = __ballot(c0 == bv), b1 = __ballot(c1 == bv);
    const int bi = b0 ? __builtin_ctzll(b0) : 64 + __builtin_ctzll(b1);
    if (bi == lane) rank[0] = j;
    if (bi == lane + 64) rank[1] = j;
    sel_sum += bv;
  }
  const float norm = renorm ? 1.f / sel_sum : 1.f;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    if (rank[s] >= 0) {
      w[(long)t * k + rank[s]] = p[s] * norm;
      ids[(long)t * k + rank[s]] = lane + 64 * s;
    }
  }
}

HS_DEVICE int pair_expert(int p, const int* ids, const int* table, const long* tokens, int top, int top_shift, long table_rows) {
  if (table == nullptr) return ids[p];
  const int t = top_shift >= 0 ? p >> top_shift : p / top;
  const long row = tokens[t];
  return table[(row >= 0 && row < table_rows ? row : 0) * top + (p - t * top)];
}

// Exclusive scan of the tile-padded counts by one wave, 2 experts per lane (E <= 128); off[128]: all of them.
HS_DEVICE void padded_offsets(const int* cnt, int* off, int E, int tile_shift, int* num_tiles, int* group_end, bool first) {
  const int lane = threadIdx.x & 63, e0 = 2 * lane, e1 = 2 * lane + 1, tile = 1 << tile_shift;
  const int a = e0 < E ? (cnt[e0] + tile - 1) >> tile_shift << tile_shift : 0;
  const int b = e1 < E ? (cnt[e1] + tile - 1) >> tile_shift << tile_shift : 0;
  int incl = a + b;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(incl, o, 64);
    if (lane >= o) incl += v;
  }
  const int excl = incl - a - b;
  off[e0] = excl;
  off[e1] = excl + a;
  if (first && group_end != nullptr) {  // per-expert end row of the padded expert-sorted slots (grouped GEMM offsets)
    if (e0 < E) group_end[e0] = excl + a;
    if (e1 < E) group_end[e1] = incl;
  }
  if (lane == 63) {
    off[128] = incl;
    if (first) *num_tiles = incl >> tile_shift;
  }
}

// The order for a GEMM of `across` tiles for each of these that takes them in rounds of `per_round`, as place << 16 | expert << 8 | pairs - 1: as they lie, but
// where it takes what whole rounds leave over by columns (pw_rest: up to two sixteenths of a round, up to three if none of it has more than 64 rows), as many of
// those that hold the fewest pairs as it is tiles of come last. Taken in another way they are better left (8 experts of 2048 x 4096, 36 of 73 tiles by
// quarters 145 -> 153 us: each workgroup has another expert's weights), and so are all partial tiles (16 experts of 1024 x 2048 in two rounds 65 -> 74). One wave,
// two experts per lane.
HS_DEVICE void order_tiles(const int* cnt, const int* off, int E, int tile_shift, int per_round, int across, int* __restrict__ order) {
  const int lane = threadIdx.x & 63, total = off[128] >> tile_shift, over = total * across % per_round, whole = total * across - over;
  // those that the left ones are of: the first group of them may start before them (the GEMM's walk: its tiles column by column)
  const int first = whole / (kTileGroup * across) * kTileGroup, taken = whole - first * across - (across - 1) * min(kTileGroup, total - first);
  const int left = over > 0 ? total - first - max(taken, 0) : 0;
  int rest[2], rank[2] = {0, 0};   // pairs of the experts' last tiles, where they are partial, and how many of those have fewer
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int x = 2 * lane + i;
    rest[i] = x < E ? cnt[x] & ((1 << tile_shift) - 1) : 0;
  }
#pragma unroll 4
  for (int x = 0; x < E; ++x) {
    const int r = cnt[x] & ((1 << tile_shift) - 1);
#pragma unroll
    for (int i = 0; i < 2; ++i) rank[i] += r > 0 && (r < rest[i] || (r == rest[i] && x < 2 * lane + i)) ? 1 : 0;
  }
  const int few = __popcll(__ballot(rest[0] > 0 && rest[0] <= 64)) + __popcll(__ballot(rest[1] > 0 && rest[1] <= 64));
  const bool moves = 16 * over <= (left <= few ? 3 : 2) * per_round;
  unsigned long moved[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) moved[i] = __ballot(moves && rest[i] > 0 && rank[i] < left);
  const int all = __popcll(moved[0]) + __popcll(moved[1]);
  const unsigned long below = (1UL << lane) - 1;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int x = 2 * lane + i;
    if (x >= E) continue;
    const bool last = moved[i] >> lane & 1;
    const int before = __popcll(moved[0] & below) + __popcll(moved[1] & below) + (i == 1 ? (int)(moved[0] >> lane & 1) : 0);
    const int t0 = off[x] >> tile_shift, t1 = (off[x] + cnt[x] + (1 << tile_shift) - 1) >> tile_shift;
    for (int t = t0; t < t1; ++t) {
      const bool partial = rest[i] > 0 && t == t1 - 1;
      order[partial && last ? total - all + rank[i] : t - before] = t << 16 | x << 8 | ((partial ? rest[i] : 1 << tile_shift) - 1);
    }
  }
}

// The places of the workgroup's pairs (experts e, pairs first + 1024 i) among their experts' pairs of this wave, which are counted in mine [128]: the same in every
// run, as those by atomics on counts of the workgroup are not, since these depend on the order between the waves. A place decides about the tile, and the packed
// GEMM sums k in another order for the tiles that whole rounds leave over: its results were repeated but for the last bits. Bits of the expert are compared over
// the wave, those that E has; experts past it, which no caller has, are at least not mixed up with others. us, by atomics -> this: 16384 pairs of 8 experts 5.7 -> 5.9, of
// 128 5.9 -> 6.4, 4096 of 8 4.2 -> 4.9, 2048 3.4 -> 4.2. (Decode steps, whose tiles of 32 are all summed alike, keep the atomics: 96 pairs of four tables 3.0 us, 3.4 this way.)
template <int PER> HS_DEVICE void wave_places(const int (&e)[PER], int first, int npairs, int E, int* mine, int (&place)[PER]) {
  const int lane = threadIdx.x & 63;
  mine[lane] = mine[lane + 64] = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    asm volatile("" ::: "memory");   // other lanes' counts are read: the LDS takes a wave's accesses in order
    const bool live = first + 1024 * i < npairs;
    unsigned long same = __ballot(live && e[i] < E);   // the lanes with this expert
    if (e[i] >= E) same = __ballot(live) & ~same;
    for (int b = 0; 1 << b < E; ++b) {
      const unsigned long set = __ballot(e[i] >> b & 1);
      same &= e[i] >> b & 1 ? set : ~set;
    }
    const int before = __popcll(same & ((1UL << lane) - 1)), known = mine[e[i]];
    place[i] = known + before;
    asm volatile("" ::: "memory");
    if (live && before == 0) mine[e[i]] = known + __popcll(same);
  }
}

// The counts of 16 waves summed to cnt, and in their place those of the waves before, of the experts 2 lane and 2 lane + 1. One wave.
HS_DEVICE void wave_totals(int (&part)[16][128], int* cnt) {
  const int lane = threadIdx.x & 63;
  int2 n[16], c = {0, 0};
#pragma unroll
  for (int w = 0; w < 16; ++w) n[w] = *reinterpret_cast<const int2*>(&part[w][2 * lane]);
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    *reinterpret_cast<int2*>(&part[w][2 * lane]) = c;
    c.x += n[w].x;
    c.y += n[w].y;
  }
  *reinterpret_cast<int2*>(&cnt[2 * lane]) = c;
}

// table (may be null): the experts come from table[tokens[t]][j] (top of them per token) instead of ids, without a
// launch of its own for the lookup (4.5 - 6.3 us); a token outside the table counts as its first entry. Workgroup b serves table b of as many
// (decode steps: the tables of all layers in one launch, 2.6 - 3.8 us instead of that for each).
// PER: pairs per thread at most, all looked up at once; a pair's place among its expert's is what the count gives it, and only slots that hold
// no pair are cleared (96 pairs 3.2 -> 2.6 us beside a second pass that counts again). SAME: places as wave_places has them.
template <int PER, bool SAME>
__global__ __launch_bounds__(1024) void moe_align_kernel(const int* __restrict__ ids, const int* __restrict__ table,
                                                         const long* __restrict__ tokens, int top, int top_shift, long table_rows,
                                                         int npairs, int E, int tile_shift,
                                                         int* __restrict__ slots, int slots_cap,
                                                         int* __restrict__ tile_expert, int tiles_cap,
                                                         int* __restrict__ num_tiles, int* __restrict__ pair_slot,
                                                         int* __restrict__ group_end, const MoeOrder order) {
  __shared__ __attribute__((aligned(16))) int part[SAME ? 16 : 1][128], cnt[128];
  __shared__ int off[129];
  const int tid = threadIdx.x, wave = tid >> 6;
  const long b = blockIdx.x;
  if (table != nullptr) table += b * table_rows * top;
  slots += b * slots_cap;
  tile_expert += b * tiles_cap;
  pair_slot += b * npairs;
  num_tiles += b;
  int e[PER], rank[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) e[i] = npairs > 0 ? pair_expert(min(tid + 1024 * i, npairs - 1), ids, table, tokens, top, top_shift, table_rows) : 0;
  if constexpr (SAME) {
    wave_places<PER>(e, tid, npairs, E, part[wave], rank);
  } else {
    if (tid < 128) cnt[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (tid + 1024 * i < npairs) rank[i] = atomicAdd(&cnt[e[i]], 1);
  }
  __syncthreads();
  if (tid < 64) {
    if constexpr (SAME) wave_totals(part, cnt);
    padded_offsets(cnt, off, E, tile_shift, num_tiles, group_end, true);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int p = tid + 1024 * i;
    if (p < npairs) {
      const int pos = off[e[i]] + rank[i] + (SAME ? part[wave][e[i]] : 0);
      slots[pos] = p;
      pair_slot[p] = pos;
    }
  }
  const int total = off[128];
  for (int x = tid >> 6; x < E; x += 16)   // the rest of every expert's last tile
    for (int s = off[x] + cnt[x] + (tid & 63); s < off[x + 1]; s += 64) slots[s] = -1;
  for (int s = total + tid; s < slots_cap; s += 1024) slots[s] = -1;
  // each expert labels its own tiles; tiles past the used range are -1
  if (tid < E)
    for (int t = off[tid] >> tile_shift; t < off[tid + 1] >> tile_shift; ++t) tile_expert[t] = tid;
  for (int t = (total >> tile_shift) + tid; t < tiles_cap; t += 1024) tile_expert[t] = -1;
  if (tid >> 6 < order.rows) order_tiles(cnt, off, E, tile_shift, order.per_round[tid >> 6], order.across[tid >> 6], order.to + (long)(tid >> 6) * tiles_cap);
}

// moe_align over many workgroups, for prefill-sized pair counts (one workgroup is bound by its compute unit's lookups and stores). Pass 1: a
// workgroup counts the experts of its PER * 1024 pairs, hist[b][E], and leaves each pair's expert and place among them in pair_slot. Pass
// 2: every workgroup sums the table (nb x E ints) into the padded expert offsets and its own prefix, then scatters its pairs; the padding slots
// (disjoint from every real slot, so no ordering between workgroups is needed) and tile tables of the experts go round the workgroups.
// us, one workgroup -> many, in brackets with the lookup of table[token]: 8000 pairs, 16 experts 7.2 -> 5.0 (13.4 -> 5.4), 16384 pairs 11.9 -> 5.2
// (24.4 -> 5.6), of 128 experts 13.8 -> 6.1 (25.4 -> 6.5), 4097 pairs of 128 experts 5.9 -> 5.6 (with an expert's rest per workgroup, not per wave, 8.9); 4096
// pairs 4.0 (5.5) on one.
template <int PER, bool SAME>
__global__ __launch_bounds__(1024) void moe_count_kernel(const int* __restrict__ ids, const int* __restrict__ table, const long* __restrict__ tokens,
                                                         int top, int top_shift, long table_rows, int npairs, int E,
                                                         int* __restrict__ pair_slot, int* __restrict__ hist) {
  __shared__ __attribute__((aligned(16))) int part[SAME ? 16 : 1][128], cnt[128];
  const int tid = threadIdx.x, b = blockIdx.x, p0 = b * PER * 1024 + tid;
  [[maybe_unused]] const int wave = tid >> 6;
  int e[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) e[i] = pair_expert(min(p0 + 1024 * i, npairs - 1), ids, table, tokens, top, top_shift, table_rows);
  if constexpr (SAME) {
    int place[PER];
    wave_places<PER>(e, p0, npairs, E, part[wave], place);
    __syncthreads();
    if (tid < 64) wave_totals(part, cnt);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (p0 + 1024 * i < npairs) pair_slot[p0 + 1024 * i] = e[i] << 16 | (part[wave][e[i]] + place[i]);
  } else {
    if (tid < 128) cnt[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (p0 + 1024 * i < npairs) pair_slot[p0 + 1024 * i] = e[i] << 16 | atomicAdd(&cnt[e[i]], 1);
    __syncthreads();
  }
  if (tid < 128) hist[b * 128 + tid] = cnt[tid];
}

template <int PER>
__global__ __launch_bounds__(1024) void moe_place_kernel(int npairs, int E, int tile_shift, const int* __restrict__ hist, int nb,
                                                         int* __restrict__ slots, int slots_cap,
                                                         int* __restrict__ tile_expert, int tiles_cap,
                                                         int* __restrict__ num_tiles, int* __restrict__ pair_slot,
                                                         int* __restrict__ group_end, const MoeOrder order) {
  __shared__ int cnt[128], pre[128], off[129], part[2][8][128];
  const int tid = threadIdx.x, b = blockIdx.x, tile = 1 << tile_shift, p0 = b * PER * 1024 + tid;
  int mine[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) mine[i] = pair_slot[min(p0 + 1024 * i, npairs - 1)];
  {  // expert totals and this workgroup's prefix over those before it
    const int x = tid & 127, g = tid >> 7;
    int c = 0, q = 0;
#pragma unroll 4
    for (int j = g; j < nb; j += 8) {
      const int h = hist[j * 128 + x];
      c += h;
      q += j < b ? h : 0;
    }
    part[0][g][x] = c;
    part[1][g][x] = q;
  }
  __syncthreads();
  if (tid < 256) {
    int c = 0;
#pragma unroll
    for (int g = 0; g < 8; ++g) c += part[tid >> 7][g][tid & 127];
    (tid < 128 ? cnt : pre)[tid & 127] = c;
  }
  __syncthreads();
  if (tid < 64) padded_offsets(cnt, off, E, tile_shift, num_tiles, group_end, b == 0);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int p = p0 + 1024 * i, x = mine[i] >> 16;
    if (p < npairs) {
      const int pos = off[x] + pre[x] + (mine[i] & 0xffff);
      slots[pos] = p;
      pair_slot[p] = pos;
    }
  }
  const int total = off[128];
  for (int x = b * 16 + (tid >> 6); x < E; x += nb * 16) {   // the rest of the experts' last tiles, their tiles' labels: an expert per wave
    for (int s = off[x] + cnt[x] + (tid & 63); s < off[x + 1]; s += 64) slots[s] = -1;
    for (int t = (off[x] >> tile_shift) + (tid & 63); t < off[x + 1] >> tile_shift; t += 64) tile_expert[t] = x;
  }
  for (int s = total + b * 1024 + tid; s < slots_cap; s += nb * 1024) slots[s] = -1;
  for (int t = (total >> tile_shift) + b * 1024 + tid; t < tiles_cap; t += nb * 1024) tile_expert[t] = -1;
  if (b == nb - 1 && tid >> 6 < order.rows) order_tiles(cnt, off, E, tile_shift, order.per_round[tid >> 6], order.across[tid >> 6], order.to + (long)(tid >> 6) * tiles_cap);
}

static int align_chunk(int npairs) { return npairs > 65536 ? 4096 : 1024; }
int moe_align_blocks(int npairs) { return npairs > 4096 ? (npairs + align_chunk(npairs) - 1) / align_chunk(npairs) : 1; }
// The tables of several layers go through one workgroup each, 16 pairs per thread at most. One table alone has no such bound; the same line is kept for it, and
// beyond it the experts are gathered first.
bool moe_align_small(int npairs) { return npairs <= 16384; }

// out[slot, N] = x[row(slot), K] . W[e, N, K]^T; row(slot) = pair / k (gather) or slot.
// A tile = 16*MT consecutive slots of one expert; each W fragment feeds MT MFMAs.
template <int MT, int KW>
__global__ __launch_bounds__(64 * KW) void moe_gemm_kernel(
    unsigned short* __restrict__ out, long out_stride, const unsigned short* __restrict__ x, long x_stride,
    const unsigned short* __restrict__ w, const int* __restrict__ slots, const int* __restrict__ tile_expert,
    int gather_k, int N, int K) {
  extern __shared__ __attribute__((aligned(16))) float red[];  // [KW][MT][64][4]
  const int tile = blockIdx.y;
  const int e = tile_expert[tile];
  if (e < 0) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, c = lane & 15;
  const int n0 = blockIdx.x * 16;
  int pr[MT];
  const unsigned short* xr[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int slot = tile * 16 * MT + 16 * t + c;
    pr[t] = slots[slot];
    const long xrow = pr[t] < 0 ? 0 : (gather_k > 0 ? pr[t] / gather_k : slot);
    xr[t] = x + xrow * x_stride + 64 * g;
  }
  const unsigned short* wr = w + ((long)e * N + min(n0 + c, N - 1)) * K + 64 * g;
  const int kw = K / KW, k0 = wave * kw, k1 = k0 + kw;
  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int kk = k0; kk < k1; kk += 256) {
    u16x8 a[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) a[s] = *reinterpret_cast<const u16x8*>(wr + kk + 8 * s);
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const u16x8 b = *reinterpret_cast<const u16x8*>(xr[t] + kk + 8 * s);
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[s]),
                                                         __builtin_bit_cast(bf16x8, b), acc[t], 0, 0, 0);
      }
  }
  if constexpr (KW > 1) {
#pragma unroll
    for (int t = 0; t < MT; ++t) *reinterpret_cast<f32x4*>(red + ((wave * MT + t) * 64 + lane) * 4) = acc[t];
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int t = 0; t < MT; ++t)
      for (int q = 1; q < KW; ++q) acc[t] += *reinterpret_cast<const f32x4*>(red + ((q * MT + t) * 64 + lane) * 4);
  }
  // C: col = slot-in-tile (lane & 15), rows n = n0 + 4g + j
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    if (pr[t] < 0) continue;
    const long slot = tile * 16 * MT + 16 * t + c;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + 4 * g + j;
      if (n < N) out[slot * out_stride + n] = f32_to_bf16(acc[t][j]);
    }
  }
}

__global__ __launch_bounds__(256) void moe_combine_kernel(unsigned short* __restrict__ out, const unsigned short* __restrict__ y,
                                                          const float* __restrict__ w, const int* __restrict__ pair_slot,
                                                          int k, int H) {
  const int t = blockIdx.x;
  for (int c = threadIdx.x; c < H / 8; c += 256) {
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < k; ++j) {
      const float wt = w[(long)t * k + j];
      const u16x8 v = *reinterpret_cast<const u16x8*>(y + (long)pair_slot[t * k + j] * H + 8 * c);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += wt * bf16_to_f32(v[e]);
    }
    u16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = f32_to_bf16(acc[e]);
    *reinterpret_cast<u16x8*>(out + (long)t * H + 8 * c) = o;
  }
}

// Split-K w2 partials ws[s][slot][H] (fp32): each pair's y row is bf16(sum over s),
// exactly what the bf16 expert GEMM output would be, then the weighted sum.
__global__ __launch_bounds__(256) void moe_combine_partial_kernel(unsigned short* __restrict__ out,
                                                                  const float* __restrict__ ws, long slab, int S,
                                                                  const float* __restrict__ w,
                                                                  const int* __restrict__ pair_slot, int k, int H) {
  const int t = blockIdx.x;
  for (int c = threadIdx.x; c < H / 8; c += 256) {
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < k; ++j) {
      const float wt = w[(long)t * k + j];
      const float* p = ws + (long)pair_slot[t * k + j] * H + 8 * c;
      f32x4 lo, hi;
      sum_slices8(lo, hi, p, slab, S);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        acc[e] += wt * bf16_to_f32(f32_to_bf16(lo[e]));
        acc[e + 4] += wt * bf16_to_f32(f32_to_bf16(hi[e]));
      }
    }
    u16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = f32_to_bf16(acc[e]);
    *reinterpret_cast<u16x8*>(out + (long)t * H + 8 * c) = o;
  }
}

// Decode MoE tail in one kernel: the weighted combine of a token's k expert rows (bf16
// y [slots, H], or fp32 w2 partials [S, slots, H] summed per pair in slice order) rounded
// to bf16 as moe_combine(_partial) writes it, then the residual add and the NEXT layer's
// RMSNorm exactly as fused_add_rmsnorm (norm.hip: same thread -> element map, same block
// reduction): bit-identical to the two-kernel chain, one launch fewer per MoE layer.
template <int NT, int VPT, bool kWF32, bool kPartial>
__global__ __launch_bounds__(NT) void moe_combine_add_rmsnorm_kernel(
    unsigned short* __restrict__ out, unsigned short* __restrict__ residual, const void* __restrict__ y, long slab,
    int S, const float* __restrict__ w, const int* __restrict__ pair_slot, int k, int H,
    const void* __restrict__ weight, float eps) {
  __shared__ float scratch[16];
  const int t = blockIdx.x;
  const int nvec = H >> 3;
  u16x8* rr = reinterpret_cast<u16x8*>(residual + (long)t * H);
  float v[VPT][8];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = threadIdx.x + i * NT;
    if (idx < nvec) {
      float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (int j = 0; j < k; ++j) {
        const float wt = w[(long)t * k + j];
        const long row = (long)pair_slot[t * k + j] * H + 8 * idx;
        if constexpr (kPartial) {
          f32x4 lo, hi;
          sum_slices8(lo, hi, static_cast<const float*>(y) + row, slab, S);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            acc[e] += wt * bf16_to_f32(f32_to_bf16(lo[e]));
            acc[e + 4] += wt * bf16_to_f32(f32_to_bf16(hi[e]));
          }
        } else {
          const u16x8 yv = *reinterpret_cast<const u16x8*>(static_cast<const unsigned short*>(y) + row);
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[e] += wt * bf16_to_f32(yv[e]);
        }
      }
      const u16x8 b = rr[idx];
      u16x8 sres;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float f = bf16_to_f32(f32_to_bf16(acc[e])) + bf16_to_f32(b[e]);
        sres[e] = f32_to_bf16(f);
        v[i][e] = bf16_to_f32(sres[e]);
      }
      rr[idx] = sres;
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += v[i][e] * v[i][e];
    }
  }
  ss = block_sum(ss, scratch);
  const float inv = rsqrtf(ss / H + eps);
  u16x8* orow = reinterpret_cast<u16x8*>(out + (long)t * H);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int idx = threadIdx.x + i * NT;
    if (idx < nvec) {
      float wv[8];
      if constexpr (kWF32) {
        const f32x4* wp = reinterpret_cast<const f32x4*>(weight) + idx * 2;
        const f32x4 w0 = wp[0], w1 = wp[1];
#pragma unroll
        for (int e = 0; e < 4; ++e) { wv[e] = w0[e]; wv[e + 4] = w1[e]; }
      } else {
        const u16x8 wb = reinterpret_cast<const u16x8*>(weight)[idx];
#pragma unroll
        for (int e = 0; e < 8; ++e) wv[e] = bf16_to_f32(wb[e]);
      }
      u16x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = f32_to_bf16(v[i][e] * inv * wv[e]);
      orow[idx] = o;
    }
  }
}

template <bool kWF32, bool kPartial>
static void mcn_launch(void* out, void* residual, const void* y, long slab, int S, const float* w, const int* ps,
                       int T, int k, int H, const void* nw, float eps, hipStream_t s) {
  auto* o = static_cast<unsigned short*>(out);
  auto* r = static_cast<unsigned short*>(residual);
  const int nvec = H / 8;
  if (norm_threads(H) == 256) {
    if (nvec <= 256) moe_combine_add_rmsnorm_kernel<256, 1, kWF32, kPartial><<<T, 256, 0, s>>>(o, r, y, slab, S, w, ps, k, H, nw, eps);
    else moe_combine_add_rmsnorm_kernel<256, 2, kWF32, kPartial><<<T, 256, 0, s>>>(o, r, y, slab, S, w, ps, k, H, nw, eps);
  } else {
    if (nvec <= 512) moe_combine_add_rmsnorm_kernel<512, 1, kWF32, kPartial><<<T, 512, 0, s>>>(o, r, y, slab, S, w, ps, k, H, nw, eps);
    else if (nvec <= 1024) moe_combine_add_rmsnorm_kernel<512, 2, kWF32, kPartial><<<T, 512, 0, s>>>(o, r, y, slab, S, w, ps, k, H, nw, eps);
    else moe_combine_add_rmsnorm_kernel<512, 4, kWF32, kPartial><<<T, 512, 0, s>>>(o, r, y, slab, S, w, ps, k, H, nw, eps);
  }
}

void launch_moe_combine_add_rmsnorm(void* out, void* residual, const void* y, long slab, int S, const float* w,
                                    const int* pair_slot, int T, int k, int H, const void* norm_w, bool norm_f32,
                                    float eps, hipStream_t s) {
  if (T <= 0) return;
  if (S > 0) {
    if (norm_f32) mcn_launch<true, true>(out, residual, y, slab, S, w, pair_slot, T, k, H, norm_w, eps, s);
    else mcn_launch<false, true>(out, residual, y, slab, S, w, pair_slot, T, k, H, norm_w, eps, s);
  } else {
    if (norm_f32) mcn_launch<true, false>(out, residual, y, slab, 0, w, pair_slot, T, k, H, norm_w, eps, s);
    else mcn_launch<false, false>(out, residual, y, slab, 0, w, pair_slot, T, k, H, norm_w, eps, s);
  }
}

void launch_moe_topk_softmax(const void* logits, bool logits_f32, float* w, int* ids, int T, int E, int k,
                             bool renorm, hipStream_t s, int splits) {
  if (T <= 0) return;
  dim3 grid((T + 3) / 4), block(256);
  if (logits_f32)
    moe_topk_softmax_kernel<float><<<grid, block, 0, s>>>(static_cast<const float*>(logits), w, ids, T, E, k,
                                                          renorm ? 1 : 0, splits);
  else
    moe_topk_softmax_kernel<unsigned short><<<grid, block, 0, s>>>(static_cast<const unsigned short*>(logits), w, ids,
                                                                   T, E, k, renorm ? 1 : 0);
}

// tiles of a power of two; hist: [moe_align_blocks, 128] where that is more than one and there is one table; same: see wave_places
template <bool SAME>
static void align(int tables, const int* ids, const int* table, const long* tokens, int top, long table_rows, int npairs, int E, int tile, int* slots,
                  int slots_cap, int* tile_expert, int tiles_cap, int* num_tiles, int* pair_slot, int* group_end, int* hist, const MoeOrder& order, hipStream_t s) {
  const int top_shift = (top & (top - 1)) == 0 ? __builtin_ctz(top) : -1, shift = __builtin_ctz(tile), nb = moe_align_blocks(npairs);
  if (nb > 1 && tables == 1) {
    const bool wide = align_chunk(npairs) > 1024;
    (wide ? moe_count_kernel<4, SAME> : moe_count_kernel<1, SAME>)<<<nb, 1024, 0, s>>>(ids, table, tokens, top, top_shift, table_rows, npairs, E, pair_slot, hist);
    (wide ? moe_place_kernel<4> : moe_place_kernel<1>)<<<nb, 1024, 0, s>>>(npairs, E, shift, hist, nb, slots, slots_cap, tile_expert, tiles_cap,
                                                                           num_tiles, pair_slot, group_end, order);
    return;
  }
  (npairs <= 1024 ? moe_align_kernel<1, SAME> : npairs <= 4096 ? moe_align_kernel<4, SAME> : moe_align_kernel<16, SAME>)<<<tables, 1024, 0, s>>>(
      ids, table, tokens, top, top_shift, table_rows, npairs, E, shift, slots, slots_cap, tile_expert, tiles_cap, num_tiles, pair_slot, group_end,
      order);
}

void launch_moe_align(const int* ids, int npairs, int E, int tile, int* slots, int slots_cap, int* tile_expert,
                      int tiles_cap, int* num_tiles, int* pair_slot, int* group_end, hipStream_t s, int* hist, bool same) {
  (same ? align<true> : align<false>)(1, ids, nullptr, nullptr, 1, 0, npairs, E, tile, slots, slots_cap, tile_expert, tiles_cap, num_tiles, pair_slot, group_end,
                                      hist, MoeOrder{}, s);
}

void launch_moe_table_align(const int* table, int tables, const long* tokens, int top, long table_rows, int npairs, int E, int tile, int* slots, int slots_cap,
                            int* tile_expert, int tiles_cap, int* num_tiles, int* pair_slot, int* hist, bool same, const MoeOrder& order, hipStream_t s) {
  (same ? align<true> : align<false>)(tables, nullptr, table, tokens, top, table_rows, npairs, E, tile, slots, slots_cap, tile_expert, tiles_cap, num_tiles,
                                      pair_slot, nullptr, hist, order, s);
}

// Prefill MoE input: xs[slot] = x[slots[slot] / k] (the token of the pair in that
// slot), zero rows for padding slots — the A operand of the grouped expert GEMM.
// One workgroup per 8 slots, 16-byte vectors.
__global__ __launch_bounds__(256) void moe_gather_kernel(unsigned short* __restrict__ out,
                                                         const unsigned short* __restrict__ x, long x_stride,
                                                         const int* __restrict__ slots, int nslots, int k, int H) {
  const int vpr = H >> 3;  // 16-byte vectors per row
  const int slot = blockIdx.x * 8 + threadIdx.x / 32;
  if (slot >= nslots) return;
  const int p = slots[slot];
  u16x8* dst = reinterpret_cast<u16x8*>(out + (long)slot * H);
  if (p < 0) {
    for (int v = threadIdx.x & 31; v < vpr; v += 32) dst[v] = u16x8{0, 0, 0, 0, 0, 0, 0, 0};
    return;
  }
  const u16x8* src = reinterpret_cast<const u16x8*>(x + (long)(p / k) * x_stride);
  for (int v = threadIdx.x & 31; v < vpr; v += 32) dst[v] = src[v];
}

void launch_moe_gather(void* out, const void* x, long x_stride, const int* slots, int nslots, int k, int H,
                       hipStream_t s) {
  if (nslots <= 0) return;
  moe_gather_kernel<<<(nslots + 7) / 8, 256, 0, s>>>(static_cast<unsigned short*>(out),
                                                     static_cast<const unsigned short*>(x), x_stride, slots, nslots,
                                                     k, H);
}

template <int MT>
static void moe_gemm_mt(void* out, long out_stride, const void* x, long x_stride, const void* w, const int* slots,
                        const int* tile_expert, int tiles_cap, int gather_k, int N, int K, hipStream_t s) {
  const int kw = (K % 1024 == 0) ? 4 : ((K % 512 == 0) ? 2 : 1);
  dim3 grid((N + 15) / 16, tiles_cap), block(64 * kw);
  const size_t smem = kw > 1 ? (size_t)kw * MT * 64 * 4 * sizeof(float) : 0;
  auto* o = static_cast<unsigned short*>(out);
  auto* xi = static_cast<const unsigned short*>(x);
  auto* wi = static_cast<const unsigned short*>(w);
  if (kw == 4)
    moe_gemm_kernel<MT, 4><<<grid, block, smem, s>>>(o, out_stride, xi, x_stride, wi, slots, tile_expert, gather_k, N, K);
  else if (kw == 2)
    moe_gemm_kernel<MT, 2><<<grid, block, smem, s>>>(o, out_stride, xi, x_stride, wi, slots, tile_expert, gather_k, N, K);
  else
    moe_gemm_kernel<MT, 1><<<grid, block, smem, s>>>(o, out_stride, xi, x_stride, wi, slots, tile_expert, gather_k, N, K);
}

void launch_moe_gemm(void* out, long out_stride, const void* x, long x_stride, const void* w, const int* slots,
                     const int* tile_expert, int tiles_cap, int tile, int gather_k, int N, int K, hipStream_t s) {
  if (tile == 16) moe_gemm_mt<1>(out, out_stride, x, x_stride, w, slots, tile_expert, tiles_cap, gather_k, N, K, s);
  else if (tile == 32) moe_gemm_mt<2>(out, out_stride, x, x_stride, w, slots, tile_expert, tiles_cap, gather_k, N, K, s);
  else moe_gemm_mt<4>(out, out_stride, x, x_stride, w, slots, tile_expert, tiles_cap, gather_k, N, K, s);
}

void launch_moe_combine(void* out, const void* y, const float* w, const int* pair_slot, int T, int k, int H,
                        hipStream_t s) {
  if (T <= 0) return;
  moe_combine_kernel<<<T, 256, 0, s>>>(static_cast<unsigned short*>(out), static_cast<const unsigned short*>(y), w,
                                       pair_slot, k, H);
}

void launch_moe_combine_partial(void* out, const float* ws, long slab, int S, const float* w, const int* pair_slot,
                                int T, int k, int H, hipStream_t s) {
  if (T <= 0) return;
  moe_combine_partial_kernel<<<T, 256, 0, s>>>(static_cast<unsigned short*>(out), ws, slab, S, w, pair_slot, k, H);
}

}  // namespace hipserve

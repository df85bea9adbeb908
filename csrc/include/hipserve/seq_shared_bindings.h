// Bindings shared by the layer-list decoders' kernel libraries (each library links its own copy of the
// kernels): products of a few rows, the expert alignment and the expert GEMMs of the mixtures of experts.
#pragma once
#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/library.h>

#include "hipserve/kernels.h"
#include "hipserve/seq_kernels.h"

namespace hipserve_shared {

inline hipStream_t cur_stream() { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream(); }

#define CHECK_DEV(x) TORCH_CHECK((x).is_cuda(), #x " must be a GPU tensor")
#define CHECK_SAME_DEV(x, y) TORCH_CHECK((x).device() == (y).device(), #x " must be on the device of " #y)
#define CHECK_CONTIG(x) TORCH_CHECK((x).is_contiguous(), #x " must be contiguous")
#define CHECK_F32(x) TORCH_CHECK((x).scalar_type() == at::kFloat && (x).is_contiguous(), #x " must be contiguous fp32")
#define CHECK_I32(x) TORCH_CHECK((x).scalar_type() == at::kInt && (x).is_contiguous(), #x " must be contiguous int32")

inline bool is_f32(const at::Tensor& t, const char* who) {
  TORCH_CHECK(t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16, who, ": bf16 or fp32 activations");
  return t.scalar_type() == at::kFloat;
}

inline const void* opt_ptr(const c10::optional<at::Tensor>& t) { return t.has_value() ? t->data_ptr() : nullptr; }
inline bool rows2d(const at::Tensor& t) { return t.dim() == 2 && t.stride(1) == 1; }

inline void moe_align(const at::Tensor& ids, int64_t E, int64_t tile, at::Tensor& slots, at::Tensor& tile_expert,
                      at::Tensor& pair_slot) {
  auto i32 = [](const at::Tensor& t) { return t.scalar_type() == at::kInt && t.is_contiguous(); };
  TORCH_CHECK(ids.is_cuda() && i32(ids) && i32(slots) && i32(tile_expert) && i32(pair_slot), "moe_align: int32 GPU tensors");
  TORCH_CHECK(E >= 1 && E <= 128, "moe_align: at most 128 experts");
  TORCH_CHECK(tile == 16 || tile == 32 || tile == 64 || tile == 128 || tile == 256);
  const int npairs = ids.numel();
  TORCH_CHECK(slots.numel() >= npairs + E * (tile - 1) && slots.numel() % tile == 0,
              "slots capacity must cover padding and be a multiple of the tile");
  TORCH_CHECK(tile_expert.numel() * tile >= slots.numel() && pair_slot.numel() >= npairs);
  c10::hip::HIPGuardMasqueradingAsCUDA g(ids.device());
  hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
  const int nb = hipserve::moe_align_blocks(npairs);
  at::Tensor scratch = at::empty({(long)(nb > 1 ? nb : 0) * 128 + 1}, ids.options());  // [hist | tile count]
  hipserve::launch_moe_align(ids.data_ptr<int>(), npairs, E, tile, slots.data_ptr<int>(), slots.numel(),
                             tile_expert.data_ptr<int>(), tile_expert.numel(),
                             scratch.data_ptr<int>() + (scratch.numel() - 1), pair_slot.data_ptr<int>(), nullptr,
                             stream, nb > 1 ? scratch.data_ptr<int>() : nullptr);
}

// moe_align of the pairs (t, j) whose expert is table[tokens[t]][j], table [rows, top]; or of every table of [L, rows, top], with outputs
// [L, slots], [L, tiles], [L, pairs]; num_tiles [L]: the tiles in use; order [n, tiles], one table: those
// as a GEMM takes them that has per_round[j] in a round, across[j] of them (none given: one) for each of these (order_tiles), place << 16 | expert << 8 | pairs - 1.
inline void moe_table_align(const at::Tensor& table, const at::Tensor& tokens, int64_t E, int64_t tile, at::Tensor& slots,
                            at::Tensor& tile_expert, at::Tensor& pair_slot, const c10::optional<at::Tensor>& num_tiles,
                            const c10::optional<at::Tensor>& order, at::IntArrayRef per_round, at::IntArrayRef across) {
  CHECK_DEV(table); CHECK_I32(table); CHECK_I32(slots); CHECK_I32(tile_expert); CHECK_I32(pair_slot);
  CHECK_SAME_DEV(tokens, table); CHECK_SAME_DEV(slots, table); CHECK_SAME_DEV(tile_expert, table); CHECK_SAME_DEV(pair_slot, table);
  const long d = table.dim(), L = d == 3 ? table.size(0) : 1;
  TORCH_CHECK((d == 2 || d == 3) && L >= 1 && table.size(d - 2) >= 1 && tokens.scalar_type() == at::kLong && tokens.is_contiguous());
  for (const at::Tensor* t : std::initializer_list<const at::Tensor*>{&slots, &tile_expert, &pair_slot})
    TORCH_CHECK(d == 2 || (t->dim() == 2 && t->size(0) == L), "moe_table_align: a row of outputs per table");
  TORCH_CHECK(E >= 1 && E <= 128, "moe_align: at most 128 experts");
  TORCH_CHECK(tile == 16 || tile == 32 || tile == 64 || tile == 128 || tile == 256);
  const long top = table.size(d - 1), npairs = tokens.numel() * top, cap = slots.numel() / L, tiles = tile_expert.numel() / L;
  TORCH_CHECK(top >= 1 && hipserve::moe_align_small(npairs), "moe_table_align: small batches");
  TORCH_CHECK(cap >= npairs + E * (tile - 1) && cap % tile == 0, "slots capacity must cover padding and be a multiple of the tile");
  TORCH_CHECK(tiles * tile >= cap && pair_slot.numel() / L >= npairs && (d == 2 || pair_slot.size(1) == npairs));
  c10::hip::HIPGuardMasqueradingAsCUDA g(table.device());
  if (num_tiles.has_value()) {
    CHECK_I32(*num_tiles); CHECK_SAME_DEV(*num_tiles, table);
    TORCH_CHECK(num_tiles->numel() == L, "moe_table_align: a count per table");
  }
  hipserve::MoeOrder orders;
  if (order.has_value()) {
    CHECK_I32(*order); CHECK_SAME_DEV(*order, table);
    TORCH_CHECK(L == 1 && order->dim() == 2 && order->size(1) == tiles && order->size(0) == (long)per_round.size() && per_round.size() <= 2 &&
                (across.empty() || across.size() == per_round.size()) && tiles < (1L << 15) && tile <= 256, "moe_table_align: orders of the tiles");
    orders.to = order->data_ptr<int>();
    orders.rows = per_round.size();
    for (size_t i = 0; i < per_round.size(); ++i) {
      TORCH_CHECK(per_round[i] >= 1 && per_round[i] < (1L << 20), "moe_table_align: tiles in a round");
      orders.per_round[i] = per_round[i];
      if (across.empty()) continue;
      TORCH_CHECK(across[i] >= 1 && across[i] < (1L << 15), "moe_table_align: tiles beside each other");
      orders.across[i] = across[i];
    }
  }
  const int nb = L == 1 ? hipserve::moe_align_blocks(npairs) : 1;
  at::Tensor hist = at::empty({nb > 1 ? nb * 128L : 0}, slots.options());
  at::Tensor count = num_tiles.has_value() ? *num_tiles : at::empty({L}, slots.options());
  hipserve::launch_moe_table_align(table.data_ptr<int>(), L, tokens.data_ptr<long>(), top, table.size(d - 2), npairs, E, tile,
                                   slots.data_ptr<int>(), cap, tile_expert.data_ptr<int>(), tiles, count.data_ptr<int>(),
                                   pair_slot.data_ptr<int>(), hist.data_ptr<int>(), num_tiles.has_value() && tile >= 128, orders, cur_stream());
}

inline bool moe_align_small(int64_t npairs) { return hipserve::moe_align_small(npairs); }

inline void expert_gemm(at::Tensor& out, const at::Tensor& x, const at::Tensor& w, const at::Tensor& slots,
                        const at::Tensor& tile_expert, int64_t tile, int64_t gather_k, int64_t act,
                        const c10::optional<at::Tensor>& row_scale, double limit, int64_t pairs, int64_t tiles) {
  auto i32 = [](const at::Tensor& t) { return t.scalar_type() == at::kInt && t.is_contiguous(); };
  TORCH_CHECK(x.is_cuda() && out.is_contiguous() && w.is_contiguous() && i32(slots) && i32(tile_expert));
  TORCH_CHECK(x.scalar_type() == at::kFloat || x.scalar_type() == at::kBFloat16, "expert_gemm: bf16 or fp32 activations");
  const bool f32 = x.scalar_type() == at::kFloat;
  TORCH_CHECK(out.scalar_type() == x.scalar_type() && w.scalar_type() == x.scalar_type());
  TORCH_CHECK(w.dim() == 3 && x.dim() == 2 && x.stride(1) == 1 && out.dim() == 2);
  const long N = w.size(1), K = w.size(2), cap = slots.numel();
  TORCH_CHECK(act >= 0 && act <= 3 && (act < 2 || N % 2 == 0),
              "expert_gemm: act 0 (none), 1 (relu^2), 2 (silu gate), 3 (clamped gate)");
  if (row_scale.has_value()) {
    CHECK_F32(*row_scale);   // one number per (token, choice) pair: the slot table holds pair indices
    TORCH_CHECK(gather_k > 0 && row_scale->numel() >= x.size(0) * gather_k, "expert_gemm: a scale per pair");
  }
  TORCH_CHECK(x.size(1) == K && out.size(1) == (act >= 2 ? N / 2 : N) && out.size(0) >= cap);
  TORCH_CHECK(tile % 32 == 0 && cap % tile == 0 && tile_expert.numel() * tile >= cap, "tiles of a multiple of 32 slots");
  TORCH_CHECK(gather_k > 0 || x.size(0) >= cap, "ungathered x needs one row per slot");
  TORCH_CHECK(pairs >= 0 && pairs <= cap, "expert_gemm: at most a pair per slot");
  TORCH_CHECK(tiles >= 0, "expert_gemm: tiles in use");   // 0: not known; else they are among the first so many
  const long ntiles = tiles > 0 ? std::min<long>(tiles, cap / tile) : cap / tile;
  c10::hip::HIPGuardMasqueradingAsCUDA g(x.device());
  hipserve::launch_expert_gemm(out.data_ptr(), x.data_ptr(), x.stride(0), w.data_ptr(), slots.data_ptr<int>(),
                               tile_expert.data_ptr<int>(), cap / tile, ntiles, tile, gather_k, N, K, act, w.size(0),
                               (const float*)opt_ptr(row_scale), (float)limit, pairs, f32,
                               c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream());
}

inline bool expert_rows_pay(int64_t tiles, int64_t pairs, int64_t cols, int64_t k) {
  constexpr int64_t kMost = 1LL << 31;
  TORCH_CHECK(tiles >= 0 && tiles < kMost && pairs >= 0 && pairs < kMost && cols >= 0 && cols < kMost && k >= 0, "expert_rows_pay: sizes");
  return hipserve::expert_rows_pay(tiles, pairs, cols, k);
}

// out = act(x . w^T + bias) of at most 64 rows: x [M, K] or [B, M, K], w [N, K] or [B, N, K], out [M, N'] or [B, M, N'].
inline void skinny_linear(at::Tensor& out, const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& bias,
                          int64_t act, double c0, double c1, int64_t act_from) {
  CHECK_DEV(x); CHECK_CONTIG(w); CHECK_SAME_DEV(w, x); CHECK_SAME_DEV(out, x);
  if (bias.has_value()) CHECK_SAME_DEV(*bias, x);
  const bool f32 = x.scalar_type() == at::kFloat;
  TORCH_CHECK((f32 || x.scalar_type() == at::kBFloat16) && w.scalar_type() == x.scalar_type() &&
              (out.scalar_type() == x.scalar_type() || out.scalar_type() == at::kFloat), "skinny_linear: bf16 or fp32 operands");
  const long d = x.dim();
  const long per = f32 ? 4 : 8;   // numbers in 16 bytes
  TORCH_CHECK((d == 2 || d == 3) && w.dim() == d && out.dim() == d, "skinny_linear: rows or batches of rows");
  const long B = d == 3 ? x.size(0) : 1, M = x.size(-2), K = x.size(-1), N = w.size(-2);
  TORCH_CHECK(w.size(-1) == K && (d == 2 || (w.size(0) == B && out.size(0) == B)) && out.size(-2) == M && M <= 64 && K % per == 0 &&
              N < (1L << 31) && K < (1L << 24) && x.stride(-2) < (1L << 24) && B < 65536, "skinny_linear: shapes");
  const bool glu = act == 3 || act == 4;
  TORCH_CHECK(act >= -1 && act <= 5 && (!glu || N % 2 == 0) && out.size(-1) == (glu ? N / 2 : N), "skinny_linear: activation");
  TORCH_CHECK(act_from >= 0 && act_from <= N && (act_from == 0 || !glu), "skinny_linear: first column of the activation");
  auto aligned = [](const at::Tensor& t) { return (uintptr_t)t.data_ptr() % 16 == 0; };
  TORCH_CHECK(x.stride(-1) == 1 && out.stride(-1) == 1 && x.stride(-2) % per == 0 && (d == 2 || x.stride(0) % per == 0) && aligned(x) &&
              aligned(w), "skinny_linear: rows at multiples of 16 bytes");
  if (bias.has_value())
    TORCH_CHECK(d == 2 && bias->scalar_type() == x.scalar_type() && bias->is_contiguous() && bias->numel() == N, "skinny_linear: bias");
  c10::hip::HIPGuardMasqueradingAsCUDA g(x.device());
  TORCH_CHECK(hipserve::launch_skinny_linear(out.data_ptr(), out.scalar_type() == at::kFloat, out.stride(-2), d == 3 ? out.stride(0) : 0, 0, 1,
                                             x.data_ptr(), x.stride(-2), d == 3 ? x.stride(0) : 0, w.data_ptr(), opt_ptr(bias), f32, B,
                                             M, N, K, act, act_from, (float)c0, (float)c1, cur_stream()), "skinny_linear: LDS");
}

inline double skinny_time(int64_t rows, int64_t cols, int64_t k, bool glu, bool f32, int64_t parts) {
  TORCH_CHECK(rows >= 0 && rows <= 64 && cols >= 0 && cols < (1L << 40) && k >= 0 && k < (1L << 30) && parts >= 1 && parts <= 64, "skinny_time: sizes");
  return hipserve::skinny_time(rows, cols, k, glu, f32, parts);
}

// out [S, M, N]: 32-bit sums over S parts of K (in 64 halves) of x [M, K] . w [N, K]^T, the bias in the first.
inline void skinny_linear_parts(at::Tensor& out, const at::Tensor& x, const at::Tensor& w, const c10::optional<at::Tensor>& bias) {
  CHECK_DEV(x); CHECK_CONTIG(w); CHECK_F32(out); CHECK_SAME_DEV(w, x); CHECK_SAME_DEV(out, x);
  if (bias.has_value()) CHECK_SAME_DEV(*bias, x);
  const bool f32 = x.scalar_type() == at::kFloat;
  TORCH_CHECK((f32 || x.scalar_type() == at::kBFloat16) && w.scalar_type() == x.scalar_type(), "skinny_linear_parts: bf16 or fp32 operands");
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && out.dim() == 3, "skinny_linear_parts: rows, and parts of rows");
  const long per = f32 ? 4 : 8, M = x.size(0), K = x.size(1), N = w.size(0), S = out.size(0);
  TORCH_CHECK(w.size(1) == K && out.size(1) == M && out.size(2) == N && M <= 64 && K % per == 0 && N < (1L << 31) && K < (1L << 24) &&
              x.stride(0) < (1L << 24) && S >= 1 && S <= 64 && S <= (K * 8 / per + 63) / 64, "skinny_linear_parts: shapes");
  auto aligned = [](const at::Tensor& t) { return (uintptr_t)t.data_ptr() % 16 == 0; };
  TORCH_CHECK(x.stride(1) == 1 && x.stride(0) % per == 0 && aligned(x) && aligned(w), "skinny_linear_parts: rows at multiples of 16 bytes");
  if (bias.has_value())
    TORCH_CHECK(bias->scalar_type() == x.scalar_type() && bias->is_contiguous() && bias->numel() == N, "skinny_linear_parts: bias");
  c10::hip::HIPGuardMasqueradingAsCUDA g(x.device());
  TORCH_CHECK(hipserve::launch_skinny_linear(out.data_ptr(), true, N, 0, M * N, S, x.data_ptr(), x.stride(0), 0, w.data_ptr(), opt_ptr(bias),
                                             f32, 1, M, N, K, -1, 0, 0.f, 0.f, cur_stream()), "skinny_linear_parts: LDS");
}

inline void check_normed_rows(const at::Tensor& out, const at::Tensor& squares, const at::Tensor& x, const at::Tensor& w,
                              const c10::optional<at::Tensor>& bias) {
  CHECK_DEV(x); CHECK_CONTIG(w); CHECK_CONTIG(out); CHECK_F32(squares); CHECK_SAME_DEV(w, x); CHECK_SAME_DEV(out, x); CHECK_SAME_DEV(squares, x);
  const bool f32 = x.scalar_type() == at::kFloat;
  const long per = f32 ? 4 : 8, M = x.size(0), K = x.size(-1), N = w.size(0);
  TORCH_CHECK((f32 || x.scalar_type() == at::kBFloat16) && w.scalar_type() == x.scalar_type(), "skinny_linear: bf16 or fp32 operands");
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && out.dim() == 2 && squares.dim() == 2 && w.size(1) == K && out.size(0) == M && M <= 32 &&
              K % per == 0 && N < (1L << 31) && K < (1L << 24) && x.stride(0) < (1L << 24), "skinny_linear: shapes");
  TORCH_CHECK(squares.size(0) == M && squares.size(1) % 4 == 0 && squares.size(1) <= 256, "skinny_linear: squares");
  auto aligned = [](const at::Tensor& t) { return (uintptr_t)t.data_ptr() % 16 == 0; };
  TORCH_CHECK(x.stride(1) == 1 && x.stride(0) % per == 0 && aligned(x) && aligned(w) && aligned(squares), "skinny_linear: rows at multiples of 16 bytes");
  if (bias.has_value()) {
    CHECK_SAME_DEV(*bias, x);
    TORCH_CHECK(bias->scalar_type() == x.scalar_type() && bias->is_contiguous() && bias->numel() == N, "skinny_linear: bias");
  }
}

// skinny_linear of rows x [M, K] without their norm's factor, 1 / sqrt(sum of the row's squares / K + eps).
inline void skinny_linear_normed(at::Tensor& out, const at::Tensor& x, const at::Tensor& squares, double eps, const at::Tensor& w,
                                 const c10::optional<at::Tensor>& bias, int64_t act, double c0, double c1, int64_t act_from) {
  check_normed_rows(out, squares, x, w, bias);
  const bool f32 = x.scalar_type() == at::kFloat, glu = act == 3 || act == 4;
  const long N = w.size(0), K = x.size(1);
  TORCH_CHECK(out.scalar_type() == x.scalar_type() || out.scalar_type() == at::kFloat, "skinny_linear: result type");
  TORCH_CHECK(act >= -1 && act <= 5 && (!glu || N % 2 == 0) && out.size(1) == (glu ? N / 2 : N) && act_from >= 0 && act_from <= N &&
              (act_from == 0 || !glu), "skinny_linear: activation");
  hipserve::SkinnyNorm norm;
  norm.squares = squares.data_ptr<float>();
  norm.blocks = squares.size(1);
  norm.cols = (float)K;
  norm.eps = (float)eps;
  c10::hip::HIPGuardMasqueradingAsCUDA g(x.device());
  TORCH_CHECK(hipserve::launch_skinny_linear_normed(out.data_ptr(), out.scalar_type() == at::kFloat, norm, x.data_ptr(), x.stride(0),
                                                    w.data_ptr(), opt_ptr(bias), f32, x.size(0), N, K, act, act_from, (float)c0, (float)c1,
                                                    cur_stream()), "skinny_linear: LDS");
}

// residual [M, N] += x . w^T + bias; out = residual * weight; squares [M, N / 16] or [M, N / 8] = the residual's squares summed over 16 or 8 columns,
// which is what a workgroup then takes (skinny_half).
inline hipserve::SkinnyNorm check_update(const at::Tensor& out, at::Tensor& squares, at::Tensor& residual, const at::Tensor& weight, const at::Tensor& x,
                                         const at::Tensor& w, const c10::optional<at::Tensor>& bias) {
  check_normed_rows(out, squares, x, w, bias);
  CHECK_F32(residual); CHECK_F32(weight); CHECK_SAME_DEV(residual, x); CHECK_SAME_DEV(weight, x);
  const long M = x.size(0), N = w.size(0);
  TORCH_CHECK(out.scalar_type() == x.scalar_type() && out.size(1) == N && residual.dim() == 2 && residual.size(0) == M && residual.size(1) == N &&
              weight.numel() == N && N % 64 == 0 && (squares.size(1) == N / 16 || squares.size(1) == N / 8), "skinny_linear_update: shapes");
  hipserve::SkinnyNorm norm;
  norm.squares = squares.data_ptr<float>();
  norm.blocks = squares.size(1);
  norm.residual = residual.data_ptr<float>();
  norm.weight = weight.data_ptr<float>();
  return norm;
}

inline void skinny_linear_update(at::Tensor& out, at::Tensor& squares, at::Tensor& residual, const at::Tensor& weight, const at::Tensor& x,
                                 const at::Tensor& w, const c10::optional<at::Tensor>& bias) {
  const auto norm = check_update(out, squares, residual, weight, x, w, bias);
  c10::hip::HIPGuardMasqueradingAsCUDA g(x.device());
  TORCH_CHECK(hipserve::launch_skinny_linear_normed(out.data_ptr(), false, norm, x.data_ptr(), x.stride(0), w.data_ptr(), opt_ptr(bias),
                                                    x.scalar_type() == at::kFloat, x.size(0), w.size(0), x.size(1), -1, 0, 0.f, 0.f, cur_stream()),
              "skinny_linear: LDS");
}

inline bool skinny_half(int64_t rows, int64_t cols, int64_t k, bool f32) {
  TORCH_CHECK(rows >= 0 && rows <= 64 && cols >= 0 && cols < (1L << 40) && k >= 0 && k < (1L << 30), "skinny_half: sizes");
  return hipserve::skinny_half(rows, (cols + 15) / 16, f32 ? 2 * k : k);
}

inline std::vector<int64_t> skinny_wide(int64_t rows, int64_t cols, int64_t k, bool f32, bool normed) {   // pieces ahead, whether half tiles
  TORCH_CHECK(rows >= 0 && rows <= 64 && cols >= 0 && cols < (1L << 40) && k >= 0 && k < (1L << 30), "skinny_wide: sizes");
  const auto w = hipserve::skinny_wide(rows, (cols + 15) / 16, f32 ? 2 * k : k, f32, normed);
  return {w.ahead, w.half};
}

inline int64_t skinny_cols(int64_t rows, int64_t cols, int64_t k) {
  TORCH_CHECK(rows >= 0 && rows <= 64 && cols >= 0 && cols < (1L << 40) && k >= 0 && k < (1L << 30), "skinny_cols: sizes");
  return hipserve::skinny_cols(rows, cols, k);
}

inline void def_moe_ops(torch::Library& m) {
  m.def("skinny_linear(Tensor(a!) out, Tensor x, Tensor w, Tensor? bias, int act, float c0, float c1, int act_from=0) -> ()");
  m.def("skinny_time(int rows, int cols, int k, bool glu, bool f32, int parts) -> float", &skinny_time);
  m.def("skinny_half(int rows, int cols, int k, bool f32) -> bool", &skinny_half);
  m.def("skinny_cols(int rows, int cols, int k) -> int", &skinny_cols);
  m.def("skinny_wide(int rows, int cols, int k, bool f32, bool normed=False) -> int[]", &skinny_wide);
  m.def("skinny_linear_parts(Tensor(a!) out, Tensor x, Tensor w, Tensor? bias) -> ()");
  m.def("skinny_linear_normed(Tensor(a!) out, Tensor x, Tensor squares, float eps, Tensor w, Tensor? bias, int act, float c0, float c1, "
        "int act_from) -> ()");
  m.def("skinny_linear_update(Tensor(a!) out, Tensor(b!) squares, Tensor(c!) residual, Tensor weight, Tensor x, Tensor w, Tensor? bias) -> ()");
  m.def("moe_align(Tensor ids, int E, int tile, Tensor(a!) slots, Tensor(b!) tile_expert, Tensor(c!) pair_slot) -> ()");
  m.def("moe_table_align(Tensor table, Tensor tokens, int E, int tile, Tensor(a!) slots, Tensor(b!) tile_expert, "
        "Tensor(c!) pair_slot, Tensor(d!)? num_tiles=None, Tensor(e!)? order=None, int[] per_round=[], int[] across=[]) -> ()");
  m.def("moe_align_small(int npairs) -> bool", &moe_align_small);
  m.def("expert_gemm(Tensor(a!) out, Tensor x, Tensor w, Tensor slots, Tensor tile_expert, int tile, int gather_k, "
        "int act, Tensor? row_scale=None, float limit=0.0, int pairs=0, int tiles=0) -> ()");
  m.def("expert_rows_pay(int tiles, int pairs, int cols, int k) -> bool", &expert_rows_pay);
}

inline void impl_moe_ops(torch::Library& m) {
  m.impl("skinny_linear", &skinny_linear);
  m.impl("skinny_linear_parts", &skinny_linear_parts);
  m.impl("skinny_linear_normed", &skinny_linear_normed);
  m.impl("skinny_linear_update", &skinny_linear_update);
  m.impl("moe_align", &moe_align);
  m.impl("moe_table_align", &moe_table_align);
  m.impl("expert_gemm", &expert_gemm);
}

}  // namespace hipserve_shared

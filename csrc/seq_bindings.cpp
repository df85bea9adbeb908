// torch.ops.hipserve_seq.* — the layer-list decoders' kernels (csrc/kernels/seq/*.hip), built as
// their own library (hipserve/_C_seq.so) so a model of these designs compiles only what it runs.
// All ops write into caller-provided outputs (no allocation except moe_align's scratch, no host sync).
#include <torch/library.h>
#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include "hipserve/kernels.h"
#include "hipserve/seq_kernels.h"
#include "hipserve/seq_shared_bindings.h"
#include "hipserve/seq_latent_bindings.h"

namespace {

using namespace hipserve_shared;

void scaled_add_group_rmsnorm(at::Tensor& out, at::Tensor& residual, const at::Tensor& w, int64_t groups, double eps,
                              const c10::optional<at::Tensor>& mix, const c10::optional<at::Tensor>& ls1,
                              const c10::optional<at::Tensor>& y, const c10::optional<at::Tensor>& pair_slot,
                              int64_t top, const c10::optional<at::Tensor>& ls2,
                              const c10::optional<at::Tensor>& extra, const c10::optional<at::Tensor>& table,
                              const c10::optional<at::Tensor>& ids) {
  CHECK_DEV(out); CHECK_CONTIG(out); CHECK_F32(residual); CHECK_F32(w);
  const bool f32 = is_f32(out, "scaled_add_group_rmsnorm");
  TORCH_CHECK(residual.dim() == 2 && out.sizes() == residual.sizes());
  const long T = residual.size(0), H = residual.size(1);
  TORCH_CHECK(groups >= 1 && H % groups == 0 && w.numel() == H && H + groups <= 15000, "group norm shape");
  if (mix.has_value()) {
    TORCH_CHECK(mix->is_contiguous() && (mix->dim() == 3 ? mix->scalar_type() == at::kFloat && mix->size(0) >= 1 && mix->size(1) == T && mix->size(2) == H
                                                         : mix->scalar_type() == out.scalar_type() && mix->sizes() == residual.sizes()));
    CHECK_SAME_DEV(*mix, out);
    TORCH_CHECK(!ls1.has_value() || (ls1->scalar_type() == at::kFloat && ls1->is_contiguous() && ls1->numel() == H));
  }
  if (y.has_value()) {
    TORCH_CHECK(y->scalar_type() == out.scalar_type() && y->is_contiguous() && y->dim() == 2 && y->size(1) == H);
    TORCH_CHECK(top >= 1 && pair_slot.has_value() && pair_slot->scalar_type() == at::kInt &&
                pair_slot->is_contiguous() && pair_slot->numel() >= T * top);
    TORCH_CHECK(ls2.has_value() && ls2->scalar_type() == at::kFloat && ls2->numel() == H);
  }
  if (extra.has_value())
    TORCH_CHECK(extra->scalar_type() == out.scalar_type() && extra->is_contiguous() && extra->sizes() == residual.sizes());
  if (table.has_value()) {
    TORCH_CHECK(table->scalar_type() == out.scalar_type() && table->is_contiguous() && table->dim() == 2 && table->size(1) == H);
    TORCH_CHECK(ids.has_value() && ids->scalar_type() == at::kLong && ids->is_contiguous() && ids->numel() == T);
    CHECK_SAME_DEV(*table, out); CHECK_SAME_DEV(*ids, out);
  }
  c10::hip::HIPGuardMasqueradingAsCUDA g(out.device());
  hipserve::launch_scaled_add_group_rmsnorm(
      out.data_ptr(), residual.data_ptr<float>(), w.data_ptr<float>(), T, H, groups, (float)eps, opt_ptr(mix),
      mix.has_value() && mix->dim() == 3 ? (int)mix->size(0) : 0,
      (const float*)opt_ptr(ls1), opt_ptr(y), (const int*)opt_ptr(pair_slot), y.has_value() ? top : 0,
      (const float*)opt_ptr(ls2), opt_ptr(extra), opt_ptr(table), table.has_value() ? ids->data_ptr<long>() : nullptr,
      table.has_value() ? table->size(0) : 0, f32, cur_stream());
}

// bf16 prompt portions on the matrix cores: qc (scratch) [heads, T, kv_rank + rot_dim] is filled here.
void mingru_scan(at::Tensor& y, at::Tensor& state, const at::Tensor& proj, const at::Tensor& b_z,
                 const at::Tensor& b_x, const at::Tensor& seq_cu, const at::Tensor& seq_ctx,
                 const at::Tensor& seq_state, int64_t max_q) {
  CHECK_DEV(proj); CHECK_CONTIG(proj); CHECK_CONTIG(y); CHECK_F32(state); CHECK_F32(b_z); CHECK_F32(b_x);
  CHECK_I32(seq_cu); CHECK_I32(seq_ctx); CHECK_I32(seq_state);
  const bool f32 = is_f32(proj, "mingru_scan");
  TORCH_CHECK(y.scalar_type() == proj.scalar_type());
  const long width = state.size(1), nseq = seq_ctx.numel();
  TORCH_CHECK(proj.dim() == 2 && proj.size(1) == 3 * width && y.numel() == proj.size(0) * width);
  TORCH_CHECK(b_z.numel() == width && b_x.numel() == width);
  TORCH_CHECK(seq_cu.numel() == nseq + 1 && seq_state.numel() >= nseq);
  c10::hip::HIPGuardMasqueradingAsCUDA g(proj.device());
  hipserve::launch_mingru_scan(y.data_ptr(), state.data_ptr<float>(), proj.data_ptr(), b_z.data_ptr<float>(),
                               b_x.data_ptr<float>(), seq_cu.data_ptr<int>(), seq_ctx.data_ptr<int>(),
                               seq_state.data_ptr<int>(), nseq, width, max_q, f32, cur_stream());
}

// mingru_scan of the rows x [M, K] of a step in which every sequence has one row at most, the product x . w^T included.
void check_mingru_product(const at::Tensor& y, const at::Tensor& state, const at::Tensor& x, const at::Tensor& w, const at::Tensor& b_z,
                          const at::Tensor& b_x, const at::Tensor& seq_cu, const at::Tensor& seq_ctx, const at::Tensor& seq_state) {
  CHECK_DEV(x); CHECK_CONTIG(w); CHECK_CONTIG(y); CHECK_F32(state); CHECK_F32(b_z); CHECK_F32(b_x);
  CHECK_I32(seq_cu); CHECK_I32(seq_ctx); CHECK_I32(seq_state);
  for (const at::Tensor* t : std::initializer_list<const at::Tensor*>{&y, &state, &w, &b_z, &b_x, &seq_cu, &seq_ctx, &seq_state}) CHECK_SAME_DEV(*t, x);
  const long per = is_f32(x, "mingru_product") ? 4 : 8, M = x.size(0), K = x.size(-1), width = state.size(1), nseq = seq_ctx.numel();
  TORCH_CHECK(y.scalar_type() == x.scalar_type() && w.scalar_type() == x.scalar_type());
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && state.dim() == 2 && w.size(0) == 3 * width && w.size(1) == K && y.numel() == M * width && M <= 64);
  TORCH_CHECK(x.stride(1) == 1 && x.stride(0) % per == 0 && K % per == 0 && K < (1L << 24) && x.stride(0) < (1L << 24) && width < (1L << 26) &&
              (uintptr_t)x.data_ptr() % 16 == 0 && (uintptr_t)w.data_ptr() % 16 == 0, "mingru_product: rows at multiples of 16 bytes");
  TORCH_CHECK(b_z.numel() == width && b_x.numel() == width && seq_cu.numel() == nseq + 1 && seq_state.numel() >= nseq);
}

void mingru_product(at::Tensor& y, at::Tensor& state, const at::Tensor& x, const at::Tensor& w, const at::Tensor& b_z,
                    const at::Tensor& b_x, const at::Tensor& seq_cu, const at::Tensor& seq_ctx, const at::Tensor& seq_state) {
  check_mingru_product(y, state, x, w, b_z, b_x, seq_cu, seq_ctx, seq_state);
  c10::hip::HIPGuardMasqueradingAsCUDA g(x.device());
  TORCH_CHECK(hipserve::launch_mingru_product(y.data_ptr(), state.data_ptr<float>(), x.data_ptr(), x.stride(0), w.data_ptr(),
                                              b_z.data_ptr<float>(), b_x.data_ptr<float>(), seq_cu.data_ptr<int>(), seq_ctx.data_ptr<int>(),
                                              seq_state.data_ptr<int>(), seq_ctx.numel(), x.size(0), state.size(1), x.size(1),
                                              x.scalar_type() == at::kFloat, cur_stream()), "mingru_product: LDS");
}

// The experts' product of expert_gemm (bf16, tiles of 32 slots) for a launch that holds a dense product of device `like`'s besides.
hipserve::ExpertRows expert_rows(at::Tensor& out, const at::Tensor& x, const at::Tensor& w, const at::Tensor& slots, const at::Tensor& tile_expert,
                                 int64_t gather_k, int64_t act, int64_t pairs, int64_t tiles, const at::Tensor& like) {
  CHECK_CONTIG(out); CHECK_CONTIG(w); CHECK_I32(slots); CHECK_I32(tile_expert);
  for (const at::Tensor* t : std::initializer_list<const at::Tensor*>{&out, &x, &w, &slots, &tile_expert}) CHECK_SAME_DEV(*t, like);
  TORCH_CHECK(out.scalar_type() == at::kBFloat16 && x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16, "experts beside: bf16");
  TORCH_CHECK(w.dim() == 3 && x.dim() == 2 && x.stride(1) == 1 && out.dim() == 2 && (act == 0 || act == 1));
  const long N = w.size(1), K = w.size(2), cap = slots.numel();
  TORCH_CHECK(x.size(1) == K && out.size(1) == N && out.size(0) >= cap && cap % 32 == 0 && tile_expert.numel() * 32 >= cap);
  TORCH_CHECK(gather_k > 0 || x.size(0) >= cap, "ungathered x needs one row per slot");
  TORCH_CHECK(pairs > 0 && pairs <= cap && tiles > 0 && N < (1L << 31) && w.size(0) < (1L << 31));
  return {out.data_ptr(), x.data_ptr(), w.data_ptr(), slots.data_ptr<int>(), tile_expert.data_ptr<int>(), x.stride(0),
          std::min<long>(tiles, cap / 32), (int)gather_k, (int)N, (int)std::min<long>(K, 1L << 30), (int)act, (int)w.size(0), (int)pairs, cap};
}

// A plain product as skinny_linear (out [M, N]) or skinny_linear_parts (out [S, M, N] in 32 bits) and the experts' in one launch; false, and nothing
// done, where there is none for these sizes.
bool skinny_linear_experts(at::Tensor& out, const at::Tensor& x, const at::Tensor& w, at::Tensor& e_out, const at::Tensor& e_x, const at::Tensor& e_w,
                           const at::Tensor& slots, const at::Tensor& tile_expert, int64_t gather_k, int64_t act, int64_t pairs, int64_t tiles) {
  CHECK_DEV(x); CHECK_CONTIG(w); CHECK_CONTIG(out); CHECK_SAME_DEV(w, x); CHECK_SAME_DEV(out, x);
  const bool f32 = out.scalar_type() == at::kFloat;
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16 && (f32 || out.scalar_type() == at::kBFloat16));
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && (out.dim() == 2 || (out.dim() == 3 && f32)), "skinny_linear_experts: rows");
  const long M = x.size(0), K = x.size(1), N = w.size(0), S = out.dim() == 3 ? out.size(0) : 1;
  TORCH_CHECK(w.size(1) == K && out.size(-2) == M && out.size(-1) == N && M <= 64 && K % 8 == 0 && N < (1L << 31) && K < (1L << 24) &&
              x.stride(0) < (1L << 24) && S >= 1 && S <= 64 && S <= (K + 63) / 64, "skinny_linear_experts: shapes");
  auto aligned = [](const at::Tensor& t) { return (uintptr_t)t.data_ptr() % 16 == 0; };
  TORCH_CHECK(x.stride(1) == 1 && x.stride(0) % 8 == 0 && aligned(x) && aligned(w), "skinny_linear_experts: rows at multiples of 16 bytes");
  const auto ex = expert_rows(e_out, e_x, e_w, slots, tile_expert, gather_k, act, pairs, tiles, x);
  c10::hip::HIPGuardMasqueradingAsCUDA g(x.device());
  return hipserve::launch_skinny_linear_experts(out.data_ptr(), f32, N, M * N, S, x.data_ptr(), x.stride(0), w.data_ptr(), M, N, K, ex, cur_stream());
}

// mingru_product and the experts' product in one launch, alike.
bool mingru_product_experts(at::Tensor& y, at::Tensor& state, const at::Tensor& x, const at::Tensor& w, const at::Tensor& b_z, const at::Tensor& b_x,
                            const at::Tensor& seq_cu, const at::Tensor& seq_ctx, const at::Tensor& seq_state, at::Tensor& e_out, const at::Tensor& e_x,
                            const at::Tensor& e_w, const at::Tensor& slots, const at::Tensor& tile_expert, int64_t gather_k, int64_t act,
                            int64_t pairs, int64_t tiles) {
  check_mingru_product(y, state, x, w, b_z, b_x, seq_cu, seq_ctx, seq_state);
  TORCH_CHECK(x.scalar_type() == at::kBFloat16, "mingru_product_experts: bf16");
  const auto ex = expert_rows(e_out, e_x, e_w, slots, tile_expert, gather_k, act, pairs, tiles, x);
  c10::hip::HIPGuardMasqueradingAsCUDA g(x.device());
  return hipserve::launch_mingru_product_experts(y.data_ptr(), state.data_ptr<float>(), x.data_ptr(), x.stride(0), w.data_ptr(), b_z.data_ptr<float>(),
                                                 b_x.data_ptr<float>(), seq_cu.data_ptr<int>(), seq_ctx.data_ptr<int>(), seq_state.data_ptr<int>(),
                                                 seq_ctx.numel(), x.size(0), state.size(1), x.size(1), ex, cur_stream());
}

}  // namespace

TORCH_LIBRARY(hipserve_seq, m) {
  hipserve_shared::def_moe_ops(m);
  m.def("scaled_add_group_rmsnorm(Tensor(a!) out, Tensor(b!) residual, Tensor w, int groups, float eps, Tensor? mix, "
        "Tensor? ls1, Tensor? y, Tensor? pair_slot, int top, Tensor? ls2, Tensor? extra, Tensor? table=None, "
        "Tensor? ids=None) -> ()");
  m.def("latent_prepare(Tensor(a!) cq, Tensor(b!) cache, Tensor proj, Tensor positions, Tensor slots, Tensor q_norm, "
        "Tensor kv_norm, Tensor inv_freq, int q_rank, int kv_rank, int rot_dim, float eps) -> ()");
  m.def("latent_attention(Tensor(a!) o_lat, Tensor q_abs, Tensor q, Tensor proj, Tensor cache, Tensor seq_cu, "
        "Tensor seq_ctx, Tensor seq_bt, int seq0, int seq1, int rows_bound, int tq, Tensor inv_freq, int heads, "
        "int dim, int rot_dim, int kv_rank, int gate_off, float scale, int window) -> ()");
  m.def("latent_attention_mfma(Tensor(a!) o_lat, Tensor(b!) qc, Tensor? q_abs, Tensor q, Tensor proj, Tensor positions, "
        "Tensor cache, Tensor seq_cu, Tensor seq_ctx, Tensor seq_bt, int seq0, int seq1, int rows_bound, "
        "Tensor inv_freq, int heads, int dim, int rot_dim, int kv_rank, int gate_off, float scale, int window, "
        "int nparts, int part_keys, Tensor(c!)? ws_acc, Tensor(d!)? ws_ml, int row_base, bool fill_qc) -> ()");
  m.def("latent_gather(Tensor(a!) lat, Tensor(b!) off, Tensor cache, Tensor seq_cu, Tensor seq_ctx, Tensor seq_bt, int window) -> ()");
  m.def("latent_prompt_attention(Tensor(a!) out, Tensor q, Tensor kv, Tensor lat, Tensor off, Tensor seq_cu, Tensor seq_ctx, "
        "Tensor positions, Tensor inv_freq, Tensor proj, int heads, int gate_off, bool channel_gate, float scale, int window) -> ()");
  m.def("latent_prompt_ok(int dim, int rot_dim, int vdim) -> bool", &latent_prompt_ok);
  m.def("latent_attention_dma_ok(int kv_rank, int rot_dim) -> bool", &latent_attention_dma_ok);
  m.def("latent_attention_mfma_ok(int kv_rank, int rot_dim) -> bool", &latent_attention_mfma_ok);
  m.def("mingru_product_time(int rows, int width, int k, bool f32) -> float", [](int64_t rows, int64_t width, int64_t k, bool f32) {
    TORCH_CHECK(rows >= 0 && rows <= 64 && width >= 0 && width < (1L << 26) && k >= 0 && k < (1L << 30), "mingru_product_time: sizes");
    return hipserve::mingru_product_time(rows, width, k, f32);
  });
  m.def("mingru_product(Tensor(a!) y, Tensor(b!) state, Tensor x, Tensor w, Tensor b_z, Tensor b_x, Tensor seq_cu, Tensor seq_ctx, "
        "Tensor seq_state) -> ()");
  m.def("mingru_product_experts(Tensor(a!) y, Tensor(b!) state, Tensor x, Tensor w, Tensor b_z, Tensor b_x, Tensor seq_cu, Tensor seq_ctx, "
        "Tensor seq_state, Tensor(c!) e_out, Tensor e_x, Tensor e_w, Tensor slots, Tensor tile_expert, int gather_k, int act, int pairs, "
        "int tiles) -> bool");
  m.def("skinny_linear_experts(Tensor(a!) out, Tensor x, Tensor w, Tensor(b!) e_out, Tensor e_x, Tensor e_w, Tensor slots, Tensor tile_expert, "
        "int gather_k, int act, int pairs, int tiles) -> bool");
  m.def("mingru_scan(Tensor(a!) y, Tensor(b!) state, Tensor proj, Tensor b_z, Tensor b_x, Tensor seq_cu, "
        "Tensor seq_ctx, Tensor seq_state, int max_q) -> ()");
}

TORCH_LIBRARY_IMPL(hipserve_seq, CUDA, m) {
  hipserve_shared::impl_moe_ops(m);
  m.impl("scaled_add_group_rmsnorm", &scaled_add_group_rmsnorm);
  m.impl("latent_prepare", &latent_prepare);
  m.impl("latent_attention", &latent_attention);
  m.impl("latent_attention_mfma", &latent_attention_mfma);
  m.impl("latent_gather", &latent_gather);
  m.impl("latent_prompt_attention", &latent_prompt_attention);
  m.impl("mingru_scan", &mingru_scan);
  m.impl("mingru_product", &mingru_product);
  m.impl("mingru_product_experts", &mingru_product_experts);
  m.impl("skinny_linear_experts", &skinny_linear_experts);
}

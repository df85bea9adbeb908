// The last product of a gated delta layer's decode step with the residual update (skinny_linear.hip), and the update of its convolution's kept inputs, in one
// launch. The inputs of shared queries and keys are read by several workgroups of the step's kernel, so they can move on only after all of it; as a
// launch of its own that is 3.1 us for 1536 channels of one sequence and 4.8 for 3072 of 16, a chain of three loads for a few KB, and nothing before the next
// step waits for it. Together, of 1024 columns one row 4.7 us, of 2048 columns 16 rows 5.6. A decode step of width 1024 with
// one such layer, one row 111.5 -> 110.7 us, three rows in 32 bits 1.1 us less, of width 2048 and 16 rows 226.0 -> 225.4.
#include "conv_update.h"
#include "hipserve/seq_kernels.h"
#include "skinny_block.h"

namespace hipserve {
namespace {

struct UpdateConvRest {
  ConvUpdate conv;
  int per_seq;   // workgroups of a sequence's channels
};
struct UpdateConvArgs {
  const void *x, *w, *p, *q;
  int x_ld, M, N, K, ni, split;
  SkinnyRest<kUpdate> rest;
  UpdateConvRest conv;
};

// Workgroups from `split` on are the convolution's, of kSkThreads channels each.
template <int XG, int NT, int DEPTH, bool F32, bool HALF>
__global__ __launch_bounds__(kSkThreads) void skinny_update_conv_kernel(
    const unsigned short* __restrict__ x, const unsigned short* __restrict__ w, void* p, const void* q, int x_ld, int M, int N, int K, int ni, int split,
    const SkinnyRest<kUpdate>, const UpdateConvRest) {
  using T = std::conditional_t<F32, float, unsigned short>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int b = blockIdx.x;
  if (b >= split) {
    const auto a = late_args<UpdateConvRest>(offsetof(UpdateConvArgs, conv));
    const int s = __builtin_amdgcn_readfirstlane((unsigned)(b - split) / (unsigned)a->per_seq);
    conv_update_block<T, 3>(s, (b - split - s * a->per_seq) * kSkThreads + threadIdx.x, a->conv.seq_cu, a->conv.seq_ctx, a->conv.seq_state,
                            static_cast<const T*>(a->conv.proj), a->conv.conv_state, a->conv.C, 4, a->conv.ld);
    return;
  }
  skinny_block<XG, NT, DEPTH, false, T, F32, kUpdate, HALF>(b, 0, 0, x, w, p, q, x_ld, M, N, K, ni, offsetof(UpdateConvArgs, rest), smem);
}

struct UpdateConvLaunch {
  void* out;
  const SkinnyNorm& norm;
  const void *x, *w, *bias;
  long x_ld;
  int M, N, K, nseq;
  const ConvUpdate& conv;
  hipStream_t s;
  template <int XG, int NT, int DEPTH, bool F32, bool HALF> bool run() const {
    constexpr int lds = Skinny<XG, NT, DEPTH, F32, HALF>::kLds, per = HALF ? 8 : 16 * NT;
    static const bool ok = allow_lds(&skinny_update_conv_kernel<XG, NT, DEPTH, F32, HALF>, lds);
    if (!ok) return false;
    const int split = (N + per - 1) / per, per_seq = (conv.C + kSkThreads - 1) / kSkThreads;
    skinny_update_conv_kernel<XG, NT, DEPTH, F32, HALF><<<split + nseq * per_seq, kSkThreads, lds, s>>>(
        (const unsigned short*)x, (const unsigned short*)w, norm.residual, norm.weight, (int)x_ld, M, N, K, norm.blocks, split,
        SkinnyRest<kUpdate>{0, N, 0, 0, -1, 0, 0.f, 0.f, norm.cols, norm.eps, out, norm.squares, bias}, UpdateConvRest{conv, per_seq});
    return true;
  }
};

}  // namespace

bool launch_skinny_update_conv(void* out, const SkinnyNorm& norm, const void* x, long x_ld, const void* w, const void* bias, bool f32, int M, int N, int K,
                               const ConvUpdate& conv, int nseq, hipStream_t s) {
  if (M <= 0 || N <= 0 || M > 32 || nseq <= 0 || conv.taps != 4) return false;
  if (f32) { x_ld *= 2; K *= 2; }   // in halves
  const UpdateConvLaunch l{out, norm, x, w, bias, x_ld, M, N, K, nseq, conv, s};
  return f32 ? run_update<true>(l, M, N, K, norm.blocks) : run_update<false>(l, M, N, K, norm.blocks);
}

}  // namespace hipserve

// The routed gated-MLP FFN as one call: permute plan, first expert GEMM with the activation, second
// with the routing weight, and the sum over each token's routes. Four to seven launches of the
// entry points they are alone, with every intermediate in one workspace. For a few tokens the
// kernels take less time than the calls around them did: 2 tokens, 128 experts top-8, 42 us of
// kernels in 73 us when each was a call of its own with its own buffers.
#include "pia_internal.h"

namespace pia {
namespace {

constexpr int FFN_BLOCK = 16;  // plan rows per block: what the expert GEMMs take per work item

struct FfnLayout {
  int64_t numel, mpad, sorted, experts, npp, align_ws, align_bytes, gemm_ws, gemm_bytes, act,
      route, total;
};

FfnLayout ffn_layout(int64_t tokens, int topk, int num_experts, int hidden, int inter, int64_t elt,
                     bool own_act, bool own_route) {
  FfnLayout o{};
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t p = at;
    at += ceil_div(bytes, 256) * 256;
    return p;
  };
  o.numel = tokens * topk;
  // every expert's padded region: numel + (E + 1)(block - 1), or one block per route if fewer
  o.mpad = o.numel < num_experts + 1 ? o.numel * FFN_BLOCK
                                     : o.numel + int64_t(num_experts + 1) * (FFN_BLOCK - 1);
  o.sorted = take(o.mpad * 4);
  o.experts = take(ceil_div(o.mpad, FFN_BLOCK) * 4);
  o.npp = take(4);
  o.align_bytes = pia_moe_align_workspace_bytes(num_experts);
  o.align_ws = take(o.align_bytes);
  o.gemm_bytes = pia_moe_expert_gemm_workspace_bytes(o.mpad, FFN_BLOCK);
  o.gemm_ws = take(o.gemm_bytes);
  o.act = own_act ? take(o.numel * inter * elt) : 0;
  o.route = own_route ? take(o.numel * hidden * elt) : 0;
  o.total = at;
  return o;
}

}  // namespace
}  // namespace pia

using namespace pia;

extern "C" int64_t pia_moe_ffn_workspace_bytes(int64_t num_tokens, int topk, int num_experts,
                                               int hidden, int inter, int dtype, int own_act,
                                               int own_route) {
  if (num_tokens < 0 || topk <= 0 || num_experts <= 0 || hidden <= 0 || inter <= 0 ||
      num_tokens > 0x7fffffff / topk)
    return 0;
  return ffn_layout(num_tokens, topk, num_experts, hidden, inter,
                    dtype == PIA_DTYPE_F32 ? 4 : 2, own_act != 0, own_route != 0)
      .total;
}

extern "C" int pia_moe_ffn(void* out, void* route_out, const void* x, int64_t ldx, const void* w1,
                           const void* w2, const float* topk_weights, const int32_t* topk_ids,
                           int64_t num_tokens, int topk, int num_experts, int hidden, int inter,
                           int activation, int weight_on_input, int dtype, void* act,
                           int64_t ld_act, void* workspace, int64_t workspace_bytes,
                           void* stream) {
  return pia_moe_ffn_bank(out, route_out, x, ldx, w1, w2, topk_weights, topk_ids, num_tokens, topk,
                          num_experts, 0, hidden, inter, activation, weight_on_input, dtype, act,
                          ld_act, workspace, workspace_bytes, stream);
}

extern "C" int pia_moe_ffn_bank(void* out, void* route_out, const void* x, int64_t ldx,
                                const void* w1, const void* w2, const float* topk_weights,
                                const int32_t* topk_ids, int64_t num_tokens, int topk,
                                int num_experts, int layer_experts, int hidden, int inter,
                                int activation, int weight_on_input, int dtype, void* act,
                                int64_t ld_act, void* workspace, int64_t workspace_bytes,
                                void* stream) {
  if (num_tokens < 0 || topk <= 0 || num_experts <= 0 || layer_experts < 0 || hidden <= 0 ||
      inter <= 0)
    return fail(PIA_EINVAL, "moe_ffn: invalid size");
  if (dtype != PIA_DTYPE_BF16 && dtype != PIA_DTYPE_F16 && dtype != PIA_DTYPE_F32)
    return fail(PIA_EUNSUPPORTED, "moe_ffn: dtype must be bf16, fp16 or fp32");
  if (num_tokens == 0) return 0;
  if (num_tokens > 0x7fffffff / topk) return fail(PIA_EINVAL, "moe_ffn: sizes must fit int32");
  if (activation < PIA_ACT_SILU || activation > PIA_ACT_GELU_TANH)
    return fail(PIA_EINVAL, "moe_ffn: unknown activation");
  if ((!out && !route_out) || !workspace || !topk_weights)
    return fail(PIA_EINVAL, "moe_ffn: null pointer");
  const FfnLayout o = ffn_layout(num_tokens, topk, num_experts, hidden, inter,
                                 dtype == PIA_DTYPE_F32 ? 4 : 2, !act, !route_out);
  if (workspace_bytes < o.total) return fail(PIA_EINVAL, "moe_ffn: workspace too small");
  if (!aligned(workspace, 256)) return fail(PIA_EINVAL, "moe_ffn: workspace must be 256-byte aligned");
  char* ws = static_cast<char*>(workspace);
  int32_t* sorted = reinterpret_cast<int32_t*>(ws + o.sorted);
  int32_t* experts = reinterpret_cast<int32_t*>(ws + o.experts);
  int32_t* npp = reinterpret_cast<int32_t*>(ws + o.npp);
  void* a = act ? act : ws + o.act;
  const int64_t lda = act ? ld_act : inter;
  void* r = route_out ? route_out : ws + o.route;
  if (int rc = pia_moe_align_block_size(sorted, experts, npp, nullptr, topk_ids, o.numel,
                                        num_experts, FFN_BLOCK, o.mpad, ws + o.align_ws,
                                        o.align_bytes, stream))
    return rc;
  if (int rc = expert_gemm(a, x, w1, topk_weights, sorted, experts, npp, o.mpad, FFN_BLOCK,
                           o.numel, topk, ldx, num_experts, layer_experts, 2 * inter, hidden, lda,
                           activation, weight_on_input ? 1 : 0, dtype, ws + o.gemm_ws,
                           o.gemm_bytes, stream))
    return rc;
  if (int rc = expert_gemm(r, a, w2, topk_weights, sorted, experts, npp, o.mpad, FFN_BLOCK, o.numel,
                           1, lda, num_experts, layer_experts, hidden, inter, hidden, PIA_ACT_NONE,
                           weight_on_input ? 0 : 1, dtype, ws + o.gemm_ws, o.gemm_bytes, stream))
    return rc;
  if (!out) return 0;
  return pia_moe_sum_reduce(out, r, num_tokens, topk, hidden, dtype, stream);
}

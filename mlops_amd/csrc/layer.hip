// Launch sequences of the MoE layer: steps of one pass that always follow one
// another, enqueued by one call from one workspace. A layer call on few
// tokens is bound by the host (14 launches of 2-7 us kernels forward, 32
// forward and backward), so the steps between the router GEMM and the up
// projection, from the activation to the combine, and from the SwiGLU
// backward to the logit gradient are one crossing of the language boundary
// each instead of one per kernel.
#include "common.h"

// router.hip: the routing of at most 64 tokens; returns 1 outside its range.
bool mi355x_route_small_serves(int tokens, int experts, int top_k, int mode, int n_group,
                               int topk_group, int segments);
int mi355x_route_small(float* logits, const float* partial, int parts, int tokens, int experts,
                       int top_k, int mode, const float* bias, int n_group, int topk_group,
                       float routed_scaling, const int32_t* forced_ids, int segments,
                       float* weights, int32_t* ids, int64_t* counts, int32_t* offsets,
                       int32_t* order, int32_t* slots, float* aux, float* prob_sum, void* stream);
// router_logits.hip: its logits in parts, and the quantized token rows.
int mi355x_router_logits_parts(int width);
int mi355x_router_logits_launch(const void* x, const void* weight, int weight_fp32, int tokens,
                                int experts, int width, float* partial, int pitch, int quantize,
                                uint8_t* q, float* scales, void* stream);

namespace {

// Walks a workspace in 256-byte steps; with a null base it only counts.
struct Carver {
  uint8_t* base;
  size_t used;
  void* take(size_t bytes) {
    void* at = base == nullptr ? nullptr : base + used;
    used += (bytes + 255) / 256 * 256;
    return at;
  }
};

struct RouteSpace {
  void *plan, *stats;
  int32_t* seg_counts;
  size_t plan_bytes, stats_bytes, total;
};
RouteSpace route_space(void* base, int tokens, int experts, int top_k, int segments, int nchunks) {
  Carver c = {(uint8_t*)base, 0};
  RouteSpace s;
  s.plan_bytes = mi355x_permute_plan_workspace_size(tokens * top_k, experts);
  s.stats_bytes = mi355x_router_stats_workspace_size(nchunks, experts);
  s.plan = c.take(s.plan_bytes);
  s.stats = c.take(s.stats_bytes);
  s.seg_counts = (int32_t*)c.take((size_t)segments * experts * sizeof(int32_t));
  s.total = c.used;
  return s;
}

struct DownSpace {
  uint8_t* q;
  float* scales;
  void *y, *tail;
  size_t tail_bytes, total;
};
DownSpace down_space(void* base, int rows, int hidden, int inter, int experts) {
  Carver c = {(uint8_t*)base, 0};
  DownSpace s;
  s.q = (uint8_t*)c.take((size_t)rows * inter);
  s.scales = (float*)c.take((size_t)rows * (inter / 128) * sizeof(float));
  s.y = c.take((size_t)rows * hidden * 2);
  s.tail_bytes = mi355x_gemm_tail_workspace_size(rows, experts, hidden, inter);
  s.tail = s.tail_bytes > 0 ? c.take(s.tail_bytes) : nullptr;
  s.total = c.used;
  return s;
}

// The backward's buffers. `gather` holds dy's transposed operand, then x's
// (the first is spent once dW2 is formed).
struct BackwardSpace {
  int32_t* blocks;
  uint8_t *dhq, *dh_t, *ap_t, *gather_t;
  float *dh_scales, *dh_t_scales, *ap_t_scales, *gather_scales, *dscore;
  void *dx, *tail, *swiglu, *router;
  size_t tail_bytes, swiglu_bytes, router_bytes, total;
};
BackwardSpace backward_space(void* base, int tokens, int hidden, int inter, int experts, int top_k,
                             int need_w13, int need_w2, int router_kernel) {
  Carver c = {(uint8_t*)base, 0};
  BackwardSpace s = {};
  const size_t rows = (size_t)tokens * top_k;
  const size_t padded = mi355x_wgrad_padded_rows((int)rows, experts);
  const size_t h = hidden, i = inter;
  s.blocks = (int32_t*)c.take(padded / 128 * 2 * sizeof(int32_t));
  s.dhq = (uint8_t*)c.take(rows * 2 * i);
  s.dh_scales = (float*)c.take(2 * i / 128 * rows * sizeof(float));
  if (need_w13) {
    s.dh_t = (uint8_t*)c.take(2 * i * padded);
    s.dh_t_scales = (float*)c.take(padded / 128 * 2 * i * sizeof(float));
  }
  if (need_w2) {
    s.ap_t = (uint8_t*)c.take(i * padded);
    s.ap_t_scales = (float*)c.take(padded / 128 * i * sizeof(float));
  }
  if (need_w13 || need_w2) {
    s.gather_t = (uint8_t*)c.take(h * padded);
    s.gather_scales = (float*)c.take(padded / 128 * h * sizeof(float));
  }
  s.dscore = (float*)c.take(rows * sizeof(float));
  s.dx = c.take(rows * h * 2);
  s.tail_bytes = mi355x_gemm_tail_workspace_size((int)rows, experts, hidden, 2 * inter);
  if (s.tail_bytes > 0) s.tail = c.take(s.tail_bytes);
  s.swiglu_bytes = mi355x_swiglu_bwd_quantize_workspace_size((int)rows, inter);
  s.swiglu = c.take(s.swiglu_bytes);
  if (router_kernel) {
    s.router_bytes = mi355x_router_weight_grad_workspace_size(tokens, experts, hidden);
    s.router = c.take(s.router_bytes);
  }
  s.total = c.used;
  return s;
}

#define STEP(call)                         \
  do {                                     \
    const int rc_ = (call);                \
    if (rc_ != MI355X_OK) return rc_;      \
  } while (0)

}  // namespace

extern "C" size_t mi355x_moe_route_workspace_size(int tokens, int experts, int top_k, int segments,
                                                  int nchunks) {
  return route_space(nullptr, tokens, experts, top_k, segments, nchunks).total;
}

extern "C" int mi355x_moe_route(const float* logits, int tokens, int experts, int top_k, int mode,
                                const float* bias, int n_group, int topk_group,
                                float routed_scaling, const int32_t* forced_ids, int segments,
                                const int32_t* seg_offsets, const int32_t* chunk_table,
                                int nchunks, float* weights, int32_t* ids, int64_t* counts,
                                int32_t* offsets, int32_t* order, int32_t* slots, float* aux,
                                float* prob_sum, void* workspace, size_t workspace_bytes,
                                void* stream) {
  MI355X_REQUIRE(tokens >= 0 && experts > 0 && top_k > 0, "moe_route: bad sizes");
  const RouteSpace s = route_space(workspace, tokens, experts, top_k, segments, nchunks);
  MI355X_REQUIRE(workspace_bytes >= s.total, "moe_route: workspace too small");
  MI355X_REQUIRE(((uintptr_t)workspace & 15) == 0,
                 "moe_route: the workspace must be 16-byte aligned");
  const int small = mi355x_route_small((float*)logits, nullptr, 0, tokens, experts, top_k, mode,
                                       bias, n_group, topk_group, routed_scaling, forced_ids,
                                       segments, weights, ids, counts, offsets, order, slots, aux,
                                       prob_sum, stream);
  if (small <= 0) return small;
  STEP(mi355x_router_topk(logits, tokens, experts, top_k, mode, bias, n_group, topk_group,
                          routed_scaling, forced_ids, weights, ids, stream));
  STEP(mi355x_permute_plan(ids, tokens * top_k, experts, counts, offsets, order, slots, s.plan,
                           s.plan_bytes, stream));
  return mi355x_router_stats(logits, ids, tokens, experts, top_k, mode, segments, seg_offsets,
                             chunk_table, nchunks, aux, prob_sum, s.seg_counts, s.stats,
                             s.stats_bytes, stream);
}

extern "C" size_t mi355x_moe_route_tokens_workspace_size(int tokens, int experts, int top_k,
                                                         int mode, int n_group, int topk_group,
                                                         int width) {
  if (width <= 0 || width % 128 != 0 || experts <= 0 || top_k <= 0 ||
      !mi355x_route_small_serves(tokens, experts, top_k, mode, n_group, topk_group, 1))
    return 0;
  const size_t pitch = ((size_t)tokens * experts + 3) / 4 * 4;
  return mi355x_router_logits_parts(width) * pitch * sizeof(float);
}

extern "C" int mi355x_moe_route_tokens(const void* x, const void* weight, int weight_fp32,
                                       int tokens, int experts, int width, int quantize,
                                       uint8_t* q, float* scales, int top_k, int mode,
                                       const float* bias, int n_group, int topk_group,
                                       float routed_scaling, const int32_t* forced_ids,
                                       float* logits, float* weights, int32_t* ids,
                                       int64_t* counts, int32_t* offsets, int32_t* order,
                                       int32_t* slots, float* aux, float* prob_sum,
                                       void* workspace, size_t workspace_bytes, void* stream) {
  const size_t need = mi355x_moe_route_tokens_workspace_size(tokens, experts, top_k, mode, n_group,
                                                             topk_group, width);
  MI355X_REQUIRE(need > 0, "moe_route_tokens: outside the range of the fused routing");
  MI355X_REQUIRE(workspace_bytes >= need, "moe_route_tokens: workspace too small");
  MI355X_REQUIRE(quantize >= MI355X_ROUTE_QUANTIZE_NONE && quantize <= MI355X_ROUTE_QUANTIZE_ROWS,
                 "moe_route_tokens: unknown quantization %d", quantize);
  MI355X_REQUIRE(quantize == MI355X_ROUTE_QUANTIZE_NONE || (q != nullptr && scales != nullptr),
                 "moe_route_tokens: the quantized rows need q and scales");
  MI355X_REQUIRE((((uintptr_t)x | (uintptr_t)weight) & 15) == 0,
                 "moe_route_tokens: operands must be 16-byte aligned");
  MI355X_REQUIRE(((uintptr_t)workspace & 15) == 0,
                 "moe_route_tokens: the workspace must be 16-byte aligned");
  float* partial = (float*)workspace;
  STEP(mi355x_router_logits_launch(x, weight, weight_fp32, tokens, experts, width, partial,
                                   (tokens * experts + 3) / 4 * 4, quantize, q, scales, stream));
  return mi355x_route_small(logits, partial, mi355x_router_logits_parts(width), tokens, experts,
                            top_k, mode, bias, n_group, topk_group, routed_scaling, forced_ids, 1,
                            weights, ids, counts, offsets, order, slots, aux, prob_sum, stream);
}

extern "C" size_t mi355x_moe_down_workspace_size(int rows, int hidden, int inter, int experts) {
  return down_space(nullptr, rows, hidden, inter, experts).total;
}

extern "C" int mi355x_moe_down(const void* h13, int tokens, int top_k, int hidden, int inter,
                               float limit, int row_scaled, const uint8_t* w2,
                               const float* w2_scale, int experts, const int32_t* offsets,
                               const int32_t* slots, const float* weights, const void* residual,
                               void* out, void* workspace, size_t workspace_bytes, void* stream) {
  MI355X_REQUIRE(tokens >= 0 && top_k > 0 && hidden > 0 && inter > 0 && inter % 128 == 0,
                 "moe_down: bad sizes");
  const int rows = tokens * top_k;
  const DownSpace s = down_space(workspace, rows, hidden, inter, experts);
  MI355X_REQUIRE(workspace_bytes >= s.total, "moe_down: workspace too small");
  MI355X_REQUIRE(((uintptr_t)workspace & 15) == 0,
                 "moe_down: the workspace must be 16-byte aligned");
  if (row_scaled)
    STEP(mi355x_swiglu_quantize_rows_current_fp8(h13, rows, inter, limit, s.q, s.scales, nullptr,
                                                 stream));
  else
    STEP(mi355x_swiglu_quantize_fp8(h13, rows, inter, limit, s.q, s.scales, nullptr, stream));
  mi355x_gemm_args g = {};
  g.a = s.q;
  g.a_scale = s.scales;
  g.w = w2;
  g.w_scale = w2_scale;
  g.offsets = offsets;
  g.out = s.y;
  g.workspace = s.tail;
  g.workspace_bytes = s.tail_bytes;
  g.rows = rows;
  g.a_rows_div = 1;
  g.experts = experts;
  g.n = hidden;
  g.k = inter;
  g.row_scaled = row_scaled;
  STEP(mi355x_gemm_fp8(&g, stream));
  return mi355x_unpermute_combine(s.y, slots, weights, residual, tokens, top_k, hidden, out,
                                  stream);
}

extern "C" size_t mi355x_moe_block_bwd_workspace_size(int tokens, int hidden, int inter,
                                                      int experts, int top_k, int need_w13,
                                                      int need_w2, int router_kernel) {
  return backward_space(nullptr, tokens, hidden, inter, experts, top_k, need_w13, need_w2,
                        router_kernel).total;
}

extern "C" size_t mi355x_moe_block_bwd_args_size(void) {
  return sizeof(mi355x_moe_block_bwd_args);
}

extern "C" int mi355x_moe_block_bwd(const mi355x_moe_block_bwd_args* a, void* stream) {
  MI355X_REQUIRE(a != nullptr && a->tokens >= 0 && a->top_k > 0 && a->hidden > 0 && a->inter > 0 &&
                     a->inter % 128 == 0 && a->hidden % 128 == 0 && a->experts > 0,
                 "moe_block_bwd: bad sizes");
  const int need_w13 = a->grad_w13 != nullptr, need_w2 = a->grad_w2 != nullptr;
  const int rows = a->tokens * a->top_k, h = a->hidden, i = a->inter;
  const BackwardSpace s =
      backward_space(a->workspace, a->tokens, h, i, a->experts, a->top_k, need_w13, need_w2,
                     a->grad_router != nullptr);
  MI355X_REQUIRE(a->workspace_bytes >= s.total, "moe_block_bwd: workspace too small");
  MI355X_REQUIRE(((uintptr_t)a->workspace & 15) == 0,
                 "moe_block_bwd: the workspace must be 16-byte aligned");
  const int padded = (int)mi355x_wgrad_padded_rows(rows, a->experts);
  STEP(mi355x_padded_row_blocks(a->offsets, a->experts, padded, s.blocks, stream));
  STEP(mi355x_swiglu_bwd_quantize(a->r, a->h13, a->route_weights, a->order, s.blocks, rows, i,
                                  padded, a->limit, s.dhq, s.dh_scales, s.dh_t, s.dh_t_scales,
                                  s.ap_t, s.ap_t_scales, s.dscore, s.swiglu, s.swiglu_bytes,
                                  stream));
  if (need_w2) {
    if (rows > 0)
      STEP(mi355x_quantize_transpose_fp8(a->dy, h, h, a->order, a->top_k, 0, s.blocks, padded,
                                         s.gather_t, s.gather_scales, stream));
    STEP(mi355x_gemm_fp8_block_wgrad(s.gather_t, s.gather_scales, h, s.ap_t, s.ap_t_scales, i,
                                     padded, a->offsets, a->experts, a->grad_w2,
                                     a->weight_grads_fp32, stream));
  }
  mi355x_gemm_args g = {};
  g.a = s.dhq;
  g.a_scale = s.dh_scales;
  g.w = a->w13;
  g.w_scale = a->w13_scale;
  g.offsets = a->offsets;
  g.out = s.dx;
  g.workspace = s.tail;
  g.workspace_bytes = s.tail_bytes;
  g.rows = rows;
  g.a_rows_div = 1;
  g.experts = a->experts;
  g.n = h;
  g.k = 2 * i;
  g.kmajor = a->w13_kmajor;
  g.w_scale_t = !a->w13_kmajor;
  STEP(mi355x_gemm_fp8(&g, stream));
  if (need_w13) {
    if (rows > 0)
      STEP(mi355x_quantize_transpose_fp8(a->x, h, h, a->order, a->top_k, 0, s.blocks, padded,
                                         s.gather_t, s.gather_scales, stream));
    STEP(mi355x_gemm_fp8_block_wgrad(s.dh_t, s.dh_t_scales, 2 * i, s.gather_t, s.gather_scales, h,
                                     padded, a->offsets, a->experts, a->grad_w13,
                                     a->weight_grads_fp32, stream));
  }
  STEP(mi355x_unpermute_sum(s.dx, a->slots, a->tokens, a->top_k, h, a->grad_x, stream));
  STEP(mi355x_router_topk_bwd_split(a->logits, a->route_weights, a->route_ids, s.dscore, a->slots,
                                    a->tokens, a->experts, a->top_k, a->mode, a->grad_aux,
                                    a->grad_prob_sum, a->offsets, a->segments, a->seg_offsets,
                                    a->seg_counts, nullptr, a->pieces, stream));
  if (a->grad_router != nullptr)
    STEP(mi355x_router_weight_grad(a->pieces, a->x, a->tokens, a->experts, h, a->grad_router,
                                   s.router, s.router_bytes, stream));
  return MI355X_OK;
}

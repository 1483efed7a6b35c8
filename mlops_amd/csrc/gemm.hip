// Entry points of the ragged grouped block-FP8 GEMMs for gfx950 (CDNA4): the
// argument checks and the choice of kernel. The grouped GEMMs are gemm_v2.hip
// (256 x 256 tiles) and gemm_tile.hip (smaller ones), the weight gradient is
// gemm_wgrad.hip.
//
// Math: every 128-wide K step is exactly one scale block of both operands,
// and one v_mfma_f32_16x16x128_f8f6f4 covers 16x16 outputs over those 128 K.
// So each MFMA produces the raw partial of one scale block, which is folded
// into the fp32 accumulator with its (row scale x weight-block scale):
//     acc += mfma(a, b, 0) * (sa[row] * sb)
// That is the reference's promoted accumulation (acc_sum += acc * scale per
// K block) at the granularity the hardware gives for free.
//
// MFMA operand layout (verified on MI355X): lane l supplies row l%16 of A
// and column l%16 of B, each as 32 consecutive K bytes starting at
// 32*(l/16); the 4 outputs of lane l are rows 4*(l/16)+i, column l%16.
#include "common.h"

namespace {

constexpr int BM = 128, BN = 128, BK = 128;  // what every GEMM's M (weight gradient), N and K are multiples of
constexpr int kMaxExperts = 512;

}  // namespace

int mi355x_gemm_v2_launch(const uint8_t* a, const float* a_scale, int rows, const uint8_t* w,
                          const float* w_scale, int w_scale_t, int experts, int n, int k,
                          const int32_t* offsets, int interleave, const void* addend, void* out,
                          uint8_t* act_q, float* act_scales, float limit, const void* lora_z,
                          const void* lora_b, int lora_rank, void* stream,
                          const int32_t* a_rows = nullptr, int a_total = 0, int a_rows_div = 1);
int mi355x_gemm_v2_kmajor_launch(const uint8_t* a, const float* a_scale, int rows,
                                 const uint8_t* w, const float* w_scale, int experts, int n, int k,
                                 const int32_t* offsets, void* out, void* stream,
                                 const int32_t* a_rows = nullptr, int a_total = 0, int a_rows_div = 1);

int mi355x_gemm_v2_rowwise_launch(const uint8_t* a, const float* a_scale, int rows,
                                  const uint8_t* w, const float* w_scale, int experts, int n,
                                  int k, const int32_t* offsets, const void* lora_z,
                                  const void* lora_b, int lora_rank, void* out, void* stream,
                                  const int32_t* a_rows = nullptr, int a_total = 0, int a_rows_div = 1);

int mi355x_wgrad_launch(const uint8_t* p, const float* p_scale, int m_features, const uint8_t* q,
                        const float* q_scale, int n_features, int padded, const int32_t* offsets,
                        int experts, void* out, int out_fp32, void* stream);

extern "C" int mi355x_gemm_fp8_block(const uint8_t* a, const float* a_scale, int rows,
                                     const uint8_t* w, const float* w_scale, int w_scale_t,
                                     int experts, int n, int k, const int32_t* offsets,
                                     int interleave, const void* addend, void* out,
                                     void* stream) {
  MI355X_REQUIRE(experts > 0 && experts <= kMaxExperts, "gemm: experts must be in [1, %d]",
                 kMaxExperts);
  MI355X_REQUIRE(n > 0 && n % BN == 0, "gemm: N must be a multiple of %d, got %d", BN, n);
  MI355X_REQUIRE(k > 0 && k % BK == 0, "gemm: K must be a multiple of %d, got %d", BK, k);
  MI355X_REQUIRE(!interleave || (n / 2) % 64 == 0,
                 "gemm: a gate/up weight needs halves that are multiples of 64");
  MI355X_REQUIRE(rows >= 0, "gemm: negative rows");
  if (rows == 0) return MI355X_OK;
  const int v2 = mi355x_gemm_v2_launch(a, a_scale, rows, w, w_scale, w_scale_t, experts, n, k,
                                       offsets, interleave, addend, out, nullptr, nullptr, 0.0f,
                                       nullptr, nullptr, 0, stream);
  if (v2 < 0) return v2;
  MI355X_REQUIRE(v2 == 0, "gemm: shape outside the pipelined kernels");
  return MI355X_OK;
}

extern "C" int mi355x_gemm_fp8_block_kmajor(const uint8_t* a, const float* a_scale, int rows,
                                            const uint8_t* w, const float* w_scale, int experts,
                                            int n, int k, const int32_t* offsets, void* out,
                                            void* stream) {
  MI355X_REQUIRE(experts > 0 && experts <= kMaxExperts,
                 "gemm_kmajor: experts must be in [1, %d]", kMaxExperts);
  MI355X_REQUIRE(n > 0 && n % 256 == 0, "gemm_kmajor: N must be a multiple of 256, got %d", n);
  MI355X_REQUIRE(k > 0 && k % BK == 0, "gemm_kmajor: K must be a multiple of %d, got %d", BK, k);
  MI355X_REQUIRE(rows >= 0, "gemm_kmajor: negative rows");
  MI355X_REQUIRE((uint64_t)(k - 1) * (uint64_t)n + 256 < (1ull << 32),
                 "gemm_kmajor: a weight slice beyond 32-bit offsets");
  if (rows == 0) return MI355X_OK;
  const int v2 = mi355x_gemm_v2_kmajor_launch(a, a_scale, rows, w, w_scale, experts, n, k, offsets,
                                              out, stream);
  if (v2 < 0) return v2;
  MI355X_REQUIRE(v2 == 0, "gemm_kmajor: shape outside the pipelined kernel");
  return MI355X_OK;
}

// Gathered-A forms: GEMM row r (expert-sorted, offsets) reads row
// a_rows[r] of a [a_total, K] and its 1x128 scales a_scale[a_total][K/128]
// (token-major, as mi355x_quantize_token_rows_fp8 writes them)
// (the activation quantized once per token; a_rows = the token of each
// routed row). Pipelined kernel only (N a multiple of 256).
static int gathered_checks(int a_total, const int32_t* a_rows, int a_rows_div, int rows, int k) {
  MI355X_REQUIRE(a_rows != nullptr && a_total > 0, "gemm gathered: a_rows and a_total required");
  MI355X_REQUIRE(a_rows_div >= 1 && (uint64_t)a_total * (uint64_t)a_rows_div < (1ull << 31),
                 "gemm gathered: a_rows_div must be >= 1 with a_total * a_rows_div < 2^31");
  MI355X_REQUIRE((uint64_t)a_total * (uint64_t)k < (1ull << 32),
                 "gemm gathered: gathered rows beyond 32-bit offsets");
  MI355X_REQUIRE(rows >= 0, "gemm gathered: negative rows");
  return MI355X_OK;
}

extern "C" int mi355x_gemm_fp8_block_gathered(const uint8_t* a, const float* a_scale, int a_total,
                                              const int32_t* a_rows, int a_rows_div, int rows, const uint8_t* w,
                                              const float* w_scale, int experts, int n, int k,
                                              const int32_t* offsets, int interleave, void* out,
                                              void* stream) {
  MI355X_REQUIRE(experts > 0 && experts <= kMaxExperts, "gemm: experts must be in [1, %d]",
                 kMaxExperts);
  MI355X_REQUIRE(n > 0 && n % 256 == 0, "gemm gathered: N must be a multiple of 256, got %d", n);
  MI355X_REQUIRE(k > 0 && k % BK == 0, "gemm: K must be a multiple of %d, got %d", BK, k);
  MI355X_REQUIRE(!interleave || (n / 2) % 128 == 0,
                 "gemm gathered: a gate/up weight needs halves that are multiples of 128");
  const int c = gathered_checks(a_total, a_rows, a_rows_div, rows, k);
  if (c != MI355X_OK) return c;
  if (rows == 0) return MI355X_OK;
  const int v2 = mi355x_gemm_v2_launch(a, a_scale, rows, w, w_scale, 0, experts, n, k, offsets,
                                       interleave, nullptr, out, nullptr, nullptr, 0.0f, nullptr,
                                       nullptr, 0, stream, a_rows, a_total, a_rows_div);
  if (v2 < 0) return v2;
  MI355X_REQUIRE(v2 == 0, "gemm gathered: shape outside the pipelined kernel");
  return MI355X_OK;
}

extern "C" int mi355x_gemm_fp8_block_kmajor_gathered(const uint8_t* a, const float* a_scale,
                                                     int a_total, const int32_t* a_rows, int a_rows_div, int rows,
                                                     const uint8_t* w, const float* w_scale,
                                                     int experts, int n, int k,
                                                     const int32_t* offsets, void* out,
                                                     void* stream) {
  MI355X_REQUIRE(experts > 0 && experts <= kMaxExperts,
                 "gemm_kmajor: experts must be in [1, %d]", kMaxExperts);
  MI355X_REQUIRE(n > 0 && n % 256 == 0, "gemm_kmajor: N must be a multiple of 256, got %d", n);
  MI355X_REQUIRE(k > 0 && k % BK == 0, "gemm_kmajor: K must be a multiple of %d, got %d", BK, k);
  MI355X_REQUIRE((uint64_t)(k - 1) * (uint64_t)n + 256 < (1ull << 32),
                 "gemm_kmajor: a weight slice beyond 32-bit offsets");
  const int c = gathered_checks(a_total, a_rows, a_rows_div, rows, k);
  if (c != MI355X_OK) return c;
  if (rows == 0) return MI355X_OK;
  const int v2 = mi355x_gemm_v2_kmajor_launch(a, a_scale, rows, w, w_scale, experts, n, k, offsets,
                                              out, stream, a_rows, a_total, a_rows_div);
  if (v2 < 0) return v2;
  MI355X_REQUIRE(v2 == 0, "gemm_kmajor: shape outside the pipelined kernel");
  return MI355X_OK;
}

extern "C" int mi355x_gemm_fp8_rowwise_gathered(const uint8_t* a, const float* a_scale,
                                                int a_total, const int32_t* a_rows, int a_rows_div, int rows,
                                                const uint8_t* w, const float* w_scale,
                                                int experts, int n, int k,
                                                const int32_t* offsets, void* out, void* stream) {
  MI355X_REQUIRE(experts > 0 && experts <= kMaxExperts, "gemm_rowwise: experts must be in [1, %d]",
                 kMaxExperts);
  MI355X_REQUIRE(n > 0 && n % 256 == 0, "gemm_rowwise: N must be a multiple of 256, got %d", n);
  MI355X_REQUIRE(k > 0 && k % BK == 0, "gemm_rowwise: K must be a multiple of %d, got %d", BK, k);
  const int c = gathered_checks(a_total, a_rows, a_rows_div, rows, k);
  if (c != MI355X_OK) return c;
  if (rows == 0) return MI355X_OK;
  const int v2 = mi355x_gemm_v2_rowwise_launch(a, a_scale, rows, w, w_scale, experts, n, k, offsets,
                                               nullptr, nullptr, 0, out, stream, a_rows, a_total, a_rows_div);
  if (v2 < 0) return v2;
  MI355X_REQUIRE(v2 == 0, "gemm_rowwise gathered: shape outside the pipelined kernel");
  return MI355X_OK;
}

extern "C" int mi355x_gemm_fp8_rowwise(const uint8_t* a, const float* a_scale, int rows,
                                       const uint8_t* w, const float* w_scale, int experts, int n,
                                       int k, const int32_t* offsets, void* out, void* stream) {
  MI355X_REQUIRE(experts > 0 && experts <= kMaxExperts, "gemm_rowwise: experts must be in [1, %d]",
                 kMaxExperts);
  MI355X_REQUIRE(n > 0 && n % 256 == 0, "gemm_rowwise: N must be a multiple of 256, got %d", n);
  MI355X_REQUIRE(k > 0 && k % BK == 0, "gemm_rowwise: K must be a multiple of %d, got %d", BK, k);
  MI355X_REQUIRE(rows >= 0, "gemm_rowwise: negative rows");
  if (rows == 0) return MI355X_OK;
  const int v2 = mi355x_gemm_v2_rowwise_launch(a, a_scale, rows, w, w_scale, experts, n, k,
                                               offsets, nullptr, nullptr, 0, out, stream);
  if (v2 < 0) return v2;
  MI355X_REQUIRE(v2 == 0, "gemm_rowwise: shape outside the pipelined kernel");
  return MI355X_OK;
}

extern "C" int mi355x_gemm_fp8_rowwise_lora(const uint8_t* a, const float* a_scale, int rows,
                                            const uint8_t* w, const float* w_scale, int experts,
                                            int n, int k, const int32_t* offsets,
                                            const void* lora_z, const void* lora_b, int lora_rank,
                                            void* out, void* stream) {
  MI355X_REQUIRE(experts > 0 && experts <= kMaxExperts,
                 "gemm_rowwise_lora: experts must be in [1, %d]", kMaxExperts);
  MI355X_REQUIRE(n > 0 && n % 256 == 0, "gemm_rowwise_lora: N must be a multiple of 256, got %d",
                 n);
  MI355X_REQUIRE(k > 0 && k % BK == 0, "gemm_rowwise_lora: K must be a multiple of %d", BK);
  MI355X_REQUIRE(lora_rank >= 16 && lora_rank <= 256 && lora_rank % 16 == 0,
                 "gemm_rowwise_lora: rank must be a multiple of 16 in [16, 256], got %d",
                 lora_rank);
  MI355X_REQUIRE(lora_z != nullptr && lora_b != nullptr, "gemm_rowwise_lora: z and b are required");
  MI355X_REQUIRE(rows >= 0, "gemm_rowwise_lora: negative rows");
  if (rows == 0) return MI355X_OK;
  const int v2 = mi355x_gemm_v2_rowwise_launch(a, a_scale, rows, w, w_scale, experts, n, k,
                                               offsets, lora_z, lora_b, lora_rank, out, stream);
  if (v2 < 0) return v2;
  MI355X_REQUIRE(v2 == 0, "gemm_rowwise_lora: shape outside the pipelined kernel");
  return MI355X_OK;
}

extern "C" int mi355x_gemm_fp8_block_lora(const uint8_t* a, const float* a_scale, int rows,
                                          const uint8_t* w, const float* w_scale, int w_scale_t,
                                          int experts, int n, int k, const int32_t* offsets,
                                          int interleave, const void* lora_z, const void* lora_b,
                                          int lora_rank, void* out, void* stream) {
  MI355X_REQUIRE(experts > 0 && experts <= kMaxExperts, "gemm_lora: experts must be in [1, %d]",
                 kMaxExperts);
  MI355X_REQUIRE(n > 0 && n % 256 == 0 && (!interleave || (n / 2) % 128 == 0),
                 "gemm_lora: N must be a multiple of 256 (2I of 128), got %d", n);
  MI355X_REQUIRE(k > 0 && k % BK == 0, "gemm_lora: K must be a multiple of %d, got %d", BK, k);
  MI355X_REQUIRE(lora_rank > 0 && lora_rank % 16 == 0 && lora_rank <= 256,
                 "gemm_lora: the (padded) rank must be a multiple of 16 in [16, 256], got %d",
                 lora_rank);
  MI355X_REQUIRE(lora_z != nullptr && lora_b != nullptr, "gemm_lora: z and b are required");
  MI355X_REQUIRE(rows >= 0, "gemm_lora: negative rows");
  if (rows == 0) return MI355X_OK;
  const int v2 = mi355x_gemm_v2_launch(a, a_scale, rows, w, w_scale, w_scale_t, experts, n, k,
                                       offsets, interleave, nullptr, out, nullptr, nullptr, 0.0f,
                                       lora_z, lora_b, lora_rank, stream);
  if (v2 < 0) return v2;
  MI355X_REQUIRE(v2 == 0, "gemm_lora: shape outside the pipelined kernel");
  return MI355X_OK;
}

extern "C" int mi355x_gemm_fp8_block_swiglu(const uint8_t* a, const float* a_scale, int rows,
                                            const uint8_t* w, const float* w_scale, int experts,
                                            int n, int k, const int32_t* offsets,
                                            const void* addend, float limit, void* h,
                                            uint8_t* act_q, float* act_scales, void* stream) {
  MI355X_REQUIRE(experts > 0 && experts <= kMaxExperts, "gemm_swiglu: experts must be in [1, %d]",
                 kMaxExperts);
  MI355X_REQUIRE(n > 0 && n % BN == 0 && (n / 2) % 128 == 0,
                 "gemm_swiglu: 2I must be a multiple of 256, got %d", n);
  MI355X_REQUIRE(k > 0 && k % BK == 0, "gemm_swiglu: K must be a multiple of %d, got %d", BK, k);
  MI355X_REQUIRE(rows >= 0, "gemm_swiglu: negative rows");
  if (rows == 0) return MI355X_OK;
  const int v2 = mi355x_gemm_v2_launch(a, a_scale, rows, w, w_scale, 0, experts, n, k, offsets, 1,
                                       addend, h, act_q, act_scales, limit, nullptr, nullptr, 0,
                                       stream);
  if (v2 <= 0) return v2;
  // Shapes outside the pipelined kernel: the GEMM, then the SwiGLU pass.
  const int rc = mi355x_gemm_fp8_block(a, a_scale, rows, w, w_scale, 0, experts, n, k, offsets, 1,
                                       addend, h, stream);
  if (rc != MI355X_OK) return rc;
  return mi355x_swiglu_quantize_fp8(h, rows, n / 2, limit, act_q, act_scales, nullptr, stream);
}

extern "C" int mi355x_gemm_fp8_block_wgrad(const uint8_t* p, const float* p_scale,
                                           int m_features, const uint8_t* q,
                                           const float* q_scale, int n_features, int padded,
                                           const int32_t* offsets, int experts, void* out,
                                           int out_fp32, void* stream) {
  MI355X_REQUIRE(experts > 0 && experts <= kMaxExperts, "wgrad: experts must be in [1, %d]",
                 kMaxExperts);
  MI355X_REQUIRE(m_features > 0 && m_features % BM == 0 && n_features > 0 && n_features % BN == 0,
                 "wgrad: feature counts must be multiples of 128");
  MI355X_REQUIRE(padded % 128 == 0, "wgrad: padded rows must be a multiple of 128");
  return mi355x_wgrad_launch(p, p_scale, m_features, q, q_scale, n_features, padded, offsets,
                             experts, out, out_fp32, stream);
}

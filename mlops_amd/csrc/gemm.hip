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
// and column l%16 of B, each as the K bytes 16g..16g+15 and 64+16g..64+16g+15
// with g = l/16; its 4 outputs are rows 4g+i, column l%16.
#include "common.h"

namespace {

constexpr int BM = 128, BN = 128, BK = 128;  // what every GEMM's M (weight gradient), N and K are multiples of
constexpr int kMaxExperts = 512;

}  // namespace

int mi355x_gemm_v2_launch(const uint8_t* a, const float* a_scale, int rows, const uint8_t* w,
                          const float* w_scale, int w_scale_t, int experts, int n, int k,
                          const int32_t* offsets, int interleave, const void* addend, void* out,
                          uint8_t* act_q, float* act_scales, float limit, const void* lora_z,
                          const void* lora_b, int lora_rank, void* stream, const int32_t* a_rows,
                          int a_rows_div, float* partial);
int mi355x_gemm_v2_kmajor_launch(const uint8_t* a, const float* a_scale, int rows,
                                 const uint8_t* w, const float* w_scale, int experts, int n, int k,
                                 const int32_t* offsets, void* out, void* stream,
                                 const int32_t* a_rows, int a_rows_div, float* partial);
int mi355x_gemm_v2_rowwise_launch(const uint8_t* a, const float* a_scale, int rows,
                                  const uint8_t* w, const float* w_scale, int experts, int n,
                                  int k, const int32_t* offsets, const void* lora_z,
                                  const void* lora_b, int lora_rank, void* out, void* stream,
                                  const int32_t* a_rows, int a_rows_div, float* partial);

int mi355x_wgrad_launch(const uint8_t* p, const float* p_scale, int m_features, const uint8_t* q,
                        const float* q_scale, int n_features, int padded, const int32_t* offsets,
                        int experts, void* out, int out_fp32, void* stream);

namespace {

// The operands every form has; the rest of the struct is zero.
mi355x_gemm_args operands(const uint8_t* a, const float* a_scale, int rows, const uint8_t* w,
                          const float* w_scale, int experts, int n, int k, const int32_t* offsets,
                          void* out) {
  mi355x_gemm_args g = {};
  g.a = a;
  g.a_scale = a_scale;
  g.rows = rows;
  g.w = w;
  g.w_scale = w_scale;
  g.experts = experts;
  g.n = n;
  g.k = k;
  g.offsets = offsets;
  g.out = out;
  g.a_rows_div = 1;
  return g;
}

// Gathered-A forms: GEMM row r (expert-sorted, offsets) reads row
// a_rows[r] of a [a_total, K] and its 1x128 scales a_scale[a_total][K/128]
// (token-major, as mi355x_quantize_token_rows_fp8 writes them): the activation
// quantized once per token, a_rows / a_rows_div the token of each routed row.
// N a multiple of 256, on the 256 x 256 tiles or the smaller ones.
int gathered_checks(const mi355x_gemm_args& g) {
  MI355X_REQUIRE(g.a_rows != nullptr && g.a_total > 0, "gemm gathered: a_rows and a_total required");
  MI355X_REQUIRE(g.a_rows_div >= 1 && (uint64_t)g.a_total * (uint64_t)g.a_rows_div < (1ull << 31),
                 "gemm gathered: a_rows_div must be >= 1 with a_total * a_rows_div < 2^31");
  MI355X_REQUIRE((uint64_t)g.a_total * (uint64_t)g.k < (1ull << 32),
                 "gemm gathered: gathered rows beyond 32-bit offsets");
  MI355X_REQUIRE(g.rows >= 0, "gemm gathered: negative rows");
  return MI355X_OK;
}

// Block-scaled, weight [E, N, K]: plain, gathered or with a rank term.
int block(const mi355x_gemm_args& g, void* stream) {
  const bool gathered = g.a_rows != nullptr, lora = g.lora_rank != 0;
  MI355X_REQUIRE(g.experts > 0 && g.experts <= kMaxExperts, "gemm: experts must be in [1, %d]",
                 kMaxExperts);
  if (gathered) {
    MI355X_REQUIRE(g.n > 0 && g.n % 256 == 0,
                   "gemm gathered: N must be a multiple of 256, got %d", g.n);
  } else if (lora) {
    MI355X_REQUIRE(g.n > 0 && g.n % 256 == 0 && (!g.interleave || (g.n / 2) % 128 == 0),
                   "gemm_lora: N must be a multiple of 256 (2I of 128), got %d", g.n);
  } else {
    MI355X_REQUIRE(g.n > 0 && g.n % BN == 0, "gemm: N must be a multiple of %d, got %d", BN, g.n);
  }
  MI355X_REQUIRE(g.k > 0 && g.k % BK == 0, "gemm: K must be a multiple of %d, got %d", BK, g.k);
  if (gathered) {
    MI355X_REQUIRE(!g.interleave || (g.n / 2) % 128 == 0,
                   "gemm gathered: a gate/up weight needs halves that are multiples of 128");
    const int c = gathered_checks(g);
    if (c != MI355X_OK) return c;
  } else if (lora) {
    MI355X_REQUIRE(g.lora_rank > 0 && g.lora_rank % 16 == 0 && g.lora_rank <= 256,
                   "gemm_lora: the (padded) rank must be a multiple of 16 in [16, 256], got %d",
                   g.lora_rank);
    MI355X_REQUIRE(g.lora_z != nullptr && g.lora_b != nullptr, "gemm_lora: z and b are required");
  } else {
    MI355X_REQUIRE(!g.interleave || (g.n / 2) % 64 == 0,
                   "gemm: a gate/up weight needs halves that are multiples of 64");
  }
  MI355X_REQUIRE(g.rows >= 0, "gemm: negative rows");
  if (g.rows == 0) return MI355X_OK;
  const int v2 = mi355x_gemm_v2_launch(g.a, g.a_scale, g.rows, g.w, g.w_scale, g.w_scale_t,
                                       g.experts, g.n, g.k, g.offsets, g.interleave, g.addend,
                                       g.out, nullptr, nullptr, 0.0f, g.lora_z, g.lora_b,
                                       g.lora_rank, stream, g.a_rows, g.a_rows_div,
                                       (float*)g.workspace);
  if (v2 < 0) return v2;
  MI355X_REQUIRE(v2 == 0, "gemm: shape outside the pipelined kernels");
  return MI355X_OK;
}

// Block-scaled, weight as stored for the forward pass [E, K, N]: plain or gathered.
int kmajor(const mi355x_gemm_args& g, void* stream) {
  MI355X_REQUIRE(g.experts > 0 && g.experts <= kMaxExperts,
                 "gemm_kmajor: experts must be in [1, %d]", kMaxExperts);
  MI355X_REQUIRE(g.n > 0 && g.n % 256 == 0, "gemm_kmajor: N must be a multiple of 256, got %d",
                 g.n);
  MI355X_REQUIRE(g.k > 0 && g.k % BK == 0, "gemm_kmajor: K must be a multiple of %d, got %d", BK,
                 g.k);
  MI355X_REQUIRE(g.rows >= 0, "gemm_kmajor: negative rows");
  MI355X_REQUIRE((uint64_t)(g.k - 1) * (uint64_t)g.n + 256 < (1ull << 32),
                 "gemm_kmajor: a weight slice beyond 32-bit offsets");
  if (g.a_rows != nullptr) {
    const int c = gathered_checks(g);
    if (c != MI355X_OK) return c;
  }
  if (g.rows == 0) return MI355X_OK;
  const int v2 = mi355x_gemm_v2_kmajor_launch(g.a, g.a_scale, g.rows, g.w, g.w_scale, g.experts,
                                              g.n, g.k, g.offsets, g.out, stream, g.a_rows,
                                              g.a_rows_div, (float*)g.workspace);
  if (v2 < 0) return v2;
  MI355X_REQUIRE(v2 == 0, "gemm_kmajor: shape outside the pipelined kernel");
  return MI355X_OK;
}

// Row-scaled, weight [E, N, K]: plain, gathered or with a rank term.
int rowwise(const mi355x_gemm_args& g, void* stream) {
  MI355X_REQUIRE(g.experts > 0 && g.experts <= kMaxExperts,
                 "gemm_rowwise: experts must be in [1, %d]", kMaxExperts);
  MI355X_REQUIRE(g.n > 0 && g.n % 256 == 0, "gemm_rowwise: N must be a multiple of 256, got %d",
                 g.n);
  MI355X_REQUIRE(g.k > 0 && g.k % BK == 0, "gemm_rowwise: K must be a multiple of %d, got %d", BK,
                 g.k);
  if (g.lora_rank != 0) {
    MI355X_REQUIRE(g.lora_rank >= 16 && g.lora_rank <= 256 && g.lora_rank % 16 == 0,
                   "gemm_rowwise_lora: rank must be a multiple of 16 in [16, 256], got %d",
                   g.lora_rank);
    MI355X_REQUIRE(g.lora_z != nullptr && g.lora_b != nullptr,
                   "gemm_rowwise_lora: z and b are required");
  }
  MI355X_REQUIRE(g.rows >= 0, "gemm_rowwise: negative rows");
  if (g.a_rows != nullptr) {
    const int c = gathered_checks(g);
    if (c != MI355X_OK) return c;
  }
  if (g.rows == 0) return MI355X_OK;
  const int v2 = mi355x_gemm_v2_rowwise_launch(g.a, g.a_scale, g.rows, g.w, g.w_scale, g.experts,
                                               g.n, g.k, g.offsets, g.lora_z, g.lora_b,
                                               g.lora_rank, g.out, stream, g.a_rows, g.a_rows_div,
                                               (float*)g.workspace);
  if (v2 < 0) return v2;
  MI355X_REQUIRE(v2 == 0, "gemm_rowwise: shape outside the pipelined kernel");
  return MI355X_OK;
}

}  // namespace

extern "C" size_t mi355x_gemm_args_size(void) { return sizeof(mi355x_gemm_args); }

extern "C" int mi355x_gemm_fp8(const mi355x_gemm_args* args, void* stream) {
  MI355X_REQUIRE(args != nullptr, "gemm: no arguments");
  mi355x_gemm_args g = *args;
  MI355X_REQUIRE((g.a_rows != nullptr) + (g.lora_rank != 0) + (g.addend != nullptr) <= 1,
                 "gemm: a gathered operand, a rank term and an addend exclude one another");
  MI355X_REQUIRE(!g.kmajor || (!g.row_scaled && !g.interleave && g.lora_rank == 0 &&
                               g.addend == nullptr),
                 "gemm: a K-major weight takes block scales and a plain or gathered operand");
  MI355X_REQUIRE(!g.row_scaled || (!g.interleave && g.addend == nullptr),
                 "gemm: row scales take no gate/up order and no addend");
  MI355X_REQUIRE(g.a_rows == nullptr || !g.w_scale_t || g.kmajor,
                 "gemm: a gathered operand takes scales in the weight's order");
  if (g.workspace != nullptr) {
    const size_t size = mi355x_gemm_tail_workspace_size(g.rows, g.experts, g.n, g.k);
    MI355X_REQUIRE(g.workspace_bytes >= size, "gemm: workspace too small");
    MI355X_REQUIRE(size == 0 || ((uintptr_t)g.workspace & 15) == 0,
                   "gemm: the workspace must be 16-byte aligned");
    if (size == 0) g.workspace = nullptr;
  }
  if (g.kmajor) return kmajor(g, stream);
  return g.row_scaled ? rowwise(g, stream) : block(g, stream);
}

extern "C" int mi355x_gemm_fp8_block(const uint8_t* a, const float* a_scale, int rows,
                                     const uint8_t* w, const float* w_scale, int w_scale_t,
                                     int experts, int n, int k, const int32_t* offsets,
                                     int interleave, const void* addend, void* out,
                                     void* stream) {
  mi355x_gemm_args g = operands(a, a_scale, rows, w, w_scale, experts, n, k, offsets, out);
  g.w_scale_t = w_scale_t;
  g.interleave = interleave;
  g.addend = addend;
  return block(g, stream);
}

extern "C" int mi355x_gemm_fp8_block_kmajor(const uint8_t* a, const float* a_scale, int rows,
                                            const uint8_t* w, const float* w_scale, int experts,
                                            int n, int k, const int32_t* offsets, void* out,
                                            void* stream) {
  return kmajor(operands(a, a_scale, rows, w, w_scale, experts, n, k, offsets, out), stream);
}

extern "C" int mi355x_gemm_fp8_block_gathered(const uint8_t* a, const float* a_scale, int a_total,
                                              const int32_t* a_rows, int a_rows_div, int rows,
                                              const uint8_t* w, const float* w_scale, int experts,
                                              int n, int k, const int32_t* offsets, int interleave,
                                              void* out, void* stream) {
  MI355X_REQUIRE(a_rows != nullptr, "gemm gathered: a_rows and a_total required");
  mi355x_gemm_args g = operands(a, a_scale, rows, w, w_scale, experts, n, k, offsets, out);
  g.a_rows = a_rows;
  g.a_total = a_total;
  g.a_rows_div = a_rows_div;
  g.interleave = interleave;
  return block(g, stream);
}

extern "C" int mi355x_gemm_fp8_block_kmajor_gathered(const uint8_t* a, const float* a_scale,
                                                     int a_total, const int32_t* a_rows,
                                                     int a_rows_div, int rows, const uint8_t* w,
                                                     const float* w_scale, int experts, int n,
                                                     int k, const int32_t* offsets, void* out,
                                                     void* stream) {
  MI355X_REQUIRE(a_rows != nullptr, "gemm gathered: a_rows and a_total required");
  mi355x_gemm_args g = operands(a, a_scale, rows, w, w_scale, experts, n, k, offsets, out);
  g.a_rows = a_rows;
  g.a_total = a_total;
  g.a_rows_div = a_rows_div;
  return kmajor(g, stream);
}

extern "C" int mi355x_gemm_fp8_rowwise_gathered(const uint8_t* a, const float* a_scale,
                                                int a_total, const int32_t* a_rows, int a_rows_div,
                                                int rows, const uint8_t* w, const float* w_scale,
                                                int experts, int n, int k, const int32_t* offsets,
                                                void* out, void* stream) {
  MI355X_REQUIRE(a_rows != nullptr, "gemm gathered: a_rows and a_total required");
  mi355x_gemm_args g = operands(a, a_scale, rows, w, w_scale, experts, n, k, offsets, out);
  g.a_rows = a_rows;
  g.a_total = a_total;
  g.a_rows_div = a_rows_div;
  return rowwise(g, stream);
}

extern "C" int mi355x_gemm_fp8_rowwise(const uint8_t* a, const float* a_scale, int rows,
                                       const uint8_t* w, const float* w_scale, int experts, int n,
                                       int k, const int32_t* offsets, void* out, void* stream) {
  return rowwise(operands(a, a_scale, rows, w, w_scale, experts, n, k, offsets, out), stream);
}

extern "C" int mi355x_gemm_fp8_rowwise_lora(const uint8_t* a, const float* a_scale, int rows,
                                            const uint8_t* w, const float* w_scale, int experts,
                                            int n, int k, const int32_t* offsets,
                                            const void* lora_z, const void* lora_b, int lora_rank,
                                            void* out, void* stream) {
  MI355X_REQUIRE(lora_rank != 0,
                 "gemm_rowwise_lora: rank must be a multiple of 16 in [16, 256], got 0");
  mi355x_gemm_args g = operands(a, a_scale, rows, w, w_scale, experts, n, k, offsets, out);
  g.lora_z = lora_z;
  g.lora_b = lora_b;
  g.lora_rank = lora_rank;
  return rowwise(g, stream);
}

extern "C" int mi355x_gemm_fp8_block_lora(const uint8_t* a, const float* a_scale, int rows,
                                          const uint8_t* w, const float* w_scale, int w_scale_t,
                                          int experts, int n, int k, const int32_t* offsets,
                                          int interleave, const void* lora_z, const void* lora_b,
                                          int lora_rank, void* out, void* stream) {
  MI355X_REQUIRE(lora_rank != 0,
                 "gemm_lora: the (padded) rank must be a multiple of 16 in [16, 256], got 0");
  mi355x_gemm_args g = operands(a, a_scale, rows, w, w_scale, experts, n, k, offsets, out);
  g.w_scale_t = w_scale_t;
  g.interleave = interleave;
  g.lora_z = lora_z;
  g.lora_b = lora_b;
  g.lora_rank = lora_rank;
  return block(g, stream);
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
                                       stream, nullptr, 1, nullptr);
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

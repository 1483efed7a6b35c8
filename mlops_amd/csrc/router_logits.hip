// Router logits of a few token rows (decode): logits[t][e] = x[t] . w[e] with
// bf16 operands (an fp32 weight rounded as it is read) and fp32 sums, and in
// the same launch the token rows quantized for the up projection.
//
// A library GEMM here is a cast of the weight, a 5-10 us kernel for 1 MB of
// operands and two launch gaps. Bound by latency and by what one CU can read
// (~57 GB/s): 16 experts x 16 tokens per block and at most a quarter of K, in
// chunks of 512: four K steps of v_mfma_f32_16x16x32_bf16 per wave with all
// their loads in flight. The quarters' sums are added in K order by the
// routing kernel that reads them: one block, so no more than four of them (14
// for width 7168 took it 21 us longer for 64 tokens of 128 experts). All
// tokens and all of K in one block of 16 waves: 5.6 us for one token of width
// 2048, 12.3 for 61, 43 for 64 of width 7168. The quantizer's rows take the
// blocks behind, one wave each. With the routing, from the token rows to the
// plan, against cast, library GEMM, quantizer and routing kernel: one token of
// width 2048 and 128 experts 9.8 us, was 18.4; 61 tokens 19.0, was 24.6; 16 of
// width 4096 and 8 experts 8.7, was 16.8; 64 of width 7168 and 128 experts
// 22.6, was 27.8 (with a bf16 weight, which needs no cast, 1.5-5 us less).
#include "row_quant.h"

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

constexpr int kLogitWaves = 4, kLogitUnroll = 4;
constexpr int kLogitK = 32 * kLogitWaves * kLogitUnroll;  // K per chunk
constexpr int kLogitParts = 4;

// Eight weights as loaded, and as an MFMA operand.
template <typename W>
struct Raw;
template <>
struct Raw<uint16_t> {
  uint4 v;
  __device__ __forceinline__ void load(const uint16_t* p) { v = *(const uint4*)p; }
  __device__ __forceinline__ bf16x8_t operand() const { return __builtin_bit_cast(bf16x8_t, v); }
};
template <>
struct Raw<float> {
  float4 a, b;
  __device__ __forceinline__ void load(const float* p) {
    a = *(const float4*)p;
    b = *(const float4*)(p + 4);
  }
  __device__ __forceinline__ bf16x8_t operand() const {
    return __builtin_bit_cast(bf16x8_t, make_uint4(pack_bf16x2(a.x, a.y), pack_bf16x2(a.z, a.w),
                                                   pack_bf16x2(b.x, b.y), pack_bf16x2(b.z, b.w)));
  }
};

template <typename W>
__global__ void __launch_bounds__(64 * kLogitWaves) router_logits_kernel(
    const uint16_t* __restrict__ x, const W* __restrict__ weight, int tokens, int experts,
    int width, int chunks, int blocks, float* __restrict__ partial, int pitch, int quantize,
    uint8_t* __restrict__ q, float* __restrict__ scales) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = lane_id();
  if ((int)blockIdx.x >= blocks) {
    const int r = (blockIdx.x - blocks) * kLogitWaves + wave;
    if (r >= tokens) return;
    const uint16_t* src = x + (size_t)r * width;
    if (quantize == MI355X_ROUTE_QUANTIZE_BLOCKS) {
      quantize_row_blocks(src, r, tokens, width, 1, q, scales);
    } else {
      const float s = quantize_row_current(src, width, q + (size_t)r * width);
      if (lane == 0) scales[r] = s;
    }
    return;
  }
  __shared__ v4f sums[kLogitWaves][64];
  const int groups = (experts + 15) / 16, tiles = (tokens + 15) / 16;
  const int e0 = (blockIdx.x % groups) * 16, t0 = (blockIdx.x / groups) % tiles * 16;
  const int part = blockIdx.x / (groups * tiles);
  const int l16 = lane & 15, k0 = 8 * (lane >> 4);
  // Rows past the last expert or token repeat it; their results are not stored.
  const W* wrow = weight + (size_t)min(e0 + l16, experts - 1) * width + k0;
  const uint16_t* xrow = x + (size_t)min(t0 + l16, tokens - 1) * width + k0;
  const int end = min((part + 1) * chunks * kLogitK, width) / 32;  // K steps
  v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int base = part * chunks * (kLogitK / 32) + wave; base < end;
       base += kLogitWaves * kLogitUnroll) {
    Raw<W> wf[kLogitUnroll];
    Raw<uint16_t> xf[kLogitUnroll];
#pragma unroll
    for (int u = 0; u < kLogitUnroll; ++u) {
      const int s = min(base + u * kLogitWaves, end - 1);
      wf[u].load(wrow + s * 32);
      xf[u].load(xrow + s * 32);
    }
    __builtin_amdgcn_sched_barrier(0);  // every load before the first wait
#pragma unroll
    for (int u = 0; u < kLogitUnroll; ++u)
      if (base + u * kLogitWaves < end)  // uniform over the wave
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[u].operand(), wf[u].operand(), acc, 0, 0,
                                                      0);
  }
  sums[wave][lane] = acc;
  __syncthreads();
  // Output (token, expert): lane 16 * (token / 4) + expert, element token % 4.
  const int row = tid >> 4, col = tid & 15;
  const float* at = (const float*)&sums[0][(row >> 2) * 16 + col] + (row & 3);
  float total = at[0];
#pragma unroll
  for (int v = 1; v < kLogitWaves; ++v) total += at[v * 256];
  const int token = t0 + row, expert = e0 + col;
  if (token < tokens && expert < experts)
    partial[part * pitch + token * experts + expert] = total;
}

}  // namespace

// Parts of K that a logit is summed in.
int mi355x_router_logits_parts(int width) {
  const int all = (width + kLogitK - 1) / kLogitK, chunks = (all + kLogitParts - 1) / kLogitParts;
  return (all + chunks - 1) / chunks;
}

// partial [parts][pitch], a part's [tokens][experts] in order; the checks are
// the caller's.
int mi355x_router_logits_launch(const void* x, const void* weight, int weight_fp32, int tokens,
                                int experts, int width, float* partial, int pitch, int quantize,
                                uint8_t* q, float* scales, void* stream) {
  const int all = (width + kLogitK - 1) / kLogitK, chunks = (all + kLogitParts - 1) / kLogitParts;
  const int blocks = (experts + 15) / 16 * ((tokens + 15) / 16) * mi355x_router_logits_parts(width);
  const int grid = blocks + (quantize != 0 ? (tokens + kLogitWaves - 1) / kLogitWaves : 0);
  auto launch = [&](auto* w) {
    hipLaunchKernelGGL(router_logits_kernel, dim3(grid), dim3(64 * kLogitWaves), 0,
                       (hipStream_t)stream, (const uint16_t*)x, w, tokens, experts, width, chunks,
                       blocks, partial, pitch, quantize, q, scales);
  };
  if (weight_fp32) launch((const float*)weight);
  else launch((const uint16_t*)weight);
  MI355X_LAUNCH_CHECK();
  return MI355X_OK;
}

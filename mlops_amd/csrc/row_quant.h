// One wave quantizing one row: the body of the row quantizers and of the
// launches that quantize token rows beside other work.
#pragma once

#include "common.h"

template <typename T>
__device__ __forceinline__ void load8(const T* p, float* v);
template <>
__device__ __forceinline__ void load8<uint16_t>(const uint16_t* p, float* v) {
  load_bf16x8(p, v);
}
template <>
__device__ __forceinline__ void load8<float>(const float* p, float* v) {
  const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
  v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

// Row r (bf16, at src) to e4m3 with one scale per 128 columns:
// scales[width/128][rows], or [rows][width/128] with row_scales. Up to four
// 512-column chunks' loads are issued before any of their stores: loads and
// stores share one completion counter, so a load issued after a store would
// wait for it.
__device__ __forceinline__ void quantize_row_blocks(const uint16_t* __restrict__ src, int r,
                                                    int rows, int width, int row_scales,
                                                    uint8_t* __restrict__ q,
                                                    float* __restrict__ scales) {
  constexpr int kChunks = 4;
  const int lane = lane_id();
  for (int base0 = 0; base0 < width; base0 += 512 * kChunks) {
    uint4 raw[kChunks];
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      const int col = base0 + c * 512 + lane * 8;
      raw[c] = col < width ? *(const uint4*)(src + col) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      if (base0 + c * 512 >= width) break;  // uniform over the wave
      const int col = base0 + c * 512 + lane * 8;
      float v[8];
      unpack_bf16x8(raw[c], v);
      float amax = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(v[i]));
      amax = group_amax<16>(amax);
      const float s = fmaxf(amax * kInv448, kMinScale);
      const uint2 packed = quant8(v, s);
      if (col < width) {
        store_stream8(q + (size_t)r * width + col, packed);
        if ((lane & 15) == 0) {
          const size_t si = row_scales ? (size_t)r * (width >> 7) + (col >> 7)
                                       : (size_t)(col >> 7) * rows + r;
          scales[si] = s;
        }
      }
    }
  }
}

// The row at src to e4m3 at dst with one scale, which is returned. Read
// twice, once for the maximum; the second read hits the caches. Four chunks'
// loads before their stores, as above.
template <typename T>
__device__ __forceinline__ float quantize_row_current(const T* __restrict__ src, int width,
                                                      uint8_t* __restrict__ dst) {
  const int lane = lane_id();
  float amax = 0.0f;
  for (int col = lane * 8; col < width; col += 512) {
    float v[8];
    load8(src + col, v);
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(v[i]));
  }
  amax = group_amax<64>(amax);
  const float s = fmaxf(amax * kInv448, kMinScale);
  for (int col0 = lane * 8; col0 < width; col0 += 4 * 512) {
    float v[4][8];
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (col0 + c * 512 < width) load8(src + col0 + c * 512, v[c]);
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (col0 + c * 512 < width) *(uint2*)(dst + col0 + c * 512) = quant8(v[c], s);
  }
  return s;
}

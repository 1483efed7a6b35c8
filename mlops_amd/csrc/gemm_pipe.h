// Pipelined block-FP8 MFMA main loop for gfx950, shared by the grouped GEMMs.
//
// Workgroup tile 256 (M) x 256 (N) x 128 (K), 8 waves (two per SIMD) in a
// 4 x 2 grid, wave tile 64 x 128 (4 x 8 blocks of
// v_mfma_f32_16x16x128_f8f6f4). Operands are copied global -> LDS by the
// CDNA4 direct loads (global_load_lds_dwordx4: no staging registers, no LDS
// store instructions) into two stages, one s_barrier per K step.
//
// Why 256 x 256: the L2 -> LDS direct-load path sustains ~54 B/clk/CU on
// MI355X (measured); a K step of this tile moves 64 KB for 16.8 MFLOP
// (256 flop/B), so the copy takes ~60% of the MFMA time and hides under it,
// where a 128 x 256 tile (171 flop/B) would make the GEMM copy-bound.
//
// LDS rows are 128 bytes, unpadded; the 16-byte unit c of row r is stored at
// unit c ^ (r & 7). A fragment lane (row l % 16, group g = l / 16) takes the
// units g and g + 4 of its row: A and B lanes agree on that K assignment, so
// the MFMA sum is unchanged, and a wave's 16 rows x 4 units per read then
// hit every bank once (measured on MI355X: full LDS read bandwidth, against
// ~63% for adjacent unit pairs under any row swizzle).
// A direct load writes 64 lanes x 16 B = 8 rows; lane L writes unit L % 8 of
// row L / 8 and so loads the logical unit (L % 8) ^ swizzle(row).
#pragma once

#include "common.h"

namespace pipe {

constexpr int BM = 256, BN = 256, BK = 128;
constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr int kStages = 2;
constexpr int A_BYTES = BM * BK;          // 32 KB
constexpr int B_BYTES = BN * BK;          // 32 KB
constexpr int SA_BYTES = BM * 4;          // row scales of A
constexpr int SB_BYTES = BN * 4;          // column scales of B (weight-gradient form)
constexpr int STAGE_BYTES = A_BYTES + B_BYTES + SA_BYTES + SB_BYTES;
constexpr int A_LOADS = A_BYTES / 1024 / kWaves;  // direct loads per wave per stage: 4
constexpr int B_LOADS = B_BYTES / 1024 / kWaves;  // 4

typedef __attribute__((address_space(3))) void* lds_ptr_t;

__device__ __forceinline__ int swz(int row) { return row & 7; }

// The direct loads are issued as inline assembly, invisible to the
// compiler's wait-count bookkeeping: it would otherwise wait for every
// in-flight load before any LDS read it cannot prove disjoint. The kernels
// count their own loads and wait with wait_and_sync<N>.
// LDS byte address of a (wave-uniform) LDS pointer, as a scalar for M0: the
// low half of the generic address (a cast to an LDS pointer would also test
// it for null, where the compiler cannot prove that it is none).
__device__ __forceinline__ uint32_t lds_addr(const uint8_t* p) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(size_t)p);
}
// Source address = wave-uniform 64-bit base (SGPRs) + per-lane 32-bit byte
// offset (one VGPR), the saddr form of the global load.
__device__ __forceinline__ void dma16(const void* base, uint32_t off, const uint8_t* lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :: "s"(lds_addr(lds)), "v"(off), "s"(base) : "memory", "m0");
}
// The same from a per-lane 64-bit address, for rows too far apart for an offset.
__device__ __forceinline__ void dma16_far(const uint8_t* src, const uint8_t* lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :: "s"(lds_addr(lds)), "v"(src) : "memory", "m0");
}
__device__ __forceinline__ void dma4(const void* base, uint32_t off, const uint8_t* lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
               :: "s"(lds_addr(lds)), "v"(off), "s"(base) : "memory", "m0");
}

// Wait until at most N direct loads of this wave are in flight, then barrier.
template <int N>
__device__ __forceinline__ void wait_and_sync() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  // gfx9 s_waitcnt: vmcnt[3:0], expcnt[6:4]=7, lgkmcnt[11:8]=15, vmcnt[5:4] in [15:14]
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Barrier that waits for this wave's LDS operations only (not for its
// in-flight global loads and stores).
__device__ __forceinline__ void lds_sync() {
  // vmcnt = 63 (no wait), expcnt = 7, lgkmcnt = 0
  __builtin_amdgcn_s_waitcnt(0xC07F);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

__device__ __forceinline__ void sync_all() {
  __builtin_amdgcn_s_waitcnt(0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// 32 fp8 K-values of one fragment row from a swizzled stage tile.
__device__ __forceinline__ v8i frag(const uint8_t* tile, int row, int lane) {
  const int g = lane >> 4;  // units g and g + 4
  const int s = swz(row);
  const uint8_t* base = tile + row * 128;
  uint4 x = *(const uint4*)(base + 16 * (g ^ s));
  uint4 y = *(const uint4*)(base + 16 * ((g + 4) ^ s));
  v8i r;
  r[0] = x.x; r[1] = x.y; r[2] = x.z; r[3] = x.w;
  r[4] = y.x; r[5] = y.y; r[6] = y.z; r[7] = y.w;
  return r;
}

// Position of 16-byte unit u in row r of a K-major stage tile: u ^ kmsw(r).
// A fragment read takes rows r .. r+7 (r % 8 == 0) in each 16-lane group and
// rows 16 apart across the four groups of a wave: the low bits spread a
// group's rows over 8 positions, and bit 3 (row / 16 odd) moves the odd
// groups to the other 8, so a 64-lane read meets each bank twice.
__device__ __forceinline__ int kmsw(int r) { return (r & 15) ^ (((r >> 4) & 1) << 3); }

// The same fragment (32 fp8 K-values of one B column) from a K-major stage
// tile: 128 K rows of 256 bytes (one byte per column), 16-byte unit u of row
// r stored at u ^ kmsw(r). ds_read_b64_tr_b8 gives lane j of each 16-lane
// group byte (j % 8) of the 8 bytes addressed by lane 2b + j / 8, as its
// byte b; so with lane i addressing K row kbase + i / 2 at column
// col0 + 8 (i % 2), lane j receives column col0 + j at K rows kbase .. +7.
// Four such reads give the K rows of frag(): 16g .. 16g+15 and
// 64+16g .. 64+16g+15 (g = lane / 16).
typedef int v2i_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ v8i frag_kmajor(const uint8_t* tile, int col0, int lane) {
  const int g = lane >> 4, j = lane & 15;
  const int unit = col0 >> 4;
  v8i r;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int row = (p >> 1) * 64 + 16 * g + (p & 1) * 8 + (j >> 1);
    const uint8_t* at = tile + row * 256 + 16 * (unit ^ kmsw(row)) + 8 * (j & 1);
    const v2i_t v = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i_t*)(lds_ptr_t)at);
    r[2 * p] = v[0];
    r[2 * p + 1] = v[1];
  }
  return r;
}

__device__ __forceinline__ v4f mfma(v8i a, v8i b) {
  const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, zero, 0, 0, 0, 0, 0, 0);
}

// The same MFMA accumulating into c (row-scaled operands: no per-block fold).
__device__ __forceinline__ v4f mfma_acc(v8i a, v8i b, v4f c) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
}

// Exclusive prefix of ceil(rows_e / tile) over experts -> prefix[0..E].
__device__ inline void tile_prefix(const int32_t* __restrict__ offsets, int experts, int tile,
                                   int* prefix, int* tmp) {
  const int t = threadIdx.x;
  const int per = (experts + kThreads - 1) / kThreads;
  int local = 0;
  for (int i = 0; i < per; ++i) {
    int e = t * per + i;
    if (e < experts) local += (offsets[e + 1] - offsets[e] + tile - 1) / tile;
  }
  tmp[t] = local;
  __syncthreads();
  for (int o = 1; o < kThreads; o <<= 1) {
    int v = t >= o ? tmp[t - o] : 0;
    __syncthreads();
    tmp[t] += v;
    __syncthreads();
  }
  int run = tmp[t] - local;
  for (int i = 0; i < per; ++i) {
    int e = t * per + i;
    if (e < experts) {
      prefix[e] = run;
      run += (offsets[e + 1] - offsets[e] + tile - 1) / tile;
    }
  }
  if (t == kThreads - 1) prefix[experts] = tmp[t];
  __syncthreads();
}

__device__ __forceinline__ int find_expert(const int* prefix, int experts, int tile) {
  int lo = 0, hi = experts - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (prefix[mid] <= tile) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Round-robin tile assignment, for grids that are no multiple of 8 workgroups.
// The others give XCD x (= workgroup % 8) the x-th eighth of the tile list, so
// that its CUs share panels in their L2 (tile_at in each kernel).
__device__ __forceinline__ int tile_of(int round, int block, int grid) {
  return round * grid + block;
}

// First K step of the 256 x 256 tile `tile` of a rotated launch, of nk. Tiles
// that share an operand panel run at the same time on neighbouring CUs of one
// XCD; consecutive tiles start one K step apart, over a window of three steps,
// so that one of them takes a panel step's L2 miss and the others find the
// line in L2 a step later. The window is kept small: a rotation over all K
// steps (7t mod nk) took the same time but spread an expert's ~30 concurrent
// tiles over its whole 5 MB of panels, more than a 4 MB L2, and the up
// projection read its operands 3.6 times from HBM instead of 1.05 times (2%
// faster over C3's four launches). Short K (under 8 steps, e.g. the down
// projection) keeps the full rotation, which measured ~3% faster there, with
// panels small enough to stay in L2. Smaller tiles start where the 256 x 256
// tile they lie in does, so that a result's sum has one order whichever tiles
// compute it.
__device__ __forceinline__ int k_rotation(int tile, int nk) {
  return nk >= 8 ? tile % 3 : (tile * 7) % nk;
}

// Tile order of a grouped GEMM by the size of one expert's weight (N x K
// bytes). Up to a few L2s' worth, tiles go row-block-major with the K
// rotation: an XCD's CUs sweep one row block's N tiles, and the whole weight
// stays cached across row blocks. Beyond that, each row block would stream the
// weight again from HBM, so tiles go in groups of n_group N tiles x all the
// expert's row blocks, unrotated, and the CUs that share a weight panel read
// it together. Measured on MI355X: Mixtral's four GEMMs (58-117 MB per
// expert) +6-14%, DeepSeek-shard up/dgrad-up (29 MB) +5-7%; the 3-15 MB
// weights of the other shapes lose 1-7% in that order.
struct Order {
  int n_group, rotate;
};
inline Order tile_order(int n, int k) {
  if ((size_t)n * (size_t)k >= ((size_t)24 << 20)) return {8, 0};
  return {0, 1};
}

// x / d for the divisor d encoded by row_div_magic (s == 0: d = 1): the
// round-down multiply-high method for unsigned division by an invariant
// integer (Granlund and Montgomery, PLDI 1994), with a 33-bit multiplier
// 2^32 + m, exact for every 32-bit x.
__device__ __forceinline__ uint32_t div_rows(uint32_t x, uint32_t m, int s) {
  const uint32_t t = __umulhi(x, m);
  const uint32_t q = (t + ((x - t) >> 1)) >> (s > 0 ? s - 1 : 0);
  return s == 0 ? x : q;  // a select: no branch around the LDS reads it feeds
}

// (m, s) for div_rows: s = ceil(log2 d), m = floor(2^32 (2^s - d) / d) + 1
// for d >= 2; (0, 0) for d = 1.
struct RowDiv {
  uint32_t m;
  int s;
};
inline RowDiv row_div_magic(int d) {
  if (d <= 1) return {0u, 0};
  int s = 0;
  while ((1 << s) < d) ++s;
  const uint64_t m = (((uint64_t)1 << 32) * (uint64_t)((1 << s) - d)) / (uint64_t)d + 1;
  return {(uint32_t)m, s};
}

// Compute units of the current device (cached; host side).
inline int cu_count() {
  static int cus[64] = {0};
  int dev = 0;
  hipGetDevice(&dev);
  if (dev < 0 || dev >= 64) dev = 0;
  if (cus[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    cus[dev] = n;
  }
  return cus[dev];
}

}  // namespace pipe

// Grouped weight-gradient GEMM:
//   out[e][m][n] = sum over expert e's padded rows k of P[m][k] * Q[n][k]
// with P, Q the feature-major e4m3 operands written by the transposing
// quantizer and one power-of-two descale per (feature, 128-row block).
//
// wgrad_v2_kernel has the main loop of the grouped GEMM (gemm_pipe.h: 256 x 256
// tile, 8 waves, direct-to-LDS loads, two stages) with one difference: both operands carry
// per-row scales that are powers of two, so the MFMA applies them itself
// (v_mfma_scale_f32_16x16x128_f8f6f4 with E8M0 scales = the fp32 exponent
// byte) and accumulates across K blocks in place: no VALU work in the loop.
// Hardware operand layout (measured on MI355X): lane l of a 16x16x128
// fragment holds K bytes [16g, 16g+16) and [64+16g, 64+16g+16), g = l / 16,
// and the scale of (row m, 32-wide K block b) is taken from lane 16b + m; a
// scale constant over the 128 K values means each lane passes its own row's.
#include "gemm_pipe.h"

using namespace pipe;

namespace {

constexpr int kMaxExperts = 512;

// q feature behind B-tile row tr, of MFMA column c of block jb: output column
// c * 8 + jb of the wave's 128, so that a lane's eight accumulator blocks are
// eight consecutive bf16 columns (one 16-byte store); with fp32 outputs
// columns 4c .. 4c + 3 of either half, so that each of the two 16-byte
// stores of a row fills whole lines (32 bytes per lane, stored as two halves
// of a line, took 930 us for 1.6 GB of gradients where this takes 269).
template <bool kFp32>
__device__ __forceinline__ int feature_col(int tr, int nt) {
  const int part = tr >> 7, local = tr & 127, c = local & 15, jb = local >> 4;
  return nt * BN + part * 128 + (kFp32 ? (jb >> 2) * 64 + c * 4 + (jb & 3) : c * 8 + jb);
}

__device__ __forceinline__ int e8m0(float pow2_scale) { return __float_as_int(pow2_scale) >> 23; }

// Whether E8M0 holds every scale added: positive normal powers of two.
struct ScalesSeen {
  uint32_t any = 0, least = 0x7f000000u, most = 0;  // bits OR-ed, their minimum, maximum
  __device__ __forceinline__ void add(float s) {
    const uint32_t bits = __float_as_uint(s);
    any |= bits;
    least = min(least, bits);
    most = max(most, bits);
  }
  template <typename... Rest>
  __device__ __forceinline__ void add(float s, Rest... rest) {
    add(s);
    add(rest...);
  }
  __device__ __forceinline__ bool e8m0() const {
    return (any & 0x807fffffu) == 0 && least >= 0x00800000u && most < 0x7f800000u;
  }
};

__device__ __forceinline__ v4f mfma_e8(v8i a, v8i b, v4f c, int sa, int sb) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, sa, 0, sb);
}

struct WTile {
  int e, mt, nt, k0, nk;  // expert, tile coordinates, first padded block, blocks
  int rot;                // K-step rotation (see wdescribe)
};

__device__ __forceinline__ WTile wdescribe(const int* prefix, int per_e, int n_tiles, int tile) {
  WTile t;
  t.e = __builtin_amdgcn_readfirstlane(tile / per_e);
  const int rem = tile - t.e * per_e;
  t.mt = __builtin_amdgcn_readfirstlane(rem / n_tiles);
  t.nt = __builtin_amdgcn_readfirstlane(rem - t.mt * n_tiles);
  t.k0 = __builtin_amdgcn_readfirstlane(prefix[t.e]);
  t.nk = __builtin_amdgcn_readfirstlane(prefix[t.e + 1] - prefix[t.e]);
  // Tiles sharing an operand panel run together on neighbouring CUs; each
  // starts at a different K step so that one takes a step's L2 miss and the
  // others hit later instead of all waiting on the same miss.
  t.rot = t.nk > 0 ? __builtin_amdgcn_readfirstlane((tile * 7) % t.nk) : 0;
  return t;
}

template <bool kFp32>
__global__ void __launch_bounds__(kThreads, 2) wgrad_v2_kernel(
    const uint8_t* __restrict__ p, const float* __restrict__ p_scale, int Mf,
    const uint8_t* __restrict__ q, const float* __restrict__ q_scale, int Nf, int padded,
    const int32_t* __restrict__ offsets, int experts, void* __restrict__ out) {
  __shared__ __align__(1024) uint8_t smem[kStages * STAGE_BYTES];
  __shared__ int prefix[kMaxExperts + 1];
  __shared__ int tmp[kThreads];
  tile_prefix(offsets, experts, 128, prefix, tmp);  // padded 128-row blocks per expert
  const int n_tiles = Nf / BN;
  const int per_e = (Mf / BM) * n_tiles;
  const int total = experts * per_e;
  const int tid = threadIdx.x, lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;  // 4 x 2 wave grid

  auto issue = [&](const WTile& t, int step, int stage) {
    const int kb = __builtin_amdgcn_readfirstlane(step + t.rot < t.nk ? step + t.rot : step + t.rot - t.nk);
    uint8_t* base = smem + stage * STAGE_BYTES;
    const size_t kblock = (size_t)(t.k0 + kb);
    const uint8_t* abase = p + kblock * 128;
    const uint8_t* bbase = q + kblock * 128;
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) {
      const int r = (wave * A_LOADS + i) * 8 + (lane >> 3);
      const uint32_t off = (uint32_t)(t.mt * BM + r) * (uint32_t)padded + 16 * ((lane & 7) ^ swz(r));
      dma16(abase, off, base + (wave * A_LOADS + i) * 1024);
    }
#pragma unroll
    for (int i = 0; i < B_LOADS; ++i) {
      const int tr = (wave * B_LOADS + i) * 8 + (lane >> 3);
      const uint32_t off = (uint32_t)feature_col<kFp32>(tr, t.nt) * (uint32_t)padded + 16 * ((lane & 7) ^ swz(tr));
      dma16(bbase, off, base + A_BYTES + (wave * B_LOADS + i) * 1024);
    }
    // Scales of this K block, stored in lane order: LDS slot wm*64 + c*4 + i
    // holds P row wm*64 + i*16 + c, slot wn*128 + c*8 + jb holds the Q row
    // of B-tile row wn*128 + jb*16 + c, so that a fragment lane (c = lane %
    // 16) fetches its 4 row scales and 8 column scales with 16-byte reads.
    // Waves 0-3 load the P scales, waves 4-7 the Q scales.
    uint8_t* sbase = base + A_BYTES + B_BYTES;
    if (wave < 4) {
      const int slot = wave * 64 + lane;
      const int row = (slot & ~63) + (slot & 3) * 16 + ((slot >> 2) & 15);
      dma4(p_scale + kblock * Mf + t.mt * BM, 4u * (uint32_t)row, sbase + wave * 256);
    } else {
      const int slot = (wave - 4) * 64 + lane;
      const int tr = (slot & ~127) + (slot & 7) * 16 + ((slot >> 3) & 15);
      dma4(q_scale + kblock * Nf, 4u * (uint32_t)feature_col<kFp32>(tr, t.nt),
           sbase + SA_BYTES + (wave - 4) * 256);
    }
  };

  // XCD-affine order: workgroup b runs on XCD b % 8, and XCD x takes a
  // contiguous range of the expert-major tile list holding 1/8 of the total
  // work (a tile costs its expert's K blocks), so an expert's operand panels
  // are fetched into one or two XCD L2s instead of all eight. The 8 x G/8
  // workgroups of an XCD take its range round-robin. Needs a grid that is a
  // multiple of 8; otherwise plain order.
  const bool affine = (gridDim.x & 7) == 0;
  const int xcd = blockIdx.x & 7, cu = blockIdx.x >> 3, per_xcd = gridDim.x >> 3;
  auto range_start = [&](int x) -> int {  // first tile of XCD x's range
    if (x <= 0) return 0;
    if (x >= 8) return total;
    const long long bound = (long long)per_e * prefix[experts] * x / 8;
    int lo = 0, hi = experts - 1;  // last e with cost before it <= bound
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if ((long long)per_e * prefix[mid] <= bound) lo = mid; else hi = mid - 1;
    }
    const int nk = prefix[lo + 1] - prefix[lo];
    const long long rem = bound - (long long)per_e * prefix[lo];
    const long long j = nk > 0 ? (rem + nk - 1) / nk : per_e;
    return lo * per_e + (int)(j < per_e ? j : per_e);
  };
  const int first = __builtin_amdgcn_readfirstlane(affine ? range_start(xcd) : 0);
  const int last = __builtin_amdgcn_readfirstlane(affine ? range_start(xcd + 1) : total);
  auto tile_at = [&](int r) -> int {
    if (!affine) return tile_of(r, blockIdx.x, gridDim.x);
    const int t = first + r * per_xcd + cu;
    return t < last ? t : total;
  };
  int round = 0;
  int tile = tile_at(0);
  if (tile >= total) return;
  WTile ct = wdescribe(prefix, per_e, n_tiles, tile);
  bool issued = false;  // whether the current tile's first step is in flight
  int stage = 0;
  for (;;) {
    if (!issued && ct.nk > 0) issue(ct, 0, stage);
    issued = false;
    const int next_tile = tile_at(round + 1);
    v4f acc[4][8];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[i][j] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};

    for (int kb = 0; kb < ct.nk; ++kb) {
      wait_and_sync<0>();
      if (kb + 1 < ct.nk) {
        issue(ct, kb + 1, stage ^ 1);
      } else if (next_tile < total) {
        const WTile nt = wdescribe(prefix, per_e, n_tiles, next_tile);
        if (nt.nk > 0) {
          issue(nt, 0, stage ^ 1);
          issued = true;
        }
      }
      const uint8_t* base = smem + stage * STAGE_BYTES;
      const uint8_t* ta = base;
      const uint8_t* tb = base + A_BYTES;
      const float* sa = (const float*)(base + A_BYTES + B_BYTES);
      const float* sb = sa + BM;
      const int c = lane & 15;
      const float4 sa4 = *(const float4*)&sa[wm * 64 + c * 4];
      const float4 sb_lo = *(const float4*)&sb[wn * 128 + c * 8];
      const float4 sb_hi = *(const float4*)&sb[wn * 128 + c * 8 + 4];
      // Reads in the order the first MFMAs consume them (the step starts
      // with every wave of the CU reading at once, so what comes first
      // decides when the matrix cores start), B fragments through a
      // three-slot ring, read two blocks ahead.
      v8i af[4], bf[3];
      bf[0] = frag(tb, wn * 128 + c, lane);
#pragma unroll
      for (int i = 0; i < 4; ++i) af[i] = frag(ta, wm * 64 + i * 16 + c, lane);
      bf[1] = frag(tb, wn * 128 + 16 + c, lane);
      __builtin_amdgcn_sched_barrier(0);
      // Exponent bytes after the fragment reads are in flight: waiting for
      // the scales then does not hold back the fragment reads.
      const int ea[4] = {e8m0(sa4.x), e8m0(sa4.y), e8m0(sa4.z), e8m0(sa4.w)};
      const int eb[8] = {e8m0(sb_lo.x), e8m0(sb_lo.y), e8m0(sb_lo.z), e8m0(sb_lo.w),
                         e8m0(sb_hi.x), e8m0(sb_hi.y), e8m0(sb_hi.z), e8m0(sb_hi.w)};
#pragma unroll
      for (int jb = 0; jb < 8; ++jb) {
        if (jb + 2 < 8) bf[(jb + 2) % 3] = frag(tb, wn * 128 + (jb + 2) * 16 + c, lane);
        // Keep the read ahead of this block's MFMAs (the scheduler would
        // otherwise sink it to shorten live ranges, leaving one group of
        // MFMAs to cover the LDS latency).
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i][jb] = mfma_e8(af[i], bf[jb % 3], acc[i][jb], ea[i], eb[jb]);
        __builtin_amdgcn_sched_barrier(0);
      }
      stage ^= 1;
    }

    // Epilogue from registers: lane (row, its 8 columns; see feature_col).
    const size_t row0 = (size_t)ct.e * Mf + ct.mt * BM + wm * 64;
    const size_t col0 = (size_t)ct.nt * BN + wn * 128 + (lane & 15) * (kFp32 ? 4 : 8);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int lrow = i * 16 + 4 * (lane >> 4) + r;
        const size_t off = (row0 + lrow) * Nf + col0;
        if constexpr (kFp32) {
          float* o = (float*)out + off;
          store_stream(o, make_uint4(__float_as_uint(acc[i][0][r]), __float_as_uint(acc[i][1][r]), __float_as_uint(acc[i][2][r]), __float_as_uint(acc[i][3][r])));
          store_stream(o + 64, make_uint4(__float_as_uint(acc[i][4][r]), __float_as_uint(acc[i][5][r]), __float_as_uint(acc[i][6][r]), __float_as_uint(acc[i][7][r])));
        } else {
          uint4 o;
          o.x = pack_bf16x2(acc[i][0][r], acc[i][1][r]);
          o.y = pack_bf16x2(acc[i][2][r], acc[i][3][r]);
          o.z = pack_bf16x2(acc[i][4][r], acc[i][5][r]);
          o.w = pack_bf16x2(acc[i][6][r], acc[i][7][r]);
          store_stream((uint16_t*)out + off, o);
        }
      }
    }
    if (next_tile >= total) break;
    ++round;
    ct = wdescribe(prefix, per_e, n_tiles, next_tile);
  }
}

// ---------------------------------------------------------------------------
// 128 x 128 tiles, two workgroups per CU: feature counts that are odd
// multiples of 128, and groups of few rows, where a tile is one or two K
// steps and its output decides (a 256 x 256 tile's epilogue then runs alone
// on its CU; two workgroups overlap one's stores with the other's copies).
// 8 waves in a 4 x 2 grid, wave tile 32 x 64 (2 x 4 blocks), two stages.
//
// kAnyScale: shapes that the 256 x 256 tiles do not take apply any fp32 scale.
// The transposing quantizer writes powers of two, so the loop lets the MFMA
// apply them as above and only gathers what it saw of them (nine VALU
// instructions a step); a wave that met others forms its part of the tile
// again, straight from memory, folding each step's raw product into the sums
// with FMAs. 1280 x 1152 and 1152 x 640, 16 experts, 12004 rows, fp32 out, us:
// 37-39 and 21 without the look, 38 and 21 with it (bf16 30 and 17, 31 and 17),
// 127 and 69 where every scale is another. (A branch in the K loop took 42 and
// 23 with powers of two: its waits come before the fragment reads, or it spills.)
namespace small {
constexpr int TM = 128, TN = 128;
constexpr int MB = 2, NB = 4;
constexpr int A_SIZE = TM * BK, B_SIZE = TN * BK;
constexpr int STAGE = A_SIZE + B_SIZE + 4 * (TM + TN);
constexpr int kStores = MB * 4;  // store instructions of a wave's epilogue
// kFar: from here on 28 padded rows exceed a 32-bit offset. Not a branch in the
// kernel, which costs the ordinary launch 6%.
constexpr int kFarRows = 1 << 27;

// frag() of one operand row's K block in memory: its units g and g + 4.
__device__ __forceinline__ v8i frag_global(const uint8_t* block, int g) {
  const uint4 x = *(const uint4*)(block + 16 * g), y = *(const uint4*)(block + 64 + 16 * g);
  return (v8i){(int)x.x, (int)x.y, (int)x.z, (int)x.w, (int)y.x, (int)y.y, (int)y.z, (int)y.w};
}
}  // namespace small

template <bool kFp32, bool kAnyScale, bool kFar>
__global__ void __launch_bounds__(kThreads, 4) wgrad_tile_kernel(
    const uint8_t* __restrict__ p, const float* __restrict__ p_scale, int Mf,
    const uint8_t* __restrict__ q, const float* __restrict__ q_scale, int Nf, int padded,
    const int32_t* __restrict__ offsets, int experts, void* __restrict__ out) {
  using namespace small;
  __shared__ __align__(1024) uint8_t smem[2 * STAGE];
  __shared__ int prefix[kMaxExperts + 1];
  padded_block_prefix<kThreads>(offsets, experts, prefix, (int*)smem);
  const int n_tiles = Nf / TN;
  const int per_e = (Mf / TM) * n_tiles;
  const int total = experts * per_e;
  const int tid = threadIdx.x, lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int lrow = lane >> 3, unit = (lane & 7) ^ (lane >> 3), c = lane & 15;

  // Where both feature counts take 256 x 256 tiles, a tile starts at the K step
  // at which the one it lies in would (wdescribe): one order of the sum
  // whichever tiles compute it.
  const int wide_n = Nf % BN == 0 && Mf % BM == 0 ? Nf / BN : 0;
  struct Tile {
    int e, mt, nt, k0, nk, rot;
  };
  auto describe = [&](int tile) -> Tile {
    Tile t;
    t.e = tile / per_e;
    const int rem = tile - t.e * per_e;
    t.mt = rem / n_tiles;
    t.nt = rem - t.mt * n_tiles;
    t.k0 = __builtin_amdgcn_readfirstlane(prefix[t.e]);
    t.nk = __builtin_amdgcn_readfirstlane(prefix[t.e + 1]) - t.k0;
    t.rot = 0;
    if (wide_n > 0 && t.nk > 0) {
      const int wide = (t.e * (Mf / BM) + t.mt / (BM / TM)) * wide_n + t.nt / (BN / TN);
      t.rot = __builtin_amdgcn_readfirstlane((wide * 7) % t.nk);
    }
    return t;
  };
  // The step-th K block of tile t into a stage. The Q row behind tile row (jb, c) of a
  // wave column is feature 4c + jb of its 64, so a lane's four blocks are
  // four consecutive output columns. Scales in lane order: P's slot
  // wm * 32 + 2c + i holds row wm * 32 + 16i + c; Q's order is natural.
  auto copy = [&](const uint8_t* base, int row, uint8_t* to) {
    if constexpr (kFar) dma16_far(base + (size_t)row * padded + 16 * unit, to);
    else dma16(base, (uint32_t)row * (uint32_t)padded + 16 * unit, to);
  };
  auto issue = [&](const Tile& t, int step, int stage) {
    uint8_t* base = smem + stage * STAGE;
    const int kb = step + t.rot < t.nk ? step + t.rot : step + t.rot - t.nk;
    const size_t block = (size_t)(t.k0 + kb);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int tr = (wave * 2 + i) * 8;
      copy(p + (size_t)(t.mt * TM + tr) * padded + block * 128, lrow, base + tr * 128);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int tr = (wave * 2 + i) * 8;
      const int feature = t.nt * TN + (tr >> 6) * 64 + (tr & 8) * 4 + ((tr >> 4) & 3);
      copy(q + (size_t)feature * padded + block * 128, 4 * lrow, base + A_SIZE + tr * 128);
    }
    uint8_t* scales = base + A_SIZE + B_SIZE;
    if (wave < 2) {
      const int slot = wave * 64 + lane;
      const int row = (slot & ~31) + (slot & 1) * 16 + ((slot >> 1) & 15);
      dma4(p_scale + block * Mf + t.mt * TM, 4u * (uint32_t)row, scales + wave * 256);
    } else if (wave < 4) {
      dma4(q_scale + block * Nf + t.nt * TN + (wave - 2) * 64, 4u * (uint32_t)lane,
           scales + TM * 4 + (wave - 2) * 256);
    }
  };

  // XCD-affine ranges balanced by cost, as in wgrad_v2_kernel, with two steps
  // added to every tile for its output.
  constexpr int kTileCost = 2;
  const bool affine = (gridDim.x & 7) == 0;
  const int xcd = blockIdx.x & 7, cu = blockIdx.x >> 3, per_xcd = gridDim.x >> 3;
  auto range_start = [&](int x) -> int {
    if (x <= 0) return 0;
    if (x >= 8) return total;
    auto before = [&](int e) -> long long {
      return (long long)per_e * (prefix[e] + kTileCost * e);
    };
    const long long bound = before(experts) * x / 8;
    int lo = 0, hi = experts - 1;  // last e with cost before it <= bound
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (before(mid) <= bound) lo = mid; else hi = mid - 1;
    }
    const int cost = prefix[lo + 1] - prefix[lo] + kTileCost;
    const long long j = (bound - before(lo) + cost - 1) / cost;
    return lo * per_e + (int)(j < per_e ? j : per_e);
  };
  const int first = __builtin_amdgcn_readfirstlane(affine ? range_start(xcd) : 0);
  const int last = __builtin_amdgcn_readfirstlane(affine ? range_start(xcd + 1) : total);
  auto tile_at = [&](int r) -> int {
    const int t = affine ? first + r * per_xcd + cu : tile_of(r, blockIdx.x, gridDim.x);
    return t < last ? t : -1;
  };
  // The issue pointer runs one step ahead, over the tiles that have steps.
  int i_round = 0, i_step = 0, i_slot = 0;
  int i_tile = tile_at(0);
  if (i_tile < 0) return;
  Tile it = describe(i_tile);
  auto skip_empty = [&]() {
    while (i_tile >= 0 && it.nk == 0) {
      i_tile = tile_at(++i_round);
      if (i_tile >= 0) it = describe(i_tile);
    }
  };
  skip_empty();
  auto issue_next = [&]() {
    if (i_tile < 0) return;
    issue(it, i_step, i_slot);
    i_slot ^= 1;
    if (++i_step == it.nk) {
      i_step = 0;
      i_tile = tile_at(++i_round);
      if (i_tile >= 0) it = describe(i_tile);
      skip_empty();
    }
  };
  issue_next();

  int slot = 0;
  bool stored = false;  // an epilogue since the last copies were issued
  for (int round = 0;; ++round) {
    const int tile = tile_at(round);
    if (tile < 0) break;
    const Tile ct = describe(tile);
    ScalesSeen seen;
    v4f acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    for (int kb = 0; kb < ct.nk; ++kb) {
      // The copies of this step are older than the last epilogue's stores,
      // which stay in flight.
      if (stored)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kStores) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      stored = false;
      issue_next();
      const uint8_t* ta = smem + slot * STAGE;
      const uint8_t* tb = ta + A_SIZE;
      const float* sa = (const float*)(tb + B_SIZE);
      const float2 sa2 = *(const float2*)&sa[wm * 32 + c * 2];
      const float4 sb4 = *(const float4*)&sa[TM + wn * 64 + c * 4];
      slot ^= 1;
      v8i af[MB], bf[NB];
#pragma unroll
      for (int i = 0; i < MB; ++i) af[i] = frag(ta, (wm * MB + i) * 16 + c, lane);
#pragma unroll
      for (int j = 0; j < NB; ++j) bf[j] = frag(tb, (wn * NB + j) * 16 + c, lane);
      if constexpr (kAnyScale) seen.add(sa2.x, sa2.y, sb4.x, sb4.y, sb4.z, sb4.w);
      const int ea[MB] = {e8m0(sa2.x), e8m0(sa2.y)};
      const int eb[NB] = {e8m0(sb4.x), e8m0(sb4.y), e8m0(sb4.z), e8m0(sb4.w)};
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int i = 0; i < MB; ++i) acc[i][j] = mfma_e8(af[i], bf[j], acc[i][j], ea[i], eb[j]);
    }
    if (kAnyScale && !__all(seen.e8m0())) {
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
      const int g = lane >> 4, prow = ct.mt * TM + wm * 32, qrow = ct.nt * TN + wn * 64 + 4 * c;
#pragma unroll 1
      for (int kb = 0; kb < ct.nk; ++kb) {
        const size_t block = (size_t)(ct.k0 + kb);
        v8i af[MB];
        float4 rs[MB];
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          af[i] = frag_global(p + (size_t)(prow + i * 16 + c) * padded + block * 128, g);
          rs[i] = *(const float4*)(p_scale + block * Mf + prow + i * 16 + 4 * g);
        }
        const float4 cs = *(const float4*)(q_scale + block * Nf + qrow);
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const v8i bf = frag_global(q + (size_t)(qrow + j) * padded + block * 128, g);
          const float s = j == 0 ? cs.x : j == 1 ? cs.y : j == 2 ? cs.z : cs.w;
#pragma unroll
          for (int i = 0; i < MB; ++i) {
            const v4f raw = mfma(af[i], bf);
            acc[i][j][0] = fmaf(raw[0], rs[i].x * s, acc[i][j][0]);
            acc[i][j][1] = fmaf(raw[1], rs[i].y * s, acc[i][j][1]);
            acc[i][j][2] = fmaf(raw[2], rs[i].z * s, acc[i][j][2]);
            acc[i][j][3] = fmaf(raw[3], rs[i].w * s, acc[i][j][3]);
          }
        }
      }
    }
    const size_t row0 = (size_t)ct.e * Mf + ct.mt * TM + wm * 32;
    const size_t col0 = (size_t)ct.nt * TN + wn * 64 + c * 4;
#pragma unroll
    for (int i = 0; i < MB; ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const size_t at = (row0 + i * 16 + 4 * (lane >> 4) + r) * Nf + col0;
        if constexpr (kFp32) {
          store_stream((float*)out + at,
                       make_uint4(__float_as_uint(acc[i][0][r]), __float_as_uint(acc[i][1][r]),
                                  __float_as_uint(acc[i][2][r]), __float_as_uint(acc[i][3][r])));
        } else {
          store_stream8((uint16_t*)out + at, make_uint2(pack_bf16x2(acc[i][0][r], acc[i][1][r]),
                                                        pack_bf16x2(acc[i][2][r], acc[i][3][r])));
        }
      }
    }
    stored = true;
  }
}

}  // namespace

// 256 x 256 tiles where both feature counts are multiples of 256, 32-bit
// offsets reach the operands and the tiles fill the CUs at least once, else
// 128 x 128 tiles. Measured on MI355X (256-
// / 128-sided tiles, bf16 out, us): 2048 x 1536, 128 experts 135 / 144 at 1021
// tokens (0.8 GB written, 5.9 TB/s) and 486 / 654 at 16384; 2048 x 512, 8
// experts (128 and 512 tiles) 22 / 15 at 2048 tokens and 60 / 37 at 8192.
// The 128 x 128 kernel it replaces at other widths, with register-staged
// copies and a VALU fold of the scales, took 271 us for the two gradients of
// 1152 x 1280 and 640, 16 experts, 12004 rows in fp32; this one takes 59.
int mi355x_wgrad_launch(const uint8_t* p, const float* p_scale, int m_features, const uint8_t* q,
                        const float* q_scale, int n_features, int padded, const int32_t* offsets,
                        int experts, void* out, int out_fp32, void* stream) {
  const bool fits = m_features % BM == 0 && n_features % BN == 0 &&
                    (uint64_t)m_features * (uint64_t)padded < (1ull << 32) &&
                    (uint64_t)n_features * (uint64_t)padded < (1ull << 32);
  const bool wide =
      fits && (long long)experts * (m_features / BM) * (n_features / BN) >= cu_count();
  const int side = wide ? BM : small::TM, slots = wide ? cu_count() : 2 * cu_count();
  const long long total = (long long)experts * (m_features / side) * (n_features / side);
  const int grid = total < slots ? (int)total : slots;
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kThreads), 0, (hipStream_t)stream, p, p_scale,
                       m_features, q, q_scale, n_features, padded, offsets, experts, out);
  };
  if (wide) out_fp32 ? launch(wgrad_v2_kernel<true>) : launch(wgrad_v2_kernel<false>);
  else if (fits)
    out_fp32 ? launch(wgrad_tile_kernel<true, false, false>)
             : launch(wgrad_tile_kernel<false, false, false>);
  else if (padded < small::kFarRows)
    out_fp32 ? launch(wgrad_tile_kernel<true, true, false>)
             : launch(wgrad_tile_kernel<false, true, false>);
  else
    out_fp32 ? launch(wgrad_tile_kernel<true, true, true>)
             : launch(wgrad_tile_kernel<false, true, true>);
  MI355X_LAUNCH_CHECK();
  return MI355X_OK;
}

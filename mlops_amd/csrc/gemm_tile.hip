// Grouped block-FP8 GEMM for few rows per expert and for widths that are odd
// multiples of 128: the same products and forms as gemm_v2.hip on smaller
// tiles (kBM x 128 x 128) with a deeper copy pipeline.
//
// With few rows per expert a launch streams every touched expert's weight
// once and is bound by HBM, so what counts is copies in flight on every CU
// and no gaps between tiles. A 256 x 256 tile copies and multiplies 256 rows
// whatever the group holds, keeps one 64 KB step in flight and leaves CUs
// idle where a launch has few tiles. Here a workgroup walks the flat
// sequence of (tile, K step) pairs of its share with an issue pointer
// kStages - 1 steps ahead of the compute pointer, across tile boundaries, so
// a tile's first steps travel under the previous tile's last ones.
//
// 8 waves in a kWM x kWN grid; a wave owns MB x NB blocks of
// v_mfma_f32_16x16x128_f8f6f4. Copies, LDS swizzle and scale folding are
// gemm_pipe.h's. A tile walks K from the step at which the 256 x 256 tile it
// lies in would start (k_rotation), so that a row's result is the same sum in
// the same order whichever tiles a launch uses.
#include "gemm_pipe.h"

using namespace pipe;

namespace {

constexpr int kMaxExperts = 512;
constexpr int TN = 128;  // columns of a tile

struct TileArgs {
  const uint8_t* a;
  const float* a_scale;
  int rows;  // pitch of the K-block-major activation scales
  const uint8_t* w;
  const float* w_scale;
  int w_scale_t, experts, N, K;
  const int32_t* offsets;
  int interleave;
  const uint16_t* addend;
  uint16_t* out;
  const uint16_t* lora_z;
  const uint16_t* lora_b;
  int lora_rank;
  const int32_t* a_rows;
  uint32_t div_m;
  int div_s;
  int rotate;  // start K as the 256 x 256 tiles do (N a multiple of 256)
};

// Position of 16-byte unit u in row r of a K-major stage tile (128 K rows of
// 128 bytes): u ^ kmsw128(r). A fragment read takes 8 consecutive rows in a
// 16-lane group (rows of a pair lie in different halves of the banks, bits
// 1-2 of the row move each pair to its own unit) and rows 16 apart across the
// groups (bit 4 moves odd groups to the other four units): a 64-lane read
// meets each bank twice, its minimum.
__device__ __forceinline__ int kmsw128(int r) { return ((r >> 1) & 3) | (((r >> 4) & 1) << 2); }

__device__ __forceinline__ v8i frag_kmajor128(const uint8_t* tile, int unit, int lane) {
  const int g = lane >> 4, j = lane & 15;
  v8i r;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int row = (p >> 1) * 64 + 16 * g + (p & 1) * 8 + (j >> 1);
    const uint8_t* at = tile + row * 128 + 16 * (unit ^ kmsw128(row)) + 8 * (j & 1);
    const v2i_t v = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i_t*)(lds_ptr_t)at);
    r[2 * p] = v[0];
    r[2 * p + 1] = v[1];
  }
  return r;
}

// Wait until at most N of this wave's global operations are in flight and its
// LDS reads are done, then barrier.
template <int N>
__device__ __forceinline__ void step_sync() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <int kBM, int kWM, int kWN, int kStages, int kWavesPerSimd, bool kRow, bool kKM,
          bool kGather, bool kLora, bool kAdd>
__global__ void __launch_bounds__(kThreads, kWavesPerSimd) grouped_tile_kernel(TileArgs g) {
  static_assert(kWM * kWN == kWaves, "wave grid");
  constexpr int MB = kBM / kWM / 16, NB = TN / kWN / 16, HB = NB / 2;
  constexpr int AL = kBM / 64, BL = TN / 64;  // direct loads per wave and step: 8 rows of 128 B each
  constexpr int A_SIZE = kBM * BK, B_SIZE = TN * BK, SA_SIZE = kBM * 4;
  constexpr int SB_SIZE = kRow ? TN * 4 : 64;
  constexpr int STAGE = A_SIZE + B_SIZE + SA_SIZE + SB_SIZE;
  constexpr int kTables = 2;  // gathered-row tables: the issued tile's and the next one's
  __shared__ __align__(1024) uint8_t smem[kStages * STAGE];
  __shared__ int prefix[kMaxExperts + 1], starts[kMaxExperts + 1];
  __shared__ int gtok[kGather ? kTables : 1][kGather ? kBM : 1];
  // 256-row blocks of the experts before each one: at most rows / 256 + experts,
  // under 2^16 for the 161 rows an expert on average that choose_tiles takes.
  // Shorts, so that two workgroups of 64-row tiles still fit a CU.
  __shared__ uint16_t wide_prefix[kBM < 256 ? kMaxExperts : 1];

  const int tid = threadIdx.x, lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / kWN, wn = wave % kWN;
  const int N = g.N, K = g.K;
  {
    // Exclusive prefix of the experts' row blocks: a wave scan, then the wave
    // totals (kThreads covers every expert).
    int* wsum = (int*)smem;
    const int lo = tid < g.experts ? g.offsets[tid] : 0;
    const int hi = tid < g.experts ? g.offsets[tid + 1] : 0;
    const int v = (hi - lo + kBM - 1) / kBM, wide = (hi - lo + BM - 1) / BM;
    int x = v, xw = wide;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64), yw = __shfl_up(xw, o, 64);
      if (lane >= o) {
        x += y;
        xw += yw;
      }
    }
    if (lane == 63) {
      wsum[wave] = x;
      wsum[kWaves + wave] = xw;
    }
    __syncthreads();
    int before = 0, before_wide = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      before += w < wave ? wsum[w] : 0;
      before_wide += w < wave ? wsum[kWaves + w] : 0;
    }
    if (tid < g.experts) {
      prefix[tid] = before + x - v;
      starts[tid] = lo;
      if constexpr (kBM < 256) wide_prefix[tid] = (uint16_t)(before_wide + xw - wide);
    }
    if (tid == g.experts - 1) {
      prefix[g.experts] = before + x;
      starts[g.experts] = hi;
    }
    __syncthreads();
  }
  const int n_tiles = N / TN, nk = K / BK;
  const int kbw = K / 128, nbw = N / 128, half_n = N / 2;
  const int total = __builtin_amdgcn_readfirstlane(prefix[g.experts]) * n_tiles;

  // XCD-affine order, as in gemm_v2.hip: XCD x (= workgroup % 8) takes the
  // x-th eighth of the expert-major tile list. Inside an expert the row
  // blocks of one column tile are neighbours: they run together on one XCD
  // and read the weight panel from HBM once.
  const bool affine = (gridDim.x & 7) == 0;
  const int xcd = blockIdx.x & 7, cu = blockIdx.x >> 3, per_xcd = gridDim.x >> 3;
  const int first = affine ? (int)((long long)total * xcd / 8) : 0;
  const int last = affine ? (int)((long long)total * (xcd + 1) / 8) : total;
  auto tile_at = [&](int r) -> int {
    const int t = affine ? first + r * per_xcd + cu : tile_of(r, blockIdx.x, gridDim.x);
    return t < last ? t : -1;
  };
  struct Tile {
    int e, row0, nvalid, nt, rot;
  };
  auto describe = [&](int tile) -> Tile {
    Tile t;
    t.e = __builtin_amdgcn_readfirstlane(find_expert(prefix, g.experts, tile / n_tiles));
    const int p0 = __builtin_amdgcn_readfirstlane(prefix[t.e]);
    const int blocks = __builtin_amdgcn_readfirstlane(prefix[t.e + 1]) - p0;
    const int local = tile - p0 * n_tiles;
    t.nt = local / blocks;
    // From LDS: a load from memory here would wait for every copy in flight.
    const int lo = __builtin_amdgcn_readfirstlane(starts[t.e]);
    const int hi = __builtin_amdgcn_readfirstlane(starts[t.e + 1]);
    t.row0 = lo + (local - t.nt * blocks) * kBM;
    t.nvalid = min(kBM, hi - t.row0);
    t.rot = 0;
    if constexpr (kBM < 256) {
      if (g.rotate) {
        const int block = wide_prefix[t.e] + (t.row0 - lo) / BM;
        t.rot = __builtin_amdgcn_readfirstlane(k_rotation(block * (N / BN) + t.nt / (BN / TN), nk));
      }
    }
    return t;
  };

  // Weight row behind tile column `c` of MFMA block jb of wave column `part`:
  // a lane's NB blocks are NB consecutive output columns. Gate/up mode:
  // blocks below HB carry gates and the others ups of consecutive j, which
  // alternate in the output.
  auto weight_row = [&](int nt, int part, int jb, int c) -> int {
    if (!g.interleave) return nt * TN + part * 16 * NB + c * NB + jb;
    const int j = nt * (TN / 2) + part * 8 * NB + HB * c + jb % HB;
    return jb < HB ? j : half_n + j;
  };

  // Direct loads of the step-th K step of tile t into a stage; rows past the
  // group's end repeat its last row.
  const int lrow = lane >> 3, unit = (lane & 7) ^ (lane >> 3);
  auto issue = [&](const Tile& t, int step, int slot, int table) {
    const int kb = step + t.rot < nk ? step + t.rot : step + t.rot - nk;
    uint8_t* base = smem + slot * STAGE;
    const size_t koff = (size_t)kb * BK;
    const uint8_t* abase = g.a + koff + (kGather ? 0 : (size_t)t.row0 * K);
#pragma unroll
    for (int i = 0; i < AL; ++i) {
      const int r = (wave * AL + i) * 8 + lrow;
      uint32_t src;
      if constexpr (kGather) src = div_rows((uint32_t)gtok[table][r], g.div_m, g.div_s);
      else src = (uint32_t)min(r, t.nvalid - 1);
      dma16(abase, src * (uint32_t)K + 16 * unit, base + (wave * AL + i) * 1024);
    }
    const uint8_t* wexp = g.w + (size_t)t.e * N * K;
#pragma unroll
    for (int i = 0; i < BL; ++i) {
      const int tr = (wave * BL + i) * 8;  // first of the copy's 8 tile rows
      uint8_t* to = base + A_SIZE + (wave * BL + i) * 1024;
      if constexpr (kKM) {
        const int r = tr + lrow;
        dma16(wexp + ((size_t)kb * BK + tr) * N + (size_t)t.nt * TN,
              (uint32_t)lrow * (uint32_t)N + 16 * ((lane & 7) ^ kmsw128(r)), to);
      } else {
        const int block = tr >> 4, c = (tr & 8) + lrow;
        const size_t row = weight_row(t.nt, block / NB, block % NB, 0);
        dma16(wexp + row * K + koff,
              (uint32_t)(c * (g.interleave ? HB : NB)) * (uint32_t)K + 16 * unit, to);
      }
    }
    uint8_t* sa = base + A_SIZE + B_SIZE;
    if constexpr (kRow) {
      // One descale per row and per column: with the tile's last step.
      if (step + 1 < nk) return;
      if (wave < kBM / 64) {
        const int r = wave * 64 + lane;
        uint32_t src;
        if constexpr (kGather) src = div_rows((uint32_t)gtok[table][r], g.div_m, g.div_s);
        else src = (uint32_t)(t.row0 + min(r, t.nvalid - 1));
        dma4(g.a_scale, 4u * src, sa + wave * 256);
      } else if (wave >= kWaves - 2) {
        const int c = (wave - (kWaves - 2)) * 64;
        dma4(g.w_scale + (size_t)t.e * N + t.nt * TN + c, 4u * (uint32_t)lane, sa + SA_SIZE + c * 4);
      }
    } else {
      if (wave < kBM / 64) {
        const int r = wave * 64 + lane;
        if constexpr (kGather) {
          const uint32_t tok = div_rows((uint32_t)gtok[table][r], g.div_m, g.div_s);
          dma4(g.a_scale + kb, 4u * tok * (uint32_t)kbw, sa + wave * 256);
        } else {
          dma4(g.a_scale + (size_t)kb * g.rows + t.row0, 4u * (uint32_t)min(r, t.nvalid - 1),
               sa + wave * 256);
        }
      } else if (wave == kWaves - 1 && lane < 2) {
        // The block scales of the tile's columns: one, or gates' and ups'.
        const int col = g.interleave ? t.nt * (TN / 2) + (lane == 0 ? 0 : half_n) : t.nt * TN;
        const size_t at = g.w_scale_t || kKM ? ((size_t)t.e * kbw + kb) * nbw
                                             : (size_t)t.e * nbw * kbw + kb;
        dma4(g.w_scale + at, 4u * (uint32_t)((col >> 7) * (g.w_scale_t || kKM ? 1 : kbw)),
             sa + SA_SIZE);
      }
    }
  };
  constexpr int kLoads = AL + BL;
  const bool scaled = !kRow && (wave < kBM / 64 || wave == kWaves - 1);  // one copy more per step

  auto load_rows = [&](int tile, int table) {
    if constexpr (kGather) {
      if (tile < 0 || wave >= kBM / 64) return;
      const Tile t = describe(tile);
      dma4(g.a_rows + t.row0, 4u * (uint32_t)min(wave * 64 + lane, t.nvalid - 1),
           (const uint8_t*)&gtok[table][wave * 64]);
    }
  };

  // The issue pointer.
  int i_round = 0, i_step = 0, i_slot = 0;
  int i_tile = tile_at(0);
  if (i_tile < 0) return;
  Tile it = describe(i_tile);
  if constexpr (kGather) {
    load_rows(i_tile, 0);
    step_sync<0>();
  }
  auto issue_next = [&]() {
    if (i_tile < 0) return;
    if constexpr (kGather) {
      if (i_step == 0) {
        // The next tile's row table travels ahead of this tile's first step:
        // it has landed, for every wave, once that step has been waited for,
        // kStages - 1 iterations on. A tile of fewer steps waits here.
        if (nk < kStages && i_round > 0) step_sync<0>();
        load_rows(tile_at(i_round + 1), (i_round + 1) & (kTables - 1));
      }
    }
    issue(it, i_step, i_slot, i_round & (kTables - 1));
    i_slot = i_slot + 1 == kStages ? 0 : i_slot + 1;
    if (++i_step == nk) {
      i_step = 0;
      i_tile = tile_at(++i_round);
      if (i_tile >= 0) it = describe(i_tile);
    }
  };
#pragma unroll
  for (int s = 0; s < kStages - 1; ++s) issue_next();

  int slot = 0;
  for (int round = 0;; ++round) {
    const int tile = tile_at(round);
    if (tile < 0) break;
    const Tile ct = describe(tile);
    const int wrows = ct.nvalid - wm * 16 * MB;  // valid rows from this wave's first on
    v4f acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (kLora) {
      // The rank term starts the accumulators (see gemm_v2.hip).
      typedef short v4s __attribute__((ext_vector_type(4)));
      const int zl = lane & 15, kq = 4 * (lane >> 4);
      for (int kc = 0; kc < g.lora_rank; kc += 16) {
        v4s zf[MB];
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          const int row = ct.row0 + min(wm * 16 * MB + i * 16 + zl, ct.nvalid - 1);
          zf[i] = *(const v4s*)(g.lora_z + (size_t)row * g.lora_rank + kc + kq);
        }
#pragma unroll
        for (int jb = 0; jb < NB; ++jb) {
          const int wrow = weight_row(ct.nt, wn, jb, zl);
          const v4s bf = *(const v4s*)(g.lora_b + ((size_t)ct.e * N + wrow) * g.lora_rank + kc + kq);
#pragma unroll
          for (int i = 0; i < MB; ++i)
            acc[i][jb] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(zf[i], bf, acc[i][jb], 0, 0, 0);
        }
      }
      if constexpr (kRow) {
        float iw[NB];
#pragma unroll
        for (int jb = 0; jb < NB; ++jb)
          iw[jb] = 1.0f / g.w_scale[(size_t)ct.e * N + weight_row(ct.nt, wn, jb, zl)];
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int row = ct.row0 + min(wm * 16 * MB + i * 16 + 4 * (lane >> 4) + r, ct.nvalid - 1);
            const float ixs = 1.0f / g.a_scale[row];
#pragma unroll
            for (int jb = 0; jb < NB; ++jb) acc[i][jb][r] = (acc[i][jb][r] * ixs) * iw[jb];
          }
      }
    }

    for (int kb = 0; kb < nk; ++kb) {
      // This step's copies, older than those of the kStages - 2 steps behind
      // it (stores, tables and first-step extras only make the wait stricter).
      if (i_tile < 0) step_sync<0>();
      else if (scaled) step_sync<(kStages - 2) * (kLoads + 1)>();
      else step_sync<(kStages - 2) * kLoads>();
      issue_next();  // into the slot that the barrier has just freed
      const uint8_t* ta = smem + slot * STAGE;
      const uint8_t* tb = ta + A_SIZE;
      const float* sa = (const float*)(tb + B_SIZE);
      const float* sb = (const float*)(tb + B_SIZE + SA_SIZE);
      slot = slot + 1 == kStages ? 0 : slot + 1;
      if (wrows <= 0) continue;  // no row of this wave is in the group
      v8i af[MB], bf[NB];
#pragma unroll
      for (int jb = 0; jb < NB; ++jb) {
        if constexpr (kKM) bf[jb] = frag_kmajor128(tb, wn * NB + jb, lane);
        else bf[jb] = frag(tb, (wn * NB + jb) * 16 + (lane & 15), lane);
      }
#pragma unroll
      for (int i = 0; i < MB; ++i) af[i] = frag(ta, (wm * MB + i) * 16 + (lane & 15), lane);
      if constexpr (kRow) {
#pragma unroll
        for (int jb = 0; jb < NB; ++jb)
#pragma unroll
          for (int i = 0; i < MB; ++i) acc[i][jb] = mfma_acc(af[i], bf[jb], acc[i][jb]);
      } else {
        const float s0 = sb[0], s1 = g.interleave ? sb[1] : s0;
        float4 s4[MB];
#pragma unroll
        for (int i = 0; i < MB; ++i) s4[i] = *(const float4*)&sa[(wm * MB + i) * 16 + 4 * (lane >> 4)];
#pragma unroll
        for (int jb = 0; jb < NB; ++jb) {
          const float s = jb < HB ? s0 : s1;
#pragma unroll
          for (int i = 0; i < MB; ++i) {
            const v4f p = mfma(af[i], bf[jb]);
            acc[i][jb][0] = fmaf(p[0], s4[i].x * s, acc[i][jb][0]);
            acc[i][jb][1] = fmaf(p[1], s4[i].y * s, acc[i][jb][1]);
            acc[i][jb][2] = fmaf(p[2], s4[i].z * s, acc[i][jb][2]);
            acc[i][jb][3] = fmaf(p[3], s4[i].w * s, acc[i][jb][3]);
          }
        }
      }
    }
    if (wrows <= 0) continue;

    // Epilogue from registers: NB consecutive columns per lane, rounded to
    // bf16 once. Ordinary stores: what follows reads these few rows at once.
    const int c = lane & 15;
    float xs[MB][4], ws[NB];
    if constexpr (kRow) {
      // The descales that came with the last step, whose slot is reused only
      // after the next barrier.
      const uint8_t* st = smem + (slot == 0 ? kStages - 1 : slot - 1) * STAGE + A_SIZE + B_SIZE;
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        const float4 v = *(const float4*)(st + ((wm * MB + i) * 16 + 4 * (lane >> 4)) * 4);
        xs[i][0] = v.x; xs[i][1] = v.y; xs[i][2] = v.z; xs[i][3] = v.w;
      }
#pragma unroll
      for (int jb = 0; jb < NB; ++jb)
        ws[jb] = ((const float*)(st + SA_SIZE))[wn * 16 * NB + c * NB + jb];
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = i * 16 + 4 * (lane >> 4) + r;
        const bool live = row < wrows;
        const size_t line = (size_t)(ct.row0 + wm * 16 * MB + row) * N + ct.nt * TN + wn * 16 * NB;
        float v[NB];
        if constexpr (kKM) {
          // Lane c holds column c of each block: neighbours swap so that an
          // even lane holds columns c, c + 1 of the first block of a pair and
          // an odd lane columns c - 1, c of the second.
#pragma unroll
          for (int jb = 0; jb < NB; jb += 2) {
            const bool odd = c & 1;
            const float mine = odd ? acc[i][jb + 1][r] : acc[i][jb][r];
            const float give = odd ? acc[i][jb][r] : acc[i][jb + 1][r];
            const float got = __int_as_float(__builtin_amdgcn_update_dpp(
                0, __float_as_int(give), 0xB1, 0xF, 0xF, true));
            const uint32_t two = odd ? pack_bf16x2(got, mine) : pack_bf16x2(mine, got);
            if (live) *(uint32_t*)(g.out + line + (jb + (odd ? 1 : 0)) * 16 + (c & ~1)) = two;
          }
          continue;
        }
#pragma unroll
        for (int jb = 0; jb < NB; ++jb) {
          const int oc = g.interleave ? (jb < HB ? 2 * jb : 2 * (jb - HB) + 1) : jb;
          v[oc] = acc[i][jb][r];
        }
        if constexpr (kRow) {
#pragma unroll
          for (int jb = 0; jb < NB; ++jb) v[jb] = (v[jb] * xs[i][r]) * ws[jb];
        }
        if (!live) continue;
        const size_t at = line + c * NB;
        if constexpr (kAdd) {
#pragma unroll
          for (int jb = 0; jb < NB; ++jb) v[jb] += bf16_to_f32(g.addend[at + jb]);
        }
        if constexpr (NB == 2) {
          *(uint32_t*)(g.out + at) = pack_bf16x2(v[0], v[1]);
        } else {
          static_assert(NB == 2 || NB == 4, "store width");
          *(uint2*)(g.out + at) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
        }
      }
    }
  }
}

template <int kBM, int kWM, int kWN, int kStages, int kWavesPerSimd>
int launch_tiles(const TileArgs& g, bool row, bool kmajor, hipStream_t stream) {
  const int upper = ((g.rows + kBM - 1) / kBM + g.experts) * (g.N / TN);
  const int slots = cu_count() * kWavesPerSimd * 4 / kWaves;
  const dim3 grid(upper < slots ? upper : slots), block(kThreads);
  const bool gather = g.a_rows != nullptr, lora = g.lora_z != nullptr, add = g.addend != nullptr;
  if constexpr (kBM == 256) {
    // N an odd multiple of 128: only these forms take it.
    if (row || kmajor || gather || lora) return 1;
  }
#define TILE_FORM(R, KM, G, L, A)                                                             \
  hipLaunchKernelGGL((grouped_tile_kernel<kBM, kWM, kWN, kStages, kWavesPerSimd, R, KM, G, L, A>), \
                     grid, block, 0, stream, g)
  if constexpr (kBM < 256) {
    if (kmajor) {
      if (gather) TILE_FORM(false, true, true, false, false);
      else TILE_FORM(false, true, false, false, false);
    } else if (row) {
      if (gather) TILE_FORM(true, false, true, false, false);
      else if (lora) TILE_FORM(true, false, false, true, false);
      else TILE_FORM(true, false, false, false, false);
    } else if (gather) {
      TILE_FORM(false, false, true, false, false);
    } else if (lora) {
      TILE_FORM(false, false, false, true, false);
    }
  }
  if (!(row || kmajor || gather || lora)) {
    if (add) TILE_FORM(false, false, false, false, true);
    else TILE_FORM(false, false, false, false, false);
  }
#undef TILE_FORM
  MI355X_LAUNCH_CHECK();
  return 0;
}

// Which tiles a launch uses, from what the host knows: the rows, the experts
// they can reach and N. K and the operand form do not enter, so every form of
// a launch sums in the same order.
enum class Tiles { kNone, k64, k128, k256 };

// Row blocks of bm rows that `rows` rows over `groups` experts make on
// average: one partial block per expert, never fewer than one each.
long long row_blocks(int rows, int groups, int bm) {
  const long long whole = rows / bm + groups / 2;
  return whole > groups ? whole : groups;
}

Tiles choose_tiles(int rows, int experts, int n) {
  const int groups = rows < experts ? rows : experts;
  const int per_group = rows / groups, cus = cu_count();
  // The loads are on the device, so the lines lie by their average. Measured on
  // MI355X, weights from HBM, us (256 x 256 tiles of gemm_v2.hip / 128-row /
  // 64-row tiles). With half of the rows on one expert, or loads after a Zipf
  // law, no line loses to the 256 x 256 tiles; with all rows on one expert the
  // 64-row tiles take 0.5 to 1.6 of their time (128 experts of hidden 2048, 768:
  // 1024 rows up 30 / 16, 4096 rows 31 / 30, 6144 rows 33 / 44).
  //
  // 64-row tiles to 48 rows a group, where the launch is HBM-bound: hidden 2048,
  // 2 x 768, 128 experts at 192 rows up 107 / 66 / 57, down 44 / 35 / 31 (6.1
  // and 5.6 TB/s of weights); at 4072 rows 137 / 97 / 88 and 64 / 51 / 48.
  if (per_group <= 48) return Tiles::k64;
  // 128-row tiles that would leave CUs without a second workgroup keep too
  // little in flight: hidden 4096, 14336, 8 experts at 256 rows down
  // 187 / 118 / 86.
  if (per_group <= 128 && row_blocks(rows, groups, 128) * (n / TN) <= cus) return Tiles::k64;
  if (n % 256 == 0) {
    // A 256 x 256 grid that fills less than half the CUs: hidden 512, 1024, 8
    // experts at 4096 rows, dx 33 / 21, down 19 / 13. Or just half of them, to
    // 160 rows a group: hidden 1024, 2048, 8 experts at 640 rows up 16 / 13.
    const long long wide = row_blocks(rows, groups, 256) * (n / 256);
    if (2 * wide < cus || (2 * wide == cus && per_group <= 160)) return Tiles::k128;
    // 128-row tiles to 64 rows a group where they make one and a half rounds of
    // two workgroups a CU or more, so that an uneven routing's extra blocks are
    // a small part. At 49 / 64 rows a group, uniform routing: hidden 7168, 2048, 32
    // experts up 191, 196 / 173, 191; hidden 4096, 14336, 8 experts up 211, 209
    // / 182, 192, gathered 236, 239 / 196, 215; hidden 2048, 768, 128 experts
    // equal. One round of them (hidden 4096, 2048, 16 experts): row-scaled up
    // 50 / 45 uniform, but 55 / 69 with experts of unequal load.
    // Beyond, 256 x 256 tiles, whose waves past the expert's rows skip their
    // work: an expert of 129 rows is one block of them and two of 128. 128
    // experts of hidden 2048, 768 at 128 rows a group up 104 / 128, down 54 / 78,
    // at 160 114 / 162 and 61 / 93. On uneven loads the two lie within 20% of
    // each other, but where the wide grid just fills the CUs a block more is a
    // round more (hidden 4096, 2048, 16 experts at 96 rows: down 25 / 30 even,
    // 55 / 35 uneven). Over 2-200 rows a group of eight layer shapes, even,
    // uniform and uneven, the lines never lose more than 5% to 256 x 256 tiles.
    if (per_group <= 64 && row_blocks(rows, groups, 128) * (n / TN) >= 3ll * cus) return Tiles::k128;
    return Tiles::kNone;
  }
  // N an odd multiple of 128 (no 256-column tile): 128-row tiles, from 161 rows
  // a group on 256 x 128 tiles once they fill the CUs three times (hidden 1152,
  // 640, 16 experts at 12004 rows: 36 us against 51; hidden 4096, 14336, 8
  // experts at 4096 rows: 789 against 742).
  if (per_group <= 160) return Tiles::k128;
  return row_blocks(rows, groups, 256) * (n / TN) >= 3ll * cus ? Tiles::k256 : Tiles::k128;
}

}  // namespace

bool mi355x_gemm_tile_serves(int rows, int experts, int n) {
  return choose_tiles(rows, experts, n) != Tiles::kNone;
}

// Returns 1 when the launch is left to the 256 x 256 tiles (gemm_v2.hip).
// `row`: row-scaled operands; `kmajor`: the weight as stored, [E, K, N].
int mi355x_gemm_tile_launch(const uint8_t* a, const float* a_scale, int rows, const uint8_t* w,
                            const float* w_scale, int w_scale_t, int experts, int n, int k,
                            const int32_t* offsets, int interleave, const void* addend,
                            const void* lora_z, const void* lora_b, int lora_rank, void* out,
                            const int32_t* a_rows, int a_rows_div, bool row, bool kmajor,
                            void* stream) {
  const RowDiv div = row_div_magic(a_rows_div);
  const TileArgs g = {a, a_scale, rows, w, w_scale, w_scale_t, experts, n, k, offsets, interleave,
                      (const uint16_t*)addend, (uint16_t*)out, (const uint16_t*)lora_z,
                      (const uint16_t*)lora_b, lora_rank, a_rows, div.m, div.s,
                      n % BN == 0 && tile_order(n, k).rotate};
  hipStream_t s = (hipStream_t)stream;
  switch (choose_tiles(rows, experts, n)) {
    // Two workgroups per CU, each with 48 KB of copies in flight.
    case Tiles::k64: return launch_tiles<64, 2, 4, 3, 4>(g, row, kmajor, s);
    // Two workgroups per CU, 32 KB each.
    case Tiles::k128: return launch_tiles<128, 2, 4, 2, 4>(g, row, kmajor, s);
    // One workgroup per CU, 96 KB.
    case Tiles::k256: return launch_tiles<256, 4, 2, 3, 2>(g, row, kmajor, s);
    default: return 1;
  }
}

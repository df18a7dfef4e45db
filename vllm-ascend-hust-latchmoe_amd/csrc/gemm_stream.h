// Weight-streaming grouped GEMM on the matrix cores, for slots of few tokens
// (row tiles of 96 rows; wide slots are several tiles).
//
// HBM bounds it: a slot of up to 96 tokens does at most 96 FLOP per weight
// byte.  The GEMV kernels pay ~70 vector instructions per row pair and token;
// here a token costs a column of an MFMA, so the weight stream sets the time
// up to a few dozen tokens per slot.
//
// A block of NWB waves owns NWB * RT tiles of 16 weight rows against one row
// tile (16 NG tokens at most).  Every wave streams its own rows, 64 columns a
// stage, as 16-byte non-temporal loads of whole 128-byte row pieces (8 lanes
// per row) into a ring of D register stages: loads laid out as the MFMA wants
// them (16 rows of 64 bytes, lanes 16 apart) reach 4.4 TB/s in this kernel,
// since the L1 serves four different lines per quad of lanes.  A stage then
// takes the detour through 2 KiB of LDS per tile that only this wave touches
// (LDS operations of one wave complete in order: no barrier).  The token rows
// of a stage are loaded once per block, shared through a double-buffered LDS
// tile, with one barrier per stage that leaves the loads in flight.
// Gate-up: a tile is 8 gate rows and the 8 matching up rows, so the halves of
// a wave hold gate and up of the same 8 act columns.
//
// Each output column starts its K loop at a phase of its own (k_phase): waves
// that walk rows of 4096 bytes in step all read the same 1/16 of the memory
// channels at a time.  A plain read of 805 MB in this access pattern took
// 140 us in step and 116 us with four phases (6.95 TB/s).
//
// Every output element accumulates its K/32 MFMA steps in the order of the
// other grouped kernels (v_mfma_f32_16x16x32_bf16 gives the bits of two
// v_mfma_f32_32x32x16_bf16 steps), so all of them give identical bits.  SPLIT
// (LMOE_PATH_STREAM) instead multiplies every stage from zero, adds the
// stages' sums four at a time and those partial sums in order: the GEMVs it
// takes over from add 64 lanes' sums pairwise, and one chain of MFMA steps
// leaves twice as many act values off what f64 sums round to (K 2048: 3.4e-4
// of them, GEMV and SPLIT 1.7e-4; K 7168: 5.7e-4, 2.1e-4, 1.7e-4).
//
// Measured, gate-up + down (us): Qwen3 shape, 128 slots, 64 tokens 179 (the
// 1.18 GB of 125 slots' weights at 6.6 TB/s), 300 tokens 194, 1024 tokens 216 to
// 231; DeepSeek-V3 expert shape, 257 slots, 700 tokens 3480, 2048 tokens (72 per
// slot) 4120.  There the token rows' loads and the output rows' stores take the
// time past the weight stream's 3.3 ms, not the MFMAs or LDS (a copy without
// most of the MFMAs: 1% less).
#pragma once

#include "gemm_mfma.h"

namespace lmoe {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kStreamBM = 96;    // rows of a row tile (block_m of the permutation)
constexpr int kStreamWaves = 4;  // waves per block
constexpr int kStreamSegment = 4;  // SPLIT: stages (of 64 columns) per partial sum

struct StreamArgs {
  const uint16_t* a;  // x [T, K] (gate-up) or act [pairs, K] (down)
  const uint16_t* w;  // slot bank
  long long w_slot_stride;
  int N, K, topk, P;  // N: output columns (gate-up: I, also the offset of the up rows)
  const int32_t* offsets;
  const int32_t* sorted_pairs;
  const int32_t* tile_off;
  const int32_t* meta;
  uint16_t* out;
};

// The chunk of row r that the lane landing at position c of a 128-byte LDS
// row holds is c ^ stream_swz(r): writes of 8 lanes per row and reads of 16
// rows at one chunk both hit distinct banks.
__device__ __forceinline__ int stream_swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// LDS ordering between the waves of a block that leaves loads in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// One row tile (n rows from sorted position p0, n <= 16 NG) against this
// wave's RT tiles of weight rows, first output column n0 (the block's: nb).  A
// wave past the last column computes the block's first columns again and
// stores none.
template <int MODE, int RT, bool SPLIT, int NG, int D>
__device__ __forceinline__ void stream_tile(const StreamArgs& g, char* smem, const int* rowid,
                                            int wave, int slot, int nb, int n0, int p0, int n) {
  constexpr int NWB = kStreamWaves;
  char* wlds = smem + wave * RT * 2048;
  char* xlds = smem + NWB * RT * 2048;
  constexpr int XL = 2 * NG <= NWB ? 1 : 2 * NG / NWB;  // token-row loads of a wave per stage
  const int lane = threadIdx.x & 63;
  const int lr = lane >> 3, lc = lane & 7;
  const int r16 = lane & 15, kg = lane >> 4;
  const int KT = g.K >> 6;
  const int rot = k_phase<MODE>(n0, KT);
  uint32_t xoff[XL];
  int xw[XL];
#pragma unroll
  for (int j = 0; j < XL; ++j) {
    // rows past n load a valid row whose result is dropped; with one token
    // group the waves load its 16 rows twice (the same values)
    const int tk = (NWB > 2 * NG ? wave % (2 * NG) : j * NWB + wave) * 8 + lr;
    const int pos = p0 + (tk < n ? tk : n - 1);
    const int row = MODE == kGateUp ? g.sorted_pairs[pos] / g.topk : pos;
    xoff[j] = static_cast<uint32_t>(row) * static_cast<uint32_t>(g.K) + lc * 8;
    xw[j] = tk * 128 + ((lc ^ stream_swz(tk)) * 16);
  }
  const uint16_t* wrow[RT][2];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int row = MODE == kGateUp ? h * g.N + n0 + 8 * t : n0 + 16 * t + 8 * h;
      wrow[t][h] = g.w + static_cast<long long>(slot) * g.w_slot_stride +
                   static_cast<long long>(row) * g.K;
    }
  const uint32_t woff = static_cast<uint32_t>(lr * g.K + lc * 8);
  constexpr f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4_t acc[RT][NG], sum[SPLIT ? RT : 1][SPLIT ? NG : 1];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int q = 0; q < NG; ++q) {
      acc[t][q] = zero;
      if constexpr (SPLIT) sum[t][q] = zero;
    }
  auto end_segment = [&]() {
    if constexpr (SPLIT) {
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int q = 0; q < NG; ++q) {
          sum[t][q] += acc[t][q];
          acc[t][q] = zero;
        }
    }
  };

  u32x4_t wb[D][RT][2], xb[D][XL];
  // stages past the last load it again (a cached line) and are not multiplied.
  // Tiles past 64 rows are often one of several of their slot, whose weights
  // the others read too: these loads are plain ones, which the caches keep.
  // An expert layer's time, plain against non-temporal (us): H 7168, I 2048,
  // 257 slots, 2048 tokens with the Zipf(1.1) rank bias (391 row tiles) 4796 /
  // 5442 (L2 hits 18% against 10% in gate-up, 41 against 29 in down); H 2048, I
  // 768, 128 slots, 1200 tokens with it 317 / 359, without (one tile of 75 rows
  // per slot) 268 / 253.
  auto load = [&](int d, int kt) {
    int kr = min(kt, KT - 1) + rot;
    if (kr >= KT) kr -= KT;
    const int ko = kr * 64;
#pragma unroll
    for (int j = 0; j < XL; ++j) xb[d][j] = *reinterpret_cast<const u32x4_t*>(g.a + ko + xoff[j]);
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x4_t* src = reinterpret_cast<const u32x4_t*>(wrow[t][h] + ko + woff);
        wb[d][t][h] = NG == 6 ? *src : __builtin_nontemporal_load(src);
      }
  };
  const int ww0 = lr * 128 + ((lc ^ stream_swz(lr)) * 16);
  const int ww1 = (8 + lr) * 128 + ((lc ^ stream_swz(8 + lr)) * 16);
  int roff[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) roff[s] = r16 * 128 + (((4 * s + kg) ^ stream_swz(r16)) * 16);
  // A wave writes the token tile of stage s only after the barrier of stage
  // s - 1, which every wave reaches after its reads of stage s - 2, the last
  // ones of the same buffer.
  auto multiply = [&](int d, int kt) {
    char* xl = xlds + (kt & 1) * (NG * 2048);
#pragma unroll
    for (int j = 0; j < XL; ++j) *reinterpret_cast<u32x4_t*>(xl + xw[j]) = xb[d][j];
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      *reinterpret_cast<u32x4_t*>(wlds + t * 2048 + ww0) = wb[d][t][0];
      *reinterpret_cast<u32x4_t*>(wlds + t * 2048 + ww1) = wb[d][t][1];
    }
    lds_barrier();
    bf16x8_t wf[2][RT];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int t = 0; t < RT; ++t)
        wf[s][t] = *reinterpret_cast<const bf16x8_t*>(wlds + t * 2048 + roff[s]);
#pragma unroll
    for (int q = 0; q < NG; ++q) {
      bf16x8_t xf[2];
#pragma unroll
      for (int s = 0; s < 2; ++s)
        xf[s] = *reinterpret_cast<const bf16x8_t*>(xl + q * 2048 + roff[s]);
      f32x4_t v[RT];
#pragma unroll
      for (int t = 0; t < RT; ++t)
        v[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[0][t], xf[0], SPLIT ? zero : acc[t][q], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < RT; ++t)
        v[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[1][t], xf[1], v[t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < RT; ++t) acc[t][q] = SPLIT ? acc[t][q] + v[t] : v[t];
    }
    if (SPLIT && (kt + 1) % kStreamSegment == 0) end_segment();  // uniform
  };
#pragma unroll
  for (int d = 0; d < D; ++d) load(d, d);
  int kt = 0;
  for (; kt + D < KT; kt += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      multiply(d, kt + d);
      __builtin_amdgcn_sched_barrier(0);
      load(d, kt + D + d);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (kt + d < KT) multiply(d, kt + d);
  end_segment();

  // epilogue: the block's bf16 tile to LDS, then 16-byte pieces of whole rows
  // out (8-byte stores from the accumulators, 32 bytes per row and wave, cost
  // the DeepSeek-V3-shaped down of 72 tokens per slot 0.3 of its 1.7 ms).
  // Lane l holds token l % 16, weight rows 4 (l / 16) .. + 3 of each tile.
  constexpr int COLS = MODE == kGateUp ? 8 * RT : 16 * RT;
  constexpr int PITCH = NWB * COLS * 2 + 16;
  constexpr int CPR = NWB * COLS / 8;  // 16-byte pieces per row
  static_assert(16 * NG * PITCH <= NWB * RT * 2048 + 2 * NG * 2048, "the tile fits the operands' LDS");
  lds_barrier();  // every wave is done with the operands
#pragma unroll
  for (int q = 0; q < NG; ++q) {
    char* row = smem + (q * 16 + r16) * PITCH + wave * COLS * 2;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      const f32x4_t v = SPLIT ? sum[SPLIT ? t : 0][SPLIT ? q : 0] : acc[t][q];
      if (MODE == kGateUp) {
        float gv[4], uv[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          gv[e] = uv[e] = v[e];
          permlane_swap<32>(gv[e], uv[e]);  // lanes < 32: own gate values, lane + 32's up values
        }
        if (lane < 32)
          *reinterpret_cast<uint2*>(row + t * 16 + kg * 8) =
              make_uint2(swiglu_bf16x2(gv[0], uv[0], gv[1], uv[1]),
                         swiglu_bf16x2(gv[2], uv[2], gv[3], uv[3]));
      } else {
        *reinterpret_cast<uint2*>(row + t * 32 + kg * 8) =
            make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
      }
    }
  }
  lds_barrier();
  for (int e = threadIdx.x; e < n * CPR; e += NWB * 64) {
    const int r = e / CPR, c = e % CPR;
    if (nb + 8 * c >= g.N) continue;  // columns of waves past the last one
    const long long dst = MODE == kGateUp ? p0 + r : rowid[r];
    *reinterpret_cast<uint4*>(g.out + dst * g.N + nb + 8 * c) =
        *reinterpret_cast<const uint4*>(smem + r * PITCH + c * 16);
  }
}

// The slot of a row tile: how many slots end at or before it.  The tile
// table is read by all lanes at once (one load's latency, where a binary
// search pays one per step).
__device__ __forceinline__ int stream_tile_slot(const int32_t* tile_off, int P, int tile) {
  const int lane = threadIdx.x & 63;
  int slot = 0;
  for (int base = 0; base < P; base += 256) {
    int32_t end[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int s = base + 64 * j + lane;
      end[j] = tile_off[min(s, P - 1) + 1];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      slot += __popcll(__ballot(base + 64 * j + lane < P && end[j] <= tile));
  }
  return slot;
}

// Waves per SIMD that the registers leave: RT 1 four, RT 2 three, with the
// partial sums three and two (two or three waves take the same time), RT 4 two.
constexpr int stream_waves(int rt, bool split) {
  return rt == 4 || (rt == 2 && split) ? 2 : rt == 1 && !split ? 4 : 3;
}

// grid (blocks of output columns, most row tiles there can be).  TWO: both
// passes of a decode layer past its bank in one launch, the tiles of g first,
// then those of g2, whose act rows follow the pairs g places (an overflow
// slot's rows stay inside the n_pairs rows of the act buffer).
template <int MODE, int RT, bool SPLIT, bool TWO>
__global__ __launch_bounds__(kStreamWaves * 64, stream_waves(RT, SPLIT)) void stream_gemm_kernel(
    StreamArgs g, StreamArgs g2, int n_pairs) {
  __shared__ __attribute__((aligned(1024))) char
      smem[kStreamWaves * RT * 2048 + 2 * (kStreamBM / 16) * 2048];
  __shared__ int rowid[kStreamBM];
  int tile = blockIdx.y;
  const int tiles = g.meta[LMOE_META_TILES];
  bool second = false;
  if (tile >= tiles) {
    if (!TWO) return;
    tile -= tiles;
    if (tile >= g2.meta[LMOE_META_TILES]) return;
    second = true;
  }
  int base = 0;
  if (TWO && second) {
    base = g.meta[LMOE_META_PAIRS];
    g = g2;
    if (MODE == kGateUp) g.out += static_cast<long long>(base) * g.N;
    else g.a += static_cast<long long>(base) * g.K;
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slot = __builtin_amdgcn_readfirstlane(stream_tile_slot(g.tile_off, g.P, tile));
  const int rt = tile - g.tile_off[slot];  // the row tile of its slot
  const int cb = blockIdx.x;
  const int p0 = g.offsets[slot] + rt * kStreamBM;
  int n = min(kStreamBM, g.offsets[slot + 1] - p0);
  if (TWO && second) n = min(n, n_pairs - base - p0);
  if (n <= 0) return;  // uniform over the block
  // destination rows, read here once: in the store loop each would be a
  // load's latency
  if (MODE == kDown && threadIdx.x < n) rowid[threadIdx.x] = g.sorted_pairs[p0 + threadIdx.x];
  constexpr int COLS = MODE == kGateUp ? 8 * RT : 16 * RT;  // output columns of a wave
  const int nb = cb * kStreamWaves * COLS;
  const int n0 = nb + wave * COLS < g.N ? nb + wave * COLS : nb;
  if (n <= 16) stream_tile<MODE, RT, SPLIT, 1, 4>(g, smem, rowid, wave, slot, nb, n0, p0, n);
  else if (n <= 32) stream_tile<MODE, RT, SPLIT, 2, 4>(g, smem, rowid, wave, slot, nb, n0, p0, n);
  else if (n <= 64) stream_tile<MODE, RT, SPLIT, 4, 2>(g, smem, rowid, wave, slot, nb, n0, p0, n);
  else stream_tile<MODE, RT, SPLIT, 6, 2>(g, smem, rowid, wave, slot, nb, n0, p0, n);
}

}  // namespace lmoe

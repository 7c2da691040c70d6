// Contraction split for launches whose tiles do not fill the chip, shared by the forward and the input-gradient GEMM.
//
// A tile of these kernels occupies a CU by itself, so a launch runs in rounds of 256 tiles and a round that holds only R
// of them costs as much as a full one: 4096 columns at 1100 tokens are 80 tiles, two thirds of the chip idle for the
// whole launch.  The tiles of whole rounds run as before; each of the R others is cut along its contraction into `s`
// ranges of stages, one workgroup each, which leave their 256 x 256 fp32 sums in the workspace (256 KB, lane contiguous).
// A second launch, one workgroup per 32 tokens of a cut tile, adds the ranges in index order (the result does not depend
// on scheduling) and applies what the kernel's own epilogue does, with the same rounding points.
// (Adding the ranges in the last workgroup of a tile to arrive, without a second launch, was built first: one CU reads
// its s x 256 KB at the latency of the memory behind the L2, 90 us per launch at s = 5, more than the split saved.)
#pragma once
#include "common.h"

#include <algorithm>

namespace {

constexpr int SPLIT_CUS = 256;
constexpr int SPLIT_QUADS = 64;  // 16-byte accumulator quads per lane: 8 token tiles x 2 column tiles x 4
constexpr size_t SPLIT_TILE_BYTES = 4 * 64 * SPLIT_QUADS * 16;

struct SplitPlan {
  int n_whole;  // tiles that run whole: ids 0 .. n_whole - 1
  int n_split;  // tiles cut into ranges
  int s;        // ranges per cut tile (1: nothing is cut)
  float us;     // estimate of the launch
  size_t bytes() const { return s > 1 ? (size_t)n_split * s * SPLIT_TILE_BYTES : 0; }
};

// A stage of 64 contraction elements takes a tile about 1.4 us where the chip is not full, from a code book too; the split
// costs the second launch and the start-up of its ranges (8 us), the sums' way to memory and back (about 4 TB/s) and, where the
// second launch does more than round and store, `finish_us` per tile.  Without whole rounds a launch is held against the split
// with `start_us` beside its stages.
// Behind whole rounds less of the tiles' time is there to be won: they start as CUs come free (10 % off).  And the whole
// tiles of a cut launch run on the flavour that can cut, which takes `whole_slow` of their time more than the one that
// cannot: with whole rounds enough in front, that is more than the cut gives (SwiGLU backward 4096 -> 14336, 6107 tokens,
// five rounds and 64 tiles: 696 us whole, 766 us cut; at 256 tokens, 56 tiles: 96 and 63 us).
inline SplitPlan plan_split(int tiles, int n_stages, float whole_slow, float finish_us = 0.f, float start_us = -3.0f) {
  constexpr float stage_us = 1.4f;
  const int rest = tiles % SPLIT_CUS, rounds = tiles / SPLIT_CUS;
  SplitPlan p{tiles, 0, 1, (rounds + (rest > 0)) * n_stages * stage_us + 8.0f};
  if (rest == 0) return p;
  const float range_us = 2.0f * SPLIT_TILE_BYTES / 4.0e6f;
  const float fixed_us = 8.0f + rest * finish_us + whole_slow * rounds * n_stages * stage_us;
  // not for a gain that the noise of a launch would hide
  float best = rounds > 0 ? 0.9f * n_stages * stage_us - 3.0f : n_stages * stage_us + start_us;
  int s_best = 1;
  for (int s = 2; s <= SPLIT_CUS / rest && 2 * s <= n_stages; ++s) {
    const float us = n_stages * stage_us / s + fixed_us + rest * s * range_us;
    if (us < best) {
      best = us;
      s_best = s;
    }
  }
  if (s_best > 1) p = SplitPlan{tiles - rest, rest, s_best, rounds * n_stages * stage_us + best};
  return p;
}

// What a workgroup of a split launch works on.
struct SplitWork {
  int tile;    // tile index
  int range;   // index of the range of a cut tile, -1: whole tile
  int cut;     // index among the cut tiles
};

FMSA_DEVI SplitWork split_work(int n_whole, int n_split, int s) {
  const int id = blockIdx.x;
  if (id < n_whole) return {xcd_remap(id, n_whole), -1, 0};
  const int u = xcd_remap(id - n_whole, n_split * s);
  return {n_whole + u / s, u % s, u / s};
}

// One range's sums: quad (mt * NT + j) * 4 + i0 of lane l of wave w at [range][w][quad][l].  Token tiles past the last row are
// not read by the second launch and not written (700 tokens, two of 24: the four GEMMs of a layer 338 -> 331 us).
template <int MT, int NT>
FMSA_DEVI void split_store(const f32x16 (&acc)[MT][NT], float* partial, int cut, int range, int s, int rows) {
  static_assert(MT * NT * 4 == SPLIT_QUADS, "a wave's accumulators");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  f32x4* dst = reinterpret_cast<f32x4*>(partial + (size_t)(cut * s + range) * (SPLIT_TILE_BYTES / 4)) + (size_t)wave * SPLIT_QUADS * 64 + lane;
  static_for<0, MT>([&](auto mt_c) {
    constexpr int mt = decltype(mt_c)::value;
    if (32 * mt >= rows) return;
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int i0 = 0; i0 < 4; ++i0)
        dst[((mt * NT + j) * 4 + i0) * 64] =
            f32x4{acc[mt][j][4 * i0], acc[mt][j][4 * i0 + 1], acc[mt][j][4 * i0 + 2], acc[mt][j][4 * i0 + 3]};
  });
}

// The sums of column tile j of token tile mt of a cut tile, all ranges in index order: register layout of the GEMM's accumulators.
// Four ranges are asked for at once: a second launch is a chain of memory latencies.
template <int NT>
FMSA_DEVI void split_load(f32x4 (&acc)[4], const float* partial, int cut, int mt, int j, int s) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const f32x4* src = reinterpret_cast<const f32x4*>(partial + (size_t)cut * s * (SPLIT_TILE_BYTES / 4)) +
                     ((size_t)wave * SPLIT_QUADS + (mt * NT + j) * 4) * 64 + lane;
  for (int r0 = 0; r0 < s; r0 += 4) {
    f32x4 v[4][4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (r0 + r < s) {
#pragma unroll
        for (int q = 0; q < 4; ++q) v[r][q] = src[(size_t)(r0 + r) * (SPLIT_TILE_BYTES / 16) + q * 64];
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (r0 + r >= s) break;
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] = r0 + r == 0 ? v[r][q] : acc[q] + v[r][q];
    }
  }
}

}  // namespace

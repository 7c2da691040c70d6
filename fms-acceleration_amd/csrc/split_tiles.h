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
#include "tile_plan.h"

namespace {


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
  constexpr int QUADS = MT * NT * 4;  // of a lane
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  f32x4* dst = reinterpret_cast<f32x4*>(partial) + ((size_t)(cut * s + range) * 4 + wave) * QUADS * 64 + lane;
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
FMSA_DEVI void split_load(f32x4 (&acc)[4], const float* partial, int cut, int mt, int j, int s, int MT) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int quads = MT * NT * 4;  // of a lane
  const size_t range = (size_t)4 * quads * 64;  // quads of a range
  const f32x4* src = reinterpret_cast<const f32x4*>(partial) + cut * s * range + ((size_t)wave * quads + (mt * NT + j) * 4) * 64 + lane;
  for (int r0 = 0; r0 < s; r0 += 4) {
    f32x4 v[4][4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (r0 + r < s) {
#pragma unroll
        for (int q = 0; q < 4; ++q) v[r][q] = src[(r0 + r) * range + q * 64];
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

// Height and cut of a launch of the tiled GEMMs (tile_plan.hip): host code.
#pragma once
#include <cstddef>

#include "common.h"

constexpr int SPLIT_CUS = 256;
constexpr size_t SPLIT_ROW_BYTES = 32 * 256 * 4;  // the fp32 sums of a token tile

inline int blocks_of(int mt, int M) { return (M + 32 * mt - 1) / (32 * mt); }

struct SplitPlan {
  int mt;       // height of a tile in token tiles of 32 rows
  int n_whole;  // tiles that run whole: ids 0 .. n_whole - 1
  int n_split;  // tiles cut into ranges
  int s;        // ranges per cut tile (1: nothing is cut)
  float us;     // estimate of the launch
  size_t ask;   // what the buffer-size query answers, bytes() or more: a call that tiles of 8 would cut is one that takes a buffer
  size_t bytes() const { return s > 1 ? (size_t)n_split * s * mt * SPLIT_ROW_BYTES : 0; }
  int blocks(int M) const { return blocks_of(mt, M); }
};

// rotating: the flavours with the rotary epilogue, which run whole tiles of 8
SplitPlan plan_fwd(const fmsa_fwd_proj* projs, int n_proj, int M, int mode, bool rotating = false);
SplitPlan plan_bwd_t(const fmsa_bwd_proj* projs, int n_proj, int M, int mode);
int bwd_t_stages(const fmsa_bwd_proj* projs, int n_proj);

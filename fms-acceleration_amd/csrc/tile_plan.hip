// Height and cut of a launch of the tiled GEMMs, and which forward the kernel for few tokens takes.  Host code: the launches are in
// gemm_fwd.hip and gemm_bwd_t.hip.
#include "tile_plan.h"

#include <algorithm>

float few_us(const fmsa_fwd_proj* projs, int n_proj, int M, int mode);  // gemm_few.hip

namespace {

constexpr int BK = 64;  // contraction elements of a stage

// What a launch takes, in us; fitted to launches of 300 to 6000 tokens of 4096 and 14336 columns, 64 to 448 stages, which it gives
// within about 5 %.
//   A stage of 64 contraction elements: stage[mt] in a tile of mt token tiles by itself, more with what else the chip computes at the
// time, power * (load / that of 256 tiles of 8)^2: many tiles lower the clock, few do not (forward 4096 x 4096, tiles of 8: 81 us for
// 48 of them, 83 for 128, 107 for 256), unpacking a tile's weights counts as 1.5 token tiles.  Whole rounds of low tiles take 6 %
// more than that.
//   A round of tiles beside its stages (fill, LoRA term, stores): fixed + fixed_row * (mt - 4), and `epilogue` where the mode computes
// there.
//   Cut tiles: `finish` for the second launch and cut_row for each token tile of a range, written and read.
struct TileCost {
  float stage[5];  // mt = 4 .. 8
  float power, fixed, fixed_row, epilogue;
  float finish, cut_row;
  float whole_slow;  // what the whole rounds in front of cut tiles take longer on the flavour that can cut, of their time
  float behind;      // of the time of a rest behind whole rounds: its tiles start as CUs come free
  float range(int mt, int tiles, float n_stages) const {
    const float load = (mt + 1.5f) * tiles * (1.0f / (9.5f * SPLIT_CUS));
    return n_stages * (stage[mt - 4] + power * load * load) + fixed + fixed_row * (mt - 4);
  }
  float round(int mt, int tiles, float n_stages) const { return range(mt, tiles, n_stages) + epilogue; }
  float rounds(int mt, int n, float n_stages) const { return n * round(mt, SPLIT_CUS, n_stages) * (mt < 8 ? 1.06f : 1.0f); }
};

// Height and cut of a launch over `cols` columns of tiles.  Low tiles unpack every weight more often but come in heights that M
// fills (1100 tokens are 5 tiles of 7 token tiles, 1120 rows, or of 8, 1280), and more of them fill the chip without a cut: 4096 x
// 4096 at 1100 / 2048 / 6000 tokens 58.8 / 78.9 / 185.6 us in tiles of 8 (3 ranges, 2 ranges, whole) and 50.4 / 63.3 / 166.4 in tiles of
// 5 (2 ranges), 4 and 6 (whole).  A chip full of tiles of 8 is the fastest: 4096 tokens 106.8, in tiles of 4 124.2.
// `low`: the launch has flavours below 8.  stay_cut: so many tiles of 8 behind whole rounds, where they are cut, stay it.
inline SplitPlan whole_tiles(int mt, int M, int cols, int n_stages, const TileCost& cost) {
  const int tiles = blocks_of(mt, M) * cols, rounds = tiles / SPLIT_CUS, rest = tiles % SPLIT_CUS;
  const float rest_us = rest ? cost.round(mt, rest, n_stages) * (rounds ? cost.behind : 1.0f) : 0.f;
  return SplitPlan{mt, tiles, 0, 1, cost.rounds(mt, rounds, n_stages) + rest_us, 0};
}

inline SplitPlan plan_tiles(int M, int cols, int n_stages, bool low, const TileCost& cost, int stay_cut = 0) {
  SplitPlan best = whole_tiles(8, M, cols, n_stages, cost);
  for (int mt = 8; mt >= (low ? 4 : 8); --mt) {
    if (mt == 7 && best.s > 1 && best.n_whole > 0 && best.n_split <= stay_cut) break;
    if (mt < 8 && mt > 4 && blocks_of(mt, M) == blocks_of(mt - 1, M)) continue;  // the lower one does the same in less
    const SplitPlan whole = whole_tiles(mt, M, cols, n_stages, cost);
    const int tiles = whole.n_whole, rest = tiles % SPLIT_CUS;
    const float whole_rounds = cost.rounds(mt, tiles / SPLIT_CUS, n_stages) * (1.0f + cost.whole_slow);
    // a lower tile, and a cut, not for a gain that the noise of a launch would hide
    if (whole.us < 0.97f * best.us) best = SplitPlan{mt, tiles, 0, 1, whole.us, best.ask};
    if (mt < 8 && best.ask == 0) continue;  // what the buffer-size query says of tiles of 8 holds: no cut, no buffer
    for (int s = 2; rest && s <= SPLIT_CUS / rest && s <= 32 && 2 * s <= n_stages; ++s) {
      const float us = whole_rounds + cost.range(mt, rest * s, (float)n_stages / s) + cost.finish + rest * s * mt * cost.cut_row;
      if (us < 0.97f * best.us) best = SplitPlan{mt, tiles - rest, rest, s, us, std::max(best.ask, (size_t)rest * s * mt * SPLIT_ROW_BYTES)};
    }
  }
  return best;
}

}  // namespace

// Height and cut of a launch.  Flavours that are compiled with them: one scale group per stage, no rotary epilogue; the lower
// heights for whole stages.
SplitPlan plan_fwd(const fmsa_fwd_proj* projs, int n_proj, int M, int mode, bool rotating) {
  int nb = 0;
  bool ok = true;
  for (int p = 0; p < n_proj; ++p) {
    const fmsa_gptq_weight& w = projs[p].w;
    nb += (w.N + 255) / 256;
    ok = ok && w.group_size % 64 == 0;
  }
  if (mode == FMSA_FWD_SWIGLU) nb = (projs[0].w.N + 127) / 128;
  if (!ok) return SplitPlan{8, ((M + 255) / 256) * nb, 0, 1, 1e9f, 0};
  // whole_slow measured per whole round, over 1 to 12 of them: nothing to 1 % of its time, 3 to 5 % with the SwiGLU epilogue
  const TileCost cost = mode == FMSA_FWD_SWIGLU ? TileCost{{0.74f, 0.83f, 0.92f, 1.05f, 1.125f}, 0.375f, 6.8f, 0.6f, 2.0f, 5.0f, 0.0073f, 0.05f, 1.0f}
                                                : TileCost{{0.74f, 0.83f, 0.92f, 1.05f, 1.125f}, 0.375f, 6.8f, 0.6f, 0.0f, 5.0f, 0.0073f, 0.01f, 1.0f};
  const int n_stages = (projs[0].w.K + BK - 1) / BK;
  if (rotating) return whole_tiles(8, M, nb, n_stages, cost);
  return plan_tiles(M, nb, n_stages, projs[0].w.K % BK == 0, cost);
}

// Whether a launch is expected to take less time on the kernel for few tokens than in 256-token tiles, cut or not.  A linear
// launch that small tiles do whole (a few stages of K) stays there, where the rotating epilogue's sums are the same.
bool gptq_lora_fwd_is_few(const fmsa_fwd_proj* projs, int n_proj, int M, int mode) {
  if (M > FMSA_FEW_MAX_TOKENS) return false;
  for (int p = 0; p < n_proj; ++p)
    if (projs[p].w.group_size % 64 != 0) return false;
  const SplitPlan plan = plan_fwd(projs, n_proj, M, mode);
  if (mode != FMSA_FWD_SWIGLU && plan.ask == 0 && plan_fwd(projs, n_proj, M, mode, true).n_whole <= SPLIT_CUS / 2) return false;
  // us there / in tiles: 4096 x 4096 at 200 / 300 / 400 tokens 21 / 30 / 40 and 26 / 28 / 30, 2048 x 2048 at 700 21 and 24, 2048 ->
  // 4096 with the SwiGLU at 200 / 300 / 400 25 / 30 / 40 and 25 / 31 / 32 (where the first estimate is high by a tenth)
  return few_us(projs, n_proj, M, mode) < (mode == FMSA_FWD_SWIGLU ? 1.2f : 1.1f) * plan.us;
}

// Whether the rotating flavours, which run whole tiles of 8, are expected to take less time than the plan and the passes over what it
// wrote (3 us and 0.4 ps an element, out of the caches that it lies in).  q, k, v of hidden 4096 (k, v of 1024) rotated in the launch /
// after it, us at 512, 1100, 2048, 3217, 4096, 8192 tokens: 87 / 49, 89 / 68, 95 / 106, 195 / 163, 198 / 213, 344 / 357; of hidden 2048
// (512) at 1100, 3217, 4096, 6000: 50 / 39, 52.3 / 51.3, 54 / 62, 108 / 91.
// Launches of a few stages that run whole either way (the same sums), below the range the estimates are fitted to, keep rotating: they end
// before the host has issued the one or two launches more (about 5 us each), so the step waits for those (hidden 1024 at 256 tokens, where
// the two ways meet, 31 / 30 us).
bool gptq_lora_fwd_rope_pays(const fmsa_fwd_proj* projs, int n_proj, int M) {
  int64_t columns = 0;
  for (int p = 0; p < n_proj; ++p) columns += projs[p].w.N;
  const SplitPlan plan = plan_fwd(projs, n_proj, M, FMSA_FWD_LINEAR);
  const float after = plan.us + 3.0f + 4.0e-7f * M * columns, rotated = plan_fwd(projs, n_proj, M, FMSA_FWD_LINEAR, true).us;
  return rotated < after || (plan.ask == 0 && rotated < 20.0f);
}

size_t gptq_lora_fwd_workspace(const fmsa_fwd_proj* projs, int n_proj, int M, int mode) {
  return plan_fwd(projs, n_proj, M, mode).ask;
}

int bwd_t_stages(const fmsa_bwd_proj* projs, int n_proj) {
  int n = 0;
  for (int p = 0; p < n_proj; ++p) n += (projs[p].w.N + BK - 1) / BK;
  return n;
}

SplitPlan plan_bwd_t(const fmsa_bwd_proj* projs, int n_proj, int M, int mode) {
  const bool swiglu = mode == FMSA_BWD_SWIGLU;
  // whole_slow measured per whole round, over 1 to 6 of them: 6 to 13 % of its time, 15 to 16 % with the SwiGLU epilogue (28672 -> 4096
  // at three rounds and 96 or 128 tiles: cutting them takes 1.9 and 0.9 % off the whole MLP step; SwiGLU 4096 -> 14336 at two rounds
  // and 48 tiles: cutting them adds 1.2 %)
  const TileCost cost = swiglu ? TileCost{{0.745f, 0.78f, 0.82f, 0.90f, 0.98f}, 0.49f, 9.5f, 1.9f, 8.0f, 13.0f, 0.0073f, 0.16f, 1.0f}
                               : TileCost{{0.745f, 0.78f, 0.82f, 0.90f, 0.98f}, 0.49f, 9.5f, 1.9f, 0.0f, 5.0f, 0.0073f, 0.10f, 0.93f};
  // (the SwiGLU backward's few tiles behind whole rounds keep the order of their sums, which tests pin: 8300 tokens, 2048 -> 2048, 8 of
  // 264 tiles, 116 us, whole in tiles of 5 98)
  bool low = true;
  for (int p = 0; p < n_proj; ++p) low = low && projs[p].w.N % BK == 0;
  return plan_tiles(M, (projs[0].w.K + 255) / 256, bwd_t_stages(projs, n_proj), low, cost, swiglu ? 8 : 0);
}

size_t gptq_lora_bwd_dx_t_workspace(const fmsa_bwd_proj* projs, int n_proj, int M) {
  return std::max(plan_bwd_t(projs, n_proj, M, FMSA_BWD_LINEAR).ask, plan_bwd_t(projs, n_proj, M, FMSA_BWD_SWIGLU).ask);
}

// The input-gradient kernel's flavours for tiles of FMSA_TILE_HEIGHT (4 to 7) token tiles of 32 rows: a translation unit a height,
// so that they compile side by side.
#include "gemm_bwd_t_tiles.h"

using namespace bwd_tiles;

#define CAT_(a, b) a##b
#define CAT(a, b) CAT_(a, b)

namespace {

template <typename T, int MODE, bool CODEBOOK, bool PK16>
void launch_mode(const BwdTArgs& a, const LowLaunch& l) {
  if (l.split) hipLaunchKernelGGL((gptq_lora_bwd_dx_t_kernel<T, false, MODE, CODEBOOK, PK16, true, FMSA_TILE_HEIGHT>), l.grid, dim3(256), 0, l.st, a);
  else hipLaunchKernelGGL((gptq_lora_bwd_dx_t_kernel<T, false, MODE, CODEBOOK, PK16, false, FMSA_TILE_HEIGHT>), l.grid, dim3(256), 0, l.st, a);
}

template <typename T, bool CODEBOOK, bool PK16>
void launch(const BwdTArgs& a, const LowLaunch& l) {
  if (l.swiglu) launch_mode<T, FMSA_BWD_SWIGLU, CODEBOOK, PK16>(a, l);
  else launch_mode<T, FMSA_BWD_LINEAR, CODEBOOK, PK16>(a, l);
}

}  // namespace

void CAT(launch_bwd_tiles_, FMSA_TILE_HEIGHT)(const BwdTArgs& a, const LowLaunch& l) {
  if (l.pk16) launch<f16_t, false, true>(a, l);
  else if (l.codebook && l.bf16) launch<bf16_t, true, false>(a, l);
  else if (l.codebook) launch<f16_t, true, false>(a, l);
  else if (l.bf16) launch<bf16_t, false, false>(a, l);
  else launch<f16_t, false, false>(a, l);
}

// The forward kernel's flavours for tiles of FMSA_TILE_HEIGHT (4 to 7) token tiles of 32 rows: a translation unit a height, so that
// they compile side by side.
#include "gemm_fwd_tiles.h"

using namespace fwd_tiles;

#define CAT_(a, b) a##b
#define CAT(a, b) CAT_(a, b)

namespace {

template <typename T, bool CODEBOOK, bool PK16>
void launch(const FwdArgs& a, const LowLaunch& l) {
  if (l.split) hipLaunchKernelGGL((gptq_lora_fwd_kernel<T, 1, false, CODEBOOK, 0, PK16, true, FMSA_TILE_HEIGHT>), l.grid, dim3(256), 0, l.st, a);
  else hipLaunchKernelGGL((gptq_lora_fwd_kernel<T, 1, false, CODEBOOK, 0, PK16, false, FMSA_TILE_HEIGHT>), l.grid, dim3(256), 0, l.st, a);
}

}  // namespace

void CAT(launch_fwd_tiles_, FMSA_TILE_HEIGHT)(const FwdArgs& a, const LowLaunch& l) {
  if (l.pk16) launch<f16_t, false, true>(a, l);
  else if (l.codebook && l.bf16) launch<bf16_t, true, false>(a, l);
  else if (l.codebook) launch<f16_t, true, false>(a, l);
  else if (l.bf16) launch<bf16_t, false, false>(a, l);
  else launch<f16_t, false, false>(a, l);
}

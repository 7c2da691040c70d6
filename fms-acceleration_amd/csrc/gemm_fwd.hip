// Fused forward: launches the kernel of gemm_fwd_tiles.h, and the second launch of tiles cut along the contraction.
#include "gemm_fwd_tiles.h"

using namespace fwd_tiles;

namespace {

// Second launch of a split call: workgroup = token tile mt (32 rows) of a cut tile and, linear, one column tile of its waves
// (SwiGLU needs both, its e and its g); lane, column and register layout of the kernel above, outputs as 8-byte stores (a row
// segment of 64 bytes is completed by four of them in L2).  A chain of memory latencies: with the ranges asked for four at a
// time (split_tiles.h) the four of a layer at 700 tokens take 49 us instead of 55 (SwiGLU 14336 columns, rank 64: 14.0 -> 11.1).
template <typename T, bool SWIGLU>
__global__ __launch_bounds__(256) void gptq_lora_fwd_finish_kernel(const FwdArgs a) {
  constexpr int NJ = SWIGLU ? 1 : NT;  // workgroups a token tile
  const int MT = a.mt, BM = 32 * MT;
  const int cut = blockIdx.x / (MT * NJ), mt = blockIdx.x / NJ % MT, j = blockIdx.x % NJ;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l32 = lane & 31, half = lane >> 5;
  int bm, bn;
  fwd_tile(a, a.n_whole + cut, bm, bn);
  const int m = bm * BM + 32 * mt + l32;
  if (bm * BM + 32 * mt >= a.M) return;  // the whole workgroup
  f32x4 acc[SWIGLU ? NT : 1][4];
  split_load<NT>(acc[0], a.partial, cut, mt, j, a.n_ranges, MT);
  if constexpr (SWIGLU) split_load<NT>(acc[1], a.partial, cut, mt, 1, a.n_ranges, MT);
  if (m >= a.M) return;
  const int p = SWIGLU ? 0 : (bn >= a.nblk_start[2] ? 2 : (bn >= a.nblk_start[1] ? 1 : 0));
  auto biased = [&](const FwdProjDev& P, const f32x4& v, int col) {
    f32x4 o = v;
    if (P.bias) {
      const u32x2 bv = *reinterpret_cast<const u32x2*>(P.bias + col);
      o += f32x4{unpack_lo<T>(bv[0]), unpack_hi<T>(bv[0]), unpack_lo<T>(bv[1]), unpack_hi<T>(bv[1])};
    }
    return u32x2{pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3])};
  };
  if constexpr (SWIGLU) {
    const int col0 = bn * 128 + 32 * wave + 4 * half;
    if (bn * 128 + 32 * wave >= a.p[0].N) return;  // N % 32 == 0: a column tile is wholly inside or outside
#pragma unroll
    for (int i0 = 0; i0 < 4; ++i0) {
      const int col = col0 + 8 * i0;
      const u32x2 ev = biased(a.p[0], acc[0][i0], col), gv = biased(a.p[1], acc[1][i0], col);
      u32x2 hv;
#pragma unroll
      for (int w = 0; w < 2; ++w) {  // f = RNE(e * sigmoid(e)) on the rounded e; h = RNE(f * g) on the rounded g
        const float e0 = unpack_lo<T>(ev[w]), e1 = unpack_hi<T>(ev[w]);
        const uint32_t fv = pack2<T>(e0 * sigmoidf_(e0), e1 * sigmoidf_(e1));
        hv[w] = pack2<T>(unpack_lo<T>(fv) * unpack_lo<T>(gv[w]), unpack_hi<T>(fv) * unpack_hi<T>(gv[w]));
      }
      *reinterpret_cast<u32x2*>(a.p[0].Y + (size_t)m * a.p[0].ldy + col) = ev;
      *reinterpret_cast<u32x2*>(a.p[1].Y + (size_t)m * a.p[1].ldy + col) = gv;
      *reinterpret_cast<u32x2*>(a.H + (size_t)m * a.ldh + col) = hv;
    }
  } else {
    const FwdProjDev P = select_proj(a, p);
    const int col0 = (bn - a.nblk_start[p]) * 256 + 64 * wave + 32 * j;
    if (col0 >= P.N) return;
#pragma unroll
    for (int i0 = 0; i0 < 4; ++i0) {
      const int col = col0 + 8 * i0 + 4 * half;
      *reinterpret_cast<u32x2*>(P.Y + (size_t)m * P.ldy + col) = biased(P, acc[0][i0], col);
    }
  }
}

}  // namespace

int launch_gptq_lora_fwd(const fmsa_fwd_proj* projs, int n_proj, const void* X, int64_t ldx, int M, int mode,
                         void* H, int64_t ldh, const fmsa_rope* rope, int act_dtype, void* workspace, size_t workspace_bytes,
                         hipStream_t st) {
  FwdArgs a{};
  if (rope) {
    a.rope_cos = rope->cos;
    a.rope_sin = rope->sin;
    a.rope_ld = rope->ld;
    a.rope_rows = rope->rows;
    a.rope_head_dim = rope->head_dim;
    a.rope_mask = rope->proj_mask;
  }
  a.X = (const uint16_t*)X;
  a.ldx = ldx;
  a.M = M;
  a.K = projs[0].w.K;
  a.mode = mode;
  a.H = (uint16_t*)H;
  a.ldh = ldh;
  int nb = 0;
  for (int p = 0; p < 3; ++p) {
    a.nblk_start[p] = (p < n_proj) ? nb : 0x7fffffff;
    if (p >= n_proj) continue;
    const fmsa_fwd_proj& s = projs[p];
    FwdProjDev& d = a.p[p];
    d.qweight = s.w.qweight;
    d.scales = s.w.scales;
    d.qzeros = s.w.qzeros;
    d.code = s.w.code;
    d.block_scale = s.w.block_scale;
    d.U = (const uint16_t*)s.U;
    d.ldu = s.ldu;
    d.B = (const uint16_t*)s.B;
    d.bias = (const uint16_t*)s.bias;
    d.Y = (uint16_t*)s.Y;
    d.ldy = s.ldy;
    d.N = s.w.N;
    d.group_size = s.w.group_size;
    d.zero_offset = s.w.zero_offset;
    d.r = s.r;
    d.s = s.s;
    nb += (s.w.N + 255) / 256;
  }
  a.nblk_start[3] = 0x7fffffff;
  if (mode == FMSA_FWD_SWIGLU) nb = (projs[0].w.N + 127) / 128;
  a.nbn = nb;
  SplitPlan plan = plan_fwd(projs, n_proj, M, mode, rope != nullptr);
  if (!workspace || workspace_bytes < plan.bytes()) plan.s = 1;  // every tile runs whole
  a.mt = plan.mt;
  a.nbm = plan.blocks(M);
  dim3 grid(a.nbm * a.nbn), block(256);
  if (plan.s > 1) {
    a.n_whole = plan.n_whole;
    a.n_cut = plan.n_split;
    a.n_ranges = plan.s;
    a.partial = (float*)workspace;
    grid = dim3(plan.n_whole + plan.n_split * plan.s);
  }
  int gps = 1;
  for (int p = 0; p < n_proj; ++p) {
    const int gsz = projs[p].w.group_size;
    if (gsz % 64 != 0) gps = (gsz % 32 == 0) ? (gps > 2 ? gps : 2) : 4;
  }
  const bool ktail = (a.K % BK) != 0;
  const bool codebook = projs[0].w.format == FMSA_WEIGHT_CODEBOOK;  // api.hip: all projections of a launch share the format
  // packed-half unpack: fp16 activations and interleaved words (api.hip: then every projection is affine, interleaved, with
  // group_size % 64 == 0, and there is no rotary epilogue)
  const bool pk16 = act_dtype == FMSA_F16 && !codebook && projs[0].w.nibble_order == 1;
  const LowLaunch low{act_dtype == FMSA_BF16, codebook, pk16, plan.s > 1, grid, st};
  auto launch_low = [&]() {
    switch (plan.mt) {
      case 7: launch_fwd_tiles_7(a, low); break;
      case 6: launch_fwd_tiles_6(a, low); break;
      case 5: launch_fwd_tiles_5(a, low); break;
      default: launch_fwd_tiles_4(a, low); break;
    }
  };
  if (plan.s > 1) {
#define SPLIT_K(TT, CB, PK)                                                                                         \
  do {                                                                                                              \
    if (ktail) hipLaunchKernelGGL((gptq_lora_fwd_kernel<TT, 1, true, CB, 0, PK, true>), grid, block, 0, st, a);      \
    else hipLaunchKernelGGL((gptq_lora_fwd_kernel<TT, 1, false, CB, 0, PK, true>), grid, block, 0, st, a);           \
  } while (0)
    if (plan.mt < 8) launch_low();
    else if (pk16) SPLIT_K(f16_t, false, true);
    else if (codebook && act_dtype == FMSA_BF16) SPLIT_K(bf16_t, true, false);
    else if (codebook) SPLIT_K(f16_t, true, false);
    else if (act_dtype == FMSA_BF16) SPLIT_K(bf16_t, false, false);
    else SPLIT_K(f16_t, false, false);
#undef SPLIT_K
    FMSA_CHECK_LAUNCH();
    const bool swiglu = mode == FMSA_FWD_SWIGLU;
    const dim3 fgrid(plan.n_split * plan.mt * (swiglu ? 1 : NT));
    if (act_dtype == FMSA_BF16) {
      if (swiglu) hipLaunchKernelGGL((gptq_lora_fwd_finish_kernel<bf16_t, true>), fgrid, block, 0, st, a);
      else hipLaunchKernelGGL((gptq_lora_fwd_finish_kernel<bf16_t, false>), fgrid, block, 0, st, a);
    } else {
      if (swiglu) hipLaunchKernelGGL((gptq_lora_fwd_finish_kernel<f16_t, true>), fgrid, block, 0, st, a);
      else hipLaunchKernelGGL((gptq_lora_fwd_finish_kernel<f16_t, false>), fgrid, block, 0, st, a);
    }
    FMSA_CHECK_LAUNCH();
    return FMSA_OK;
  }
#define LAUNCH3(TT, KT, CB)                                                                          \
  do {                                                                                               \
    if (rope && rope->dtype == FMSA_F32) hipLaunchKernelGGL((gptq_lora_fwd_kernel<TT, 1, false, CB, 2>), grid, block, 0, st, a); \
    else if (rope) hipLaunchKernelGGL((gptq_lora_fwd_kernel<TT, 1, false, CB, 1>), grid, block, 0, st, a); /* api.hip: gps 1, no K tail */ \
    else if (gps == 1) hipLaunchKernelGGL((gptq_lora_fwd_kernel<TT, 1, KT, CB>), grid, block, 0, st, a);  \
    else if (gps == 2) hipLaunchKernelGGL((gptq_lora_fwd_kernel<TT, 2, KT, CB>), grid, block, 0, st, a); \
    else hipLaunchKernelGGL((gptq_lora_fwd_kernel<TT, 4, KT, CB>), grid, block, 0, st, a);           \
  } while (0)
#define LAUNCH2(TT, KT)          \
  do {                           \
    if (codebook) LAUNCH3(TT, KT, true); \
    else LAUNCH3(TT, KT, false); \
  } while (0)
#define LAUNCH(TT)            \
  do {                        \
    if (ktail) LAUNCH2(TT, true); \
    else LAUNCH2(TT, false);  \
  } while (0)
  if (plan.mt < 8) {
    launch_low();
  } else if (pk16) {
    if (ktail) hipLaunchKernelGGL((gptq_lora_fwd_kernel<f16_t, 1, true, false, 0, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((gptq_lora_fwd_kernel<f16_t, 1, false, false, 0, true>), grid, block, 0, st, a);
  } else if (act_dtype == FMSA_BF16) {
    LAUNCH(bf16_t);
  } else {
    LAUNCH(f16_t);
  }
#undef LAUNCH
#undef LAUNCH2
#undef LAUNCH3
  FMSA_CHECK_LAUNCH();
  return FMSA_OK;
}

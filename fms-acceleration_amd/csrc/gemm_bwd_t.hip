// Fused input gradient on the transposed twin: launches the kernel of gemm_bwd_t_tiles.h, the second launch of tiles
// cut along the contraction, and the kernels that build the twin and the forward's interleaved copy.
#include "gemm_bwd_t_tiles.h"

using namespace bwd_tiles;

namespace {

// Second launch of a split call: workgroup = token tile mt (32 rows) and NJ column tiles of the waves of a cut tile; lane, column
// and register layout and the rounding points of the kernel above, outputs as 8-byte stores.  One column tile instead of both
// in a workgroup: twice the waves in flight and half the registers (4096 -> 2048, 300 tokens: 27.6 -> 22.1 us for the layer's
// six; at 80 cut tiles of rank 64 the sums' bytes bound it either way, 27 us).
template <typename T, int MODE, int NJ>
__global__ __launch_bounds__(256) void gptq_lora_bwd_dx_t_finish_kernel(const BwdTArgs a) {
  constexpr bool swiglu = MODE == FMSA_BWD_SWIGLU;
  // The two column tiles share the 128-byte lines of what is read and written row by row, so their workgroups are 8 ids
  // apart, on one XCD; token tile 0 of consecutive cuts goes to different ones.  (On two XCDs the SwiGLU's six arrays moved half
  // a line at a time: 4096 -> 14336, 64 / 256 tokens, 45 / 70 us a call, and 39 / 61 this way; 4096 of 2048 at 512 41 and 36.)
  static_assert(NT == 2 && (NJ == 1 || NJ == 2), "a wave's column tiles");
  const int cut = blockIdx.x / (8 * (NT / NJ)), mt = (blockIdx.x + cut) % 8, jt = NJ == 1 ? blockIdx.x / 8 % NT : 0;
  const int MT = a.mt, BM = 32 * MT;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l32 = lane & 31, half = lane >> 5;
  int bm, bk;
  bwd_tile(a, a.n_whole + cut, bm, bk);
  const int m = bm * BM + 32 * mt + l32;
  if (mt >= MT || bm * BM + 32 * mt >= a.M) return;  // the whole workgroup
  const bool m_ok = m < a.M;
  // A workgroup is short and few are resident, so its time is its chain of memory latencies: the mask, four rank steps of
  // every projection and the sums are each asked for in one go (one step and one load after the other: 32 us at 80 tiles,
  // rank 64).
  bool any_lora = false;
  for (int p = 0; p < a.n_proj; ++p) any_lora = any_lora || select_proj(a, p).r > 0;
  const bool has_mask = a.mask_src != nullptr && any_lora;
  const int col0 = bk * 256 + 64 * wave + 32 * jt;
  u32x2 mask[NJ][4];
  f32x4 acc[NJ][4];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
#pragma unroll
    for (int i0 = 0; i0 < 4; ++i0) {
      const int col = col0 + 32 * j + 8 * i0 + 4 * half;
      mask[j][i0] = u32x2{0u, 0u};
      if (has_mask && m_ok && col < a.K) mask[j][i0] = *reinterpret_cast<const u32x2*>(a.mask_src + (size_t)m * a.ldmask + col);
    }
    split_load<NT>(acc[j], a.partial, cut, mt, jt + j, a.n_ranges, MT);
  }
  f32x16 lora[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i) lora[j][i] = 0.f;
  for (int p = 0; p < a.n_proj; ++p) {
    const BwdTProjDev P = select_proj(a, p);
    if (P.r <= 0) continue;
    f32x16 tmp[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int i = 0; i < 16; ++i) tmp[j][i] = 0.f;
    for (int j0 = 0; j0 < P.r; j0 += 64) {
      u32x4 tf[4], af[4][NJ];
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const int ko = j0 + 16 * st + 8 * half;
        tf[st] = u32x4{0u, 0u, 0u, 0u};
        if (m_ok && ko < P.r) tf[st] = *reinterpret_cast<const u32x4*>(P.T + (size_t)m * P.ldt + ko);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const int col = col0 + 32 * j;
          af[st][j] = u32x4{0u, 0u, 0u, 0u};
          if (col < a.K && ko < P.r) af[st][j] = *reinterpret_cast<const u32x4*>(P.At + (size_t)(col + l32) * P.r + ko);
        }
      }
#pragma unroll
      for (int st = 0; st < 4; ++st)
        if (j0 + 16 * st < P.r) {
#pragma unroll
          for (int j = 0; j < NJ; ++j) tmp[j] = mfma32<T>(af[st][j], tf[st], tmp[j]);
        }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int i = 0; i < 16; ++i) lora[j][i] += P.s * tmp[j][i];
  }
  if (!m_ok) return;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    if (col0 + 32 * j >= a.K) continue;
#pragma unroll
    for (int i0 = 0; i0 < 4; ++i0) {
      const int col = col0 + 32 * j + 8 * i0 + 4 * half;
      const u32x2 bv = {pack2<T>(acc[j][i0][0], acc[j][i0][1]), pack2<T>(acc[j][i0][2], acc[j][i0][3])};
      const u32x2 mv = mask[j][i0];
      u32x2 lv = {0u, 0u};
      if (any_lora) lv = u32x2{pack2<T>(lora[j][4 * i0], lora[j][4 * i0 + 1]), pack2<T>(lora[j][4 * i0 + 2], lora[j][4 * i0 + 3])};
      if constexpr (swiglu) {
        const size_t o = (size_t)m * a.ldeg + col;
        const u32x2 ev = *reinterpret_cast<const u32x2*>(a.e + o), gv = *reinterpret_cast<const u32x2*>(a.g + o);
        u32x2 hv, dgv, dev;
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          uint32_t h, dg, de;
          swiglu_bwd_pair<T>(ev[w], gv[w], bv[w], lv[w], mv[w], has_mask, h, dg, de);
          hv[w] = h;
          dgv[w] = dg;
          dev[w] = de;
        }
        *reinterpret_cast<u32x2*>(a.h + o) = hv;
        *reinterpret_cast<u32x2*>(a.e + o) = dgv;
        *reinterpret_cast<u32x2*>(a.g + o) = dev;
      } else {
        u32x2 ov = bv;
        if (any_lora) {
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            const float l0 = (!has_mask || (mv[w] & 0x7fffu)) ? unpack_lo<T>(lv[w]) : 0.f;
            const float l1 = (!has_mask || ((mv[w] >> 16) & 0x7fffu)) ? unpack_hi<T>(lv[w]) : 0.f;
            ov[w] = pack2<T>(unpack_lo<T>(bv[w]) + l0, unpack_hi<T>(bv[w]) + l1);
          }
        }
        *reinterpret_cast<u32x2*>(a.dX + (size_t)m * a.lddx + col) = ov;
      }
    }
  }
}

// qweight [K/8, N] (nibble j of word [k8, n] = q[8 k8 + j, n]) -> qweight_t [N/8, K]: word [n8, k] holds q[k, 8 n8 + e]
// with element e = 2p at nibble position p and e = 2p + 1 at position 4 + p.  One thread per 8 x 8 block of nibbles:
// 8 adjacent words in, 8 adjacent words out.  Runs once per frozen weight.
__global__ __launch_bounds__(256) void gptq_transpose_kernel(const uint32_t* __restrict__ qweight, int K8, int N8,
                                                             uint32_t* __restrict__ out) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)K8 * N8) return;
  // consecutive threads walk k8 first, so that the 32-byte output segments of a warp are adjacent
  const int k8 = (int)(idx % K8), n8 = (int)(idx / K8);
  const int N = N8 * 8, K = K8 * 8;
  uint32_t in[8], o[8];
  const u32x4* src = reinterpret_cast<const u32x4*>(qweight + (size_t)k8 * N + 8 * n8);
  const u32x4 a = src[0], b = src[1];
  in[0] = a[0]; in[1] = a[1]; in[2] = a[2]; in[3] = a[3];
  in[4] = b[0]; in[5] = b[1]; in[6] = b[2]; in[7] = b[3];
#pragma unroll
  for (int i = 0; i < 8; ++i) {  // output word i: row k = 8 k8 + i; element j comes from input word j (column 8 n8 + j)
    uint32_t w = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) w |= ((in[j] >> (4 * i)) & 0xFu) << (4 * ((j >> 1) + 4 * (j & 1)));
    o[i] = w;
  }
  u32x4* dst = reinterpret_cast<u32x4*>(out + (size_t)n8 * K + 8 * k8);
  dst[0] = u32x4{o[0], o[1], o[2], o[3]};
  dst[1] = u32x4{o[4], o[5], o[6], o[7]};
}

// The same re-ordering inside the words of the checkpoint layout itself (no transpose): out word [k8, n] holds
// q[8 k8 + e, n] with element 2p at nibble position p and element 2p + 1 at position 4 + p.  Four words per thread.
__global__ __launch_bounds__(256) void gptq_interleave_kernel(const u32x4* __restrict__ in, int64_t quads, u32x4* __restrict__ out) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= quads) return;
  const u32x4 w = in[idx];
  u32x4 o;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    uint32_t v = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) v |= ((w[c] >> (4 * e)) & 0xFu) << (4 * ((e >> 1) + 4 * (e & 1)));
    o[c] = v;
  }
  out[idx] = o;
}

}  // namespace

int launch_gptq_interleave(const int32_t* qweight, int K, int N, int32_t* out, hipStream_t st) {
  const int64_t quads = (int64_t)(K / 8) * N / 4;
  dim3 grid((unsigned)((quads + 255) / 256)), block(256);
  hipLaunchKernelGGL(gptq_interleave_kernel, grid, block, 0, st, (const u32x4*)qweight, quads, (u32x4*)out);
  FMSA_CHECK_LAUNCH();
  return FMSA_OK;
}

int launch_gptq_transpose(const int32_t* qweight, int K, int N, int32_t* out, hipStream_t st) {
  const int64_t total = (int64_t)(K / 8) * (N / 8);
  dim3 grid((unsigned)((total + 255) / 256)), block(256);
  hipLaunchKernelGGL(gptq_transpose_kernel, grid, block, 0, st, (const uint32_t*)qweight, K / 8, N / 8, (uint32_t*)out);
  FMSA_CHECK_LAUNCH();
  return FMSA_OK;
}

// Which flavour of the twin kernel a call can take: 0 none (a projection without its twin, or a group that does not hold
// whole 64-column wave tiles), 1 the fp32 scale / offset tables, 2 the packed-half unpack (fp16 activations, affine
// weights, every projection with its fp16 offset table).
int bwd_dx_twin_flavour(const fmsa_bwd_proj* projs, int n_proj, int act_dtype) {
  bool fp32_tables = true, pk16 = act_dtype == FMSA_F16;
  for (int p = 0; p < n_proj; ++p) {
    const fmsa_bwd_proj& s = projs[p];
    if (!s.qweight_t || s.w.group_size % 64 != 0) return 0;
    const bool cb = s.w.format == FMSA_WEIGHT_CODEBOOK;
    fp32_tables = fp32_tables && (cb || (s.scale_f32 && s.nsz));
    pk16 = pk16 && !cb && s.negzp_f16 && s.w.scales;
  }
  return pk16 ? 2 : (fp32_tables ? 1 : 0);
}

int launch_gptq_lora_bwd_dx_t(const fmsa_bwd_proj* projs, int n_proj, int M, int mode, void* dX, int64_t lddx,
                              void* e, void* g, void* h_out, int64_t ldeg, int act_dtype, void* workspace,
                              size_t workspace_bytes, hipStream_t st) {
  BwdTArgs a{};
  a.n_proj = n_proj;
  a.M = M;
  a.K = projs[0].w.K;
  a.dX = (uint16_t*)dX;
  a.lddx = lddx;
  a.e = (uint16_t*)e;
  a.g = (uint16_t*)g;
  a.h = (uint16_t*)h_out;
  a.ldeg = ldeg;
  bool ntail = false;
  for (int p = 0; p < n_proj; ++p) {
    const fmsa_bwd_proj& s = projs[p];
    BwdTProjDev& d = a.p[p];
    const bool cb = s.w.format == FMSA_WEIGHT_CODEBOOK;
    d.qt = s.qweight_t;
    d.sc = cb ? s.w.block_scale : s.scale_f32;
    d.nsz = cb ? nullptr : s.nsz;
    d.sc16 = s.w.scales;
    d.nz16 = (const uint16_t*)s.negzp_f16;
    d.code = s.w.code;
    d.dY = (const uint16_t*)s.dY;
    d.lddy = s.lddy;
    d.T = (const uint16_t*)s.T;
    d.ldt = s.ldt;
    d.At = (const uint16_t*)s.At;
    d.N = s.w.N;
    d.group_size = s.w.group_size;
    d.r = s.r;
    d.s = s.s;
    if (s.mask_src && s.r > 0) {
      a.mask_src = (const uint16_t*)s.mask_src;
      a.ldmask = s.ldmask;
    }
    ntail = ntail || (s.w.N % BK != 0);
  }
  SplitPlan plan = plan_bwd_t(projs, n_proj, M, mode);
  if (!workspace || workspace_bytes < plan.bytes()) plan.s = 1;  // every tile runs whole
  a.mt = plan.mt;
  a.nbm = plan.blocks(M);
  a.nbk = (a.K + 255) / 256;
  dim3 grid(a.nbm * a.nbk), block(256);
  if (plan.s > 1) {
    a.n_whole = plan.n_whole;
    a.n_cut = plan.n_split;
    a.n_ranges = plan.s;
    a.n_stages_all = bwd_t_stages(projs, n_proj);
    a.partial = (float*)workspace;
    grid = dim3(plan.n_whole + plan.n_split * plan.s);
  }
  const bool codebook = projs[0].w.format == FMSA_WEIGHT_CODEBOOK;  // api.hip: all projections of a launch share the format
  const bool pk16 = bwd_dx_twin_flavour(projs, n_proj, act_dtype) == 2;
#define LAUNCH_S(TT, NTL, MD, CB, PK)                                                                                       \
  do {                                                                                                                    \
    if (plan.s > 1) hipLaunchKernelGGL((gptq_lora_bwd_dx_t_kernel<TT, NTL, MD, CB, PK, true>), grid, block, 0, st, a);     \
    else hipLaunchKernelGGL((gptq_lora_bwd_dx_t_kernel<TT, NTL, MD, CB, PK>), grid, block, 0, st, a);                      \
  } while (0)
#define LAUNCH_PK(MD)                                                                                          \
  do {                                                                                                         \
    if (ntail) LAUNCH_S(f16_t, true, MD, false, true);                                                         \
    else LAUNCH_S(f16_t, false, MD, false, true);                                                              \
  } while (0)
#define LAUNCH_C(TT, MD, CB)                                                                             \
  do {                                                                                                   \
    if (ntail) LAUNCH_S(TT, true, MD, CB, false);                                                        \
    else LAUNCH_S(TT, false, MD, CB, false);                                                             \
  } while (0)
#define LAUNCH_M(TT, MD)                  \
  do {                                    \
    if (codebook) LAUNCH_C(TT, MD, true); \
    else LAUNCH_C(TT, MD, false);         \
  } while (0)
#define LAUNCH(TT)                                              \
  do {                                                          \
    if (mode == FMSA_BWD_SWIGLU) LAUNCH_M(TT, FMSA_BWD_SWIGLU); \
    else LAUNCH_M(TT, FMSA_BWD_LINEAR);                         \
  } while (0)
  if (plan.mt < 8) {
    const LowLaunch low{act_dtype == FMSA_BF16, codebook, pk16, mode == FMSA_BWD_SWIGLU, plan.s > 1, grid, st};
    switch (plan.mt) {
      case 7: launch_bwd_tiles_7(a, low); break;
      case 6: launch_bwd_tiles_6(a, low); break;
      case 5: launch_bwd_tiles_5(a, low); break;
      default: launch_bwd_tiles_4(a, low); break;
    }
  } else if (pk16) {
    if (mode == FMSA_BWD_SWIGLU) LAUNCH_PK(FMSA_BWD_SWIGLU);
    else LAUNCH_PK(FMSA_BWD_LINEAR);
  } else if (act_dtype == FMSA_BF16) {
    LAUNCH(bf16_t);
  } else {
    LAUNCH(f16_t);
  }
#undef LAUNCH
#undef LAUNCH_M
#undef LAUNCH_C
#undef LAUNCH_PK
#undef LAUNCH_S
  FMSA_CHECK_LAUNCH();
  if (plan.s > 1) {
    // Many ranks are another chain of reads, of T by every column tile: both in a workgroup where ranks add up to 128 and the
    // workgroups still are two to a CU, or many (one / both, us a call: q, k, v of rank 64 at 2048 tokens, K 4096, 128 tiles, 126.5 /
    // 123.0, K 2048, 64 tiles, 56.0 / 52.1, rank 128 69 / 61; 2560 tokens, K 2048, 80 tiles, 80.3 / 80.4, K 3072, 72, 1.05 of the time)
    int ranks = 0;
    for (int p = 0; p < n_proj; ++p) ranks += projs[p].r;
    const bool both = mode != FMSA_BWD_SWIGLU && ranks >= 128 && (plan.n_split == 64 || plan.n_split > 96);
    const dim3 fgrid(plan.n_split * 8 * (both ? 1 : NT));
#define FINISH(TT)                                                                                                                     \
  do {                                                                                                                                 \
    if (mode == FMSA_BWD_SWIGLU) hipLaunchKernelGGL((gptq_lora_bwd_dx_t_finish_kernel<TT, FMSA_BWD_SWIGLU, 1>), fgrid, block, 0, st, a); \
    else if (both) hipLaunchKernelGGL((gptq_lora_bwd_dx_t_finish_kernel<TT, FMSA_BWD_LINEAR, 2>), fgrid, block, 0, st, a);              \
    else hipLaunchKernelGGL((gptq_lora_bwd_dx_t_finish_kernel<TT, FMSA_BWD_LINEAR, 1>), fgrid, block, 0, st, a);                        \
  } while (0)
    if (act_dtype == FMSA_BF16) FINISH(bf16_t);
    else FINISH(f16_t);
#undef FINISH
    FMSA_CHECK_LAUNCH();
  }
  return FMSA_OK;
}

// Standalone SwiGLU forward / backward (UL/swiglu.py:20-98).  The fused GEMM epilogues apply the
// same arithmetic; these kernels serve the paths that cannot fuse it (act-order weights, whose
// gate/up/down projections each walk K in their own order) and the unfused baseline.
// HBM-bound: 16-byte vectors, one pass.
#include "common.h"

namespace {

template <typename T>
__global__ __launch_bounds__(256) void swiglu_fwd_kernel(const uint16_t* __restrict__ e, const uint16_t* __restrict__ g,
                                                         uint16_t* __restrict__ h, int M, int I, int64_t ld) {
  const int64_t vec = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // over M * I / 8
  const int per_row = I / 8;
  if (vec >= (int64_t)M * per_row) return;
  const int64_t off = (vec / per_row) * ld + (vec % per_row) * 8;
  const u32x4 ev = *reinterpret_cast<const u32x4*>(e + off);
  const u32x4 gv = *reinterpret_cast<const u32x4*>(g + off);
  u32x4 hv;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float e0 = unpack_lo<T>(ev[i]), e1 = unpack_hi<T>(ev[i]);
    const uint32_t f = pack2<T>(e0 * sigmoidf_(e0), e1 * sigmoidf_(e1));
    hv[i] = pack2<T>(unpack_lo<T>(f) * unpack_lo<T>(gv[i]), unpack_hi<T>(f) * unpack_hi<T>(gv[i]));
  }
  *reinterpret_cast<u32x4*>(h + off) = hv;
}

// in place: h_out <- f*g, e <- d_g = dh*f, g <- d_e
template <typename T>
__global__ __launch_bounds__(256) void swiglu_bwd_kernel(const uint16_t* __restrict__ dh, int64_t lddh,
                                                         uint16_t* __restrict__ e, uint16_t* __restrict__ g,
                                                         uint16_t* __restrict__ h, int M, int I, int64_t ld) {
  const int64_t vec = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int per_row = I / 8;
  if (vec >= (int64_t)M * per_row) return;
  const int64_t row = vec / per_row, col = (vec % per_row) * 8;
  const int64_t off = row * ld + col;
  const u32x4 dv = *reinterpret_cast<const u32x4*>(dh + row * lddh + col);
  const u32x4 ev = *reinterpret_cast<const u32x4*>(e + off);
  const u32x4 gv = *reinterpret_cast<const u32x4*>(g + off);
  u32x4 hv, dgv, dev;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float hh[2], dg[2], de[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float e32 = j ? unpack_hi<T>(ev[i]) : unpack_lo<T>(ev[i]);
      const float g32 = j ? unpack_hi<T>(gv[i]) : unpack_lo<T>(gv[i]);
      const float DW = j ? unpack_hi<T>(dv[i]) : unpack_lo<T>(dv[i]);
      const float se = sigmoidf_(e32);
      const float f = unpack1<T>(pack1<T>(se * e32));
      hh[j] = f * g32;
      dg[j] = DW * f;
      const float dgt = unpack1<T>(pack1<T>(DW * g32));
      de[j] = dgt * se * (1.0f + e32 * (1.0f - se));
    }
    hv[i] = pack2<T>(hh[0], hh[1]);
    dgv[i] = pack2<T>(dg[0], dg[1]);
    dev[i] = pack2<T>(de[0], de[1]);
  }
  *reinterpret_cast<u32x4*>(h + off) = hv;
  *reinterpret_cast<u32x4*>(e + off) = dgv;
  *reinterpret_cast<u32x4*>(g + off) = dev;
}

// ---- adapter pack ------------------------------------------------------------------------------
// One launch turns the two LoRA parameters (any float type) into the four activation-type copies
// the GEMM kernels read: A [r, K], A^T [K, r], B [N, r], B^T [r, N].  Each conversion is one RNE
// rounding of the parameter value (the `.to(dtype)` of UL/gptq/fast_lora.py:167).
template <typename TIN> FMSA_DEVI float load_param(const void* p, int64_t i);
template <> FMSA_DEVI float load_param<float>(const void* p, int64_t i) { return reinterpret_cast<const float*>(p)[i]; }
template <> FMSA_DEVI float load_param<bf16_t>(const void* p, int64_t i) { return bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(p)[i]); }
template <> FMSA_DEVI float load_param<f16_t>(const void* p, int64_t i) { return fp16_bits_to_f32(reinterpret_cast<const uint16_t*>(p)[i]); }

// The adapters of one fused operator go out together (one launch instead of one per projection); workgroup ids
// are laid end to end over the jobs.
struct LoraPackArgs {
  fmsa_lora_pack_job j[FMSA_LORA_PACK_MAX_JOBS];
  int block_start[FMSA_LORA_PACK_MAX_JOBS];
  int n_jobs;
};
FMSA_DEVI float load_param_rt(const void* p, int64_t i, int dtype) {
  if (dtype == FMSA_F32) return load_param<float>(p, i);
  return dtype == FMSA_BF16 ? load_param<bf16_t>(p, i) : load_param<f16_t>(p, i);
}

// A workgroup takes a tile of 4096 elements (1024 up to rank 16 and of matrices up to 128 Ki elements, which are a matter of
// latency: 2048 x 2048 of rank 32 4.2 us with the large tile, 3.6 with the small one) of one matrix
// (A [r, K] or B [N, r]), as many ranks wide as there are (a power of two from 8 to 64), in 4-element pieces: the rounded copy
// leaves row by row as it came, the transposed copy through LDS, so that both are written in whole lines.  (One thread per
// element wrote the transposed copies 2 bytes at a time, r or N elements apart; q, k, v / the MLP's three of 4096 and 14336: 5.0 /
// 9.6 -> 3.7 / 4.5 us at rank 32, 9.0 / 21 -> 4.1 / 5.8 at rank 64.)
__host__ __device__ inline int pack_log2_ranks(int r) { return r > 32 ? 6 : (r > 16 ? 5 : (r > 8 ? 4 : 3)); }
__host__ __device__ inline int pack_log2_tile(int r, int n) { return r > 16 && (int64_t)r * n > (1 << 17) ? 12 : 10; }
__host__ __device__ inline int pack_tiles(int r, int n) {  // of a matrix of r ranks and n columns (A) or rows (B)
  const int lr = pack_log2_ranks(r), ln = pack_log2_tile(r, n) - lr;
  return ((r + (1 << lr) - 1) >> lr) * ((n + (1 << ln) - 1) >> ln);
}
template <typename T>
__global__ __launch_bounds__(256) void lora_pack_kernel(const LoraPackArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t tile[128 * 34];  // 2^log_rows rows of 2^log_cols + 2: the most for 32 ranks of B
  // the job that owns this workgroup, copied field by field (no runtime index into the argument struct)
  fmsa_lora_pack_job J = a.j[0];
  int start = 0;
#pragma unroll
  for (int q = 1; q < FMSA_LORA_PACK_MAX_JOBS; ++q)
    if (q < a.n_jobs && (int)blockIdx.x >= a.block_start[q]) {
      J = a.j[q];
      start = a.block_start[q];
    }
  const int lr = pack_log2_ranks(J.r), rt = (J.r + (1 << lr) - 1) >> lr, n_a = pack_tiles(J.r, J.K);
  int t = blockIdx.x - start;
  const bool is_a = t < n_a;
  if (!is_a) t -= n_a;
  const int rows = is_a ? J.r : J.N, cols = is_a ? J.K : J.r;
  const int log_tile = pack_log2_tile(J.r, is_a ? J.K : J.N), log_rows = is_a ? lr : log_tile - lr, log_cols = log_tile - log_rows;
  const int rank0 = (t % rt) << lr, other0 = (t / rt) << (log_tile - lr);
  const int row0 = is_a ? rank0 : other0, col0 = is_a ? other0 : rank0;
  const int stride = (1 << log_cols) + 2;
  const void* src = is_a ? J.A : J.B;
  uint16_t* copy = reinterpret_cast<uint16_t*>(is_a ? J.A16 : J.B16);
  uint16_t* turned = reinterpret_cast<uint16_t*>(is_a ? J.At16 : J.Bt16);
  // parameters may be views into a flat buffer and begin anywhere; ranks, K and N of the fused operators are multiples of 8
  const bool f32 = J.param_dtype == FMSA_F32, wide = cols % 4 == 0 && reinterpret_cast<uintptr_t>(src) % (f32 ? 16 : 8) == 0;
  const bool wide_copy = cols % 4 == 0 && reinterpret_cast<uintptr_t>(copy) % 8 == 0;
  const bool wide_turned = rows % 4 == 0 && reinterpret_cast<uintptr_t>(turned) % 8 == 0;
#pragma unroll 4
  for (int i = 0; i < 1 << (log_tile - 10); ++i) {
    const int p = threadIdx.x + 256 * i, rr = p >> (log_cols - 2), piece = 4 * (p & ((1 << (log_cols - 2)) - 1));
    if (row0 + rr >= rows || col0 + piece >= cols) continue;
    const int64_t at = (int64_t)(row0 + rr) * cols + col0 + piece;
    const int n = min(4, cols - (col0 + piece));
    f32x4 f = {0.f, 0.f, 0.f, 0.f};
    if (wide && f32) {
      f = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(src) + at);
    } else if (wide) {
      const u32x2 w = *reinterpret_cast<const u32x2*>(reinterpret_cast<const uint16_t*>(src) + at);
      if (J.param_dtype == FMSA_BF16)
        f = f32x4{unpack_lo<bf16_t>(w[0]), unpack_hi<bf16_t>(w[0]), unpack_lo<bf16_t>(w[1]), unpack_hi<bf16_t>(w[1])};
      else
        f = f32x4{unpack_lo<f16_t>(w[0]), unpack_hi<f16_t>(w[0]), unpack_lo<f16_t>(w[1]), unpack_hi<f16_t>(w[1])};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (e < n) f[e] = load_param_rt(src, at + e, J.param_dtype);
    }
    const u32x2 v = {pack2<T>(f[0], f[1]), pack2<T>(f[2], f[3])};
    if (copy && wide_copy) {
      *reinterpret_cast<u32x2*>(copy + at) = v;
    } else if (copy) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (e < n) copy[at + e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
    }
    uint32_t* l = reinterpret_cast<uint32_t*>(tile + rr * stride + piece);
    l[0] = v[0];
    l[1] = v[1];
  }
  __syncthreads();
  if (!turned) return;
#pragma unroll 4
  for (int i = 0; i < 1 << (log_tile - 10); ++i) {
    const int p = threadIdx.x + 256 * i, cc = p >> (log_rows - 2), piece = 4 * (p & ((1 << (log_rows - 2)) - 1));
    if (col0 + cc >= cols || row0 + piece >= rows) continue;
    uint16_t* out = turned + (int64_t)(col0 + cc) * rows + row0 + piece;
    if (wide_turned) {
      const uint16_t* l = tile + piece * stride + cc;
      *reinterpret_cast<u32x2*>(out) = u32x2{l[0] | (uint32_t)l[stride] << 16, l[2 * stride] | (uint32_t)l[3 * stride] << 16};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (row0 + piece + e < rows) out[e] = tile[(piece + e) * stride + cc];
    }
  }
}

}  // namespace

int launch_swiglu_fwd(const void* e, const void* g, void* h, int M, int I, int64_t ld, int act_dtype, hipStream_t st) {
  const int64_t nvec = (int64_t)M * (I / 8);
  dim3 grid((unsigned)((nvec + 255) / 256)), block(256);
  if (act_dtype == FMSA_BF16)
    hipLaunchKernelGGL(swiglu_fwd_kernel<bf16_t>, grid, block, 0, st, (const uint16_t*)e, (const uint16_t*)g,
                       (uint16_t*)h, M, I, ld);
  else
    hipLaunchKernelGGL(swiglu_fwd_kernel<f16_t>, grid, block, 0, st, (const uint16_t*)e, (const uint16_t*)g,
                       (uint16_t*)h, M, I, ld);
  FMSA_CHECK_LAUNCH();
  return FMSA_OK;
}

int launch_swiglu_bwd(const void* dh, int64_t lddh, void* e, void* g, void* h, int M, int I, int64_t ld, int act_dtype,
                      hipStream_t st) {
  const int64_t nvec = (int64_t)M * (I / 8);
  dim3 grid((unsigned)((nvec + 255) / 256)), block(256);
  if (act_dtype == FMSA_BF16)
    hipLaunchKernelGGL(swiglu_bwd_kernel<bf16_t>, grid, block, 0, st, (const uint16_t*)dh, lddh, (uint16_t*)e,
                       (uint16_t*)g, (uint16_t*)h, M, I, ld);
  else
    hipLaunchKernelGGL(swiglu_bwd_kernel<f16_t>, grid, block, 0, st, (const uint16_t*)dh, lddh, (uint16_t*)e,
                       (uint16_t*)g, (uint16_t*)h, M, I, ld);
  FMSA_CHECK_LAUNCH();
  return FMSA_OK;
}

int launch_lora_pack_batch(const fmsa_lora_pack_job* jobs, int n_jobs, int act_dtype, hipStream_t st) {
  LoraPackArgs a{};
  a.n_jobs = n_jobs;
  int64_t blocks = 0;
  for (int q = 0; q < n_jobs; ++q) {
    a.j[q] = jobs[q];
    a.block_start[q] = (int)blocks;
    blocks += pack_tiles(jobs[q].r, jobs[q].K) + pack_tiles(jobs[q].r, jobs[q].N);
  }
  dim3 grid((unsigned)blocks), block(256);
  if (act_dtype == FMSA_BF16)
    hipLaunchKernelGGL(lora_pack_kernel<bf16_t>, grid, block, 0, st, a);
  else
    hipLaunchKernelGGL(lora_pack_kernel<f16_t>, grid, block, 0, st, a);
  FMSA_CHECK_LAUNCH();
  return FMSA_OK;
}

// The rank-r LoRA GEMMs.  Both stream one [M, C] activation matrix exactly once and are bound
// by HBM bandwidth, not by arithmetic:
//   lora_down  out[M, r]  = X[M, C] * Wd[r, C]^T          (U = Xd A^T,  T = dY B)
//   lora_grad  out[r, C]  = scale * L[M, r]^T * R[M, C]    (dA, dB: a reduction over tokens)
#include "common.h"

#include <algorithm>

namespace {

// The big operand is read exactly once: its loads carry the non-temporal hint (`nt`: direct-to-LDS loads through the
// aux operand, register loads through __builtin_nontemporal_load), so that the stream does not push the small operand
// that every workgroup re-reads (Wd, L) out of L2.  Worth 5-10 % of the launch at 235 MB and rank <= 32.
// ---- lora_down ----------------------------------------------------------------------------------
// One workgroup = 16 * MTL tokens; its NW waves split C into NW contiguous slices and each runs
// MFMA 16x16x32 over its slice (X fragments straight from global: 16 rows x 64 B per load; a Wd
// fragment is loaded once per step and used for all MTL token tiles).  The kernel lives on memory
// latency, so a workgroup is up to 16 waves: that many independent load streams per CU are what
// keeps enough bytes in flight.  The NW partial [16 * MTL x r] tiles are summed through LDS in a
// fixed order: the upper half of the waves hands its tiles to the lower half, whose sums are then
// added up by all threads.
// With few tokens one workgroup per 16 of them leaves most CUs idle and every wave with a long serial walk over its slice
// (40 us at 1100 tokens x 4096, rank 64; 17 us for ONE token), so the columns are also split over gridDim.y workgroups:
// their fp32 sums go to partial[split][M][r], which lora_down_reduce_kernel adds in index order.
template <typename T, int RT, int MTL, int NW>
FMSA_DEVI void lora_down_tile(const uint16_t* __restrict__ X, int64_t ldx, const uint16_t* __restrict__ Wd, int M, int C, int r,
                              uint16_t* __restrict__ out, int64_t ldo, float* __restrict__ partial, int n_split) {
  constexpr int NH = NW / 2;
  __shared__ float red[NH][MTL][RT][64][4];
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int l16 = lane & 15, q = lane >> 4;
  const int m_base = blockIdx.x * (16 * MTL);
  // slice boundaries in units of 32 columns
  const int n32 = (C + 31) / 32;
  const int slice = blockIdx.y * NW + wave, n_slices = n_split * NW;
  const int per = (n32 + n_slices - 1) / n_slices;
  const int c_begin = min(C, slice * per * 32);
  const int c_end = min(C, (slice + 1) * per * 32);

  f32x4 acc[MTL][RT];
#pragma unroll
  for (int u = 0; u < MTL; ++u)
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  const uint16_t* xrow[MTL];
  bool m_ok[MTL];
#pragma unroll
  for (int u = 0; u < MTL; ++u) {
    const int m = m_base + 16 * u + l16;
    m_ok[u] = m < M;
    xrow[u] = X + (size_t)(m_ok[u] ? m : 0) * ldx + 8 * q;
  }
#pragma unroll 4
  for (int c0 = c_begin; c0 < c_end; c0 += 32) {
    const bool c_ok = (c0 + 8 * q) < c_end;
    u32x4 xf[MTL];
#pragma unroll
    for (int u = 0; u < MTL; ++u) {
      xf[u] = u32x4{0u, 0u, 0u, 0u};
      if (m_ok[u] && c_ok) xf[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(xrow[u] + c0));
    }
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      const int j = 16 * t + l16;
      u32x4 wf = {0u, 0u, 0u, 0u};
      if (j < r && c_ok) wf = *reinterpret_cast<const u32x4*>(Wd + (size_t)j * C + c0 + 8 * q);
#pragma unroll
      for (int u = 0; u < MTL; ++u) acc[u][t] = mfma16<T>(xf[u], wf, acc[u][t]);  // D[i = token][j = rank]
    }
  }
  if (wave >= NH) {
#pragma unroll
    for (int u = 0; u < MTL; ++u)
#pragma unroll
      for (int t = 0; t < RT; ++t) *reinterpret_cast<f32x4*>(red[wave - NH][u][t][lane]) = acc[u][t];
  }
  __syncthreads();
  if (wave < NH) {
#pragma unroll
    for (int u = 0; u < MTL; ++u)
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        const f32x4 o = *reinterpret_cast<const f32x4*>(red[wave][u][t][lane]);
        *reinterpret_cast<f32x4*>(red[wave][u][t][lane]) = acc[u][t] + o;
      }
  }
  __syncthreads();
  // lane l of a tile holds D[4*(l>>4) + i][l & 15]; all threads sum MTL*RT*256 outputs over the NH slots
  for (int o = tid; o < MTL * RT * 256; o += 64 * NW) {
    const int u = o / (RT * 256), t = (o >> 8) % RT, ln = (o >> 2) & 63, i = o & 3;
    float v = red[0][u][t][ln][i];
#pragma unroll
    for (int w = 1; w < NH; ++w) v += red[w][u][t][ln][i];
    const int row = m_base + 16 * u + 4 * (ln >> 4) + i;
    const int j = 16 * t + (ln & 15);
    if (row < M && j < r) {
      if (partial)
        partial[((size_t)blockIdx.y * M + row) * r + j] = v;
      else
        out[(size_t)row * ldo + j] = pack1<T>(v);
    }
  }
}

template <typename T, int RT, int MTL, int NW>
__global__ __launch_bounds__(64 * NW) void lora_down_kernel(const uint16_t* __restrict__ X, int64_t ldx,
                                                            const uint16_t* __restrict__ Wd, int M, int C, int r,
                                                            uint16_t* __restrict__ out, int64_t ldo, float* __restrict__ partial) {
  lora_down_tile<T, RT, MTL, NW>(X, ldx, Wd, M, C, r, out, ldo, partial, gridDim.y);
}

// Several products over the same few tokens in one launch (q, k, v; gate, up): blockIdx.z names the job.  A launch of one
// of them is 14 us at 1100 tokens, rank 64, most of it ramp and latency; its column sums are another launch.
struct LoraDownJobDev {
  const uint16_t* X;
  const uint16_t* Wd;
  uint16_t* out;
  float* partial;
  int64_t ldx, ldo;
  int C, r, n_split;
};
struct LoraDownArgs {
  LoraDownJobDev j[FMSA_LORA_DOWN_MAX_JOBS];
  int M, r_max;
};
FMSA_DEVI LoraDownJobDev select_down_job(const LoraDownArgs& a, int q) { return q == 0 ? a.j[0] : (q == 1 ? a.j[1] : a.j[2]); }

template <typename T, int RT, int MTL, int NW>
__global__ __launch_bounds__(64 * NW) void lora_down_batch_kernel(const LoraDownArgs a) {
  const LoraDownJobDev J = select_down_job(a, blockIdx.z);
  if ((int)blockIdx.y >= J.n_split) return;
  lora_down_tile<T, RT, MTL, NW>(J.X, J.ldx, J.Wd, a.M, J.C, J.r, J.out, J.ldo, J.partial, J.n_split);
}

// ---- lora_down, a few hundred tokens ---------------------------------------------------------------------
// Between the few tokens of a generation step and the thousands that fill the chip by themselves, the fragment kernel above is
// bound by the address path of its loads: a fragment's four rows in every four lanes go one by one, 16 bytes per clock and CU,
// and every 16 tokens read all of Wd that way.  Here a workgroup owns 64 tokens and 64 ranks at most; its four waves take the
// 64-wide chunks of the columns in turn, each through LDS of its own (no barrier: direct loads of 8 rows x 128 bytes, slot s
// of row i holding the 16 bytes s ^ ((i >> 1) & 7), two chunks in flight), and their sums meet in LDS in wave order.  Columns are
// split over workgroups as in the kernels around it; ranks above 64 are further workgroups.
// LINES: rows begin on 128-byte lines, so a chunk's piece of a row is one line, read once and past the caches.  Other rows share
// their lines between neighbouring chunks, which come from L2 the second time (16383 tokens of 5464 columns, rank 32 / 64: 42.6 /
// 52.6 -> 30.7 / 35.6 us).
constexpr int LM_NW = 4, LM_MT = 4;  // waves; 16-token tiles
constexpr int lm_vmcnt(int n) { return (n & 0xF) | ((n >> 4) << 14) | 0x0F70; }  // s_waitcnt operand: vmcnt(n) only, n < 64

template <typename T, int RT, bool LINES>
__global__ __launch_bounds__(64 * LM_NW) void lora_down_mid_kernel(const LoraDownArgs a) {
  // one array per buffer, so that the compiler's wait counts tell reads of one from loads in flight into the other
  __shared__ __attribute__((aligned(1024))) uint16_t b0[LM_NW * (LM_MT + RT) * 1024];
  __shared__ __attribute__((aligned(1024))) uint16_t b1[LM_NW * (LM_MT + RT) * 1024];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 15, kq = lane >> 4;
  const int rank_blocks = (a.r_max + 63) / 64;
  const LoraDownJobDev J = select_down_job(a, blockIdx.z / rank_blocks);
  const int r0 = 64 * (blockIdx.z % rank_blocks);
  if ((int)blockIdx.y >= J.n_split || r0 >= J.r) return;
  const int m0 = blockIdx.x * (16 * LM_MT), C = J.C;
  const int rows = min(16 * LM_MT, a.M - m0), ranks = min(64, J.r - r0);
  const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(J.X + (size_t)m0 * J.ldx, (size_t)rows * J.ldx * 2);
  const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(J.Wd + (size_t)r0 * C, (size_t)ranks * C * 2);
  // the lane's 16 bytes of row 8 i + (lane >> 3): chunk piece (lane & 7) ^ ((row >> 1) & 7); rows 16 apart share it
  uint32_t x_off[2], w_off[2], piece[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = 8 * i + (lane >> 3);
    piece[i] = 8 * ((lane & 7) ^ ((row >> 1) & 7));
    x_off[i] = (uint32_t)((row * J.ldx + piece[i]) * 2);
    w_off[i] = (uint32_t)((row * (int64_t)C + piece[i]) * 2);
  }
  const uint32_t x_tile = (uint32_t)(16 * J.ldx * 2), w_tile = (uint32_t)(16 * (int64_t)C * 2);
  uint32_t frag[2];  // the lane's fragment of a tile's 32-wide half t
#pragma unroll
  for (int t = 0; t < 2; ++t) frag[t] = (uint32_t)(c * 128 + 16 * ((4 * t + kq) ^ ((c >> 1) & 7)));
  const int n_chunks = (C + 63) / 64, n_slices = J.n_split * LM_NW, slice = blockIdx.y * LM_NW + wave;
  const int n_it = (n_chunks + n_slices - 1) / n_slices;
  f32x4 acc[LM_MT][RT];
#pragma unroll
  for (int u = 0; u < LM_MT; ++u)
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  // columns past C (and chunks past the wave's last) are out of range by their lane offsets: zeros, and no traffic
  auto load = [&](int it, uint16_t* buf) {
    const int col = 64 * (slice + n_slices * it);
    char* dst = reinterpret_cast<char*>(buf) + wave * ((LM_MT + RT) * 2048);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t dead = col + (int)piece[i] < C ? 0u : 0x80000000u;
#pragma unroll
      for (int u = 0; u < LM_MT; ++u)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(x_rsrc, (__attribute__((address_space(3))) void*)(dst + u * 2048 + i * 1024), 16,
                                                 (x_off[i] + u * x_tile) | dead, (uint32_t)col * 2, 0, LINES ? 2 : 0);
#pragma unroll
      for (int t = 0; t < RT; ++t)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, (__attribute__((address_space(3))) void*)(dst + (LM_MT + t) * 2048 + i * 1024), 16,
                                                 (w_off[i] + t * w_tile) | dead, (uint32_t)col * 2, 0, 0);
    }
  };
  auto multiply = [&](const uint16_t* buf) {
    __builtin_amdgcn_s_waitcnt(lm_vmcnt(2 * (LM_MT + RT)));  // the other buffer's loads are younger
    __builtin_amdgcn_sched_barrier(0);
    const char* src = reinterpret_cast<const char*>(buf) + wave * ((LM_MT + RT) * 2048);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      u32x4 xf[LM_MT];
#pragma unroll
      for (int u = 0; u < LM_MT; ++u) xf[u] = *reinterpret_cast<const u32x4*>(src + u * 2048 + frag[h]);
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        const u32x4 wf = *reinterpret_cast<const u32x4*>(src + (LM_MT + t) * 2048 + frag[h]);
#pragma unroll
        for (int u = 0; u < LM_MT; ++u) acc[u][t] = mfma16<T>(xf[u], wf, acc[u][t]);  // D[i = token][j = rank]
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // the fragments have arrived before the buffer is loaded again
  };
  load(0, b0);
  __builtin_amdgcn_sched_barrier(0);  // the counted wait takes b1's loads to be younger, and the compiler knows of no order between them
  load(1, b1);
  for (int it = 0; it < n_it; it += 2) {
    multiply(b0);
    load(it + 2, b0);
    multiply(b1);
    load(it + 3, b1);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // the surplus direct loads, every wave's
  __syncthreads();
  float(*red)[LM_MT][RT][64][4] = reinterpret_cast<float(*)[LM_MT][RT][64][4]>(b0);
#pragma unroll
  for (int u = 0; u < LM_MT; ++u)
#pragma unroll
    for (int t = 0; t < RT; ++t) *reinterpret_cast<f32x4*>(red[wave][u][t][lane]) = acc[u][t];
  __syncthreads();
  // wave = token tile: lane holds D[4 kq + i][c] of every rank tile
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    f32x4 v = *reinterpret_cast<const f32x4*>(red[0][wave][t][lane]);
#pragma unroll
    for (int w = 1; w < LM_NW; ++w) v += *reinterpret_cast<const f32x4*>(red[w][wave][t][lane]);
    const int j = r0 + 16 * t + c;
    if (j >= J.r) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = m0 + 16 * wave + 4 * kq + i;
      if (m >= a.M) continue;
      if (J.partial)
        J.partial[((size_t)blockIdx.y * a.M + m) * J.r + j] = v[i];
      else
        J.out[(size_t)m * J.ldo + j] = pack1<T>(v[i]);
    }
  }
}
static_assert(LM_MT == LM_NW, "one token tile of the sums per wave");

// ---- lora_down, staged ----------------------------------------------------------------------------
// The same product for the large-M case, with X going through LDS: a direct load of one wave moves a
// whole 1 KB run of one row (512 columns), where the fragment loads above fetch 64 B of each of 16
// rows per instruction.  Workgroup = 32 tokens, 8 waves; a stage = 32 rows x 512 columns (32 KB) in
// one of four LDS buffers, so up to two stages are in flight while a third is multiplied.  Slot c of
// row m holds chunk c ^ (m & 15) of the row's run (the permutation is applied on the global side: a
// direct load writes lane p's 16 bytes to slot p), which spreads the 16 rows a fragment read touches
// over all banks.  Wave w multiplies columns 64w .. 64w+63 of every stage; its Wd fragments come
// straight from global (L2) one stage ahead.  Partial sums of the 8 waves are added as above.
template <typename T, int RT, int MTL>
__global__ __launch_bounds__(512) void lora_down_staged_kernel(const uint16_t* __restrict__ X, int64_t ldx,
                                                               const uint16_t* __restrict__ Wd, int M, int C, int r,
                                                               uint16_t* __restrict__ out, int64_t ldo) {
  constexpr int NW = 8, NH = 4, ROWS = 16 * MTL, SC = 512;  // a wave moves 2 * MTL rows per stage
  static_assert(RT <= 8 && (MTL == 1 || MTL == 2), "rank tiles are reduced four at a time through one stage buffer");
  // four separate arrays: every access names its buffer statically, so the compiler's wait counts
  // can tell reads of one buffer from direct loads in flight into the others
  __shared__ __attribute__((aligned(1024))) uint16_t s0[ROWS * SC];
  __shared__ __attribute__((aligned(1024))) uint16_t s1[ROWS * SC];
  __shared__ __attribute__((aligned(1024))) uint16_t s2[ROWS * SC];
  __shared__ __attribute__((aligned(1024))) uint16_t s3[ROWS * SC];
  auto buf = [&](auto b_c) -> char* {
    constexpr int b = decltype(b_c)::value;
    return reinterpret_cast<char*>(b == 0 ? s0 : (b == 1 ? s1 : (b == 2 ? s2 : s3)));
  };
  using B0 = std::integral_constant<int, 0>;
  using B1 = std::integral_constant<int, 1>;
  using B2 = std::integral_constant<int, 2>;
  using B3 = std::integral_constant<int, 3>;
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int uwave = __builtin_amdgcn_readfirstlane(wave);
  const int l16 = lane & 15, q = lane >> 4;
  const int m_base = blockIdx.x * ROWS;
  const int rows_valid = min(ROWS, M - m_base);
  const int n_stages = (C + SC - 1) / SC;
  const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(X + (size_t)m_base * ldx, (size_t)rows_valid * ldx * 2);
  const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(Wd, (size_t)r * C * 2);

  // direct loads: wave w moves rows RPW * w .. of a stage
  // (arrays of fixed size and the template parameter itself in the loops: a local constant that depends on MTL,
  // used inside the generic lambdas below, makes the host pass drop the kernel's stub without a diagnostic)
  uint32_t d_off[4], d_col[4];
#pragma unroll
  for (int i = 0; i < 2 * MTL; ++i) {
    const int row = 2 * MTL * wave + i;
    d_col[i] = 8 * (lane ^ (row & 15));
    d_off[i] = (uint32_t)((row * ldx + d_col[i]) * 2);
  }
  auto dma = [&](int st, auto b_c) {
#pragma unroll
    for (int i = 0; i < 2 * MTL; ++i) {
      const uint32_t dead = (st * SC + (int)d_col[i]) < C ? 0u : 0x80000000u;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(x_rsrc, (__attribute__((address_space(3))) void*)(buf(b_c) + (2 * MTL * uwave + i) * (SC * 2)),
                                               16, d_off[i] | dead, (uint32_t)st * (SC * 2), 0, 2);
    }
  };
  // Wd fragments of the wave's two 32-column steps of a stage
  uint32_t w_off[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) w_off[t] = (uint32_t)(((16 * t + l16) * (int64_t)C + 8 * q) * 2);
  auto wld = [&](int st, u32x4(&wf)[2][RT]) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int c0 = st * SC + 32 * (2 * wave + kk);
      const uint32_t dead = (c0 + 8 * q) < C ? 0u : 0x80000000u;
#pragma unroll
      for (int t = 0; t < RT; ++t) wf[kk][t] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, (w_off[t] + 2 * c0) | dead, 0, 0);
    }
  };
  f32x4 acc[MTL][RT];
#pragma unroll
  for (int u = 0; u < MTL; ++u)
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto mul = [&](auto b_c, const u32x4(&wf)[2][RT]) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int chunk = 4 * (2 * wave + kk) + q;
#pragma unroll
      for (int u = 0; u < MTL; ++u) {
        const u32x4 xf = *reinterpret_cast<const u32x4*>(buf(b_c) + (16 * u + l16) * (SC * 2) + ((chunk ^ l16) * 16));
#pragma unroll
        for (int t = 0; t < RT; ++t) acc[u][t] = mfma16<T>(xf, wf[kk][t], acc[u][t]);  // D[i = token][j = rank]
      }
    }
  };
  // s_waitcnt vmcnt(n) only (expcnt / lgkmcnt fields left at their maxima)
  constexpr int YOUNGER = 4 * MTL + 4 * RT;  // loads a wave issues after the direct loads of a stage and before that stage's turn
  constexpr int WAIT_STEADY = (YOUNGER & 0xF) | ((YOUNGER >> 4) << 14) | 0x0F70;
  constexpr int YOUNGER0 = 4 * MTL + 2 * RT;  // ... for stage 0 (prologue order)
  constexpr int WAIT_FIRST = (YOUNGER0 & 0xF) | ((YOUNGER0 >> 4) << 14) | 0x0F70;
  // one stage: its own direct loads have landed -> barrier (all waves' parts are there, and everybody has
  // left the buffer that is re-filled next) -> requests two and three stages ahead -> multiply
  u32x4 wa[2][RT], wb[2][RT];
  auto turn = [&](int st, auto cur_c, auto refill_c, const u32x4(&wcur)[2][RT], u32x4(&wnext)[2][RT]) {
    if (st == 0)
      __builtin_amdgcn_s_waitcnt(WAIT_FIRST);
    else
      __builtin_amdgcn_s_waitcnt(WAIT_STEADY);
    // a bare barrier: the fence of __syncthreads() would wait for ALL direct loads in flight (they
    // are stores to LDS), the two stages ahead included
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    wld(st + 1, wnext);
    dma(st + 3, refill_c);
    mul(cur_c, wcur);
  };
  dma(0, B0{});
  dma(1, B1{});
  dma(2, B2{});
  wld(0, wa);
  for (int st = 0; st < n_stages; st += 4) {
    turn(st, B0{}, B3{}, wa, wb);
    turn(st + 1, B1{}, B0{}, wb, wa);
    turn(st + 2, B2{}, B1{}, wa, wb);
    turn(st + 3, B3{}, B2{}, wb, wa);
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // the surplus direct loads (all lanes out of range) have landed too
  __syncthreads();

  // the waves' partial tiles are added through stage buffer 0, RC rank tiles at a time ([NH][MTL][RC] KB <= its size)
  constexpr int RC = RT < 4 ? RT : 4;
  float(*red)[MTL][RC][64][4] = reinterpret_cast<float(*)[MTL][RC][64][4]>(s0);
  static_for<0, RT / RC>([&](auto c_c) {
    constexpr int t0 = decltype(c_c)::value * RC;
    if (wave >= NH) {
#pragma unroll
      for (int u = 0; u < MTL; ++u)
#pragma unroll
        for (int t = 0; t < RC; ++t) *reinterpret_cast<f32x4*>(red[wave - NH][u][t][lane]) = acc[u][t0 + t];
    }
    __syncthreads();
    if (wave < NH) {
#pragma unroll
      for (int u = 0; u < MTL; ++u)
#pragma unroll
        for (int t = 0; t < RC; ++t) {
          const f32x4 o = *reinterpret_cast<const f32x4*>(red[wave][u][t][lane]);
          *reinterpret_cast<f32x4*>(red[wave][u][t][lane]) = acc[u][t0 + t] + o;
        }
    }
    __syncthreads();
    for (int o = tid; o < MTL * RC * 256; o += 64 * NW) {
      const int u = o / (RC * 256), t = (o >> 8) % RC, ln = (o >> 2) & 63, i = o & 3;
      float v = red[0][u][t][ln][i];
#pragma unroll
      for (int w = 1; w < NH; ++w) v += red[w][u][t][ln][i];
      const int row = m_base + 16 * u + 4 * (ln >> 4) + i;
      const int j = 16 * (t0 + t) + (ln & 15);
      if (row < M && j < r) out[(size_t)row * ldo + j] = pack1<T>(v);
    }
    if constexpr (t0 + RC < RT) __syncthreads();  // the next four rank tiles reuse the buffer
  });
}

// ---- lora_down, staged, many tokens per workgroup, columns split over workgroups ----------------------
// Every workgroup of the kernels above reads all of Wd, which at 16-32 tokens per workgroup is r / 16 .. r / 32 times
// the bytes of X it consumes: from rank 32 on the L2 traffic of Wd, not HBM, sets the pace.  Here a workgroup owns
// 32 * G tokens and one of `n_split` contiguous column ranges: the stages of a 512-column chunk are its G row groups one
// after the other, multiplied by the same Wd fragments (loaded once per chunk), so Wd is read once per 32 * G tokens;
// the column split gives the chip its workgroups back when M / (32 * G) falls short of the CUs.  With n_split > 1 the
// fp32 sums of the ranges go to partial[split][M][r] and lora_down_reduce_kernel adds them in index order (same result
// whatever the scheduling) and rounds once.  Stage buffers, swizzle and the waits are those of the kernel above.
template <typename T, int RT, int G>
__global__ __launch_bounds__(512) void lora_down_split_kernel(const uint16_t* __restrict__ X, int64_t ldx,
                                                              const uint16_t* __restrict__ Wd, int M, int C, int r,
                                                              uint16_t* __restrict__ out, int64_t ldo,
                                                              float* __restrict__ partial, int n_tb, int n_split) {
  constexpr int NW = 8, NH = 4, MTL = 2, ROWS = 32, SC = 512;
  static_assert(G == 2 || G == 4, "a chunk's row groups fill the four stage buffers a whole number of times");
  static_assert(G * MTL * RT <= 32, "accumulator registers");
  __shared__ __attribute__((aligned(1024))) uint16_t s0[ROWS * SC];
  __shared__ __attribute__((aligned(1024))) uint16_t s1[ROWS * SC];
  __shared__ __attribute__((aligned(1024))) uint16_t s2[ROWS * SC];
  __shared__ __attribute__((aligned(1024))) uint16_t s3[ROWS * SC];
  auto buf = [&](auto b_c) -> char* {
    constexpr int b = decltype(b_c)::value;
    return reinterpret_cast<char*>(b == 0 ? s0 : (b == 1 ? s1 : (b == 2 ? s2 : s3)));
  };
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int uwave = __builtin_amdgcn_readfirstlane(wave);
  const int l16 = lane & 15, q = lane >> 4;
  const int tb = blockIdx.x % n_tb, sp = blockIdx.x / n_tb;
  const int m_base = tb * (ROWS * G);
  const int rows_valid = min(ROWS * G, M - m_base);
  // this workgroup's chunks [ch_lo, ch_hi) of 512 columns
  const int n_chunks = (C + SC - 1) / SC;
  const int per = (n_chunks + n_split - 1) / n_split;
  const int ch_lo = min(n_chunks, sp * per), ch_hi = min(n_chunks, ch_lo + per);
  const int n_stages = (ch_hi - ch_lo) * G;
  const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(X + (size_t)m_base * ldx, (size_t)rows_valid * ldx * 2);
  const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(Wd, (size_t)r * C * 2);

  // direct loads: wave w moves rows 4 w .. 4 w + 3 of a stage (row group g of the workgroup's tokens)
  uint32_t d_off[4], d_col[4];
#pragma unroll
  for (int i = 0; i < 2 * MTL; ++i) {
    const int row = 2 * MTL * wave + i;
    d_col[i] = 8 * (lane ^ (row & 15));
    d_off[i] = (uint32_t)((row * ldx + d_col[i]) * 2);
  }
  const uint32_t group_bytes = (uint32_t)(ROWS * ldx * 2);
  // stage st = chunk ch_lo + st / G, row group st % G; stages past the last one load nothing (every lane out of range)
  auto dma = [&](int st, auto b_c) {
    const int ch = ch_lo + st / G, g = st % G;
#pragma unroll
    for (int i = 0; i < 2 * MTL; ++i) {
      const uint32_t dead = (ch < ch_hi && (ch * SC + (int)d_col[i]) < C) ? 0u : 0x80000000u;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(x_rsrc, (__attribute__((address_space(3))) void*)(buf(b_c) + (2 * MTL * uwave + i) * (SC * 2)),
                                               16, (d_off[i] + (uint32_t)g * group_bytes) | dead, (uint32_t)ch * (SC * 2), 0, 2);
    }
  };
  uint32_t w_off[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) w_off[t] = (uint32_t)(((16 * t + l16) * (int64_t)C + 8 * q) * 2);
  auto wld = [&](int ch, u32x4(&wf)[2][RT]) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int c0 = ch * SC + 32 * (2 * wave + kk);
      const uint32_t dead = (ch < ch_hi && (c0 + 8 * q) < C) ? 0u : 0x80000000u;
#pragma unroll
      for (int t = 0; t < RT; ++t) wf[kk][t] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, (w_off[t] + 2 * c0) | dead, 0, 0);
    }
  };
  f32x4 acc[G][MTL][RT];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int u = 0; u < MTL; ++u)
#pragma unroll
      for (int t = 0; t < RT; ++t) acc[g][u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto mul = [&](auto b_c, auto g_c, const u32x4(&wf)[2][RT]) {
    constexpr int g = decltype(g_c)::value;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int chunk = 4 * (2 * wave + kk) + q;
#pragma unroll
      for (int u = 0; u < MTL; ++u) {
        const u32x4 xf = *reinterpret_cast<const u32x4*>(buf(b_c) + (16 * u + l16) * (SC * 2) + ((chunk ^ l16) * 16));
#pragma unroll
        for (int t = 0; t < RT; ++t) acc[g][u][t] = mfma16<T>(xf, wf[kk][t], acc[g][u][t]);
      }
    }
  };
  // Loads a wave issues after the direct loads of stage st and before that stage's turn: the direct loads of the two
  // stages after it (2 x 4), and one batch of Wd fragments when turn st - 1 or st - 2 closed a chunk (g = 0 or 1).
  // A smaller count than the true one only waits longer, so the first turns use the same figures.
  auto wait_for = [&](auto g_c) {
    constexpr int g = decltype(g_c)::value;
    constexpr int YOUNGER = 4 * MTL + ((g == 0 || g == 1) ? 2 * RT : 0);
    __builtin_amdgcn_s_waitcnt((YOUNGER & 0xF) | ((YOUNGER >> 4) << 14) | 0x0F70);
  };
  u32x4 wa[2][RT], wb[2][RT];
  // turn st: its direct loads have landed -> barrier -> (last row group of a chunk: the next chunk's Wd fragments) ->
  // the direct loads three stages ahead -> multiply
  auto turn = [&](int st, auto cur_c, auto refill_c, auto g_c, const u32x4(&wcur)[2][RT], u32x4(&wnext)[2][RT]) {
    constexpr int g = decltype(g_c)::value;
    wait_for(g_c);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (g == G - 1) wld(ch_lo + st / G + 1, wnext);
    dma(st + 3, refill_c);
    mul(cur_c, g_c, wcur);
  };
  using B0 = std::integral_constant<int, 0>;
  using B1 = std::integral_constant<int, 1>;
  using B2 = std::integral_constant<int, 2>;
  using B3 = std::integral_constant<int, 3>;
  dma(0, B0{});
  dma(1, B1{});
  dma(2, B2{});
  wld(ch_lo, wa);
  if constexpr (G == 2) {
    for (int st = 0; st < n_stages; st += 4) {  // two chunks per round
      turn(st, B0{}, B3{}, B0{}, wa, wb);
      turn(st + 1, B1{}, B0{}, B1{}, wa, wb);
      turn(st + 2, B2{}, B1{}, B0{}, wb, wa);
      turn(st + 3, B3{}, B2{}, B1{}, wb, wa);
    }
  } else {
    for (int st = 0; st < n_stages; st += 8) {
      turn(st, B0{}, B3{}, B0{}, wa, wb);
      turn(st + 1, B1{}, B0{}, B1{}, wa, wb);
      turn(st + 2, B2{}, B1{}, B2{}, wa, wb);
      turn(st + 3, B3{}, B2{}, B3{}, wa, wb);
      turn(st + 4, B0{}, B3{}, B0{}, wb, wa);
      turn(st + 5, B1{}, B0{}, B1{}, wb, wa);
      turn(st + 6, B2{}, B1{}, B2{}, wb, wa);
      turn(st + 7, B3{}, B2{}, B3{}, wb, wa);
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);  // the surplus direct loads (all lanes out of range) have landed too
  __syncthreads();

  // the waves' partial tiles are added through stage buffer 0, one row group and RC rank tiles at a time
  constexpr int RC = RT < 4 ? RT : 4;
  float(*red)[MTL][RC][64][4] = reinterpret_cast<float(*)[MTL][RC][64][4]>(s0);
  float* const pdst = partial + (size_t)sp * M * r;
  static_for<0, G>([&](auto g_c) {
    constexpr int g = decltype(g_c)::value;
    static_for<0, RT / RC>([&](auto c_c) {
      constexpr int t0 = decltype(c_c)::value * RC;
      if (wave >= NH) {
#pragma unroll
        for (int u = 0; u < MTL; ++u)
#pragma unroll
          for (int t = 0; t < RC; ++t) *reinterpret_cast<f32x4*>(red[wave - NH][u][t][lane]) = acc[g][u][t0 + t];
      }
      __syncthreads();
      if (wave < NH) {
#pragma unroll
        for (int u = 0; u < MTL; ++u)
#pragma unroll
          for (int t = 0; t < RC; ++t) {
            const f32x4 o = *reinterpret_cast<const f32x4*>(red[wave][u][t][lane]);
            *reinterpret_cast<f32x4*>(red[wave][u][t][lane]) = acc[g][u][t0 + t] + o;
          }
      }
      __syncthreads();
      for (int o = tid; o < MTL * RC * 256; o += 64 * NW) {
        const int u = o / (RC * 256), t = (o >> 8) % RC, ln = (o >> 2) & 63, i = o & 3;
        float v = red[0][u][t][ln][i];
#pragma unroll
        for (int w = 1; w < NH; ++w) v += red[w][u][t][ln][i];
        const int row = m_base + ROWS * g + 16 * u + 4 * (ln >> 4) + i;
        const int j = 16 * (t0 + t) + (ln & 15);
        if (row < M && j < r) {
          if (n_split == 1)
            out[(size_t)row * ldo + j] = pack1<T>(v);
          else
            pdst[(size_t)row * r + j] = v;
        }
      }
      __syncthreads();  // the next tiles reuse the buffer
    });
  });
}

// out[m, j] = round(sum over splits, in index order, of partial[split][m][j]); r % 8 == 0: four ranks per thread
template <typename T>
FMSA_DEVI void lora_down_reduce(const float* __restrict__ partial, int n_split, int M, int r, uint16_t* __restrict__ out, int64_t ldo) {
  const int64_t q4 = (int64_t)blockIdx.x * 256 + threadIdx.x;  // quad of ranks
  const int per_row = r / 4;
  if (q4 >= (int64_t)M * per_row) return;
  const int m = (int)(q4 / per_row), j = 4 * (int)(q4 % per_row);
  const size_t plane = (size_t)M * r;
  f32x4 v = *reinterpret_cast<const f32x4*>(partial + (size_t)m * r + j);
#pragma unroll 8
  for (int s = 1; s < n_split; ++s) v += *reinterpret_cast<const f32x4*>(partial + s * plane + (size_t)m * r + j);
  u32x2 o;
  o[0] = pack2<T>(v[0], v[1]);
  o[1] = pack2<T>(v[2], v[3]);
  *reinterpret_cast<u32x2*>(out + (size_t)m * ldo + j) = o;
}

template <typename T>
__global__ __launch_bounds__(256) void lora_down_reduce_kernel(const float* __restrict__ partial, int n_split, int M, int r,
                                                               uint16_t* __restrict__ out, int64_t ldo) {
  lora_down_reduce<T>(partial, n_split, M, r, out, ldo);
}
template <typename T>
__global__ __launch_bounds__(256) void lora_down_reduce_batch_kernel(const LoraDownArgs a) {
  const LoraDownJobDev J = select_down_job(a, blockIdx.y);
  if (!J.partial) return;  // rounded by the first launch
  lora_down_reduce<T>(J.partial, J.n_split, a.M, J.r, J.out, J.ldo);
}

// ---- lora_grad ----------------------------------------------------------------------------------
// out[j, c] = sum_m L[m, j] * R[m, c]: the contraction runs over tokens, which is the row index of
// both row-major operands, so each MFMA fragment (8 consecutive contraction elements per lane) is a
// column walk.  Tiles of 32 tokens are staged through LDS (coalesced 16-byte global loads in, transposing
// 8-byte reads out: column_frag below); token e of a tile is the MFMA's contraction index e, rows are padded
// by 32 B.
// Pass 1: workgroup = 256 columns of R (eight waves) x one fixed range of tokens (split); wave w owns columns
// 32w .. 32w+31 (two 16-wide MFMA tiles) and all r ranks.  Partial sums go to partial[split][r][C]
// (fp32).  Pass 2 adds the splits in index order, so the result does not depend on scheduling.
constexpr int LG_TM = 32;               // tokens per tile
constexpr int LG_TC_T = 256;   // columns of R per workgroup (8 waves x 32)

// Several gradients over the same M tokens go out as ONE launch of each pass (the dA of stacked
// adapters and their dB's; a launch of a small gradient alone neither fills the chip nor hides its
// own start-up): workgroup ids are laid end to end over the jobs.
struct LoraGradJobDev {
  const uint16_t* L;
  const uint16_t* R;
  void* out;
  float* partial;  // [splits][r][C] of this job, or [splits][C][r] where the output is transposed
  int64_t ldl, ldr;
  int C, r, splits, rows_per_split;
  int block_start;   // first workgroup of the job in pass 1
  int rblock_start;  // ... in pass 2
  int transpose_out, out_dtype;
  float scale;
  int per_thread;  // elements of the output that a thread of pass 2 adds: 4 or 1
  // optional second product of the same pass over R: T[M, r] = R * Wt^T (see below)
  const uint16_t* Wt;  // [r, C]
  float* tpart;        // [column blocks][M][r]
  uint16_t* T;
  int64_t ldt;
};
struct LoraGradArgs {
  LoraGradJobDev j[FMSA_LORA_GRAD_MAX_JOBS];
  int n_jobs, M, act_dtype;
};
// the job that owns workgroup `block` (wave-uniform), copied field by field: indexing the
// kernel-argument struct with a runtime value would force a copy of it into scratch memory
template <bool REDUCE>
FMSA_DEVI LoraGradJobDev select_job(const LoraGradArgs& a, int block) {
  LoraGradJobDev J = a.j[0];
#pragma unroll
  for (int q = 1; q < FMSA_LORA_GRAD_MAX_JOBS; ++q)
    if (q < a.n_jobs && block >= (REDUCE ? a.j[q].rblock_start : a.j[q].block_start)) J = a.j[q];
  return J;
}

// WITH_T: a job with Wt set also produces T = R * Wt^T (the `dY @ B` every backward needs next to
// dB = s * dY^T U: both read dY, which is the whole cost of either).  The R tile is in LDS anyway, and
// row-major, which is the natural MFMA layout for a contraction over columns: wave w multiplies the
// tile's 32 tokens by its own 32 columns (2 * rt MFMAs per tile), the four waves' partial tiles meet in
// LDS and are summed in wave order by the whole workgroup one iteration later (behind the barrier the
// loop has anyway), and leave as the column block's partial T[column block][token][rank] (fp32).  The
// reduce pass adds the column blocks in index order and rounds once: deterministic like the rest.
// Eight waves and 256 columns per workgroup: the L tile every workgroup re-reads is r / 256 of the R bytes it consumes
// (a four-wave, 128-column workgroup measured slower at every rank: 44.6 vs 41.8 us over 235 MB at rank 16).
template <typename T, int RT, bool WITH_T>
__global__ __launch_bounds__(512) void lora_grad_partial_kernel(const LoraGradArgs a) {
  constexpr int NWV = 8;  // waves
  constexpr int NTH = 64 * NWV;             // threads
  constexpr int TC = 32 * NWV;              // columns of R per workgroup
  constexpr int LG_RSTRIDE = TC + 16;       // elements: row + 32 B pad
  constexpr int LSTRIDE = (RT == 1) ? 16 : RT * 16 + 16;  // elements; row pitch = 8 banks mod 32
  __shared__ __attribute__((aligned(16))) uint16_t r_lds[2][LG_TM * LG_RSTRIDE];
  __shared__ __attribute__((aligned(16))) uint16_t l_lds[2][LG_TM * LSTRIDE];
  __shared__ __attribute__((aligned(16))) float t_lds[WITH_T ? 2 : 1][WITH_T ? NWV : 1][2][WITH_T ? RT : 1][64][WITH_T ? 4 : 1];
  const LoraGradJobDev J = select_job<false>(a, blockIdx.x);
  const uint16_t* __restrict__ L = J.L;
  const uint16_t* __restrict__ R = J.R;
  float* __restrict__ partial = J.partial;
  const int64_t ldl = J.ldl, ldr = J.ldr;
  const int M = a.M, C = J.C, r = J.r, rows_per_split = J.rows_per_split;
  const int rt = (r + 15) / 16;  // 16-rank tiles this job uses of the RT the launch is built for
  const int ncb = (C + TC - 1) / TC;
  const int local = blockIdx.x - J.block_start;
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int l16 = lane & 15, kg = lane >> 4;
  const int split = local / ncb;
  const int c0 = (local % ncb) * TC;
  const int m_begin = split * rows_per_split;
  const int m_end = min(M, m_begin + rows_per_split);
  const int n_tiles = (m_end - m_begin + LG_TM - 1) / LG_TM;

  // global -> LDS assignment: R tile = 32 rows x TC/8 chunks of 16 B -> 2 chunks per thread (16 rows per pass);
  // L tile = 32 rows x (RT*2) chunks = 64*RT chunks -> LP per thread (chunk tid + NTH*p), threads
  // past the last chunk idle
  const int r_row = tid / (TC / 8), r_chunk = tid % (TC / 8);
  const bool r_col_ok = (c0 + 8 * r_chunk) < C;  // C % 8 == 0
  constexpr int LP = (64 * RT + NTH - 1) / NTH;
  int l_row[LP], l_chunk[LP];
  bool l_thread[LP], l_col_ok[LP];
#pragma unroll
  for (int p = 0; p < LP; ++p) {
    const int ci = tid + NTH * p;
    l_row[p] = ci / (2 * RT);
    l_chunk[p] = ci % (2 * RT);
    l_thread[p] = ci < 64 * RT;
    l_col_ok[p] = 8 * l_chunk[p] < r;  // r % 8 == 0
  }

  u32x4 rst[2], lst[LP];
  auto load_tile = [&](int tile) {
    const int m0 = m_begin + tile * LG_TM;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int m = m0 + r_row + 16 * p;
      rst[p] = u32x4{0u, 0u, 0u, 0u};
      if (m < m_end && r_col_ok) rst[p] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(R + (size_t)m * ldr + c0 + 8 * r_chunk));
    }
#pragma unroll
    for (int p = 0; p < LP; ++p) {
      lst[p] = u32x4{0u, 0u, 0u, 0u};
      const int m = m0 + l_row[p];
      if (l_thread[p] && m < m_end && l_col_ok[p]) lst[p] = *reinterpret_cast<const u32x4*>(L + (size_t)m * ldl + 8 * l_chunk[p]);
    }
  };
  auto commit_tile = [&](int buf) {
#pragma unroll
    for (int p = 0; p < 2; ++p)
      *reinterpret_cast<u32x4*>(&r_lds[buf][(r_row + 16 * p) * LG_RSTRIDE + 8 * r_chunk]) = rst[p];
#pragma unroll
    for (int p = 0; p < LP; ++p)
      if (l_thread[p]) *reinterpret_cast<u32x4*>(&l_lds[buf][l_row[p] * LSTRIDE + 8 * l_chunk[p]]) = lst[p];
  };
  // The MFMA operand of a 16-column tile starting at column `col0`: lane 16 kg + m gets column col0 + m at the 8 tokens
  // 8 kg .. 8 kg + 7 (contraction index k = 8 kg + e <-> token 8 kg + e of the tile).  Two transposing LDS reads
  // (ds_read_b64_tr_b16) do it: in a group of 16 lanes, lane 4 a + b receives element b of the four 16-bit values that
  // lanes a, a + 4, a + 8, a + 12 address, so lane j of the group addresses token 8 kg + 4 h + j / 4, columns
  // col0 + 4 (j % 4) .. + 3 (h = 0, 1: the two reads).  Was eight 16-bit reads and their packing per operand.
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  auto column_frag = [&](const uint16_t* base, int stride, int col0) {
    const uint16_t* p = base + (8 * kg + (l16 >> 2)) * stride + col0 + 4 * (l16 & 3);
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p + 4 * stride));
    const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
    return u32x4{l2[0], l2[1], h2[0], h2[1]};
  };

  f32x4 acc[2][RT];
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[g][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  // T product: this lane's Wt fragments (rank 16t + l16, columns c0 + 32*wave + 8*kg ..), fixed for the workgroup
  const bool with_t = WITH_T && J.Wt != nullptr;
  u32x4 wtf[RT];
  if constexpr (WITH_T) {
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      wtf[t] = u32x4{0u, 0u, 0u, 0u};
      const int j = 16 * t + l16, c = c0 + 32 * wave + 8 * kg;
      if (with_t && j < r && c < C) wtf[t] = *reinterpret_cast<const u32x4*>(J.Wt + (size_t)j * C + c);
    }
  }
  // sums the four waves' partial T tiles of token tile `tile` (parked in t_lds[tile & 1]) and stores them
  auto flush_t = [&](int tile) {
    if constexpr (WITH_T) {
      if (!with_t) return;
      const int tb = tile & 1;
      const int m0 = m_begin + tile * LG_TM;
      float* dst = J.tpart + ((size_t)(local % ncb) * M) * r;
      for (int v = tid; v < LG_TM * 16 * RT; v += NTH) {
        const int j = v % (16 * RT), m = v / (16 * RT);
        const int u = m >> 4, ln = ((m & 15) >> 2) * 16 + (j & 15), i = m & 3, t = j >> 4;
        float sum = t_lds[tb][0][u][t][ln][i];
#pragma unroll
        for (int w = 1; w < NWV; ++w) sum += t_lds[tb][w][u][t][ln][i];
        if (m0 + m < m_end && j < r) dst[(size_t)(m0 + m) * r + j] = sum;
      }
    }
  };

  if (n_tiles > 0) {
    load_tile(0);
    commit_tile(0);
  }
  __syncthreads();
  for (int tile = 0; tile < n_tiles; ++tile) {
    const int buf = tile & 1;
    if (tile + 1 < n_tiles) load_tile(tile + 1);
    if (tile > 0) flush_t(tile - 1);
    if constexpr (WITH_T) {
      if (with_t) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const u32x4 yf = *reinterpret_cast<const u32x4*>(&r_lds[buf][(16 * u + l16) * LG_RSTRIDE + 32 * wave + 8 * kg]);
#pragma unroll
          for (int t = 0; t < RT; ++t)
            if (t < rt)
              *reinterpret_cast<f32x4*>(t_lds[buf][wave][u][t][lane]) = mfma16<T>(yf, wtf[t], f32x4{0.f, 0.f, 0.f, 0.f});  // D[token][rank]
        }
      }
    }
    u32x4 lf[RT], rf[2];
#pragma unroll
    for (int t = 0; t < RT; ++t)
      if (t < rt) lf[t] = column_frag(l_lds[buf], LSTRIDE, 16 * t);
#pragma unroll
    for (int g = 0; g < 2; ++g) rf[g] = column_frag(r_lds[buf], LG_RSTRIDE, 32 * wave + 16 * g);
#pragma unroll
    for (int t = 0; t < RT; ++t)
      if (t < rt) {
#pragma unroll
        for (int g = 0; g < 2; ++g) acc[g][t] = mfma16<T>(rf[g], lf[t], acc[g][t]);  // D[c][j]
      }
    if (tile + 1 < n_tiles) commit_tile(buf ^ 1);
    __syncthreads();
  }
  if (n_tiles > 0) flush_t(n_tiles - 1);
  // lane holds D[c = 4*kg + i][j = l16]: four consecutive columns -> one 16-byte store, or, for a transposed output, its
  // rank of four columns (16 lanes: 64 bytes of a column's row of ranks)
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const int c = c0 + 32 * wave + 16 * g + 4 * kg;
    if (c >= C) continue;  // C % 8 == 0: the four columns are inside
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      const int j = 16 * t + l16;
      if (j >= r) continue;
      if (J.transpose_out) {
#pragma unroll
        for (int i = 0; i < 4; ++i) partial[((size_t)split * C + c + i) * r + j] = acc[g][t][i];
      } else {
        *reinterpret_cast<f32x4*>(partial + ((size_t)split * r + j) * C + c) = acc[g][t];
      }
    }
  }
}

// Four elements of a gradient from `at` on
FMSA_DEVI void grad_store4(const LoraGradJobDev& J, size_t at, f32x4 v) {
  v *= J.scale;
  const bool aligned = reinterpret_cast<uintptr_t>(J.out) % 16 == 0;
  if (J.out_dtype == FMSA_F32) {
    float* out = reinterpret_cast<float*>(J.out) + at;
    if (aligned) {
      *reinterpret_cast<f32x4*>(out) = v;
    } else {
      for (int i = 0; i < 4; ++i) out[i] = v[i];
    }
  } else {
    uint16_t* out = reinterpret_cast<uint16_t*>(J.out) + at;
    const u32x2 o = J.out_dtype == FMSA_BF16 ? u32x2{pack2<bf16_t>(v[0], v[1]), pack2<bf16_t>(v[2], v[3])}
                                             : u32x2{pack2<f16_t>(v[0], v[1]), pack2<f16_t>(v[2], v[3])};
    if (aligned) {
      *reinterpret_cast<u32x2*>(out) = o;
    } else {
      for (int i = 0; i < 4; ++i) out[i] = (uint16_t)(o[i >> 1] >> (16 * (i & 1)));
    }
  }
}

// The sums of a job's splits, in the output's order (which the partial sums are in too), V elements a thread: four, whose loads
// are whole lines (the transposed outputs were written 4 bytes at a time, r elements apart, 10.5 us where the sums of q, k, v at
// rank 64 and 1100 tokens take 6), or one, of straight outputs in launches that four leave short of workgroups (below).
template <int V> FMSA_DEVI void grad_reduce(const LoraGradJobDev& J, int idx) {
  using fv = std::conditional_t<V == 4, f32x4, float>;
  const float* src = J.partial + idx;
  const size_t step = (size_t)J.r * J.C;
  fv v{};
  int sp = 0;
  for (; sp + 8 <= J.splits; sp += 8) {  // eight loads in flight, summed in index order
    fv p[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) p[k] = *reinterpret_cast<const fv*>(src + (size_t)(sp + k) * step);
#pragma unroll
    for (int k = 0; k < 8; ++k) v += p[k];
  }
#pragma unroll 4
  for (; sp < J.splits; ++sp) v += *reinterpret_cast<const fv*>(src + (size_t)sp * step);
  if constexpr (V == 1) {
    v *= J.scale;
    if (J.out_dtype == FMSA_F32) reinterpret_cast<float*>(J.out)[idx] = v;
    else reinterpret_cast<uint16_t*>(J.out)[idx] = J.out_dtype == FMSA_BF16 ? pack1<bf16_t>(v) : pack1<f16_t>(v);
  } else {
    grad_store4(J, idx, v);
  }
}

__global__ __launch_bounds__(256) void lora_grad_reduce_kernel(const LoraGradArgs a) {
  const LoraGradJobDev J = select_job<true>(a, blockIdx.x);
  const int r = J.r, C = J.C;
  const int nb_grad = (r * C / J.per_thread + 255) / 256;
  const int lb = blockIdx.x - J.rblock_start;
  if (lb >= nb_grad) {  // the job's T: column blocks added in index order, one rounding; four ranks per thread
    const int64_t ti = ((int64_t)(lb - nb_grad) * 256 + threadIdx.x) * 4;
    if (ti >= (int64_t)a.M * r) return;  // r % 8 == 0: the four stay inside one token's row
    const int m = (int)(ti / r), j = (int)(ti % r);
    const int ncb = (C + LG_TC_T - 1) / LG_TC_T;
    // eight loads in flight per thread (a plain loop waits for each load before it issues the next); the sum
    // itself stays in index order
    const float* src = J.tpart + (size_t)m * r + j;
    const size_t step = (size_t)a.M * r;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    int cb = 0;
    for (; cb + 8 <= ncb; cb += 8) {
      f32x4 p[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) p[k] = *reinterpret_cast<const f32x4*>(src + (size_t)(cb + k) * step);
#pragma unroll
      for (int k = 0; k < 8; ++k) v += p[k];
    }
    for (; cb < ncb; ++cb) v += *reinterpret_cast<const f32x4*>(src + (size_t)cb * step);
    u32x2 pk;
    pk[0] = a.act_dtype == FMSA_BF16 ? pack2<bf16_t>(v[0], v[1]) : pack2<f16_t>(v[0], v[1]);
    pk[1] = a.act_dtype == FMSA_BF16 ? pack2<bf16_t>(v[2], v[3]) : pack2<f16_t>(v[2], v[3]);
    *reinterpret_cast<u32x2*>(J.T + (size_t)m * J.ldt + j) = pk;
    return;
  }
  const int at = lb * 256 + threadIdx.x;
  if (J.per_thread == 4) {
    if (4 * at < r * C) grad_reduce<4>(J, 4 * at);
  } else if (at < r * C) {
    grad_reduce<1>(J, at);
  }
}

// The same gradients in one launch: workgroup = 64 columns of R, its eight waves share the tokens (wave w takes tiles w, w + 8, ..),
// every wave stages its own tiles through its own part of LDS, and the waves' sums meet there in wave order, so nothing goes
// through memory and nothing is waited for but a wave's own loads.  The two-pass kernel above gives a gradient of few tokens one
// workgroup for 256 columns, which walks the tokens tile after tile (2048 columns: 8 workgroups), and a second launch.
constexpr int LGW_WAVES = 8;
constexpr int LGW_COLS = 64;
constexpr int LGW_RSTRIDE = LGW_COLS + 16;  // elements
constexpr int LGW_SUM = LGW_COLS + 4;       // floats: a rank's row of sums
template <int RT> constexpr int lgw_lstride() { return RT == 1 ? 16 : RT * 16 + 16; }
template <int RT> constexpr int lgw_round() { return RT < 2 ? 1 : 2; }  // 16-rank tiles summed at a time
template <int RT> constexpr int lgw_lds() {
  constexpr int stage = LGW_WAVES * LG_TM * (LGW_RSTRIDE + lgw_lstride<RT>()) * 2, sums = LGW_WAVES * lgw_round<RT>() * 16 * LGW_SUM * 4;
  return stage > sums ? stage : sums;
}

template <typename T, int RT>
__global__ __launch_bounds__(64 * LGW_WAVES) void lora_grad_waves_kernel(const LoraGradArgs a) {
  constexpr int LSTRIDE = lgw_lstride<RT>(), ROUND = lgw_round<RT>(), G = LGW_COLS / 16;
  __shared__ __attribute__((aligned(16))) char lds[lgw_lds<RT>()];
  const LoraGradJobDev J = select_job<false>(a, blockIdx.x);
  const int M = a.M, C = J.C, r = J.r, rt = (r + 15) / 16;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l16 = lane & 15, kg = lane >> 4;
  const int c0 = (blockIdx.x - J.block_start) * LGW_COLS;
  const int n_tiles = (M + LG_TM - 1) / LG_TM;
  uint16_t* r_lds = reinterpret_cast<uint16_t*>(lds) + wave * LG_TM * (LGW_RSTRIDE + LSTRIDE);
  uint16_t* l_lds = r_lds + LG_TM * LGW_RSTRIDE;
  // R tile: 32 rows x 8 chunks of 16 B, 4 a lane (8 rows a pass: whole lines); L tile: 32 rows x 2 RT chunks, RT a lane
  const int r_row = lane >> 3, r_chunk = lane & 7;
  const bool r_ok = c0 + 8 * r_chunk < C;  // C % 8 == 0
  u32x4 rst[4], lst[RT];
  auto load_tile = [&](int tile) {
    const int m0 = tile * LG_TM;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int m = m0 + r_row + 8 * p;
      rst[p] = u32x4{0u, 0u, 0u, 0u};
      if (m < M && r_ok) rst[p] = *reinterpret_cast<const u32x4*>(J.R + (size_t)m * J.ldr + c0 + 8 * r_chunk);
    }
#pragma unroll
    for (int p = 0; p < RT; ++p) {
      const int ci = lane + 64 * p, row = ci / (2 * RT), chunk = ci % (2 * RT), m = m0 + row;
      lst[p] = u32x4{0u, 0u, 0u, 0u};
      if (m < M && 8 * chunk < r) lst[p] = *reinterpret_cast<const u32x4*>(J.L + (size_t)m * J.ldl + 8 * chunk);  // r % 8 == 0
    }
  };
  // a wave's own stage: its lanes exchange data, so neither side of a fence moves past it
  auto own_stage_fence = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  auto column_frag = [&](const uint16_t* base, int stride, int col0) {  // as in the kernel above
    const uint16_t* p = base + (8 * kg + (l16 >> 2)) * stride + col0 + 4 * (l16 & 3);
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p + 4 * stride));
    const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
    return u32x4{l2[0], l2[1], h2[0], h2[1]};
  };
  f32x4 acc[G][RT];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[g][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (wave < n_tiles) load_tile(wave);
  for (int tile = wave; tile < n_tiles; tile += LGW_WAVES) {
    own_stage_fence();
#pragma unroll
    for (int p = 0; p < 4; ++p) *reinterpret_cast<u32x4*>(r_lds + (r_row + 8 * p) * LGW_RSTRIDE + 8 * r_chunk) = rst[p];
#pragma unroll
    for (int p = 0; p < RT; ++p) {
      const int ci = lane + 64 * p;
      *reinterpret_cast<u32x4*>(l_lds + ci / (2 * RT) * LSTRIDE + 8 * (ci % (2 * RT))) = lst[p];
    }
    own_stage_fence();
    if (tile + LGW_WAVES < n_tiles) load_tile(tile + LGW_WAVES);
    u32x4 rf[G];
#pragma unroll
    for (int g = 0; g < G; ++g) rf[g] = column_frag(r_lds, LGW_RSTRIDE, 16 * g);
#pragma unroll
    for (int t = 0; t < RT; ++t)
      if (t < rt) {
        const u32x4 lf = column_frag(l_lds, LSTRIDE, 16 * t);
#pragma unroll
        for (int g = 0; g < G; ++g) acc[g][t] = mfma16<T>(rf[g], lf, acc[g][t]);  // D[c][j]
      }
  }
  // ROUND rank tiles at a time: every wave's sums to LDS (rank-major), added in wave order, scaled, rounded once and stored
  float* sums = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int t0 = 0; t0 < RT; t0 += ROUND) {
    if (t0 >= rt) break;
    __syncthreads();
#pragma unroll
    for (int t = 0; t < ROUND; ++t)
#pragma unroll
      for (int g = 0; g < G; ++g)
        *reinterpret_cast<f32x4*>(sums + ((wave * ROUND + t) * 16 + l16) * LGW_SUM + 16 * g + 4 * kg) = acc[g][t0 + t];
    __syncthreads();
    // four columns of a rank, or, for a transposed output, four ranks of a column
    const int quads = ROUND * 16 * LGW_COLS / 4;
    if (tid < quads) {
      const bool tr = J.transpose_out;
      const int j = tr ? 4 * (tid % (ROUND * 4)) : tid / (LGW_COLS / 4), c = tr ? tid / (ROUND * 4) : 4 * (tid % (LGW_COLS / 4));
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < LGW_WAVES; ++w) {
        const float* src = sums + (w * ROUND * 16 + j) * LGW_SUM + c;
        v += tr ? f32x4{src[0], src[LGW_SUM], src[2 * LGW_SUM], src[3 * LGW_SUM]} : *reinterpret_cast<const f32x4*>(src);
      }
      const int jr = 16 * t0 + j;
      if (c0 + c < C && jr < r) grad_store4(J, tr ? (size_t)(c0 + c) * r + jr : (size_t)jr * C + c0 + c, v);
    }
  }
}

}  // namespace

int lora_grad_splits(int M, int C) {
  const int ncb = (C + LG_TC_T - 1) / LG_TC_T;
  // about two 512-thread workgroups per CU (16 waves), but at least 512 tokens (16 tiles) per split: shorter
  // splits spend their time in the prologue and in writing / re-reading partial sums.  (The count equals what
  // 1024 / number of 128-column blocks gave for widths that are multiples of 256; part of the workspace contract.)
  int splits = 512 / ncb;
  const int max_splits = (M + 511) / 512;
  if (splits > max_splits) splits = max_splits;
  if (splits < 1) splits = 1;
  return splits;
}

// n_split > 1: the fragment kernel with its columns split over workgroups, sums to `partial` (the caller reduces them)
static int launch_lora_down_plain(const void* X, int64_t ldx, const void* Wd, int M, int C, int r, int act_dtype, void* out,
                                  int64_t ldo, float* partial, int n_split, hipStream_t st) {
  // 32 tokens per workgroup once that still leaves a workgroup per CU (halves the re-reads of Wd)
  const int mtl = (M >= 32 * 256 && r <= 64) ? 2 : 1;
  constexpr int NW = 8;  // waves per workgroup: measured best of 4 / 8 / 16 at 8192 tokens
  dim3 grid((M + 16 * mtl - 1) / (16 * mtl), n_split), block(64 * NW);
  const int rt = (r + 15) / 16;
  // staged kernel: 32 (from 8192 tokens) or 16 (from 4096) tokens per workgroup, worth it once that gives every CU a
  // workgroup and the rows are long enough to amortise its pipeline fill (measured at 8192 tokens: 59 -> 48 us at
  // C = 14336, r = 16; 32 -> 28 us at C = 4096, r = 48; 20 -> 21 us at C = 4096, r = 16; at 4096 tokens, C = 28672,
  // r = 64: 205 us with the fragment loads above)
  // (the staged kernel walks all columns: it leaves no partial sums)
  const bool staged = n_split == 1 && M >= 16 * 256 && rt <= 8 && (C >= 8192 || (rt >= 2 && C >= 2048));
  if (staged) {
    const int smtl = M >= 32 * 256 ? 2 : 1;
    dim3 sgrid((M + 16 * smtl - 1) / (16 * smtl)), sblock(512);
#define SLAUNCH(TT, RT)                                                                                                           \
  do {                                                                                                                            \
    if (smtl == 2)                                                                                                                \
      hipLaunchKernelGGL((lora_down_staged_kernel<TT, RT, 2>), sgrid, sblock, 0, st, (const uint16_t*)X, ldx, (const uint16_t*)Wd, \
                         M, C, r, (uint16_t*)out, ldo);                                                                           \
    else                                                                                                                          \
      hipLaunchKernelGGL((lora_down_staged_kernel<TT, RT, 1>), sgrid, sblock, 0, st, (const uint16_t*)X, ldx, (const uint16_t*)Wd, \
                         M, C, r, (uint16_t*)out, ldo);                                                                           \
  } while (0)
#define SDISPATCH(TT)                        \
  switch (rt) {                              \
    case 1: SLAUNCH(TT, 1); break;           \
    case 2: SLAUNCH(TT, 2); break;           \
    case 3: case 4: SLAUNCH(TT, 4); break;   \
    default: SLAUNCH(TT, 8); break;          \
  }
    if (act_dtype == FMSA_BF16) {
      SDISPATCH(bf16_t)
    } else {
      SDISPATCH(f16_t)
    }
#undef SDISPATCH
#undef SLAUNCH
    FMSA_CHECK_LAUNCH();
    return FMSA_OK;
  }
#define LAUNCH(TT, RT)                                                                                                       \
  do {                                                                                                                       \
    if (mtl == 2)                                                                                                            \
      hipLaunchKernelGGL((lora_down_kernel<TT, RT, (RT > 4 ? 1 : 2), NW>), grid, block, 0, st, (const uint16_t*)X, ldx,       \
                         (const uint16_t*)Wd, M, C, r, (uint16_t*)out, ldo, partial);                                        \
    else                                                                                                                     \
      hipLaunchKernelGGL((lora_down_kernel<TT, RT, 1, NW>), grid, block, 0, st, (const uint16_t*)X, ldx, (const uint16_t*)Wd, \
                         M, C, r, (uint16_t*)out, ldo, partial);                                                             \
  } while (0)
#define DISPATCH(TT)            \
  switch (rt) {                 \
    case 1: LAUNCH(TT, 1); break; \
    case 2: LAUNCH(TT, 2); break; \
    case 3: case 4: LAUNCH(TT, 4); break; \
    default: LAUNCH(TT, 8); break; \
  }
  if (act_dtype == FMSA_BF16) {
    DISPATCH(bf16_t)
  } else {
    DISPATCH(f16_t)
  }
#undef DISPATCH
#undef LAUNCH
  FMSA_CHECK_LAUNCH();
  return FMSA_OK;
}

// Whether products over M tokens take the kernel of 64-token workgroups: `columns` in all, of one product (`single`) or of a batch;
// `lines`: every product's columns are whole 128-byte lines, and so, as a rule, its rows (the size query knows no strides).  us with
// the other kernels / with it, over 5100 forms of one product and 1900 of batches:
//
// Below 2048 tokens from the traffic on that the fragment kernel's loads are bound by, X and the re-reads of Wd.
//   rank 8, half of whose tile the fragment kernel does not read: 22 MB up to 8192 columns (4096 at 1300 tokens, 21 MB, 7.8 / 8.6;
//     5120 at 1536, 31 MB, 9.5 / 8.2), 52 MB above (8192 at 1300, 43 MB, 11.1 / 11.8; 14336 at 1100, 63 MB, 13.8 / 12.0), a batch
//     35 MB (q, k, v of 4096 and 1024 at 1300, 32 MB, 9.8 / 10.8, at 1536, 38 MB, 14.7 / 11.4); 14 MB where rows are no whole lines,
//     which the fragment kernel reads worst (8224 at 900, 30 MB, 11.0 / 7.3)
//   rank 16: 15 MB (4096 at 900, 15 MB, 8.0 / 8.6; 8192 at 512, 17 MB, 8.9 / 7.0)
//   rank 32: 18 MB, a batch 14 (11008 at 256, 17 MB, 9.0 / 9.9; 4096 at 1100, 27 MB, 10.4 / 9.0; q, k, v at 512, rank 24, 16 MB, 10.1 /
//     9.3)
//   rank 64: 22 MB (1100 tokens of 2048, 23 MB, 10.0 / 9.2), 33 where rows are no whole lines (5472 twice at 200, 26 MB, 8.7 / 9.8),
//     34 for a product of up to 512 tokens, whose column ranges fill the chip evenly (8192 at 384, 31 MB, 10.2 / 11.4; 11008 at 320,
//     35 MB, 13.3 / 11.9)
//   rank 96: 24 MB, a batch 18 (1056 at 1300, 19 MB, 8.3 / 9.2; q, k, v at 256, 22 MB, 13.9 / 10.6)
//   above, always: its eight rank tiles are one long chain there (1024 columns at 65 tokens 8.8 / 7.7, gate and up at 2047 131 / 48)
//
// From 2048 tokens and columns on (below, 1024 columns at 3000 tokens 7.5 / 9.9) against the staged kernels of 64 tokens up to rank
// 32 and 128 above, whose workgroups run one to a CU and are at their best where their ranges make one even round.
//   up to rank 16: long rows of less than 4096 tokens, where they need a second round (14336 at 3217 26 / 20, 28672 at 2500 42 / 29;
//     one round: 14336 at 4095 23 / 28, 8192 at 2048 10.1 / 10.6), and a good part of it where rows are no whole lines (10976 at 2300,
//     288 workgroups, 17.5 / 15.5, at 2800, 264, 15.2 / 16.1)
//   rank 32: all (2048 at 8192 11.0 / 10.4, 14336 at 3217 31 / 21) but 8192 at 16384, one round, 51 / 55
//   rank 64: all (4096 at 8192 25 / 20, 28672 at 7000 115 / 93) but long rows where the others have one round (28672 at 8192 95 / 98)
//     and the longest of the most tokens (14336 at 16384 94 / 102, 11008 at 16383 92 / 78)
//   rank 32 and 64, rows that are no whole lines: up to 140 M elements (7200 at 12000 68 / 39, at 20000 87 / 98; 10976 at 16384 63 / 71),
//     but not the 8192 columns and a few that leave most waves a step of nothing (8224 at 3500 tokens, rank 32, 18 / 22, at 7000, rank
//     64, 36 / 43)
//   above: all (14336 at 4096 81 / 46, 28672 at 8192 194 / 165) but the longest of the most tokens (14336 at 16383 186 / 197)
// Short rows of many tokens at rank 16 and below (4096 at 16384: 39 / 26) would need a buffer that the size query does not ask for.
static int staged_workgroups(int M, int64_t columns, int r);
static bool down_is_mid(int M, int r_max, int64_t columns, bool lines, bool single) {
  if (M <= 64) return false;  // few tokens: the ranges of the products straight from the parameters are the fragment kernel's
  if (M >= 2048) {
    if (columns < 2048) return false;
    const bool wide = columns >= 8192, many = M > 127 * 128;
    const int64_t elements = M * columns;
    if (r_max <= 16) return wide && M < 4096 && (lines || columns >= 9216) && staged_workgroups(M, columns, r_max) > (lines ? 256 : 280);
    if (lines) {
      if (r_max <= 32) return !(many && wide && columns < 11008);
      if (many && columns >= 12800) return false;
      return r_max > 64 || elements < 200000000 || staged_workgroups(M, columns, r_max) != 256;
    }
    if (r_max > 64) return !(many && columns >= 9216);
    return elements < 140000000 && !(wide && columns < 9216 && M < 9000 && (r_max <= 32 || M >= 5000));
  }
  const int64_t bytes = (int64_t)((M + 15) / 16) * (16 + std::max(16, r_max)) * columns * 2;
  if (r_max > 96) return true;
  if (r_max > 64) return bytes >= (single ? 24000000 : 18000000);
  if (r_max > 32) return bytes >= (single && M <= 512 ? 34000000 : (lines ? 22000000 : 33000000));
  if (r_max > 16) return bytes >= (single ? 18000000 : 14000000);
  if (r_max > 8) return bytes >= 15000000;
  if (!lines) return bytes >= 14000000;
  return bytes >= (!single ? 35000000 : (columns < 8192 ? 22000000 : 52000000));
}
static bool down_is_mid(int M, int C, int r) { return down_is_mid(M, r, C, C % 64 == 0, true); }
// column ranges: a step of two chunks of 64 columns a wave, the last range shorter (rounded down, 1056 columns took every wave two
// steps; rank 128 at 128 tokens 9.7 -> 8.7 us), and no more workgroups than run at once (one per CU, two up to rank 16)
static int down_mid_split(int M, int C, int r_max, int blocks_per_row) {
  const int blocks = ((M + 16 * LM_MT - 1) / (16 * LM_MT)) * blocks_per_row, slots = r_max <= 16 ? 512 : 256;
  return std::max(1, std::min(slots / blocks, ((C + 63) / 64 + 2 * LM_NW - 1) / (2 * LM_NW)));
}
static int rank_blocks(int r) { return (r + 63) / 64; }

static int launch_down_mid(LoraDownArgs& a, int n_jobs, int act_dtype, hipStream_t st) {
  int split_max = 1, r_max = 0;
  bool sums = false, lines = true;
  for (int q = 0; q < n_jobs; ++q) {
    lines = lines && a.j[q].ldx % 64 == 0 && reinterpret_cast<uintptr_t>(a.j[q].X) % 128 == 0;
    if (a.j[q].n_split == 1) a.j[q].partial = nullptr;
    sums = sums || a.j[q].partial;
    split_max = std::max(split_max, a.j[q].n_split);
    r_max = std::max(r_max, a.j[q].r);
  }
  a.r_max = r_max;
  const dim3 grid((a.M + 16 * LM_MT - 1) / (16 * LM_MT), split_max, n_jobs * rank_blocks(r_max)), block(64 * LM_NW);
  const dim3 rgrid((unsigned)(((int64_t)a.M * (r_max / 4) + 255) / 256), n_jobs);
  const int rt = (std::min(r_max, 64) + 15) / 16;
#define MID_RT(TT, RT)                                                                                       \
  do {                                                                                                       \
    if (lines) hipLaunchKernelGGL((lora_down_mid_kernel<TT, RT, true>), grid, block, 0, st, a);               \
    else hipLaunchKernelGGL((lora_down_mid_kernel<TT, RT, false>), grid, block, 0, st, a);                    \
  } while (0)
#define MID(TT)                                                                                       \
  do {                                                                                                \
    if (rt <= 1) MID_RT(TT, 1);                                                                        \
    else if (rt == 2) MID_RT(TT, 2);                                                                   \
    else MID_RT(TT, 4);                                                                                \
    if (sums) hipLaunchKernelGGL((lora_down_reduce_batch_kernel<TT>), rgrid, dim3(256), 0, st, a);     \
  } while (0)
  if (act_dtype == FMSA_BF16) MID(bf16_t);
  else MID(f16_t);
#undef MID
#undef MID_RT
  FMSA_CHECK_LAUNCH();
  return FMSA_OK;
}

int launch_lora_down(const void* X, int64_t ldx, const void* Wd, int M, int C, int r, int act_dtype, void* out,
                     int64_t ldo, hipStream_t st) {
  return launch_lora_down_plain(X, ldx, Wd, M, C, r, act_dtype, out, ldo, nullptr, 1, st);
}

namespace {
// Shape of the split launch: row groups per workgroup, column ranges, or g = 0 when the kernels without workspace do as
// well or the matrix is too small.  (At rank 16 and below Wd is a small part of the traffic; what the split kernel adds there
// is 64 tokens per workgroup with 1 KB row runs through LDS and column ranges that keep every CU busy: 21 -> 17 us on
// 8192 x 4096.)
struct DownSplit {
  int g, n_tb, n_split;
};
DownSplit lora_down_split_shape(int M, int C, int r, bool few_tokens) {
  const int rt = (std::min(r, 64) + 15) / 16;  // ranks above 64 go out 64 at a time (accumulator registers)
  if (M < 2048 || C < 2048) {
    // The columns of few tokens, where a wave has enough to walk through that the second launch pays: columns times rank
    // tiles of 4096 and more (us whole / split at 300 tokens: 1024 columns 4.4 / 5.5 at rank 16, 7.2 / 7.1 at 64,
    // 11.3 / 9.5 at 128; 2048 columns 6.1 / 6.1 at rank 16, 7.9 / 6.5 at 32; 4096 columns 9.5 / 7.1 at rank 16).
    // From 2048 tokens on the token blocks fill the chip (1024 columns, rank 64, 3000 tokens: 7.5 / 9.9).
    if (!few_tokens || M >= 2048 || (int64_t)C * ((r + 15) / 16) < 4096) return {0, 0, 0};
    // g = 1: the fragment kernel, columns split until two workgroups per CU are there or a wave is down to two steps of 32
    const int n_tb = (M + 15) / 16;
    const int n_split = std::min(512 / n_tb, C / 512);
    if (n_split < 2) return {0, 0, 0};
    return {1, n_tb, n_split};
  }
  if (rt < 2 && M >= 16384) return {0, 0, 0};  // rank 16 and below with a workgroup per CU anyway: the 32-token kernels do as well
  const int g = rt <= 2 ? 2 : 4;  // rank 32: 64 tokens per workgroup; 48 / 64: 128
  const int n_tb = (M + 32 * g - 1) / (32 * g);
  const int n_chunks = (C + 511) / 512;
  int n_split = (256 + n_tb - 1) / n_tb;                 // a workgroup per CU at least
  n_split = std::max(1, std::min(n_split, n_chunks / 2));  // two chunks per range at least
  return {g, n_tb, n_split};
}
}  // namespace

static int staged_workgroups(int M, int64_t columns, int r) {
  const DownSplit d = lora_down_split_shape(M, (int)columns, r, true);
  return d.n_tb * d.n_split;
}

static size_t down_mid_bytes(int M, int C, int r) {
  const int n = down_mid_split(M, C, r, rank_blocks(r));
  return n > 1 ? (size_t)n * M * r * sizeof(float) : 0;
}

static size_t down_split_bytes(int M, int C, int r, bool few_tokens) {
  const DownSplit d = lora_down_split_shape(M, C, r, few_tokens);
  const int ranks = d.g == 1 ? r : std::min(r, 64);
  return d.g && d.n_split > 1 ? (size_t)d.n_split * (size_t)M * (size_t)ranks * sizeof(float) : 0;
}

// Enough for either kernel, so that the answer for a shape does not depend on which of them is the faster one today.
size_t lora_down_workspace(int M, int C, int r, bool few_tokens) {
  const bool mid = (few_tokens || M >= 2048) && down_is_mid(M, C, r);
  return std::max(mid ? down_mid_bytes(M, C, r) : 0, down_split_bytes(M, C, r, few_tokens));
}

// The split kernel where it pays and the caller brought the partial-sum buffer (or none is needed); launch_lora_down otherwise.
int launch_lora_down_ws(const void* X, int64_t ldx, const void* Wd, int M, int C, int r, int act_dtype, void* out,
                        int64_t ldo, void* workspace, size_t workspace_bytes, bool few_tokens, hipStream_t st) {
  const size_t need = lora_down_workspace(M, C, r, few_tokens);
  // a buffer smaller than the query's answer is as good as none; the reduce pass stores four ranks at a time
  const bool sums = workspace && workspace_bytes >= need && (uintptr_t)out % 8 == 0 && ldo % 4 == 0;
  if ((few_tokens || M >= 2048) && down_is_mid(M, C, r) && (sums || !down_mid_bytes(M, C, r))) {
    LoraDownArgs a{};
    a.M = M;
    a.j[0] = {(const uint16_t*)X, (const uint16_t*)Wd, (uint16_t*)out, (float*)workspace, ldx, ldo, C, r, down_mid_split(M, C, r, rank_blocks(r))};
    return launch_down_mid(a, 1, act_dtype, st);
  }
  const DownSplit d = lora_down_split_shape(M, C, r, few_tokens);
  if (!d.g || (down_split_bytes(M, C, r, few_tokens) && !sums))
    return launch_lora_down(X, ldx, Wd, M, C, r, act_dtype, out, ldo, st);
  auto reduce = [&]() -> int {
    const int64_t quads = (int64_t)M * (r / 4);
    dim3 rgrid((unsigned)((quads + 255) / 256));
    if (act_dtype == FMSA_BF16)
      hipLaunchKernelGGL((lora_down_reduce_kernel<bf16_t>), rgrid, dim3(256), 0, st, (const float*)workspace, d.n_split, M, r,
                         (uint16_t*)out, ldo);
    else
      hipLaunchKernelGGL((lora_down_reduce_kernel<f16_t>), rgrid, dim3(256), 0, st, (const float*)workspace, d.n_split, M, r,
                         (uint16_t*)out, ldo);
    FMSA_CHECK_LAUNCH();
    return FMSA_OK;
  };
  if (d.g == 1) {
    if (int rc = launch_lora_down_plain(X, ldx, Wd, M, C, r, act_dtype, out, ldo, (float*)workspace, d.n_split, st)) return rc;
    return reduce();
  }
  if (r > 64) {
    // 64 ranks per pass over X (launches on one stream run in order, so the passes share the workspace); cheaper than one
    // pass whose accumulators and double-buffered Wd fragments do not fit the registers
    for (int r0 = 0; r0 < r; r0 += 64) {
      const int rc = launch_lora_down_ws(X, ldx, (const uint16_t*)Wd + (size_t)r0 * C, M, C, std::min(64, r - r0), act_dtype,
                                         (uint16_t*)out + r0, ldo, workspace, workspace_bytes, few_tokens, st);
      if (rc != FMSA_OK) return rc;
    }
    return FMSA_OK;
  }
  const int rt = (r + 15) / 16;
  dim3 grid(d.n_tb * d.n_split), block(512);
#define SPLIT_LAUNCH(TT, RT, G)                                                                                                  \
  hipLaunchKernelGGL((lora_down_split_kernel<TT, RT, G>), grid, block, 0, st, (const uint16_t*)X, ldx, (const uint16_t*)Wd, M, \
                     C, r, (uint16_t*)out, ldo, (float*)workspace, d.n_tb, d.n_split)
#define SPLIT_DISPATCH(TT)                            \
  switch (rt) {                                       \
    case 1: SPLIT_LAUNCH(TT, 1, 2); break;            \
    case 2: SPLIT_LAUNCH(TT, 2, 2); break;            \
    default: SPLIT_LAUNCH(TT, 4, 4); break;           \
  }
  if (act_dtype == FMSA_BF16) {
    SPLIT_DISPATCH(bf16_t)
  } else {
    SPLIT_DISPATCH(f16_t)
  }
#undef SPLIT_DISPATCH
#undef SPLIT_LAUNCH
  FMSA_CHECK_LAUNCH();
  if (d.n_split > 1) return reduce();
  return FMSA_OK;
}

// One launch for up to FMSA_LORA_DOWN_MAX_JOBS products over the same tokens, for few tokens (the rule of the g = 1 split).
static int down_batch_split(int M, int C, int n_jobs) {
  const int n_tb = (M + 15) / 16;
  return std::max(1, std::min(512 / (n_tb * n_jobs), C / 512));
}
static int max_rank(const fmsa_lora_down_job* jobs, int n_jobs) {
  int r = 0;
  for (int q = 0; q < n_jobs; ++q) r = std::max(r, jobs[q].r);
  return r;
}

// Column ranges of lora_down (one job) and of the batched launch over few tokens
int lora_down_few_splits(int M, int C, int r, int n_jobs) {
  if (n_jobs > 1) return down_batch_split(M, C, n_jobs);
  const DownSplit d = lora_down_split_shape(M, C, r, true);
  return d.g == 1 ? d.n_split : 1;
}

static bool down_batch_is_mid(const fmsa_lora_down_job* jobs, int n_jobs, int M) {
  int64_t columns = 0;
  bool lines = true;
  for (int q = 0; q < n_jobs; ++q) {
    columns += jobs[q].C;
    lines = lines && jobs[q].C % 64 == 0;
  }
  return down_is_mid(M, max_rank(jobs, n_jobs), columns, lines, n_jobs == 1);
}
static int down_batch_split_any(const fmsa_lora_down_job* jobs, int q, int n_jobs, int M) {
  const int r_max = max_rank(jobs, n_jobs);
  return down_batch_is_mid(jobs, n_jobs, M) ? down_mid_split(M, jobs[q].C, r_max, n_jobs * rank_blocks(r_max))
                                            : down_batch_split(M, jobs[q].C, n_jobs);
}

size_t lora_down_batch_workspace(const fmsa_lora_down_job* jobs, int n_jobs, int M) {
  size_t bytes = 0;
  for (int q = 0; q < n_jobs; ++q) bytes += (size_t)down_batch_split_any(jobs, q, n_jobs, M) * M * jobs[q].r * sizeof(float);
  return bytes;
}

int launch_lora_down_batch(const fmsa_lora_down_job* jobs, int n_jobs, int M, int act_dtype, void* workspace, hipStream_t st) {
  LoraDownArgs a{};
  a.M = M;
  const int r_max = max_rank(jobs, n_jobs);
  int split_max = 1;
  float* p = (float*)workspace;
  for (int q = 0; q < n_jobs; ++q) {
    const fmsa_lora_down_job& s = jobs[q];
    LoraDownJobDev& d = a.j[q];
    d.X = (const uint16_t*)s.X;
    d.Wd = (const uint16_t*)s.Wd;
    d.out = (uint16_t*)s.out;
    d.ldx = s.ldx;
    d.ldo = s.ldout;
    d.C = s.C;
    d.r = s.r;
    d.n_split = down_batch_split_any(jobs, q, n_jobs, M);
    d.partial = p;
    p += (size_t)d.n_split * M * s.r;
    split_max = std::max(split_max, d.n_split);
  }
  if (down_batch_is_mid(jobs, n_jobs, M)) return launch_down_mid(a, n_jobs, act_dtype, st);
  constexpr int NW = 8;
  const dim3 grid((M + 15) / 16, split_max, n_jobs), block(64 * NW);
  const dim3 rgrid((unsigned)(((int64_t)M * (r_max / 4) + 255) / 256), n_jobs);
  const int rt = (r_max + 15) / 16;
#define BATCH(TT)                                                                                            \
  do {                                                                                                       \
    if (rt <= 1) hipLaunchKernelGGL((lora_down_batch_kernel<TT, 1, 1, NW>), grid, block, 0, st, a);              \
    else if (rt <= 2) hipLaunchKernelGGL((lora_down_batch_kernel<TT, 2, 1, NW>), grid, block, 0, st, a);         \
    else if (rt <= 4) hipLaunchKernelGGL((lora_down_batch_kernel<TT, 4, 1, NW>), grid, block, 0, st, a);         \
    else hipLaunchKernelGGL((lora_down_batch_kernel<TT, 8, 1, NW>), grid, block, 0, st, a);                      \
    hipLaunchKernelGGL((lora_down_reduce_batch_kernel<TT>), rgrid, dim3(256), 0, st, a);                      \
  } while (0)
  if (act_dtype == FMSA_BF16) BATCH(bf16_t);
  else BATCH(f16_t);
#undef BATCH
  FMSA_CHECK_LAUNCH();
  return FMSA_OK;
}

namespace {
size_t job_partial_bytes(const fmsa_lora_grad_job& s, int M) {
  return (size_t)lora_grad_splits(M, s.C) * (size_t)s.r * (size_t)s.C * sizeof(float);
}
// Whether a launch's gradients come from one launch (lora_grad_waves_kernel).  us in two passes / there: q, k, v of hidden 2048 at 300
// tokens, rank 16, 13.2 / 6.3; 14336 and 4096 at 1100, rank 64, 22 / 14; gate and up of 4096 -> 14336 at 3217, rank 64, 87 / 50.  All of
// 36 forms, 2048 to 28672 columns, ranks 8 to 64: at 64 tokens 342 / 254, 512 706 / 331, 1100 778 / 469, 2048 1012 / 703, 4096 1534 /
// 1278, 8192 1570 / 1581.  Not where T comes along; above 2048 tokens for ranks that T never comes along with (smaller ones have the
// sums of a launch with T, and are a copy that takes more bytes in flight: 14336 and 4096 at 3217, rank 8, 23.9 / 25.7), and there
// not where few workgroups hold many ranks over more than 12 token tiles a wave (q, k, v of 2048 at 4096, stacked ranks 96, 25.5 /
// 28.1); and not where the stores of many ranks are all there is to do (8192 -> 28672 at 300, rank 64, 27.8 / 32).
bool lora_grad_in_one_launch(const fmsa_lora_grad_job* jobs, int n_jobs, int M) {
  int r_max = 0, blocks = 0;
  for (int q = 0; q < n_jobs; ++q) {
    if (jobs[q].Wt) return false;
    blocks += (jobs[q].C + LGW_COLS - 1) / LGW_COLS;
    r_max = std::max(r_max, jobs[q].r);
  }
  if (M <= 512) return r_max <= 64 || blocks <= 512;
  if (M <= 2048) return true;
  return M <= 4096 && r_max > 32 && (r_max <= 64 || blocks >= 128 || M <= 3072);
}
size_t job_tpart_bytes(const fmsa_lora_grad_job& s, int M) {
  return s.Wt ? (size_t)((s.C + LG_TC_T - 1) / LG_TC_T) * (size_t)M * (size_t)s.r * sizeof(float) : 0;
}
}  // namespace

size_t lora_grad_batch_workspace(const fmsa_lora_grad_job* jobs, int n_jobs, int M) {
  size_t bytes = 0;
  for (int q = 0; q < n_jobs; ++q) bytes += job_partial_bytes(jobs[q], M) + job_tpart_bytes(jobs[q], M);
  return bytes;
}

int launch_lora_grad_batch(const fmsa_lora_grad_job* jobs, int n_jobs, int M, int act_dtype, void* workspace, hipStream_t st) {
  LoraGradArgs a{};
  a.n_jobs = n_jobs;
  a.M = M;
  a.act_dtype = act_dtype;
  bool any_t = false;
  int64_t elements = 0;
  for (int q = 0; q < n_jobs; ++q) {
    any_t = any_t || jobs[q].Wt != nullptr;
    elements += (int64_t)jobs[q].r * jobs[q].C;
  }
  const bool waves = lora_grad_in_one_launch(jobs, n_jobs, M);
  const int tc = waves ? LGW_COLS : LG_TC_T;
  int blocks = 0, rblocks = 0, r_max = 0;
  size_t ws_off = 0;
  for (int q = 0; q < n_jobs; ++q) {
    const fmsa_lora_grad_job& s = jobs[q];
    LoraGradJobDev& d = a.j[q];
    d.L = (const uint16_t*)s.L;
    d.R = (const uint16_t*)s.R;
    d.out = s.out;
    d.partial = reinterpret_cast<float*>(reinterpret_cast<char*>(workspace) + ws_off);
    d.ldl = s.ldl;
    d.ldr = s.ldr;
    d.C = s.C;
    d.r = s.r;
    d.splits = lora_grad_splits(M, s.C);
    const int rows = (M + d.splits - 1) / d.splits;
    d.rows_per_split = ((rows + LG_TM - 1) / LG_TM) * LG_TM;
    d.block_start = blocks;
    d.rblock_start = rblocks;
    d.transpose_out = s.transpose_out;
    d.out_dtype = s.out_dtype;
    d.scale = s.scale;
    blocks += ((s.C + tc - 1) / tc) * (waves ? 1 : d.splits);
    // one element a thread: straight sums over several splits, in launches of fewer than 1024 workgroups with four (us with four /
    // one; single outputs: 4096 of rank 64 at 3217 tokens 25.2 / 22.8, 14336 of rank 32 at 8192 50.6 / 46.9, of rank 64 at 1100
    // 25.3 / 23.7, of rank 128 at 3217, 1792 workgroups, 58.8 / 60.4; q, k, v of rank 128 at 2048, 2304, 54 / 58; 14336 of rank 128
    // at 300 tokens, one split, 23.7 / 27.3)
    d.per_thread = !s.transpose_out && d.splits > 1 && elements < 1024 * 1024 ? 1 : 4;
    rblocks += (s.r * s.C / d.per_thread + 255) / 256;
    ws_off += job_partial_bytes(s, M);
    if (s.Wt) {
      d.Wt = (const uint16_t*)s.Wt;
      d.T = (uint16_t*)s.T;
      d.ldt = s.ldt;
      d.tpart = reinterpret_cast<float*>(reinterpret_cast<char*>(workspace) + ws_off);
      ws_off += job_tpart_bytes(s, M);
      rblocks += (int)(((int64_t)M * s.r / 4 + 255) / 256);
    }
    r_max = s.r > r_max ? s.r : r_max;
  }
  dim3 grid1(blocks), grid2(rblocks), block(256), block1(512);
  const int rt = (r_max + 15) / 16;
  if (waves) {
#define LAUNCH(TT)                                                                                                           \
  do {                                                                                                                      \
    if (rt == 1) hipLaunchKernelGGL((lora_grad_waves_kernel<TT, 1>), grid1, block1, 0, st, a);                               \
    else if (rt == 2) hipLaunchKernelGGL((lora_grad_waves_kernel<TT, 2>), grid1, block1, 0, st, a);                          \
    else if (rt <= 4) hipLaunchKernelGGL((lora_grad_waves_kernel<TT, 4>), grid1, block1, 0, st, a);                          \
    else hipLaunchKernelGGL((lora_grad_waves_kernel<TT, 8>), grid1, block1, 0, st, a);                                       \
  } while (0)
    if (act_dtype == FMSA_BF16) LAUNCH(bf16_t);
    else LAUNCH(f16_t);
#undef LAUNCH
    FMSA_CHECK_LAUNCH();
    return FMSA_OK;
  }
#define LAUNCH(TT, RT, WT) hipLaunchKernelGGL((lora_grad_partial_kernel<TT, RT, WT>), grid1, block1, 0, st, a)
#define DISPATCH(TT)                                                  \
  switch (rt) {                                                       \
    case 1: if (any_t) LAUNCH(TT, 1, true); else hipLaunchKernelGGL((lora_grad_partial_kernel<TT, 1, false>), grid1, block1, 0, st, a); break; \
    case 2: if (any_t) LAUNCH(TT, 2, true); else hipLaunchKernelGGL((lora_grad_partial_kernel<TT, 2, false>), grid1, block1, 0, st, a); break; \
    case 3: case 4: hipLaunchKernelGGL((lora_grad_partial_kernel<TT, 4, false>), grid1, block1, 0, st, a); break; \
    default: hipLaunchKernelGGL((lora_grad_partial_kernel<TT, 8, false>), grid1, block1, 0, st, a); break;         \
  }
  if (act_dtype == FMSA_BF16) {
    DISPATCH(bf16_t)
  } else {
    DISPATCH(f16_t)
  }
#undef DISPATCH
#undef LAUNCH
  FMSA_CHECK_LAUNCH();
  hipLaunchKernelGGL(lora_grad_reduce_kernel, grid2, block, 0, st, a);
  FMSA_CHECK_LAUNCH();
  return FMSA_OK;
}

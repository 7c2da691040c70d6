// Fused forward:  Y = X * deq(W) + s * U * B^T (+ bias), optional SwiGLU over a gate/up pair.
//
// Tiling (one workgroup = 4 waves = 256 lanes, one workgroup per CU):
//   workgroup tile  256 tokens x 256 output columns, K walked in stages of 64
//   wave tile       256 tokens x 64 columns = 8 x 2 MFMA 32x32x16 tiles, 256 fp32 accumulators
//   X operand       global -> LDS directly (buffer loads with the LDS bit: no staging registers, no
//                   ds_write), two stage buffers of 256 rows x 128 B, loaded one stage ahead.
//                   A direct load places lane p's 16 bytes at slot p of a 1 KB block, so the
//                   bank-conflict-free layout is obtained on the global side: slot c of row r holds
//                   the 8-element chunk c ^ ((r >> 1) & 7) of that row.  One barrier per stage.
//   W operand       never touches LDS: one packed int32 (8 nibbles along K at one column) is
//                   exactly the 8-element MFMA fragment of the lane that owns that column, so each
//                   lane loads its own words (a wave reads 2 x 128 B contiguous per load), unpacks
//                   them in registers and feeds the MFMA directly.  Each wave owns distinct
//                   columns, so no weight is unpacked twice inside a workgroup.
// The MFMA is issued as D^T = W^T-fragment x X-fragment: a lane then holds 4 consecutive output
// columns per accumulator quad, which turns the epilogue stores into 8-byte vectors.
// The rank-r LoRA term is one extra MFMA step per 16 ranks in the epilogue, scaled by s in fp32
// before the single rounding of the output.
//
// The kernel itself; gemm_fwd.hip plans and launches it, gemm_fwd_low.hip holds the flavours of lower tiles.
#pragma once
#include "common.h"
#include "split_tiles.h"

namespace fwd_tiles {

constexpr int BK = 64;
constexpr int EP_ROWS = 64;          // tokens per epilogue pass
constexpr int EP_STRIDE_L = 256 + 8;  // plane row stride (elements), linear: one plane of 256 columns
constexpr int EP_STRIDE_S = 128 + 8;  // SwiGLU: three planes (e, g, h) of 128 columns
constexpr int NBUF = 2;  // LDS stage buffers / register slots for the weight words
constexpr int NT = 2;

struct FwdProjDev {
  const int32_t* qweight;
  const uint16_t* scales;
  const int32_t* qzeros;
  const float* code;         // code-book format only
  const float* block_scale;  // code-book format only: fp32 [K / group_size, N]
  const uint16_t* U;
  int64_t ldu;
  const uint16_t* B;
  const uint16_t* bias;
  uint16_t* Y;
  int64_t ldy;
  int N, group_size, zero_offset, r;
  float s;
};

struct FwdArgs {
  FwdProjDev p[3];
  int nblk_start[4];
  const uint16_t* X;
  int64_t ldx;
  int M, K, mode, nbm, nbn;
  uint16_t* H;
  int64_t ldh;
  // rotary embedding in the epilogue (linear mode): projections whose bit is set in rope_mask leave rotated
  const void* rope_cos;
  const void* rope_sin;
  int64_t rope_ld;
  int rope_rows, rope_head_dim, rope_mask;
  // contraction split (SPLIT flavours): tiles n_whole .. n_whole + n_cut - 1 are cut into n_ranges ranges of stages
  int n_whole, n_cut, n_ranges, mt;  // mt: token tiles of a tile
  float* partial;
};

// a.p[p] for a runtime (wave-uniform) p without dynamic indexing of the kernel-argument struct,
// which would force a copy of it into scratch memory.
FMSA_DEVI FwdProjDev select_proj(const FwdArgs& a, int p) { return p == 0 ? a.p[0] : (p == 1 ? a.p[1] : a.p[2]); }

// token block and column block of tile pid: grouped-M order
FMSA_DEVI void fwd_tile(const FwdArgs& a, int pid, int& bm, int& bn) {
  constexpr int GROUP_M = 4;  // token blocks per group: 4 x 8 tiles in flight per XCD share X and W tiles in its L2
  const int width = GROUP_M * a.nbn;
  const int first_m = (pid / width) * GROUP_M;
  const int gsz = min(a.nbm - first_m, GROUP_M);
  bm = first_m + (pid % width) % gsz;
  bn = (pid % width) / gsz;
}

// GPS = scale groups per 64-wide K stage: 1 for group_size % 64 == 0, 2 / 4 for group sizes 32 / 16.
// CODEBOOK: the nibbles index a 16-entry table and one fp32 scale per (group, column) multiplies the entry
// (W = code[q] * block_scale) instead of the affine GPTQ form W = scale * (q - zero); the codes come from a table of pairs in
// LDS, two per 8-byte read, which leaves the LDS pipe the room that one ds_bpermute per code did not and takes 40 vector
// instructions a step less than 16 rounded products per block kept in registers and looked up with byte permutes did: 16384
// tokens, 4096 -> 14336 with the SwiGLU and 14336 -> 4096 together 5100 -> 4757 us (1213 TFLOP/s; affine 1264).
// ROPE (1: cos / sin tables in the activation type, 2: in fp32; 0: none): the Q / K projections of an attention block
// leave the kernel with the rotary embedding applied
// (kernels/unsloth/rope_embedding.py:36-65 of the reference: (q1, q2) <- (q1 cos - q2 sin, q2 cos + q1 sin) on the two
// halves of every head, on the projection output ROUNDED to the storage type, fp32 arithmetic, one more rounding).
// PK16 (fp16 activations, affine weights whose words hold their nibbles interleaved -- element 2p at position p, element
// 2p + 1 at position 4 + p --, one scale group per stage): a fragment register is (((w >> 4p) & 0x000F000F) | 0x64006400)
// + (-(1024 + z)) [exact] times the fp16 scale [one rounding] in packed half arithmetic: RNE_fp16(s * (q - z)) bit for bit
// in 15 instead of 22 instructions per word.
// SPLIT: the tiles that do not fill a round of the chip are cut along K (split_tiles.h); a template parameter, because the
// flavours without it are scheduled instruction by instruction.
// MT: token tiles of 32 rows, the tile's height (split_tiles.h says when fewer than 8 are taken).
template <typename T, int GPS, bool KTAIL, bool CODEBOOK, int ROPE = 0, bool PK16 = false, bool SPLIT = false, int MT = 8>
__global__ __launch_bounds__(256) void gptq_lora_fwd_kernel(const FwdArgs a) {
  static_assert(MT == 8 || (MT >= 4 && MT < 8 && GPS == 1 && !KTAIL && ROPE == 0), "lower tiles: one scale group per stage, whole stages");
  constexpr int BM = 32 * MT;
  static_assert(!PK16 || (std::is_same<T, f16_t>::value && !CODEBOOK && GPS == 1 && ROPE == 0), "packed half unpack");
  // two separate arrays (not one 2-D array): every access names its buffer statically, which is
  // what lets the compiler see that fragment reads of one buffer do not depend on the direct loads
  // in flight into the other
  __shared__ __attribute__((aligned(1024))) uint16_t lds0[BM * BK];
  __shared__ __attribute__((aligned(1024))) uint16_t lds1[BM * BK];
  // CODEBOOK: the pair table until the epilogue, the adapter's staged operands behind it (the strictest alignment puts the
  // array at LDS address 0: no base to add to a lookup)
  constexpr int PAIR_BYTES = CODEBOOK ? 256 * 32 * 8 : 0;
  constexpr int LORA_BYTES = (16 + 4 * NT) * 1024;
  __shared__ alignas(CODEBOOK ? 2048 : 16) uint16_t ep_planes[CODEBOOK ? (PAIR_BYTES + LORA_BYTES) / 2 : 3 * EP_ROWS * EP_STRIDE_S];  // >= EP_ROWS * EP_STRIDE_L
  static_assert(sizeof(ep_planes) >= 3 * EP_ROWS * EP_STRIDE_S * 2, "the SwiGLU planes must fit");
  static_assert(3 * EP_STRIDE_S >= EP_STRIDE_L, "the linear plane must fit");
  auto lds_buf = [&](auto b_c) -> char* {
    constexpr int b = decltype(b_c)::value;
    return reinterpret_cast<char*>(b == 0 ? lds0 : lds1);
  };

  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int l32 = lane & 31;
  const int half = lane >> 5;

  // ---- tile assignment: XCD-contiguous ranges, then grouped-M order inside the range --------
  SplitWork work{0, -1, 0};
  if constexpr (SPLIT) work = split_work(a.n_whole, a.n_cut, a.n_ranges);
  const int pid = SPLIT ? work.tile : xcd_remap(blockIdx.x, a.nbm * a.nbn);
  int bm, bn;
  fwd_tile(a, pid, bm, bn);
  const int m0 = bm * BM;

  int pj[NT], col0[NT];
  bool active[NT];
  if (a.mode == FMSA_FWD_SWIGLU) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      pj[j] = j;
      col0[j] = bn * 128 + wave * 32;
    }
  } else {
    int p = 0;
    if (bn >= a.nblk_start[1]) p = 1;
    if (bn >= a.nblk_start[2]) p = 2;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      pj[j] = p;
      col0[j] = (bn - a.nblk_start[p]) * 256 + wave * 64 + j * 32;
    }
  }
  const char* qbase[NT];
  const char* scbase[NT];
  const char* zbase[NT];
  int Np[NT], zshift[NT], gs[NT];
  float zoff[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const FwdProjDev P = select_proj(a, pj[j]);
    active[j] = col0[j] < P.N;
    if (!active[j]) col0[j] = 0;
    const int col = col0[j] + l32;
    // wave-uniform by construction; readfirstlane tells the compiler so (scalar offsets below)
    Np[j] = __builtin_amdgcn_readfirstlane(P.N);
    gs[j] = __builtin_amdgcn_readfirstlane(P.group_size);
    qbase[j] = reinterpret_cast<const char*>(P.qweight);
    scbase[j] = CODEBOOK ? reinterpret_cast<const char*>(P.block_scale) : reinterpret_cast<const char*>(P.scales);
    zbase[j] = reinterpret_cast<const char*>(P.qzeros);
    zshift[j] = 4 * (col & 7);
    zoff[j] = (float)P.zero_offset;
  }

  // code book: entry [16 hi + lo][copy] = (code[lo], code[hi]) as fp32, 32 copies of 8 bytes; lane l32 reads copy l32, so no two
  // lanes of a half wave meet in a bank whatever the codes are, and the address is one byte permute (byte << 8 | 8 * copy).
  // Copies 16-31 hold the second column tile's book; where the two differ (SwiGLU) a tile has 16 copies.
  uint32_t pair_lane[NT];
  if constexpr (CODEBOOK) {
    const float* c0 = select_proj(a, pj[0]).code;
    const float* c1 = select_proj(a, pj[1]).code;
#pragma unroll
    for (int j = 0; j < NT; ++j) pair_lane[j] = c0 == c1 ? (uint32_t)(8 * l32) : (uint32_t)(8 * (l32 & 15) + 128 * j);
    // thread: entry lo = tid >> 4, copies 2 * (tid & 15) and the next, all hi
    const float* c = (tid & 15) < 8 ? c0 : c1;
    const uint32_t lo = __float_as_uint(c[tid >> 4]);
    u32x4* dst = reinterpret_cast<u32x4*>(ep_planes) + tid;
#pragma unroll
    for (int hi = 0; hi < 16; ++hi) {
      const uint32_t up = __float_as_uint(c[hi]);
      dst[256 * hi] = u32x4{lo, up, lo, up};
    }
  }

  const int K = a.K;
  // this workgroup's stages st0 .. st_end - 1 of the contraction
  int st0 = 0, st_end = (K + BK - 1) / BK;
  if constexpr (SPLIT) {
    if (work.range >= 0) {
      const int n = st_end;
      st0 = work.range * n / a.n_ranges;
      st_end = (work.range + 1) * n / a.n_ranges;
    }
  }

  f32x16 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mt][j][i] = 0.f;

  // ---- operand addressing: buffer loads (SGPR resource + 32-bit lane offset + SGPR offset) -----
  // No 64-bit address arithmetic in the loop, and lanes whose offset falls outside the resource
  // read zeros: rows past M need no predication.
  // X tile: wave w fills rows 8 MT w .. 8 MT (w + 1) - 1 of a stage buffer with MT direct loads; load i covers
  // 8 rows from 8 (MT w + i), lane p writes slot (p & 7) of row 8 (MT w + i) + (p >> 3), which holds chunk
  // (p & 7) ^ ((row >> 1) & 7) of that row.
  const int uwave = __builtin_amdgcn_readfirstlane(wave);
  const int rows_valid = min(BM, a.M - m0);
  const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(a.X + (size_t)m0 * a.ldx, (size_t)rows_valid * a.ldx * 2);
  uint32_t x_off[8];  // (not MT: a builtin whose operands have dependent types is checked in the host pass, too)
  const int chunk_even = (lane & 7) ^ (lane >> 4);  // chunk fetched for even eights of rows; odd ones: ^ 4
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int row = 8 * (MT * wave + i) + (lane >> 3);
    const int chunk = chunk_even ^ (4 * ((MT * wave + i) & 1));
    x_off[i] = (uint32_t)((row * a.ldx + 8 * chunk) * 2);
  }
  // fragment reads: row 32*mt + l32, chunk 2t + half -> slot (2t + half) ^ ((l32 >> 1) & 7)
  uint32_t lds_r_off[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) lds_r_off[t] = (uint32_t)(l32 * (BK * 2) + 16 * ((2 * t + half) ^ ((l32 >> 1) & 7)));
  // weights: word (k8, col) at k8*N*4 + col*4; the lane part is (half*N + col)*4
  __amdgpu_buffer_rsrc_t q_rsrc[NT], sc_rsrc[NT], z_rsrc[NT];
  uint32_t q_off[NT], sc_off[NT], z_off[NT];
  uint32_t q_stage_bytes[NT], q_step_bytes[NT], q_last[NT];
  int n_groups_j[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n_groups = (K + gs[j] - 1) / gs[j];
    n_groups_j[j] = n_groups;
    q_rsrc[j] = make_rsrc(qbase[j], (size_t)(K >> 3) * Np[j] * 4);
    sc_rsrc[j] = make_rsrc(scbase[j], (size_t)n_groups * Np[j] * (CODEBOOK ? 4 : 2));
    z_rsrc[j] = make_rsrc(zbase[j], CODEBOOK ? 0 : (size_t)n_groups * (Np[j] >> 3) * 4);
    q_off[j] = (uint32_t)((half * Np[j] + col0[j] + l32) * 4);
    sc_off[j] = (uint32_t)((col0[j] + l32) * (CODEBOOK ? 4 : 2));
    z_off[j] = (uint32_t)(((col0[j] + l32) >> 3) * 4);
    q_step_bytes[j] = (uint32_t)Np[j] * 8;    // two packed rows per 16-wide K step
    q_stage_bytes[j] = (uint32_t)Np[j] * 32;  // eight packed rows per stage
    q_last[j] = (uint32_t)((K >> 3) - 2) * Np[j] * 4;
  }

  // Weight words, scales and zero words in two register slots (slot = stage % 2), loaded one
  // stage ahead together with X.
  uint32_t qw[NBUF][NT][4];
  uint16_t sc_raw[NBUF][NT][GPS];
  uint32_t zw_raw[NBUF][NT][GPS];  // code-book format: the fp32 block scale
  float sf[NT][GPS], sf16[NT][GPS], nsz[NT][GPS];
  uint32_t sp16[NT], nz16[NT];  // PK16: the stage's scale and -(1024 + zero) as fp16 pairs (both halves equal)
  const uint32_t pk_mask = opaque(0x000F000Fu), pk_bias = opaque(0x64006400u);  // in vector registers: the and-or takes no literal
  // group index of the stage being loaded, advanced without a division when GPS == 1
  int g_ld[NT], k_in_g[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    g_ld[j] = k_in_g[j] = 0;
    if constexpr (SPLIT) {
      g_ld[j] = __builtin_amdgcn_readfirstlane(st0 * BK / gs[j]);
      k_in_g[j] = __builtin_amdgcn_readfirstlane(st0 * BK % gs[j]);
    }
  }
  // issue the global loads of stage `st` (st0 <= st < st_end) into slot SB; nothing here may read
  // the loaded registers, or the wave would wait for the load on the spot
  auto load_stage = [&](int st, auto sb_c) {
    constexpr int SB = decltype(sb_c)::value;
    const uint32_t x_soff = (uint32_t)st * (BK * 2);
    // K % 64 == 32 (KTAIL): in the last stage the upper half of the stage lies past K.  Its X
    // columns are forced out of range (zeros); the weight rows are clamped to valid memory.
    uint32_t poison[2] = {0u, 0u};
    if constexpr (KTAIL) {
      poison[0] = ((st * BK + 8 * chunk_even) < K) ? 0u : 0x80000000u;
      poison[1] = ((st * BK + 8 * (chunk_even ^ 4)) < K) ? 0u : 0x80000000u;
    }
    char* lw = lds_buf(sb_c) + uwave * (8 * MT * BK * 2);
#pragma unroll
    for (int i = 0; i < MT; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(x_rsrc, (__attribute__((address_space(3))) void*)(lw + i * (8 * BK * 2)),
                                               16, x_off[i] | poison[i & 1], x_soff, 0, 0);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const uint32_t qs = (uint32_t)st * q_stage_bytes[j];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        uint32_t so = qs + t * q_step_bytes[j];
        if constexpr (KTAIL) so = min(so, q_last[j]);
        qw[SB][j][t] = __builtin_amdgcn_raw_buffer_load_b32(q_rsrc[j], q_off[j], so, 0);
      }
#pragma unroll
      for (int u = 0; u < GPS; ++u) {
        int gu;
        if constexpr (GPS == 1) {
          gu = min(g_ld[j], n_groups_j[j] - 1);
        } else {
          const int ku = st * BK + u * (BK / GPS);
          gu = (ku < K ? ku : st * BK) / gs[j];
        }
        gu = __builtin_amdgcn_readfirstlane(gu);  // uniform; keeps the scalar offsets out of vector registers
        if constexpr (CODEBOOK) {
          zw_raw[SB][j][u] = __builtin_amdgcn_raw_buffer_load_b32(sc_rsrc[j], sc_off[j], (uint32_t)gu * Np[j] * 4, 0);
        } else {
          sc_raw[SB][j][u] = __builtin_amdgcn_raw_buffer_load_b16(sc_rsrc[j], sc_off[j], (uint32_t)gu * Np[j] * 2, 0);
          zw_raw[SB][j][u] = __builtin_amdgcn_raw_buffer_load_b32(z_rsrc[j], z_off[j], (uint32_t)gu * (Np[j] >> 3) * 4, 0);
        }
      }
      if constexpr (GPS == 1) {  // uniform scalar bookkeeping, no division
        k_in_g[j] += BK;
        const bool wrap = k_in_g[j] >= gs[j];
        k_in_g[j] -= wrap ? gs[j] : 0;
        g_ld[j] += wrap ? 1 : 0;
      }
    }
  };
  // make the scales / zeros of slot SB current
  auto commit_stage = [&](auto sb_c) {
    constexpr int SB = decltype(sb_c)::value;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
#pragma unroll
      for (int u = 0; u < GPS; ++u) {
        if constexpr (CODEBOOK) {
          sf[j][u] = __uint_as_float(zw_raw[SB][j][u]);
        } else if constexpr (PK16) {
          sp16[j] = (uint32_t)sc_raw[SB][j][u] * 0x00010001u;
          const float nz = -(1024.0f + (float)((zw_raw[SB][j][u] >> zshift[j]) & 0xFu) + zoff[j]);  // exact in fp16
          nz16[j] = pack2<f16_t>(nz, nz);
        } else {
          sf[j][u] = fp16_bits_to_f32(sc_raw[SB][j][u]);
          sf16[j][u] = sf[j][u] * 0.0625f;
          const float z = (float)((zw_raw[SB][j][u] >> zshift[j]) & 0xFu) + zoff[j];
          nsz[j][u] = -sf[j][u] * z;  // exact: 11-bit x 5-bit
        }
      }
    }
  };

  // Software pipeline at the granularity of one 16-wide MFMA K step: while the 16 MFMAs of step t
  // run, the 8 X fragments of step t+1 are read from LDS and its 2 weight fragments are unpacked,
  // into the other half of xf / wf.  The stage barrier sits after step 2, so step 3 can already
  // fetch step 0 of the next stage from the next LDS buffer.
  u32x4 xf[2][MT], wf[2][NT];
  const char* const pairs = reinterpret_cast<const char*>(ep_planes);
  // the codes of a word's byte: elements 2 byte, 2 byte + 1 = fragment register `byte`
  auto look_up = [&](uint32_t w, int j, auto byte_c) -> u32x2 {
    return *reinterpret_cast<const u32x2*>(pairs + __builtin_amdgcn_perm(w, pair_lane[j], 0x0C0C0400u + 256 * decltype(byte_c)::value));
  };
  // code * block scale in fp32, one rounding
  auto scaled = [&](const u32x2& v, float sc) -> uint32_t { return pack2<T>(__uint_as_float(v[0]) * sc, __uint_as_float(v[1]) * sc); };
  auto prefetch = [&](auto sb_c, auto t_c, auto par_c) {
    constexpr int SB = decltype(sb_c)::value;
    constexpr int t = decltype(t_c)::value;
    constexpr int par = decltype(par_c)::value;
    const char* lr = lds_buf(sb_c) + lds_r_off[t];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) xf[par][mt] = *reinterpret_cast<const u32x4*>(lr + mt * 32 * BK * 2);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      if constexpr (CODEBOOK) {
        u32x2 v[4];
        static_for<0, 4>([&](auto r_c) { v[decltype(r_c)::value] = look_up(qw[SB][j][t], j, r_c); });
#pragma unroll
        for (int r = 0; r < 4; ++r) wf[par][j][r] = scaled(v[r], sf[j][t * GPS / 4]);
      } else if constexpr (PK16) {
        static_for<0, 4>([&](auto r_c) {
          constexpr int r = decltype(r_c)::value;
          wf[par][j][r] = pk_sub_mul_f16(((qw[SB][j][t] >> (4 * r)) & pk_mask) | pk_bias, nz16[j], sp16[j]);
        });
      } else {
        wf[par][j] = dequant8<T>(qw[SB][j][t], sf[j][t * GPS / 4], sf16[j][t * GPS / 4], nsz[j][t * GPS / 4]);
      }
    }
  };
  auto mfma_step = [&](auto par_c) {
    constexpr int par = decltype(par_c)::value;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[mt][j] = mfma32<T>(wf[par][j], xf[par][mt], acc[mt][j]);
  };
  // One wave per SIMD issues strictly in order, and an MFMA that finds the matrix pipe busy stalls
  // everything behind it.  The other instructions of a step therefore have to sit BETWEEN its 16
  // MFMAs (each occupies the pipe for 8 issue slots): per MFMA 3 VALU, every second one an LDS
  // read, and in step 0 also the global loads of a later stage with their scalar offset math.
  auto interleave = [&](auto with_vmem_c) {
    constexpr bool with_vmem = decltype(with_vmem_c)::value;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
      if (CODEBOOK || (i & 1) == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (with_vmem) {
        if (i < 6)
          __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
        else
          __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // nothing from the next step (or the stage hand-over) moves up
  };
  using WithVmem = std::integral_constant<bool, true>;
  using NoVmem = std::integral_constant<bool, false>;
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;

  // One 64-wide K stage out of LDS buffer / register slot SB = s % 2.  Steps 0-2 read the stage's
  // fragments; then every wave waits for its own loads of stage s + 1 (issued one stage earlier),
  // and the barrier makes all four waves' parts visible and closes the reads of buffer SB.  Step 3
  // therefore is where the loads of stage s + 2 go out, into the buffer and register slot this
  // stage has just vacated.  The last two stages re-load the final stage (no branch); that data
  // is never read.
  constexpr int WAIT_VM0 = 0x0F70;  // s_waitcnt vmcnt(0) only
  // one 16-wide K step: the MFMAs of parity `cur` while fragments and weights of (buffer nb, step nt)
  // are produced into parity `nx`
  auto step = [&](auto nb_c, auto nt_c, auto nx_c, auto cur_c, auto vmem_c) {
    prefetch(nb_c, nt_c, nx_c);
    mfma_step(cur_c);
    interleave(vmem_c);
  };
  // The step with one scale group per stage written slot by slot, as the input-gradient kernel on the transposed
  // twin does: the 16 MFMAs of parity `cur`, behind each one its share of the work that produces step (nb, nt) into
  // parity `nx` -- a fragment read behind the first eight, one unpacked fragment register (2 conversions, 2
  // multiply-adds, 1 packed conversion) behind every even one -- and, in the last step of a stage, the 20 loads of
  // stage `st_next` into buffer / slot `lb`.  A scheduling fence closes every slot: the order below is the schedule
  // (about 1 % faster than what the group-barrier matcher makes of the same step; the fragment reads spread over the
  // odd slots instead measured no gain).  From a code book the 8 lookups lead, two behind each of the first four, the fragment
  // reads follow, and a register's product comes about four MFMAs after its lookup.
  constexpr bool HAND = GPS == 1;
  // load number `idx` of stage `st` into slot SB (GPS == 1): the MT loads of the X tile (direct loads), 8 weight words
  // (4 j + t), scale and zero word of column tile 0, of column tile 1 (code book: the block scale in the scale's place)
  auto load_piece = [&](int st, auto sb_c, auto idx_c) {
    constexpr int SB = decltype(sb_c)::value;
    constexpr int idx = decltype(idx_c)::value;
    if constexpr (idx < MT) {
      uint32_t poison = 0u;
      if constexpr (KTAIL) poison = ((st * BK + 8 * (chunk_even ^ (4 * (idx & 1)))) < K) ? 0u : 0x80000000u;
      char* lw = lds_buf(sb_c) + uwave * (8 * MT * BK * 2);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(x_rsrc, (__attribute__((address_space(3))) void*)(lw + idx * (8 * BK * 2)), 16,
                                               x_off[idx] | poison, (uint32_t)st * (BK * 2), 0, 0);
    } else if constexpr (idx < MT + 8) {
      constexpr int j = (idx - MT) >> 2, t = (idx - MT) & 3;
      uint32_t so = (uint32_t)st * q_stage_bytes[j] + t * q_step_bytes[j];
      if constexpr (KTAIL) so = min(so, q_last[j]);
      qw[SB][j][t] = __builtin_amdgcn_raw_buffer_load_b32(q_rsrc[j], q_off[j], so, 0);
    } else {
      constexpr int j = (idx - MT - 8) >> 1;
      const int gu = __builtin_amdgcn_readfirstlane(min(g_ld[j], n_groups_j[j] - 1));
      if constexpr (((idx - MT - 8) & 1) == 0) {
        if constexpr (CODEBOOK) zw_raw[SB][j][0] = __builtin_amdgcn_raw_buffer_load_b32(sc_rsrc[j], sc_off[j], (uint32_t)gu * Np[j] * 4, 0);
        else sc_raw[SB][j][0] = __builtin_amdgcn_raw_buffer_load_b16(sc_rsrc[j], sc_off[j], (uint32_t)gu * Np[j] * 2, 0);
      } else {
        if constexpr (!CODEBOOK) zw_raw[SB][j][0] = __builtin_amdgcn_raw_buffer_load_b32(z_rsrc[j], z_off[j], (uint32_t)gu * (Np[j] >> 3) * 4, 0);
        k_in_g[j] += BK;  // uniform scalar bookkeeping, no division
        const bool wrap = k_in_g[j] >= gs[j];
        k_in_g[j] -= wrap ? gs[j] : 0;
        g_ld[j] += wrap ? 1 : 0;
      }
    }
  };
  auto step_hand = [&](auto nb_c, auto nt_c, auto nx_c, auto cur_c, auto vmem_c, int st_next, auto lb_c) {
    constexpr int SB = decltype(nb_c)::value;
    constexpr int t = decltype(nt_c)::value;
    constexpr int par = decltype(nx_c)::value;
    constexpr int cur = decltype(cur_c)::value;
    constexpr bool with_vmem = decltype(vmem_c)::value;
    const char* lr = lds_buf(nb_c) + lds_r_off[t];
    auto mfma_slot = [&](int slot) { acc[slot >> 1][slot & 1] = mfma32<T>(wf[cur][slot & 1], xf[cur][slot >> 1], acc[slot >> 1][slot & 1]); };
    auto frag = [&](int mt) { xf[par][mt] = *reinterpret_cast<const u32x4*>(lr + mt * 32 * BK * 2); };
    auto fence = [&]() { __builtin_amdgcn_sched_barrier(0); };
    constexpr int SLOTS = 2 * MT, EXTRA = MT + 12 - SLOTS;
    // the MT + 12 loads: one a slot, the last EXTRA ride with the last slots'
    auto dma = [&](auto u_c) {
      constexpr int u = decltype(u_c)::value;
      if constexpr (with_vmem) {
        load_piece(st_next, lb_c, u_c);
        if constexpr (u >= SLOTS - EXTRA) load_piece(st_next, lb_c, std::integral_constant<int, u + EXTRA>{});
      }
    };
    uint32_t nib[NT][2];  // [tile][0]: nibbles 0, 2, 4, 6 in bytes 0..3; [1]: 16 * nibbles 1, 3, 5, 7 (the scale is pre-divided)
    auto masks = [&](auto j_c) {
      constexpr int j = decltype(j_c)::value;
      if constexpr (!PK16) {
        nib[j][0] = opaque(qw[SB][j][t] & 0x0F0F0F0Fu);
        nib[j][1] = opaque(qw[SB][j][t] & 0xF0F0F0F0u);
      }
    };
    auto piece = [&](auto j_c, auto reg_c) {
      constexpr int j = decltype(j_c)::value;
      constexpr int reg = decltype(reg_c)::value;
      if constexpr (PK16) {
        wf[par][j][reg] = pk_sub_mul_f16(((qw[SB][j][t] >> (4 * reg)) & pk_mask) | pk_bias, nz16[j], sp16[j]);
        return;
      }
      float b0, b1;
      if constexpr (reg == 0) {
        b0 = ubyte0(nib[j][0]);
        b1 = ubyte0(nib[j][1]);
      } else if constexpr (reg == 1) {
        b0 = ubyte1(nib[j][0]);
        b1 = ubyte1(nib[j][1]);
      } else if constexpr (reg == 2) {
        b0 = ubyte2(nib[j][0]);
        b1 = ubyte2(nib[j][1]);
      } else {
        b0 = ubyte3(nib[j][0]);
        b1 = ubyte3(nib[j][1]);
      }
      wf[par][j][reg] = pack2<T>(__builtin_fmaf(sf[j][0], b0, nsz[j][0]), __builtin_fmaf(sf16[j][0], b1, nsz[j][0]));
    };
    if constexpr (CODEBOOK) {
      u32x2 v[NT][4];
      constexpr int ROOM = SLOTS - 5 < 8 ? SLOTS - 5 : 8;  // slots that the 8 products spread over
      static_for<0, SLOTS>([&](auto u_c) {
        constexpr int u = decltype(u_c)::value;
        mfma_slot(u);
        if constexpr (u < 4) {
          constexpr int j = u & 1, b = 2 * (u >> 1);
          v[j][b] = look_up(qw[SB][j][t], j, std::integral_constant<int, b>{});
          v[j][b + 1] = look_up(qw[SB][j][t], j, std::integral_constant<int, b + 1>{});
        }
        if constexpr (u >= 4 && u < 4 + MT) frag(u - 4);
        static_for<0, 8>([&](auto p_c) {
          constexpr int p = decltype(p_c)::value, j = p & 1, reg = p >> 1;
          if constexpr (u == 5 + p * ROOM / 8) wf[par][j][reg] = scaled(v[j][reg], sf[j][0]);
        });
        dma(u_c);
        fence();
      });
      return;
    }
    static_for<0, SLOTS>([&](auto u_c) {
      constexpr int u = decltype(u_c)::value;
      mfma_slot(u);
      if constexpr (u == 0) masks(std::integral_constant<int, 0>{});
      if constexpr (u == SLOTS / 2) masks(std::integral_constant<int, 1>{});
      static_for<0, 8>([&](auto p_c) {
        constexpr int p = decltype(p_c)::value;
        if constexpr (u == p * SLOTS / 8) piece(std::integral_constant<int, (p >> 2)>{}, std::integral_constant<int, (p & 3)>{});
      });
      if constexpr (u < MT) frag(u);
      dma(u_c);
      fence();
    });
  };
  auto stage = [&](int s, auto sb_c) {
    constexpr int SB = decltype(sb_c)::value;
    using S1 = std::integral_constant<int, SB ^ 1>;
    if constexpr (HAND) {
      step_hand(sb_c, I1{}, I1{}, I0{}, NoVmem{}, 0, sb_c);
      step_hand(sb_c, I2{}, I0{}, I1{}, NoVmem{}, 0, sb_c);
      step_hand(sb_c, I3{}, I1{}, I0{}, NoVmem{}, 0, sb_c);
    } else {
      step(sb_c, I1{}, I1{}, I0{}, NoVmem{});
      step(sb_c, I2{}, I0{}, I1{}, NoVmem{});
      step(sb_c, I3{}, I1{}, I0{}, NoVmem{});
    }
    __builtin_amdgcn_s_waitcnt(WAIT_VM0);
    commit_stage(S1{});
    __syncthreads();
    if constexpr (HAND) {
      step_hand(S1{}, I0{}, I0{}, I1{}, WithVmem{}, min(s + 2, st_end - 1), sb_c);
    } else {
      load_stage(min(s + 2, st_end - 1), sb_c);
      step(S1{}, I0{}, I0{}, I1{}, WithVmem{});
    }
  };

  // LoRA operands of ranks 0..15 (the whole adapter up to rank 16): direct loads into the epilogue planes,
  // which are idle until the epilogue, issued here so that their latency is not exposed after the main loop.
  // KB (8u + mt): rows 32mt..32mt+31 of U of the tile's u-th projection, 16 B per (row, rank half) at slot
  // 2 * row + half.  KB (16 + NT * wave + j): the same for the wave's 32 rows of B of column tile j.
  // Ranks past r and rows past M / N arrive as zeros through the range check.
  char* const lora_lds = reinterpret_cast<char*>(ep_planes) + PAIR_BYTES;
  static_assert(sizeof(ep_planes) >= PAIR_BYTES + LORA_BYTES, "LoRA operands must fit into the epilogue planes");
  const bool lora_any = (a.p[0].r | a.p[1].r | a.p[2].r) != 0;
  if (lora_any) {
    const int prow = lane >> 1, phalf = lane & 1;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const FwdProjDev P = select_proj(a, pj[j]);
      const int rp = __builtin_amdgcn_readfirstlane(P.r);
      const uint32_t dead = (8 * phalf < rp) ? 0u : 0x80000000u;
      if (j == 0 || a.mode == FMSA_FWD_SWIGLU) {  // linear mode: both column tiles belong to one projection
        const __amdgpu_buffer_rsrc_t u_rs = make_rsrc(P.U + (size_t)m0 * P.ldu, rp > 0 ? (size_t)rows_valid * P.ldu * 2 : 0);
#pragma unroll
        for (int i = 0; i < 2; ++i)
          if (MT == 8 || 2 * uwave + i < MT)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                u_rs, (__attribute__((address_space(3))) void*)(lora_lds + (8 * j + 2 * uwave + i) * 1024), 16,
                (uint32_t)(((64 * wave + 32 * i + prow) * P.ldu + 8 * phalf) * 2) | dead, 0, 0, 0);
      }
      const __amdgpu_buffer_rsrc_t b_rs = make_rsrc(P.B, rp > 0 ? (size_t)P.N * rp * 2 : 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rs, (__attribute__((address_space(3))) void*)(lora_lds + (16 + NT * uwave + j) * 1024),
                                               16, (uint32_t)(((col0[j] + prow) * rp + 8 * phalf) * 2) | dead, 0, 0, 0);
    }
  }
  load_stage(st0, I0{});
  __builtin_amdgcn_s_waitcnt(WAIT_VM0);
  commit_stage(I0{});
  __syncthreads();
  load_stage(min(st0 + 1, st_end - 1), I1{});
  prefetch(I0{}, I0{}, I0{});

  // whole pairs in a single-exit loop (slots 0, 1), then the odd stage
  const int s_full = st0 + ((st_end - st0) & ~1);
  int s = st0;
  for (; s < s_full; s += NBUF) {
    stage(s, I0{});
    stage(s + 1, I1{});
  }
  if (s < st_end) stage(s, I0{});

  // ---- LoRA term as extra contraction steps: acc += U[:, j0..j0+15] x (s * B[:, j0..j0+15])^T -------
  // s * B is rounded to the storage type, the rounding point of the reference's
  // `(X @ A.t()) @ (s * B.t())` (UL/gptq/fast_lora.py:167-169).  Rows past M read zeros through the
  // buffer resource.
  // One loop for both modes (no mode branch around the accumulators): tile j takes U and B of its
  // own projection -- gate / up in SwiGLU mode, twice the same projection otherwise.
  {
    const uint16_t* Uj[NT];
    const uint16_t* Bj[NT];
    int rj[NT];
    int64_t lduj[NT];
    float sj[NT];
    __amdgpu_buffer_rsrc_t u_rsrc[NT];
    int r_max = 0;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const FwdProjDev P = select_proj(a, pj[j]);
      rj[j] = __builtin_amdgcn_readfirstlane(P.r);
      sj[j] = P.s;
      Uj[j] = P.U;
      Bj[j] = P.B;
      lduj[j] = P.ldu;
      u_rsrc[j] = make_rsrc(P.U + (size_t)m0 * P.ldu, rj[j] > 0 ? (size_t)rows_valid * P.ldu * 2 : 0);
      r_max = max(r_max, rj[j]);
    }
    if (SPLIT && work.range > 0) r_max = 0;  // the adapter's term goes into the first range of a cut tile
    const uint32_t slot = (uint32_t)(2 * l32 + half) * 16;
    const int u_region = a.mode == FMSA_FWD_SWIGLU ? 8 : 0;  // KB between the U blocks of column tiles 0 and 1
    for (int j0 = 0; j0 < r_max; j0 += 16) {
      const int ko = j0 + 8 * half;
      u32x4 uf[NT][MT], bw[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        u32x4 bf = {0u, 0u, 0u, 0u};
        if (j0 == 0) {  // staged in LDS before the main loop
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) uf[j][mt] = *reinterpret_cast<const u32x4*>(lora_lds + (u_region * j + mt) * 1024 + slot);
          bf = *reinterpret_cast<const u32x4*>(lora_lds + (16 + NT * wave + j) * 1024 + slot);
        } else {
          const bool live = ko < rj[j];
          const uint32_t dead = live ? 0u : 0x80000000u;
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            uf[j][mt] = __builtin_amdgcn_raw_buffer_load_b128(u_rsrc[j], (uint32_t)(((32 * mt + l32) * lduj[j] + ko) * 2) | dead, 0, 0);
          if (live) bf = *reinterpret_cast<const u32x4*>(Bj[j] + (size_t)(col0[j] + l32) * rj[j] + ko);
        }
#pragma unroll
        for (int w = 0; w < 4; ++w) bw[j][w] = pack2<T>(sj[j] * unpack_lo<T>(bf[w]), sj[j] * unpack_hi<T>(bf[w]));
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[mt][j] = mfma32<T>(bw[j], uf[j][mt], acc[mt][j]);
    }
  }

  if constexpr (SPLIT) {
    if (work.range >= 0) {
      __builtin_amdgcn_s_waitcnt(WAIT_VM0);  // the surplus direct loads of the last stage have landed
      split_store(acc, a.partial, work.cut, work.range, a.n_ranges, rows_valid);
      return;
    }
  }

  // ---- epilogue ---------------------------------------------------------------------------
  // accumulator register 4*i0+i1 of acc[mt][j] is Y[m0 + 32*mt + l32][col0[j] + 8*i0 + 4*half + i1].
  // 64 tokens at a time the rounded outputs go through LDS planes (8-byte writes per lane) and
  // leave as 16-byte row segments through buffer stores: rows past M and columns past N are
  // dropped by the range check, so there are no branches.
  const bool swiglu = a.mode == FMSA_FWD_SWIGLU;
  const FwdProjDev PL = select_proj(a, pj[0]);
  const int cb = swiglu ? bn * 128 : (bn - a.nblk_start[pj[0]]) * 256;  // first output column of the tile
  const int lcol = swiglu ? wave * 32 : wave * 64;                      // wave's first column inside the tile
  const int estride = swiglu ? EP_STRIDE_S : EP_STRIDE_L;              // plane row stride, elements
  uint16_t* plane0 = ep_planes;
  uint16_t* plane1 = ep_planes + EP_ROWS * EP_STRIDE_S;
  uint16_t* plane2 = ep_planes + 2 * EP_ROWS * EP_STRIDE_S;
  // coalesced side: linear 32 chunks per row (8 rows per sweep), SwiGLU 16 chunks per row (16 rows)
  const int cchunk = swiglu ? (tid & 15) : (tid & 31);
  const int crow = swiglu ? (tid >> 4) : (tid >> 5);
  const int crows_per_it = swiglu ? 16 : 8;
  const int n_out = swiglu ? a.p[0].N : PL.N;
  const uint32_t col_dead = (cb + 8 * cchunk) < n_out ? 0u : 0x80000000u;
  const int64_t ld0 = swiglu ? a.p[0].ldy : PL.ldy;
  const __amdgpu_buffer_rsrc_t y0_rsrc = make_rsrc((swiglu ? a.p[0].Y : PL.Y) + (size_t)m0 * ld0, (size_t)rows_valid * ld0 * 2);
  const __amdgpu_buffer_rsrc_t y1_rsrc = make_rsrc(a.p[1].Y + (size_t)m0 * a.p[1].ldy, swiglu ? (size_t)rows_valid * a.p[1].ldy * 2 : 0);
  const __amdgpu_buffer_rsrc_t h_rsrc = make_rsrc(a.H + (size_t)m0 * a.ldh, swiglu ? (size_t)rows_valid * a.ldh * 2 : 0);
  const uint32_t y0_voff = (uint32_t)((crow * ld0 + cb + 8 * cchunk) * 2) | col_dead;
  const uint32_t y1_voff = (uint32_t)((crow * a.p[1].ldy + cb + 8 * cchunk) * 2) | col_dead;
  const uint32_t h_voff = (uint32_t)((crow * a.ldh + cb + 8 * cchunk) * 2) | col_dead;
  const uint32_t y0_row = __builtin_amdgcn_readfirstlane((uint32_t)(ld0 * 2));
  const uint32_t y1_row = __builtin_amdgcn_readfirstlane((uint32_t)(a.p[1].ldy * 2));
  const uint32_t h_row = __builtin_amdgcn_readfirstlane((uint32_t)(a.ldh * 2));
  // bias of the lane's 4 x 4 columns per tile
  float bias_v[NT][16];
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const FwdProjDev P = select_proj(a, pj[j]);
#pragma unroll
    for (int i = 0; i < 16; ++i) bias_v[j][i] = 0.f;
    if (P.bias) {
#pragma unroll
      for (int i0 = 0; i0 < 4; ++i0) {
        const u32x2 bv = *reinterpret_cast<const u32x2*>(P.bias + col0[j] + 8 * i0 + 4 * half);
        bias_v[j][4 * i0 + 0] = unpack_lo<T>(bv[0]);
        bias_v[j][4 * i0 + 1] = unpack_hi<T>(bv[0]);
        bias_v[j][4 * i0 + 2] = unpack_lo<T>(bv[1]);
        bias_v[j][4 * i0 + 3] = unpack_hi<T>(bv[1]);
      }
    }
  }
  // rotary embedding (ROPE flavour, tiles of a projection named by rope_mask): the thread's pair of half-head chunks
  bool rope_on = false;
  int rp_row = 0, rp_c1 = 0, rp_c2 = 0, rp_cw = 0, rp_pos0 = 0;
  uint32_t rp_voff = 0;
  u32x4 rp_c[EP_ROWS / 16][2], rp_s[EP_ROWS / 16][2];  // cos / sin of the pair's 8 columns per sweep of the pass, as loaded:
                                                       // one 16-byte word of 16-bit values or two of fp32
  if constexpr (ROPE != 0) {
    rope_on = ((a.rope_mask >> pj[0]) & 1) != 0;
    const int hd = a.rope_head_dim, hpc = hd >> 4;  // 8-column chunks per half head (a power of two)
    const int pi = tid & 15;
    const int head = pi >> (31 - __builtin_clz(hpc)), within = pi & (hpc - 1);
    rp_row = tid >> 4;
    rp_c1 = head * (hd >> 3) + within;
    rp_c2 = rp_c1 + hpc;
    rp_cw = 8 * within;
    rp_pos0 = (m0 + rp_row) % a.rope_rows;
    rp_voff = (uint32_t)((rp_row * ld0 + cb + 8 * rp_c1) * 2) | ((cb + 8 * rp_c1) < n_out ? 0u : 0x80000000u);
  }
  __syncthreads();  // (the stage buffers are not reused, but all waves are past the main loop)

  static_for<0, (MT + 1) / 2>([&](auto q_c) {
    constexpr int q = decltype(q_c)::value;
    constexpr int ROWS = MT - 2 * q < 2 ? 32 : EP_ROWS;  // of this pass
    if constexpr (ROPE != 0) {
      // cos / sin of this pass's rows, asked for before the accumulators are packed so that they arrive behind that work
      if (rope_on) {
        static_for<0, EP_ROWS / 16>([&](auto it_c) {
          constexpr int it = decltype(it_c)::value;
          int pos = rp_pos0 + EP_ROWS * q + 16 * it;  // token row m0 + ... takes table row (token row) % rope_rows
          if (pos >= a.rope_rows) pos %= a.rope_rows;
          const int64_t cso = (int64_t)pos * a.rope_ld + rp_cw;
          // kept as loaded and unpacked where they are used: an ALU operation here would make the wave wait for the load
          // before it goes on to pack its accumulators
          if constexpr (ROPE == 2) {
            const u32x4* cp = reinterpret_cast<const u32x4*>(reinterpret_cast<const float*>(a.rope_cos) + cso);
            const u32x4* sp = reinterpret_cast<const u32x4*>(reinterpret_cast<const float*>(a.rope_sin) + cso);
            rp_c[it][0] = cp[0];
            rp_c[it][1] = cp[1];
            rp_s[it][0] = sp[0];
            rp_s[it][1] = sp[1];
          } else {
            rp_c[it][0] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(a.rope_cos) + cso);
            rp_s[it][0] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(a.rope_sin) + cso);
          }
        });
      }
    }
    static_for<0, ROWS / 32>([&](auto ml_c) {
      constexpr int ml = decltype(ml_c)::value;
      constexpr int mt = 2 * q + ml;
      const int prow = 32 * ml + l32;
      if (swiglu) {
#pragma unroll
        for (int i0 = 0; i0 < 4; ++i0) {
          u32x2 ev, gv, hv;
          float hf[4];
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            ev[w] = pack2<T>(acc[mt][0][4 * i0 + 2 * w] + bias_v[0][4 * i0 + 2 * w],
                             acc[mt][0][4 * i0 + 2 * w + 1] + bias_v[0][4 * i0 + 2 * w + 1]);
            gv[w] = pack2<T>(acc[mt][1][4 * i0 + 2 * w] + bias_v[1][4 * i0 + 2 * w],
                             acc[mt][1][4 * i0 + 2 * w + 1] + bias_v[1][4 * i0 + 2 * w + 1]);
            // f = RNE(e32 * sigmoid(e32)) on the rounded e; h = RNE(f * g) on the rounded g
            const float e0 = unpack_lo<T>(ev[w]), e1 = unpack_hi<T>(ev[w]);
            const uint32_t fv = pack2<T>(e0 * sigmoidf_(e0), e1 * sigmoidf_(e1));
            hf[2 * w] = unpack_lo<T>(fv) * unpack_lo<T>(gv[w]);
            hf[2 * w + 1] = unpack_hi<T>(fv) * unpack_hi<T>(gv[w]);
          }
          hv[0] = pack2<T>(hf[0], hf[1]);
          hv[1] = pack2<T>(hf[2], hf[3]);
          const int o = prow * EP_STRIDE_S + lcol + 8 * i0 + 4 * half;
          *reinterpret_cast<u32x2*>(plane0 + o) = ev;
          *reinterpret_cast<u32x2*>(plane1 + o) = gv;
          *reinterpret_cast<u32x2*>(plane2 + o) = hv;
        }
      } else {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int i0 = 0; i0 < 4; ++i0) {
            u32x2 yv;
            yv[0] = pack2<T>(acc[mt][j][4 * i0 + 0] + bias_v[j][4 * i0 + 0], acc[mt][j][4 * i0 + 1] + bias_v[j][4 * i0 + 1]);
            yv[1] = pack2<T>(acc[mt][j][4 * i0 + 2] + bias_v[j][4 * i0 + 2], acc[mt][j][4 * i0 + 3] + bias_v[j][4 * i0 + 3]);
            *reinterpret_cast<u32x2*>(plane0 + prow * EP_STRIDE_L + lcol + 32 * j + 8 * i0 + 4 * half) = yv;
          }
      }
    });
    __syncthreads();
    if (swiglu) {
#pragma unroll
      for (int it = 0; it < ROWS / 16; ++it) {
        const int row = crow + 16 * it;
        const uint32_t srow = (uint32_t)(EP_ROWS * q + 16 * it);
        const int o = row * EP_STRIDE_S + 8 * cchunk;
        __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4*>(plane0 + o), y0_rsrc, y0_voff, srow * y0_row, STORE_NT);
        __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4*>(plane1 + o), y1_rsrc, y1_voff, srow * y1_row, STORE_NT);
        __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4*>(plane2 + o), h_rsrc, h_voff, srow * h_row, STORE_NT);
      }
    } else {
      if (ROPE != 0 && rope_on) {
        // Two half-head chunks per thread: 8 columns of the first half of a head and the 8 columns half a head
        // further (heads do not straddle the 256-column tile), so every cos / sin value is loaded and unpacked once
        // for the two outputs it makes.  16 pairs per row, 16 rows per sweep.
        static_for<0, EP_ROWS / 16>([&](auto it_c) {
          constexpr int it = decltype(it_c)::value;
          const int row = rp_row + 16 * it;
          const uint32_t srow = (uint32_t)(EP_ROWS * q + 16 * it);
          u32x4 v1 = *reinterpret_cast<const u32x4*>(plane0 + row * EP_STRIDE_L + 8 * rp_c1);
          u32x4 v2 = *reinterpret_cast<const u32x4*>(plane0 + row * EP_STRIDE_L + 8 * rp_c2);
          static_for<0, 4>([&](auto w_c) {
            constexpr int w = decltype(w_c)::value;  // values 2w and 2w + 1 of the 8 columns
            float c0, c1, s0, s1;
            if constexpr (ROPE == 2) {
              c0 = __uint_as_float(rp_c[it][w >> 1][2 * (w & 1)]);
              c1 = __uint_as_float(rp_c[it][w >> 1][2 * (w & 1) + 1]);
              s0 = __uint_as_float(rp_s[it][w >> 1][2 * (w & 1)]);
              s1 = __uint_as_float(rp_s[it][w >> 1][2 * (w & 1) + 1]);
            } else {
              c0 = unpack_lo<T>(rp_c[it][0][w]);
              c1 = unpack_hi<T>(rp_c[it][0][w]);
              s0 = unpack_lo<T>(rp_s[it][0][w]);
              s1 = unpack_hi<T>(rp_s[it][0][w]);
            }
            const float a0 = unpack_lo<T>(v1[w]), a1 = unpack_hi<T>(v1[w]);  // first half of the head
            const float b0 = unpack_lo<T>(v2[w]), b1 = unpack_hi<T>(v2[w]);  // second half
            v1[w] = pack2<T>(a0 * c0 - b0 * s0, a1 * c1 - b1 * s1);
            v2[w] = pack2<T>(b0 * c0 + a0 * s0, b1 * c1 + a1 * s1);
          });
          __builtin_amdgcn_raw_buffer_store_b128(v1, y0_rsrc, rp_voff, srow * y0_row, STORE_NT);
          __builtin_amdgcn_raw_buffer_store_b128(v2, y0_rsrc, rp_voff + (uint32_t)(a.rope_head_dim), srow * y0_row, STORE_NT);
        });
      } else {
#pragma unroll
        for (int it = 0; it < ROWS / 8; ++it) {
          const int row = crow + 8 * it;
          const uint32_t srow = (uint32_t)(EP_ROWS * q + 8 * it);
          __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4*>(plane0 + row * EP_STRIDE_L + 8 * cchunk), y0_rsrc,
                                                 y0_voff, srow * y0_row, STORE_NT);
        }
      }
    }
    __syncthreads();
  });
  (void)estride;
  (void)crows_per_it;
  (void)active;
}

// Launches the flavours of one height below 8 (gemm_fwd_low.hip).
struct LowLaunch {
  bool bf16, codebook, pk16, split;
  dim3 grid;
  hipStream_t st;
};

}  // namespace fwd_tiles

void launch_fwd_tiles_4(const fwd_tiles::FwdArgs& a, const fwd_tiles::LowLaunch& l);
void launch_fwd_tiles_5(const fwd_tiles::FwdArgs& a, const fwd_tiles::LowLaunch& l);
void launch_fwd_tiles_6(const fwd_tiles::FwdArgs& a, const fwd_tiles::LowLaunch& l);
void launch_fwd_tiles_7(const fwd_tiles::FwdArgs& a, const fwd_tiles::LowLaunch& l);

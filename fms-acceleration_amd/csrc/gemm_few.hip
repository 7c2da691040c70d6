// Forward of few tokens: Y = X * deq(W) + s * U * B^T (+ bias), optional SwiGLU over a gate / up pair.
//
// Up to a few dozen tokens a launch is one pass over the packed weights: 8 MB for 4096 x 4096, 59 MB for gate and up of
// 4096 x 14336, against X and Y of kilobytes.  The 256-token tiles of gemm_fwd.hip keep at most 240 workgroups of one wave
// per SIMD busy on that, issue 32 matrix instructions per weight fragment of which one has tokens in it, and need a second
// launch for the sums of their ranges.  Here:
//   workgroup  16 * CT output columns (of each projection it serves) for 16 * MT tokens; its waves share the contraction: wave
//              w of NW takes the 64-wide chunks w, w + NW, ..  4096 columns are 256 workgroups without cutting K between
//              workgroups, so there is no second launch, and the chunks the waves have in flight (8 to 16 KB per CU and
//              workgroup) are what the memory's latency asks for.
//   W operand  a lane's packed word is its 8-element fragment of MFMA 16x16x32 as in gemm_fwd.hip, and is unpacked the same
//              way, with the same rounding: RNE(s * (q - z)).  16 lanes read 64 B of a row of words with CT = 1 (the
//              neighbouring workgroup, on the same XCD, takes the other half of the line) and 128 B with CT = 2.
//   X operand  every workgroup reads all of X (from L2), through LDS of the wave's own.
// The waves' tiles are added in LDS in wave order, so the result does not depend on scheduling.
// Measured next to the 256-token tiles cut along K and their second launch, us at 1 / 12 / 64 tokens, rank 16: 4096 x 4096 33.6
// -> 6.3 / 6.4 / 12.2, q, k, v of 4096 and 1024 columns 36.4 -> 8.4 / 8.7 / 12.5, gate and up of 4096 x 14336 64 -> 22 / 22 / 41,
// 14336 x 4096 52 -> 12.4 / 12.4 / 28.  Bound by latency and the unpack at one token (30 vector instructions per 64 words of a
// wave, 12 of the 22 us), by the reads of X towards 64 tokens.
#include "common.h"

int lora_down_few_splits(int M, int C, int r, int n_jobs);  // lora_skinny.hip

namespace {

constexpr int FEW_BK = 64;  // contraction elements per chunk
constexpr int FEW_STAGE = 16 * FEW_BK;  // elements of 16 rows of a chunk
constexpr int few_vmcnt(int n) { return (n & 0xF) | ((n >> 4) << 14) | 0x0F70; }  // s_waitcnt operand: vmcnt(n) only, n < 64
constexpr int FEW_DOWN_NW = 8;

struct FewProjDev {
  const int32_t* qweight;
  const uint16_t* scales;
  const int32_t* qzeros;
  const float* code;
  const float* block_scale;
  const uint16_t* U;  // [M, r] in the activation type, or nullptr: sum the ranges of `partial`
  int64_t ldu;
  const void* A;  // rank-r product: [r, K] in the parameters' type
  const void* B;  // [N, r]
  const uint16_t* bias;
  uint16_t* Y;
  int64_t ldy;
  int N, zero_offset, r, u_col;  // u_col: first column of this projection in `partial`
  uint32_t group_magic;          // chunk -> group: (chunk * magic) >> 32; 0: every chunk is a group
  int param_dtype;               // of A and B: FMSA_F32, or the activation type
  float s;
};

struct FewArgs {
  FewProjDev p[3];
  int nblk_start[3];
  const uint16_t* X;
  int64_t ldx;
  const uint16_t* Xd;  // input of the rank-r products (the model's K order)
  int64_t ldxd;
  int M, K, n_cb, n_tb, swiglu;
  uint16_t* H;
  int64_t ldh;
  float* partial;  // [n_ranges][M][r_all] fp32 sums of the rank-r products
  int n_ranges, r_all;
};

FMSA_DEVI uint32_t few_group(uint32_t chunk, uint32_t magic) { return magic ? __umulhi(chunk, magic) : chunk; }

FMSA_DEVI FewProjDev few_proj(const FewArgs& a, int p) { return p == 0 ? a.p[0] : (p == 1 ? a.p[1] : a.p[2]); }

// Eight consecutive parameters as an MFMA fragment, rounded to the activation type.
template <typename T> FMSA_DEVI u32x4 few_params(const void* base, size_t at, bool f32) {
  if (!f32) return *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(base) + at);
  const f32x4* p = reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(base) + at);
  const f32x4 a = p[0], b = p[1];
  return u32x4{pack2<T>(a[0], a[1]), pack2<T>(a[2], a[3]), pack2<T>(b[0], b[1]), pack2<T>(b[2], b[3])};
}

// FMT 0: affine words in the checkpoint's nibble order; 1: interleaved words, packed-half unpack (fp16); 2: code book
// (codes from a table of pairs in LDS, two per 8-byte read).
template <typename T, int FMT, int NP, int MT, int CT, int NW, int DEPTH, int WPE>
__global__ __launch_bounds__(64 * NW, WPE) void gptq_lora_fwd_few_kernel(const FewArgs a) {
  static_assert(CT == 1 || CT == 2, "columns per lane");
  static_assert(DEPTH == 2 || DEPTH == 4, "stage buffers");
  static_assert((DEPTH - 1) * (2 * MT + 4 * NP) < 64, "vmcnt");
  static_assert(NP * CT <= 2, "the waves' sums must fit into a stage buffer");
  static_assert(FMT != 1 || std::is_same<T, f16_t>::value, "packed half unpack");
  // one array per stage buffer: an access names its buffer statically, so the compiler's wait counts tell the reads of one
  // from the direct loads in flight into the others
  __shared__ __attribute__((aligned(1024))) uint16_t st0[NW * MT * FEW_STAGE];
  __shared__ __attribute__((aligned(1024))) uint16_t st1[NW * MT * FEW_STAGE];
  __shared__ __attribute__((aligned(1024))) uint16_t st2[DEPTH > 2 ? NW * MT * FEW_STAGE : 8];
  __shared__ __attribute__((aligned(1024))) uint16_t st3[DEPTH > 2 ? NW * MT * FEW_STAGE : 8];
  // Code book: entry [16 hi + lo][copy] = (code[lo], code[hi]) as fp32, a lane's copy by its number: with 16 of them 16 lanes never
  // meet in a bank.  The LDS pipe bound the launches while every code was a ds_bpermute of its own (16 of them and 36 vector
  // instructions for the two words of a column, 8 reads and 20 now): the launches of a layer of hidden 4096 at 12 / 64 / 300 tokens, three
  // ranks, 263 / 500 / 301 -> 213 / 407 / 217 us, of hidden 2048 140 / 256 / 320 -> 131 / 230 / 252; affine words take 204 / 395 / 203.
  // COPIES leaves as many workgroups on a CU as run there without the table.
  constexpr int COPIES = FMT == 2 ? (MT == 1 ? 16 : 8) : 0;
  __shared__ __attribute__((aligned(1024))) u32x2 pairs[FMT == 2 ? 256 * COPIES : 1];
  auto stage = [&](auto d_c) -> char* {
    constexpr int d = decltype(d_c)::value;
    return reinterpret_cast<char*>(d == 0 ? st0 : (d == 1 ? st1 : (d == 2 ? st2 : st3)));
  };
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, c = lane & 15, kq = lane >> 4;

  // token blocks of one column block are neighbours: they read the same weights
  const int pid = xcd_remap(blockIdx.x, a.n_cb * a.n_tb);
  const int cb = pid / a.n_tb, m0 = (pid % a.n_tb) * (16 * MT);
  int p0 = 0;
  if (NP == 1) p0 = cb >= a.nblk_start[2] ? 2 : (cb >= a.nblk_start[1] ? 1 : 0);
  const int n0 = (NP == 1 ? cb - (p0 == 0 ? 0 : (p0 == 1 ? a.nblk_start[1] : a.nblk_start[2])) : cb) * (16 * CT);
  const int col = n0 + CT * c;  // the lane's first column; tile j of the wave holds columns n0 + CT * row + j

  FewProjDev P[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) P[p] = few_proj(a, NP == 1 ? p0 : p);

  f32x4 acc[NP][CT][MT];
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[p][j][mt] = f32x4{0.f, 0.f, 0.f, 0.f};

  // ---- LoRA term: 32 ranks per matrix step; (projection, rank step, token tile) in turn over the waves, ahead of the wave's
  // stream of weights, so that its few small loads do not queue behind that ----
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int r = __builtin_amdgcn_readfirstlane(P[p].r);
    const bool f32 = P[p].param_dtype == FMSA_F32;
    for (int rs = 0; rs * 32 < r; ++rs) {
      const int ko = 32 * rs + 8 * kq;
      static_for<0, MT>([&](auto mt_c) {
        constexpr int mt = decltype(mt_c)::value;
        if (((rs * MT + mt) * NP + p) % NW != wave) return;
        const int m = m0 + 16 * mt + c;
        u32x4 bf[CT];
#pragma unroll
        for (int j = 0; j < CT; ++j) {
          bf[j] = u32x4{0u, 0u, 0u, 0u};
          if (ko < r) bf[j] = few_params<T>(P[p].B, (size_t)(col + j) * r + ko, f32);
        }
        u32x4 uf = {0u, 0u, 0u, 0u};
        if (ko < r && m < a.M) {
          if (P[p].U) {
            uf = *reinterpret_cast<const u32x4*>(P[p].U + (size_t)m * P[p].ldu + ko);
          } else {
            const f32x4* src = reinterpret_cast<const f32x4*>(a.partial + (size_t)m * a.r_all + P[p].u_col + ko);
            const size_t step = (size_t)a.M * a.r_all / 4;
            f32x4 lo, hi;
            for (int i0 = 0; i0 < a.n_ranges; i0 += 8) {  // eight ranges asked for at once, added in index order
              f32x4 part[8][2];
#pragma unroll
              for (int i = 0; i < 8; ++i) {
                const size_t at = (size_t)min(i0 + i, a.n_ranges - 1) * step;  // the surplus re-reads the last range
                part[i][0] = src[at];
                part[i][1] = src[at + 1];
              }
#pragma unroll
              for (int i = 0; i < 8; ++i) {
                if (i0 + i == 0) {
                  lo = part[i][0];
                  hi = part[i][1];
                } else if (i0 + i < a.n_ranges) {
                  lo += part[i][0];
                  hi += part[i][1];
                }
              }
            }
            uf = u32x4{pack2<T>(lo[0], lo[1]), pack2<T>(lo[2], lo[3]), pack2<T>(hi[0], hi[1]), pack2<T>(hi[2], hi[3])};
          }
        }
#pragma unroll
        for (int j = 0; j < CT; ++j) {
#pragma unroll
          for (int w = 0; w < 4; ++w) bf[j][w] = pack2<T>(P[p].s * unpack_lo<T>(bf[j][w]), P[p].s * unpack_hi<T>(bf[j][w]));
          acc[p][j][mt] = mfma16<T>(bf[j], uf, acc[p][j][mt]);
        }
      });
    }
  }

  __amdgpu_buffer_rsrc_t q_rsrc[NP], s_rsrc[NP], z_rsrc[NP];
  uint32_t q_off[NP], s_off[NP], z_off[NP], q_chunk[NP], q_half[NP];
  int zshift[NP], N[NP];
  float zoff[NP];
  const int n_chunks = (a.K + FEW_BK - 1) / FEW_BK;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    N[p] = __builtin_amdgcn_readfirstlane(P[p].N);
    const int n_groups = (int)few_group(n_chunks - 1, P[p].group_magic) + 1;
    q_rsrc[p] = make_rsrc(P[p].qweight, (size_t)(a.K >> 3) * N[p] * 4);
    s_rsrc[p] = FMT == 2 ? make_rsrc(P[p].block_scale, (size_t)n_groups * N[p] * 4) : make_rsrc(P[p].scales, (size_t)n_groups * N[p] * 2);
    z_rsrc[p] = make_rsrc(P[p].qzeros, FMT == 2 ? 0 : (size_t)n_groups * (N[p] >> 3) * 4);
    q_off[p] = (uint32_t)((kq * N[p] + col) * 4);
    s_off[p] = (uint32_t)(col * (FMT == 2 ? 4 : 2));
    z_off[p] = (uint32_t)((col >> 3) * 4);
    q_half[p] = (uint32_t)N[p] * 16;   // four rows of words: 32 contraction elements
    q_chunk[p] = (uint32_t)N[p] * 32;
    zshift[p] = 4 * (col & 7);
    zoff[p] = (float)P[p].zero_offset;
  }
  // X: the wave's chunk of 16 * MT rows goes through its own 2 KB * MT of a stage buffer by direct loads, 8 rows x 128 B
  // each; a fragment load from global has four rows in every four lanes, which the address path takes one by one (16 B per
  // clock and CU: 4096 x 4096 at 32 tokens 11.4 us that way).  Slot s of row r holds the 16 bytes s ^ ((r >> 1) & 7), so that
  // the fragment reads spread over all banks.  Nobody else touches the wave's part: no barrier.
  const int rows = min(16 * MT, a.M - m0);
  const __amdgpu_buffer_rsrc_t x_rsrc = make_rsrc(a.X + (size_t)m0 * a.ldx, (size_t)rows * a.ldx * 2);
  static_assert(MT <= 4, "x_off");
  uint32_t x_off[8];  // (of fixed size: the host pass drops the stub of a kernel whose direct loads index one sized by MT)
  // the lane's 16 bytes of its row: slot lane & 7 of row 8 i + (lane >> 3)
#pragma unroll
  for (int i = 0; i < 2 * MT; ++i) {
    const int row = 8 * i + (lane >> 3), chunk = (lane & 7) ^ ((row >> 1) & 7);
    x_off[i] = (uint32_t)((row * a.ldx + 8 * chunk) * 2);
  }
  uint32_t x_lds[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) x_lds[t] = (uint32_t)(wave * MT * FEW_STAGE * 2 + c * 128 + 16 * ((4 * t + kq) ^ ((c >> 1) & 7)));

  // DEPTH chunks in flight.  Loads of a chunk past the wave's last one, and of the half chunk past K, are out of range by
  // their lane offsets: zeros, and no traffic.
  uint32_t qw[DEPTH][NP][2][CT], sc[DEPTH][NP][CT], zw[DEPTH][NP];
  auto load = [&](int chunk, auto d_c) {
    constexpr int d = decltype(d_c)::value;
    const uint32_t dead0 = chunk * FEW_BK < a.K ? 0u : 0x80000000u;
    const uint32_t dead1 = chunk * FEW_BK + 32 < a.K ? 0u : 0x80000000u;
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) {
      // half chunk past K: the lanes that fetch its 16-byte pieces (4..7 of a row)
      const uint32_t dead = (((lane & 7) ^ (((8 * i + (lane >> 3)) >> 1) & 7)) & 4) ? dead1 : dead0;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(x_rsrc, (__attribute__((address_space(3))) void*)(stage(d_c) + wave * (MT * FEW_STAGE * 2) + i * 1024),
                                               16, x_off[i] | dead, (uint32_t)chunk * (FEW_BK * 2), 0, 0);
    }
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const uint32_t g = __builtin_amdgcn_readfirstlane(few_group((uint32_t)chunk, P[p].group_magic));
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const uint32_t so = (uint32_t)chunk * q_chunk[p] + t * q_half[p];
        const uint32_t vo = q_off[p] | (t ? dead1 : dead0);
        if constexpr (CT == 1) {
          qw[d][p][t][0] = __builtin_amdgcn_raw_buffer_load_b32(q_rsrc[p], vo, so, 0);
        } else {
          const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(q_rsrc[p], vo, so, 0);
          qw[d][p][t][0] = v[0];
          qw[d][p][t][1] = v[1];
        }
      }
      if constexpr (FMT == 2) {
        if constexpr (CT == 1) {
          sc[d][p][0] = __builtin_amdgcn_raw_buffer_load_b32(s_rsrc[p], s_off[p] | dead0, g * (uint32_t)N[p] * 4, 0);
        } else {
          const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(s_rsrc[p], s_off[p] | dead0, g * (uint32_t)N[p] * 4, 0);
          sc[d][p][0] = v[0];
          sc[d][p][1] = v[1];
        }
      } else {
        if constexpr (CT == 1)
          sc[d][p][0] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(s_rsrc[p], s_off[p] | dead0, g * (uint32_t)N[p] * 2, 0);
        else
          sc[d][p][0] = __builtin_amdgcn_raw_buffer_load_b32(s_rsrc[p], s_off[p] | dead0, g * (uint32_t)N[p] * 2, 0);
        zw[d][p] = __builtin_amdgcn_raw_buffer_load_b32(z_rsrc[p], z_off[p] | dead0, g * (uint32_t)(N[p] >> 3) * 4, 0);
      }
    }
  };
  // The table is written while the first chunks are on their way: the book's entries are asked for ahead of them, and the barrier
  // waits for the LDS writes alone.  Where the two projections' books differ, each has half of the copies.
  uint32_t pair_lane[NP];
  constexpr int PAIR_VEC = 256 * COPIES / 2, PAIR_TURNS = FMT == 2 ? PAIR_VEC / (64 * NW) : 0;  // 16-byte writes, two copies each
  static_assert(FMT != 2 || PAIR_VEC % (64 * NW) == 0, "every thread writes as many entries");
  u32x2 entry[FMT == 2 ? PAIR_TURNS : 1];
  if constexpr (FMT == 2) {
    const float *c0 = P[0].code, *c1 = P[NP - 1].code;
#pragma unroll
    for (int p = 0; p < NP; ++p)
      pair_lane[p] = c0 == c1 ? (uint32_t)(8 * (lane & (COPIES - 1))) : (uint32_t)(8 * (lane & (COPIES / 2 - 1)) + 4 * COPIES * p);
#pragma unroll
    for (int k = 0; k < PAIR_TURNS; ++k) {
      const int v = tid + 64 * NW * k, e = v / (COPIES / 2);
      const float* book = v % (COPIES / 2) < COPIES / 4 ? c0 : c1;
      entry[k] = u32x2{__float_as_uint(book[e & 15]), __float_as_uint(book[e >> 4])};
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  const uint32_t pk_mask = opaque(0x000F000Fu), pk_bias = opaque(0x64006400u);
  auto multiply = [&](auto d_c) {
    constexpr int d = decltype(d_c)::value;
    // the direct loads of this chunk have landed: at most the loads of the DEPTH - 1 younger chunks are outstanding
    __builtin_amdgcn_s_waitcnt(few_vmcnt((DEPTH - 1) * (2 * MT + NP * (FMT == 2 ? 3 : 4))));
    __builtin_amdgcn_sched_barrier(0);
    u32x4 xf[2][MT];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) xf[t][mt] = *reinterpret_cast<const u32x4*>(stage(d_c) + x_lds[t] + mt * 2048);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        u32x4 wf[2];
        if constexpr (FMT == 2) {
          const float bs = __uint_as_float(sc[d][p][j]);
          u32x2 v[2][4];
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const uint32_t w = qw[d][p][t][j];
            static_for<0, 4>([&](auto b_c) {  // the codes of byte b: elements 2b, 2b + 1
              constexpr int b = decltype(b_c)::value, at = COPIES == 16 ? 7 : 6;
              const uint32_t byte = 8 * b < at ? w << (at - 8 * b) : w >> (8 * b - at);
              v[t][b] = *reinterpret_cast<const u32x2*>(reinterpret_cast<const char*>(pairs) + ((byte & (0xFFu << at)) | pair_lane[p]));
            });
          }
#pragma unroll
          for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int b = 0; b < 4; ++b) wf[t][b] = pack2<T>(__uint_as_float(v[t][b][0]) * bs, __uint_as_float(v[t][b][1]) * bs);
        } else {
          const uint16_t sb = (uint16_t)(sc[d][p][0] >> (16 * j));
          const float z = (float)((zw[d][p] >> (zshift[p] + 4 * j)) & 0xFu) + zoff[p];
          if constexpr (FMT == 1) {
            const uint32_t sp = (uint32_t)sb * 0x00010001u;
            const float nz = -(1024.0f + z);  // exact in fp16
            const uint32_t nzp = pack2<f16_t>(nz, nz);
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
              for (int r = 0; r < 4; ++r) wf[t][r] = pk_sub_mul_f16(((qw[d][p][t][j] >> (4 * r)) & pk_mask) | pk_bias, nzp, sp);
          } else {
            const float sf = fp16_bits_to_f32(sb);
#pragma unroll
            for (int t = 0; t < 2; ++t) wf[t] = dequant8<T>(qw[d][p][t][j], sf, sf * 0.0625f, -sf * z);
          }
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[p][j][mt] = mfma16<T>(wf[t], xf[t][mt], acc[p][j][mt]);
      }
    }
  };

  // turn `it` of the wave: chunk wave + NW * it
  const int n_it = (n_chunks + NW - 1) / NW;
  static_for<0, DEPTH>([&](auto d_c) {
    load(wave + NW * decltype(d_c)::value, d_c);
    // the counted wait for a chunk takes the loads of the younger ones to be younger: nothing but this keeps the compiler, which
    // knows the buffers for separate arrays, from issuing them first
    __builtin_amdgcn_sched_barrier(0);
  });
  if constexpr (FMT == 2) {
#pragma unroll
    for (int k = 0; k < PAIR_TURNS; ++k)
      reinterpret_cast<u32x4*>(pairs)[tid + 64 * NW * k] = u32x4{entry[k][0], entry[k][1], entry[k][0], entry[k][1]};
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0) only
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int it = 0; it < n_it; it += DEPTH)
    static_for<0, DEPTH>([&](auto d_c) {
      constexpr int d = decltype(d_c)::value;
      multiply(d_c);
      // the fragments of buffer d have arrived (their matrix steps were issued) before it is loaded again: a direct load is
      // not ordered behind LDS reads that are still queued
      __builtin_amdgcn_sched_barrier(0);
      load(wave + NW * (it + DEPTH + d), d_c);
    });

  // ---- the waves' sums, through stage buffer 0 (the surplus direct loads have landed, every wave's) ----
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __syncthreads();
  float(*red)[MT][NP * CT][64][4] = reinterpret_cast<float(*)[MT][NP * CT][64][4]>(st0);
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) *reinterpret_cast<f32x4*>(red[wave][mt][p * CT + j][lane]) = acc[p][j][mt];
  __syncthreads();
  if (tid >= 64 * MT) return;
  // thread (token tile = wave, lane): columns n0 + 4 CT kq .. + 4 CT - 1 of token 16 * wave + c
  const int m = m0 + 16 * wave + c;
  if (m >= a.M) return;
  const int oc = n0 + 4 * CT * kq;
  float v[NP][4 * CT];
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      f32x4 sum = *reinterpret_cast<const f32x4*>(red[0][wave][p * CT + j][lane]);
#pragma unroll
      for (int w = 1; w < NW; ++w) sum += *reinterpret_cast<const f32x4*>(red[w][wave][p * CT + j][lane]);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[p][CT * i + j] = sum[i];
    }
  uint32_t y[NP][2 * CT];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    if (P[p].bias) {
#pragma unroll
      for (int i = 0; i < 2 * CT; ++i) {
        const uint32_t b = *reinterpret_cast<const uint32_t*>(P[p].bias + oc + 2 * i);
        v[p][2 * i] += unpack_lo<T>(b);
        v[p][2 * i + 1] += unpack_hi<T>(b);
      }
    }
#pragma unroll
    for (int i = 0; i < 2 * CT; ++i) y[p][i] = pack2<T>(v[p][2 * i], v[p][2 * i + 1]);
  }
  auto store = [&](uint16_t* dst, const uint32_t(&o)[2 * CT]) {
    if constexpr (CT == 1)
      *reinterpret_cast<u32x2*>(dst) = u32x2{o[0], o[1]};
    else
      *reinterpret_cast<u32x4*>(dst) = u32x4{o[0], o[1], o[2], o[3]};
  };
#pragma unroll
  for (int p = 0; p < NP; ++p)
    if (P[p].Y) store(P[p].Y + (size_t)m * P[p].ldy + oc, y[p]);
  if constexpr (NP == 2) {  // f = RNE(e * sigmoid(e)) on the rounded e; h = RNE(f * g) on the rounded g
    uint32_t h[2 * CT];
#pragma unroll
    for (int i = 0; i < 2 * CT; ++i) {
      const float e0 = unpack_lo<T>(y[0][i]), e1 = unpack_hi<T>(y[0][i]);
      const uint32_t fv = pack2<T>(e0 * sigmoidf_(e0), e1 * sigmoidf_(e1));
      h[i] = pack2<T>(unpack_lo<T>(fv) * unpack_lo<T>(y[1][i]), unpack_hi<T>(fv) * unpack_hi<T>(y[1][i]));
    }
    store(a.H + (size_t)m * a.ldh + oc, h);
  }
}

// U = Xd A^T of every projection, as fp32 sums of `n_ranges` ranges of K that the kernel above adds in index order and
// rounds once; slices and order of sums are lora_down_kernel's.  blockIdx.x: range; blockIdx.y: 16 ranks of one projection; blockIdx.z: 64 tokens.  A is read in the
// parameters' own type, so that a pass without a backward packs nothing.
template <typename T>
__global__ __launch_bounds__(64 * FEW_DOWN_NW) void lora_down_few_kernel(const FewArgs a) {
  constexpr int MT = 4;
  __shared__ __attribute__((aligned(16))) float red[FEW_DOWN_NW][MT][64][4];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c = lane & 15, kq = lane >> 4;
  int p = 0, rt = blockIdx.y;
  const int t0 = (a.p[0].r + 15) / 16, t1 = (a.p[1].r + 15) / 16;
  if (rt >= t0) { rt -= t0; p = 1; }
  if (p == 1 && rt >= t1) { rt -= t1; p = 2; }
  const FewProjDev P = few_proj(a, p);
  const int j = 16 * rt + c;  // the lane's rank
  const bool f32 = P.param_dtype == FMSA_F32;
  const int m0 = blockIdx.z * (16 * MT), n_mt = (min(16 * MT, a.M - m0) + 15) / 16;
  // slices in units of 32 columns
  const int n32 = (a.K + 31) / 32, slice = blockIdx.x * FEW_DOWN_NW + wave, n_slices = a.n_ranges * FEW_DOWN_NW;
  const int per = (n32 + n_slices - 1) / n_slices;
  const int c_begin = min(a.K, slice * per * 32), c_end = min(a.K, (slice + 1) * per * 32);
  f32x4 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = c_begin + 8 * kq; k < c_end; k += 32) {  // K % 32 == 0: the four quarters of a wave leave together
    u32x4 af = {0u, 0u, 0u, 0u};
    if (j < P.r) af = few_params<T>(P.A, (size_t)j * a.K + k, f32);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if (mt >= n_mt) continue;
      const int m = m0 + 16 * mt + c;
      u32x4 xf = {0u, 0u, 0u, 0u};
      if (m < a.M) xf = *reinterpret_cast<const u32x4*>(a.Xd + (size_t)m * a.ldxd + k);
      acc[mt] = mfma16<T>(xf, af, acc[mt]);  // D[i = token][j = rank]
    }
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) *reinterpret_cast<f32x4*>(red[wave][mt][lane]) = acc[mt];
  __syncthreads();
  const int mt = wave;  // one token tile per wave
  if (mt >= n_mt) return;
  // in lora_down_kernel's order: upper half of the waves onto the lower, then those
  f32x4 sum;
#pragma unroll
  for (int w = 0; w < FEW_DOWN_NW / 2; ++w) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(red[w][mt][lane]) + *reinterpret_cast<const f32x4*>(red[w + FEW_DOWN_NW / 2][mt][lane]);
    sum = w == 0 ? v : sum + v;
  }
  if (j >= P.r) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + 16 * mt + 4 * kq + i;
    if (m < a.M) a.partial[((size_t)blockIdx.x * a.M + m) * a.r_all + P.u_col + j] = sum[i];
  }
}
static_assert(FEW_DOWN_NW >= 4, "one token tile of the sums per wave");

// Waves, chunks in flight and the waves per SIMD the registers are held to, by token tiles; 4096 x 4096 / gate and up of
// 4096 x 14336, us.  One token tile: 8 waves, two chunks, two workgroups per CU 6.3 / 22.3 (four chunks 6.6 / 23.5; 16 waves
// 7.3 / 35.8; 32 columns a workgroup 8.3).  Two: 8.1 / 31.6 (gate and up with 8 waves 36.4).  Four: 32 columns a workgroup 12.2
// / 41.3 (16 columns: q, k, v of 4096 and 1024 columns 12.5 -> 19.9; gate and up with 8 waves 50.3).
template <typename T, int FMT>
int few_launch(const FewArgs& a, int mt, hipStream_t st) {
  const dim3 grid(a.n_cb * a.n_tb);
#define FEW_K(NP, MT, CT, NW, DEPTH, WPE) \
  hipLaunchKernelGGL((gptq_lora_fwd_few_kernel<T, FMT, NP, MT, CT, NW, DEPTH, WPE>), grid, dim3(64 * NW), 0, st, a)
  if (a.swiglu) {
    if (mt == 1) FEW_K(2, 1, 1, 8, 2, 4);
    else if (mt == 2) FEW_K(2, 2, 1, 4, 4, 4);
    else FEW_K(2, 4, 1, 4, 2, 2);
  } else {
    if (mt == 1) FEW_K(1, 1, 1, 8, 2, 4);
    else if (mt == 2) FEW_K(1, 2, 1, 8, 2, 4);
    else FEW_K(1, 4, 2, 8, 2, 2);
  }
#undef FEW_K
  FMSA_CHECK_LAUNCH();
  return FMSA_OK;
}

FewProjDev few_weight(const fmsa_gptq_weight& w) {
  FewProjDev d{};
  d.qweight = w.qweight;
  d.scales = w.scales;
  d.qzeros = w.qzeros;
  d.code = w.code;
  d.block_scale = w.block_scale;
  d.N = w.N;
  d.zero_offset = w.zero_offset;
  // ceil(2^32 / d): exact for chunk * d < 2^32
  const uint64_t per_group = w.group_size / FEW_BK;
  d.group_magic = per_group == 1 ? 0u : (uint32_t)((0x100000000ull + per_group - 1) / per_group);
  return d;
}

int few_gemm(FewArgs& a, const fmsa_gptq_weight& w0, int n_proj, int mode, int act_dtype, hipStream_t st) {
  const int mt = a.M <= 16 ? 1 : (a.M <= 32 ? 2 : 4);
  const int ct = (mt == 4 && mode != FMSA_FWD_SWIGLU) ? 2 : 1;
  a.swiglu = mode == FMSA_FWD_SWIGLU;
  int nb = 0;
  for (int p = 0; p < 3; ++p) {
    a.nblk_start[p] = p < n_proj ? nb : 0x7fffffff;
    if (p < n_proj) nb += a.p[p].N / (16 * ct);
  }
  a.n_cb = a.swiglu ? a.p[0].N / (16 * ct) : nb;
  a.n_tb = (a.M + 16 * mt - 1) / (16 * mt);
  const bool codebook = w0.format == FMSA_WEIGHT_CODEBOOK;
  if (act_dtype == FMSA_BF16) return codebook ? few_launch<bf16_t, 2>(a, mt, st) : few_launch<bf16_t, 0>(a, mt, st);
  if (codebook) return few_launch<f16_t, 2>(a, mt, st);
  return w0.nibble_order == 1 ? few_launch<f16_t, 1>(a, mt, st) : few_launch<f16_t, 0>(a, mt, st);
}

}  // namespace

// Estimate of a launch, us.  Up to 64 tokens it is always the faster one (measured above); beyond, in token blocks of 64, a
// linear launch goes in whole rounds of one workgroup per CU (4096 columns and K: 12.2 us at 64 and 12.8 at 128 tokens, one
// round; 21.7 and 22.4 at 192 and 256, two; 2048 -> 2048 8.0 to 8.7 from 64 to 256 tokens; 14336 -> 4096 28 to 30 a round),
// two workgroups with the SwiGLU per CU share it more evenly (4096 -> 14336: 43, 72, 101, 130 us at 64, 128, 192, 256 tokens);
// from a code book 4 to 10 % more.
float few_us(const fmsa_fwd_proj* projs, int n_proj, int M, int mode) {
  if (M <= 64) return 0.f;
  const bool codebook = projs[0].w.format == FMSA_WEIGHT_CODEBOOK;
  const float k = (float)projs[0].w.K, tb = (float)((M + 63) / 64);
  if (mode == FMSA_FWD_SWIGLU) {
    const float rounds = projs[0].w.N / 16 * tb / 512.f;
    return 4.f + 0.0022f * k + rounds * (4.f + 0.0031f * k) * (codebook ? 1.08f : 1.f);
  }
  int cols = 0;
  for (int p = 0; p < n_proj; ++p) cols += projs[p].w.N;
  const int rounds = (int)((cols / 32 * tb + 255.f) / 256.f);
  return 2.5f + rounds * (1.9f + 0.00185f * k * (codebook ? 1.08f : 1.f));
}

// U given (in the activation type), adapters packed.
int launch_gptq_lora_fwd_few(const fmsa_fwd_proj* projs, int n_proj, const void* X, int64_t ldx, int M, int mode, void* H, int64_t ldh,
                             int act_dtype, hipStream_t st) {
  FewArgs a{};
  a.X = (const uint16_t*)X;
  a.ldx = ldx;
  a.M = M;
  a.K = projs[0].w.K;
  a.H = (uint16_t*)H;
  a.ldh = ldh;
  for (int p = 0; p < n_proj; ++p) {
    const fmsa_fwd_proj& s = projs[p];
    FewProjDev& d = a.p[p];
    d = few_weight(s.w);
    d.U = (const uint16_t*)s.U;
    d.ldu = s.ldu;
    d.B = s.B;
    d.bias = (const uint16_t*)s.bias;
    d.Y = (uint16_t*)s.Y;
    d.ldy = s.ldy;
    d.r = s.r;
    d.s = s.s;
    d.param_dtype = act_dtype;
  }
  return few_gemm(a, projs[0].w, n_proj, mode, act_dtype, st);
}

// Ranges of K of the rank-r products: those that the same call takes over packed adapters (one lora_down of the stacked
// adapters, one batched launch of them, a single one), so that U comes out the same to the last bit.
static int few_ranges(const fmsa_few_proj* projs, int n_proj, int M) {
  int r_all = 0, live = 0;
  for (int p = 0; p < n_proj; ++p) {
    r_all += projs[p].r;
    live += projs[p].r > 0;
  }
  const bool stacked = live == n_proj && n_proj > 1 && r_all <= 128;
  return lora_down_few_splits(M, projs[0].w.K, r_all, stacked ? 1 : live);
}

size_t lora_few_workspace(const fmsa_few_proj* projs, int n_proj, int M) {
  size_t r_all = 0;
  for (int p = 0; p < n_proj; ++p) r_all += projs[p].r;
  return r_all * M * 4 * few_ranges(projs, n_proj, M);
}

// U and Y from the parameters themselves: two launches, one without adapters.
int launch_lora_few(const fmsa_few_proj* projs, int n_proj, const void* X, int64_t ldx, int M, int mode, void* H, int64_t ldh,
                    int act_dtype, void* workspace, hipStream_t st) {
  FewArgs a{};
  a.X = a.Xd = (const uint16_t*)X;
  a.ldx = a.ldxd = ldx;
  a.M = M;
  a.K = projs[0].w.K;
  a.H = (uint16_t*)H;
  a.ldh = ldh;
  a.partial = (float*)workspace;
  a.n_ranges = few_ranges(projs, n_proj, M);
  int tiles = 0;
  for (int p = 0; p < n_proj; ++p) {
    const fmsa_few_proj& s = projs[p];
    FewProjDev& d = a.p[p];
    d = few_weight(s.w);
    d.A = s.A;
    d.B = s.B;
    d.bias = (const uint16_t*)s.bias;
    d.Y = (uint16_t*)s.Y;
    d.ldy = s.ldy;
    d.r = s.r;
    d.s = s.s;
    d.param_dtype = s.param_dtype;
    d.u_col = a.r_all;
    a.r_all += s.r;
    tiles += (s.r + 15) / 16;
  }
  if (tiles > 0) {
    const dim3 grid(a.n_ranges, tiles, (M + 63) / 64), block(64 * FEW_DOWN_NW);
    if (act_dtype == FMSA_BF16) hipLaunchKernelGGL((lora_down_few_kernel<bf16_t>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((lora_down_few_kernel<f16_t>), grid, block, 0, st, a);
    FMSA_CHECK_LAUNCH();
  }
  return few_gemm(a, projs[0].w, n_proj, mode, act_dtype, st);
}

// Tiled (prefill) GEMM for bf16 activations x 4-bit weights (W4A16: codes
// two per byte with the even k in the low nibble; MXFP4: e2m1 + one e8m0
// scale per 32 k; NVFP4: e2m1 + one bf16 scale per 16 k; INT4: offset-binary
// integers + one bf16 scale per 32 / 64 / 128 k), dense or grouped.
//
// Restates the reference's W4A16 path (`layers/adapter/linear_common.py:
// 188-209` -> `kernels/megablox/gmm_v2.py:452-462`: blocks below 256 k are
// dequantized to the activation dtype and multiplied in bf16 with f32
// accumulation). Expanding the codes on the fly gives the same bf16 weights
// as dequantizing the whole matrix first: exact for e8m0 scales, one
// round-to-nearest-even of value * scale for the bf16 NVFP4 / INT4 scales.
//
// Design for gfx950 (w4_gemm_kernel):
//  * output tile BM tokens x 256 weight rows of 32 x 32 MFMA blocks (weight
//    block first, activation block second: v_mfma_f32_32x32x16_bf16). Each of
//    4 wavefronts owns 64 weight rows for all BM tokens, so it expands its
//    rows once; two workgroups share a CU (80 KB of LDS, 256 VGPRs), or
//    two K groups of 4 wavefronts share a workgroup (KG 2) where the tiles
//    only fill one workgroup per CU: one wavefront's instructions issue in
//    order, and it takes a second one to put the expansion of one beside the
//    MFMAs of the other;
//  * what bounds it: from ~1000 tokens the expansion, the MFMAs and the copies
//    into LDS, which overlap in part only (K 2880, N 5760, 4096 / 8192 tokens
//    133 / 258 us, 1.05 PFLOP/s; MFMAs busy 41 % of the SIMDs' cycles); a
//    routed expert's few rows, the weight stream as well (GPT-OSS MoE, 512 /
//    2048 tokens 794 / 1112 us in 64-byte pieces -> 457 / 654 us; its gate_up
//    fetches 1.36 GB for 1.13 GB of codes and scales);
//  * a wavefront's codes are copied as whole 128-byte lines of its own rows
//    (256 k, four stages) into its own LDS rows and from there into
//    registers at the start of the line, which frees the buffer for the next
//    line: 64 KB per CU stay in flight. 64-byte pieces of rows of 1440 bytes
//    touch a line more often than it stays in the L2. A wavefront owns every
//    fourth row of the tile, whose lines start at the same place (see `ph`);
//  * activations: stages of 64 k (128 bytes of each row) in a ring of three
//    sets, copied two sets ahead, one barrier per set;
//  * in a stage, lane l (row l % 32, half h = l / 32) feeds k in
//    [32h, 32h + 32): that is one e8m0 block (two NVFP4 blocks), 16
//    contiguous code bytes and one scale byte (NVFP4: one 4-byte bf16 pair;
//    INT4: one bf16 group scale). Each 16-k step expands 8 codes to bf16 with
//    the scale applied (v_cvt_scalef32_pk_bf16_fp4 for e8m0; unscaled
//    conversion, f32 product and bf16 rounding for NVFP4 and INT4);
//    activation and weight use the same lane -> k assignment, so the
//    products pair up whatever order the MFMA sums;
//  * LDS rows of 128 bytes hold the 16-byte chunk c of row r at slot
//    c ^ ((r & 7) ^ ((r >> 3) & 1)), so that the operand reads are
//    conflict-free;
//  * the epilogue applies bias, fused activation and routing weight (the
//    weights carry no other scale).

#include <algorithm>
#include <cstdlib>

#include "gemm_tile.h"

namespace {

using rsrc_t = __amdgpu_buffer_rsrc_t;
constexpr int kW4BN = 256;  // weight rows per tile

__device__ __forceinline__ int w4_swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// 8 e2m1 codes (one dword, low nibble first) -> 8 bf16 times `scale`
__device__ __forceinline__ bf16x8 w4_expand(uint32_t d, float scale) {
  union {
    bf16x2 h[4];
    bf16x8 v;
  } u;
  u.h[0] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, scale, 0);
  u.h[1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, scale, 1);
  u.h[2] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, scale, 2);
  u.h[3] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, scale, 3);
  return u.v;
}

__device__ __forceinline__ bf16x8 as_bf16x8_u4(const uint4& x) {
  union {
    uint4 u;
    bf16x8 v;
  } c;
  c.u = x;
  return c.v;
}

// FMT: 0 MXFP4, 1 NVFP4, 2 INT4
template <int BM, int KG, bool ACT, int FMT>
__global__ __launch_bounds__(KG * kThreads, 2) void w4_gemm_kernel(const GemmParams p, int m_tiles, int n_tiles) {
  constexpr bool NV = FMT == 1, I4 = FMT == 2;
  constexpr int BN = kW4BN;
  constexpr int NI = 2, MJ = BM / 32;     // 32-row weight blocks, 32-token blocks per wavefront
  constexpr int BNO = ACT ? BN / 2 : BN;  // output channels per tile
  constexpr int PB = BM >= 128 ? 1 : 2;  // 64-k stages per barrier
  constexpr int NT = KG * kThreads;
  constexpr int RING = 3;                 // sets of PB activation stages in LDS
  constexpr int SB = BM * 128;            // bytes of a stage
  constexpr int AB = PB * SB;             // bytes of a set
  constexpr int WB = 64 * 128;            // bytes of a wavefront's code lines

  // per K group: codes [4 wavefronts][64 rows][128 B], activations
  // [RING][PB][BM][128 B]: 80 KB with KG 1, so that two workgroups share a CU
  constexpr int GB = 4 * WB + RING * AB;
  __shared__ __align__(1024) uint8_t smem_all[KG * GB];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3;
  const int kgrp = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 8);
  uint8_t* const smem = smem_all + kgrp * GB;
  uint8_t* const sX = smem + 4 * WB;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem_all + kgrp * GB;

  int g, row0, rows, ntile;
  if (p.group_offs) {
    if (!tile_group_xcd<BM>(p, blockIdx.x, n_tiles, g, row0, rows, ntile, reinterpret_cast<int*>(smem_all))) return;
    __syncthreads();  // the group has been read everywhere: the buffers are free
  } else {
    int mt;
    if (!tile_dense(blockIdx.x, m_tiles, n_tiles, mt, ntile)) return;
    g = 0;
    row0 = mt * BM;
    rows = min(BM, p.M - row0);
  }
  g = __builtin_amdgcn_readfirstlane(g);
  const int n0 = ntile * BNO;
  const int nlim = ACT ? p.N / 2 : p.N;
  // global weight row of tile row r (gate rows, then up rows with ACT); rows
  // past the end are clamped (their outputs are never stored)
  auto wrow_global = [&](int r) {
    if (ACT) return (r < BN / 2 ? 0 : p.N / 2) + min(n0 + (r % (BN / 2)), nlim - 1);
    return min(n0 + r, nlim - 1);
  };
  // tile row of this wavefront's row m of weight block i
  auto wrow = [&](int i, int m) { return i * (BN / 2) + 4 * m + wave; };

  // epilogue inputs (loaded now, staged in LDS at the end): token routing
  // weight and output row; weight-row bias
  float e_rw = 1.0f, e_bs = 0.0f;
  int e_yr = 0;
  if (tid < BM) {
    const int R = row0 + min(tid, rows - 1);
    if (p.row_weight) e_rw = bf16_to_f32(p.row_weight[R]);
    e_yr = p.y_rows ? p.y_rows[R] : R;
  }
  if (tid < BN && p.bias) e_bs = p.bias[(int64_t)g * p.bias_gstride + wrow_global(tid)];

  // split-K: the workgroup's stages of 64 k; its K groups take consecutive parts
  const int NU = p.K / 64;
  int u0 = (int)((int64_t)NU * blockIdx.z / p.ksplit);
  int KS = (int)((int64_t)NU * (blockIdx.z + 1) / p.ksplit) - u0;
  const int sets = cdiv(cdiv(KS, KG), PB);  // barriers that every K group reaches
  if constexpr (KG == 2) {
    const int h = (KS + 1) / 2;
    u0 += kgrp * h;
    KS = kgrp ? KS - h : h;
  }

  // ---- activation copies: one instruction = 8 rows x 128 bytes (lane -> row
  // l >> 3, slot l & 7; the slot of chunk c of row r is c ^ w4_swz(r))
  constexpr int XI = BM / 32;  // per wavefront and stage; copy j covers rows 32 j .. 32 j + 31
  const uint8_t* xp[XI];
#pragma unroll
  for (int j = 0; j < XI; ++j) {
    const int r = (wave + 4 * j) * 8 + (lane >> 3);
    const int R = row0 + min(r, rows - 1);
    const int ar = p.a_rows ? p.a_rows[R] : R;
    xp[j] = static_cast<const uint8_t*>(p.a) + (uint64_t)(uint32_t)ar * ((uint64_t)p.lda * 2) +
            (uint32_t)(((lane & 7) ^ w4_swz(r)) * 16 + u0 * 128);
  }
  const uint32_t xdst = lds0 + 4 * WB + wave * 1024;

  // ---- code copies: whole 128-byte lines (256 k) of the wavefront's own 64
  // rows, 8 rows per instruction. Row bytes are K / 2, any multiple of 32, so
  // consecutive rows start at up to four different places of a line (phases
  // of 32 bytes); rows four apart share one, and a wavefront owns every
  // fourth row. Stage s of the wavefront is quarter (s + ph) % 4 of its line
  // (s + ph) / 4.
  const uint8_t* wbase = p.w + (int64_t)g * p.w_gstride;
  const int rowb = p.K / 2;
  const int ph = __builtin_amdgcn_readfirstlane(
      (int)((((uint64_t)reinterpret_cast<uintptr_t>(wbase) + (uint64_t)(uint32_t)wrow_global(wrow(0, 0)) * (uint64_t)p.ldw) >> 5) +
            (uint64_t)u0) & 3);
  constexpr int WI = 8;
  uint32_t roff[WI];
#pragma unroll
  for (int j = 0; j < WI; ++j)
    roff[j] = (uint32_t)wrow_global(wrow(j / 4, (j % 4) * 8 + (lane >> 3))) * (uint32_t)p.ldw;
  const int wc16 = ((lane & 7) ^ (lane >> 3)) * 16;  // chunk of even j (odd j: the neighbour)
  const uint32_t wdst = lds0 + wave * WB;
  auto copy_line = [&](int q) {  // line q of the slice, clamped to the rows
    const int b = (u0 - ph) * 32 + q * 128;
    const uint32_t b0 = (uint32_t)min(max(b + wc16, 0), rowb - 16);
    const uint32_t b1 = (uint32_t)min(max(b + (wc16 ^ 16), 0), rowb - 16);
#pragma unroll
    for (int j = 0; j < WI; ++j) lds_copy16(wbase, roff[j] + (j & 1 ? b1 : b0), wdst + j * 1024);
  };

  // ---- weight scales: lane (row l % 32, half h) of weight block i needs, for
  // stage u, e8m0 byte 2 u + h of its row; NVFP4: the bf16 pair 4 u + 2 h;
  // INT4: the bf16 scale of k 64 u + 32 h. Loaded for the four stages of a line.
  constexpr int kSB = NV || I4 ? 2 : 1;  // bytes per scale
  constexpr int SW = NV || I4 ? 4 : 2;   // registers per weight block and line
  const rsrc_t eres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<void*>(static_cast<const void*>(static_cast<const uint8_t*>(p.w_scale) + (int64_t)g * p.ws_gstride * kSB)),
      (short)0, (int)std::min<int64_t>((int64_t)p.N * p.ldws * kSB, 0x7fffffff), 0x00020000);
  const int rl = lane & 31, kh = lane >> 5;
  uint32_t eoff[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i)
    eoff[i] = (uint32_t)wrow_global(wrow(i, rl)) * (uint32_t)(p.ldws * kSB) + (NV ? kh * 4 : 0);
  const int lg = I4 ? (p.wq_group == 32 ? 5 : (p.wq_group == 64 ? 6 : 7)) : 0;  // log2(group)
  constexpr int NSC = NI * (NV || I4 ? 4 : 2);  // loads
  uint32_t we[NI][SW], wn[NI][SW];  // the line in use and the next one
  // scales of stages s .. s + 3 of the slice (those past the end of K: of a
  // valid stage or zero, for no product). Every call makes NSC loads.
  auto load_scales = [&](int s) {
    const int u = u0 + s;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if constexpr (NV) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          wn[i][k] = __builtin_amdgcn_raw_buffer_load_b32(eres, eoff[i], (uint32_t)min(u + k, NU - 1) * 8u, 0);
      } else if constexpr (I4) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const uint32_t k0 = (uint32_t)min(u + k, NU - 1) * 64u + (uint32_t)kh * 32u;
          wn[i][k] = __builtin_amdgcn_raw_buffer_load_b16(eres, eoff[i] + (k0 >> lg) * 2u, 0, 0);
        }
      } else {
        // pairs of stages: 4 bytes, the last stage of an odd K / 64 2 bytes
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int v = min(u + 2 * k, NU - 1);
          if (v + 1 < NU) wn[i][k] = __builtin_amdgcn_raw_buffer_load_b32(eres, eoff[i], (uint32_t)v * 2u, 0);
          else wn[i][k] = __builtin_amdgcn_raw_buffer_load_b16(eres, eoff[i], (uint32_t)v * 2u, 0);
        }
      }
    }
  };

  f32x16 acc[NI][MJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  // The K pipeline over the first MJE 32-token blocks of the tile (MJ: all
  // of them); the accumulators of the others keep their zeros.
  auto pipeline = [&](auto mje_c) {
    constexpr int MJE = decltype(mje_c)::value;
    constexpr int XC = PB * MJE;  // copies per set
    auto copy_x = [&](int ks, int buf) {  // the set of stages ks .. ks + PB - 1
#pragma unroll
      for (int h = 0; h < PB; ++h)
#pragma unroll
        for (int j = 0; j < MJE; ++j)
          lds_copy16(xp[j] + min(ks + h, KS - 1) * 128, xdst + buf * AB + h * SB + j * 4096);
    };
    uint4 wc[4][NI];  // codes of a line's four stages
    auto read_line = [&]() {
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const int r = i * 32 + rl;
          wc[k][i] = *reinterpret_cast<const uint4*>(smem + wave * WB + r * 128 + (((2 * k + kh) ^ w4_swz(r)) * 16));
        }
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the codes are in registers
    };
    if (KS <= 0) return;
    const int last_line = (KS - 1 + ph) >> 2;
    load_scales(0);
    copy_line(0);
    copy_x(0, 0);
    if (KS > PB) copy_x(PB, 1);
    wait_copies_upto<0>();
    asm volatile("" ::: "memory");
    // the first line starts in quarter ph: its scales move to their quarters
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if constexpr (NV || I4) {
        const uint32_t e0 = wn[i][0], e1 = wn[i][1], e2 = wn[i][2];
        if (ph == 1) wn[i][1] = e0, wn[i][2] = e1, wn[i][3] = e2;
        else if (ph == 2) wn[i][2] = e0, wn[i][3] = e1;
        else if (ph == 3) wn[i][3] = e0;
      } else {
        const uint64_t e = ((uint64_t)wn[i][1] << 32 | wn[i][0]) << (16 * ph);
        wn[i][0] = (uint32_t)e;
        wn[i][1] = (uint32_t)(e >> 32);
      }
    }
    int buf = 0;
    // ---- stages. Per set of PB stages: wait for its activations (the next
    // set's, and a line and scales copied meanwhile, stay in flight) ->
    // barrier: they have landed everywhere, and everybody is done with the
    // previous set -> copy the set after the next into its buffer. At the
    // start of a line the wavefront takes its codes into registers, which
    // frees the line buffer for the next line, four stages ahead of its use:
    // what a workgroup has in flight from memory sets the rate at which it
    // can stream weights.
    auto stage = [&](auto k_c, int s) __attribute__((always_inline)) {
      constexpr int K4 = decltype(k_c)::value;
      const int line = (s + ph) >> 2;
      const bool first = PB == 1 || !(s & 1);  // of its set
      if (first) {
        // issued after the set's activations: those of the next set, and
        // scales and codes of a line taken since (in this line's first stage)
        if (s > 0) {
          if (s + PB >= KS) wait_copies_upto<0>();
          else if (K4 != 0 && (PB == 2 || K4 == 1 || s == 1) && line < last_line)
            wait_copies_upto<XC + NSC + WI>();
          else wait_copies_upto<XC>();
        }
        stage_barrier();
      } else if (K4 == 0) {
        // a line that starts inside a set: two sets' activations were copied after it
        if (s + 3 >= KS) wait_copies_upto<0>();
        else if (s == 1) wait_copies_upto<XC>();
        else wait_copies_upto<2 * XC>();
        asm volatile("" ::: "memory");
      }
      if (K4 == 0 || s == 0) {
        read_line();
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int k = 0; k < SW; ++k) we[i][k] = wn[i][k];
        if (line < last_line) {
          load_scales(4 * (line + 1) - ph);
          asm volatile("" ::: "memory");
          copy_line(line + 1);
        }
      }
      if (first && s + 2 * PB < KS) copy_x(s + 2 * PB, buf == 0 ? 2 : buf - 1);
      const uint8_t* sA = sX + buf * AB + (first ? 0 : SB);
      if (PB == 1 || !first) buf = buf == 2 ? 0 : buf + 1;

      float scale[NI], scale1[NI];
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        if constexpr (NV) {  // scale for 16-k steps 0-1, scale1 for 2-3
          scale[i] = bits_f32(we[i][K4] << 16);
          scale1[i] = bits_f32(we[i][K4] & 0xffff0000u);
        } else if constexpr (I4) {
          scale[i] = bits_f32(we[i][K4] << 16);
        } else {
          scale[i] = e8m0_to_f32(we[i][K4 / 2] >> ((K4 & 1) * 16 + 8 * kh));
        }
      }
      uint4 xa[2][MJE];
      auto read_x = [&](int q) {
#pragma unroll
        for (int j = 0; j < MJE; ++j) {
          const int r = j * 32 + rl;
          xa[q & 1][j] = *reinterpret_cast<const uint4*>(sA + r * 128 + (((kh * 4 + q) ^ w4_swz(r)) * 16));
        }
      };
      read_x(0);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (q < 3) read_x(q + 1);
        bf16x8 wv[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          // dword q of the lane's 16 code bytes feeds 16-k step q
          const uint4 c4 = wc[K4][i];
          const uint32_t d = q == 0 ? c4.x : (q == 1 ? c4.y : (q == 2 ? c4.z : c4.w));
          if constexpr (NV) wv[i] = as_bf16x8_u4(nvfp4x8_to_bf16(d, q < 2 ? scale[i] : scale1[i]));
          else if constexpr (I4) wv[i] = as_bf16x8_u4(int4x8_to_bf16(d, scale[i]));
          else wv[i] = w4_expand(d, scale[i]);
        }
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < MJE; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv[i], as_bf16x8_u4(xa[q & 1][j]), acc[i][j], 0, 0, 0);
      }
    };
    for (int s = -ph; s < KS; s += 4) {
      if (s >= 0) stage(std::integral_constant<int, 0>{}, s);
      if (s + 1 >= 0 && s + 1 < KS) stage(std::integral_constant<int, 1>{}, s + 1);
      if (s + 2 >= 0 && s + 2 < KS) stage(std::integral_constant<int, 2>{}, s + 2);
      if (s + 3 >= 0 && s + 3 < KS) stage(std::integral_constant<int, 3>{}, s + 3);
    }
  };
  // A tile with few valid tokens -- a routed expert's last tile -- copies and
  // multiplies its occupied 32-token blocks only.
  const int rows_u = __builtin_amdgcn_readfirstlane(rows);
  if constexpr (MJ == 4) {
    if (rows_u <= 32) pipeline(std::integral_constant<int, 1>{});
    else if (rows_u <= 64) pipeline(std::integral_constant<int, 2>{});
    else if (rows_u <= 96) pipeline(std::integral_constant<int, 3>{});
    else pipeline(std::integral_constant<int, 4>{});
  } else if constexpr (MJ == 2) {
    if (rows_u <= 32) pipeline(std::integral_constant<int, 1>{});
    else pipeline(std::integral_constant<int, 2>{});
  } else {
    pipeline(std::integral_constant<int, MJ>{});
  }

  if constexpr (KG == 2)
    for (int b = cdiv(KS, PB); b < sets; ++b) stage_barrier();

  // ---- epilogue: per 32-token block, the workgroup's f32 sums in LDS
  // ([32 tokens][256 tile rows], row n of token t at n ^ 4 (t % 16); the
  // second K group adds to the first's), then 8 output channels of a token
  // per thread
  __syncthreads();  // every wavefront is done with the stage buffers
  float* reg = reinterpret_cast<float*>(smem_all);
  float* s_rw = reinterpret_cast<float*>(smem_all + 4 * WB);
  float* s_bs = s_rw + BM;
  int* s_yr = reinterpret_cast<int*>(s_bs + BN);
  static_assert(32 * BN * 4 <= 4 * WB && (2 * BM + BN) * 4 <= RING * AB, "epilogue regions");
  if (tid < BM) {
    s_rw[tid] = e_rw;
    s_yr[tid] = e_yr;
  }
  if (tid < BN) s_bs[tid] = e_bs;
#pragma unroll
  for (int j = 0; j < MJ; ++j) {
    if (j * 32 >= rows_u) break;
    if (j) __syncthreads();  // the previous block has been read
#pragma unroll
    for (int kk = 0; kk < KG; ++kk) {
      if (kgrp == kk) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int m = 8 * (r / 4) + 4 * kh + (r % 4);  // MFMA row of register r
            float& d = reg[rl * BN + (wrow(i, m) ^ (4 * (rl & 15)))];
            d = kk ? d + acc[i][j][r] : acc[i][j][r];
          }
      }
      __syncthreads();
    }
    if (p.ksplit > 1) {
      // raw sums to the f32 workspace [ksplit][M][N]; the finishing kernel
      // adds the slices in order and runs the epilogue
      float* plane = p.partial + (int64_t)blockIdx.z * p.M * p.N;
      for (int e = tid; e < 32 * BN / 4; e += NT) {
        const int t = e / (BN / 4), r = (e % (BN / 4)) * 4;
        const int tr = j * 32 + t;
        const int c = n0 + (ACT ? r % (BN / 2) : r);  // output channel of the quad
        if (tr >= rows || c >= nlim) continue;
        const float4 v = tile_quad<BN>(reg, t, r);
        float* dst = plane + (int64_t)(row0 + tr) * p.N + (ACT && r >= BN / 2 ? p.N / 2 : 0) + c;
        if (c + 4 <= nlim && (p.N & 3) == 0 && (!ACT || (p.N & 7) == 0)) {
          *reinterpret_cast<float4*>(dst) = v;
        } else {
          const float f[4] = {v.x, v.y, v.z, v.w};
          for (int k = 0; k < 4 && c + k < nlim; ++k) dst[k] = f[k];
        }
      }
      continue;
    }
    tile_finish_rows<32, NT, BN, ACT, false>(p, reg, tid, j * 32, rows, n0, nlim, s_rw, s_bs, nullptr, s_yr);
  }
}

// The wavefronts split the 256 weight rows (each expands its own 64 rows
// once per stage and reuses them for all BM tokens); WN = 4 always.
template <int BM>
struct W4Shape {
  static constexpr int WN = 4;                  // wavefronts along weight rows
  static constexpr int WM = 1;                  // along tokens
  static constexpr int TN = kW4BN / WN;         // weight rows per wavefront
  static constexpr int TM = BM / WM;            // tokens per wavefront
  static constexpr int NI = TN / 32;
  static constexpr int MJ = TM / 32;
  static_assert(NI >= 1 && MJ >= 1, "tile too small");
};

// Under-filled dense problems of the costlier formats (1 NVFP4, 2 INT4;
// w4_plan_dense has the rule): one workgroup per tile whose stages of 64 k --
// activations, codes and scales alike -- run through a ring of four, copied
// four stages ahead, with the operand reads and copies of a stage spread
// over its MFMAs. It spends fewer instructions per stage than the line
// pipeline above, and with one workgroup per CU that is what counts: NVFP4 K
// 2880, N 5760 at 128 / 203 tokens 22.6 / 27.7 us against 26.0 / 32.0. What
// bounds it are the chains of a stage -- waits, barrier, operand reads, about
// 180 vector instructions of expansion and few MFMAs (203 tokens: vector ALU
// busy 23 % of the wave-cycles, MFMAs 7 % of the SIMDs'): two K groups of four
// wavefronts (KG 2, their sums added through LDS) take 0.84 us per stage of
// each, one alone 0.50.
template <int BM, int KG, bool ACT, int FMT>
__global__ __launch_bounds__(KG * kThreads) void w4_ring_kernel(const GemmParams p, int m_tiles, int n_tiles) {
  constexpr bool NV = FMT == 1, I4 = FMT == 2;
  using S = W4Shape<BM>;
  constexpr int BN = kW4BN;
  constexpr int NI = S::NI, MJ = S::MJ, TN = S::TN, TM = S::TM;
  constexpr int BNO = ACT ? BN / 2 : BN;  // output channels per tile
  static_assert(!ACT || NI % 2 == 0, "fused activation pairs gate and up blocks");

  // four LDS stages of 64 k per K group: activations [BM][128 B], codes [BN][32 B]
  constexpr int AB = BM * 128, WB = BN * 32;
  __shared__ __align__(1024) uint8_t sA0s[KG * AB], sA1s[KG * AB], sA2s[KG * AB], sA3s[KG * AB];
  __shared__ __align__(1024) uint8_t sW0s[KG * WB], sW1s[KG * WB], sW2s[KG * WB], sW3s[KG * WB];
  __shared__ float s_sx[BM], s_rw[BM], s_ws[BN], s_bs[BN];
  __shared__ int s_yr[BM];

  // K group of the wavefront; threads and wavefronts count within the group
  const int kg = KG > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / kThreads) : 0;
  const int tid = KG > 1 ? (int)threadIdx.x % kThreads : (int)threadIdx.x;
  uint8_t *sA0 = sA0s + kg * AB, *sA1 = sA1s + kg * AB, *sA2 = sA2s + kg * AB, *sA3 = sA3s + kg * AB;
  uint8_t *sW0 = sW0s + kg * WB, *sW1 = sW1s + kg * WB, *sW2 = sW2s + kg * WB, *sW3 = sW3s + kg * WB;
  const int lane = tid & 63, wave = tid >> 6;
  const int wn = wave % S::WN, wm = wave / S::WN;

  int mt, ntile;
  if (!tile_dense(blockIdx.x, m_tiles, n_tiles, mt, ntile)) return;
  const int row0 = mt * BM, rows = min(BM, p.M - row0);
  const int n0 = ntile * BNO;
  const int nlim = ACT ? p.N / 2 : p.N;
  // global weight row of tile LDS row r (gate rows, then up rows with ACT);
  // rows past the end are clamped (their outputs are never stored)
  auto wrow_global = [&](int r) {
    if (ACT) return (r < BN / 2 ? 0 : p.N / 2) + min(n0 + (r % (BN / 2)), nlim - 1);
    return min(n0 + r, nlim - 1);
  };

  // epilogue inputs (loaded now, staged in LDS at the end): token routing
  // weight and output row; weight-row bias. No activation / channel scales.
  float e_rw = 1.0f, e_bs = 0.0f;
  int e_yr = 0;
  if (tid < BM) {
    const int R = row0 + min(tid, rows - 1);
    if (p.row_weight) e_rw = bf16_to_f32(p.row_weight[R]);
    e_yr = p.y_rows ? p.y_rows[R] : R;
  }
  if (tid < BN && p.bias) e_bs = p.bias[wrow_global(tid)];

  // ---- LDS copies (16 bytes per lane) ----
  // activations: one instruction = 8 rows x 128 bytes (lane -> row l >> 3,
  // slot l & 7, fetching the chunk that the row's swizzle stores there);
  // codes: 32 rows x 32 bytes (lane -> row l >> 1, half l & 1). Scales:
  // lane (row l % 32, half h) of weight block i needs e8m0 byte 2*stage + h
  // of its row (NVFP4: bf16 scales 4*stage + 2h and + 1, one 4-byte load;
  // INT4: bf16 scale (64*stage + 32h) / group).
  static_assert(NV || I4, "bf16 scales");
  constexpr int kSB = 2;  // bytes per scale
  constexpr int XI = BM / 32;  // activation copies per wavefront
  constexpr int WI = 2;        // code copies per wavefront
  const uint8_t* xbase = static_cast<const uint8_t*>(p.a);
  const uint8_t* wbase = p.w;
  const rsrc_t eres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<void*>(static_cast<const void*>(p.w_scale)),
      (short)0, (int)std::min<int64_t>((int64_t)p.N * p.ldws * kSB, 0x7fffffff), 0x00020000);
  const uint64_t lda_b = (uint64_t)p.lda * 2;
  uint32_t xrow[XI], woff[WI];
  int xcx[XI];
#pragma unroll
  for (int j = 0; j < XI; ++j) {
    const int r = (wave + 4 * j) * 8 + (lane >> 3);
    const int R = row0 + min(r, rows - 1);
    xrow[j] = (uint32_t)(p.a_rows ? p.a_rows[R] : R);
    xcx[j] = ((lane & 7) ^ w4_swz(r)) * 16;
  }
#pragma unroll
  for (int j = 0; j < WI; ++j) {
    const int r = (wave + 4 * j) * 32 + (lane >> 1);
    woff[j] = (uint32_t)wrow_global(r) * (uint32_t)p.ldw + (lane & 1) * 16;
  }

  // split-K: this workgroup's K range in 64-k stages, dealt to the K groups
  // (the first may have one stage more: `most`, the others at least `least`)
  const int NU = p.K / 64;
  const int wg0 = (int)((int64_t)NU * blockIdx.z / p.ksplit);
  const int u1 = (int)((int64_t)NU * (blockIdx.z + 1) / p.ksplit);
  const int most = cdiv(u1 - wg0, KG), least = (u1 - wg0) / KG;
  const int u0 = wg0 + kg * most;
  const int KS = kg == 0 ? most : least;
  const int rl = lane & 31, kh = lane >> 5;
  auto wrow = [&](int i) { return tile_wrow<BN, TN, NI, ACT>(wn, i); };
  uint32_t eoff[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i)
    eoff[i] = (uint32_t)wrow_global(wrow(i) + rl) * (uint32_t)(p.ldws * kSB) + (NV ? kh * 4 : 0);
  const int lg = I4 ? (p.wq_group == 32 ? 5 : (p.wq_group == 64 ? 6 : 7)) : 0;  // log2(group)
  uint32_t we[4][NI];  // scales of the stages in flight (stage s in set s % 4)
  auto copy_stage = [&](uint8_t* dA, uint8_t* dW, int e, int ks) {
    // (a group without stages fetches one that it never uses)
    const uint32_t st = (uint32_t)(KG > 1 ? min(u0 + max(ks, 0), NU - 1) : u0 + ks);
#pragma unroll
    for (int j = 0; j < WI; ++j) {
      uint32_t o = woff[j];
      asm volatile("" : "+v"(o));
      __builtin_amdgcn_global_load_lds(wbase + (o + st * 32u), QMOE_LDS(dW + (wave + 4 * j) * 1024), 16, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < XI; ++j) {
      uint32_t r = xrow[j];
      asm volatile("" : "+v"(r));
      const uint8_t* src = xbase + (uint64_t)r * lda_b + (st * 128u + xcx[j]);
      __builtin_amdgcn_global_load_lds(src, QMOE_LDS(dA + (wave + 4 * j) * 1024), 16, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if constexpr (NV) {
        we[e][i] = __builtin_amdgcn_raw_buffer_load_b32(eres, eoff[i], st * 8u, 0);
      } else {
        const uint32_t gi = (st * 64u + (uint32_t)kh * 32u) >> lg;  // group of the lane's 32 k
        we[e][i] = __builtin_amdgcn_raw_buffer_load_b16(eres, eoff[i] + gi * 2u, 0, 0);
      }
    }
  };

  uint4 wc[2][NI];  // codes: dword q feeds 16-k step q
  uint4 xa[2][MJ][4];  // activations: [block][16-k step]
  f32x16 acc[NI][MJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  // The K pipeline over the first MJE 32-token blocks of the tile (MJ: all
  // of them); the accumulators of the others keep their zeros.
  auto pipeline = [&](auto mje_c) {
    constexpr int MJE = decltype(mje_c)::value;
    // ---- operands of one stage into register set t ----
    auto read_stage = [&](const uint8_t* sA, const uint8_t* sW, int t) {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int r = wrow(i) + rl;
        wc[t][i] = *reinterpret_cast<const uint4*>(sW + r * 32 + kh * 16);
      }
#pragma unroll
      for (int j = 0; j < MJE; ++j) {
        const int r = wm * TM + j * 32 + rl;
        const uint8_t* row = sA + r * 128;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          xa[t][j][q] = *reinterpret_cast<const uint4*>(row + (((kh * 4 + q) ^ w4_swz(r)) * 16));
      }
    };

    // k-step outer, blocks inner: consecutive MFMAs go to different
    // accumulators, and a step's expansions overlap the previous step's MFMAs
    auto mma_stage = [&](int t, const uint32_t (&eb)[NI]) {
      float scale[NI], scale1[NI];  // NVFP4: scale for 16-k steps 0-1, scale1 for 2-3
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        if constexpr (NV) {
          scale[i] = bits_f32(eb[i] << 16);
          scale1[i] = bits_f32(eb[i] & 0xffff0000u);
        } else {
          scale[i] = bits_f32(eb[i] << 16);
        }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        bf16x8 wv[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const uint32_t d = q == 0 ? wc[t][i].x : (q == 1 ? wc[t][i].y : (q == 2 ? wc[t][i].z : wc[t][i].w));
          if constexpr (NV) wv[i] = as_bf16x8_u4(nvfp4x8_to_bf16(d, q < 2 ? scale[i] : scale1[i]));
          else wv[i] = as_bf16x8_u4(int4x8_to_bf16(d, scale[i]));
        }
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < MJE; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv[i], as_bf16x8_u4(xa[t][j][q]), acc[i][j], 0, 0, 0);
      }
    };

    constexpr int CPS = WI + XI + NI;        // vector-memory loads per wavefront per stage
    constexpr int NM = NI * MJE * 4;         // MFMAs per stage
    constexpr int NR = NI + MJE * 4;         // LDS operand reads per stage
    // Stage s lives in buffer s % 4 and is copied four stages ahead. Stage s:
    // wait for the own copy of stage s+1 -> barrier (stage s+1 has landed
    // everywhere, and every wavefront holds stage s in registers, so buffer
    // s % 4 is free) -> copy stage s+4 into it -> MFMAs of stage s with the
    // operand reads of stage s+1 among the first half and the copies among
    // the second. Copies past the end refetch the last stage into a consumed
    // buffer (never read again).
    // (stage s's scale bytes are register set s % 4; they are taken before
    // the set is reloaded with stage s+4)
    auto stage = [&](uint8_t* fA, uint8_t* fW, const uint8_t* nA, const uint8_t* nW, int e, int s, int t) {
      wait_copies_upto<2 * CPS>();
      stage_barrier();
      uint32_t eb[NI];
#pragma unroll
      for (int i = 0; i < NI; ++i) eb[i] = we[e][i];
      copy_stage(fA, fW, e, min(s + 4, KS - 1));
      if (KG > 1 && s >= KS) return;  // the other group's last stage
      mma_stage(t, eb);
      read_stage(nA, nW, t ^ 1);
      interleave<0, NM, NR, CPS>();
    };
    if (most > 0) {
      copy_stage(sA0, sW0, 0, 0);
      copy_stage(sA1, sW1, 1, min(1, KS - 1));
      copy_stage(sA2, sW2, 2, min(2, KS - 1));
      copy_stage(sA3, sW3, 3, min(3, KS - 1));
      wait_copies_upto<3 * CPS>();
      __syncthreads();
      read_stage(sA0, sW0, 0);
      int s = 0;
      for (; s + 4 <= least; s += 4) {
        stage(sA0, sW0, sA1, sW1, 0, s, 0);
        stage(sA1, sW1, sA2, sW2, 1, s + 1, 1);
        stage(sA2, sW2, sA3, sW3, 2, s + 2, 0);
        stage(sA3, sW3, sA0, sW0, 3, s + 3, 1);
      }
      if (s < most) stage(sA0, sW0, sA1, sW1, 0, s, 0);
      if (s + 1 < most) stage(sA1, sW1, sA2, sW2, 1, s + 1, 1);
      if (s + 2 < most) stage(sA2, sW2, sA3, sW3, 2, s + 2, 0);
      if (KG > 1 && s + 3 < most) stage(sA3, sW3, sA0, sW0, 3, s + 3, 1);
    }

  };
  // A 64-token tile with at most 32 valid tokens runs the MFMAs of its first
  // 32-token block only: the others' sums belong to no token. The expansion of
  // the weight codes, the copies and the barriers are the same.
  const int rows_u = __builtin_amdgcn_readfirstlane(rows);
  if constexpr (MJ == 2) {
    if (rows_u <= 32) pipeline(std::integral_constant<int, 1>{});
    else pipeline(std::integral_constant<int, 2>{});
  } else {
    pipeline(std::integral_constant<int, MJ>{});
  }
  if constexpr (KG > 1) {
    // the second group's sums, through its own code stages, added to the first's
    static_assert(KG == 2 && NI * MJ * 16 * 64 * 4 <= WB, "exchange region");
    wait_copies_upto<0>();
    __syncthreads();  // every wavefront is done with the stage buffers
    float* ex = reinterpret_cast<float*>(wave == 0 ? sW0s : wave == 1 ? sW1s : wave == 2 ? sW2s : sW3s) + WB / 4 + lane;
    if (kg == 1) {
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < MJ; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) ex[((i * MJ + j) * 16 + r) * 64] = acc[i][j][r];
    }
    if (kg == 0) {
      if (tid < BM) {
        s_sx[tid] = 1.0f;
        s_rw[tid] = e_rw;
        s_yr[tid] = e_yr;
      }
      if (tid < BN) {
        s_ws[tid] = 1.0f;
        s_bs[tid] = e_bs;
      }
    }
    __syncthreads();
    if (kg == 1) return;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < MJ; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] += ex[((i * MJ + j) * 16 + r) * 64];
  }
  if (p.ksplit > 1) {
    tile_store_partials<BN, TN, TM, NI, MJ, ACT, false>(p, acc, row0, rows, n0, nlim, wn, wm, lane);
    return;
  }
  if constexpr (KG == 1) {
    wait_copies_upto<0>();
    __syncthreads();  // every wavefront is done with the stage buffers
    if (tid < BM) {
      s_sx[tid] = 1.0f;
      s_rw[tid] = e_rw;
      s_yr[tid] = e_yr;
    }
    if (tid < BN) {
      s_ws[tid] = 1.0f;
      s_bs[tid] = e_bs;
    }
    __syncthreads();
  }
  // a wavefront's f32 region [32 tokens][TN rows]: an activation stage for
  // 64-token tiles, a code stage for 32-token tiles
  static_assert(32 * TN * 4 <= (BM >= 64 ? BM * 128 : BN * 32), "epilogue region");
  uint8_t* regb;
  if constexpr (BM >= 64) regb = wave == 0 ? sA0 : wave == 1 ? sA1 : wave == 2 ? sA2 : sA3;
  else regb = wave == 0 ? sW0 : wave == 1 ? sW1 : wave == 2 ? sW2 : sW3;
  tile_epilogue<BN, TN, TM, NI, MJ, ACT>(p, acc, reinterpret_cast<float*>(regb), s_sx, s_rw, s_yr, s_ws, s_bs,
                                        n0, nlim, rows, wn, wm, lane);
}

template <int BM, int KG, bool ACT, int FMT>
void w4_launch_shape(const GemmParams& p, hipStream_t st) {
  const int nout = ACT ? p.N / 2 : p.N;
  const int n_tiles = cdiv(nout, ACT ? kW4BN / 2 : kW4BN);
  const unsigned ks = (unsigned)std::max(1, p.ksplit);
  const int m_tiles = cdiv(p.M, BM) + (p.group_offs ? std::min(p.slots, p.M) : 0);
  const int grid = cdiv(m_tiles * n_tiles, kXcds) * kXcds;
  hipLaunchKernelGGL((w4_gemm_kernel<BM, KG, ACT, FMT>), dim3(grid, 1, ks), dim3(KG * kThreads), 0, st, p, m_tiles,
                     n_tiles);
}

template <int BM, int KG, int FMT>
void w4_launch_act(const GemmParams& p, hipStream_t st) {
  if (p.act != QA_NONE) w4_launch_shape<BM, KG, true, FMT>(p, st);
  else w4_launch_shape<BM, KG, false, FMT>(p, st);
}

template <int BM, int KG>
void w4_launch_fmt(const GemmParams& p, int fmt, hipStream_t st) {
  if (fmt == 1) w4_launch_act<BM, KG, 1>(p, st);
  else if (fmt == 2) w4_launch_act<BM, KG, 2>(p, st);
  else w4_launch_act<BM, KG, 0>(p, st);
}

template <int BM, int KG, int FMT>
void w4_launch_ring(const GemmParams& p, hipStream_t st) {
  const bool act = p.act != QA_NONE;
  const int n_tiles = cdiv(act ? p.N / 2 : p.N, act ? kW4BN / 2 : kW4BN), m_tiles = cdiv(p.M, BM);
  const dim3 grid(cdiv(m_tiles * n_tiles, kXcds) * kXcds, 1, (unsigned)std::max(1, p.ksplit));
  if (act) hipLaunchKernelGGL((w4_ring_kernel<BM, KG, true, FMT>), grid, dim3(KG * kThreads), 0, st, p, m_tiles, n_tiles);
  else hipLaunchKernelGGL((w4_ring_kernel<BM, KG, false, FMT>), grid, dim3(KG * kThreads), 0, st, p, m_tiles, n_tiles);
}

// The kernel of a problem: token-tile height, K groups of wavefronts per
// workgroup, K slices, and whether the ring kernel runs it.
struct W4Plan {
  int bm = 128, kgroups = 1, ksplit = 1;
  bool ring = false;
};

// One round of workgroups on MI355X takes `start` + `stage` us per 64-k stage
// of a K group, by kernel and format (MXFP4, NVFP4, INT4). Fitted to 171 dense
// problems per format (K 512..14336, N 128..32768, 65..4096 tokens, one to 12
// slices), which they meet within 8 % (rms).
struct W4Time {
  int bm, kgroups;
  bool ring;
  float start[3], stage[3];
};
constexpr W4Time kW4Times[] = {
    {32, 2, false, {6.7f, 7.5f, 8.0f}, {0.63f, 1.07f, 1.29f}},
    {64, 2, false, {9.4f, 10.0f, 10.3f}, {0.87f, 1.25f, 1.47f}},
    {128, 2, false, {13.4f, 13.8f, 14.0f}, {1.34f, 1.68f, 1.93f}},
    {64, 1, false, {9.7f, 9.9f, 10.4f}, {0.90f, 1.26f, 1.44f}},
    {128, 1, false, {9.2f, 8.5f, 9.3f}, {1.51f, 1.84f, 2.09f}},
    {32, 1, true, {0, 6.0f, 0}, {0, 0.50f, 0}},
    {32, 2, true, {0, 7.6f, 0}, {0, 0.84f, 0}},
    {64, 1, true, {0, 0, 7.9f}, {0, 0, 0.77f}},
};

// Dense problems of more than one round of 64-token tiles (two workgroups of
// one K group per CU) take 128-token tiles (64-token ones lose 5 to 30 % from
// there on). The others take the kernel and K split of the least time: two K
// groups where the workgroups fill only one per CU, one group above that; a
// split only within one workgroup per CU, which also bounds its f32 slices to
// 256 tiles; the ring kernel up to 256 tokens. The XCDs are dealt whole tiles,
// so a count is rounded up to 8. The ring ends at K 8192 (NVFP4 K 14336, N
// 4096, 129 tokens 56.6 us, the line kernel 46.6). Measured against the rules
// before (the largest tiles on at least 130 CUs, at most 4 slices of at least
// 28 stages, the ring up to K 4096): MXFP4 / NVFP4 / INT4 4 / 6 / 9 % faster
// over 192 problems, e.g. K 2880, N 5760, 700 tokens 46.5 / 57.0 / 61.6 -> 31.6 / 41.6 / 46.1 us,
// NVFP4 / INT4 K 7168, N 256, 128 tokens 24.9 / 29.0 -> 15.9 / 20.4.
W4Plan w4_plan_dense(const GemmParams& p, int fmt, int n_tiles, int force_bm, int force_ks) {
  const int nu = p.K / 64;
  auto workgroups = [&](int bm, int ks) { return cdiv<int64_t>((int64_t)cdiv(p.M, bm) * n_tiles, kXcds) * kXcds * ks; };
  W4Plan best;
  if (force_bm) {
    best.bm = force_bm;
    best.ksplit = std::max(force_ks, 1);
    best.kgroups = force_bm == 32 || workgroups(force_bm, best.ksplit) <= 256 ? 2 : 1;
    return best;
  }
  if (!force_ks && workgroups(64, 1) > 512) return best;
  float best_us = -1.0f;
  for (int k : {1, 2, 3, 4, 6, 8, 12}) {
    const int ks = force_ks ? force_ks : k;
    if (!force_ks && ks > 1 && nu / ks < 4) break;
    for (const W4Time& t : kW4Times) {
      if (t.ring && (t.start[fmt] == 0 || p.M > 256 || p.K > 8192)) continue;
      const int64_t n = workgroups(t.bm, ks), round = t.kgroups == 1 && !t.ring ? 512 : 256;
      if (round == 512 && n <= 256) continue;  // one workgroup per CU: two K groups
      if (!force_ks && n > (ks > 1 ? 256 : t.bm == 32 && !t.ring ? 512 : round)) continue;
      float us = (float)cdiv(n, round) * (t.start[fmt] + t.stage[fmt] * (float)cdiv(cdiv(nu, ks), t.kgroups));
      if (ks > 1) us += 2.5f + 0.4e-6f * (float)((int64_t)p.M * p.N * 4 * ks);  // the finishing launch and its slices
      if (best_us < 0 || us < best_us) {
        best_us = us;
        best.bm = t.bm;
        best.kgroups = t.kgroups;
        best.ksplit = ks;
        best.ring = t.ring;
      }
    }
    if (force_ks) break;
  }
  return best;
}

// m-tiles of `bm` rows that the groups are expected to need: those of equal
// groups, or of groups whose last tiles are half filled on average
int w4_group_tiles(const GemmParams& p, int bm) {
  const int groups = std::max(1, std::min(p.slots, p.M));
  return std::max(groups * cdiv(p.M / groups, bm), p.M / bm + groups / 2);
}

// Routed experts. Tiles that about fill one workgroup per CU run two K groups
// in each; beyond 40 rows per expert 128-token tiles, unless one round of
// 64-token tiles (two workgroups per CU) holds them all. Measured on MI355X
// (one group, 64 / 128 tokens; two groups, 64 / 128): MXFP4, 4 experts, K
// 2880, N 5760, 16 rows each 27.6 / 29.7; 21.8 / 23.9 us, 128 rows 39.8 / 63.4;
// 31.9 / 55.0; 8 experts, 128 rows 57.2 / 86.0; 64.9 / 105.7; 16 experts, N
// 2880, 64 rows 50.2 / 46.6; 58.0 / 38.9; GPT-OSS MoE layer (128 experts), 32 /
// 64 rows 518 / 797 in 64-token tiles, 532 / 696 in 128-token tiles.
W4Plan w4_plan_grouped(const GemmParams& p, int n_tiles, int force_bm, int force_ks) {
  constexpr int kFill = 272;  // the estimate, a little over 256
  auto count = [&](int bm) { return (int64_t)w4_group_tiles(p, bm) * n_tiles; };
  const int rows = p.M / std::max(1, std::min(p.slots, p.M));
  W4Plan r;
  if (force_bm) r.bm = std::max(force_bm, 64);
  else if (count(64) <= kFill || rows <= 40) r.bm = 64;
  else r.bm = count(128) <= kFill || count(64) > 512 ? 128 : 64;
  r.kgroups = count(r.bm) <= kFill ? 2 : 1;
  r.ksplit = std::max(force_ks, 1);
  return r;
}

// The plan of a problem that the kernels take (qmoe_w4_plan checks that).
// QMOE_W4_BM forces the line kernel in that tile height, QMOE_W4_KSPLIT the K
// split (tuning knobs).
W4Plan w4_choose(const GemmParams& p, int fmt, int n_tiles) {
  const char* env = getenv("QMOE_W4_BM");
  const int bm = env && (atoi(env) == 128 || atoi(env) == 64 || atoi(env) == 32) ? atoi(env) : 0;
  const char* ks_env = getenv("QMOE_W4_KSPLIT");
  const int ks = ks_env && atoi(ks_env) > 0 ? std::min(atoi(ks_env), p.K / 64) : 0;
  return p.group_offs ? w4_plan_grouped(p, n_tiles, bm, ks) : w4_plan_dense(p, fmt, n_tiles, bm, ks);
}

}  // namespace

// Whether the W4A16 tiled kernels take the problem (K % 64, 16-byte aligned
// rows, even scale rows, codes < 4 GiB per group), and its plan: token-tile
// height, K split and the f32 workspace the split needs ([ksplit][M][N]).
// `fmt`: 0 MXFP4 (e8m0 per 32 k), 1 NVFP4 (bf16 per 16 k), 2 INT4 (bf16 per
// wq_group k).
bool qmoe_w4_plan(const GemmParams& p, int fmt, int* bm_out, int* ksplit_out, int64_t* ws_bytes) {
  if (p.M <= 0 || p.K <= 0 || (p.K % 64) != 0 || p.N <= 0) return false;
  if (p.act != QA_NONE && (p.N % 2) != 0) return false;
  if ((p.lda % 8) != 0 || (p.ldw % 16) != 0 || (fmt != 2 && (p.ldws % 2) != 0)) return false;
  if (fmt == 2 && ((p.wq_group != 32 && p.wq_group != 64 && p.wq_group != 128) || (p.K % p.wq_group) != 0))
    return false;
  // scale alignment mask: 4-byte bf16 pairs (NVFP4), 2-byte e8m0 pairs (MXFP4), bf16 (INT4)
  const int sal = fmt == 1 ? 3 : 1;
  if ((reinterpret_cast<uintptr_t>(p.a) & 15) || (reinterpret_cast<uintptr_t>(p.w) & 15) ||
      (p.w_gstride % 16) != 0 || (reinterpret_cast<uintptr_t>(p.w_scale) & sal) ||
      (fmt != 2 && (p.ws_gstride % 2) != 0))
    return false;
  if ((int64_t)p.ldw * p.N >= ((int64_t)1 << 32) || (int64_t)p.ldws * (fmt ? 2 : 1) * p.N >= ((int64_t)1 << 31))
    return false;
  const int nout = p.act != QA_NONE ? p.N / 2 : p.N;
  const int n_tiles = cdiv(nout, p.act != QA_NONE ? kW4BN / 2 : kW4BN);
  const W4Plan plan = w4_choose(p, fmt, n_tiles);
  const int bm = plan.bm, ksplit = plan.ksplit;
  const int m_tiles0 = p.group_offs ? cdiv(p.M, bm) + std::min(p.slots, p.M) : cdiv(p.M, bm);
  if ((int64_t)m_tiles0 * n_tiles > (1 << 30)) return false;
  *bm_out = bm;
  *ksplit_out = ksplit;
  *ws_bytes = ksplit > 1 ? (int64_t)ksplit * p.M * p.N * 4 : 0;
  return true;
}

// Launch per the plan (the caller sized the workspace); with a K split the
// finishing kernel runs the epilogue.
int qmoe_w4_launch(GemmParams p, int fmt, void* workspace, int64_t ws_bytes, hipStream_t st) {
  int bm = 0, ksplit = 1;
  int64_t need = 0;
  if (!qmoe_w4_plan(p, fmt, &bm, &ksplit, &need)) return QMOE_ERR_ARG;
  p.ksplit = ksplit;
  if (ksplit > 1) {
    if (!workspace || ws_bytes < need) return QMOE_ERR_WORKSPACE;
    p.partial = static_cast<float*>(workspace);
  }
  const W4Plan plan =
      w4_choose(p, fmt, cdiv(p.act != QA_NONE ? p.N / 2 : p.N, p.act != QA_NONE ? kW4BN / 2 : kW4BN));
  if (plan.ring) {
    if (fmt == 2) w4_launch_ring<64, 1, 2>(p, st);
    else plan.kgroups == 2 ? w4_launch_ring<32, 2, 1>(p, st) : w4_launch_ring<32, 1, 1>(p, st);
  } else if (bm == 128) {
    plan.kgroups == 2 ? w4_launch_fmt<128, 2>(p, fmt, st) : w4_launch_fmt<128, 1>(p, fmt, st);
  } else if (bm == 64) {
    plan.kgroups == 2 ? w4_launch_fmt<64, 2>(p, fmt, st) : w4_launch_fmt<64, 1>(p, fmt, st);
  } else {
    w4_launch_fmt<32, 2>(p, fmt, st);
  }
  if (ksplit > 1) {
    const int nout = p.act != QA_NONE ? p.N / 2 : p.N;
    const dim3 rg((unsigned)cdiv(nout, 512), (unsigned)cdiv(p.M, 4), 1);
    if (p.act != QA_NONE)
      hipLaunchKernelGGL((tile_splitk_finish_kernel<false, true, kScNone>), rg, dim3(kThreads), 0, st, p);
    else
      hipLaunchKernelGGL((tile_splitk_finish_kernel<false, false, kScNone>), rg, dim3(kThreads), 0, st, p);
  }
  return hipGetLastError() == hipSuccess ? QMOE_OK : QMOE_ERR_LAUNCH;
}

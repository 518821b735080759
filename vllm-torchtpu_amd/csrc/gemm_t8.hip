// Tiles of eight wavefronts (one workgroup per CU, two wavefronts per SIMD):
// block-scaled FP8 (QK_W8A8_BLK: 128 x 128 tiles of e4m3 weights or the
// grouped matmul's per-channel e4m3 or e5m2 weights, activation scales per 128 or 512
// columns) and bf16 x bf16 (QK_W16A16), dense or grouped.
//
//  * What bounds it: the matrix cores with the vector ALU and the operand
//    reads beside them. A block-scaled tile adds every 128-k block's sums,
//    scaled, to its accumulators: 16 FMAs per 32 x 32 block against two MFMAs
//    of 64 cycles. With one wavefront per SIMD (gemm_f8.hip) these alternate
//    and the second accumulator set in AGPRs costs another 16 moves; with two
//    wavefronts of at most 256 VGPRs the MFMAs write VGPRs directly, and one
//    wavefront scales while the other multiplies.
//  * Output tile BM tokens x 256 weight rows; wavefront (wn, wm), wn < 4,
//    wm < 2, owns 64 weight rows (two 32-row blocks) and the 32-token blocks
//    wm, wm + 2, ..., so that a tile with few tokens loads both halves alike.
//    Measured against the four-wavefront and generic tiles (block FP8 K 7168, N
//    18432, 2048 / 8192 tokens, quantization included: 396 / 1516 -> 339 / 1223
//    us; DeepSeek-V3 routed experts, 2048 tokens 2530 -> 2252 us; bf16 K 4096, N
//    6144, 1024 tokens 78.6 -> 59.3 us).
//  * Stages of 128 bytes of every row (128 e4m3 / 64 bf16 values), copied
//    straight into a ring of LDS stages (two of 64 KB for 256 tokens, three of
//    48 KB for 128); one barrier per stage.
//  * The epilogue takes 64 tokens at a time through LDS (32 x 256 f32 sums per
//    token block) and finishes 8 channels of a token per thread.

#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "gemm_tile.h"
#include "stream_load.h"

namespace {

constexpr int kT8Threads = 512;
constexpr int kT8BN = 256;

__device__ __forceinline__ int t8_swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// Wait until at most n vector-memory operations are outstanding; n, known at
// run time (wave-uniform), is one stage's copies, 4 to 7 (else: all)
__device__ __forceinline__ void t8_wait(int n) {
  switch (n) {
    case 4: wait_copies_upto<4>(); break;
    case 5: wait_copies_upto<5>(); break;
    case 6: wait_copies_upto<6>(); break;
    case 7: wait_copies_upto<7>(); break;
    default: wait_copies_upto<0>(); break;
  }
}

// lds_copy16 (gemm_tile.h) of four offsets from one scalar base, to `lds` + 0,
// 8, 16 and 24 KB: the move of the base that its wait states need, once for the
// four (bf16 K 4096, N 6144, 1024 tokens 60.4 -> 59.5 us).
__device__ __forceinline__ void t8_copy4(const uint8_t* base, const uint32_t (&off)[4], uint32_t lds) {
  const uint8_t* b;
  asm volatile(
      "s_mov_b64 %0, %6\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %0\n\t"
      "s_add_u32 m0, m0, 0x2000\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %3, %0\n\t"
      "s_add_u32 m0, m0, 0x2000\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %4, %0\n\t"
      "s_add_u32 m0, m0, 0x2000\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %5, %0"
      : "=&s"(b)
      : "s"(lds), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(base)
      : "m0", "scc", "memory");
}

// F8: block-scaled 1-byte floats; else bf16. WPC (F8): one weight scale per
// weight row, applied in the epilogue, instead of one per 128 x 128 tile. WF:
// weight format code of the MFMA, 0 e4m3, 1 e5m2 (activations are e4m3).
template <bool F8, int BM, bool ACT, bool WPC, int WF>
__global__ __launch_bounds__(kT8Threads, 2) void t8_gemm_kernel(const GemmParams p, int m_tiles, int n_tiles) {
  constexpr int BN = kT8BN, BNO = ACT ? BN / 2 : BN;
  constexpr int NI = 2, MJ = BM / 64;            // 32-row weight blocks, 32-token blocks per wavefront
  constexpr int RING = BM > 128 ? 2 : 3;
  constexpr int WB = BN * 128, XB = BM * 128;    // bytes of a stage
  constexpr int STG = WB + XB + (F8 ? BM * 4 : 0);
  __shared__ __align__(1024) uint8_t smem[RING * STG];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem;

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 3, wm = wave >> 2;

  int g, row0, rows, ntile;
  if (p.group_offs) {
    if (!tile_group_xcd<BM>(p, blockIdx.x, n_tiles, g, row0, rows, ntile, reinterpret_cast<int*>(smem))) return;
    __syncthreads();  // the group has been read everywhere: the buffers are free
  } else {
    int mt;
    if (!tile_dense(blockIdx.x, m_tiles, n_tiles, mt, ntile)) return;
    g = 0;
    row0 = mt * BM;
    rows = min(BM, p.M - row0);
  }
  g = __builtin_amdgcn_readfirstlane(g);
  const int rows_u = __builtin_amdgcn_readfirstlane(rows);
  const int n0 = ntile * BNO;
  const int nlim = ACT ? p.N / 2 : p.N;
  // global weight row of tile row r (gate rows, then up rows with ACT); rows
  // past the end are clamped (their outputs are never stored). With ACT a
  // wavefront's first block holds gate rows and its second the matching up
  // rows.
  auto wrow_global = [&](int r) {
    if (ACT) return (r < BN / 2 ? 0 : p.N / 2) + min(n0 + (r % (BN / 2)), nlim - 1);
    return min(n0 + r, nlim - 1);
  };
  auto wrow = [&](int i) { return ACT ? i * (BN / 2) + wn * 32 : wn * 64 + i * 32; };

  // epilogue inputs (loaded now, staged in LDS at the end)
  float e_rw = 1.0f, e_bs = 0.0f, e_ws = 1.0f;
  int e_yr = 0;
  if (tid < BM) {
    const int R = row0 + min(tid, rows - 1);
    if (p.row_weight) e_rw = bf16_to_f32(p.row_weight[R]);
    e_yr = p.y_rows ? p.y_rows[R] : R;
  }
  if (tid < BN) {
    if (p.bias) e_bs = p.bias[(int64_t)g * p.bias_gstride + wrow_global(tid)];
    if constexpr (F8 && WPC) e_ws = static_cast<const float*>(p.w_scale)[(int64_t)g * p.ws_gstride + wrow_global(tid)];
  }

  // ---- copies: one instruction = 8 rows x 128 bytes (lane -> row l >> 3, slot
  // l & 7; the slot of chunk c of row r is c ^ t8_swz(r)); wavefront w copies
  // the row groups w, w + 8, ... of both operands. Activation row groups past
  // the tile's rows are left out.
  constexpr int WI = BN / 64, XI = BM / 64;
  const uint64_t ab = F8 ? 1 : 2;
  const uint8_t* wbase = p.w + (int64_t)g * p.w_gstride;
  const int cchunk = ((lane & 7) ^ ((lane >> 3) ^ (wave & 1))) * 16;
  uint32_t woff[WI];
#pragma unroll
  for (int j = 0; j < WI; ++j)
    woff[j] = (uint32_t)wrow_global((wave + 8 * j) * 8 + (lane >> 3)) * (uint32_t)p.ldw + (uint32_t)cchunk;
  const uint8_t* xp[XI];
  int nx = 0;
#pragma unroll
  for (int j = 0; j < XI; ++j) {
    const int r = (wave + 8 * j) * 8 + (lane >> 3);
    const int R = row0 + min(r, rows - 1);
    const int ar = p.a_rows ? p.a_rows[R] : R;
    xp[j] = static_cast<const uint8_t*>(p.a) + (uint64_t)(uint32_t)ar * ((uint64_t)p.lda * ab) + (uint32_t)cchunk;
    nx += (wave + 8 * j) * 8 < rows_u ? 1 : 0;
  }
  // F8: the activation scales of a stage, 64 tokens per wavefront
  const float* sp = p.a_scale;
  const bool sc_mine = F8 && wave * 64 < BM && wave * 64 < rows_u;
  if constexpr (F8) {
    const int R = row0 + min(min(wave, BM / 64 - 1) * 64 + lane, rows - 1);
    sp += (int64_t)(p.a_rows ? p.a_rows[R] : R) * p.lds_a;
  }
  const int a_kshift = p.a_kshift, w_kshift = p.w_kshift;
  const uint32_t cw = lds0 + wave * 1024;
  auto copy_stage = [&](int s, int buf) {
    const uint32_t d = __builtin_amdgcn_readfirstlane(cw + buf * STG);
    const uint64_t b = reinterpret_cast<uint64_t>(wbase) + (uint64_t)(uint32_t)s * 128u;
    const uint8_t* ws = reinterpret_cast<const uint8_t*>(
        (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(b >> 32)) << 32 |
        (uint32_t)__builtin_amdgcn_readfirstlane((int)b));
    static_assert(WI == 4, "weight copies of a stage");
    t8_copy4(ws, woff, d);
#pragma unroll
    for (int j = 0; j < XI; ++j)
      if (j < nx) lds_copy16(xp[j] + (int64_t)s * 128, d + WB + j * 8192);
    if (sc_mine) lds_copy4(sp + (s >> a_kshift), lds0 + buf * STG + WB + XB + wave * 256);
  };
  const int per_stage = WI + nx + (sc_mine ? 1 : 0);

  const int KS = F8 ? p.K / 128 : p.K / 64;
  const int rl = lane & 31, kh = lane >> 5;
  // the weight scale of this wavefront's rows, tile layout (block i's rows lie
  // in one 128-row tile). Read through the constant address space, as scalar
  // loads: a vector load's wait would drain the copies in flight.
  typedef const float __attribute__((address_space(4))) CFloat;
  CFloat* wsp[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i)
    wsp[i] = (CFloat*)(uintptr_t)(static_cast<const float*>(p.w_scale) +
                                  (F8 && !WPC ? (int64_t)g * p.ws_gstride +
                                                    (int64_t)(__builtin_amdgcn_readfirstlane(wrow_global(wrow(i))) / 128) *
                                                        p.ldws
                                              : 0));

  f32x16 acc[NI][MJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  // The K pipeline over the wavefront's first MJE token blocks (those with a
  // token); the accumulators of the others keep their zeros.
  auto pipeline = [&](auto mje_c) {
    constexpr int MJE = decltype(mje_c)::value;
#pragma unroll
    for (int r = 0; r < (F8 ? RING - 1 : RING); ++r)
      if (r < KS) copy_stage(r, r);
    // Per stage: its first operands are in registers (read during the last
    // MFMAs of the stage before). All but the last MFMA step run while the
    // next step's operands are read; then the next stage's copies have landed
    // (the one after's stay in flight with three buffers) -> barrier: they
    // have landed everywhere, and everybody holds this stage's last operands,
    // so that its buffer takes the copies of stage s + RING -> the last step,
    // while the next stage's first operands are read.
    auto landed = [&](int ahead) {
      if (ahead && RING == 3) t8_wait(per_stage * ahead);
      else wait_copies_upto<0>();
    };
    auto chunk = [&](const uint8_t* base, int row, int c) {
      return *reinterpret_cast<const uint4*>(base + (row + rl) * 128 + ((c ^ t8_swz(rl)) * 16));
    };
    landed(0);
    stage_barrier();
    int buf = 0;
    if constexpr (F8) {
      auto frag = [&](const uint8_t* base, int row, int t) {
        const uint4 a = chunk(base, row, 4 * t + 2 * kh), b = chunk(base, row, 4 * t + 2 * kh + 1);
        i32x8 r;
        r[0] = a.x; r[1] = a.y; r[2] = a.z; r[3] = a.w;
        r[4] = b.x; r[5] = b.y; r[6] = b.z; r[7] = b.w;
        return r;
      };
      // (a second set of weight operands, read ahead, would not fit the 256
      // VGPRs: the stage's operands are read behind its barrier)
      for (int s = 0; s < KS; ++s) {
        if (s > 0) {
          landed(RING == 3 && s + 1 < KS ? 1 : 0);
          stage_barrier();
        }
        // (after the first operand reads, which the first MFMAs wait for)
        auto refill = [&]() {
          if (s + RING - 1 < KS) copy_stage(s + RING - 1, buf == 0 ? RING - 1 : buf - 1);
        };
        if constexpr (MJE == 0) refill();
        if constexpr (MJE > 0) {
          const uint8_t* sW = smem + buf * STG;
          const uint8_t* sX = sW + WB;
          const float* sS = reinterpret_cast<const float*>(sX + XB);
          i32x8 wf[NI][2];
          float sw[NI];
#pragma unroll
          for (int i = 0; i < NI; ++i) {
            wf[i][0] = frag(sW, wrow(i), 0);
            wf[i][1] = frag(sW, wrow(i), 1);
            sw[i] = WPC ? 1.0f : wsp[i][s >> w_kshift];
          }
          // block pair n's MFMAs, then the scaling of pair n - 1
          f32x16 tmp[2];
          float sc[2];
          i32x8 xf[2];
          xf[0] = frag(sX, wm * 32, 0);
          xf[1] = frag(sX, wm * 32, 1);
          refill();
#pragma unroll
          for (int n = 0; n <= NI * MJE; ++n) {
            if (n < NI * MJE) {
              const int i = n % NI, j = n / NI, row = (2 * j + wm) * 32;
              if (i == 0 && j > 0) {
                xf[0] = frag(sX, row, 0);
                xf[1] = frag(sX, row, 1);
              }
              sc[n & 1] = sS[row + rl] * sw[i];
              tmp[n & 1] =
                  __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wf[i][0], xf[0], f32x16{}, WF, 0, 0, 127, 0, 127);
              tmp[n & 1] =
                  __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wf[i][1], xf[1], tmp[n & 1], WF, 0, 0, 127, 0, 127);
            }
            if (n > 0) {
              const int i = (n - 1) % NI, j = (n - 1) / NI;
#pragma unroll
              for (int r = 0; r < 16; ++r) acc[i][j][r] += tmp[(n - 1) & 1][r] * sc[(n - 1) & 1];
            }
          }
        }
        buf = buf == RING - 1 ? 0 : buf + 1;
      }
    } else {
      union B8 {
        uint4 u;
        bf16x8 v;
      };
      constexpr int MR = MJE > 0 ? MJE : 1;
      B8 wf[2][NI], xf[2][MR];
      auto read_q = [&](int b, int q) {
        const uint8_t* sW = smem + b * STG;
#pragma unroll
        for (int i = 0; i < NI; ++i) wf[q & 1][i].u = chunk(sW, wrow(i), 2 * q + kh);
#pragma unroll
        for (int j = 0; j < MJE; ++j) xf[q & 1][j].u = chunk(sW + WB, (2 * j + wm) * 32, 2 * q + kh);
      };
      auto mma = [&](int q) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < MJE; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[q & 1][i].v, xf[q & 1][j].v, acc[i][j], 0, 0, 0);
      };
      if constexpr (MJE > 0) read_q(0, 0);
      for (int s = 0; s < KS; ++s) {
        const int nb = buf == RING - 1 ? 0 : buf + 1;
        if constexpr (MJE > 0) {
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            read_q(buf, q + 1);
            mma(q);
          }
        }
        if (s + 1 < KS) landed(s + 2 < KS ? 1 : 0);
        stage_barrier();
        if (s + RING < KS) copy_stage(s + RING, buf);
        asm volatile("" ::: "memory");
        if constexpr (MJE > 0) {
          if (s + 1 < KS) read_q(nb, 0);
          mma(3);
        }
        buf = nb;
      }
    }
  };
  // token blocks 2 j + wm with a token
  const int mje = max(0, (cdiv(rows_u, 32) - wm + 1) / 2);
  if constexpr (MJ == 4) {
    if (mje == 0) pipeline(std::integral_constant<int, 0>{});
    else if (mje == 1) pipeline(std::integral_constant<int, 1>{});
    else if (mje == 2) pipeline(std::integral_constant<int, 2>{});
    else if (mje == 3) pipeline(std::integral_constant<int, 3>{});
    else pipeline(std::integral_constant<int, 4>{});
  } else {
    if (mje == 0) pipeline(std::integral_constant<int, 0>{});
    else if (mje == 1) pipeline(std::integral_constant<int, 1>{});
    else pipeline(std::integral_constant<int, 2>{});
  }

  // ---- epilogue: 64 tokens at a time, f32 sums in LDS ([64 tokens][256 tile
  // rows], row n of token t at n ^ 4 (t % 16)), then 8 output channels of a
  // token per thread
  __syncthreads();  // every wavefront is done with the stage buffers
  float* reg = reinterpret_cast<float*>(smem);
  float* s_rw = reg + 64 * BN;
  float *s_bs = s_rw + BM, *s_ws = s_bs + BN;
  int* s_yr = reinterpret_cast<int*>(s_ws + BN);
  static_assert((64 * BN + 2 * BM + 2 * BN) * 4 <= RING * STG, "epilogue regions");
  if (tid < BM) {
    s_rw[tid] = e_rw;
    s_yr[tid] = e_yr;
  }
  if (tid < BN) {
    s_bs[tid] = e_bs;
    s_ws[tid] = e_ws;
  }
#pragma unroll
  for (int j = 0; j < MJ; ++j) {
    if (j * 64 >= rows_u) break;
    if (j) __syncthreads();  // the previous tokens have been read
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = wrow(i) + q * 8 + kh * 4;  // tile row of the register quad
        *reinterpret_cast<float4*>(reg + (wm * 32 + rl) * BN + (n ^ (4 * (rl & 15)))) =
            make_float4(acc[i][j][q * 4], acc[i][j][q * 4 + 1], acc[i][j][q * 4 + 2], acc[i][j][q * 4 + 3]);
      }
    __syncthreads();
    tile_finish_rows<64, kT8Threads, BN, ACT, F8 && WPC>(p, reg, tid, j * 64, rows, n0, nlim, s_rw, s_bs, s_ws, s_yr);
  }
}

template <bool F8, int BM, bool ACT, bool WPC, int WF = 0>
void t8_launch_shape(const GemmParams& p, hipStream_t st) {
  const int n_tiles = cdiv(ACT ? p.N / 2 : p.N, ACT ? kT8BN / 2 : kT8BN);
  const int m_tiles = cdiv(p.M, BM) + (p.group_offs ? std::min(p.slots, p.M) : 0);
  const int grid = cdiv(m_tiles * n_tiles, kXcds) * kXcds;
  hipLaunchKernelGGL((t8_gemm_kernel<F8, BM, ACT, WPC, WF>), dim3(grid), dim3(kT8Threads), 0, st, p, m_tiles, n_tiles);
}

template <bool WPC, int WF = 0>
void t8_launch_f8(const GemmParams& p, int bm, hipStream_t st) {
  const bool act = p.act != QA_NONE;
  if (bm == 256) act ? t8_launch_shape<true, 256, true, WPC, WF>(p, st) : t8_launch_shape<true, 256, false, WPC, WF>(p, st);
  else act ? t8_launch_shape<true, 128, true, WPC, WF>(p, st) : t8_launch_shape<true, 128, false, WPC, WF>(p, st);
}

// Dense: how many 256-token tiles (of every weight tile) come first; the rows
// after them run as 128-token tiles in a second launch. The candidates are
// 128-token tiles alone, 256-token tiles alone, and whole rounds of 256-token
// tiles over the 256 CUs with the last round, or the last two, as 128-token
// tiles. A round of 256-token tiles takes 1.57 to 1.73 times one of 128-token
// tiles (K 7168, N 18432, 512 / 1024 / 4096 / 8192 tokens 142 / 211 / 735 /
// 1469 us in 128-token tiles, 119 / 236 / 642 / 1246 in 256-token tiles).
// Measured, two heights / 128 / 256 alone: e4m3 K 7168, N 18432 at 1024 / 2048
// tokens 197 / 205 / 227, 311 / 341 / 347 us; K 4096, N 6144 at 3000 116 / 125
// / 141; bf16 K 7168, N 18432 at 1024 296 / 325 / 364, K 4096, N 6144 at 3000
// 171 / 185 / 209.
int t8_tall_tiles(int M, int n_tiles) {
  const int64_t m256 = cdiv(M, 256), rounds = cdiv<int64_t>(m256 * n_tiles, 256);
  int64_t best = 0, best_cost = -1;
  auto consider = [&](int64_t tall) {
    const int64_t rest = std::max<int64_t>(M - tall * 256, 0);
    int64_t cost = cdiv<int64_t>(tall * n_tiles, 256) * 168 + cdiv<int64_t>(cdiv<int64_t>(rest, 128) * n_tiles, 256) * 100;
    if (tall > 0 && rest > 0) cost += 10;  // the second launch
    if (best_cost < 0 || cost < best_cost) best = tall, best_cost = cost;
  };
  consider(0);
  consider(m256);
  for (int64_t r = rounds - 1; r > 0 && r >= rounds - 2; --r) consider(r * 256 / n_tiles);
  return (int)best;
}

// The rows from `row` on of a dense problem
GemmParams t8_rows_from(GemmParams p, int row, int a_bytes) {
  p.M -= row;
  if (p.a_rows) {
    p.a_rows += row;
  } else {
    p.a = static_cast<const uint8_t*>(p.a) + (int64_t)row * p.lda * a_bytes;
    if (p.a_scale) p.a_scale += (int64_t)row * p.lds_a;
  }
  if (p.row_weight) p.row_weight += row;
  if (p.y_rows) p.y_rows += row;
  else p.y += (int64_t)row * p.ldy;
  return p;
}

void t8_launch(const GemmParams& p, bool f8, int bm, hipStream_t st) {
  if (!f8) bm == 256 ? t8_launch_shape<false, 256, false, false>(p, st) : t8_launch_shape<false, 128, false, false>(p, st);
  else if (p.w_kshift >= 31) p.wfmt == 2 ? t8_launch_f8<true, 1>(p, bm, st) : t8_launch_f8<true>(p, bm, st);
  else t8_launch_f8<false>(p, bm, st);
}

int t8_n_tiles(const GemmParams& p) {
  return cdiv(p.act != QA_NONE ? p.N / 2 : p.N, p.act != QA_NONE ? kT8BN / 2 : kT8BN);
}

// Token-tile height of routed experts, 0 for gemm_f8.hip's tiles. An expert is
// taken to hold the average rows and a sixteenth more. A round of 256-token
// tiles over the 256 CUs takes about 1.68 times one of 128-token tiles
// (measured, 128 / 256, us: DeepSeek-V3 routed experts, K 7168, N 4096, 64
// experts, 96 / 128 / 200 / 300 rows each 390 / 450, 576 / 486, 738 / 578, 921
// / 1193; 8 experts, K 2048, N 7168, 128 / 300 rows 55 / 33, 76 / 89). Below
// 200 tiles of 128 tokens the smaller ones of gemm_f8.hip put more CUs to work
// (8 experts, K 7168, N 4096, 64 / 96 rows 51 / 56 us there, 56 / 70 here; K
// 14336, N 4096, 96 rows 118 / 155), and so do its 128-row weight tiles for
// tile-scaled experts of few rows without an activation (K 2048, N 7168: 32
// experts, 8 / 48 rows 88 / 104 there, 94 / 110 here; 64 experts, 48 rows 198
// both; 256 experts, 32 rows 768 / 736). `tiles`: weight scales per 128 x 128.
int t8_grouped_tile(const GemmParams& p, bool tiles) {
  const int groups = std::max(1, std::min(p.slots, p.M)), rows = p.M / groups;
  const int64_t n = (int64_t)groups * t8_n_tiles(p);
  auto tiles_of = [&](int bm) { return n * cdiv(rows + rows / 16, bm); };
  if ((p.K % 256) == 0 && (rows == 0 ? n : tiles_of(128)) < 200) return 0;
  if ((p.K % 256) == 0 && tiles && p.act == QA_NONE && rows <= 48 && n < 1024) return 0;
  return cdiv<int64_t>(tiles_of(256), 256) * 168 < cdiv<int64_t>(tiles_of(128), 256) * 100 ? 256 : 128;
}

}  // namespace

// Token-tile height of the problem on this kernel (256 also where the last
// rows of a dense problem run as 128-token tiles), 0 when another one takes
// it. `f8`: block-scaled codes (else bf16 on both sides).
int qmoe_t8_plan(const GemmParams& p, bool f8) {
  if (p.M <= 0 || p.N <= 0 || p.K <= 0 || (p.K % (f8 ? 128 : 64)) != 0) return 0;
  if (p.act != QA_NONE && (p.N % 2) != 0) return 0;
  const bool wpc = p.w_kshift >= 31;
  if (f8 && (p.wfmt == 1 || (p.wfmt != 0 && !wpc) || (!wpc && (p.ws_bn != 128 || (p.act != QA_NONE && ((p.N / 2) % 128) != 0))))) return 0;
  if (((p.lda * (f8 ? 1 : 2)) % 16) != 0 || (p.ldw % 16) != 0 || (p.w_gstride % 16) != 0) return 0;
  if ((reinterpret_cast<uintptr_t>(p.a) & 15) || (reinterpret_cast<uintptr_t>(p.w) & 15)) return 0;
  if ((int64_t)p.ldw * p.N >= ((int64_t)1 << 32)) return 0;
  // bf16: dense linears (the grouped bf16 layers keep the generic tiles)
  if (!f8 && (p.group_offs || p.act != QA_NONE)) return 0;
  const char* env = getenv("QMOE_T8_BM");  // tuning knob: 128, 256 or 0 (off)
  if (env) return atoi(env) == 128 || atoi(env) == 256 ? atoi(env) : 0;
  if (p.group_offs) return t8_grouped_tile(p, f8 && !wpc);
  // Dense, if it has work for more than half of the CUs; else the smaller
  // tiles and K splits of the other kernels (K 4096, N 4096, 1024 tokens, 128
  // tiles: 50 us here, 41 there; K 2048, N 7168, 1000 tokens, 224 tiles: 32
  // and 42).
  const int n_tiles = t8_n_tiles(p), tall = t8_tall_tiles(p.M, n_tiles);
  // bf16 of a width that 256-row tiles pad by a third or more over the generic
  // tiles' 128 rows: up to 128 channels and 257 to 384 (K 2880, 40000 tokens, N
  // 64 / 320: 76 / 135 us here, 58 / 121 there; N 640 184 here, 209 there)
  if (!f8 && 3 * 2 * cdiv(p.N, 256) >= 4 * cdiv(p.N, 128)) return 0;
  // block-scaled, 257 to 320 tokens over more than one round of 128-token tiles:
  // five 64-token tiles pad less than three of 128 or two of 256 (300 tokens, K
  // 1536 / 7168, N 24576: 36 / 114 us here, 30 / 97 there; one round, K 7168, N
  // 18432: 69 here, 74 there)
  if (f8 && p.act == QA_NONE && (p.K % 256) == 0 && p.M > 256 && p.M <= 320 && 3 * (int64_t)n_tiles > 256) return 0;
  const int64_t tiles = (int64_t)(tall + cdiv(std::max(p.M - (int64_t)tall * 256, (int64_t)0), (int64_t)128)) * n_tiles;
  return tiles >= 140 ? (tall ? 256 : 128) : 0;
}

int qmoe_t8_launch(GemmParams p, bool f8, hipStream_t st) {
  const int bm = qmoe_t8_plan(p, f8);
  if (!bm) return QMOE_ERR_ARG;
  p.ksplit = 1;
  const bool forced = getenv("QMOE_T8_BM") != nullptr;
  const int tall = bm == 256 && !p.group_offs && !forced ? t8_tall_tiles(p.M, t8_n_tiles(p)) : 0;
  if (tall > 0 && (int64_t)tall * 256 < p.M) {
    GemmParams top = p;
    top.M = tall * 256;
    t8_launch(top, f8, 256, st);
    t8_launch(t8_rows_from(p, tall * 256, f8 ? 1 : 2), f8, 128, st);
  } else {
    t8_launch(p, f8, bm, st);
  }
  return hipGetLastError() == hipSuccess ? QMOE_OK : QMOE_ERR_LAUNCH;
}

// Linear with a few dozen to a few hundred activation rows on the matrix cores, for weights packed in MFMA operand order: the
// waves of a workgroup share ONE output tile and split K.
//
// A batch of this size has few output tiles: with 128-row x 256-column tiles and one K loop per tile, 93 rows of a
// 2048 x 6144 matrix are 16 workgroups on 256 CUs, each walking all of K (43 us for 6 MB of weights).  Here the tile is
// (32 TM) rows x (32 TN) channels, wave w of NW takes the K blocks w, w + NW, ... (128 bytes of an activation row each), and the
// waves' sums meet in LDS in wave order: enough workgroups and waves to fill the chip, no workspace, no second launch, the
// same bits on every run.
//
// A wave works on its own: its weights come straight from memory in operand order (1 KB contiguous per load), its activation
// rows as whole 128-byte lines (8 rows per load instruction; one row per lane would touch 32 lines and be bound by the L1's
// tag rate) that pass through the wave's own 4 TM KB of LDS, 16-byte pieces placed at piece ^ (row / 2 % 8): conflict-free
// both ways, and no barrier, since one wave's LDS operations execute in order.  D blocks are in flight per wave in registers.
//
// RP: how many 8-row pieces of a 32-row tile are loaded, staged and summed (4: all).  Up to eight rows need one: the matrix instructions'
// other columns then hold whatever the LDS held, which reaches no sum of a stored row.  Same bits; W4A16, one to eight tokens: 2048 x 2048
// 5.85 -> 5.1 us, 6144 x 2048 6.2 -> 5.5, 2560 x 9728 14.0 -> 11.9 (a GEMV of fp32 FMAs took 5.5 / 5.9 / 15.9 for one token), 22016 x 4096
// 18.9 -> 18.7.
//
// A traits class T supplies Args (tile-independent arguments with members M, N), KB-independent geometry and the operand type:
//   kblocks(a)                        K blocks of 128 activation bytes
//   activations(a) / row_bytes(a)     base and length in bytes of a row (16-byte multiple)
//   struct W                          a block's packed weights of one 32-channel column
//   Col col(a, nb, lane)              per-lane addressing of column block nb
//   load(rsrc, col, kb, W&)           requests a block (past the end: zeros)
//   operand(W, d)                     the lane's operand of matrix instruction d = 0..3
//   mma(w, x, acc), Acc               the instruction, weights first: acc[4g + e] = C[row l % 32][channel 8g + 4 (l / 32) + e]
//   store(a, m, n, sum[4])            epilogue of four consecutive channels (n % 4 == 0; may reach past N)
#pragma once
#include "qcommon.h"

namespace mllmhip {

// (one tile by eight waves: 128 registers, two workgroups per CU)
template <class T, int TM, int TN, int NW, int D, int RP = 4>
__global__ __launch_bounds__(NW * 64, TM * TN == 1 && NW == 8 ? 4 : 1) void wk_gemm_kernel(typename T::Args a) {
  typedef typename T::Acc Acc;  // sixteen 32-bit sums
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 31, hi = lane >> 5;
  const int tilesM = (a.M + 32 * TM - 1) / (32 * TM), tilesN = (a.N + 32 * TN - 1) / (32 * TN);
  // row tiles of one column tile are neighbours on ONE XCD: its L2 fetches their weights once
  const int tile = xcd_run(blockIdx.x, tilesM * tilesN);
  const int m0 = (tile % tilesM) * 32 * TM, n0 = (tile / tilesM) * 32 * TN;

  const uint32_t rowb = (uint32_t)T::row_bytes(a);
  const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(T::activations(a)), 0, (uint32_t)a.M * rowb, 0x00020000);
  const __amdgpu_buffer_rsrc_t rW = T::weights(a);
  // activation piece c of a lane: row 8 c + lane / 8, 16-byte column lane % 8; rows past M repeat the last one (never stored)
  constexpr int CA = RP * TM;
  uint32_t offA[CA];
#pragma unroll
  for (int c = 0; c < CA; c++) offA[c] = (uint32_t)min(m0 + 8 * c + (lane >> 3), a.M - 1) * rowb + (lane & 7) * 16;
  const uint32_t colb = (lane & 7) * 16;
  typename T::Col col[TN];
#pragma unroll
  for (int j = 0; j < TN; j++) col[j] = T::col(a, n0 / 32 + j, lane);

  unsigned char* stage = smem + wave * (TM * 4096);
  unsigned char* wr[2];  // pieces c even / odd: (row / 2) % 8 = 4 (c % 2) + lane / 16
#pragma unroll
  for (int p = 0; p < 2; p++) wr[p] = stage + (lane >> 3) * 128 + (((lane & 7) ^ ((4 * p + (lane >> 4)) & 7)) * 16);
  const unsigned char* rd[4];
#pragma unroll
  for (int d = 0; d < 4; d++) rd[d] = stage + lrow * 128 + (((2 * d + hi) ^ ((lrow >> 1) & 7)) * 16);

  const int nblk = T::kblocks(a);
  const int cnt = wave < nblk ? (nblk - wave + NW - 1) / NW : 0;  // blocks of this wave

  u32x4 ga[D][CA];
  typename T::W w[D][TN];
  auto request = [&](int s, int it) {
    const int kb = wave + it * NW;
    const bool in = it < cnt;
    const bool ok = in && (uint32_t)kb * 128u + colb < rowb;
#pragma unroll
    for (int c = 0; c < CA; c++) ga[s][c] = __builtin_amdgcn_raw_buffer_load_b128(rA, ok ? offA[c] : 0xffffffffu, kb * 128, 0);
#pragma unroll
    for (int j = 0; j < TN; j++) T::load(rW, col[j], in ? kb : -1, w[s][j]);
  };
  Acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0;

#pragma unroll
  for (int s = 0; s < D; s++) request(s, s);
  auto work = [&](int s, int next, bool more) {
#pragma unroll
    for (int c = 0; c < CA; c++) *reinterpret_cast<u32x4*>(wr[c & 1] + c * 1024) = ga[s][c];
    typename T::W wc[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) wc[j] = w[s][j];
    if (more) request(s, next);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 0; d < 4; d++) {
      typename T::X x[TM];
#pragma unroll
      for (int i = 0; i < TM; i++) x[i] = *reinterpret_cast<const typename T::X*>(rd[d] + i * 4096);
#pragma unroll
      for (int j = 0; j < TN; j++) {
        const typename T::X o = T::operand(wc[j], d);
#pragma unroll
        for (int i = 0; i < TM; i++) acc[i][j] = T::mma(o, x[i], acc[i][j]);
      }
    }
  };
  int it = 0;
  for (; it + D <= cnt; it += D) {
#pragma unroll
    for (int s = 0; s < D; s++) work(s, it + s + D, true);
  }
#pragma unroll
  for (int s = 0; s < D - 1; s++)
    if (it + s < cnt) work(s, 0, false);

  // the waves' sums meet in LDS: [wave][i][j][g][half] of 33 16-byte slots (32 rows and one of padding)
  constexpr int PER = TM * TN * 8 * 33;  // slots of a wave
  typedef typename T::Sum4 Sum4;
  __syncthreads();
  Sum4* part = reinterpret_cast<Sum4*>(smem);
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        Sum4 v;
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = acc[i][j][4 * g + e];
        if (RP == 4 || lrow < 8 * RP) part[wave * PER + ((i * TN + j) * 8 + 2 * g + hi) * 33 + lrow] = v;
      }
  __syncthreads();
  // consecutive lanes take consecutive quads of channels of a row
  constexpr int QUADS = 8 * TN, OUT = 8 * RP * TM * QUADS;
#pragma unroll
  for (int o = tid; o < OUT; o += NW * 64) {
    const int q = o % QUADS, m = o / QUADS;
    const int slot = (((m >> 5) * TN + (q >> 3)) * 8 + (q & 7)) * 33 + (m & 31);
    Sum4 v = part[slot];
#pragma unroll
    for (int ww = 1; ww < NW; ww++) v += part[ww * PER + slot];
    if (m0 + m < a.M) T::store(a, m0 + m, n0 + 4 * q, v);
  }
}

template <int TM, int TN, int NW>
constexpr size_t wk_gemm_lds() {
  constexpr size_t stage = (size_t)NW * TM * 4096, sums = (size_t)NW * TM * TN * 8 * 33 * 16;
  return stage > sums ? stage : sums;
}

template <class T, int TM, int TN, int NW, int D, int RP = 4>
int wk_gemm_launch(const typename T::Args& a, hipStream_t st) {
  constexpr size_t lds = wk_gemm_lds<TM, TN, NW>();
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  static_assert(RP == 4 || TM == 1, "fewer rows than a tile: one row tile");
  if (a.M > 8 * RP * TM && RP < 4) return MLLM_HIP_E_BADARG;
  auto kern = wk_gemm_kernel<T, TM, TN, NW, D, RP>;
  if (lds > 64 * 1024)
    HIP_RET(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  const unsigned grid = (unsigned)(((a.M + 32 * TM - 1) / (32 * TM)) * ((a.N + 32 * TN - 1) / (32 * TN)));
  hipLaunchKernelGGL(kern, dim3(grid), dim3(NW * 64), lds, st, a);
  return (int)hipGetLastError();
}

// Tiles of 64 x 64 by four waves, two blocks ahead, two workgroups per CU; where every tile has a CU to itself, by eight: one wave per SIMD
// dequantizes and multiplies in turns, with a second one the two overlap.  Eight / four waves, median (range) over 730 shapes of Q4_0, Q8_0, Q4_K,
// Q6_K and W4A16: 129 to 256 tiles 0.96 (0.91 to 1.02) up to K 1500, 0.93 (0.86 to 0.98) up to 4000, 0.87 (0.82 to 0.99) beyond; 257 to 384 tiles
// 1.02 to 1.25, more 0.99 to 1.44.  Up to six blocks most waves have one block or none (W4A16: four 1.06, six 1.02, eight 0.99).
constexpr int64_t WK_EIGHT_TILES = 256, WK_EIGHT_BLOCKS = 7;
inline bool wk_eight(int64_t M, int64_t N, int64_t blocks) {
  return ((M + 63) / 64) * ((N + 63) / 64) <= WK_EIGHT_TILES && blocks >= WK_EIGHT_BLOCKS;
}
template <class T>
int wk_gemm_64x64(const typename T::Args& a, hipStream_t st) {
  if (wk_eight(a.M, a.N, T::kblocks(a))) return wk_gemm_launch<T, 2, 2, 8, 1>(a, st);
  return wk_gemm_launch<T, 2, 2, 4, 2>(a, st);
}

// What a form of a GEMM is expected to take, in us: fixed + rounds * (round + block * K blocks) + mk * M K + mn * M N (in millions).  A round
// is one tile per CU; up to `cap` tiles share a CU, each further one at `share` of the first, and a partly filled last round counts `whole` of a
// whole one.  The callers' constants are fitted to measured times (each says how well); the form with the least cost is launched.
// Up to 32 rows the choice looks at the tiles alone: a row's bits do not depend on how many rows come with it.
struct FormCost {
  int bm, bn, cap;                    // tile: rows x channels
  float share, whole, fixed, round, block, mk, mn;
};
inline float form_cost(const FormCost& f, int64_t M, int64_t N, int64_t K, int64_t blocks) {
  const int64_t tiles = ((M + f.bm - 1) / f.bm) * ((N + f.bn - 1) / f.bn), chip = 256 * (int64_t)f.cap;
  const float part = (float)tiles / 256.f, m = 1e-6f * (float)(M > 32 ? M : 32);
  float rounds;
  if (tiles <= chip) rounds = 1.f + f.share * (f.whole * (float)((tiles + 255) / 256) + (1.f - f.whole) * (part > 1.f ? part : 1.f) - 1.f);
  else rounds = (1.f + f.share * (float)(f.cap - 1)) * (f.whole * (float)((tiles + chip - 1) / chip) + (1.f - f.whole) * part / (float)f.cap);
  return f.fixed + rounds * (f.round + f.block * (float)blocks) + m * (f.mk * (float)K + f.mn * (float)N);
}

}  // namespace mllmhip

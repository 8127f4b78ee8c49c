// W8A8 Linear for prefill on gfx950: per-token dynamic int8 activation quantization + int8 MFMA GEMM with int32
// accumulation and a per-token x per-channel scale epilogue.
//
// Semantics (the reference's CUDA path, restated):
//   activation quant   pymllm/tests/bench_w8a8_activation_quant.py:20-26
//                      absmax = max(amax|x|, 1e-10); scale = absmax/127; q = clamp(round_half_even(x/scale), -128, 127)
//   GEMM + epilogue    pymllm/quantization/methods/compressed_tensors.py:450-468 (apply)
//                      mllm-kernel/mllm_kernel/cuda/csrc/cutlass_extensions/epilogue/epilogue_per_row_per_col_scale.h:273-280
//                      y = out_dtype( float(acc_int32) * (w_scale[n] * x_scale[m]) + bias[n] )
// The int32 accumulators are exact, so they match any other exact implementation bit for bit.
#include "qcommon.h"
#include <algorithm>

#include "wk_gemm.h"

namespace mllmhip {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// =========================================================================================================
// per-token dynamic quantization: one workgroup per row
// =========================================================================================================
template <int XT>
__device__ __forceinline__ float load_x1(const void* x, int64_t i) {
  return XT == MLLM_HIP_F32 ? reinterpret_cast<const float*>(x)[i] : bf16_to_f32(reinterpret_cast<const uint16_t*>(x)[i]);
}
template <int XT>
__device__ __forceinline__ void load_x8v(const void* x, int64_t i, float (&v)[8]) {
  if (XT == MLLM_HIP_F32) {
    const float4* p = reinterpret_cast<const float4*>(reinterpret_cast<const float*>(x) + i);
    const float4 a = p[0], b = p[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
    const u32x4 r = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(x) + i);
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int j = 0; j < 4; j++) {
      v[2 * j] = __uint_as_float(w[j] << 16);
      v[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
    }
  }
}
__device__ __forceinline__ int quant1(float x, float scale) {
  float r = rintf(x / scale);  // IEEE division, round half to even
  r = fminf(127.f, fmaxf(-128.f, r));
  return (int)r;
}
// Eight codes of a row.  The IEEE division of every element is eleven instructions; with inv = 1 / scale, correctly rounded once per row, a
// product, its remainder and one correction give the correctly rounded quotient (no difference beside any half-way point of the codes for any
// significand of the scale; the remainder is exact unless |x| is below 2^-102, whose code is 0 either way: no scale is below 2^-41).
// |x / scale| <= 127 but for rounding, so that adding 1.5 * 2^23 rounds half to even and leaves the code in the low byte; a NaN becomes -128 as
// above.  scale is infinite only for a row that holds an infinity: inv is 0 then, and with rem_scale 0 in its place the quotients are 0, and
// NaN where x / scale is.
struct RowScale {
  float rem_scale, inv;
};
__device__ __forceinline__ RowScale row_scale(float scale) { return {scale < __builtin_inff() ? scale : 0.f, 1.0f / scale}; }
__device__ __forceinline__ uint2 quant8(const float (&v)[8], RowScale s) {
  uint32_t b[8];
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const float q0 = v[e] * s.inv, q = fmaf(fmaf(-q0, s.rem_scale, v[e]), s.inv, q0);
    b[e] = __float_as_uint(fmaxf(-128.f, q) + 12582912.f);
  }
  return make_uint2(__builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u) | __builtin_amdgcn_perm(b[3], b[2], 0x04000c0cu),
                    __builtin_amdgcn_perm(b[5], b[4], 0x0c0c0400u) | __builtin_amdgcn_perm(b[7], b[6], 0x04000c0cu));
}

// NI > 0: the row (K <= NI * 2048, K % 8 == 0) stays in registers between the maximum and the rounding, eight elements per
// lane and item; NI == 0: any K, the row is read twice (the second time from cache).
template <int XT, int NI>
__global__ __launch_bounds__(256) void per_token_quant_kernel(const void* __restrict__ x, int8_t* __restrict__ q,
                                                              float* __restrict__ scale, int K) {
  __shared__ float s_max[4];
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x;
  const bool vec = (K % 8) == 0;
  const int64_t base = row * K;
  float amax = 0.f;
  float held[NI > 0 ? NI : 1][8];
  if (NI > 0) {
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int k = (tid + 256 * i) * 8;
      load_x8v<XT>(x, base + (k < K ? k : K - 8), held[i]);  // clamped: lanes past the row re-read its tail and are not stored
#pragma unroll
      for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(held[i][e]));
    }
  } else if (vec) {
    for (int k = tid * 8; k < K; k += 256 * 8) {
      float v[8];
      load_x8v<XT>(x, base + k, v);
#pragma unroll
      for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(v[e]));
    }
  } else {
    for (int k = tid; k < K; k += 256) amax = fmaxf(amax, fabsf(load_x1<XT>(x, base + k)));
  }
  // wave max with DPP, then across the four waves through LDS
  amax = fmaxf(amax, dpp_f<0xB1>(amax));
  amax = fmaxf(amax, dpp_f<0x4E>(amax));
  amax = fmaxf(amax, dpp_f<0x141>(amax));
  amax = fmaxf(amax, dpp_f<0x140>(amax));
  amax = max16(amax);
  amax = max32(amax);
  if ((tid & 63) == 0) s_max[tid >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
  amax = fmaxf(amax, 1e-10f);
  const float sc = amax / 127.0f;
  const RowScale rs = row_scale(sc);
  if (tid == 0) scale[row] = sc;
  if (NI > 0) {
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int k = (tid + 256 * i) * 8;
      if (k < K) *reinterpret_cast<uint2*>(q + base + k) = quant8(held[i], rs);
    }
  } else if (vec) {
    for (int k = tid * 8; k < K; k += 256 * 8) {
      float v[8];
      load_x8v<XT>(x, base + k, v);
      *reinterpret_cast<uint2*>(q + base + k) = quant8(v, rs);
    }
  } else {
    for (int k = tid; k < K; k += 256) q[base + k] = (int8_t)quant1(load_x1<XT>(x, base + k), sc);
  }
}

// =========================================================================================================
// int8 GEMM  C[m][n] = sum_k A[m][k] * W[n][k]   (both operands K-contiguous)
// =========================================================================================================
struct W8A8Args {
  const int8_t* A;      // [M][K]
  const int8_t* W;      // [N][K]
  const float* xs;      // [M]
  const float* ws;      // [N]
  const float* bias;    // [N] or null
  uint16_t* C;          // bf16 [M][N] or null
  int32_t* acc;         // int32 [M][N] or null
  int M, N, K;
};

// Workgroup tile BM x BN, K step 64 bytes; waves laid out (BM/WM) x (BN/WN), each owning WM x WN as 32x32 MFMA tiles
// (v_mfma_i32_32x32x32_i8: every lane supplies 16 consecutive k of one row of A and of one row of W).
// Global -> registers -> LDS with the loads of the next D K steps in flight during the MFMAs.  LDS rows are 64 bytes,
// unpadded: measured on MI355X, 16-byte operand reads run at the full LDS rate (about 64 B/clk/CU) for every row stride
// except multiples of 128 bytes.
template <int BM, int BN, int WM, int WN, int D>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64) void w8a8_gemm_kernel(W8A8Args a) {
  constexpr int BK = 64, LDK = 64;
  constexpr int NT = (BM / WM) * (BN / WN) * 64;
  constexpr int CA = BM * 4 / NT, CB = BN * 4 / NT;  // 16-byte chunks per thread and K step
  static_assert(BM * 4 % NT == 0 && BN * 4 % NT == 0, "tile must split evenly over the threads");
  constexpr int TM = WM / 32, TN = WN / 32;
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int STAGE = (BM + BN) * LDK;  // one K step: A rows then W rows

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / (BN / WN), wn = wave % (BN / WN);

  // XCD-aware tile order: workgroup i runs on XCD i % 8, so give each XCD a contiguous run of tiles (same A panel)
  const int tilesN = (a.N + BN - 1) / BN, tilesM = (a.M + BM - 1) / BM;
  const int total = tilesM * tilesN;
  int tile = blockIdx.x;
  if (total % 8 == 0) tile = (blockIdx.x % 8) * (total / 8) + blockIdx.x / 8;
  const int m0 = (tile / tilesN) * BM, n0 = (tile % tilesN) * BN;

  const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.A), 0, (uint32_t)((int64_t)a.M * a.K), 0x00020000);
  const __amdgpu_buffer_rsrc_t rW = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.W), 0, (uint32_t)((int64_t)a.N * a.K), 0x00020000);

  // chunk c of a thread: row = (tid + c*NT) / 4, 16-byte column = (tid + c*NT) % 4
  uint32_t offA[CA], offB[CB];
#pragma unroll
  for (int c = 0; c < CA; c++) {
    const int idx = tid + c * NT, row = m0 + idx / 4;
    offA[c] = row < a.M ? (uint32_t)((int64_t)row * a.K + (idx % 4) * 16) : 0xffffffffu;
  }
#pragma unroll
  for (int c = 0; c < CB; c++) {
    const int idx = tid + c * NT, row = n0 + idx / 4;
    offB[c] = row < a.N ? (uint32_t)((int64_t)row * a.K + (idx % 4) * 16) : 0xffffffffu;
  }
  // D register sets hold the global loads of the next D K steps while they are in flight (HBM/L2 latency is several
  // K steps of MFMA work); loads are issued unconditionally (past K they are out of range or unused) so that the
  // hardware wait counters stay exact.
  u32x4 gA[D][CA], gB[D][CB];
  auto gload = [&](int k0, u32x4 (&ga)[CA], u32x4 (&gb)[CB]) {
#pragma unroll
    for (int c = 0; c < CA; c++) {
      const bool ok = offA[c] != 0xffffffffu && k0 + ((tid + c * NT) % 4) * 16 < a.K;
      ga[c] = __builtin_amdgcn_raw_buffer_load_b128(rA, ok ? offA[c] + k0 : 0xffffffffu, 0, 0);
    }
#pragma unroll
    for (int c = 0; c < CB; c++) {
      const bool ok = offB[c] != 0xffffffffu && k0 + ((tid + c * NT) % 4) * 16 < a.K;
      gb[c] = __builtin_amdgcn_raw_buffer_load_b128(rW, ok ? offB[c] + k0 : 0xffffffffu, 0, 0);
    }
  };
  auto sstore = [&](int buf, const u32x4 (&ga)[CA], const u32x4 (&gb)[CB]) {
#pragma unroll
    for (int c = 0; c < CA; c++) {
      const int idx = tid + c * NT;
      *reinterpret_cast<u32x4*>(smem + buf * STAGE + (idx / 4) * LDK + (idx % 4) * 16) = ga[c];
    }
#pragma unroll
    for (int c = 0; c < CB; c++) {
      const int idx = tid + c * NT;
      *reinterpret_cast<u32x4*>(smem + buf * STAGE + (BM + idx / 4) * LDK + (idx % 4) * 16) = gb[c];
    }
  };

  v16i acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0;

  const int KT = (a.K + BK - 1) / BK;
  // K step s lives in register set s % D from its issue until it is written to LDS buffer s % 2 one step before use
#pragma unroll
  for (int d = 0; d < D; d++) gload(d * BK, gA[d], gB[d]);
  sstore(0, gA[0], gB[0]);
  __syncthreads();
  const int lrow = lane & 31, lk = (lane >> 5) * 16;
  for (int kt0 = 0; kt0 < KT; kt0 += D) {
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int kt = kt0 + d;
      if (kt < KT) {  // uniform
        const int buf = kt & 1;
        gload((kt + D) * BK, gA[d], gB[d]);  // set d was written to LDS one step ago: free again
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
          v4i fa[TM], fb[TN];
#pragma unroll
          for (int i = 0; i < TM; i++)
            fa[i] = *reinterpret_cast<const v4i*>(smem + buf * STAGE + (wm * WM + i * 32 + lrow) * LDK + ks * 32 + lk);
#pragma unroll
          for (int j = 0; j < TN; j++)
            fb[j] = *reinterpret_cast<const v4i*>(smem + buf * STAGE + (BM + wn * WN + j * 32 + lrow) * LDK + ks * 32 + lk);
#pragma unroll
          for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
        sstore(buf ^ 1, gA[(d + 1) % D], gB[(d + 1) % D]);  // K step kt + 1
        __syncthreads();
      }
    }
  }

  // epilogue.  32x32 accumulator layout: register r of lane l holds row 8*(r/4) + 4*(l/32) + r%4, column l%32.
  // The row / column scales and the bias of the tile go through LDS once (the staging buffers are free after the last
  // barrier), so the per-element work is three fp32 operations and a store, with no loads or branches on full tiles.
  float* sXs = reinterpret_cast<float*>(smem);
  float* sWs = sXs + BM;
  float* sBi = sWs + BN;
  for (int i = tid; i < BM; i += NT) sXs[i] = (a.xs && m0 + i < a.M) ? a.xs[m0 + i] : 0.f;
  for (int i = tid; i < BN; i += NT) {
    sWs[i] = (a.ws && n0 + i < a.N) ? a.ws[n0 + i] : 0.f;
    sBi[i] = (a.bias && n0 + i < a.N) ? a.bias[n0 + i] : 0.f;
  }
  __syncthreads();
  const bool full = m0 + BM <= a.M && n0 + BN <= a.N;
  const int hi4 = 4 * (lane >> 5);
#pragma unroll
  for (int j = 0; j < TN; j++) {
    const int cn = wn * WN + j * 32 + lrow;
    const int n = n0 + cn;
    const bool nok = n < a.N;
    const float wsn = sWs[cn], bn = sBi[cn];
#pragma unroll
    for (int i = 0; i < TM; i++) {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int rm = wm * WM + i * 32 + 8 * g + hi4;  // first of four consecutive rows
        const f32x4 xs4 = *reinterpret_cast<const f32x4*>(&sXs[rm]);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int m = m0 + rm + e;
          const int v = acc[i][j][4 * g + e];
          if (full || (nok && m < a.M)) {
            if (a.acc) a.acc[(int64_t)m * a.N + n] = v;
            if (a.C) {
              float f = (float)v * (wsn * xs4[e]);
              if (a.bias) f += bn;
              a.C[(int64_t)m * a.N + n] = f32_to_bf16(f);
            }
          }
        }
      }
    }
  }
}

// Weight layout for the large-problem kernel below: the matrix in v_mfma_i32_32x32x32_i8 operand order.  Block (nb, kb)
// of 32 rows x 32 bytes is 1 KB, lane l = (row l%32, k-half l/32) owns bytes [16 l, 16 l + 16); blocks are ordered
// [nb][kb] with N padded to 32 and K to 128 by zeros.  A wave's 16-byte operand load then reads one contiguous KB
// (8 cache lines) instead of 32 bytes from each of 32 rows (32 cache lines, each touched again by the next three loads).
__host__ __device__ inline int64_t w8a8_packed_k(int64_t K) { return (K + 127) / 128 * 128; }
__host__ __device__ inline int64_t w8a8_packed_n(int64_t N) { return (N + 31) / 32 * 32; }

__global__ __launch_bounds__(256) void w8a8_prepack_kernel(const int8_t* __restrict__ W, u32x4* __restrict__ P, int N, int K,
                                                           int64_t chunks) {
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;  // one 16-byte piece of the packed matrix
  if (c >= chunks) return;
  const int kbs = (int)(w8a8_packed_k(K) / 32);
  const int l = (int)(c % 64);
  const int64_t blk = c / 64;
  const int kb = (int)(blk % kbs), nb = (int)(blk / kbs);
  const int n = nb * 32 + (l & 31), k = kb * 32 + (l >> 5) * 16;
  u32x4 v = {0, 0, 0, 0};
  if (n < N && k < K) v = *reinterpret_cast<const u32x4*>(W + (int64_t)n * K + k);  // K % 16 == 0
  P[c] = v;
}

// Large-problem kernel.  Measured on this part: a 16-byte LDS read of a whole wave occupies the CU's LDS pipe for 16
// cycles (64 B/clk/CU) while one v_mfma_i32_32x32x32_i8 occupies a SIMD for 32, so a wave that pulls both operands of a
// 64x64 tile through LDS is LDS-bound at under half the matrix rate.  Here only the activation tile goes through LDS;
// the four waves of a workgroup sit side by side along N, each owns (32 TM) x (32 TN) outputs and fetches ITS weight
// operands straight from global memory into registers in MFMA layout, one K step (128 bytes) ahead: every operand
// register is reloaded for the next step right after its last use.  PK: weights in the prepacked layout above; else
// the plain [N][K] matrix with K % 128 == 0.
// The weights are the MFMA's first operand, so that a lane ends up with four CONSECUTIVE output columns per row.
// Scheduling barriers pin the hand-made software pipeline: left alone, the compiler sinks all global loads to the end
// of the loop body and exposes their latency.
// WPS: waves per SIMD the register budget is held to (workgroups of 4 waves: WPS workgroups per CU).
// G == 2: eight waves, the second four take the second half of K with a stage of their own; their sums join the first's in LDS (exact).
template <int TM, int TN, bool PK, int WPS, int G = 1>
__global__ __launch_bounds__(256 * G) __attribute__((amdgpu_waves_per_eu(WPS, WPS))) void w8a8_gemm_nsplit_kernel(W8A8Args a) {
  constexpr int BK = 128, LDK = 144, KS = BK / 32;
  constexpr int BM = TM * 32, WN = TN * 32, BN = 4 * WN;
  constexpr int CA = BM * (BK / 16) / 256;  // 16-byte activation chunks per thread and K step
  constexpr int STAGE = BM * LDK;
  extern __shared__ __align__(16) unsigned char smem_all[];

  const int group = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  unsigned char* const smem = smem_all + group * 2 * STAGE;
  const int tid = G == 1 ? threadIdx.x : threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
  const int lrow = lane & 31, hi = lane >> 5;
  const int tilesN = (a.N + BN - 1) / BN, tilesM = (a.M + BM - 1) / BM;
  const int tile = xcd_run(blockIdx.x, tilesM * tilesN);           // one run of tiles per XCD ...
  const int m0 = (tile % tilesM) * BM, n0 = (tile / tilesM) * BN;  // ... that shares a slice of the weights

  // Rows past the end are clamped to the last row (their results are never stored).  Activation bytes past K belong to
  // the next row and meet zero weights (PK) or do not occur (K % 128 == 0); reads past the buffers return zero.
  const int Kw = PK ? (int)w8a8_packed_k(a.K) : a.K;
  const int64_t wbytes = PK ? w8a8_packed_n(a.N) * Kw : (int64_t)a.N * a.K;
  const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.A), 0, (uint32_t)((int64_t)a.M * a.K), 0x00020000);
  const __amdgpu_buffer_rsrc_t rW = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.W), 0, (uint32_t)wbytes, 0x00020000);
  uint32_t offA[CA];
#pragma unroll
  for (int c = 0; c < CA; c++) {
    const int idx = tid + c * 256;
    offA[c] = (uint32_t)((int64_t)min(m0 + idx / 8, a.M - 1) * a.K + (idx % 8) * 16);
  }
  uint32_t offB[TN];
#pragma unroll
  for (int j = 0; j < TN; j++) {
    const int nrow = n0 + wave * WN + j * 32;
    offB[j] = PK ? (uint32_t)((int64_t)min(nrow, (int)w8a8_packed_n(a.N) - 32) * Kw + lane * 16)
                 : (uint32_t)((int64_t)min(nrow + lrow, a.N - 1) * a.K + hi * 16);
  }

  auto loadA = [&](int k0, u32x4 (&ga)[CA]) {
#pragma unroll
    for (int c = 0; c < CA; c++) ga[c] = __builtin_amdgcn_raw_buffer_load_b128(rA, offA[c], k0, 0);
  };
  auto storeA = [&](int buf, const u32x4 (&ga)[CA]) {
#pragma unroll
    for (int c = 0; c < CA; c++) {
      const int idx = tid + c * 256;
      *reinterpret_cast<u32x4*>(smem + buf * STAGE + (idx / 8) * LDK + (idx % 8) * 16) = ga[c];
    }
  };
  auto loadB = [&](int k0, int ks, int j) -> v4i {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rW, offB[j], (k0 + ks * 32) * (PK ? 32 : 1), 0);
    return v4i{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
  };
  auto readA = [&](int buf, int ks, v4i (&fa)[TM]) {
#pragma unroll
    for (int i = 0; i < TM; i++)
      fa[i] = *reinterpret_cast<const v4i*>(smem + buf * STAGE + (i * 32 + lrow) * LDK + ks * 32 + hi * 16);
  };

  v16i acc[TN][TM];
#pragma unroll
  for (int j = 0; j < TN; j++)
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[j][i][r] = 0;

  // K steps of these waves: all of them, or one of the halves (idle: how many fewer the second has, whose barriers it keeps)
  const int KT = Kw / BK, per = (KT + G - 1) / G, kt0 = group * per, kt1 = min(KT, kt0 + per), idle = G == 1 ? 0 : per - (kt1 - kt0);
  u32x4 ga[CA];
  v4i fb[KS][TN];
  v4i fa[2][TM];
  loadA(kt0 * BK, ga);
#pragma unroll
  for (int ks = 0; ks < KS; ks++)
#pragma unroll
    for (int j = 0; j < TN; j++) fb[ks][j] = loadB(kt0 * BK, ks, j);
  storeA(0, ga);
  __syncthreads();
  readA(0, 0, fa[0]);

  for (int kt = kt0; kt < kt1; kt++) {
    const int buf = (kt - kt0) & 1, k1 = (kt + 1) * BK;
    loadA(k1, ga);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      if (ks < KS - 1) {
        readA(buf, ks + 1, fa[(ks + 1) & 1]);  // the next sub-step's activations while this one's MFMAs run
      } else {
        storeA(buf ^ 1, ga);  // free since the previous barrier; its loads were issued a whole K step ago
        __syncthreads();
        readA(buf ^ 1, 0, fa[(ks + 1) & 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < TN; j++) {
#pragma unroll
        for (int i = 0; i < TM; i++)
          acc[j][i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[ks][j], fa[ks & 1][i], acc[j][i], 0, 0, 0);
        fb[ks][j] = loadB(k1, ks, j);  // the operand of the next K step, into the register that just became free
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  for (int i = 0; i < idle; i++) __syncthreads();
  __syncthreads();  // all LDS reads done before the scales overwrite the tiles
  if constexpr (G == 2) {
    v4i* part = reinterpret_cast<v4i*>(smem_all);
    auto quad = [&](int j, int i, int g) -> v4i& { return part[(((wave * TN + j) * TM + i) * 4 + g) * 64 + lane]; };
    if (group == 1) {
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int g = 0; g < 4; g++) quad(j, i, g) = v4i{acc[j][i][4 * g], acc[j][i][4 * g + 1], acc[j][i][4 * g + 2], acc[j][i][4 * g + 3]};
    }
    __syncthreads();
    if (group == 0) {
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int g = 0; g < 4; g++) {
            const v4i v = quad(j, i, g);
#pragma unroll
            for (int e = 0; e < 4; e++) acc[j][i][4 * g + e] += v[e];
          }
    }
    __syncthreads();
  }

  // acc[j][i][4g+e] = C[m0 + 32i + lrow][n0 + wave*WN + 32j + 8g + 4hi + e]
  float* sXs = reinterpret_cast<float*>(smem_all);
  float* sWs = sXs + BM;
  float* sBi = sWs + BN;
  for (int i = tid; i < BM; i += 256) sXs[i] = (a.xs && m0 + i < a.M) ? a.xs[m0 + i] : 0.f;
  for (int i = tid; i < BN; i += 256) {
    sWs[i] = (a.ws && n0 + i < a.N) ? a.ws[n0 + i] : 0.f;
    sBi[i] = (a.bias && n0 + i < a.N) ? a.bias[n0 + i] : 0.f;
  }
  __syncthreads();
  // bf16 output only: the column scales sit in registers, and each 32-row slab
  // of results is turned through LDS so that a wave stores whole rows of the workgroup's BN columns (runs of whole
  // cache lines, 16 bytes per lane).
  constexpr int ROWB = 2 * BN + 16;
  unsigned char* patch = smem_all + 4096;
  static_assert((BM + 2 * BN) * 4 <= 4096, "scales overlap the store patch");
  // 16-byte pieces; those of ragged edges fall outside the buffer (whose end a row or column past the tile must not wrap over)
  const bool pieces = a.N % 8 == 0 && reinterpret_cast<uintptr_t>(a.C) % 16 == 0 && ((int64_t)a.M + BM) * a.N * 2 < ((int64_t)1 << 32);
  if (pieces && a.C && !a.acc) {
    const __amdgpu_buffer_rsrc_t rC = __builtin_amdgcn_make_buffer_rsrc(a.C, 0, (uint32_t)((int64_t)a.M * a.N * 2), 0x00020000);
    f32x4 ws4[TN][4], bi4[TN][4];
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        ws4[j][g] = *reinterpret_cast<const f32x4*>(&sWs[wave * WN + j * 32 + 8 * g + 4 * hi]);
        bi4[j][g] = *reinterpret_cast<const f32x4*>(&sBi[wave * WN + j * 32 + 8 * g + 4 * hi]);
      }
    const bool has_bias = a.bias != nullptr;
    constexpr int CPR = BN / 8;  // 16-byte pieces per row
    constexpr int RPW = 8 / G;   // rows per wave
    static_assert((RPW * CPR) % 64 == 0, "a wave stores whole rows");
#pragma unroll
    for (int i = 0; i < TM; i++) {
      const float xsm = sXs[i * 32 + lrow];
      if (group == 0) {
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int g = 0; g < 4; g++) {
            float f[4];
#pragma unroll
            for (int e = 0; e < 4; e++) f[e] = (float)acc[j][i][4 * g + e] * (ws4[j][g][e] * xsm);
            if (has_bias) {
#pragma unroll
              for (int e = 0; e < 4; e++) f[e] += bi4[j][g][e];
            }
            *reinterpret_cast<uint2*>(patch + lrow * ROWB + (wave * WN + j * 32 + 8 * g + 4 * hi) * 2) =
                uint2{pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3])};
          }
      }
      __syncthreads();
#pragma unroll
      for (int t = 0; t < RPW * CPR / 64; t++) {  // wave w stores rows RPW w .. RPW (w + 1) - 1
        const int c = lane + 64 * t;
        const int row = (group * 4 + wave) * RPW + c / CPR, cc = c % CPR;
        const u32x4 v = *reinterpret_cast<const u32x4*>(patch + row * ROWB + cc * 16);
        const int n = n0 + cc * 8;
        // (a row past M lies past the end of the buffer)
        __builtin_amdgcn_raw_buffer_store_b128(v, rC, n < a.N ? (uint32_t)(m0 + i * 32 + row) * (uint32_t)a.N * 2u + (uint32_t)n * 2u : 0xffffffffu, 0, 0);
      }
      if (i + 1 < TM) __syncthreads();
    }
    return;
  }
  if (group != 0) return;
#pragma unroll
  for (int i = 0; i < TM; i++) {
    const int m = m0 + i * 32 + lrow;
    const float xsm = sXs[i * 32 + lrow];
#pragma unroll
    for (int j = 0; j < TN; j++) {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int cn = wave * WN + j * 32 + 8 * g + 4 * hi;
        const int n = n0 + cn;
        const f32x4 ws4 = *reinterpret_cast<const f32x4*>(&sWs[cn]);
        const f32x4 bi4 = *reinterpret_cast<const f32x4*>(&sBi[cn]);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          if (m < a.M && n + e < a.N) {
            const int v = acc[j][i][4 * g + e];
            if (a.acc) a.acc[(int64_t)m * a.N + n + e] = v;
            if (a.C) {
              float f = (float)v * (ws4[e] * xsm);
              if (a.bias) f += bi4[e];
              a.C[(int64_t)m * a.N + n + e] = (uint16_t)pack_bf16(f, 0.f);
            }
          }
        }
      }
    }
  }
}

template <int TM, int TN, bool PK, int WPS>
static int launch_w8a8_nsplit(const W8A8Args& a, hipStream_t st) {
  constexpr int BM = TM * 32, BN = 4 * TN * 32;
  constexpr size_t stage = 2 * (size_t)BM * 144, patch = 4096 + 32 * (2 * (size_t)BN + 16);
  const size_t lds = stage > patch ? stage : patch;
  const unsigned grid = (unsigned)(((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN));
  hipLaunchKernelGGL((w8a8_gemm_nsplit_kernel<TM, TN, PK, WPS>), dim3(grid), dim3(256), lds, st, a);
  return (int)hipGetLastError();
}

// K in halves, eight waves per tile
template <int TM, int TN>
static int launch_w8a8_halves(const W8A8Args& a, hipStream_t st) {
  constexpr int BM = TM * 32, BN = 4 * TN * 32;
  constexpr size_t stage = 4 * (size_t)BM * 144, patch = 4096 + 32 * (2 * (size_t)BN + 16), sums = (size_t)BM * BN * 4;
  constexpr size_t lds = std::max(stage, std::max(patch, sums));
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  auto kern = w8a8_gemm_nsplit_kernel<TM, TN, true, 2, 2>;
  if (lds > 64 * 1024)
    HIP_RET(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  const unsigned grid = (unsigned)(((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN));
  hipLaunchKernelGGL(kern, dim3(grid), dim3(512), lds, st, a);
  return (int)hipGetLastError();
}

static int g_w8a8_ntile = 0;  // weights-from-global kernel: 0 = heuristic, 1 = 128x384, 2 = 64x384, 3 = 128x128, 4 = 64x128, 5 = 128x256

// Tile choice for the weights-from-global kernel: the biggest tile that still gives every CU work.
template <bool PK>
static int launch_w8a8_nsplit_auto(const W8A8Args& a, hipStream_t st) {
  auto tiles = [&](int bm, int bn) { return (int64_t)((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn); };
  int t = g_w8a8_ntile;
  if (!t) {
    if (a.M > 64 && tiles(128, 384) >= 192) t = 1;
    else if (tiles(64, 384) >= 192 || a.N <= 128) t = 2;
    else if (a.M > 64 && tiles(128, 128) >= 192) t = 3;
    else t = 4;
  }
  switch (t) {
    case 1: return launch_w8a8_nsplit<4, 3, PK, 1>(a, st);
    case 2: return launch_w8a8_nsplit<2, 3, PK, 2>(a, st);
    case 3: return launch_w8a8_nsplit<4, 1, PK, 2>(a, st);
    case 5: return launch_w8a8_nsplit<4, 2, PK, 2>(a, st);
    default: return launch_w8a8_nsplit<2, 1, PK, 2>(a, st);
  }
}

template <int BM, int BN, int WM, int WN, int D>
static int launch_w8a8(const W8A8Args& a, hipStream_t st) {
  constexpr int NT = (BM / WM) * (BN / WN) * 64;
  const size_t lds = 2 * (size_t)(BM + BN) * 64;
  const unsigned grid = (unsigned)(((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN));
  auto kern = w8a8_gemm_kernel<BM, BN, WM, WN, D>;
  if (lds > 64 * 1024)
    HIP_RET(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(kern, dim3(grid), dim3(NT), lds, st, a);
  return (int)hipGetLastError();
}

static int g_w8a8_tile = 0;  // 0 = heuristic, 1 = 256x192, 2 = 128x128, 3 = 64x64, 4 = weights-from-global tiles

}  // namespace mllmhip

using namespace mllmhip;

MLLM_API int mllm_hip_w8a8_set_tuning(int tile) {
  if (tile < 0 || tile > 4) return MLLM_HIP_E_BADARG;
  g_w8a8_tile = tile;
  return 0;
}

// ---- decode: a few tokens against the prepacked weights --------------------------------------------------------------------
// The tile kernels above spend a 128-row tile on a decode token and leave most CUs idle (9728 x 2560 at one token: 16 us;
// 2560 x 9728: 41 us).  Here a workgroup takes one block row of the packed matrix (32 weight rows) and its waves stride over
// the K blocks, eight 1 KB blocks requested per wave before the first is multiplied (the first batch ahead of the copy of
// the tokens' codes into LDS, which it does not depend on); v_dot4_i32_i8 sums, the two K halves of a block met by a wave
// shuffle, the waves through LDS.  Integer sums are exact: the epilogue is the tile kernels' and so are the bits.
//
// XT: the tokens themselves instead of their codes: every workgroup quantizes all of them while its first weights are on their way, the waves
// divided among the tokens, in place of a launch of its own (about 2.5 us).  Same codes, scales and results.  us, quantized in a launch before /
// here: one token of 1536 x 2048 5.6 / 4.2, 3584 x 3584 6.1 / 4.8, 18 944 x 3584 15.1 / 13.9, 3584 x 18 944 21.6 / 15.3; two of 4096 x 4096
// 7.1 / 5.8; four of 2048 x 6144 9.7 / 8.8.  Two workgroups per CU have to fit (64 VGPRs): with 76, 18 944 x 3584 takes 16.8.
constexpr int W8G_MAXW = 16;
constexpr int W8G_CODES = -1;
template <int MT, int XT>
__global__ __launch_bounds__(W8G_MAXW * 64) __attribute__((amdgpu_waves_per_eu(8))) void w8a8_gemv_packed_kernel(W8A8Args a, const void* x) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int Kp = (int)w8a8_packed_k(a.K), kbs = Kp / 32;
  u32x4* sx = reinterpret_cast<u32x4*>(smem);                          // [MT][Kp / 16] the tokens' codes, zero past K and M
  int* s_part = reinterpret_cast<int*>(smem + (size_t)MT * Kp);        // [wave][MT][32]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nthreads = blockDim.x, nwaves = nthreads >> 6;
  const int r = lane & 31, h = lane >> 5;
  const int nb = blockIdx.x;
  const u32x4* P = reinterpret_cast<const u32x4*>(a.W) + (size_t)nb * kbs * 64 + lane;
  constexpr int UB = 8;
  u32x4 wv[UB];
  auto load_batch = [&](int kb0) {
#pragma unroll
    for (int u = 0; u < UB; u++) {
      const int kb = kb0 + u * nwaves;
      wv[u] = u32x4{0u, 0u, 0u, 0u};
      if (kb < kbs) wv[u] = P[(size_t)kb * 64];
    }
  };
  load_batch(wave);
  const int cpr = Kp / 16;  // 16-byte pieces per token
  __shared__ float s_max[W8G_MAXW], s_scale[MT];
  if constexpr (XT != W8G_CODES) {
    constexpr int HELD = 1;                                   // items of eight elements that stay in registers (two: 76 VGPRs)
    const int wpt = nwaves / MT, step = wpt * 64;             // (at least one wave per token; nwaves a multiple of MT)
    const int m = wave / wpt, t = tid - m * step;
    const int64_t base = (int64_t)min(m, a.M - 1) * a.K;
    float held[HELD][8], amax = 0.f;
    auto item = [&](int c, float (&v)[8]) { load_x8v<XT>(x, base + min(c * 8, a.K - 8), v); };  // (past the row: its tail again)
    auto most = [&](const float (&v)[8]) {
#pragma unroll
      for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(v[e]));
    };
#pragma unroll
    for (int i = 0; i < HELD; i++) item(t + i * step, held[i]);
#pragma unroll
    for (int i = 0; i < HELD; i++) most(held[i]);
    for (int c = t + HELD * step; c * 8 < a.K; c += step) {
      float v[8];
      item(c, v);
      most(v);
    }
    amax = fmaxf(amax, dpp_f<0xB1>(amax));
    amax = fmaxf(amax, dpp_f<0x4E>(amax));
    amax = fmaxf(amax, dpp_f<0x141>(amax));
    amax = fmaxf(amax, dpp_f<0x140>(amax));
    amax = max16(amax);
    amax = max32(amax);
    if (lane == 0) s_max[wave] = amax;
    __syncthreads();
    for (int w = 0; w < wpt; w++) amax = fmaxf(amax, s_max[m * wpt + w]);
    const float sc = fmaxf(amax, 1e-10f) / 127.0f;
    const RowScale rs = row_scale(sc);
    if (t == 0) s_scale[m] = sc;
    uint2* row = reinterpret_cast<uint2*>(sx + m * cpr);
    auto put = [&](int c, const float (&v)[8]) {
      if (c * 8 < Kp) row[c] = c * 8 < a.K && m < a.M ? quant8(v, rs) : make_uint2(0u, 0u);
    };
#pragma unroll
    for (int i = 0; i < HELD; i++) put(t + i * step, held[i]);
    for (int c = t + HELD * step; c * 8 < Kp; c += step) {
      float v[8];
      item(c, v);
      put(c, v);
    }
  } else
  for (int i = tid; i < MT * cpr; i += nthreads) {
    const int m = i / cpr, c = i - m * cpr;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (m < a.M && c * 16 < a.K) v = *reinterpret_cast<const u32x4*>(a.A + (size_t)m * a.K + c * 16);  // K % 16 == 0
    sx[i] = v;
  }
  __syncthreads();
  int acc[MT];
#pragma unroll
  for (int m = 0; m < MT; m++) acc[m] = 0;
  for (int kb0 = wave; kb0 < kbs; kb0 += nwaves * UB) {
    if (kb0 != wave) load_batch(kb0);
#pragma unroll
    for (int u = 0; u < UB; u++) {
      const int kb = kb0 + u * nwaves;
      if (kb < kbs) {  // uniform
#pragma unroll
        for (int m = 0; m < MT; m++) {
          const u32x4 xv = sx[m * cpr + kb * 2 + h];
          int s = acc[m];
          s = __builtin_amdgcn_sdot4((int)wv[u].x, (int)xv.x, s, false);
          s = __builtin_amdgcn_sdot4((int)wv[u].y, (int)xv.y, s, false);
          s = __builtin_amdgcn_sdot4((int)wv[u].z, (int)xv.z, s, false);
          s = __builtin_amdgcn_sdot4((int)wv[u].w, (int)xv.w, s, false);
          acc[m] = s;
        }
      }
    }
  }
#pragma unroll
  for (int m = 0; m < MT; m++) {
    acc[m] = sum32(acc[m]);
    if (h == 0) s_part[(wave * MT + m) * 32 + r] = acc[m];
  }
  __syncthreads();
  for (int i = tid; i < MT * 32; i += nthreads) {
    const int m = i >> 5, n = nb * 32 + (i & 31);
    if (m < a.M && n < a.N) {
      int v = 0;
      for (int w = 0; w < nwaves; w++) v += s_part[(w * MT + m) * 32 + (i & 31)];
      if (a.acc) a.acc[(int64_t)m * a.N + n] = v;
      if (a.C) {
        float f = (float)v * (a.ws[n] * (XT == W8G_CODES ? a.xs[m] : s_scale[m]));
        if (a.bias) f += a.bias[n];
        a.C[(int64_t)m * a.N + n] = (uint16_t)pack_bf16(f, 0.f);
      }
    }
  }
}
// The packed matrix as wk_gemm.h reads it: a block is 128 elements, operand d the 16 bytes of the lane's row in the d-th 32 of them.
// Integer sums are exact, the epilogue is the tile kernels': the same bits as every other form.
struct W8A8Waves {
  typedef W8A8Args Args;
  typedef v16i Acc;
  typedef v4i Sum4;
  typedef v4i X;
  struct W {
    u32x4 q[4];
  };
  typedef uint32_t Col;
  static __host__ __device__ __forceinline__ int kblocks(const Args& a) { return (a.K + 127) / 128; }
  static __device__ __forceinline__ int row_bytes(const Args& a) { return a.K; }
  static __device__ __forceinline__ const void* activations(const Args& a) { return a.A; }
  static __device__ __forceinline__ __amdgpu_buffer_rsrc_t weights(const Args& a) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.W), 0, (uint32_t)(w8a8_packed_n(a.N) * w8a8_packed_k(a.K)), 0x00020000);
  }
  static __device__ __forceinline__ Col col(const Args& a, int nb, int lane) {
    nb = min(nb, (int)(w8a8_packed_n(a.N) / 32) - 1);
    return (uint32_t)((int64_t)nb * 32 * w8a8_packed_k(a.K) + lane * 16);
  }
  static __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, Col c, int kb, W& w) {
#pragma unroll
    for (int d = 0; d < 4; d++) w.q[d] = __builtin_amdgcn_raw_buffer_load_b128(r, kb < 0 ? 0xffffffffu : c + d * 1024, kb * 4096, 0);
  }
  static __device__ __forceinline__ X operand(const W& w, int d) { return __builtin_bit_cast(v4i, w.q[d]); }
  static __device__ __forceinline__ Acc mma(const X& w, const X& x, const Acc& acc) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(w, x, acc, 0, 0, 0); }
  static __device__ __forceinline__ void store(const Args& a, int m, int n, const v4i& v) {
    const int64_t at = (int64_t)m * a.N + n;
    float f[4];
    if (a.C) {
      const float xs = a.xs[m];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        f[e] = n + e < a.N ? (float)v[e] * (a.ws[n + e] * xs) : 0.f;
        if (a.bias && n + e < a.N) f[e] += a.bias[n + e];
      }
      if (n + 3 < a.N && a.N % 4 == 0 && reinterpret_cast<uintptr_t>(a.C) % 8 == 0) {
        *reinterpret_cast<uint2*>(a.C + at) = uint2{pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3])};
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (n + e < a.N) a.C[at + e] = (uint16_t)pack_bf16(f[e], 0.f);
      }
    }
    if (a.acc) {
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (n + e < a.N) a.acc[at + e] = v[e];
    }
  }
};
static int g_w8a8_decode = 1;  // 0: only the weights-from-global tiles (comparison runs and tests)
static int g_w8a8_decode_mfma_from = 5;  // token counts from this one up take the matrix cores (at four tokens the two are even: 6144 x 2048
                                         // 5.9 us here, 6.1 there; 2560 x 9728 10.4 against 9.5; at one 5.3 / 6.1 and 8.1 / 9.4)
// false where the dot kernel does not apply; x: the tokens (a.A and a.xs are not read then), null: their codes
static bool launch_w8a8_gemv_packed(const W8A8Args& a, hipStream_t st, int* rc, const void* x = nullptr, int x_dtype = 0) {
  if (a.M >= g_w8a8_decode_mfma_from || !g_w8a8_decode) return false;
  const int Kp = (int)w8a8_packed_k(a.K), kbs = Kp / 32;
  const int nwaves = kbs >= 32 ? W8G_MAXW : 4;
  if (a.M > (x ? 4 : 8)) return false;
  // Three and four tokens are quantized by every workgroup only while there are few of them: four of 4096 (weights' rows 8192 / 10 240 / 12 288)
  // 8.6 -> 7.7 us, 13.1 -> 12.7, 12.3 -> 12.7; three of 3584 x 18 944 17.2 -> 18.4.  One and two gain up to 4748 workgroups.
  if (x && a.M > 2 && w8a8_packed_n(a.N) / 32 > 320) return false;
  const int MT = a.M <= 1 ? 1 : (a.M <= 2 ? 2 : (a.M <= 4 ? 4 : 8));
  const size_t lds = (size_t)MT * Kp + (size_t)nwaves * MT * 32 * 4;
  if (lds > (x ? 159u : 160u) * 1024) return false;
  const dim3 grid((unsigned)(w8a8_packed_n(a.N) / 32));
  auto go = [&](auto kern) {
    if (lds > 63 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
      return (int)hipGetLastError();
    hipLaunchKernelGGL(kern, grid, dim3(nwaves * 64), lds, st, a, x);
    return (int)hipGetLastError();
  };
  if (!x)
    *rc = MT == 1   ? go(w8a8_gemv_packed_kernel<1, W8G_CODES>)
          : MT == 2 ? go(w8a8_gemv_packed_kernel<2, W8G_CODES>)
          : MT == 4 ? go(w8a8_gemv_packed_kernel<4, W8G_CODES>)
                    : go(w8a8_gemv_packed_kernel<8, W8G_CODES>);
  else if (x_dtype == MLLM_HIP_F32)
    *rc = MT == 1   ? go(w8a8_gemv_packed_kernel<1, MLLM_HIP_F32>)
          : MT == 2 ? go(w8a8_gemv_packed_kernel<2, MLLM_HIP_F32>)
                    : go(w8a8_gemv_packed_kernel<4, MLLM_HIP_F32>);
  else
    *rc = MT == 1   ? go(w8a8_gemv_packed_kernel<1, MLLM_HIP_BF16>)
          : MT == 2 ? go(w8a8_gemv_packed_kernel<2, MLLM_HIP_BF16>)
                    : go(w8a8_gemv_packed_kernel<4, MLLM_HIP_BF16>);
  return true;
}
// Whether a tile form runs as halves of K by eight waves: up to 256 tiles every tile has a CU to itself, and one wave per SIMD waits for its own
// loads; above that two workgroups share a CU and the four are faster (1.13 to 1.28 of the time with halves).  Halves / whole over 1500 shapes of 5 to 3000 rows,
// mean (most): 64 x 128 five blocks of 128 1.01 (1.03), six 0.98 (1.00), sixteen 0.94, more 0.85 to 0.90; 128 x 128 eight 1.01 (1.03), nine to sixteen 0.98 (1.025),
// up to 32 0.94, more 0.90.  One tile of rows and more than 192 of channels, where the weights' bytes are the bound: 1.02 (1.05) up to 23 blocks, 0.94 beyond.
// 128 x 256 (1.10 to 0.97) and 64 x 384 (1.11 to 1.03) stay with four.
static bool w8a8_halves(int form, int64_t M, int64_t N, int64_t K) {
  if (form != 3 && form != 4) return false;
  const int bm = form == 3 ? 64 : 128;
  const int64_t tiles = ((M + bm - 1) / bm) * ((N + 127) / 128), blocks = (K + 127) / 128;
  if (M <= 64 && tiles > 192 && blocks < 24) return false;
  return tiles <= 256 && blocks >= (form == 3 ? 6 : 10);
}
// Which matrix-core form runs against packed weights.  Waves that split K (wk_gemm.h) from a few tokens to about the batch whose
// large tiles fill the chip (93 x 2560 x 9728: 38 -> 11 us, 300 x 2560 x 9728: 41 -> 20, 32 x 4096 x 4096: 13.5 -> 7.6), then the
// weights-from-global tiles.  Over 1850 random shapes (5 to 6000 rows, 64 to 22 000 channels, K 64 to 10 000) the choice takes 1.008 times the
// best form's time on average (40 % more at worst, 814 x 1200 x 3200; more than 10 % in 43) and is more than 5 % slower than the tiles by
// rows and columns alone that ran before in 17 (2806 x 208 x 3968: 14.7, 11.5 at most).  More than 32 rows: fitted to 1300 of them within 5 to
// 8 % (rms, where a form is near the best); a table fitted to 170 shapes of 93 rows and more, without the prices of M K and M N, made the
// choice 1.021, 169 and 97 (1811 x 264 x 1280 7.6 us, 6.4 now), but is as good up to 32 rows (1.009 of the best) and stays there.
// Costs are those of four waves: with a gain of halves taken off them, 190 of 1500 shapes went from tiles of 64 x 128 (or 64 x 64 by eight waves) to halves of larger
// ones, 1.01 of their time on average, 71 of them 3 to 22 % slower and 34 3 to 15 % faster (1155 x 1912 x 4288 28.7 -> 31.3 us, 927 x 1032 x 9728 33.5 -> 40.9).
static int w8a8_packed_form(int64_t M, int64_t N, int64_t K) {
  constexpr int forms = 8;
  static const FormCost many[forms] = {
      {32, 32, 1, 1.0f, 0.75f, 3.143f, 0.5845f, 0.08189f, 0.0852f, 0.8638f},  // 8 waves, two workgroups per CU
      {32, 64, 1, 1.0f, 1.00f, 2.442f, 1.744f, 0.1177f, 0.08201f, 1.227f},    // 8 waves
      {64, 64, 1, 1.0f, 1.00f, 2.549f, 2.125f, 0.1942f, 0.1198f, 1.73f},      // 8 waves
      {64, 128, 1, 1.0f, 0.75f, 3.462f, 0.3554f, 0.2758f, 0.05724f, 0.4347f},  // weights-from-global tiles
      {128, 128, 1, 1.0f, 0.50f, 4.155f, 0.355f, 0.501f, 0.2004f, 0.3674f},
      {128, 256, 1, 1.0f, 1.00f, 5.54f, 0.f, 0.7006f, 0.1384f, 0.3784f},
      {64, 384, 1, 1.0f, 1.00f, 4.842f, 0.03656f, 0.5477f, 0.07742f, 0.48f},
      {128, 384, 1, 1.0f, 1.00f, 3.357f, 4.175f, 0.9135f, 0.3508f, 0.3465f}};
  static const FormCost few[forms] = {{32, 32, 1, 1.f, 0.50f, 2.89f, 0.79f, 0.1048f, 0.f, 0.f},   {32, 64, 1, 1.f, 1.00f, 1.94f, 2.55f, 0.1276f, 0.f, 0.f},
                                      {64, 64, 1, 1.f, 1.00f, 0.89f, 4.64f, 0.1776f, 0.f, 0.f},   {64, 128, 1, 1.f, 0.00f, 3.34f, 0.f, 0.4102f, 0.f, 0.f},
                                      {128, 128, 1, 1.f, 0.50f, 2.82f, 1.34f, 0.5597f, 0.f, 0.f}, {128, 256, 1, 1.f, 0.75f, 0.f, 6.71f, 0.6615f, 0.f, 0.f},
                                      {64, 384, 1, 1.f, 0.75f, 0.f, 5.22f, 0.5796f, 0.f, 0.f},    {128, 384, 1, 1.f, 1.00f, 0.f, 9.57f, 0.86f, 0.f, 0.f}};
  const FormCost* cost = M <= 32 ? few : many;
  int form = 0;
  float best = 0.f;
  for (int f = 0; f < forms; f++) {
    const float c = form_cost(cost[f], M, N, K, (K + 127) / 128);
    if (f == 0 || c < best) {
      best = c;
      form = f;
    }
  }
  return form;
}
static int launch_w8a8_packed_auto(const W8A8Args& a, hipStream_t st) {
  if (g_w8a8_ntile || !g_w8a8_decode) return launch_w8a8_nsplit_auto<true>(a, st);
  const int form = w8a8_packed_form(a.M, a.N, a.K);
  const bool halves = w8a8_halves(form, a.M, a.N, a.K);
  switch (form) {
    case 0: return wk_gemm_launch<W8A8Waves, 1, 1, 8, 2>(a, st);
    case 1: return wk_gemm_launch<W8A8Waves, 1, 2, 8, 1>(a, st);
    case 2: return wk_gemm_launch<W8A8Waves, 2, 2, 8, 1>(a, st);
    case 3: return halves ? launch_w8a8_halves<2, 1>(a, st) : launch_w8a8_nsplit<2, 1, true, 2>(a, st);
    case 4: return halves ? launch_w8a8_halves<4, 1>(a, st) : launch_w8a8_nsplit<4, 1, true, 2>(a, st);
    case 5: return launch_w8a8_nsplit<4, 2, true, 2>(a, st);
    case 6: return launch_w8a8_nsplit<2, 3, true, 2>(a, st);
    default: return launch_w8a8_nsplit<4, 3, true, 1>(a, st);
  }
}
MLLM_API int mllm_hip_w8a8_packed_form(int64_t M, int64_t N, int64_t K) {
  if (M < 1 || N < 1 || K < 1) return 0;
  return M < 5 ? 9 : 1 + w8a8_packed_form(M, N, K);
}
MLLM_API int mllm_hip_w8a8_packed_halves(int64_t M, int64_t N, int64_t K) {
  return M >= 5 && N >= 1 && K >= 1 && w8a8_halves(w8a8_packed_form(M, N, K), M, N, K);
}
MLLM_API int mllm_hip_w8a8_set_decode(int gemv) {
  if (gemv != 0 && gemv != 1) return MLLM_HIP_E_BADARG;
  g_w8a8_decode = gemv;
  return 0;
}
MLLM_API int mllm_hip_w8a8_set_decode_mfma_from(int tokens) {
  if (tokens < 1 || tokens > 33) return MLLM_HIP_E_BADARG;
  g_w8a8_decode_mfma_from = tokens;
  return 0;
}

MLLM_API int mllm_hip_w8a8_nsplit_set_tuning(int tile) {
  if (tile < 0 || tile > 5) return MLLM_HIP_E_BADARG;
  g_w8a8_ntile = tile;
  return 0;
}

static int check_per_token_quant(const void* x, int x_dtype, const int8_t* q, const float* scale, int64_t M, int64_t K) {
  if (!x || !q || !scale || M <= 0 || K <= 0 || (x_dtype != MLLM_HIP_F32 && x_dtype != MLLM_HIP_BF16))
    return MLLM_HIP_E_BADARG;
  if (M > INT32_MAX || K > INT32_MAX) return MLLM_HIP_E_SHAPE;
  if (K % 8 == 0 && (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(q) % 8)) return MLLM_HIP_E_ALIGN;
  return 0;
}
MLLM_API int mllm_hip_per_token_quant_int8(const void* x, int x_dtype, int8_t* q, float* scale, int64_t M, int64_t K,
                                           void* stream) {
  RC_RET(check_per_token_quant(x, x_dtype, q, scale, M, K));
  const int ni = (K % 8 == 0 && K >= 8 && K <= 4 * 2048) ? (K <= 2048 ? 1 : (K <= 4096 ? 2 : 4)) : 0;
#define PTQ(XT_, NI_) \
  hipLaunchKernelGGL((per_token_quant_kernel<XT_, NI_>), dim3((unsigned)M), dim3(256), 0, (hipStream_t)stream, x, q, scale, (int)K)
#define PTQ_T(XT_)          \
  if (ni == 1) PTQ(XT_, 1); \
  else if (ni == 2) PTQ(XT_, 2); \
  else if (ni == 4) PTQ(XT_, 4); \
  else PTQ(XT_, 0)
  if (x_dtype == MLLM_HIP_F32) {
    PTQ_T(MLLM_HIP_F32);
  } else {
    PTQ_T(MLLM_HIP_BF16);
  }
#undef PTQ_T
#undef PTQ
  return (int)hipGetLastError();
}

MLLM_API int mllm_hip_w8a8_gemm(const int8_t* xq, const float* x_scale, const int8_t* W, const float* w_scale,
                                const float* bias, void* out_bf16, int32_t* acc_out, int64_t M, int64_t N, int64_t K,
                                void* stream) {
  if (!xq || !W || M <= 0 || N <= 0 || K <= 0 || (!out_bf16 && !acc_out)) return MLLM_HIP_E_BADARG;
  if (out_bf16 && (!x_scale || !w_scale)) return MLLM_HIP_E_BADARG;
  if (K % 16) return MLLM_HIP_E_SHAPE;
  if (M * K >= ((int64_t)1 << 32) || N * K >= ((int64_t)1 << 32) || M > INT32_MAX || N > INT32_MAX) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(xq) % 16 || reinterpret_cast<uintptr_t>(W) % 16) return MLLM_HIP_E_ALIGN;
  W8A8Args a{xq, W, x_scale, w_scale, bias, (uint16_t*)out_bf16, acc_out, (int)M, (int)N, (int)K};
  hipStream_t st = (hipStream_t)stream;
  int tile = g_w8a8_tile;
  if (!tile) {
    const int64_t mid = ((M + 127) / 128) * ((N + 127) / 128);
    // the 256x192 tile is compiled and tested but measured slower than 128x128
    tile = (K % 128 == 0 && mid >= 256) ? 4 : mid >= 128 ? 2 : 3;
  }
  if (tile == 4 && K % 128) tile = 2;
  switch (tile) {
    case 4: return launch_w8a8_nsplit_auto<false>(a, st);
    case 1: return launch_w8a8<256, 192, 128, 96, 4>(a, st);
    case 2: return launch_w8a8<128, 128, 64, 64, 4>(a, st);
    default: return launch_w8a8<64, 64, 32, 32, 2>(a, st);
  }
}

MLLM_API size_t mllm_hip_w8a8_packed_bytes(int64_t N, int64_t K) {
  if (N <= 0 || K <= 0) return 0;
  return (size_t)(w8a8_packed_n(N) * w8a8_packed_k(K));
}

MLLM_API int mllm_hip_w8a8_prepack(const int8_t* W, int64_t N, int64_t K, void* packed, void* stream) {
  if (!W || !packed || N <= 0 || K <= 0) return MLLM_HIP_E_BADARG;
  if (K % 16 || N > INT32_MAX || K > INT32_MAX || w8a8_packed_n(N) * w8a8_packed_k(K) >= ((int64_t)1 << 32)) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(W) % 16 || reinterpret_cast<uintptr_t>(packed) % 16) return MLLM_HIP_E_ALIGN;
  const int64_t chunks = w8a8_packed_n(N) * w8a8_packed_k(K) / 16;
  hipLaunchKernelGGL(w8a8_prepack_kernel, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, (hipStream_t)stream, W,
                     reinterpret_cast<u32x4*>(packed), (int)N, (int)K, chunks);
  return (int)hipGetLastError();
}

static int check_w8a8_gemm_packed(const int8_t* xq, const float* x_scale, const void* W_packed, const float* w_scale, const void* out_bf16,
                                  const int32_t* acc_out, int64_t M, int64_t N, int64_t K) {
  if (!xq || !W_packed || M <= 0 || N <= 0 || K <= 0 || (!out_bf16 && !acc_out)) return MLLM_HIP_E_BADARG;
  if (out_bf16 && (!x_scale || !w_scale)) return MLLM_HIP_E_BADARG;
  if (K % 16) return MLLM_HIP_E_SHAPE;
  if (M * K >= ((int64_t)1 << 32) || w8a8_packed_n(N) * w8a8_packed_k(K) >= ((int64_t)1 << 32) || M > INT32_MAX || N > INT32_MAX)
    return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(xq) % 16 || reinterpret_cast<uintptr_t>(W_packed) % 16) return MLLM_HIP_E_ALIGN;
  return 0;
}
MLLM_API int mllm_hip_w8a8_gemm_packed(const int8_t* xq, const float* x_scale, const void* W_packed, const float* w_scale,
                                       const float* bias, void* out_bf16, int32_t* acc_out, int64_t M, int64_t N,
                                       int64_t K, void* stream) {
  RC_RET(check_w8a8_gemm_packed(xq, x_scale, W_packed, w_scale, out_bf16, acc_out, M, N, K));
  W8A8Args a{xq, reinterpret_cast<const int8_t*>(W_packed), x_scale, w_scale, bias, (uint16_t*)out_bf16, acc_out, (int)M, (int)N, (int)K};
  int rc = 0;
  if (launch_w8a8_gemv_packed(a, (hipStream_t)stream, &rc)) return rc;  // up to four tokens
  return launch_w8a8_packed_auto(a, (hipStream_t)stream);
}

MLLM_API size_t mllm_hip_w8a8_workspace_bytes(int64_t M, int64_t K) {
  if (M <= 0 || K <= 0) return 0;
  return align_up((size_t)M * K, 256) + align_up((size_t)M * 4, 256);
}

MLLM_API int mllm_hip_w8a8_linear(const void* x, int x_dtype, const int8_t* W, const float* w_scale, const float* bias,
                                  void* out_bf16, int64_t M, int64_t N, int64_t K, void* workspace, void* stream) {
  // everything the second step would reject is rejected before the first one is launched
  if (!workspace || !W || !w_scale || !out_bf16 || N <= 0) return MLLM_HIP_E_BADARG;
  if (K > 0 && K % 16) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(workspace) % 16 || reinterpret_cast<uintptr_t>(W) % 16) return MLLM_HIP_E_ALIGN;
  int8_t* q = reinterpret_cast<int8_t*>(workspace);
  float* xs = reinterpret_cast<float*>(reinterpret_cast<char*>(workspace) + align_up((size_t)M * K, 256));
  int rc = mllm_hip_per_token_quant_int8(x, x_dtype, q, xs, M, K, stream);
  if (rc) return rc;
  return mllm_hip_w8a8_gemm(q, xs, W, w_scale, bias, out_bf16, nullptr, M, N, K, stream);
}

MLLM_API int mllm_hip_w8a8_linear_packed(const void* x, int x_dtype, const void* W_packed, const float* w_scale,
                                         const float* bias, void* out_bf16, int64_t M, int64_t N, int64_t K,
                                         void* workspace, void* stream) {
  // everything the second step would reject is rejected before the first one is launched
  if (!workspace || !W_packed || !w_scale || !out_bf16 || N <= 0) return MLLM_HIP_E_BADARG;
  if (K > 0 && K % 16) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(workspace) % 16 || reinterpret_cast<uintptr_t>(W_packed) % 16) return MLLM_HIP_E_ALIGN;
  int8_t* q = reinterpret_cast<int8_t*>(workspace);
  float* xs = reinterpret_cast<float*>(reinterpret_cast<char*>(workspace) + align_up((size_t)M * K, 256));
  RC_RET(check_per_token_quant(x, x_dtype, q, xs, M, K));
  RC_RET(check_w8a8_gemm_packed(q, xs, W_packed, w_scale, out_bf16, nullptr, M, N, K));
  W8A8Args a{q, reinterpret_cast<const int8_t*>(W_packed), xs, w_scale, bias, (uint16_t*)out_bf16, nullptr, (int)M, (int)N, (int)K};
  int rc = 0;
  // (results over the tokens: they are all read first)
  const uintptr_t xa = reinterpret_cast<uintptr_t>(x), ya = reinterpret_cast<uintptr_t>(out_bf16);
  const bool apart = xa + (uintptr_t)M * K * (x_dtype == MLLM_HIP_F32 ? 4 : 2) <= ya || ya + (uintptr_t)M * N * 2 <= xa;
  if (apart && launch_w8a8_gemv_packed(a, (hipStream_t)stream, &rc, x, x_dtype)) return rc;
  RC_RET(mllm_hip_per_token_quant_int8(x, x_dtype, q, xs, M, K, stream));
  return mllm_hip_w8a8_gemm_packed(q, xs, W_packed, w_scale, bias, out_bf16, nullptr, M, N, K, stream);
}

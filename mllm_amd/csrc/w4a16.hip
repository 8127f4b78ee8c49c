// W4A16 Linear for prefill on gfx950: bf16 activations x uint4 weights with per-group fp16 scales and uint4 zero-points
// (group size a multiple of 64 along K, 128 in the checkpoints), fp32 accumulation, bf16 output.
//
// Semantics (the reference runs this on CUDA through Marlin; restated in closed form):
//   dequantization      mllm-kernel/mllm_kernel/cuda/csrc/gemm/marlin/dequant.h:18-26 (q - zp), marlin_template.h:153-168 (x scale)
//   checkpoint scheme   pymllm/quantization/methods/awq_marlin.py:274-449
//   test formula        mllm-kernel/tests/test_gptq_marlin.py:143-146
//   w_bf16[n][k] = bf16_rne( float(q[n][k] - zp[n][k/g]) * fp32(scale[n][k/g]) )   (the product is exact in fp32: <= 16 bits)
//   C[m][n]      = bf16_rne( sum_k A[m][k] * w_bf16[n][k]  (+ bias[n]) ),  fp32 accumulate on the matrix cores
// Storage: qw uint8 [N][K/2], element 2j in the low nibble of byte j; scales fp16 [N][K/g]; zero-points uint8
// [N][ceil(K/g/2)], group 2i in the low nibble of byte i.
//
// Weights are fetched packed (16 bytes = 32 elements per lane), dequantized once per workgroup in registers and staged
// as bf16 in LDS next to the activation tile; the matrix cores read both operands from LDS.
#include "qcommon.h"
#include <algorithm>

#include "wk_gemm.h"

namespace mllmhip {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

// eight elements of one packed dword -> four dwords of bf16 pairs, element order kept.
// (q - zp) * s == fma(q, s, -zp*s) exactly: both products and their sum need at most 16 significant bits.
// A nibble alone in a byte is q * 2^-9 as an fp8 number (e4m3: below 16 the pattern counts, denormal or not), and
// v_cvt_pk_f32_fp8 converts two bytes in the 4.3 clocks that v_cvt_f32_ubyteN takes for one: the fma takes s * 2^9 (exact).  Clocks
// per dword and wave, alone: 62, with a conversion per element 78.  us, before / now: 93 x 2048 x 6144 10.6 / 10.1, 2048 x
// 9728 x 2560 105.3 / 102.9, 1 x 2280 x 4480 7.1 / 6.7, 1709 x 1208 x 6784 67.9 / 62.6; 0.962 of the time over 26 sizes, none slower.
struct DequantNibbles {
  uint32_t lo, hi;  // bytes: elements 0,2,4,6 / 1,3,5,7
  f32x2 l, h;
  __device__ __forceinline__ explicit DequantNibbles(uint32_t w) : lo(w & 0x0f0f0f0fu), hi((w >> 4) & 0x0f0f0f0fu) {}
  // elements 2 b, 2 b + 1 (b = 0..3 in this order); s9 = s * 2^9
  __device__ __forceinline__ uint32_t pair(int b, float s9, float nzs) {
    if (b == 0) l = __builtin_amdgcn_cvt_pk_f32_fp8((int)lo, false), h = __builtin_amdgcn_cvt_pk_f32_fp8((int)hi, false);
    if (b == 2) l = __builtin_amdgcn_cvt_pk_f32_fp8((int)lo, true), h = __builtin_amdgcn_cvt_pk_f32_fp8((int)hi, true);
    return pack_bf16(fmaf(l[b & 1], s9, nzs), fmaf(h[b & 1], s9, nzs));
  }
};
__device__ __forceinline__ void dequant8(uint32_t w, float s, float nzs, uint32_t (&out)[4]) {
  DequantNibbles q(w);
  const float s9 = s * 512.f;
#pragma unroll
  for (int b = 0; b < 4; b++) out[b] = q.pair(b, s9, nzs);
}

struct W4A16Args {
  const uint16_t* A;    // bf16 [M][K]
  const uint8_t* qw;    // [N][K/2]
  const uint16_t* s;    // fp16 [N][G]
  const uint8_t* zp;    // [N][(G+1)/2]
  const uint16_t* bias; // bf16 [N] or null
  uint16_t* C;          // bf16 [M][N]
  int M, N, K, group;
};

// Workgroup tile BM x BN, K step 64 elements; waves (BM/WM) x (BN/WN), each WM x WN as 32x32 tiles of
// v_mfma_f32_32x32x16_bf16 (every lane supplies 8 consecutive k of one row of A and of one row of W).
// LDS rows hold 64 bf16 = 128 bytes, padded to 144 so that 16-byte reads of 16 neighbouring rows hit distinct banks.
template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64) void w4a16_gemm_kernel(W4A16Args a) {
  constexpr int BK = 64, LDK = 144;
  constexpr int NT = (BM / WM) * (BN / WN) * 64;
  constexpr int CA = BM * 8 / NT;                 // 16-byte activation chunks (8 bf16) per thread and K step
  constexpr int CB = (BN * 2 + NT - 1) / NT;      // 16-byte packed weight chunks (32 elements) per thread and K step
  static_assert(BM * 8 % NT == 0, "activation tile must split evenly over the threads");
  constexpr int TM = WM / 32, TN = WN / 32;
  constexpr int STAGE = (BM + BN) * LDK;
  extern __shared__ __align__(16) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / (BN / WN), wn = wave % (BN / WN);
  const int G = a.K / a.group, zpb = (G + 1) / 2;

  const int tilesN = (a.N + BN - 1) / BN, tilesM = (a.M + BM - 1) / BM;
  const int total = tilesM * tilesN;
  int tile = blockIdx.x;
  if (total % 8 == 0) tile = (blockIdx.x % 8) * (total / 8) + blockIdx.x / 8;  // one run of tiles per XCD
  const int m0 = (tile / tilesN) * BM, n0 = (tile % tilesN) * BN;

  const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.A), 0, (uint32_t)((int64_t)a.M * a.K * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rW = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.qw), 0, (uint32_t)((int64_t)a.N * a.K / 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rS = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.s), 0, (uint32_t)((int64_t)a.N * G * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rZ = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.zp), 0, (uint32_t)((int64_t)a.N * zpb), 0x00020000);

  // activation chunk c: row = idx / 8, 16-byte column = idx % 8 ; weight chunk c: row = idx / 2, half = idx % 2
  uint32_t offA[CA];
#pragma unroll
  for (int c = 0; c < CA; c++) {
    const int idx = tid + c * NT, row = m0 + idx / 8;
    offA[c] = row < a.M ? (uint32_t)(((int64_t)row * a.K + (idx % 8) * 8) * 2) : 0xffffffffu;
  }
  int wrow[CB];
  bool wok[CB];
#pragma unroll
  for (int c = 0; c < CB; c++) {
    const int idx = tid + c * NT;
    wrow[c] = n0 + idx / 2;
    wok[c] = idx < BN * 2 && wrow[c] < a.N;
  }
  u32x4 gA[CA], gW[CB];
  uint16_t gS[CB];
  uint8_t gZ[CB];
  auto gload = [&](int k0) {
#pragma unroll
    for (int c = 0; c < CA; c++) {
      const bool ok = offA[c] != 0xffffffffu && k0 + ((tid + c * NT) % 8) * 8 < a.K;
      gA[c] = __builtin_amdgcn_raw_buffer_load_b128(rA, ok ? offA[c] + (uint32_t)k0 * 2u : 0xffffffffu, 0, 0);
    }
    const int g = k0 / a.group;
#pragma unroll
    for (int c = 0; c < CB; c++) {
      const int half = (tid + c * NT) & 1;
      const bool ok = wok[c] && k0 + half * 32 < a.K;
      gW[c] = __builtin_amdgcn_raw_buffer_load_b128(rW, ok ? (uint32_t)(((int64_t)wrow[c] * a.K + k0 + half * 32) / 2) : 0xffffffffu, 0, 0);
      gS[c] = __builtin_amdgcn_raw_buffer_load_b16(rS, ok ? (uint32_t)(((int64_t)wrow[c] * G + g) * 2) : 0xffffffffu, 0, 0);
      gZ[c] = __builtin_amdgcn_raw_buffer_load_b8(rZ, ok ? (uint32_t)((int64_t)wrow[c] * zpb + (g >> 1)) : 0xffffffffu, 0, 0);
    }
  };
  auto sstore = [&](int buf, int k0) {
    unsigned char* base = smem + buf * STAGE;
#pragma unroll
    for (int c = 0; c < CA; c++) {
      const int idx = tid + c * NT;
      *reinterpret_cast<u32x4*>(base + (idx / 8) * LDK + (idx % 8) * 16) = gA[c];
    }
    const int g = k0 / a.group;
#pragma unroll
    for (int c = 0; c < CB; c++) {
      const int idx = tid + c * NT;
      if (idx < BN * 2) {
        const float s = f16bits_to_f32(gS[c]);
        const float z = (float)((g & 1) ? (gZ[c] >> 4) : (gZ[c] & 15));
        const float nzs = -(z * s);  // exact: 4-bit integer times an 11-bit significand
        const uint32_t w[4] = {gW[c].x, gW[c].y, gW[c].z, gW[c].w};
        unsigned char* dst = base + (BM + idx / 2) * LDK + (idx & 1) * 64;
#pragma unroll
        for (int j = 0; j < 4; j++) {
          uint32_t o[4];
          dequant8(w[j], s, nzs, o);
          *reinterpret_cast<u32x4*>(dst + j * 16) = u32x4{o[0], o[1], o[2], o[3]};
        }
      }
    }
  };

  v16f acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

  const int KT = (a.K + BK - 1) / BK;
  gload(0);
  sstore(0, 0);
  __syncthreads();
  const int lrow = lane & 31, lk = (lane >> 5) * 16;
  for (int kt = 0; kt < KT; kt++) {
    const int buf = kt & 1;
    if (kt + 1 < KT) gload((kt + 1) * BK);
    const unsigned char* base = smem + buf * STAGE;
#pragma unroll
    for (int ks = 0; ks < 4; ks++) {
      bf16x8 fa[TM], fb[TN];
#pragma unroll
      for (int i = 0; i < TM; i++)
        fa[i] = *reinterpret_cast<const bf16x8*>(base + (wm * WM + i * 32 + lrow) * LDK + ks * 32 + lk);
#pragma unroll
      for (int j = 0; j < TN; j++)
        fb[j] = *reinterpret_cast<const bf16x8*>(base + (BM + wn * WN + j * 32 + lrow) * LDK + ks * 32 + lk);
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
    if (kt + 1 < KT) sstore(buf ^ 1, (kt + 1) * BK);
    __syncthreads();
  }

  // epilogue.  32x32 accumulator layout: register r of lane l holds row 8*(r/4) + 4*(l/32) + r%4, column l%32.
#pragma unroll
  for (int j = 0; j < TN; j++) {
    const int n = n0 + wn * WN + j * 32 + lrow;
    const bool nok = n < a.N;
    const float bn = (nok && a.bias) ? bf16_to_f32(a.bias[n]) : 0.f;
#pragma unroll
    for (int i = 0; i < TM; i++) {
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int m = m0 + wm * WM + i * 32 + 8 * (r / 4) + 4 * (lane >> 5) + (r % 4);
        if (nok && m < a.M) {
          float f = acc[i][j][r];
          if (a.bias) f += bn;
          a.C[(int64_t)m * a.N + n] = f32_to_bf16(f);
        }
      }
    }
  }
}

// dequantized weight table (parity probe and the definition of "dequantized weight values")
__global__ void w4a16_dequant_kernel(const uint8_t* __restrict__ qw, const uint16_t* __restrict__ s,
                                     const uint8_t* __restrict__ zp, uint16_t* __restrict__ w, int64_t N, int64_t K, int group) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // one packed dword = 8 elements
  if (i >= N * K / 8) return;
  const int64_t n = i / (K / 8), k = (i % (K / 8)) * 8;
  const int G = (int)(K / group), zpb = (G + 1) / 2, g = (int)(k / group);
  const float sc = f16bits_to_f32(s[n * G + g]);
  const uint8_t zb = zp[n * zpb + (g >> 1)];
  const float z = (float)((g & 1) ? (zb >> 4) : (zb & 15));
  const uint32_t word = *reinterpret_cast<const uint32_t*>(qw + (n * K + k) / 2);
  uint32_t o[4];
  dequant8(word, sc, -(z * sc), o);
  *reinterpret_cast<u32x4*>(w + n * K + k) = u32x4{o[0], o[1], o[2], o[3]};
}

// ---------------------------------------------------------------------------------------------------------
// Prepacked weights + weights-from-global kernel (the fast path for prefill-sized M).
//
// Measured on this part: a 16-byte LDS read of a whole wave occupies the CU's LDS pipe for 16 cycles (64 B/clk/CU) while
// one v_mfma_f32_32x32x16_bf16 occupies a SIMD for 32, so a wave that pulls both operands of a 64x64 tile through LDS is
// LDS-bound at under half the matrix rate, and dequantized weights staged in LDS cost that bandwidth twice (write +
// reads).  Here only the activation tile goes through LDS.  The four waves of a workgroup sit side by side along N, each
// owns (32 TM) x (32 TN) outputs, loads ITS packed 4-bit weights straight from global memory (16 bytes per lane = the
// lane's operands of four MFMA K steps), dequantizes them in registers one MFMA step ahead of their use, and no weight
// is dequantized twice inside a workgroup.
//
// Packed layout (one pass over the checkpoint tensors, mllm_hip_w4a16_prepack):
//   q   [N/32][K/64][64 lanes][16 bytes]: lane l = (row l%32, half l/32); dword d of its 16 bytes holds the eight
//       elements k = 64 kb + 16 d + 8 (l/32) + 0..7 of its row, element e in nibble e (the checkpoint's own dword).
//       N is padded to 32 rows and K to 128 elements with zeros.
//   sz  [N/32][K/group][32 rows][2 floats]: (scale, -zero_point * scale) of the row's group, both exact in fp32.
__host__ __device__ inline int64_t w4a16_packed_n(int64_t N) { return (N + 31) / 32 * 32; }
__host__ __device__ inline int64_t w4a16_packed_k(int64_t K) { return (K + 127) / 128 * 128; }
__host__ __device__ inline int64_t w4a16_packed_qbytes(int64_t N, int64_t K) { return w4a16_packed_n(N) * w4a16_packed_k(K) / 2; }

__global__ __launch_bounds__(256) void w4a16_prepack_q_kernel(const uint8_t* __restrict__ qw, uint32_t* __restrict__ P, int N,
                                                              int K, int64_t words) {
  const int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x;  // one dword = 8 elements of the packed matrix
  if (w >= words) return;
  const int kbs = (int)(w4a16_packed_k(K) / 64);
  const int d = (int)(w % 4), l = (int)((w / 4) % 64);
  const int64_t blk = w / 256;
  const int kb = (int)(blk % kbs), nb = (int)(blk / kbs);
  const int n = nb * 32 + (l & 31), k = kb * 64 + d * 16 + (l >> 5) * 8;
  uint32_t v = 0;
  if (n < N && k < K) v = *reinterpret_cast<const uint32_t*>(qw + ((int64_t)n * K + k) / 2);
  P[w] = v;
}
__global__ __launch_bounds__(256) void w4a16_prepack_sz_kernel(const uint16_t* __restrict__ s, const uint8_t* __restrict__ zp,
                                                               float2* __restrict__ SZ, int N, int G, int64_t count) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // (nb, g, row)
  if (i >= count) return;
  const int row = (int)(i % 32), g = (int)((i / 32) % G), nb = (int)(i / 32 / G);
  const int n = nb * 32 + row;
  float2 v = {0.f, 0.f};
  if (n < N) {
    const float sc = f16bits_to_f32(s[(int64_t)n * G + g]);
    const uint8_t zb = zp[(int64_t)n * ((G + 1) / 2) + (g >> 1)];
    const float z = (float)((g & 1) ? (zb >> 4) : (zb & 15));
    v = float2{sc, -(z * sc)};
  }
  SZ[i] = v;
}

struct W4A16PArgs {
  const uint16_t* A;     // bf16 [M][K]
  const uint8_t* P;      // packed q then sz
  const uint16_t* bias;  // bf16 [N] or null
  uint16_t* C;           // bf16 [M][N]
  int M, N, K, group;
};


// One output tile (32 TM rows from m0) x (128 TN columns from n0) by the four waves of a workgroup.  G == 2: by eight, the second four take the
// second half of K with a stage of their own; their sums join the first's in LDS.
template <int TM, int TN, int BK, int G = 1>
__device__ __forceinline__ void w4a16_nsplit_tile(const W4A16PArgs& a, const int m0, const int n0, unsigned char* smem_all) {
  static_assert(BK == 64 || BK == 128, "K step of one or two 64-element weight blocks");
  constexpr int LDK = 2 * BK + 16, KS = BK / 16, NH = BK / 64;  // LDS row in bytes; MFMA steps; weight blocks per K step
  constexpr int CPRA = BK / 8;                                  // 16-byte activation chunks per row and K step
  constexpr int BM = TM * 32, WN = TN * 32, BN = 4 * WN;
  constexpr int CA = BM * (2 * BK / 16) / 256;  // 16-byte activation chunks per thread and K step
  static_assert(CA >= 1, "tile too small for 256 threads");
  constexpr int STAGE = BM * LDK;

  const int group = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  unsigned char* const smem = smem_all + group * 2 * STAGE;
  const int tid = G == 1 ? threadIdx.x : threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
  const int lrow = lane & 31, hi = lane >> 5;

  const int Kp = (int)w4a16_packed_k(a.K), kbs = Kp / 64, groups = a.K / a.group, g64 = a.group / 64;
  const int64_t qbytes = w4a16_packed_qbytes(a.N, a.K);
  const int nbs = (int)(w4a16_packed_n(a.N) / 32);
  const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.A), 0, (uint32_t)((int64_t)a.M * a.K * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rQ = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.P), 0, (uint32_t)qbytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rS = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.P + qbytes), 0, (uint32_t)((int64_t)nbs * groups * 256), 0x00020000);

  // activation chunk: row idx / CPRA, 16-byte column idx % CPRA.  Rows past M are clamped (never stored); columns past K
  // read as zeros so that the zero-padded tail of the weights never meets another row's values.
  uint32_t offA[CA];
  int colA[CA];
#pragma unroll
  for (int c = 0; c < CA; c++) {
    const int idx = tid + c * 256;
    colA[c] = (idx % CPRA) * 8;
    offA[c] = (uint32_t)(((int64_t)min(m0 + idx / CPRA, a.M - 1) * a.K + colA[c]) * 2);
  }
  uint32_t offQ[TN], offS[TN];
#pragma unroll
  for (int j = 0; j < TN; j++) {
    const int nb = min((n0 + wave * WN) / 32 + j, nbs - 1);
    offQ[j] = (uint32_t)((int64_t)nb * kbs * 1024 + lane * 16);
    offS[j] = (uint32_t)(((int64_t)nb * groups * 32 + lrow) * 8);
  }
  auto loadA = [&](int k0, u32x4 (&ga)[CA]) {
#pragma unroll
    for (int c = 0; c < CA; c++)
      ga[c] = __builtin_amdgcn_raw_buffer_load_b128(rA, k0 + colA[c] < a.K ? offA[c] : 0xffffffffu, k0 * 2, 0);
  };
  auto storeA = [&](int buf, const u32x4 (&ga)[CA]) {
#pragma unroll
    for (int c = 0; c < CA; c++) {
      const int idx = tid + c * 256;
      *reinterpret_cast<u32x4*>(smem + buf * STAGE + (idx / CPRA) * LDK + (idx % CPRA) * 16) = ga[c];
    }
  };
  auto readA = [&](int buf, int ks, bf16x8 (&fa)[TM]) {
#pragma unroll
    for (int i = 0; i < TM; i++)
      fa[i] = *reinterpret_cast<const bf16x8*>(smem + buf * STAGE + (i * 32 + lrow) * LDK + ks * 32 + hi * 16);
  };
  // the packed weights and the (scale, -zp*scale) pair of 64-element block kb of column block j
  auto loadQ = [&](int kb, int j) -> u32x4 { return __builtin_amdgcn_raw_buffer_load_b128(rQ, offQ[j], kb * 1024, 0); };
  auto loadS = [&](int kb, int j) -> u32x2 {
    return __builtin_amdgcn_raw_buffer_load_b64(rS, offS[j], min(kb / g64, groups - 1) * 256, 0);
  };
  auto dequant = [&](const u32x4& q, const u32x2& sz, int d) -> bf16x8 {
    uint32_t o[4];
    dequant8(q[d], __uint_as_float(sz.x), __uint_as_float(sz.y), o);
    return __builtin_bit_cast(bf16x8, u32x4{o[0], o[1], o[2], o[3]});
  };

  v16f acc[TN][TM];
#pragma unroll
  for (int j = 0; j < TN; j++)
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[j][i][r] = 0.f;

  // K steps of these waves: all of them, or one of the halves (idle: how many fewer the second has, whose barriers it keeps)
  const int KT = Kp / BK, per = (KT + G - 1) / G, kt0 = group * per, kt1 = min(KT, kt0 + per), idle = G == 1 ? 0 : per - (kt1 - kt0);
  u32x4 ga[CA];
  u32x4 rq[NH][TN];  // packed weights of the 64-element blocks of a K step
  u32x2 rs[NH][TN];
  bf16x8 fb[2][TN];  // dequantized operands of MFMA step ks (set ks & 1)
  bf16x8 fa[2][TM];
  loadA(kt0 * BK, ga);
#pragma unroll
  for (int h = 0; h < NH; h++)
#pragma unroll
    for (int j = 0; j < TN; j++) {
      rq[h][j] = loadQ(kt0 * NH + h, j);
      rs[h][j] = loadS(kt0 * NH + h, j);
    }
  storeA(0, ga);
  __syncthreads();
  readA(0, 0, fa[0]);
#pragma unroll
  for (int j = 0; j < TN; j++) fb[0][j] = dequant(rq[0][j], rs[0][j], 0);

  for (int kt = kt0; kt < kt1; kt++) {
    const int buf = (kt - kt0) & 1, k1 = (kt + 1) * BK;
    loadA(k1, ga);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      if (ks < KS - 1) {
        readA(buf, ks + 1, fa[(ks + 1) & 1]);  // the next step's activations while this one's MFMAs run
      } else {
        storeA(buf ^ 1, ga);  // free since the previous barrier; its loads were issued a whole K step ago
        __syncthreads();
        readA(buf ^ 1, 0, fa[(ks + 1) & 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
      const int nh = ((ks + 1) / 4) % NH, nd = (ks + 1) % 4;  // block and dword of the NEXT MFMA step's weights
#pragma unroll
      for (int j = 0; j < TN; j++) {
        // One wave per SIMD issues in order: the dequantization of the next step's operand (19 vector instructions) is
        // cut into TM pieces, one in the shadow of each MFMA (32 cycles), and pinned there; left to the scheduler, the
        // MFMAs queue up back to back and the matrix pipe idles behind them while the VALU work runs.
        DequantNibbles next(rq[nh][j][nd]);
        const float s9 = __uint_as_float(rs[nh][j].x) * 512.f, nzs = __uint_as_float(rs[nh][j].y);
        uint32_t o[4];
#pragma unroll
        for (int i = 0; i < TM; i++) {
          acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[ks & 1][j], fa[ks & 1][i], acc[j][i], 0, 0, 0);
#pragma unroll
          for (int b = i * 4 / TM; b < (i + 1) * 4 / TM; b++)
            o[b] = next.pair(b, s9, nzs);
          __builtin_amdgcn_sched_barrier(0);
        }
        fb[(ks + 1) & 1][j] = __builtin_bit_cast(bf16x8, u32x4{o[0], o[1], o[2], o[3]});
        if (nd == 3) {  // last dword of that half consumed: fetch the same half of the next K step into its registers
          rq[nh][j] = loadQ((kt + 1) * NH + nh, j);
          rs[nh][j] = loadS((kt + 1) * NH + nh, j);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  for (int i = 0; i < idle; i++) __syncthreads();
  __syncthreads();  // all LDS reads done before the epilogue reuses the tiles
  if constexpr (G == 2) {  // the second half's sums join the first's
    f32x4* part = reinterpret_cast<f32x4*>(smem_all);
    auto quad = [&](int j, int i, int g) -> f32x4& { return part[(((wave * TN + j) * TM + i) * 4 + g) * 64 + lane]; };
    if (group == 1) {
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int g = 0; g < 4; g++) quad(j, i, g) = f32x4{acc[j][i][4 * g], acc[j][i][4 * g + 1], acc[j][i][4 * g + 2], acc[j][i][4 * g + 3]};
    }
    __syncthreads();
    if (group == 0) {
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int g = 0; g < 4; g++) {
            const f32x4 v = quad(j, i, g);
#pragma unroll
            for (int e = 0; e < 4; e++) acc[j][i][4 * g + e] += v[e];
          }
    }
    __syncthreads();
  }

  // acc[j][i][4g+e] = C[m0 + 32i + lrow][n0 + wave*WN + 32j + 8g + 4hi + e]
  float* sBi = reinterpret_cast<float*>(smem_all);
  for (int i = tid; i < BN; i += 256) sBi[i] = (a.bias && n0 + i < a.N) ? bf16_to_f32(a.bias[n0 + i]) : 0.f;
  __syncthreads();
  constexpr int ROWB = 2 * BN + 16;
  unsigned char* patch = smem_all + 4096;
  static_assert(BN * 4 <= 4096, "bias overlaps the store patch");
  const bool has_bias = a.bias != nullptr;
  // 16-byte pieces; those of ragged edges fall outside the buffer (whose end a row or column past the tile must not wrap over)
  const bool pieces = a.N % 8 == 0 && reinterpret_cast<uintptr_t>(a.C) % 16 == 0 && ((int64_t)a.M + BM) * a.N * 2 < ((int64_t)1 << 32);
  if (pieces) {
    const __amdgpu_buffer_rsrc_t rC = __builtin_amdgcn_make_buffer_rsrc(a.C, 0, (uint32_t)((int64_t)a.M * a.N * 2), 0x00020000);
    // each 32-row slab of results is turned through LDS so that a wave stores whole rows of the
    // workgroup's BN columns (runs of whole cache lines, 16 bytes per lane)
    f32x4 bi4[TN][4];
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int g = 0; g < 4; g++) bi4[j][g] = *reinterpret_cast<const f32x4*>(&sBi[wave * WN + j * 32 + 8 * g + 4 * hi]);
    constexpr int CPR = BN / 8;  // 16-byte pieces per row
    constexpr int RPW = 8 / G;   // rows per wave
    static_assert((RPW * CPR) % 64 == 0, "a wave stores whole rows");
#pragma unroll
    for (int i = 0; i < TM; i++) {
      if (group == 0) {
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int g = 0; g < 4; g++) {
            float f[4];
#pragma unroll
            for (int e = 0; e < 4; e++) f[e] = acc[j][i][4 * g + e];
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
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const int cn = wave * WN + j * 32 + 8 * g + 4 * hi;
        const f32x4 bi4 = *reinterpret_cast<const f32x4*>(&sBi[cn]);
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (m < a.M && n0 + cn + e < a.N) {
            float f = acc[j][i][4 * g + e];
            if (has_bias) f += bi4[e];
            a.C[(int64_t)m * a.N + n0 + cn + e] = (uint16_t)pack_bf16(f, 0.f);
          }
      }
  }
}

// Tile schedule.  Full tiles (32 TM rows) cover the first `big_cols` column tiles, half-height tiles the remaining column
// tiles.  The host picks big_cols so that the full tiles fill whole rounds of the chip's workgroup slots and the remainder,
// which would otherwise occupy a whole further round at a fraction of the chip, runs as twice as many tiles of half the
// duration; the half-height tiles are the FIRST workgroups of the grid (2048 x 9728 x 2560: 108 -> 101 us; as the last
// workgroups 107).
// WPS: waves per SIMD the register budget is held to (workgroups of 4 waves: WPS workgroups per CU).
template <int TM, int TN, int BK, int WPS, int G = 1>
__global__ __launch_bounds__(256 * G) __attribute__((amdgpu_waves_per_eu(WPS, WPS))) void w4a16_gemm_nsplit_kernel(W4A16PArgs a, int big_cols) {
  constexpr int BM = TM * 32, BN = 4 * TN * 32;
  extern __shared__ __align__(16) unsigned char smem[];
  const int tilesM = (a.M + BM - 1) / BM;
  const int nbig = tilesM * big_cols;
  // The half-height tiles come FIRST in the grid: at the start every CU holds two workgroups, half-height ones beside full
  // ones, and the slots they free take full tiles; as the last round of the launch the half-height tiles ran one to a CU, a
  // wave alone on its SIMD (whose vector and matrix instructions do not overlap).
  constexpr int HM = BM / 2;
  const int tilesH = (a.M + HM - 1) / HM;
  const int nsmall = TM >= 2 ? (int)gridDim.x - nbig : 0;
  int b = (int)blockIdx.x - nsmall;
  if (b >= 0) {
    // Workgroup b runs on XCD b % 8, and every XCD has its own L2.  An XCD takes a block of the tile grid, two blocks along
    // M by four along N where the counts divide: it then reads half of the activations and a quarter of the weights
    // (a run of whole tile columns per XCD reads ALL of the activations and an eighth of the weights: for 2048 x 9728 x 2560
    // 11.8 MB per XCD against 7.9)
    int tm = b % tilesM, tn = b / tilesM;
    if (tilesM % 2 == 0 && big_cols % 4 == 0) {
      const int xcd = b & 7, seq = b >> 3, hm = tilesM / 2, qn = big_cols / 4;
      tm = (xcd & 1) * hm + seq % hm;
      tn = (xcd >> 1) * qn + seq / hm;
    } else {
      b = xcd_run(b, nbig);  // one run of tiles per XCD that shares a slice of the weights
      tm = b % tilesM;
      tn = b / tilesM;
    }
    w4a16_nsplit_tile<TM, TN, BK, G>(a, tm * BM, tn * BN, smem);
  } else {
    if constexpr (TM >= 2 && G == 1) {
      b = (int)blockIdx.x;
      w4a16_nsplit_tile<TM / 2, TN, BK>(a, (b % tilesH) * HM, (big_cols + b / tilesH) * BN, smem);
    }
  }
}

// dequantized weight table from the PACKED form, through the same dequant8 and (scale, -zp*scale) pairs as the GEMM
__global__ void w4a16_dequant_packed_kernel(const uint8_t* __restrict__ P, uint16_t* __restrict__ w, int N, int K, int group) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // one dword = 8 elements of the table
  if (i >= (int64_t)N * K / 8) return;
  const int n = (int)(i / (K / 8)), k = (int)(i % (K / 8)) * 8;
  const int kbs = (int)(w4a16_packed_k(K) / 64), G = K / group;
  const int nb = n / 32, row = n % 32, kb = k / 64, d = (k % 64) / 16, hi = (k % 16) / 8;
  const uint32_t word = reinterpret_cast<const uint32_t*>(P)[(((int64_t)nb * kbs + kb) * 64 + hi * 32 + row) * 4 + d];
  const float2 sz = reinterpret_cast<const float2*>(P + w4a16_packed_qbytes(N, K))[((int64_t)nb * G + k / group) * 32 + row];
  uint32_t o[4];
  dequant8(word, sz.x, sz.y, o);
  *reinterpret_cast<u32x4*>(w + (int64_t)n * K + k) = u32x4{o[0], o[1], o[2], o[3]};
}

static int g_w4a16_tail = 1;  // half-height tiles for a short last round (0 switches the schedule off: tuning/tests)

// K in halves, eight waves per tile
template <int TM, int TN, int BK>
static int launch_w4a16_halves(const W4A16PArgs& a, hipStream_t st) {
  constexpr int BM = TM * 32, BN = 4 * TN * 32;
  constexpr size_t stage = 4 * (size_t)BM * (2 * BK + 16), patch = 4096 + 32 * (2 * (size_t)BN + 16), sums = (size_t)BM * BN * 4;
  constexpr size_t lds = std::max(stage, std::max(patch, sums));
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  auto kern = w4a16_gemm_nsplit_kernel<TM, TN, BK, 2, 2>;
  if (lds > 64 * 1024)
    HIP_RET(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  const int tilesM = (a.M + BM - 1) / BM, tilesN = (a.N + BN - 1) / BN;
  hipLaunchKernelGGL(kern, dim3((unsigned)(tilesM * tilesN)), dim3(512), lds, st, a, tilesN);
  return (int)hipGetLastError();
}

template <int TM, int TN, int BK, int WPS>
static int launch_w4a16_nsplit(const W4A16PArgs& a, hipStream_t st) {
  constexpr int BM = TM * 32, BN = 4 * TN * 32;
  constexpr size_t stage = 2 * (size_t)BM * (2 * BK + 16), patch = 4096 + 32 * (2 * (size_t)BN + 16);
  const size_t lds = stage > patch ? stage : patch;
  auto kern = w4a16_gemm_nsplit_kernel<TM, TN, BK, WPS>;
  static int slots = 0;  // workgroups the chip holds at once
  if (!slots) {
    if (lds > 64 * 1024)
      HIP_RET(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    int dev = 0, cus = 0, per_cu = 0;
    HIP_RET(hipGetDevice(&dev));
    HIP_RET(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    HIP_RET(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kern), 256, lds));
    slots = cus * (per_cu > 0 ? per_cu : 1);
  }
  const int tilesM = (a.M + BM - 1) / BM, tilesN = (a.N + BN - 1) / BN;
  const int64_t total = (int64_t)tilesM * tilesN;
  int big_cols = tilesN;
  if (g_w4a16_tail && TM >= 2 && total > slots && total % slots) {
    // columns whose full tiles fit into whole rounds; the remaining columns as half tiles if that ends earlier
    const int cols = (int)(total / slots * slots / tilesM);
    const int64_t halves = (int64_t)(tilesN - cols) * ((a.M + BM / 2 - 1) / (BM / 2));
    const double as_full = (double)((total + slots - 1) / slots);
    // a half tile takes about 0.6 of a full one: it dequantizes the same weights for half the rows
    const double with_tail = (double)(((int64_t)cols * tilesM + slots - 1) / slots) + 0.6 * (double)((halves + slots - 1) / slots);
    if (with_tail < as_full) big_cols = cols;
  }
  const int64_t grid = (int64_t)tilesM * big_cols + (int64_t)(tilesN - big_cols) * ((a.M + BM / 2 - 1) / (BM / 2));
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), lds, st, a, big_cols);
  return (int)hipGetLastError();
}

// The packed matrix as wk_gemm.h reads it: a block is 64 elements, one 16-byte piece of codes per lane and the (scale, -zp * scale)
// pair of the lane's row; operand d is dword d, dequantized as everywhere else.
struct W4A16Waves {
  typedef W4A16PArgs Args;
  typedef v16f Acc;
  typedef f32x4 Sum4;
  typedef bf16x8 X;
  struct W {
    u32x4 q;
    u32x2 sz;
  };
  struct Col {
    uint32_t q, sz;
    int g64, last;
  };
  static __host__ __device__ __forceinline__ int kblocks(const Args& a) { return (a.K + 63) / 64; }
  static __device__ __forceinline__ int row_bytes(const Args& a) { return a.K * 2; }
  static __device__ __forceinline__ const void* activations(const Args& a) { return a.A; }
  static __device__ __forceinline__ __amdgpu_buffer_rsrc_t weights(const Args& a) {
    const int64_t bytes = w4a16_packed_qbytes(a.N, a.K) + w4a16_packed_n(a.N) * (a.K / a.group) * 8;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.P), 0, (uint32_t)bytes, 0x00020000);
  }
  static __device__ __forceinline__ Col col(const Args& a, int nb, int lane) {
    const int kbs = (int)(w4a16_packed_k(a.K) / 64), G = a.K / a.group;
    nb = min(nb, (int)(w4a16_packed_n(a.N) / 32) - 1);
    return Col{(uint32_t)((int64_t)nb * kbs * 1024 + lane * 16), (uint32_t)(w4a16_packed_qbytes(a.N, a.K) + ((int64_t)nb * G * 32 + (lane & 31)) * 8),
               a.group / 64, G - 1};
  }
  static __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, const Col& c, int kb, W& w) {
    w.q = __builtin_amdgcn_raw_buffer_load_b128(r, kb < 0 ? 0xffffffffu : c.q, kb * 1024, 0);
    w.sz = __builtin_amdgcn_raw_buffer_load_b64(r, kb < 0 ? 0xffffffffu : c.sz, min(kb / c.g64, c.last) * 256, 0);
  }
  static __device__ __forceinline__ X operand(const W& w, int d) {
    uint32_t o[4];
    dequant8(w.q[d], __uint_as_float(w.sz.x), __uint_as_float(w.sz.y), o);
    return __builtin_bit_cast(bf16x8, u32x4{o[0], o[1], o[2], o[3]});
  }
  static __device__ __forceinline__ Acc mma(const X& w, const X& x, const Acc& acc) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, x, acc, 0, 0, 0); }
  static __device__ __forceinline__ void store(const Args& a, int m, int n, f32x4 v) {
    uint16_t* c = a.C + (int64_t)m * a.N + n;
    if (n + 3 < a.N && a.N % 4 == 0 && reinterpret_cast<uintptr_t>(a.C) % 8 == 0) {
      if (a.bias) {
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] += bf16_to_f32(a.bias[n + e]);
      }
      *reinterpret_cast<uint2*>(c) = uint2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
      return;
    }
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (n + e < a.N) c[e] = (uint16_t)pack_bf16(a.bias ? v[e] + bf16_to_f32(a.bias[n + e]) : v[e], 0.f);
  }
};

static int g_w4a16_ptile = 0;  // packed path: 0 = heuristic, 1 = 128x384, 2 = 64x384, 3 = 128x128, 4 = 64x128, 5 = 128x256

static int g_w4a16_waves = 1;  // 0: only the weights-from-global tiles (comparison runs and tests)

// us that halves of K (eight waves) save a tile form, 0 where the four waves run: up to 256 tiles every tile has a CU to itself, and one wave per
// SIMD dequantizes and multiplies in turns; above that two workgroups share a CU and the four are faster (1.05 to 1.3 of the time with halves).
// Fitted to 71 to 84 shapes each within 1.7 % (rms).  Halves / whole, median over 298 shapes of 65 to 1500 rows: K up to 1500 0.91 to 0.97, up to 4000 0.79
// to 0.87, beyond 0.73 to 0.83; the sums of 128 x 384 do not fit the LDS.
static float w4a16_halves_gain(int form, int64_t M, int64_t N, int64_t K) {
  struct Gain {
    int bm, bn;
    float less, block;
  };
  static const Gain gains[] = {{128, 128, 1.23f, 0.1892f}, {128, 256, 1.553f, 0.1981f}, {}, {64, 128, 0.671f, 0.094f}, {64, 384, 1.781f, 0.173f}};  // forms 4 to 8
  if (form < 4 || form > 8 || !gains[form - 4].bm) return 0.f;
  const Gain& g = gains[form - 4];
  if (((M + g.bm - 1) / g.bm) * ((N + g.bn - 1) / g.bn) > 256) return 0.f;
  return std::max(0.f, g.block * (float)((K + 63) / 64) - g.less);
}

// Which form runs.  The waves-split-K forms (wk_gemm.h) serve from one token to about the batch whose large tiles fill the chip;
// 93 x 2048 x 6144: 43.6 -> 10.5 us, 1 x 2560 x 9728: 15.9 (a GEMV of fp32 FMAs) -> 11.9, 300 x 9728 x 2560: 36 -> 28, 2048 rows as before.
// Two tables: where tiles of 128 x 256 would be fewer than 192, costs fitted to 1703 random shapes (5 to 6000 rows, 64 to 22 000 channels, K 64
// to 10 000) within 4 to 8 % (rms, where a form is near the best); from 192 tiles on, costs fitted to 98 shapes of 512 and more channels, which
// are within 0.2 % of the best form there on average, 8 % at worst.  Over all the choice takes 1.009 times the best form's time (28 % more at
// worst, 1194 x 392 x 8960; more than 10 % in 34) and is more than 5 % slower than the tiles by rows and columns alone that ran before in 7;
// the second table for all sizes, without the tiles of 64 rows, made that 1.037, 266 and 130 (3500 x 456 x 1280: 18.3 us, 14.0 now).
static int w4a16_packed_form(int64_t M, int64_t N, int64_t K, bool tiles_only) {
  // Up to eight K blocks and 64 rows: four waves, since of more most have nothing to multiply and all of them meet.  us, as many waves as
  // below / four: 1 x 1440 x 128 3.76 / 2.85, 8 x 4096 x 512 3.99 / 3.26, 32 x 9728 x 512 4.44 / 4.40, 64 x 9728 x 128 5.40 / 3.84 (a GEMV of
  // fp32 FMAs took 3.4 for the first)
  if (!tiles_only && K <= 512 && M <= 64) return 9;
  constexpr int waves = 4, most = 9;
  static const FormCost few[most] = {
      {32, 32, 1, 1.0f, 1.00f, 2.408f, 1.616f, 0.06823f, 0.292f, 3.379f},     // 16 waves
      {32, 32, 1, 1.0f, 0.75f, 3.452f, 0.1624f, 0.07441f, 0.3295f, 2.168f},   // 8 waves, two workgroups per CU
      {32, 64, 1, 1.0f, 1.00f, 3.91f, 0.1143f, 0.1137f, 0.1157f, 1.484f},     // 8 waves
      {64, 64, 1, 1.0f, 0.75f, 4.599f, 0.03457f, 0.1918f, 0.2428f, 0.9395f},  // 4 waves, two workgroups per CU, or 8
      {128, 128, 3, 0.7f, 0.25f, 4.537f, 0.f, 0.631f, 0.288f, 0.3427f},       // weights-from-global tiles
      {128, 256, 1, 1.0f, 0.50f, 5.655f, 0.f, 0.8938f, 0.1696f, 0.3077f},
      {128, 384, 1, 1.0f, 1.00f, 4.017f, 3.449f, 1.104f, 0.1419f, 0.348f},
      {64, 128, 2, 0.6f, 0.50f, 3.84f, 0.1499f, 0.4126f, 0.1031f, 0.5252f},
      {64, 384, 1, 1.0f, 0.50f, 5.6f, 0.f, 0.8473f, 0.1218f, 0.3584f}};
  static const FormCost many[] = {{32, 32, 1, 1.f, 0.75f, 1.32f, 2.22f, 0.0906f, 0.f, 0.f},   {32, 32, 1, 1.f, 0.50f, 3.15f, 0.54f, 0.0879f, 0.f, 0.f},
                                  {32, 64, 1, 1.f, 0.75f, 3.20f, 0.85f, 0.1206f, 0.f, 0.f},   {64, 64, 1, 1.f, 0.50f, 3.79f, 0.95f, 0.2008f, 0.f, 0.f},
                                  {128, 128, 1, 1.f, 0.00f, 5.66f, 0.f, 0.6687f, 0.f, 0.f},   {128, 256, 1, 1.f, 0.75f, 7.69f, 0.46f, 0.8890f, 0.f, 0.f},
                                  {128, 384, 1, 1.f, 1.00f, 3.20f, 12.54f, 1.0826f, 0.f, 0.f}};
  const bool large = ((M + 127) / 128) * ((N + 255) / 256) >= 192;
  const FormCost* cost = large ? many : few;
  const int forms = large ? 7 : most;
  // What eight waves save comes off: halves of K as above; 64 x 64 fitted to 70 shapes of 100 to 256 such tiles, 2.2 % rms; over 250 shapes the choice takes
  // 0.981 of the time with four waves throughout, 41 of them 3 to 20 % less (119 x 7224 x 4416 20.6 -> 17.1 us).  Where a form of the waves that split K is the
  // cheapest by four, halves of K of a tile take its place only
  //  * with 2.8 us per million results added where rows are no multiple of 16 bytes: the tiles store those an element at a time (1.4 to 3 us by form, the
  //    waves' forms nothing), which had 40 of 372 such shapes 3 to 25 % slower (778 x 1915 x 1792 15.2 -> 19.1 us); not
  //    for many rows of long K, where the waves' forms take more than their costs.  Over 1872 such shapes 0.896 of the time of four waves, 20 of them 3 to 9 % slower
  //  * on 128 x 128 at 0.94 of the cost: at 0.95 to 0.975 of 32 x 64's 9 of 12 shapes were 2 to 7 % slower (258 x 6832 x 5120 39.8 -> 42.8)
  auto cheapest = [&](bool eight, bool split) {
    int form = -1;
    float best = 0.f;
    for (int f = tiles_only ? waves : 0; f < forms; f++) {
      float c = form_cost(cost[f], M, N, K, (K + 63) / 64);
      if (eight) {
        c -= w4a16_halves_gain(f, M, N, K);
        if (f == 3 && ((M + 63) / 64) * ((N + 63) / 64) <= WK_EIGHT_TILES) c -= 0.0322f * (float)((K + 63) / 64);
        if (split && f >= waves && N % 8 != 0 && (M < 900 || K < 3000)) c += 2.8e-6f * (float)(M > 32 ? M : 32) * (float)N;
        if (split && f == waves) c *= 1.06f;
      }
      if (form < 0 || c < best) {
        best = c;
        form = f;
      }
    }
    return form;
  };
  return cheapest(true, cheapest(false, false) < waves);
}
static int launch_w4a16_auto(const W4A16PArgs& a, hipStream_t st) {
  static const int tiles[] = {-1, 6, 8, 4, 7, 5};  // of g_w4a16_ptile
  const int form = g_w4a16_ptile ? tiles[g_w4a16_ptile] : w4a16_packed_form(a.M, a.N, a.K, !g_w4a16_waves);
  const bool halves = !g_w4a16_ptile && w4a16_halves_gain(form, a.M, a.N, a.K) > 0.f;  // (a tile asked for runs by four waves)
  if (a.M <= 8) switch (form) {  // one piece of eight rows; faster at every size measured (512 to 22016 channels, K 512 to 11008)
    case 0: return wk_gemm_launch<W4A16Waves, 1, 1, 16, 2, 1>(a, st);
    case 1: return wk_gemm_launch<W4A16Waves, 1, 1, 8, 3, 1>(a, st);
    case 2: return wk_gemm_launch<W4A16Waves, 1, 2, 8, 1, 1>(a, st);
    case 9: return wk_gemm_launch<W4A16Waves, 1, 1, 4, 1, 1>(a, st);
  }
  switch (form) {
    case 0: return wk_gemm_launch<W4A16Waves, 1, 1, 16, 2>(a, st);
    case 1: return wk_gemm_launch<W4A16Waves, 1, 1, 8, 3>(a, st);
    case 2: return wk_gemm_launch<W4A16Waves, 1, 2, 8, 1>(a, st);
    case 3: return wk_gemm_64x64<W4A16Waves>(a, st);
    case 4: return halves ? launch_w4a16_halves<4, 1, 64>(a, st) : launch_w4a16_nsplit<4, 1, 64, 3>(a, st);
    case 5: return halves ? launch_w4a16_halves<4, 2, 64>(a, st) : launch_w4a16_nsplit<4, 2, 64, 2>(a, st);
    case 6: return launch_w4a16_nsplit<4, 3, 128, 1>(a, st);
    case 7: return halves ? launch_w4a16_halves<2, 1, 128>(a, st) : launch_w4a16_nsplit<2, 1, 128, 2>(a, st);
    case 8: return halves ? launch_w4a16_halves<2, 3, 128>(a, st) : launch_w4a16_nsplit<2, 3, 128, 2>(a, st);
    default: return wk_gemm_launch<W4A16Waves, 1, 1, 4, 1>(a, st);
  }
}

template <int BM, int BN, int WM, int WN>
static int launch_w4a16(const W4A16Args& a, hipStream_t st) {
  constexpr int NT = (BM / WM) * (BN / WN) * 64;
  const size_t lds = 2 * (size_t)(BM + BN) * 144;
  const unsigned grid = (unsigned)(((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN));
  auto kern = w4a16_gemm_kernel<BM, BN, WM, WN>;
  if (lds > 64 * 1024)
    HIP_RET(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(kern, dim3(grid), dim3(NT), lds, st, a);
  return (int)hipGetLastError();
}

static int g_w4a16_tile = 0;  // 0 = heuristic, 1 = 256x192, 2 = 128x128, 3 = 64x64

}  // namespace mllmhip

using namespace mllmhip;

MLLM_API int mllm_hip_w4a16_set_tuning(int tile) {
  if (tile < 0 || tile > 3) return MLLM_HIP_E_BADARG;
  g_w4a16_tile = tile;
  return 0;
}

MLLM_API int mllm_hip_w4a16_packed_form(int64_t M, int64_t N, int64_t K) {
  return M < 1 || N < 1 || K < 1 ? 0 : 1 + w4a16_packed_form(M, N, K, false);
}
MLLM_API int mllm_hip_w4a16_packed_eight(int64_t M, int64_t N, int64_t K) {
  if (M < 1 || N < 1 || K < 1) return 0;
  const int form = w4a16_packed_form(M, N, K, false);
  return form == 3 ? wk_eight(M, N, (K + 63) / 64) : w4a16_halves_gain(form, M, N, K) > 0.f;
}
MLLM_API int mllm_hip_w4a16_packed_set_tuning(int tile) {
  if (tile < 0 || (tile & 15) > 5 || tile > 31) return MLLM_HIP_E_BADARG;
  g_w4a16_ptile = tile & 15;
  g_w4a16_tail = !(tile & 16);
  return 0;
}

static int check_w4a16(const void* qw, const void* s, const void* zp, int64_t N, int64_t K, int group) {
  if (!qw || !s || !zp || N <= 0 || K <= 0 || group <= 0) return MLLM_HIP_E_BADARG;
  if (group % 64 || K % group) return MLLM_HIP_E_SHAPE;
  if (N * K / 2 >= ((int64_t)1 << 32) || N > INT32_MAX || K > INT32_MAX) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(qw) % 16) return MLLM_HIP_E_ALIGN;
  return 0;
}

MLLM_API int mllm_hip_w4a16_gemm(const void* a_bf16, const uint8_t* qw, const uint16_t* scales, const uint8_t* zeros,
                                 const void* bias_bf16, void* c_bf16, int64_t M, int64_t N, int64_t K, int group,
                                 void* stream) {
  int rc = check_w4a16(qw, scales, zeros, N, K, group);
  if (rc) return rc;
  if (!a_bf16 || !c_bf16 || M <= 0) return MLLM_HIP_E_BADARG;
  if (M * K * 2 >= ((int64_t)1 << 32) || M > INT32_MAX) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(a_bf16) % 16) return MLLM_HIP_E_ALIGN;
  W4A16Args a{(const uint16_t*)a_bf16, qw, scales, zeros, (const uint16_t*)bias_bf16, (uint16_t*)c_bf16,
              (int)M, (int)N, (int)K, group};
  hipStream_t st = (hipStream_t)stream;
  int tile = g_w4a16_tile;
  if (!tile) {
    const int64_t big = ((M + 255) / 256) * ((N + 191) / 192);
    const int64_t mid = ((M + 127) / 128) * ((N + 127) / 128);
    (void)big;  // the 256x192 tile is compiled and tested but measured slower than 128x128 so far
    tile = mid >= 128 ? 2 : 3;
  }
  switch (tile) {
    case 1: return launch_w4a16<256, 192, 128, 96>(a, st);
    case 2: return launch_w4a16<128, 128, 64, 64>(a, st);
    default: return launch_w4a16<64, 64, 32, 32>(a, st);
  }
}

MLLM_API int mllm_hip_w4a16_dequantize(const uint8_t* qw, const uint16_t* scales, const uint8_t* zeros, void* w_bf16,
                                       int64_t N, int64_t K, int group, void* stream) {
  int rc = check_w4a16(qw, scales, zeros, N, K, group);
  if (rc) return rc;
  if (!w_bf16) return MLLM_HIP_E_BADARG;
  const int64_t words = N * K / 8;
  hipLaunchKernelGGL(w4a16_dequant_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, (hipStream_t)stream, qw,
                     scales, zeros, (uint16_t*)w_bf16, N, K, group);
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------------
// AWQ checkpoint tensors -> the row-major layout of this file (the unpacking half of what the reference does in
// AWQMarlinLinearMethod.process_weights_after_loading, pymllm/quantization/methods/awq_marlin.py:366-410).
//   qweight int32 [K][N/8], qzeros int32 [K/group][N/8]: eight 4-bit codes of eight neighbouring output columns per dword,
//   nibble position p holding column 8 j + {0,2,4,6,1,3,5,7}[p] (awq_marlin.py:202-213 unpack_cols followed by the
//   undo_interleave of :248-257; awq_marlin_repack.cuh:108-110 reads column c from nibble {0,4,1,5,2,6,3,7}[c]);
//   scales fp16 [K/group][N].
// The weight codes are transposed through LDS in 64 x 64 tiles so that both the checkpoint reads and the [N][K/2] writes
// are whole 32-byte runs.
__device__ __forceinline__ int awq_nibble_of_column(int c) { return ((c & 1) << 2) | (c >> 1); }  // {0,4,1,5,2,6,3,7}[c]

__global__ __launch_bounds__(256) void awq_unpack_q_kernel(const uint32_t* __restrict__ qweight, uint32_t* __restrict__ qw,
                                                           int N, int K) {
  __shared__ uint32_t tile[64][9];  // [k][column dword], one pad dword against bank conflicts of the column reads
  const int n0 = blockIdx.x * 64, k0 = blockIdx.y * 64, t = threadIdx.x;
  const int nd = N / 8;
  for (int i = t; i < 512; i += 256) {
    const int k = k0 + i / 8, j = n0 / 8 + i % 8;
    tile[i / 8][i % 8] = (k < K && j < nd) ? qweight[(int64_t)k * nd + j] : 0u;
  }
  __syncthreads();
  for (int i = t; i < 512; i += 256) {
    const int r = i / 8, kd = i % 8;  // output row n0 + r, its dword of elements k0 + 8 kd .. + 7
    const int n = n0 + r, k = k0 + kd * 8;
    if (n >= N || k >= K) continue;
    const int sh = 4 * awq_nibble_of_column(r & 7);
    uint32_t v = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) v |= ((tile[kd * 8 + e][r >> 3] >> sh) & 15u) << (4 * e);
    qw[((int64_t)n * K + k) / 8] = v;
  }
}

__global__ __launch_bounds__(256) void awq_unpack_sz_kernel(const uint32_t* __restrict__ qzeros, const uint16_t* __restrict__ s_in,
                                                            uint16_t* __restrict__ s_out, uint8_t* __restrict__ z_out, int N,
                                                            int G) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // (group, n): neighbouring threads read neighbouring columns
  if (i >= (int64_t)N * G) return;
  const int n = (int)(i % N), g = (int)(i / N);
  s_out[(int64_t)n * G + g] = s_in[(int64_t)g * N + n];
  if (g & 1) return;  // one thread per byte of zero points: groups g (low nibble) and g + 1 (high nibble)
  const int sh = 4 * awq_nibble_of_column(n & 7), nd = N / 8;
  uint32_t z = (qzeros[(int64_t)g * nd + n / 8] >> sh) & 15u;
  if (g + 1 < G) z |= ((qzeros[(int64_t)(g + 1) * nd + n / 8] >> sh) & 15u) << 4;
  z_out[(int64_t)n * ((G + 1) / 2) + g / 2] = (uint8_t)z;
}

MLLM_API int mllm_hip_w4a16_from_awq(const int32_t* qweight, const int32_t* qzeros, const uint16_t* scales, int64_t N,
                                     int64_t K, int group, uint8_t* qw, uint16_t* scales_out, uint8_t* zeros_out,
                                     void* stream) {
  if (!qweight || !qzeros || !scales || !qw || !scales_out || !zeros_out || N <= 0 || K <= 0 || group <= 0)
    return MLLM_HIP_E_BADARG;
  if (N % 8 || K % 8 || K % group) return MLLM_HIP_E_SHAPE;
  if (N * K / 2 >= ((int64_t)1 << 32) || N > INT32_MAX || K > INT32_MAX) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(qw) % 4 || reinterpret_cast<uintptr_t>(qweight) % 4 ||
      reinterpret_cast<uintptr_t>(qzeros) % 4)
    return MLLM_HIP_E_ALIGN;
  const int G = (int)(K / group);
  if ((K + 63) / 64 > 65535) return MLLM_HIP_E_SHAPE;
  hipLaunchKernelGGL(awq_unpack_q_kernel, dim3((unsigned)((N + 63) / 64), (unsigned)((K + 63) / 64)), dim3(256), 0,
                     (hipStream_t)stream, reinterpret_cast<const uint32_t*>(qweight), reinterpret_cast<uint32_t*>(qw), (int)N,
                     (int)K);
  hipLaunchKernelGGL(awq_unpack_sz_kernel, dim3((unsigned)((N * G + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     reinterpret_cast<const uint32_t*>(qzeros), scales, scales_out, zeros_out, (int)N, G);
  return (int)hipGetLastError();
}

MLLM_API size_t mllm_hip_w4a16_packed_bytes(int64_t N, int64_t K, int group) {
  if (N <= 0 || K <= 0 || group <= 0 || group % 64 || K % group) return 0;
  return (size_t)(w4a16_packed_qbytes(N, K) + w4a16_packed_n(N) * (K / group) * 8);
}

MLLM_API int mllm_hip_w4a16_prepack(const uint8_t* qw, const uint16_t* scales, const uint8_t* zeros, int64_t N, int64_t K,
                                    int group, void* packed, void* stream) {
  int rc = check_w4a16(qw, scales, zeros, N, K, group);
  if (rc) return rc;
  if (!packed) return MLLM_HIP_E_BADARG;
  if (reinterpret_cast<uintptr_t>(packed) % 16) return MLLM_HIP_E_ALIGN;
  if (mllm_hip_w4a16_packed_bytes(N, K, group) >= ((size_t)1 << 32)) return MLLM_HIP_E_SHAPE;
  const int64_t words = w4a16_packed_qbytes(N, K) / 4;
  hipLaunchKernelGGL(w4a16_prepack_q_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, (hipStream_t)stream, qw,
                     reinterpret_cast<uint32_t*>(packed), (int)N, (int)K, words);
  const int G = (int)(K / group);
  const int64_t count = w4a16_packed_n(N) * G;
  hipLaunchKernelGGL(w4a16_prepack_sz_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, (hipStream_t)stream, scales,
                     zeros, reinterpret_cast<float2*>(reinterpret_cast<char*>(packed) + w4a16_packed_qbytes(N, K)), (int)N, G,
                     count);
  return (int)hipGetLastError();
}

MLLM_API int mllm_hip_w4a16_set_decode(int gemv) {
  if (gemv != 0 && gemv != 1) return MLLM_HIP_E_BADARG;
  g_w4a16_waves = gemv;
  return 0;
}
MLLM_API int mllm_hip_w4a16_set_decode_mfma_from(int tokens) {  // (every token count is on the matrix cores)
  return tokens < 1 || tokens > 33 ? MLLM_HIP_E_BADARG : 0;
}

MLLM_API int mllm_hip_w4a16_gemm_packed(const void* a_bf16, const void* packed, const void* bias_bf16, void* c_bf16,
                                        int64_t M, int64_t N, int64_t K, int group, void* stream) {
  if (!a_bf16 || !packed || !c_bf16 || M <= 0 || N <= 0 || K <= 0 || group <= 0) return MLLM_HIP_E_BADARG;
  if (group % 64 || K % group) return MLLM_HIP_E_SHAPE;
  if (M * K * 2 >= ((int64_t)1 << 32) || M > INT32_MAX || N > INT32_MAX ||
      mllm_hip_w4a16_packed_bytes(N, K, group) >= ((size_t)1 << 32))
    return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(a_bf16) % 16 || reinterpret_cast<uintptr_t>(packed) % 16) return MLLM_HIP_E_ALIGN;
  W4A16PArgs a{(const uint16_t*)a_bf16, (const uint8_t*)packed, (const uint16_t*)bias_bf16, (uint16_t*)c_bf16,
               (int)M, (int)N, (int)K, group};
  return launch_w4a16_auto(a, (hipStream_t)stream);
}

MLLM_API int mllm_hip_w4a16_dequantize_packed(const void* packed, void* w_bf16, int64_t N, int64_t K, int group, void* stream) {
  if (!packed || !w_bf16 || N <= 0 || K <= 0 || group <= 0) return MLLM_HIP_E_BADARG;
  if (group % 64 || K % group || N > INT32_MAX || K > INT32_MAX) return MLLM_HIP_E_SHAPE;
  const int64_t words = N * K / 8;
  hipLaunchKernelGGL(w4a16_dequant_packed_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     (const uint8_t*)packed, (uint16_t*)w_bf16, (int)N, (int)K, group);
  return (int)hipGetLastError();
}

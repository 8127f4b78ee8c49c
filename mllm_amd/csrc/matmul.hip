// Activation x activation MatMul on the matrix cores (the kMatMul factory slot of the backend: attention scores, attention
// x values and the MoE gate logits of the reference run through it, mllm/backends/cpu/ops/MatMulOp.cpp:27-61 with the batch
// loop of mllm/backends/cpu/kernels/common/ggml/matmul.cpp / mllm_blas).  Not a quantized path.
//   fp32 operands   v_mfma_f32_32x32x2f32: exact fp32 products, fp32 accumulation (the CPU's arithmetic in another order); larger products from
//                   three bf16 parts per operand, to within 2^-34 of a product (matmul_split_kernel)
//   bf16 / fp16     v_mfma_f32_32x32x16_{bf16,f16}: exact products, fp32 accumulation, one rounding of the result
// One launch covers the whole batch (a stride of 0 broadcasts an operand).
//
// Workgroup = 2 x 2 waves, each wave (32 TM) x (32 TN) outputs, K step 32.  Both operand tiles sit in LDS with
// 16 bytes of padding per row, as [row][k] whichever way the tensor is laid out in memory (fp32 [K][rows] operands stay [k][row]).  Inside a K step lane half h takes k = 16 h .. 16 h + 15 of its row, for both
// operands alike: the order in which an MFMA walks k is free, and this way every lane fetches its operands of the whole
// step with 16-byte LDS reads.
#include <algorithm>
#include <cmath>

#include "qcommon.h"

namespace mllmhip {

typedef __bf16 mm_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 mm_f16x8 __attribute__((ext_vector_type(8)));
typedef float mm_f32x16 __attribute__((ext_vector_type(16)));

struct MMArgs {
  const void* A;
  const void* B;
  void* C;
  int M, N, K, batch;
  int64_t sA, sB, sC;  // batch strides in elements
  int vecA, vecB;      // aligned 16-byte loads of whole rows (base, leading dimension and batch stride all multiples of 16 bytes)
};

// The grid of a launch of `total` workgroups (below 2^31): HIP counts the work-items of a dimension in 32 bits, which 2^24 workgroups of
// 256 threads no longer fit, so that more than 2^21 are rows of 2^21 (a multiple of the XCDs).  The last row may reach past the end.
static dim3 mm_grid(int64_t total) {
  constexpr int64_t ROW = 1 << 21;
  return total <= ROW ? dim3((unsigned)total) : dim3((unsigned)ROW, (unsigned)((total + ROW - 1) / ROW));
}
__device__ __forceinline__ int mm_block() { return (int)(blockIdx.y * gridDim.x + blockIdx.x); }
// n / d for the same n in every lane; inv = mm_inv(d, n's bound): a division instruction sequence costs a small product as much as a K step
static uint32_t mm_inv(int64_t d, int64_t bound) { return d > 1 && bound <= 65536 ? (uint32_t)(((1ull << 32) + d - 1) / d) : 0u; }
__device__ __forceinline__ int mm_div(int n, int d, uint32_t inv) {
  return d == 1 ? n : inv ? (int)__umulhi((uint32_t)n, inv) : n / d;  // (n, d < 2^16: exact)
}

template <int DT>
struct MMElem {
  using type = uint16_t;
};
template <>
struct MMElem<MLLM_HIP_F32> {
  using type = float;
};

// One operand tile of ROWS x 32 elements from global memory into registers, then into LDS.
// CONTIG_K: the tensor is [rows][K] (k contiguous); otherwise it is [K][rows].  In LDS the tile is [row][k], except that an fp32
// tensor [K][rows] stays [k][row]: v_mfma_f32_32x32x2f32 takes one k per lane half, so a lane's operand is one dword and
// neighbouring lanes read neighbouring dwords.  A 16-bit tensor [K][rows] is loaded as two neighbouring k of four rows per
// thread and vector, which makes one dword of LDS per row.
// Whole tiles load whole vectors whatever the alignment of the rows (odd row lengths among them); rows past the end repeat the
// last ones (their results are never stored).  A K step that ends behind K, and a last tile of rows that are not a multiple of
// the vector in a [K][rows] tensor, load element by element with zeros outside; MM_VECTORS: the shape has neither but K steps whose
// vectors lie inside or outside as a whole (mm_vectors below), and no element by element code: the short products that this is for
// are bound by their few K steps (bf16 1000 x 8 x 8 x 8: 4.7 us by elements, 3.3; 8 x 800 x 64 x 200 5.7 / 4.8).  MM_STEP: one K step, element
// by element and nothing else: 0.3 to 0.5 us of a launch are waits for code (8 x 69 x 7 x 18 bf16 4.84 us with the general form's, 4.4).
// MM_NARROW: rows past the end are not requested again but stay zero (mm_narrow below).
enum { MM_ANY, MM_VECTORS, MM_STEP, MM_NARROW };
template <typename E, int ROWS, bool CONTIG_K, int FORM, int NT = 256>
struct MMTile {
  static constexpr bool VECTORS = FORM == MM_VECTORS;
  static constexpr int VE = 16 / (int)sizeof(E);
  static constexpr bool KROWS = !CONTIG_K && sizeof(E) == 4;   // [k][row] in LDS
  static constexpr bool PAIRS = !CONTIG_K && sizeof(E) == 2;   // two k of four rows per vector
  static constexpr int RV = CONTIG_K ? 1 : 4;                  // rows of a vector
  static constexpr int LD = KROWS ? ROWS + VE : 32 + VE;
  static constexpr int SIZE = KROWS ? 32 * LD : ROWS * LD;     // elements in LDS
  static constexpr int NV = ROWS * 32 / VE / NT;               // 16-byte vectors per thread
  static_assert(ROWS * 32 / VE % NT == 0, "tile must split evenly over the threads");
  u32x4 v[NV];
  const E* p[NV];
  bool whole, inside[FORM == MM_NARROW ? NV : 1];

  static __device__ __forceinline__ uint32_t bits(E e) {
    if constexpr (sizeof(E) == 4) return __builtin_bit_cast(uint32_t, e);
    else return (uint32_t)e;
  }
  // j is a compile-time constant after unrolling; the element goes through a plain dword first (a bit cast applied directly
  // to q[j] was compiled as a read of element 0)
  static __device__ __forceinline__ E elem(u32x4 q, int j) {
    const uint32_t d = sizeof(E) == 4 ? q[j] : (q[j >> 1] >> (16 * (j & 1)));
    if constexpr (sizeof(E) == 4) return __builtin_bit_cast(E, d);
    else return (E)d;
  }
  static __device__ __forceinline__ void place(int c, int& r, int& k) {  // first element of vector c of this thread inside the tile
    const int idx = c * NT + (int)threadIdx.x;
    if (CONTIG_K) r = idx / (32 / VE), k = (idx % (32 / VE)) * VE;
    else if (PAIRS) k = idx / (ROWS / 4) * 2, r = (idx % (ROWS / 4)) * 4;
    else k = idx / (ROWS / VE), r = (idx % (ROWS / VE)) * VE;
  }
  __device__ __forceinline__ void start(const E* __restrict__ X, int row0, int rows, int K) {
    if (FORM == MM_STEP) return;
    whole = CONTIG_K || VECTORS || (rows >= RV && (row0 + ROWS <= rows || rows % RV == 0));  // (the same in every thread)
#pragma unroll
    for (int c = 0; c < NV; ++c) {
      int r, k;
      place(c, r, k);
      if constexpr (FORM == MM_NARROW) {
        inside[c] = row0 + r < rows;
        v[c] = u32x4{0u, 0u, 0u, 0u};
      }
      if (CONTIG_K) p[c] = X + (int64_t)min(row0 + r, rows - 1) * K + k;
      else p[c] = X + (int64_t)k * rows + (whole ? min(row0 + r, rows - RV) : 0);
    }
  }
  static __device__ __forceinline__ u32x4 vector(const E* __restrict__ at, int rows) {
    u32x4 q;
    if constexpr (PAIRS) {
      u32x2 lo, hi;
      __builtin_memcpy(&lo, at, 8);
      __builtin_memcpy(&hi, at + rows, 8);
      q = u32x4{lo.x, lo.y, hi.x, hi.y};
    } else {
      __builtin_memcpy(&q, at, 16);
    }
    return q;
  }
  __device__ __forceinline__ void load(const E* __restrict__ X, int row0, int k0, int rows, int K) {
    if (FORM != MM_STEP && (VECTORS || whole) && k0 + 32 <= K) {
      const int64_t step = CONTIG_K ? (int64_t)k0 : (int64_t)k0 * rows;
#pragma unroll
      for (int c = 0; c < NV; ++c)
        if (FORM != MM_NARROW || inside[FORM == MM_NARROW ? c : 0]) v[c] = vector(p[c] + step, rows);
      return;
    }
    if constexpr (VECTORS) {
      const int64_t step = CONTIG_K ? (int64_t)k0 : (int64_t)k0 * rows;
#pragma unroll
      for (int c = 0; c < NV; ++c) {
        int r, k;
        place(c, r, k);
        v[c] = u32x4{0u, 0u, 0u, 0u};
        if (k0 + k < K) v[c] = vector(p[c] + step, rows);
      }
      return;
    }
#pragma unroll
    for (int c = 0; c < NV; ++c) {
      int r, k;
      place(c, r, k);
      r += row0;
      k += k0;
      u32x4 q = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int j = 0; j < VE; ++j) {
        const int rj = CONTIG_K ? r : PAIRS ? r + j % 4 : r + j, kj = CONTIG_K ? k + j : PAIRS ? k + j / 4 : k;
        const uint32_t e = rj < rows && kj < K ? bits(X[CONTIG_K ? (int64_t)rj * K + kj : (int64_t)kj * rows + rj]) : 0u;
        if constexpr (sizeof(E) == 4) q[j] = e;
        else q[j >> 1] |= e << (16 * (j & 1));
      }
      v[c] = q;
    }
  }
  __device__ __forceinline__ void store(E* __restrict__ s) const {
#pragma unroll
    for (int c = 0; c < NV; ++c) {
      int r, k;
      place(c, r, k);
      if constexpr (CONTIG_K) {
        *reinterpret_cast<u32x4*>(s + r * LD + k) = v[c];
      } else if constexpr (KROWS) {
        *reinterpret_cast<u32x4*>(s + k * LD + r) = v[c];
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          *reinterpret_cast<uint32_t*>(s + (r + j) * LD + k) = __builtin_amdgcn_perm(v[c][2 + (j >> 1)], v[c][j >> 1], j & 1 ? 0x07060302u : 0x05040100u);
      }
    }
  }
  // fp32: the operand of instruction 4 q + s of a K step (k = 16 h + 4 q + s) for s = 0 .. 3, row r of the tile
  static __device__ __forceinline__ f32x4 four(const E* __restrict__ s, int r, int h, int q) {
    static_assert(sizeof(E) == 4 || !KROWS, "");
    const float* f = reinterpret_cast<const float*>(s);
    if constexpr (!KROWS) return *reinterpret_cast<const f32x4*>(f + r * LD + 16 * h + 4 * q);
    else return f32x4{f[(16 * h + 4 * q) * LD + r], f[(16 * h + 4 * q + 1) * LD + r], f[(16 * h + 4 * q + 2) * LD + r], f[(16 * h + 4 * q + 3) * LD + r]};
  }
};

// one K step of fp32 instructions from the two tiles in LDS
template <typename TileA, typename TileB, int TM, int TN>
__device__ __forceinline__ void mm_f32_step(const float* sA, const float* sB, int wm, int wn, int r, int h, mm_f32x16 (&acc)[TM][TN]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {  // four k of this lane's sixteen at a time
    f32x4 fa[TM], fb[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[i] = TileA::four(sA, wm * 32 * TM + i * 32 + r, h, q);
#pragma unroll
    for (int j = 0; j < TN; ++j) fb[j] = TileB::four(sB, wn * 32 * TN + j * 32 + r, h, q);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i][s], fb[j][s], acc[i][j], 0, 0, 0);
  }
}
template <int DT, int TM, int TN, int BM, int BN>
__device__ __forceinline__ void mm_store(const MMArgs& a, typename MMElem<DT>::type* C, int m0, int n0, int wm, int wn, int r, int h, const mm_f32x16 (&acc)[TM][TN]) {
  // 32x32 accumulator layout: register v of lane l holds row 8 (v / 4) + 4 (l / 32) + v % 4, column l % 32
  auto put = [&](int m, int n, float f) {
    if constexpr (DT == MLLM_HIP_F32) C[(int64_t)m * a.N + n] = f;
    else if constexpr (DT == MLLM_HIP_BF16) C[(int64_t)m * a.N + n] = f32_to_bf16(f);
    else C[(int64_t)m * a.N + n] = f32_to_f16bits(f);
  };
  const bool full = m0 + BM <= a.M && n0 + BN <= a.N;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + wn * 32 * TN + j * 32 + r;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = m0 + wm * 32 * TM + i * 32 + 8 * (v / 4) + 4 * h + (v % 4);
        if (full || (n < a.N && m < a.M)) put(m, n, acc[i][j][v]);
      }
  }
}

// Bound by the matrix pipe in fp32 (157 TFLOP/s nominal; larger fp32 products run in matmul_split_kernel), by LDS reads and the output in 16 bits.  The next K step is loaded into
// registers during this one's matrix instructions.  One LDS stage: a second one halves the workgroups of a CU, which hide
// the barriers better (fp32 8 x 3108 x 777 x 128: 59 us, 62 with two stages).  The tiles of one batch entry are
// neighbours on one XCD, whose L2 then holds that entry's operands.  16 bits, large tile: 128 registers, four waves per SIMD instead of
// three (4096 x 4096 x 4096 bf16: 236 -> 180 us).
//   (heads x rows x keys x d) fp32 8 x 3108 x 777 x 128: scores 80 -> 59 us, values 97 -> 65; bf16 33 -> 23, 70 -> 26 (odd row lengths
//   loaded element by element and transposed through 16 two-byte LDS stores before)
template <int DT, bool TA, bool TB, int TM, int TN, int FORM>
__global__ __launch_bounds__(256, (TM * TN == 4 && DT != MLLM_HIP_F32) ? 4 : 1) void matmul_kernel(MMArgs a, int tiles, int tilesM, uint32_t inv_tiles, uint32_t inv_tilesM) {
  using E = typename MMElem<DT>::type;
  constexpr int BM = 64 * TM, BN = 64 * TN;
  // A is [M][K], or [K][M] when transposed; B is [K][N], or [N][K] when transposed
  typedef MMTile<E, BM, !TA, FORM> TileA;
  typedef MMTile<E, BN, TB, FORM == MM_NARROW ? MM_ANY : FORM> TileB;
  __shared__ __align__(16) E sA[TileA::SIZE];
  __shared__ __align__(16) E sB[TileB::SIZE];

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1, r = lane & 31, h = lane >> 5;
  const int KT = FORM == MM_STEP ? 1 : (a.K + 31) / 32;
  const int total = tiles * a.batch, b = mm_block();
  if (b >= total) return;  // (uniform)
  const int t = xcd_run(b, total), z = mm_div(t, tiles, inv_tiles), in = t - z * tiles;
  const int tn = mm_div(in, tilesM, inv_tilesM), n0 = tn * BN, m0 = (in - tn * tilesM) * BM;
  const E* A = reinterpret_cast<const E*>(a.A) + z * a.sA;
  const E* B = reinterpret_cast<const E*>(a.B) + z * a.sB;
  E* C = reinterpret_cast<E*>(a.C) + z * a.sC;

  TileA ta;
  TileB tb;
  mm_f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  ta.start(A, m0, a.M, a.K);
  tb.start(B, n0, a.N, a.K);
  ta.load(A, m0, 0, a.M, a.K);
  tb.load(B, n0, 0, a.N, a.K);
  for (int kt = 0; kt < KT; ++kt) {
    __syncthreads();  // the previous step's LDS reads are done
    ta.store(sA);
    tb.store(sB);
    __syncthreads();
    if (kt + 1 < KT) {
      ta.load(A, m0, (kt + 1) * 32, a.M, a.K);
      tb.load(B, n0, (kt + 1) * 32, a.N, a.K);
    }
    if constexpr (DT == MLLM_HIP_F32) {
      mm_f32_step<TileA, TileB, TM, TN>(sA, sB, wm, wn, r, h, acc);
    } else {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        u32x4 fa[TM], fb[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) fa[i] = *reinterpret_cast<const u32x4*>(sA + (wm * 32 * TM + i * 32 + r) * TileA::LD + 16 * h + 8 * q);
#pragma unroll
        for (int j = 0; j < TN; ++j) fb[j] = *reinterpret_cast<const u32x4*>(sB + (wn * 32 * TN + j * 32 + r) * TileB::LD + 16 * h + 8 * q);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            if constexpr (DT == MLLM_HIP_BF16)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(mm_bf16x8, fa[i]),
                                                                  __builtin_bit_cast(mm_bf16x8, fb[j]), acc[i][j], 0, 0, 0);
            else
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(mm_f16x8, fa[i]),
                                                                 __builtin_bit_cast(mm_f16x8, fb[j]), acc[i][j], 0, 0, 0);
          }
      }
    }
  }

  mm_store<DT, TM, TN, BM, BN>(a, C, m0, n0, wm, wn, r, h, acc);
}

// fp32 operands on the bf16 matrix instructions, which do sixteen times the products per clock.  A float is the sum of three bf16 numbers,
// exactly: x0 = bf16(x), x1 = bf16(x - x0), x2 = x - x0 - x1.  Eight of the nine products are multiplied; x2 y2 is below 2^-34 of a product.
// An instruction cuts off what it adds to a larger sum where the fp32 ones round, so the products but x0 y0 have a sum of their own, the smallest first, which
// is added at the end: a single product is within 0.506 ulp (fp32 instructions 0.5; without x1 y2 and x2 y1 and in one sum 1.43), the results are nearer to
// 64 bits than theirs (8 x 3108 x 777 x 128: 0.65e-7 of the norm against 2.03e-7, x 128 x 777: 1.6e-7 against 5.0e-7).
// Bound by the matrix pipe at the clock it holds under this load, by LDS reads (nine 16-byte reads per sixteen instructions; a wave tile of 32 x
// 64) and by the splitting (six vector instructions per element), which share the issue slots; the matrix instructions alone take 23 us per 128 k of
// 8 x 3072 x 768, the fp32 ones 45.  K steps of sixteen in two LDS buffers, one barrier each; one (large tile, two accumulators) to four workgroups
// per CU.  On the large tile three of the splitting's instructions follow each matrix instruction: in front of them all, they took their time alone,
// two waves per SIMD or not (8 x 3108 x 128 x 777: 50 -> 43 us, 2048 x 2048 x 2048 131 -> 112; on the small one, bound by LDS reads at 64 bytes
// per clock, nothing).  Waves of 64 x 64 read less (4096 x 4096 x 1024 233 -> 220) but have 256 registers and, one per SIMD, nothing beside them (8 x 3108 x 128 x 777: 48).  One LDS buffer with steps of 32, operands read a step ahead, and tiles of 64 x 128 with four waves were no faster.
//   8 x 3108 x 777 x 128 (scores): 61 -> 55 us, x 128 x 777 (values): 61.5 -> 43; 8 x 4096 x 1024 x 128: 85 -> 80
struct MMParts {
  uint32_t p[3];
};
__device__ __forceinline__ MMParts mm_split(float a, float b) {  // two neighbouring k of a row
  MMParts s;
  s.p[0] = pack_bf16(a, b);
  a -= __uint_as_float(s.p[0] << 16), b -= __uint_as_float(s.p[0] & 0xffff0000u);
  s.p[1] = pack_bf16(a, b);
  a -= __uint_as_float(s.p[1] << 16), b -= __uint_as_float(s.p[1] & 0xffff0000u);
  s.p[2] = pack_bf16(a, b);
  return s;
}
// An operand tile of ROWS x 16 elements (K >= 16): in LDS [row][part][k], 16 bytes of padding per row (16-byte reads of neighbouring rows
// meet different banks).  A last K step that ends behind K is moved back to end at K, and what the step before it has multiplied is zero
// in it: every load is whole, without a branch.  Rows past the end repeat the last one.
template <int ROWS, bool CONTIG_K, int NT>
struct MMSplitTile {
  static constexpr int LD = 3 * 32 + 16, SIZE = ROWS * LD;  // bytes
  static_assert(ROWS * 4 == NT && ROWS >= 64, "four k of one row per thread");
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t off, ld;
  u32x4 v[2];  // two K steps in flight
  static __device__ __forceinline__ int row() { return CONTIG_K ? (int)threadIdx.x / 4 : (int)threadIdx.x % ROWS; }
  static __device__ __forceinline__ int kfirst() {  // of the step's 16
    return CONTIG_K ? (int)threadIdx.x % 4 * 4 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / ROWS) * 4;  // (the same in a wave)
  }
  __device__ __forceinline__ void start(const float* X, int row0, int rows, int K) {
    rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(X), 0, (uint32_t)rows * (uint32_t)K * 4u, 0x00020000);
    const uint32_t r = (uint32_t)min(row0 + row(), rows - 1);
    off = CONTIG_K ? (r * (uint32_t)K + kfirst()) * 4u : r * 4u;
    ld = (uint32_t)rows * 4u;
  }
  __device__ __forceinline__ void load(int d, int k) {  // k: the first of the step's 16
    if constexpr (CONTIG_K) {
      v[d] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, k * 4, 0);
    } else {
      const uint32_t at = (uint32_t)(k + kfirst()) * ld;
#pragma unroll
      for (int e = 0; e < 4; e++) v[d][e] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, off, at + e * ld, 0);
    }
  }
  // skip: how many k of the step are not its own
  __device__ __forceinline__ void store(unsigned char* s, int d, int skip, float& most) {
    if (__builtin_expect(skip != 0, 0)) {
      asm volatile("");  // (a branch: selects in every step cost more)
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (kfirst() + e < skip) v[d][e] = 0u;
    }
    const f32x4 x = __builtin_bit_cast(f32x4, v[d]);
    most = fmaxf(fmaxf(most, fabsf(x[0])), fabsf(x[1]));
    most = fmaxf(fmaxf(most, fabsf(x[2])), fabsf(x[3]));
    const MMParts a = mm_split(x[0], x[1]), b = mm_split(x[2], x[3]);
    unsigned char* at = s + row() * LD + kfirst() * 2;
#pragma unroll
    for (int i = 0; i < 3; i++) *reinterpret_cast<u32x2*>(at + 32 * i) = u32x2{a.p[i], b.p[i]};
  }
};

template <bool TA, bool TB, int WM, int WN, int TM, int TN>
__global__ __launch_bounds__(WM * WN * 64, TM * TN == 1 ? 4 : 2) void matmul_split_kernel(MMArgs a, int tiles, int tilesM, uint32_t inv_tiles, uint32_t inv_tilesM) {
  constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN, NT = WM * WN * 64;
  typedef MMSplitTile<BM, !TA, NT> SplitA;
  typedef MMSplitTile<BN, TB, NT> SplitB;
  typedef MMTile<float, BM, !TA, MM_ANY, NT> TileA;
  typedef MMTile<float, BN, TB, MM_ANY, NT> TileB;
  constexpr int BUF = SplitA::SIZE + SplitB::SIZE, F32 = (TileA::SIZE + TileB::SIZE) * 4;
  __shared__ __align__(16) unsigned char smem[2 * BUF > F32 ? 2 * BUF : F32];

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / WN, wn = wave % WN, r = lane & 31, h = lane >> 5;
  const int total = tiles * a.batch, b = mm_block();
  if (b >= total) return;  // (uniform)
  const int t = xcd_run(b, total), z = mm_div(t, tiles, inv_tiles), in = t - z * tiles;
  const int tn = mm_div(in, tilesM, inv_tilesM), n0 = tn * BN, m0 = (in - tn * tilesM) * BM;
  const float* A = reinterpret_cast<const float*>(a.A) + z * a.sA;
  const float* B = reinterpret_cast<const float*>(a.B) + z * a.sB;
  float* C = reinterpret_cast<float*>(a.C) + z * a.sC;

  mm_f32x16 acc[TM][TN];
  auto clear = [&](mm_f32x16 (&x)[TM][TN]) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) x[i][j][v] = 0.f;
  };
  clear(acc);
  float mostA = 0.f, mostB = 0.f;  // of the rows that this thread loads of
  {
    mm_f32x16 low[TM][TN];  // the products but x0 y0
    clear(low);
    SplitA ta;
    SplitB tb;
    ta.start(A, m0, a.M, a.K);
    tb.start(B, n0, a.N, a.K);
    const int steps = (a.K + 15) / 16;
    auto load = [&](int d, int step) {  // (past the last step: that one again)
      const int k = min(step * 16, a.K - 16);
      ta.load(d, k);
      tb.load(d, k);
    };
    auto store = [&](int d, int skip) {  // d = step % 2
      ta.store(smem + d * BUF, d, skip, mostA);
      tb.store(smem + d * BUF + SplitA::SIZE, d, skip, mostB);
    };
    const unsigned char *pa = smem + (wm * 32 * TM + r) * SplitA::LD + 16 * h, *pb = smem + SplitA::SIZE + (wn * 32 * TN + r) * SplitB::LD + 16 * h;
    auto skip = [&](int step) { return max(step * 16 + 16 - a.K, 0); };
    load(0, 0);
    load(1, 1);
    store(0, 0);
    load(0, 2);
    __syncthreads();
    // step s's tile is in LDS, steps s + 1 and s + 2 are on their way (past the end the last step again, which nothing reads)
    auto work = [&](int d, int step, int skip) {
      mm_bf16x8 fa[TM][3], fb[TN][3];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int u = 0; u < 3; ++u) fa[i][u] = *reinterpret_cast<const mm_bf16x8*>(pa + d * BUF + i * 32 * SplitA::LD + u * 32);
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int u = 0; u < 3; ++u) fb[j][u] = *reinterpret_cast<const mm_bf16x8*>(pb + d * BUF + j * 32 * SplitB::LD + u * 32);
      __builtin_amdgcn_sched_barrier(0);
      store(1 - d, skip);
      load(1 - d, step + 3);
      if constexpr (TM * TN == 1) __builtin_amdgcn_sched_barrier(0);
      auto mul = [&](mm_f32x16 (&to)[TM][TN], int u, int w) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) to[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][u], fb[j][w], to[i][j], 0, 0, 0);
      };
      mul(low, 2, 1), mul(acc, 0, 0), mul(low, 1, 2), mul(low, 2, 0), mul(low, 0, 2), mul(low, 1, 1), mul(low, 1, 0), mul(low, 0, 1);
      if constexpr (TM * TN > 1) {  // the splitting in the shadows of the matrix instructions
#pragma unroll
        for (int q = 0; q < 8 * TM * TN; q++) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x2, 3, 0);
        }
      }
      __syncthreads();
    };
    int step = 0;
    for (; step + 3 < steps; step += 2) work(0, step, 0), work(1, step + 1, 0);
#pragma unroll 1
    for (; step < steps; step += 2) {
      work(0, step, skip(step + 1));
      if (step + 1 < steps) work(1, step + 1, skip(step + 2));
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] += low[i][j][v];
  }
  // An infinity or a NaN in an operand, and a float that rounds to an infinity in bf16, leave a NaN here.  Parts below 2^-133 vanish: at most
  // 2^-103 of a product of operands below 2^30.  Results that are no numbers, of rows or columns with a larger operand, or between 0 and 2^-66 are
  // multiplied again with fp32 instructions; so are results of zero of a row and a column that are not all zeros, of which one has an element with parts that may be
  // below the normal bf16 numbers (below 2^-103: the sum may be zero because they vanished).  Every result is judged by its own row and column: what else its tile holds
  // does not change its bits.
  constexpr uint32_t LOW = (127u - 66u) << 24;
  auto twice = [](float f) { return (__float_as_uint(f) << 1) - 1u; };  // the magnitude's bits, less one: a zero is ~0u, 0 < |f| < 2^-66 below LOW - 1
  float check = 0.f;
  uint32_t least = ~0u, greatest = 0;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        check = fmaf(acc[i][j][v], 0.f, check);
        least = min(least, twice(acc[i][j][v])), greatest = max(greatest, twice(acc[i][j][v]));
      }
  const bool look = __syncthreads_or(check != 0.f || fmaxf(mostA, mostB) >= 0x1p30f || least < LOW - 1u || greatest == ~0u);
  {  // 32x32 accumulator layout as in mm_store; rows past the end lie past the end of the buffer
    const __amdgpu_buffer_rsrc_t rC = __builtin_amdgcn_make_buffer_rsrc(C, 0, (uint32_t)a.M * (uint32_t)a.N * 4u, 0x00020000);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + wn * 32 * TN + j * 32 + r;
      if (n < a.N) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const uint32_t at = ((uint32_t)(m0 + wm * 32 * TM + i * 32 + 4 * h) * (uint32_t)a.N + n) * 4u;
#pragma unroll
          for (int v = 0; v < 16; ++v)
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[i][j][v]), rC, at + (uint32_t)(8 * (v / 4) + v % 4) * (uint32_t)a.N * 4u, 0, 0);
        }
      }
    }
  }
  if (!look) return;

  enum : uint32_t { BIG = 1, SMALL = 2, NONZERO = 4 };
  uint32_t* flags = reinterpret_cast<uint32_t*>(smem);  // of the tile's rows of A, then of its columns of B
  for (int i = threadIdx.x; i < BM + BN; i += NT) flags[i] = 0u;
  __syncthreads();
  const int rowA = SplitA::row(), rowB = BM + SplitB::row();
  if (mostA > 0.f) atomicOr(&flags[rowA], mostA >= 0x1p30f ? BIG | NONZERO : NONZERO);
  if (mostB > 0.f) atomicOr(&flags[rowB], mostB >= 0x1p30f ? BIG | NONZERO : NONZERO);
  __syncthreads();
  // Small elements are looked for only where a result is zero though neither its row nor its column is: padded rows, caches not yet filled and
  // zero columns cost nothing, the look where zeros come of other elements 17 % of a tile (8 x 3108 x 128 x 777: dense 49 us, a zero row, column or
  // unfilled rows 49 to 52, other zeros in each tile 58).  Keeping the smallest element as well would cost the staging 1.5 instructions per element.
  bool open = false;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const uint32_t column = flags[BM + wn * 32 * TN + j * 32 + r];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) open |= acc[i][j][v] == 0.f && (column & flags[wm * 32 * TM + i * 32 + 8 * (v / 4) + 4 * h + v % 4] & NONZERO);
  }
  if (__syncthreads_or(open)) {
    SplitA ta;
    SplitB tb;
    ta.start(A, m0, a.M, a.K);
    tb.start(B, n0, a.N, a.K);
    constexpr int U = 4;  // K steps on their way at once
    uint32_t leastA = ~0u, leastB = ~0u;
    auto low = [&](uint32_t& l, u32x4 x) {
#pragma unroll
      for (int e = 0; e < 4; e++) l = min(l, (x[e] << 1) - 1u);
    };
#pragma unroll 1
    for (int k = 0; k < a.K; k += 16 * U) {
      u32x4 xa[U], xb[U];
#pragma unroll
      for (int u = 0; u < U; u++) {  // (past the end: the last 16 k again)
        ta.load(0, min(k + 16 * u, a.K - 16)), xa[u] = ta.v[0];
        tb.load(0, min(k + 16 * u, a.K - 16)), xb[u] = tb.v[0];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; u++) low(leastA, xa[u]), low(leastB, xb[u]);
    }
    constexpr uint32_t PARTS = (24u << 24) - 1u;  // |x| < 2^-103
    if (leastA < PARTS) atomicOr(&flags[rowA], SMALL);
    if (leastB < PARTS) atomicOr(&flags[rowB], SMALL);
    __syncthreads();
  }
  static_assert(TM * TN <= 2, "a bit per result of a lane");
  uint32_t wanted = 0;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const uint32_t column = flags[BM + wn * 32 * TN + j * 32 + r];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const uint32_t row = flags[wm * 32 * TM + i * 32 + 8 * (v / 4) + 4 * h + v % 4], either = row | column;
        const float f = acc[i][j][v];
        const bool w = !(fabsf(f) < __builtin_inff()) || (either & BIG) || twice(f) < LOW - 1u || (f == 0.f && (row & column & NONZERO) && (either & SMALL));
        wanted |= (uint32_t)w << (16 * (i * TN + j) + v);
      }
  }
  if (!__syncthreads_or(wanted != 0u)) return;

  // The next K step is loaded during this one's instructions, as in matmul_kernel; waves of which nothing is wanted multiply nothing.  8 x 3108 x 128 x
  // 777: one NaN row 81 us, a large or tiny row in every tile 102 (dense 49, fp32 instructions 61.5); a step loaded when it is needed: 109, 110.
  float *sA = reinterpret_cast<float*>(smem), *sB = sA + TileA::SIZE;
  TileA ta;
  TileB tb;
  clear(acc);
  ta.start(A, m0, a.M, a.K);
  tb.start(B, n0, a.N, a.K);
  ta.load(A, m0, 0, a.M, a.K);
  tb.load(B, n0, 0, a.N, a.K);
  const bool mine = __any(wanted != 0u);
#pragma unroll 1
  for (int k = 0; k < a.K; k += 32) {
    ta.store(sA);
    tb.store(sB);
    __syncthreads();
    if (k + 32 < a.K) {
      ta.load(A, m0, k + 32, a.M, a.K);
      tb.load(B, n0, k + 32, a.N, a.K);
    }
    if (mine) mm_f32_step<TileA, TileB, TM, TN>(sA, sB, wm, wn, r, h, acc);
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = m0 + wm * 32 * TM + i * 32 + 8 * (v / 4) + 4 * h + v % 4, n = n0 + wn * 32 * TN + j * 32 + r;
        if ((wanted >> (16 * (i * TN + j) + v) & 1) && m < a.M && n < a.N) C[(int64_t)m * a.N + n] = acc[i][j][v];
      }
}

// Up to four rows of A [M][K] against B [K][N] (attention probabilities x values of a decode token): a GEMV per row, bound by
// reading B once, which the tile kernel above walks with one workgroup per 64 columns and a K step at a time (32 heads x
// 8192 x 128 bf16: 158 us, 0.43 TB/s).  Here a workgroup of sixteen waves takes 2^lpr_log2 x VE columns (VE elements = 16
// bytes per lane); a lane takes four neighbouring k per pass, whose elements of A are one load per row (one load per element of A
// beside each load of B bound the kernel before: 8 x 4 x 8000 x 128 bf16 48.6 -> 20.9 us), the waves stride over K; fp32 sums per lane,
// then over the lanes of a column (wave shuffles), then over the waves in order through LDS.  Exact products, fp32 sums in
// another order than the tile kernel's.  The column blocks of a batch entry run on one XCD: they share the cache lines of B.
template <int DT>
__device__ __forceinline__ float mm_to_f32(typename MMElem<DT>::type e) {
  if constexpr (DT == MLLM_HIP_F32) return e;
  else if constexpr (DT == MLLM_HIP_BF16) return bf16_to_f32(e);
  else return f16bits_to_f32(e);
}
constexpr int MMR_WAVES = 16;
template <int DT, int MR>
__global__ __launch_bounds__(MMR_WAVES * 64) void matmul_rows_kernel(MMArgs a, int lpr_log2, int col_blocks, uint32_t inv_blocks) {
  using E = typename MMElem<DT>::type;
  constexpr int VE = 16 / (int)sizeof(E), UB = 4;
  typedef E AV __attribute__((ext_vector_type(UB)));
  extern __shared__ __align__(16) unsigned char mmr_smem[];
  float* s_part = reinterpret_cast<float*>(mmr_smem);  // [wave][row][column of the workgroup]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lpr = 1 << lpr_log2, rpw = 64 >> lpr_log2, ncols = lpr * VE;
  const int col = (lane & (lpr - 1)) * VE, sub = lane >> lpr_log2;
  const int total = col_blocks * a.batch;
  if (mm_block() >= total) return;  // (uniform)
  const int b = xcd_run(mm_block(), total), z = mm_div(b, col_blocks, inv_blocks), nb = (b - z * col_blocks) * ncols;
  const int n0 = nb + col, nc = min(n0, a.N - VE);  // (N % VE == 0: a lane's columns are all inside or all outside)
  const E* A = reinterpret_cast<const E*>(a.A) + z * a.sA;
  const E* B = reinterpret_cast<const E*>(a.B) + z * a.sB + nc;
  E* C = reinterpret_cast<E*>(a.C) + z * a.sC;
  const E* Am[MR];
#pragma unroll
  for (int m = 0; m < MR; m++) Am[m] = A + (int64_t)min(m, a.M - 1) * a.K;
  float acc[MR][VE];
#pragma unroll
  for (int m = 0; m < MR; m++)
#pragma unroll
    for (int j = 0; j < VE; j++) acc[m][j] = 0.f;
  auto mac = [&](u32x4 bv, int m, E e) {
    const float am = mm_to_f32<DT>(e);
#pragma unroll
    for (int j = 0; j < VE; j++) acc[m][j] = fmaf(am, mm_to_f32<DT>(MMTile<E, 64, true, MM_ANY>::elem(bv, j)), acc[m][j]);
  };
  const int kstep = MMR_WAVES * rpw * UB;
  int k = (wave * rpw + sub) * UB;
#pragma unroll 2
  for (; k + UB <= a.K; k += kstep) {
    u32x4 bv[UB];
    AV av[MR];
#pragma unroll
    for (int u = 0; u < UB; u++) bv[u] = *reinterpret_cast<const u32x4*>(B + (int64_t)(k + u) * a.N);
#pragma unroll
    for (int m = 0; m < MR; m++) __builtin_memcpy(&av[m], Am[m] + k, sizeof(AV));
#pragma unroll
    for (int u = 0; u < UB; u++)
#pragma unroll
      for (int m = 0; m < MR; m++) mac(bv[u], m, av[m][u]);
  }
  for (; k < a.K; k++) {  // one lane group of one wave ends here at most
    const u32x4 bv = *reinterpret_cast<const u32x4*>(B + (int64_t)k * a.N);
#pragma unroll
    for (int m = 0; m < MR; m++) mac(bv, m, Am[m][k]);
    if (k + 1 == a.K) break;
  }
#pragma unroll
  for (int m = 0; m < MR; m++)
#pragma unroll
    for (int j = 0; j < VE; j++) {
      float v = acc[m][j];
      for (int off = lpr; off < 64; off <<= 1) v += __shfl_xor(v, off, 64);
      if (sub == 0) s_part[((size_t)wave * MR + m) * ncols + col + j] = v;
    }
  __syncthreads();
  for (int i = tid; i < MR * ncols; i += MMR_WAVES * 64) {
    const int m = i / ncols, c = i - m * ncols, n = nb + c;
    if (m < a.M && n < a.N) {
      float f = 0.f;
#pragma unroll
      for (int w = 0; w < MMR_WAVES; w++) f += s_part[((size_t)w * MR + m) * ncols + c];
      if constexpr (DT == MLLM_HIP_F32) C[(int64_t)m * a.N + n] = f;
      else if constexpr (DT == MLLM_HIP_BF16) C[(int64_t)m * a.N + n] = f32_to_bf16(f);
      else C[(int64_t)m * a.N + n] = f32_to_f16bits(f);
    }
  }
}
// the launch shape of the kernel above; false where it does not apply (the tile kernel then)
template <int DT>
static bool launch_matmul_rows(const MMArgs& a, hipStream_t st, int* rc) {
  constexpr int VE = 16 / (int)sizeof(typename MMElem<DT>::type);
  if (a.M > 4 || !a.vecB || a.N % VE || a.K < 256) return false;
  int lg = 0;
  while (lg < 6 && (VE << lg) < a.N) lg++;
  // narrower column blocks while the launch has fewer than 128 workgroups, down to 64 bytes of a row per workgroup
  while (lg > 2 && (int64_t)a.batch * ((a.N + (VE << lg) - 1) / (VE << lg)) < 128) lg--;
  const int mr = a.M <= 1 ? 1 : (a.M <= 2 ? 2 : 4);
  while (lg > 0 && (size_t)MMR_WAVES * mr * (VE << lg) * sizeof(float) > 64 * 1024) lg--;  // the waves' partial sums fit 64 KB of LDS
  const int ncols = VE << lg;
  const int64_t cols = (a.N + ncols - 1) / ncols;
  if (cols * a.batch > 0x7fffffff) return false;
  const dim3 grid = mm_grid(cols * a.batch);
  const uint32_t inv = mm_inv(cols, cols * a.batch);
  const size_t lds = (size_t)MMR_WAVES * mr * ncols * sizeof(float);
  if (mr == 1) hipLaunchKernelGGL((matmul_rows_kernel<DT, 1>), grid, dim3(MMR_WAVES * 64), lds, st, a, lg, (int)cols, inv);
  else if (mr == 2) hipLaunchKernelGGL((matmul_rows_kernel<DT, 2>), grid, dim3(MMR_WAVES * 64), lds, st, a, lg, (int)cols, inv);
  else hipLaunchKernelGGL((matmul_rows_kernel<DT, 4>), grid, dim3(MMR_WAVES * 64), lds, st, a, lg, (int)cols, inv);
  *rc = (int)hipGetLastError();
  return true;
}

// Up to four rows of A [M][K] against B [N][K] (a decode token's queries x keys): dot products, bound by reading B once.  The tile
// kernel multiplies 64 rows for them, which in fp32 takes as long as the read.  A group of 2^g_log2 lanes holds 16-byte pieces of the
// rows of A and takes UB rows of B, all requested before the first is multiplied; the lanes' sums meet through wave shuffles.
// fp32: 8 x 4 x 8000 x 128 13.7 -> 9.8 us (3.3 TB/s), 8 x 1 x 8000 x 128 13.5 -> 5.5; bf16: 8 x 1 x 8000 x 128 5.6 -> 4.2.  1 x 1 x 64 x 2048 (router logits): fp32 52.6 -> 11.3,
// bf16 21.8 -> 5.4.
template <int DT, int MR, int UB>
__global__ __launch_bounds__(256) void matmul_dots_kernel(MMArgs a, int g_log2, int col_blocks, uint32_t inv_blocks) {
  using E = typename MMElem<DT>::type;
  constexpr int VE = 16 / (int)sizeof(E);
  __shared__ float s_out[MR][256 * UB / 4];  // at least four lanes per row of B
  const int tid = threadIdx.x, g = 1 << g_log2, sub = tid & (g - 1), groups = 256 >> g_log2, grp = tid >> g_log2, per = groups * UB;
  const int total = col_blocks * a.batch;
  if (mm_block() >= total) return;  // (uniform)
  const int b = xcd_run(mm_block(), total), z = mm_div(b, col_blocks, inv_blocks), n0 = (b - z * col_blocks) * per;
  const E* A = reinterpret_cast<const E*>(a.A) + z * a.sA;
  const E* B = reinterpret_cast<const E*>(a.B) + z * a.sB;
  E* C = reinterpret_cast<E*>(a.C) + z * a.sC;
  float acc[UB][MR];
#pragma unroll
  for (int u = 0; u < UB; u++)
#pragma unroll
    for (int m = 0; m < MR; m++) acc[u][m] = 0.f;
#pragma unroll UB == 1 ? 4 : 1
  for (int k = sub * VE; k < a.K; k += g * VE) {  // (K % VE == 0; once for rows of up to 64 pieces)
    u32x4 av[MR], bv[UB];
#pragma unroll
    for (int m = 0; m < MR; m++) av[m] = *reinterpret_cast<const u32x4*>(A + (int64_t)min(m, a.M - 1) * a.K + k);
#pragma unroll
    for (int u = 0; u < UB; u++) bv[u] = *reinterpret_cast<const u32x4*>(B + (int64_t)min(n0 + grp + u * groups, a.N - 1) * a.K + k);
#pragma unroll
    for (int u = 0; u < UB; u++)
#pragma unroll
      for (int j = 0; j < VE; j++) {
        const float bf = mm_to_f32<DT>(MMTile<E, 64, true, MM_ANY>::elem(bv[u], j));
#pragma unroll
        for (int m = 0; m < MR; m++) acc[u][m] = fmaf(mm_to_f32<DT>(MMTile<E, 64, true, MM_ANY>::elem(av[m], j)), bf, acc[u][m]);
      }
  }
#pragma unroll
  for (int u = 0; u < UB; u++)
#pragma unroll
    for (int m = 0; m < MR; m++) {
      float v = acc[u][m];
      v += dpp_f<0xB1>(v);  // (a group has four lanes or more)
      v += dpp_f<0x4E>(v);
      if (g > 4) v += dpp_f<0x141>(v);
      if (g > 8) v += dpp_f<0x140>(v);
      if (g > 16) v = sum16(v);
      if (g > 32) v = sum32(v);
      if (sub == 0) s_out[m][u * groups + grp] = v;
    }
  __syncthreads();
  for (int i = tid; i < MR * per; i += 256) {
    const int m = i / per, c = i - m * per;
    if (m < a.M && n0 + c < a.N) {
      const float f = s_out[m][c];
      if constexpr (DT == MLLM_HIP_F32) C[(int64_t)m * a.N + n0 + c] = f;
      else if constexpr (DT == MLLM_HIP_BF16) C[(int64_t)m * a.N + n0 + c] = f32_to_bf16(f);
      else C[(int64_t)m * a.N + n0 + c] = f32_to_f16bits(f);
    }
  }
}
// the launch shape of the kernel above; false where it does not apply (the tile kernel then: 16-bit operands with three or four
// short rows cost less there, 5.8 against 6.0 us at 8 x 4 x 8000 x 128; 1 x 4 x 64 x 2048: 18.7 / 6.0)
template <int DT>
static bool launch_matmul_dots(const MMArgs& a, hipStream_t st, int* rc) {
  constexpr int VE = 16 / (int)sizeof(typename MMElem<DT>::type);
  if (a.M > 4 || (a.M > 2 && DT != MLLM_HIP_F32 && a.K < 256) || !a.vecA || !a.vecB) return false;  // (aligned rows: K % VE == 0)
  int lg = 2;
  while (lg < 6 && (VE << lg) < a.K) lg++;
  if (((int64_t)a.N + 3) / 4 * a.batch > 0x7fffffff) return false;  // (a workgroup takes four rows of B at least)
  auto go = [&](auto kern, int ub) {
    const int per = (256 >> lg) * ub;
    const int64_t cols = ((int64_t)a.N + per - 1) / per;
    hipLaunchKernelGGL(kern, mm_grid(cols * a.batch), dim3(256), 0, st, a, lg, (int)cols, mm_inv(cols, cols * a.batch));
    return (int)hipGetLastError();
  };
  // four rows of B per group where that leaves 128 workgroups or more, else one (8 x 4 x 8000 x 128 fp32: 9.8 us / 13.1; 2 x 4 x
  // 777 x 128: 5.0 / 4.1)
  const int64_t per4 = (256 >> lg) * 4;
  if ((a.N + per4 - 1) / per4 * a.batch >= 128)
    *rc = a.M <= 1 ? go(matmul_dots_kernel<DT, 1, 4>, 4) : a.M <= 2 ? go(matmul_dots_kernel<DT, 2, 4>, 4) : go(matmul_dots_kernel<DT, 4, 4>, 4);
  else
    *rc = a.M <= 1 ? go(matmul_dots_kernel<DT, 1, 1>, 1) : a.M <= 2 ? go(matmul_dots_kernel<DT, 2, 1>, 1) : go(matmul_dots_kernel<DT, 4, 1>, 1);
  return true;
}

// The tile of 128 x 128 or of 64 x 64.  A wave of the larger one does four matrix instructions per pair of operand reads
// instead of one per pair, but fewer workgroups fit a CU and the last round and the edges of the output stay emptier.
//   fp32 (bound by the matrix pipe, two large tiles per CU at a time): rounds over the 256 CUs; 2048 x 4096 x 1000: 138 us large, 153
//     small; 3000 x 3000 x 3000 (2.25 rounds): 604 / 527; K = 64 is mostly epilogue: 4 x 4000 x 1000 x 64: 34 / 31
//   16 bits (bound by loads and LDS, more workgroups per CU hide them): us of a K of 2048 against tiles per CU, B [N][K]: 4096 x 4096 x 4096
//     180 large, 298 small, 1000 x 3000 x 700: 24 / 20; where an operand is [K][rows] the large tile gains less (4096^3: 340 / 371)
static int g_matmul_tile = 0;   // mllm_hip_matmul_set_tile
static int g_matmul_split = 0;  // mllm_hip_matmul_set_split
template <int DT, bool TA, bool TB>
static bool matmul_large_tile(const MMArgs& a) {
  if (g_matmul_tile) return g_matmul_tile == 128;
  const double large = (double)((a.M + 127) / 128) * ((a.N + 127) / 128) * a.batch / 256;
  const double small = (double)((a.M + 63) / 64) * ((a.N + 63) / 64) * a.batch / 256;
  if (DT == MLLM_HIP_F32) return a.K >= 128 && 4. * std::ceil(large) < 1.13 * std::ceil(small);
  if (a.K < 256) return false;
  return !TA && TB ? 30. + 17. * large < 9. + 9.3 * small : 40. + 36. * large < 11.7 * small;
}

// A short product all of whose vectors lie inside K and the rows, or outside K, as a whole (whatever the alignment in memory).  From K =
// 512 on the two are even (1000 x 1000 x 1000 bf16 17.1 / 17.1 us, fp32 26.4 / 26.4 to 27.4); whole K steps gain 0.1 to 0.3 us of a
// launch (64 x 128 x 128 x 128 bf16 4.44 -> 4.21) and nothing in many rounds (fp32 8 x 3108 x 777 x 128: 58.4 / 59.8).
template <int DT, bool TA, bool TB>
static bool mm_vectors(const MMArgs& a) {
  constexpr bool f32 = DT == MLLM_HIP_F32;
  if (a.K >= 512 || (a.K % 32 == 0 && (double)((a.M + 63) / 64) * ((a.N + 63) / 64) * a.batch > 1024)) return false;
  auto fits = [&](bool contig_k, int rows) { return contig_k ? a.K % (f32 ? 4 : 8) == 0 : rows % 4 == 0 && (f32 || a.K % 2 == 0); };
  return fits(!TA, a.M) && fits(TB, a.N);
}

// Few rows of A against many of B, fp32 [M][K] x [N][K]: the tile's other rows would repeat A's last one through the L1, whose requests are
// what such a product waits for when it fills the chip.  us, repeated / left out: 33 x 12 x 2732 x 1080 171 / 146, 48 x 8 x 2840 x 624 127 /
// 113, 16 x 20 x 3148 x 692 (800 tiles) 59.1 / 56.8; with fewer tiles the branch costs more (10 x 20 x 920 x 432, 150 tiles: 12.6 / 13.3),
// in the other orders and in 16 bits up to 1.6 times as much.
template <int DT, bool TA, bool TB>
static bool mm_narrow(const MMArgs& a) {
  return DT == MLLM_HIP_F32 && !TA && TB && a.M <= 32 && (int64_t)((a.N + 63) / 64) * a.batch >= 800;
}

// fp32: the side of the tile of matmul_split_kernel, 0 where fp32 instructions are as fast or needed.  Costs in us of the three forms fitted to 4800
// random shapes in all orders (1 to 64 x 5 to 4096 x 5 to 4096 x 16 to 2048, a third of them attention of 64 to 1024 tokens), those of the large tile
// again to 900 of more than one small tile per CU: the choice takes 0.864 of the fp32 instructions' time on average over those, the best of the three 0.859 (0.879
// before the large tile's splitting moved).  Large tiles whose edges cover more than 1.2 of what small ones do cost 6 % more than that (42 x 157 x 721 x 1301 130 us on
// small ones, 151), and the fp32 instructions no less than for 48 from 33 on (17 x 382 x 515 x 35 10.9 us, 8.4 from parts): over 2372 shapes near the limits 0.970 of the time of the
// choice before those two costs and that move, 45 more than 3 % slower, up to 10 % (60, up to 18 %, without).  A gain of less than 4 % in the costs stays with
// fp32 instructions, and so do K below 32 (59 x 397 x 1677 x 24: 45.4 us, 57 with parts) and up to one small tile per CU, where the order decides
// and tiles do not (1 x 1701 x 245 x 1964 with A [K][M] 74 / 56, 8 x 20 x 168 x 1765 42 / 50).  With costs of the parts alone every launch
// above a floor took them, and the large tile too early: 8 x 504 x 504 x 128 9.4 / 12.2 us, 8 x 1308 x 327 x 64 11.2 / 16.1.  Few rows x
// [N][K] over many tiles stay with the form for those.
static int mm_split_side(const MMArgs& a, bool nt) {
  constexpr int64_t LIMIT = (int64_t)1 << 32;  // byte offsets in 32 bits
  if (a.K < 16 || (int64_t)a.M * a.K * 4 >= LIMIT || (int64_t)a.N * a.K * 4 >= LIMIT || ((int64_t)a.M + 128) * a.N * 4 >= LIMIT) return 0;
  if (g_matmul_split) return g_matmul_split < 0 ? 0 : g_matmul_split;
  if (g_matmul_tile) return 0;
  if (nt && mm_narrow<MLLM_HIP_F32, false, true>(a)) return 0;
  const double K = a.K, t64 = (double)((a.M + 63) / 64) * ((a.N + 63) / 64) * a.batch / 256, t128 = (double)((a.M + 127) / 128) * ((a.N + 127) / 128) * a.batch / 256;
  if (t64 <= 1. || a.K < 32) return 0;
  const double steps = a.K > 32 ? std::max(K, 48.) : K;  // the fp32 instructions' tiles take K in steps of 32: 33 elements cost as many as 48
  const double pad = (double)((a.M + 127) / 128 * 2) * ((a.N + 127) / 128 * 2) / ((double)((a.M + 63) / 64) * ((a.N + 63) / 64));  // large tiles' area over small ones'
  const double us64 = 3.6 + 0.80 * t64 + K * (0.0225 + 0.0152 * (0.49 * std::ceil(t64) + 0.51 * t64 - 1.));
  const double us128 = (2.14 + 6.02 * std::max(t128, 1.) + K * (0.0384 + 0.0503 * (std::ceil(t128) - 1.))) * (pad > 1.2 ? 1.06 : 1.);
  const double f32 = 3.06 + 0.869 * t64 + steps * (0.024 + 0.020 * (0.93 * std::ceil(t64) + 0.07 * t64 - 1.));
  if (std::min(us64, us128) > 0.96 * f32) return 0;
  return us128 < us64 ? 128 : 64;
}

template <int DT, bool TA, bool TB>
static int launch_matmul(const MMArgs& a, hipStream_t st) {
  if constexpr (!TA && !TB) {
    int rc = 0;
    if (launch_matmul_rows<DT>(a, st, &rc)) return rc;
  }
  if constexpr (!TA && TB) {
    int rc = 0;
    if (launch_matmul_dots<DT>(a, st, &rc)) return rc;
  }
  auto run = [&](auto kern, int bm, int bn, int threads) {
    const int64_t tilesM = (a.M + bm - 1) / bm, tiles = tilesM * ((a.N + bn - 1) / bn);
    if (tiles > 0x7fffffff) return MLLM_HIP_E_SHAPE;
    const int most = (int)std::min<int64_t>(a.batch, 0x7fffffff / tiles);  // batch entries per launch
    using E = typename MMElem<DT>::type;
    for (int z = 0; z < a.batch; z += most) {
      MMArgs p = a;
      p.A = reinterpret_cast<const E*>(a.A) + z * a.sA;
      p.B = reinterpret_cast<const E*>(a.B) + z * a.sB;
      p.C = reinterpret_cast<E*>(a.C) + z * a.sC;
      p.batch = std::min(most, a.batch - z);
      hipLaunchKernelGGL(kern, mm_grid(tiles * p.batch), dim3(threads), 0, st, p, (int)tiles, (int)tilesM, mm_inv(tiles, tiles * p.batch), mm_inv(tilesM, tiles));
    }
    return (int)hipGetLastError();
  };
  auto go = [&](auto kern, int side) { return run(kern, side, side, 256); };
  if constexpr (DT == MLLM_HIP_F32) {
    switch (mm_split_side(a, !TA && TB)) {
      case 64: return run(matmul_split_kernel<TA, TB, 2, 2, 1, 1>, 64, 64, 256);
      case 128: return run(matmul_split_kernel<TA, TB, 4, 2, 1, 2>, 128, 128, 512);
    }
  }
  if (matmul_large_tile<DT, TA, TB>(a)) return go(matmul_kernel<DT, TA, TB, 2, 2, MM_ANY>, 128);
  if constexpr (DT == MLLM_HIP_F32 && !TA && TB) {
    if (a.K > 32 && mm_narrow<DT, TA, TB>(a)) return go(matmul_kernel<DT, TA, TB, 1, 1, MM_NARROW>, 64);
  }
  if (mm_vectors<DT, TA, TB>(a)) return go(matmul_kernel<DT, TA, TB, 1, 1, MM_VECTORS>, 64);
  if (a.K <= 32) return go(matmul_kernel<DT, TA, TB, 1, 1, MM_STEP>, 64);
  return go(matmul_kernel<DT, TA, TB, 1, 1, MM_ANY>, 64);
}

template <int DT>
static int launch_matmul_t(const MMArgs& a, int ta, int tb, hipStream_t st) {
  if (ta && tb) return launch_matmul<DT, true, true>(a, st);
  if (ta) return launch_matmul<DT, true, false>(a, st);
  if (tb) return launch_matmul<DT, false, true>(a, st);
  return launch_matmul<DT, false, false>(a, st);
}

}  // namespace mllmhip

using namespace mllmhip;

MLLM_API int mllm_hip_matmul_batched(const void* A, const void* B, void* C, int dtype, int64_t batch, int64_t M, int64_t N,
                                     int64_t K, int64_t stride_a, int64_t stride_b, int64_t stride_c, int transpose_a,
                                     int transpose_b, void* stream) {
  if (!A || !B || !C || M <= 0 || N <= 0 || K <= 0 || batch <= 0 || stride_a < 0 || stride_b < 0 || stride_c < 0)
    return MLLM_HIP_E_BADARG;
  if (dtype != MLLM_HIP_F32 && dtype != MLLM_HIP_BF16 && dtype != MLLM_HIP_F16) return MLLM_HIP_E_BADARG;
  if (M > INT32_MAX || N > INT32_MAX || K > INT32_MAX || batch > INT32_MAX) return MLLM_HIP_E_SHAPE;
  if ((M + 63) / 64 > 65535) return MLLM_HIP_E_SHAPE;
  if (batch > 1 && stride_c < M * N) return MLLM_HIP_E_SHAPE;  // outputs of different batch entries must not overlap
  const int es = dtype == MLLM_HIP_F32 ? 4 : 2;
  if (reinterpret_cast<uintptr_t>(A) % es || reinterpret_cast<uintptr_t>(B) % es || reinterpret_cast<uintptr_t>(C) % es)
    return MLLM_HIP_E_ALIGN;
  const int ve = 16 / es;
  auto vec_ok = [&](const void* p, int64_t ld, int64_t stride) {
    return reinterpret_cast<uintptr_t>(p) % 16 == 0 && ld % ve == 0 && (batch == 1 || stride % ve == 0);
  };
  MMArgs a{A, B, C, (int)M, (int)N, (int)K, (int)batch, stride_a, stride_b, stride_c,
           vec_ok(A, transpose_a ? M : K, stride_a) ? 1 : 0, vec_ok(B, transpose_b ? K : N, stride_b) ? 1 : 0};
  hipStream_t st = (hipStream_t)stream;
  switch (dtype) {
    case MLLM_HIP_F32: return launch_matmul_t<MLLM_HIP_F32>(a, transpose_a, transpose_b, st);
    case MLLM_HIP_BF16: return launch_matmul_t<MLLM_HIP_BF16>(a, transpose_a, transpose_b, st);
    default: return launch_matmul_t<MLLM_HIP_F16>(a, transpose_a, transpose_b, st);
  }
}

MLLM_API int mllm_hip_matmul_set_tile(int side) {
  if (side != 0 && side != 64 && side != 128) return MLLM_HIP_E_BADARG;
  g_matmul_tile = side;
  return 0;
}

MLLM_API int mllm_hip_matmul_set_split(int side) {
  if (side != -1 && side != 0 && side != 64 && side != 128) return MLLM_HIP_E_BADARG;
  g_matmul_split = side;
  return 0;
}

MLLM_API int mllm_hip_matmul_split_side(int64_t batch, int64_t M, int64_t N, int64_t K, int transpose_a, int transpose_b) {
  if (batch < 1 || M < 1 || N < 1 || K < 1 || batch > INT32_MAX || M > INT32_MAX || N > INT32_MAX || K > INT32_MAX) return 0;
  MMArgs a{};
  a.batch = (int)batch, a.M = (int)M, a.N = (int)N, a.K = (int)K;
  return mm_split_side(a, !transpose_a && transpose_b);
}

MLLM_API int mllm_hip_matmul_f32(const float* A, const float* B, float* C, int64_t M, int64_t N, int64_t K, int transpose_a,
                                 int transpose_b, void* stream) {
  return mllm_hip_matmul_batched(A, B, C, MLLM_HIP_F32, 1, M, N, K, 0, 0, 0, transpose_a, transpose_b, stream);
}

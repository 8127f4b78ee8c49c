// Block-quantized GEMM for many activation rows on gfx950, and the MoE expert FFN built on it.
//
//   y[row][n] = sum_b fp32(dW[n][b] * dX[row][b]) * int32(sum_32 qW * qX)       (every Linear of the reference's CPU path)
//
// Reference semantics:
//   expert loop           mllm/models/qwen3_moe/modeling_qwen3_moe_fa2.hpp:175-238 (moeInfer), :98-100 (Qwen3MoeMLP)
//   each Linear           mllm/backends/cpu/kernels/common/ggml/matmul.cpp:148-206 (Q8_0 activations, block dots)
//   SiLU                  mllm/backends/cpu/kernels/x86/silu.cpp:16-27   x * (1 / (1 + exp_poly(-x))), math.hpp:19-72
// The per-block int32 sums come from v_mfma_i32_32x32x32_i8 (K = 32 = one quantization block per instruction, exact);
// they are scaled and accumulated in fp32 on the vector ALU.  Tokens are the MFMA rows, weight rows the MFMA columns, so
// a lane owns one output channel: its weight scale is a scalar per block and stores are contiguous across lanes.
#include "qgemv_kernel.h"
#include "qgemm_layout.h"
#include "kquant_layout.h"
#include "wk_gemm.h"

namespace mllmhip {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int TOK_TILE = 64;    // activation rows per workgroup tile (2 MFMA row tiles)
constexpr int TT = TOK_TILE / 32;
constexpr int KCH = 8;          // blocks per K chunk staged in LDS

// ---------------------------------------------------------------------------------------------------------
// routing: histogram, offsets, expert-sorted order and the tile list, one workgroup
// ---------------------------------------------------------------------------------------------------------
struct RouteOut {
  int* counts;       // [E]
  int* offsets;      // [E + 1]
  int* sorted_idx;   // [T*k]  flat index t*k + j of the entry at each expert-sorted position
  int* tile_expert;  // [max_tiles]
  int* tile_row0;    // [max_tiles]  first sorted position of the tile
  int* tile_rows;    // [max_tiles]  rows in the tile (<= TOK_TILE)
  int* ntiles;       // [1]
};

// GROUPED: an expert's tiles are neighbours in the list (full tiles, then its partial tile), the experts in the order of
// their numbers; otherwise all full tiles come first.  (Measured and dropped for the grouped list: experts in order of
// falling row counts, so that the short tiles end a launch: 4 % slower on 512 tokens x 8 of 128 experts -- the heavy
// experts' tiles are bound by arithmetic and the light ones by memory, and a list that mixes them overlaps the two.)
template <bool GROUPED = false>
__device__ __forceinline__ void moe_route_body(const int32_t* __restrict__ ids, int n, int E, int tile_h, const RouteOut& o, int* s_cnt) {
  // s_cnt: [E] counts, [E] cursors, [E] scan scratch x 3
  int* s_cur = s_cnt + E;
  int* s_off = s_cur + E;   // exclusive scan of the counts
  int* s_full = s_off + E;  // exclusive scan of the full-tile counts
  int* s_part = s_full + E; // exclusive scan of the partial-tile flags
  __shared__ int s_tot[3];
  for (int e = threadIdx.x; e < E; e += blockDim.x) s_cnt[e] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const int e = ids[i];
    if (e >= 0 && e < E) atomicAdd(&s_cnt[e], 1);
  }
  __syncthreads();
  // three exclusive scans over the experts, one wave each (E is at most a few thousand: 64 experts per step)
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (wave < 3) {
    int* dst = wave == 0 ? s_off : wave == 1 ? s_full : s_part;
    int run = 0;
    for (int base = 0; base < E; base += 64) {
      const int e = base + lane;
      const int c = e < E ? s_cnt[e] : 0;
      const int v = wave == 0 ? c : wave == 1 ? c / tile_h : (c % tile_h != 0);
      int incl = v;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int t = __shfl_up(incl, d, 64);
        if (lane >= d) incl += t;
      }
      if (e < E) dst[e] = run + incl - v;
      run += __shfl(incl, 63, 64);
    }
    if (lane == 0) s_tot[wave] = run;
  }
  __syncthreads();
  // tile list, full tiles first so that the long-running workgroups start early (GROUPED: expert by expert)
  for (int e = threadIdx.x; e < E; e += blockDim.x) {
    const int c = s_cnt[e], base = s_off[e];
    o.counts[e] = c;
    o.offsets[e] = base;
    s_cur[e] = base;
    const int nf = c / tile_h;
    for (int t = 0; t < nf; t++) {
      const int slot = s_full[e] + t + (GROUPED ? s_part[e] : 0);
      o.tile_expert[slot] = e;
      o.tile_row0[slot] = base + t * tile_h;
      o.tile_rows[slot] = tile_h;
    }
    if (c % tile_h) {
      const int slot = GROUPED ? s_full[e] + nf + s_part[e] : s_tot[1] + s_part[e];
      o.tile_expert[slot] = e;
      o.tile_row0[slot] = base + nf * tile_h;
      o.tile_rows[slot] = c % tile_h;
    }
  }
  if (threadIdx.x == 0) {
    o.offsets[E] = s_tot[0];
    o.ntiles[0] = s_tot[1] + s_tot[2];
  }
  __syncthreads();
  // the order inside an expert does not matter: every row is computed independently of its neighbours
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const int e = ids[i];
    if (e >= 0 && e < E) o.sorted_idx[atomicAdd(&s_cur[e], 1)] = i;
  }
}

__global__ __launch_bounds__(1024) void moe_route_kernel(const int32_t* __restrict__ ids, int n, int E, int tile_h, RouteOut o) {
  extern __shared__ int s_route[];
  moe_route_body(ids, n, E, tile_h, o, s_route);
}

// identity routing for a plain Linear over M rows
__global__ void identity_tiles_kernel(int M, int tile_h, RouteOut o) {
  const int nt = (M + tile_h - 1) / tile_h;
  for (int t = threadIdx.x; t < nt; t += blockDim.x) {
    o.tile_expert[t] = 0;
    o.tile_row0[t] = t * tile_h;
    o.tile_rows[t] = min(tile_h, M - t * tile_h);
  }
  if (threadIdx.x == 0) o.ntiles[0] = nt;
}

// The routing pass keeps five int arrays of E entries in LDS: E is limited to what fits the 64 KB a launch gets without
// raising the kernel's dynamic-LDS attribute.  The launch status is read before anything that consumes the tile list is
// queued: a consumer must never walk a list the routing pass did not write.
constexpr int MOE_MAX_EXPERTS = 3072;
static int launch_route(const int32_t* ids, int64_t entries, int E, int tile_h, const RouteOut& ro, hipStream_t st) {
  if (E <= 0 || E > MOE_MAX_EXPERTS) return MLLM_HIP_E_SHAPE;
  hipLaunchKernelGGL(moe_route_kernel, dim3(1), dim3(1024), 5 * (size_t)E * sizeof(int), st, ids, (int)entries, E, tile_h, ro);
  return (int)hipGetLastError();
}
static int launch_identity_tiles(int64_t M, int tile_h, const RouteOut& ro, hipStream_t st) {
  hipLaunchKernelGGL(identity_tiles_kernel, dim3(1), dim3(256), 0, st, (int)M, tile_h, ro);
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------------
// Q8_0 activation quantization to codes + the fp32 scale that takes part in the arithmetic
// (quantize_row_q8_0, AVX2 branch, ggml/quantize/quantize_q8.cpp:106-190)
// ---------------------------------------------------------------------------------------------------------
__global__ void quant_rows_kernel(const void* __restrict__ x, int x_dtype, int8_t* __restrict__ codes,
                                  float* __restrict__ deff, int64_t nblocks, int x86_scale) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nblocks) return;
  float v[32];
  uint32_t q[8];
  int sum;
  load_block_f32(x, x_dtype, i * QK, v);
  uint16_t bits = quantize_block_q8_0(v, q, sum);
  if (x86_scale) bits = x86_scale_bits(bits);
  deff[i] = f16bits_to_f32(bits);
  u32x4* out = reinterpret_cast<u32x4*>(codes + i * QK);
  out[0] = u32x4{q[0], q[1], q[2], q[3]};
  out[1] = u32x4{q[4], q[5], q[6], q[7]};
}

// ---------------------------------------------------------------------------------------------------------
// the tile kernel
// ---------------------------------------------------------------------------------------------------------
struct QGemmArgs {
  const char* W0;        // packed weights of matrix 0 (gate, or the only matrix), expert e at W0 + e * wstride
  const char* W1;        // packed weights of matrix 1 (up) for the fused gate/up mode
  size_t wstride;
  const int8_t* aq;      // activation codes  [rows][K]
  const float* ad;       // activation scales [rows][K/32]
  const int* a_index;    // activation row of each sorted position is a_index[pos] / a_div ; null: the position itself
  int a_div;
  int a_rows;            // rows of aq
  const int* o_index;    // output row of each sorted position (null: the position itself)
  float* out;            // fp32 [..][N]   (plain / down mode)
  const float* bias;     // [N] or null    (plain mode)
  int8_t* hq;            // gate/up mode: int8 codes of silu(g)*u  [rows][N]
  float* hd;             // gate/up mode: their scales              [rows][N/32]
  const int* tile_expert;
  const int* tile_row0;
  const int* tile_rows;
  const int* ntiles;
  int N, K;
  int x86_scale;
};

// weight codes of one block for the lane's output channel as signed int8: lanes 0..31 supply elements 0..15, lanes 32..63
// elements 16..31 (Q4_0: low / high nibbles of the same 16 bytes; Q8_0: first / second code plane).
template <int WT>
__device__ __forceinline__ v4i weight_operand(const u32x4& q, int hi) {
  if (WT == MLLM_HIP_Q4_0) {
    const uint32_t sh = hi ? 4u : 0u;
    const uint32_t d[4] = {q.x, q.y, q.z, q.w};
    v4i r;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint32_t nib = (d[j] >> sh) & 0x0f0f0f0fu;                    // bytes 0..15
      r[j] = (int)(((nib | 0x80808080u) - 0x08080808u) ^ 0x80808080u);    // per-byte (v - 8), no borrow between bytes
    }
    return r;
  } else {
    return v4i{(int)q.x, (int)q.y, (int)q.z, (int)q.w};
  }
}

// the SiLU operator runs over whole [rows, I] tensors with I a multiple of 32: always the vector form
__device__ __forceinline__ float silu_f(float x) { return x * (1.0f / (1.0f + exp_poly(-x))); }

constexpr int PLANE = TOK_TILE * 16 + 16;          // LDS bytes of one (block, half) plane of activation codes, padded
constexpr int SA_BYTES = KCH * 2 * PLANE;
constexpr int SDX_BYTES = KCH * TOK_TILE * 4;
constexpr int SU_LD = 128 + 4;                     // row stride (floats) of the up -> gate hand-over tile
constexpr int SU_BYTES = TOK_TILE * SU_LD * 4;

// Workgroup tile: up to TOK_TILE activation rows x 128 output channels; a wave owns 32 channels (one MFMA column tile) and
// all 32-row tiles.  K is walked in chunks of 8 blocks:
//   * the rows' int8 codes (128 x 256 B) and fp32 scales of the chunk are staged in LDS once per workgroup, laid out as
//     [block][half][row] 16-byte words so that operand reads of neighbouring rows are neighbouring words;
//   * each lane keeps its channel's 8 weight blocks and 8 scales of the chunk in registers;
//   * the next chunk's global loads (activations and weights) are in flight while the current chunk is computed.
// MODE 0: one weight matrix, out[o_index[pos]][n] = acc (+ bias).
// MODE 1: eight waves; waves 0..3 run the gate matrix, waves 4..7 the up matrix over the same channels; the up
//         accumulators are handed over through LDS and the gate waves emit h = silu(g) * u quantized to Q8_0 (the 32
//         channels of a wave are exactly one block of the next Linear's input).
template <int WT, int MODE>
__global__ __launch_bounds__(MODE == 1 ? 512 : 256) void qgemm_tile_kernel(QGemmArgs a) {
  constexpr int NT = MODE == 1 ? 512 : 256;
  constexpr int UA = TOK_TILE * 16 / NT;  // 16-byte activation words per thread and chunk
  extern __shared__ __align__(16) unsigned char smem[];
  unsigned char* sA = smem;
  float* sDx = reinterpret_cast<float*>(smem + SA_BYTES);
  float* sU = reinterpret_cast<float*>(smem);  // MODE 1 hand-over tile, reuses the staging area after the last chunk

  const int tile = blockIdx.x;
  if (tile >= min(a.ntiles[0], (int)gridDim.x)) return;
  const int e = a.tile_expert[tile], row0 = a.tile_row0[tile], rows = a.tile_rows[tile];
  const int ntt = (rows + 31) >> 5;
  const int last_njg = (rows - 32 * (ntt - 1) + 7) >> 3;  // 8-row groups in the last 32-row tile
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lrow = lane & 31, hi = lane >> 5;
  const int nb = a.K / QK, nbp = (int)scale_row_stride(a.K);
  const int mat = MODE == 1 ? (wave >> 2) : 0;
  const int nt = blockIdx.y * 4 + (wave & 3);  // this wave's tile of 32 output channels
  const bool nvalid = nt * 32 < a.N;
  const int n = min(nt * 32 + lrow, a.N - 1);

  const PackedView w = packed_view(WT, (mat ? a.W1 : a.W0) + (size_t)e * a.wstride, a.N, a.K);
  const u32x4* wq = (WT == MLLM_HIP_Q8_0 && hi) ? w.q1 : w.q0;

  const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(a.aq), 0, (uint32_t)((int64_t)a.a_rows * a.K), 0x00020000);
  const __amdgpu_buffer_rsrc_t rD = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.ad), 0, (uint32_t)((int64_t)a.a_rows * nb * 4), 0x00020000);

  // staging assignment: word u = tid + i*NT of the chunk -> row u/16, 16-byte column u%16 (= block*2 + half)
  uint32_t abase[UA];
#pragma unroll
  for (int i = 0; i < UA; i++) {
    const int u = tid + i * NT, p = u >> 4;
    uint32_t off = 0xffffffffu;
    if (p < rows) {
      const int r = a.a_index ? a.a_index[row0 + p] / a.a_div : row0 + p;
      off = (uint32_t)((int64_t)r * a.K + (u & 15) * 16);
    }
    abase[i] = off;
  }
  // scales: thread t < 2*TOK_TILE -> row t/2, blocks (t%2)*4 .. +4 of the chunk
  uint32_t dbase = 0xffffffffu;
  if (tid < 2 * TOK_TILE && (tid >> 1) < rows) {
    const int p = tid >> 1;
    const int r = a.a_index ? a.a_index[row0 + p] / a.a_div : row0 + p;
    dbase = (uint32_t)(((int64_t)r * nb + (tid & 1) * 4) * 4);
  }

  u32x4 pa[UA];
  float pd[4];
  u32x4 bq[KCH], bqn[KCH], bs, bsn;
  auto gload_act = [&](int b0) {
#pragma unroll
    for (int i = 0; i < UA; i++) {
      const int blk = ((tid + i * NT) & 15) >> 1;
      const bool ok = abase[i] != 0xffffffffu && b0 + blk < nb;
      pa[i] = __builtin_amdgcn_raw_buffer_load_b128(rA, ok ? abase[i] + (uint32_t)b0 * QK : 0xffffffffu, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const bool ok = dbase != 0xffffffffu && b0 + (tid & 1) * 4 + j < nb;
      pd[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rD, ok ? dbase + (uint32_t)(b0 + j) * 4 : 0xffffffffu, 0, 0));
    }
  };
  auto sstore_act = [&]() {
#pragma unroll
    for (int i = 0; i < UA; i++) {
      const int u = tid + i * NT;
      *reinterpret_cast<u32x4*>(sA + (u & 15) * PLANE + (u >> 4) * 16) = pa[i];
    }
    if (tid < 2 * TOK_TILE) {
#pragma unroll
      for (int j = 0; j < 4; j++) sDx[((tid & 1) * 4 + j) * TOK_TILE + (tid >> 1)] = pd[j];
    }
  };
  auto gload_w = [&](int b0, u32x4 (&q)[KCH], u32x4& sc) {
#pragma unroll
    for (int k = 0; k < KCH; k++) q[k] = wq[(int64_t)n * nb + min(b0 + k, nb - 1)];
    sc = *reinterpret_cast<const u32x4*>(w.d + (int64_t)n * nbp + min(b0, nbp - KCH));
  };

  float acc[TT][16];
#pragma unroll
  for (int tt = 0; tt < TT; tt++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[tt][r] = 0.f;

  gload_act(0);
  gload_w(0, bq, bs);
  sstore_act();
  __syncthreads();

  for (int b0 = 0; b0 < nb; b0 += KCH) {
    // the next chunk's loads are issued unconditionally (past the end they are clamped or out of range and unused): a
    // branch around them would leave the number of loads in flight unknown and force a full wait before the MFMAs
    const bool more = b0 + KCH < nb;
    gload_act(b0 + KCH);
    gload_w(b0 + KCH, bqn, bsn);
    if (nvalid) {
      const uint32_t sw[4] = {bs.x, bs.y, bs.z, bs.w};
#pragma unroll
      for (int k = 0; k < KCH; k++) {
        if (b0 + k < nb) {
          const v4i fb = weight_operand<WT>(bq[k], hi);
          const float dw = f16bits_to_f32((uint16_t)(sw[k >> 1] >> (16 * (k & 1))));
#pragma unroll
          for (int tt = 0; tt < TT; tt++) {
            if (tt < ntt) {
              const v4i fa = *reinterpret_cast<const v4i*>(sA + (k * 2 + hi) * PLANE + (tt * 32 + lrow) * 16);
              v16i z;
#pragma unroll
              for (int r = 0; r < 16; r++) z[r] = 0;
              const v16i is = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa, fb, z, 0, 0, 0);
              const int njg = (tt == ntt - 1) ? last_njg : 4;
              // accumulator register r of lane l: row 8*(r/4) + 4*(l/32) + r%4, column l%32
#pragma unroll
              for (int j = 0; j < 4; j++) {
                if (j < njg) {
                  const f32x4 dx = *reinterpret_cast<const f32x4*>(&sDx[k * TOK_TILE + tt * 32 + 8 * j + 4 * hi]);
#pragma unroll
                  for (int i = 0; i < 4; i++) acc[tt][4 * j + i] = fmaf(dw * dx[i], (float)is[4 * j + i], acc[tt][4 * j + i]);
                }
              }
            }
          }
        }
      }
    }
    __syncthreads();  // every wave is done with the staged chunk
    if (more) {
      sstore_act();
#pragma unroll
      for (int k = 0; k < KCH; k++) bq[k] = bqn[k];
      bs = bsn;
    }
    __syncthreads();
  }

  if (MODE == 1) {
    // up waves hand their accumulators to the gate waves of the same channels (the staging area is free now)
    if (mat == 1 && nvalid) {
#pragma unroll
      for (int tt = 0; tt < TT; tt++)
        if (tt < ntt)
#pragma unroll
          for (int r = 0; r < 16; r++)
            sU[(tt * 32 + 8 * (r / 4) + 4 * hi + (r % 4)) * SU_LD + (wave & 3) * 32 + lrow] = acc[tt][r];
    }
    __syncthreads();
    if (mat == 1 || !nvalid) return;
#pragma unroll
    for (int tt = 0; tt < TT; tt++) {
      if (tt >= ntt) continue;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int p = tt * 32 + 8 * (r / 4) + 4 * hi + (r % 4);  // row within the tile, same for the 32 lanes of a half
        const float h = silu_f(acc[tt][r]) * sU[p * SU_LD + (wave & 3) * 32 + lrow];
        float amax = fabsf(h);
        amax = fmaxf(amax, dpp_f<0xB1>(amax));
        amax = fmaxf(amax, dpp_f<0x4E>(amax));
        amax = fmaxf(amax, dpp_f<0x141>(amax));
        amax = fmaxf(amax, dpp_f<0x140>(amax));
        amax = max16(amax);
        const float d = amax / 127.f;
        const float idv = (amax != 0.f) ? 127.f / amax : 0.f;
        int qi = (int)rintf(h * idv);
        qi = min(127, max(-128, qi));
        if (p < rows) {
          a.hq[(int64_t)(row0 + p) * a.N + n] = (int8_t)qi;
          if (lrow == 0) {
            uint16_t bits = f32_to_f16bits(d);
            if (a.x86_scale) bits = x86_scale_bits(bits);
            a.hd[(int64_t)(row0 + p) * (a.N / QK) + nt] = f16bits_to_f32(bits);
          }
        }
      }
    }
  } else {
    if (!nvalid) return;
#pragma unroll
    for (int tt = 0; tt < TT; tt++) {
      if (tt >= ntt) continue;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int p = tt * 32 + 8 * (r / 4) + 4 * hi + (r % 4);
        if (p < rows && nt * 32 + lrow < a.N) {
          const int64_t orow = a.o_index ? a.o_index[row0 + p] : row0 + p;
          float v = acc[tt][r];
          if (a.bias) v = a.bias[n] + v;
          a.out[orow * a.N + n] = v;
        }
      }
    }
  }
}

// =========================================================================================================
// Matrix-core path for many rows: fp16 operands with the block scales folded in
//
//   y[row][n] = sum_k xh[row][k] * wh[n][k],   xh = fp16(dX * qX) (the Q8_0 round trip of the activations, exact product
//   rounded once to fp16), wh = fp16(dW * qW) (likewise), fp32 accumulation in v_mfma_f32_32x32x16_f16.
//
// The block-dot form above needs three vector-ALU operations per (row, channel, block) to scale and add the int32 block
// sums, which bounds it far below the matrix rate.  Folding the scales into 16-bit operands moves that work to the
// operands: about two operations per WEIGHT element per 32*TM rows, nothing per accumulator.  Both roundings are to 11
// significant bits (relative error <= 2^-12 each), which keeps the result within about 3e-4 relative L2 of the
// reference's fp32 block arithmetic.  |dX*qX| and |dW*qW| must stay below 65504 (fp16).
//
// Weight layout ("gemm-packed", mllm_hip_q_gemm_prepack): codes in v_mfma_*_32x32x16 operand order, N padded to 32 rows
// and K to 128 elements with zero blocks;
//   Q4_0  q  [N/32][K/64][64 lanes][16 B]: lane l = (row l%32, half l/32); dword d of its 16 bytes holds the eight
//            elements k = 64 kb + 16 d + 8 (l/32) + 0..7: element 2i in nibble i, element 2i+1 in nibble 4+i (so that
//            (dword >> 4i) & 0x000f000f is the pair (2i, 2i+1) in the two halves of a register)
//   Q8_0  q  [N/32][K/64][2][64 lanes][16 B]: plane p holds d = 2p, 2p+1; each d is two dwords of four codes in byte
//            order e0, e2, e1, e3
//   scales   [N/32][K/64][32 rows] dwords: fp16 scale of block 2kb | fp16 scale of block 2kb+1 << 16, after the
//            weight_scale_mode decoding
// Kernel structure as the W4A16 weights-from-global kernel: four waves side by side along N, activations via LDS,
// weights straight from global memory two K steps ahead, dequantized one MFMA step ahead in the shadows of the MFMAs.
// =========================================================================================================
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));


// one output dword of the code area per thread
template <int WT>
__global__ __launch_bounds__(256) void qg_prepack_q_kernel(const unsigned char* __restrict__ blocks, uint32_t* __restrict__ P,
                                                           int N, int K, int64_t words) {
  const int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (w >= words) return;
  const int kbs = (int)(qg_kp(K) / 64), nblk = K / QK;
  constexpr int BS = WT == MLLM_HIP_Q4_0 ? 18 : 34;
  uint32_t v = 0;
  if (WT == MLLM_HIP_Q4_0) {
    const int d = (int)(w % 4), l = (int)((w / 4) % 64);
    const int64_t blk = w / 256;
    const int kb = (int)(blk % kbs), nb = (int)(blk / kbs);
    const int n = nb * 32 + (l & 31), k0 = kb * 64 + d * 16 + (l >> 5) * 8;
    if (n < N && k0 < K) {
      const unsigned char* qs = blocks + ((int64_t)n * nblk + k0 / QK) * BS + 2;
      const int o = k0 % QK;  // 0, 8, 16, 24: elements o..o+7 are the low (o < 16) or high nibbles of qs[o % 16 ..]
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const uint32_t byte = qs[(o & 15) + i];
        const uint32_t e = o < 16 ? (byte & 15u) : (byte >> 4);
        v |= e << (4 * ((i >> 1) + 4 * (i & 1)));
      }
    }
  } else {
    const int x = (int)(w % 4), l = (int)((w / 4) % 64), pl = (int)((w / 256) % 2);
    const int64_t blk = w / 512;
    const int kb = (int)(blk % kbs), nb = (int)(blk / kbs);
    const int d = 2 * pl + x / 2;
    const int n = nb * 32 + (l & 31), k0 = kb * 64 + d * 16 + (l >> 5) * 8 + 4 * (x % 2);
    if (n < N && k0 < K) {
      const unsigned char* qs = blocks + ((int64_t)n * nblk + k0 / QK) * BS + 2 + k0 % QK;
      v = (uint32_t)qs[0] | ((uint32_t)qs[2] << 8) | ((uint32_t)qs[1] << 16) | ((uint32_t)qs[3] << 24);
    }
  }
  P[w] = v;
}
template <int WT>
__global__ __launch_bounds__(256) void qg_prepack_s_kernel(const unsigned char* __restrict__ blocks, uint32_t* __restrict__ S,
                                                           int N, int K, int x86_scale, int64_t count) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // (nb, kb, row)
  if (i >= count) return;
  const int kbs = (int)(qg_kp(K) / 64), nblk = K / QK;
  constexpr int BS = WT == MLLM_HIP_Q4_0 ? 18 : 34;
  const int row = (int)(i % 32), kb = (int)((i / 32) % kbs), nb = (int)(i / 32 / kbs);
  const int n = nb * 32 + row;
  uint32_t v = 0;
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int b = 2 * kb + h;
    if (n < N && b < nblk) {
      const unsigned char* p = blocks + ((int64_t)n * nblk + b) * BS;
      uint16_t bits = (uint16_t)(p[0] | (p[1] << 8));
      if (x86_scale) {  // as mllm_hip_q_prepack: the field holds the pattern as a half-precision NUMBER
        const float num = f16bits_to_f32(bits);
        bits = (num >= 0.f && num < 65536.f) ? (uint16_t)(uint32_t)num : (uint16_t)0;
      }
      v |= (uint32_t)bits << (16 * h);
    }
  }
  S[i] = v;
}

// activations: Q8_0 quantization (bit-exact codes and scale) and back to fp16 in one pass, eight elements per thread (four lanes of a
// block), so that a wave reads and writes whole cache lines: 2048 x 2560 bf16 7.1 us with a block per thread, 6.1 this way
// (xl, when asked for: the rounding residual dX*qX - xh, exact in fp16, for the two-term gate/up path)
__global__ __launch_bounds__(256) void qg_act_kernel(const void* __restrict__ x, int x_dtype, uint16_t* __restrict__ xh, uint16_t* __restrict__ xl,
                                                     int64_t nblocks, int x86_scale) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // whole blocks only: the four lanes of a block are here or not together
  if (i >= nblocks * 4) return;
  float v[8];
  if (x_dtype == MLLM_HIP_F32) {
    const f32x4* p = reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(x) + i * 8);
    const f32x4 a = p[0], b = p[1];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      v[e] = a[e];
      v[4 + e] = b[e];
    }
  } else {
    const u32x4 r = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(x) + i * 8);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      v[2 * e] = __uint_as_float(r[e] << 16);
      v[2 * e + 1] = __uint_as_float(r[e] & 0xffff0000u);
    }
  }
  float amax = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(v[e]));
  amax = fmaxf(amax, dpp_f<0xB1>(amax));
  amax = fmaxf(amax, dpp_f<0x4E>(amax));
  const float id = (amax != 0.f) ? 127.f / amax : 0.f;
  uint16_t bits = f32_to_f16bits(amax / 127.f);
  if (x86_scale) bits = x86_scale_bits(bits);
  const float d = f16bits_to_f32(bits);
  uint32_t o[4], ol[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const float a = d * (float)min(127, max(-128, (int)rintf(v[2 * j] * id)));  // exact in fp32: 11 x 8 bits
    const float b = d * (float)min(127, max(-128, (int)rintf(v[2 * j + 1] * id)));
    const uint16_t ha = f32_to_f16bits(a), hb = f32_to_f16bits(b);
    o[j] = (uint32_t)ha | ((uint32_t)hb << 16);
    ol[j] = (uint32_t)f32_to_f16bits(a - f16bits_to_f32(ha)) | ((uint32_t)f32_to_f16bits(b - f16bits_to_f32(hb)) << 16);
  }
  *reinterpret_cast<u32x4*>(xh + i * 8) = u32x4{o[0], o[1], o[2], o[3]};
  if (xl) *reinterpret_cast<u32x4*>(xl + i * 8) = u32x4{ol[0], ol[1], ol[2], ol[3]};
}

struct QG2Args {
  const char* W0;        // gemm-packed weights of matrix 0 (gate, or the only matrix), expert e at W0 + e * wstride
  const char* W1;        // gemm-packed weights of matrix 1 (up) in the fused gate/up mode
  size_t wstride;
  const uint16_t* xh;    // fp16 activations [a_rows][K]
  const uint16_t* xl;    // their rounding residuals, same shape (two-term mode only)
  const int* a_index;    // activation row of sorted position pos is a_index[pos] / a_div ; null: pos itself
  int a_div;
  int a_rows;
  const int* o_index;    // output row of sorted position pos (null: pos itself)
  float* out;            // fp32 [..][N]       (one-matrix mode)
  const float* bias;     // [N] or null        (one-matrix mode)
  uint16_t* hh;          // gate/up mode: fp16 Q8_0 round trip of silu(g)*u, [rows][N]
  const int* tile_expert;
  const int* tile_row0;
  const int* tile_rows;
  const int* ntiles;
  int N, K;
  int wtype;
  int x86_scale;
  int ksplit;            // one-matrix mode: K is cut into this many ranges (blockIdx.z), each writing its own partial result
  float* partial;        // [ksplit][a_rows][N] when ksplit > 1
  int halves;            // a plain Linear: workgroups of eight waves, each four of them half of K
  int big_cols;          // a plain Linear (no tile list): column tiles that run as full-height tiles
};

// the scale of dword d (K elements 16 d .. 16 d + 15 of a 64-element step) in both halves; for Q4_K also the offset
template <int WT>
__device__ __forceinline__ f16x2 qg_scale2(const uint32_t (&s)[qg_scale_dwords(WT)], int d) {
  uint32_t h;
  if constexpr (WT == MLLM_HIP_Q6_K) {
    const uint32_t v = s[d >> 1];
    h = (d & 1) ? (v >> 16) : (v & 0xffffu);
  } else {
    h = d < 2 ? (s[0] & 0xffffu) : (s[0] >> 16);
  }
  return __builtin_bit_cast(f16x2, h | (h << 16));
}
template <int WT>
__device__ __forceinline__ f16x2 qg_offset2(const uint32_t (&s)[qg_scale_dwords(WT)], int d) {
  const uint32_t v = s[qg_scale_dwords(WT) - 1], h = d < 2 ? (v & 0xffffu) : (v >> 16);
  return __builtin_bit_cast(f16x2, h | (h << 16));
}

// (w & mask) | base in one instruction
__device__ __forceinline__ uint32_t qg_under(uint32_t w, uint32_t mask, uint32_t base) {
  return (uint32_t)__builtin_amdgcn_bitop3_b32((int)w, (int)mask, (int)base, 0xea);
}
// pair `b` (elements 2b, 2b+1) of the eight weights of one MFMA step, scaled: one dword of two fp16.  With PREC == 2 also
// the rounding residual of the product (exact: the error of a product of two fp16 numbers is an fp16 number).
// Q4_K: the sub-block's value is ds * q - dm (q = 0..15): one fused multiply-add, one rounding; Q6_K: codes widened to
// int8 at load time, ds the scale of the step's 16 elements: the Q8_0 arithmetic.
// Nibbles at bits 4 b + 0..3 go into the mantissa of 1024 (b even) or as they are into that of 64 (b odd), one shift for two of the four
// pairs; bytes are put under the mantissa of 1024 by a permutation.  Clocks of a wave per instruction, four waves per SIMD: 2.3 for a shift, an and / or / xor,
// 2.5 for three-input logic, 4.2 for a permutation, packed fp16 and conversions: mask and exponent in one instruction take 2.5 instead of 4.6 (bytes
// by a shift and three-input logic instead of the permutation: no faster).  In a graph, three shifts and and / or on bytes / one shift, permutations, us: 2048 x 9728 x 2560
// Q6_K 119.3 / 117.7, Q4_0 115.9 / 113.0; 131 x 2560 x 9728 Q6_K 28.3 / 25.9, Q8_0 27.7 / 25.4, Q4_0 26.0 / 25.0, Q4_K 25.4 / 24.4.  And, or / three-input logic, Q4_0:
// 111 x 5376 x 4736 21.7 / 20.3, 531 x 4144 x 2848 32.9 / 31.8, 2048 x 9728 x 2560 (bound by the matrix pipe at the clock that it holds) 117.2 / 115.0.
template <int WT, int PREC>
__device__ __forceinline__ uint32_t qg_pair(const u32x4 (&rq)[qg_nibbles(WT) ? 1 : 2], int d, int b, f16x2 dd, f16x2 dm, uint32_t& lo) {
  uint32_t t;
  float off;
  if (qg_nibbles(WT)) {
    const uint32_t w = b < 2 ? rq[0][d] : rq[0][d] >> 8;
    t = b & 1 ? qg_under(w, 0x00f000f0u, 0x54005400u) : qg_under(w, 0x000f000fu, 0x64006400u);  // 64 + q or 1024 + q in both halves
    off = b & 1 ? 64.f : 1024.f;
    if (WT == MLLM_HIP_Q4_0) off += 8.f;
  } else {
    const uint32_t w = rq[d >> 1][2 * (d & 1) + (b >> 1)] ^ 0x80808080u;  // codes + 128, bytes e0 e2 e1 e3
    t = __builtin_amdgcn_perm(0x64646464u, w, b & 1 ? 0x04030401u : 0x04020400u);
    off = 1152.f;
  }
  const f16x2 c = __builtin_bit_cast(f16x2, t) - f16x2{(_Float16)off, (_Float16)off};  // v_pk_add_f16: the code, exact
  if (WT == MLLM_HIP_Q4_K) {
    static_assert(WT != MLLM_HIP_Q4_K || PREC == 1, "one-term operands only");
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(c, dd, -dm));  // v_pk_fma_f16
  }
  const f16x2 r = c * dd;                                          // v_pk_mul_f16: one rounding
  if (PREC == 2) lo = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(c, dd, -r));  // v_pk_fma_f16
  return __builtin_bit_cast(uint32_t, r);
}

// One tile: `rows` (<= 32 TM) sorted positions from row0 x 128 TN channels from n0, NW weight matrices (1, or gate + up).
// PREC == 2 carries both operands as fp16 value + fp16 residual and adds the two first-order cross terms
// (wh*xh + wl*xh + wh*xl): the operands are then exact and the result is the fp32 sum of exact products.  The gate/up
// stage needs it: its output is re-quantized to Q8_0, and a relative perturbation eps of the values in front of that
// rounding step flips codes often enough to come out as about sqrt(eps/40) in relative L2.
// G == 2 (one matrix): eight waves, the second four take the second half of K with a stage of their own; their sums join the first
// four's through LDS.
template <int WT, int NW, int TM, int TN, int PREC, int G = 1>
__device__ __forceinline__ void qg_tile(const QG2Args& a, const int e, const int row0, const int rows, const int n0,
                                        unsigned char* smem_all) {
  constexpr int BK = 64, LDK = 2 * BK + 16, KS = BK / 16;
  constexpr int BM = TM * 32, WN = TN * 32;
  constexpr int CA = TM;  // 16-byte activation chunks per thread and K step: 32 TM rows x 8 chunks over 256 threads
  constexpr int STAGE = PREC * BM * LDK;  // value rows, then residual rows
  constexpr int QW = qg_nibbles(WT) ? 1 : 2;
  constexpr int SDW = qg_scale_dwords(WT);

  static_assert(G == 1 || NW == 1, "halves of K: one matrix");
  const int group = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  unsigned char* const smem = smem_all + group * 2 * STAGE;
  const int tid = G == 1 ? threadIdx.x : threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
  const int lrow = lane & 31, hi = lane >> 5;
  const int Kp = (int)qg_kp(a.K), kbs = Kp / 64, nbs = (int)(qg_np(a.N) / 32);
  const int64_t qbytes = qg_qbytes(WT, a.N, a.K), wbytes = qg_bytes(WT, a.N, a.K);

  const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.xh), 0, (uint32_t)((int64_t)a.a_rows * a.K * 2), 0x00020000);
  __amdgpu_buffer_rsrc_t rW[NW];
  rW[0] = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(a.W0 + (size_t)e * a.wstride), 0, (uint32_t)wbytes, 0x00020000);
  if (NW == 2) rW[NW - 1] = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(a.W1 + (size_t)e * a.wstride), 0, (uint32_t)wbytes, 0x00020000);

  // activation chunk c of a thread: tile row (tid + 256 c) / 8, 16-byte column (tid + 256 c) % 8.  Rows past `rows` repeat
  // the last one (never stored); columns past K read as zeros so that the zero-padded weight tail meets no other row.
  uint32_t offA[CA];
  const int colA = (tid % 8) * 8;
#pragma unroll
  for (int c = 0; c < CA; c++) {
    const int pos = row0 + min((tid + c * 256) / 8, rows - 1);
    const int arow = a.a_index ? a.a_index[pos] / a.a_div : pos;
    offA[c] = (uint32_t)(((int64_t)arow * a.K + colA) * 2);
  }
  uint32_t offQ[TN], offS[TN];
#pragma unroll
  for (int j = 0; j < TN; j++) {
    const int nb = min((n0 + wave * WN) / 32 + j, nbs - 1);
    offQ[j] = (uint32_t)((int64_t)nb * kbs * (1024 * QW) + lane * 16);
    offS[j] = (uint32_t)(qbytes + ((int64_t)nb * kbs * 32 + lrow) * 4 * SDW);
  }
  const __amdgpu_buffer_rsrc_t rAl = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(PREC == 2 ? a.xl : a.xh), 0, (uint32_t)((int64_t)a.a_rows * a.K * 2), 0x00020000);
  auto loadA = [&](int k0, u32x4 (&ga)[PREC][CA]) {
    const bool ok = k0 + colA < a.K;
#pragma unroll
    for (int c = 0; c < CA; c++) {
      ga[0][c] = __builtin_amdgcn_raw_buffer_load_b128(rA, ok ? offA[c] : 0xffffffffu, k0 * 2, 0);
      if (PREC == 2) ga[PREC - 1][c] = __builtin_amdgcn_raw_buffer_load_b128(rAl, ok ? offA[c] : 0xffffffffu, k0 * 2, 0);
    }
  };
  auto storeA = [&](int buf, const u32x4 (&ga)[PREC][CA]) {
#pragma unroll
    for (int p = 0; p < PREC; p++)
#pragma unroll
      for (int c = 0; c < CA; c++) {
        const int idx = tid + c * 256;
        *reinterpret_cast<u32x4*>(smem + buf * STAGE + (p * BM + idx / 8) * LDK + (idx % 8) * 16) = ga[p][c];
      }
  };
  auto readA = [&](int buf, int ks, f16x8 (&fa)[PREC][TM]) {
#pragma unroll
    for (int p = 0; p < PREC; p++)
#pragma unroll
      for (int i = 0; i < TM; i++)
        fa[p][i] = *reinterpret_cast<const f16x8*>(smem + buf * STAGE + (p * BM + i * 32 + lrow) * LDK + ks * 32 + hi * 16);
  };

  v16f acc[NW][TN][TM];
#pragma unroll
  for (int w = 0; w < NW; w++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[w][j][i][r] = 0.f;

  u32x4 ga[PREC][CA];
  u32x4 rq[2][NW][TN][QW];      // packed codes of K steps kt (set kt & 1) and kt + 1
  uint32_t rs[2][NW][TN][SDW];  // their scale records
  f16x8 fb[2][NW][TN][PREC];    // dequantized operands of MFMA step ks (set ks & 1): value, residual
  f16x8 fa[2][PREC][TM];
  auto loadS = [&](uint32_t (&r)[SDW], int w, int j, int kb) {
    if (SDW == 1) {
      r[0] = __builtin_amdgcn_raw_buffer_load_b32(rW[w], offS[j], kb * 128, 0);
    } else {
      const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rW[w], offS[j], kb * 256, 0);
      r[0] = v.x;
      r[SDW - 1] = v.y;
    }
  };
  auto loadW = [&](int set, int kb) {
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
      for (int j = 0; j < TN; j++) {
#pragma unroll
        for (int p = 0; p < QW; p++) rq[set][w][j][p] = __builtin_amdgcn_raw_buffer_load_b128(rW[w], offQ[j], (kb * QW + p) * 1024, 0);
        loadS(rs[set][w][j], w, j, kb);
      }
  };
  // K range of these waves: all of it or (short batches, one matrix) range blockIdx.z of a.ksplit, written to its own partial result, and
  // of that one of the G halves; the ranges and halves start at even K steps
  int kt0 = 0, kt1 = Kp / BK, idle = 0;  // even
  float* outp = a.out;
  const float* biasp = a.bias;
  if (NW == 1 && a.ksplit > 1) {
    const int per = ((kt1 + a.ksplit - 1) / a.ksplit + 1) / 2 * 2;
    kt0 = (int)blockIdx.z * per;
    kt1 = min(kt1, kt0 + per);
    outp = a.partial + (size_t)blockIdx.z * a.a_rows * a.N;
    biasp = nullptr;
  }
  if (G == 2) {
    const int per = ((kt1 - kt0) / 2 + 1) / 2 * 2, all = kt1;
    kt0 += group * per;
    kt1 = min(all, kt0 + per);
    idle = per - (kt1 - kt0);
  }
  loadA(kt0 * BK, ga);
  loadW(0, kt0);
  loadW(1, kt0 + 1);
  storeA(0, ga);
  __syncthreads();
  readA(0, 0, fa[0]);
#pragma unroll
  for (int w = 0; w < NW; w++)
#pragma unroll
    for (int j = 0; j < TN; j++) {
      const f16x2 dd = qg_scale2<WT>(rs[0][w][j], 0), dm = qg_offset2<WT>(rs[0][w][j], 0);
      uint32_t o[4], ol[4] = {0, 0, 0, 0};
#pragma unroll
      for (int b = 0; b < 4; b++) o[b] = qg_pair<WT, PREC>(rq[0][w][j], 0, b, dd, dm, ol[b]);
      fb[0][w][j][0] = __builtin_bit_cast(f16x8, u32x4{o[0], o[1], o[2], o[3]});
      if (PREC == 2) fb[0][w][j][PREC - 1] = __builtin_bit_cast(f16x8, u32x4{ol[0], ol[1], ol[2], ol[3]});
    }

  // one K step (64 elements) with its weights in register set CUR; refills that set with K step kt + 2 when done with it
  auto kstep = [&](auto cur_tag, int kt) {
    constexpr int CUR = decltype(cur_tag)::value;
    const int buf = kt & 1;
    loadA((kt + 1) * BK, ga);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      if (ks < KS - 1) {
        readA(buf, ks + 1, fa[(ks + 1) & 1]);  // the next step's activations while this one's MFMAs run
      } else {
        storeA(buf ^ 1, ga);
        __syncthreads();
        readA(buf ^ 1, 0, fa[(ks + 1) & 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
      const int ns = ks < KS - 1 ? CUR : CUR ^ 1, nd = (ks + 1) % KS;  // register set and dword of the NEXT step's weights
#pragma unroll
      for (int w = 0; w < NW; w++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
          // the dequantization of the next step's operand is cut into TM pieces, one pinned into the shadow of each MFMA
          const f16x2 dd = qg_scale2<WT>(rs[ns][w][j], nd), dm = qg_offset2<WT>(rs[ns][w][j], nd);
          uint32_t o[4], ol[4] = {0, 0, 0, 0};
#pragma unroll
          for (int i = 0; i < TM; i++) {
            acc[w][j][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[ks & 1][w][j][0], fa[ks & 1][0][i], acc[w][j][i], 0, 0, 0);
            if (PREC == 2) {
              acc[w][j][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[ks & 1][w][j][PREC - 1], fa[ks & 1][0][i], acc[w][j][i], 0, 0, 0);
              acc[w][j][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[ks & 1][w][j][0], fa[ks & 1][PREC - 1][i], acc[w][j][i], 0, 0, 0);
            }
#pragma unroll
            for (int b = i * 4 / TM; b < (i + 1) * 4 / TM; b++) o[b] = qg_pair<WT, PREC>(rq[ns][w][j], nd, b, dd, dm, ol[b]);
            __builtin_amdgcn_sched_barrier(0);
          }
          fb[(ks + 1) & 1][w][j][0] = __builtin_bit_cast(f16x8, u32x4{o[0], o[1], o[2], o[3]});
          if (PREC == 2) fb[(ks + 1) & 1][w][j][PREC - 1] = __builtin_bit_cast(f16x8, u32x4{ol[0], ol[1], ol[2], ol[3]});
          if (ks == KS - 2) {  // the set's last dword is consumed: fetch K step kt + 2 into it
#pragma unroll
            for (int p = 0; p < QW; p++)
              rq[CUR][w][j][p] = __builtin_amdgcn_raw_buffer_load_b128(rW[w], offQ[j], ((kt + 2) * QW + p) * 1024, 0);
            loadS(rs[CUR][w][j], w, j, kt + 2);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
    }
  };
  for (int kt = kt0; kt < kt1; kt += 2) {
    kstep(std::integral_constant<int, 0>{}, kt);
    kstep(std::integral_constant<int, 1>{}, kt + 1);
  }
  for (int i = 0; i < idle; i++) __syncthreads();  // the barriers of the steps the other half of K still has
  __syncthreads();
  if (G == 2) {
    f32x4* part = reinterpret_cast<f32x4*>(smem_all);
    if (group == 1) {
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int g = 0; g < 4; g++)
            part[(((wave * TN + j) * TM + i) * 4 + g) * 64 + lane] = f32x4{acc[0][j][i][4 * g], acc[0][j][i][4 * g + 1], acc[0][j][i][4 * g + 2], acc[0][j][i][4 * g + 3]};
    }
    __syncthreads();
    if (group == 0) {
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int g = 0; g < 4; g++) {
            const f32x4 v = part[(((wave * TN + j) * TM + i) * 4 + g) * 64 + lane];
#pragma unroll
            for (int q = 0; q < 4; q++) acc[0][j][i][4 * g + q] += v[q];
          }
    }
    __syncthreads();
  }

  // acc[w][j][i][4g+e] = result[row0 + 32i + lrow][n0 + wave*WN + 32j + 8g + 4hi + e]
  if (NW == 1 && a.N % 4 == 0) {
    // each 32-row slab is turned through LDS so that a wave stores whole rows of the workgroup's columns, 16 bytes per lane (a lane's
    // own quads lie in 32 different rows: 2048 x 9728 x 2560 128 -> 125 us)
    constexpr int BN = 4 * WN, ROWB = 4 * BN + 16, QPR = BN / 4;  // QPR: 16-byte pieces per row
    constexpr int RPW = 8 / G;                                    // rows per wave
    static_assert(RPW * QPR % 64 == 0, "a wave stores whole rows");
    const int wall = group * 4 + wave;
#pragma unroll
    for (int i = 0; i < TM; i++) {
      if (group == 0) {
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int g = 0; g < 4; g++)
            *reinterpret_cast<f32x4*>(smem_all + lrow * ROWB + (wave * WN + j * 32 + 8 * g + 4 * hi) * 4) =
                f32x4{acc[0][j][i][4 * g], acc[0][j][i][4 * g + 1], acc[0][j][i][4 * g + 2], acc[0][j][i][4 * g + 3]};
      }
      __syncthreads();
      const int q = lane % QPR, n = n0 + 4 * q;
      f32x4 bi = {0.f, 0.f, 0.f, 0.f};
      if (biasp && n < a.N) bi = *reinterpret_cast<const f32x4*>(biasp + n);
#pragma unroll
      for (int t = 0; t < RPW * QPR / 64; t++) {
        const int rl = wall * RPW + t * (64 / QPR) + lane / QPR, r = i * 32 + rl;
        f32x4 v = *reinterpret_cast<const f32x4*>(smem_all + rl * ROWB + q * 16);
        if (biasp) v += bi;
        if (r < rows && n < a.N) {
          const int pos = row0 + r;
          *reinterpret_cast<f32x4*>(outp + (int64_t)(a.o_index ? a.o_index[pos] : pos) * a.N + n) = v;
        }
      }
      if (i + 1 < TM) __syncthreads();
    }
  } else if (NW == 1) {
#pragma unroll
    for (int i = 0; i < TM; i++) {
      const int r = i * 32 + lrow;
      if (r < rows && group == 0) {
        const int pos = row0 + r;
        float* orow = outp + (int64_t)(a.o_index ? a.o_index[pos] : pos) * a.N;
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int q = 0; q < 16; q++) {
            const int n = n0 + wave * WN + j * 32 + 8 * (q / 4) + 4 * hi + q % 4;
            if (n < a.N) orow[n] = biasp ? acc[0][j][i][q] + biasp[n] : acc[0][j][i][q];
          }
      }
    }
  } else {
    // h = silu(gate) * up, Q8_0 round trip over each block of 32 channels (a block is one column tile j: 16 channels in
    // this lane, 16 in lane ^ 32), written as fp16 for the next Linear
#pragma unroll
    for (int i = 0; i < TM; i++) {
      const int r = i * 32 + lrow;
#pragma unroll
      for (int j = 0; j < TN; j++) {
        float h[16];
        float amax = 0.f;
#pragma unroll
        for (int q = 0; q < 16; q++) {
          h[q] = silu_f(acc[0][j][i][q]) * acc[NW - 1][j][i][q];
          amax = fmaxf(amax, fabsf(h[q]));
        }
        amax = max32(amax);
        const float d = amax / 127.f;
        const float idv = (amax != 0.f) ? 127.f / amax : 0.f;
        uint16_t bits = f32_to_f16bits(d);
        if (a.x86_scale) bits = x86_scale_bits(bits);
        const float deff = f16bits_to_f32(bits);
        if (r < rows) {
          uint16_t* hrow = a.hh + (int64_t)(row0 + r) * a.N;
#pragma unroll
          for (int g = 0; g < 4; g++) {
            const int n = n0 + wave * WN + j * 32 + 8 * g + 4 * hi;
            uint32_t o[2];
#pragma unroll
            for (int e2 = 0; e2 < 2; e2++) {
              const int q0 = min(127, max(-128, (int)rintf(h[4 * g + 2 * e2] * idv)));
              const int q1 = min(127, max(-128, (int)rintf(h[4 * g + 2 * e2 + 1] * idv)));
              o[e2] = (uint32_t)f32_to_f16bits(deff * (float)q0) | ((uint32_t)f32_to_f16bits(deff * (float)q1) << 16);
            }
            if (n + 3 < a.N) *reinterpret_cast<uint2*>(hrow + n) = uint2{o[0], o[1]};
          }
        }
      }
    }
  }
}

constexpr int QG_TILE_H = 128;
constexpr int QG_SLOTS = 512;  // tiles in flight: two workgroups on each of 256 CUs

// MODE 0: one matrix, 128 x 256 tiles, one-term operands.  MODE 1: gate and up together with two-term operands; a tile of
// the list is cut into halves of 64 rows (blockIdx.z) x 128 channels.
// The tile height follows the rows the tile really has: short tiles skip the MFMAs of empty row blocks.
template <int WT, int MODE, int G = 1>
__global__ __launch_bounds__(256 * G) __attribute__((amdgpu_waves_per_eu(2, 2))) void qg_kernel(QG2Args a) {
  extern __shared__ __align__(16) unsigned char smem[];
  int e, row0, rows, n0 = blockIdx.y * (MODE == 1 ? 128 : 256);
  if (MODE == 1 || a.ntiles) {
    const int t = blockIdx.x;
    if (t >= min(a.ntiles[0], (int)gridDim.x)) return;
    e = a.tile_expert[t];
    row0 = a.tile_row0[t];
    rows = a.tile_rows[t];
  } else {
    // A plain Linear.  The column tiles behind big_cols run as half-height tiles, which are the first workgroups of the grid: the
    // full-height tiles fill whole rounds of the chip, and short tiles share their CUs with full ones.
    const int tilesM = (a.a_rows + QG_TILE_H - 1) / QG_TILE_H, tilesH = (a.a_rows + QG_TILE_H / 2 - 1) / (QG_TILE_H / 2);
    const int nbig = tilesM * a.big_cols, nsmall = (int)gridDim.x - nbig;
    int b = (int)blockIdx.x - nsmall;
    e = 0;
    if (b < 0) {
      b = (int)blockIdx.x;
      row0 = b % tilesH * (QG_TILE_H / 2);
      rows = min(QG_TILE_H / 2, a.a_rows - row0);
      n0 = (a.big_cols + b / tilesH) * 256;
    } else {
      // Row tiles in multiples of eight, from 16 on: in the grid's order an XCD takes every eighth of them, whose activations stay in its
      // L2 (1.00 to 1.11 of the time otherwise over 110 shapes of 2048 to 8192 rows; 0.90 to 1.04 with eight row tiles).
      int tm, tn;
      if (tilesM % 8 == 0 && tilesM >= 16) {
        tm = b % tilesM;
        tn = b / tilesM;
      } else if (tilesM % 2 == 0 && a.big_cols % 4 == 0) {  // an XCD takes half of the rows of a quarter of the columns
        const int xcd = b & 7, seq = b >> 3, hm = tilesM / 2, qn = a.big_cols / 4;
        tm = (xcd & 1) * hm + seq % hm;
        tn = (xcd >> 1) * qn + seq / hm;
      } else {
        b = xcd_run(b, nbig);
        tm = b % tilesM;
        tn = b / tilesM;
      }
      row0 = tm * QG_TILE_H;
      rows = min(QG_TILE_H, a.a_rows - row0);
      n0 = tn * 256;
    }
  }
  if constexpr (MODE == 1) {
    row0 += 64 * blockIdx.z;
    rows -= 64 * blockIdx.z;
    if (rows <= 0) return;
    if (rows > 32) qg_tile<WT, 2, 2, 1, 2>(a, e, row0, min(rows, 64), n0, smem);
    else qg_tile<WT, 2, 1, 1, 2>(a, e, row0, rows, n0, smem);
  } else {
    if (rows > 64) qg_tile<WT, 1, 4, 2, 1, G>(a, e, row0, rows, n0, smem);
    else if (rows > 32) qg_tile<WT, 1, 2, 2, 1, G>(a, e, row0, rows, n0, smem);
    else qg_tile<WT, 1, 1, 2, 1, G>(a, e, row0, rows, n0, smem);
  }
}

template <int MODE>
static int launch_qg(const QG2Args& a, unsigned max_tiles, hipStream_t st) {
  constexpr int TN = MODE == 1 ? 1 : 2;
  dim3 grid(max_tiles, (unsigned)((a.N + 128 * TN - 1) / (128 * TN)), MODE == 1 ? 2 : (unsigned)(a.ksplit > 1 ? a.ksplit : 1));
  if (MODE == 0 && !a.ntiles) {
    const int64_t cols = grid.y, tilesH = (a.a_rows + QG_TILE_H / 2 - 1) / (QG_TILE_H / 2);
    grid.x = (unsigned)(max_tiles * a.big_cols + tilesH * (cols - a.big_cols));
    grid.y = 1;
  }
  if (MODE == 0 && a.halves) {
    constexpr size_t lds = 128 * 1024;  // the sums of four waves
    auto go = [&](auto kern) {
      HIP_RET(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
      hipLaunchKernelGGL(kern, grid, dim3(512), lds, st, a);
      return (int)hipGetLastError();
    };
    switch (a.wtype) {
      case MLLM_HIP_Q4_0: return go(qg_kernel<MLLM_HIP_Q4_0, 0, 2>);
      case MLLM_HIP_Q8_0: return go(qg_kernel<MLLM_HIP_Q8_0, 0, 2>);
      case MLLM_HIP_Q4_K: return go(qg_kernel<MLLM_HIP_Q4_K, 0, 2>);
      default: return go(qg_kernel<MLLM_HIP_Q6_K, 0, 2>);
    }
  }
  const size_t lds = 2 * (size_t)QG_TILE_H * (2 * 64 + 16);  // MODE 1: half the rows, value + residual (and the 32 rows of 256 sums of the epilogue)
  if (a.wtype == MLLM_HIP_Q4_0) hipLaunchKernelGGL((qg_kernel<MLLM_HIP_Q4_0, MODE>), grid, dim3(256), lds, st, a);
  else if (a.wtype == MLLM_HIP_Q8_0) hipLaunchKernelGGL((qg_kernel<MLLM_HIP_Q8_0, MODE>), grid, dim3(256), lds, st, a);
  else if constexpr (MODE == 0) {  // the super-block formats: plain Linear only
    if (a.wtype == MLLM_HIP_Q4_K) hipLaunchKernelGGL((qg_kernel<MLLM_HIP_Q4_K, 0>), grid, dim3(256), lds, st, a);
    else hipLaunchKernelGGL((qg_kernel<MLLM_HIP_Q6_K, 0>), grid, dim3(256), lds, st, a);
  } else return MLLM_HIP_E_BADARG;
  return (int)hipGetLastError();
}

// =========================================================================================================
// Exact block sums on the matrix cores ("qx"): the reference's arithmetic itself for many rows
//
//   y[row][n] = sum_b fp32(dW[n][b] * dX[row][b]) * float(sum_32 qW * qX)
//
// (llamafile_sgemm.cpp:697-743: Cv += set1(dW * dX) * float(int32 block sum)).  Per 32-row x 32-channel tile and block, two
// matrix instructions, sixteen conversions and sixteen fp32 FMAs:
//   * the block sum: one v_mfma_i32_32x32x32_i8 on the codes.  A nibble enters as the byte 16 (q - 8): the nibble in the high half,
//     its top bit inverted, one three-input logic operation (and a shift for the low nibbles).  The 16 goes out behind the last
//     block: a power of two moves through products and sums unrounded (|sum| <= 2^19, scales below 2^16: far from the ends of fp32).
//   * the 32 x 32 scale products dW[n] * dX[row]: an outer product of the two fp16 scales sitting in one K slot of otherwise
//     zero fp16 operands; an 11-bit by 11-bit product is exact in fp32.
//   * acc = fma(dW * dX, float(block sum), acc): the reference's operation.  Only the order in which blocks are added differs
//     from the CPU path.
// Same gemm-packed weights and tile list as the fp16-operand kernel.  Activations: Q8_0 codes as bytes [rows][K] in the order in
// which a lane's weights come out of their dwords (QX_ORDER below), and the fp16 scales of two blocks per dword.
//
// What bounds it: the vector ALU (160 instructions of 4 clocks per K step and wave, 32 clocks for each of the 8 matrix instructions beside
// them: three waves per SIMD keep it busy), with few rows per expert the weights (5.8 TB/s for 128 tokens), and the last round of workgroups.
// Codes as fp16 numbers (offsets in the mantissas of 1024 and 64) gave the sums as floats at 3.5 matrix instructions per block, but in
// 242 registers, and more than there are for Q8_0: two waves per SIMD, and a wave's own chain of instructions was what a workgroup took, with a neighbour or
// without (Q4_0 26 us, Q8_0 with registers in memory 70).  us of an FFN of 128 experts of 2048 x 768, top-8, before / now: 512 tokens
// Q4_0 145 / 122, Q8_0 269 / 173; 128 tokens Q4_0 102 / 95; 317 tokens, top-4, 512 elements Q8_0 149 / 105 (in a graph, routing and activations in it).
// =========================================================================================================
struct QXArgs {
  const char* W0;        // gemm-packed weights of matrix 0 (gate, or the only matrix), expert e at W0 + e * wstride
  const char* W1;        // matrix 1 (up) in the gate/up mode
  size_t wstride;
  const uint8_t* xq;     // Q8_0 codes of the activations [a_rows][K], a block's 32 in QX_ORDER
  const uint32_t* xd;    // [a_rows][KD] fp16 scales of blocks 2j | 2j+1 (zero past the end)
  const int* a_index;    // activation row of sorted position pos is a_index[pos] / a_div ; null: pos itself
  int a_div;
  int a_rows;
  const int* o_index;    // output row of sorted position pos (null: pos itself)
  float* out;            // fp32 [..][N]       (one-matrix mode)
  const float* bias;     // [N] or null        (one-matrix mode)
  uint8_t* hq;           // gate/up mode: Q8_0 codes of silu(g)*u [rows][N], as xq
  uint32_t* hd;          // gate/up mode: their scales [rows][ceil(N/64)], as xd
  const int* tile_expert;
  const int* tile_row0;
  const int* tile_rows;
  const int* ntiles;
  int N, K;
  int x86_scale;
  int half_tiles;        // tiles of at most sixteen rows take the 16-row form (same bits; 0: comparison runs and tests)
};

// QX_ORDER: lane half hi of the 32-row operand takes the elements 8 hi .. 8 hi + 7 and 16 + 8 hi .. of a block (bytes 16 hi .. 16 hi + 15 of the
// stored block), each eight in the order of the weights' dwords: Q4_0 low nibbles 0 4 1 5, high nibbles 2 6 3 7; Q8_0 0 2 1 3, 4 6 5 7.
// lo, hi: the codes 0..3 and 4..7
template <int WT>
__device__ __forceinline__ u32x2 qx_order(uint32_t lo, uint32_t hi) {
  if (WT == MLLM_HIP_Q4_0) return u32x2{__builtin_amdgcn_perm(hi, lo, 0x05010400u), __builtin_amdgcn_perm(hi, lo, 0x07030602u)};
  return u32x2{__builtin_amdgcn_perm(0u, lo, 0x03010200u), __builtin_amdgcn_perm(0u, hi, 0x03010200u)};
}
// constants in registers (three-input logic takes no literal)
struct QXConst {
  uint32_t m, x;
};
__device__ __forceinline__ QXConst qx_const() {
  QXConst c{0xf0f0f0f0u, 0x80808080u};
  asm volatile("" : "+v"(c.m), "+v"(c.x));
  return c;
}
// four low / high nibbles of a dword as bytes 16 (q - 8)
__device__ __forceinline__ uint32_t qx_high(uint32_t v, const QXConst& c) { return (v & c.m) ^ c.x; }
__device__ __forceinline__ uint32_t qx_low(uint32_t v, const QXConst& c) { return qx_high(v << 4, c); }
constexpr float QX_UNIT(int wt) { return wt == MLLM_HIP_Q4_0 ? 0.0625f : 1.f; }  // of the codes' products
// K steps of weights and activations in flight per wave, in the 32-row and the 16-row form (512 tokens, Q4_0, of the FFN's time with 2 / 4: 2 / 2
// 1.014, 2 / 6 1.04; a Q8_0 wave has registers for two)
constexpr int QX_ST = 2;
constexpr int QX_ST16(int wt) { return wt == MLLM_HIP_Q4_0 ? 4 : 2; }

// One tile: `rows` (<= 32) sorted positions from row0 x 128 TN channels from n0, NW weight matrices (1, or gate + up).
template <int WT, int NW, int TN>
__device__ __forceinline__ void qx_tile(const QXArgs& a, const int e, const int row0, const int rows, const int n0,
                                        unsigned char* smem) {
  constexpr int BK = 64, LDK = BK + 16;  // bytes of codes per row and K step; pitch in LDS (sixteen rows' reads cover all banks)
  constexpr int BM = 32, WN = TN * 32;
  constexpr int STAGE = BM * LDK + BM * 4;  // code rows, then the rows' scale pairs
  constexpr int QW = WT == MLLM_HIP_Q4_0 ? 1 : 2;
  constexpr int ST = QX_ST;                 // K steps of weights in flight per wave

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lrow = lane & 31, hi = lane >> 5;
  const int Kp = (int)qg_kp(a.K), kbs = Kp / 64, nbs = (int)(qg_np(a.N) / 32), KD = (a.K + 63) / 64;
  const int64_t qbytes = qg_qbytes(WT, a.N, a.K), wbytes = qg_bytes(WT, a.N, a.K);

  const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.xq), 0, (uint32_t)((int64_t)a.a_rows * a.K), 0x00020000);
  const __amdgpu_buffer_rsrc_t rD = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(a.xd), 0, (uint32_t)((int64_t)a.a_rows * KD * 4), 0x00020000);
  __amdgpu_buffer_rsrc_t rW[NW];
  rW[0] = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(a.W0 + (size_t)e * a.wstride), 0, (uint32_t)wbytes, 0x00020000);
  if (NW == 2) rW[NW - 1] = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(a.W1 + (size_t)e * a.wstride), 0, (uint32_t)wbytes, 0x00020000);

  // activations of a thread: tile row tid / 8, eight codes from 8 (tid % 8).  Rows past `rows` repeat the last one (never
  // stored); columns past K read as zeros (out-of-range buffer offsets).
  const int colA = (tid % 8) * 8;
  auto arow_of = [&](int r) -> uint32_t {
    const int pos = row0 + min(r, rows - 1);
    return (uint32_t)(a.a_index ? a.a_index[pos] / a.a_div : pos);
  };
  const uint32_t offA = arow_of(tid / 8) * (uint32_t)a.K + colA;
  // the scales of a row and K step: threads 0 .. 31, one row each
  const uint32_t offD = tid < BM ? arow_of(tid) * (uint32_t)(KD * 4) : 0xffffffffu;
  uint32_t offQ[TN], offS[TN];
#pragma unroll
  for (int j = 0; j < TN; j++) {
    const int nb = min((n0 + wave * WN) / 32 + j, nbs - 1);
    offQ[j] = (uint32_t)((int64_t)nb * kbs * (1024 * QW) + lane * 16);
    offS[j] = (uint32_t)(qbytes + ((int64_t)nb * kbs * 32 + lrow) * 4);
  }
  // Activations travel as many K steps ahead of their use as the weights, in as many register sets.  Vector memory returns in order:
  // the wait for a step's activations also waits for every load issued before them, and a shorter lead would be the weights' lead too.
  u32x2 ga[ST];
  uint32_t gd[ST] = {};
  auto loadA = [&](int set, int kt) {
    ga[set] = __builtin_amdgcn_raw_buffer_load_b64(rA, kt * BK + colA < a.K ? offA : 0xffffffffu, kt * BK, 0);
    if (tid < BM) gd[set] = __builtin_amdgcn_raw_buffer_load_b32(rD, kt < KD ? offD : 0xffffffffu, kt * 4, 0);
  };
  auto storeA = [&](int set, int buf) {
    *reinterpret_cast<u32x2*>(smem + buf * STAGE + (tid / 8) * LDK + colA) = ga[set];
    if (tid < BM) *reinterpret_cast<uint32_t*>(smem + buf * STAGE + BM * LDK + tid * 4) = gd[set];
  };

  v16f acc[NW][TN];
#pragma unroll
  for (int w = 0; w < NW; w++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[w][j][r] = 0.f;

  u32x4 rq[ST][NW][TN][QW];  // packed codes of the K steps in flight (ring, slot = step % ST)
  uint32_t rs[ST][NW][TN];   // their scale dwords
  auto loadW1 = [&](int slot, int kt, int w, int j) {  // steps past the end read nothing (zeros): the ring is always full
#pragma unroll
    for (int p = 0; p < QW; p++)
      rq[slot][w][j][p] = __builtin_amdgcn_raw_buffer_load_b128(rW[w], kt < kbs ? offQ[j] : 0xffffffffu, (kt * QW + p) * 1024, 0);
    rs[slot][w][j] = __builtin_amdgcn_raw_buffer_load_b32(rW[w], kt < kbs ? offS[j] : 0xffffffffu, kt * 128, 0);
  };
  // Scale operand of the weights: the fp16 scale of the step's first block in K slot 0 (low half of the first register), of
  // its second block in K slot 1 (high half), in the lanes of the low K half only; every other K slot is zero.  The
  // activations' scale pair is used as it comes (first register of an otherwise zero operand): what a K slot holds does not
  // matter where the other operand is zero.
  const uint32_t msk0 = hi ? 0u : 0x0000ffffu, msk1 = hi ? 0u : 0xffff0000u;
  const v16f zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const QXConst kc = qx_const();
  const v16i izero = {};

  // A "group" is one (block, matrix, column tile): two matrix instructions, in their shadow the unpacking of the NEXT group's weights,
  // sixteen conversions and FMAs.
  constexpr int G = 2 * NW * TN;  // groups per K step: block-major, then matrix, then column tile
  v4i fw;                         // codes of the next group
  u32x2 sw = {0u, 0u}, rec = {0u, 0u};  // its scale operand, the rows' (K slots 0 to 3 of either half)
  asm("" : "+v"(sw), "+v"(rec));        // (known to be zero, the upper register would be written again for every group)
  auto unpack = [&](const u32x4 (&q)[QW], uint32_t s, int b) {
    if (WT == MLLM_HIP_Q4_0) fw = v4i{(int)qx_low(q[0][2 * b], kc), (int)qx_high(q[0][2 * b], kc), (int)qx_low(q[0][2 * b + 1], kc), (int)qx_high(q[0][2 * b + 1], kc)};
    else fw = __builtin_bit_cast(v4i, q[QW == 2 ? b : 0]);
    sw.x = s & (b ? msk1 : msk0);
  };

  const int nsteps = (kbs + ST - 1) / ST * ST;
#pragma unroll
  for (int s = 0; s < ST; s++) {
    loadA(s, s);
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
      for (int j = 0; j < TN; j++) loadW1(s, s, w, j);
  }
  storeA(0, 0);
  unpack(rq[0][0][0], rs[0][0][0], 0);
  __syncthreads();

  // one K step (64 elements = two blocks) with its weights in ring slot SLOT; refills the slot with step kt + ST
  auto kstep = [&](auto slot_tag, int kt) {
    constexpr int SLOT = decltype(slot_tag)::value;
    constexpr int NSLOT = (SLOT + 1) % ST;
    const int buf = kt & 1;
    loadA(SLOT, kt + ST);  // the set whose step (kt) is in LDS already
    v4i fb[2];
#pragma unroll
    for (int b = 0; b < 2; b++) fb[b] = *reinterpret_cast<const v4i*>(smem + buf * STAGE + lrow * LDK + b * 32 + hi * 16);
    rec.x = *reinterpret_cast<const uint32_t*>(smem + buf * STAGE + BM * LDK + lrow * 4);
#pragma unroll
    for (int g = 0; g < G; g++) {
      const int b = g / (NW * TN), w = (g / TN) % NW, j = g % TN;
      // the next group: (b', w', j') in this step, or the first group of the next step (ring slot NSLOT)
      const bool last = g == G - 1;
      const int gn = last ? 0 : g + 1;
      const int bn = gn / (NW * TN), wn = (gn / TN) % NW, jn = gn % TN;
      __builtin_amdgcn_sched_barrier(0);
      const v16i D = __builtin_amdgcn_mfma_i32_32x32x32_i8(fw, fb[b], izero, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      const v16f T = __builtin_amdgcn_mfma_f32_32x32x8f16(__builtin_bit_cast(f16x4, sw), __builtin_bit_cast(f16x4, rec), zero16, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (last) {
        unpack(rq[NSLOT][wn][jn], rs[NSLOT][wn][jn], bn);
      } else {
        unpack(rq[SLOT][wn][jn], rs[SLOT][wn][jn], bn);
        if (bn == 1) loadW1(SLOT, kt + ST, wn, jn);  // both blocks of (wn, jn) are unpacked: its ring registers are free
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < 16; r++) acc[w][j][r] = fmaf(T[r], (float)D[r], acc[w][j][r]);
      asm volatile("" : "+v"(acc[w][j]));  // pins the FMAs here (the compiler otherwise sinks them to the end of the body)
    }
    storeA(NSLOT, buf ^ 1);
    __syncthreads();
  };
  for (int kt = 0; kt < nsteps; kt += ST) {
    kstep(std::integral_constant<int, 0>{}, kt);
    kstep(std::integral_constant<int, 1>{}, kt + 1);
  }

  if (QX_UNIT(WT) != 1.f) {
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[w][j][r] *= QX_UNIT(WT);
  }
  // acc[w][j][4g+e] = result[row0 + lrow][n0 + wave*WN + 32j + 8g + 4hi + e]
  if (NW == 1) {
    if (lrow < rows) {
      const int pos = row0 + lrow;
      float* orow = a.out + (int64_t)(a.o_index ? a.o_index[pos] : pos) * a.N;
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const int n = n0 + wave * WN + j * 32 + 8 * g + 4 * hi;
          f32x4 v = {acc[0][j][4 * g], acc[0][j][4 * g + 1], acc[0][j][4 * g + 2], acc[0][j][4 * g + 3]};
          if (n + 3 < a.N && a.N % 4 == 0) {
            if (a.bias) v += *reinterpret_cast<const f32x4*>(a.bias + n);
            *reinterpret_cast<f32x4*>(orow + n) = v;
          } else {
#pragma unroll
            for (int e2 = 0; e2 < 4; e2++)
              if (n + e2 < a.N) orow[n + e2] = a.bias ? v[e2] + a.bias[n + e2] : v[e2];
          }
        }
    }
  } else {
    // h = silu(gate) * up, quantized to Q8_0 over each block of 32 channels (a block is one column tile j: 16 channels in
    // this lane, 16 in lane ^ 32): the next Linear's activation format
    const int nblk = a.N / QK, KDo = (a.N + 63) / 64;
#pragma unroll
    for (int j = 0; j < TN; j++) {
      float h[16];
      float amax = 0.f;
#pragma unroll
      for (int q = 0; q < 16; q++) {
        h[q] = silu_f(acc[0][j][q]) * acc[NW - 1][j][q];
        amax = fmaxf(amax, fabsf(h[q]));
      }
      amax = max32(amax);
      const float d = amax / 127.f;
      const float idv = (amax != 0.f) ? 127.f / amax : 0.f;
      uint16_t bits = f32_to_f16bits(d);
      if (a.x86_scale) bits = x86_scale_bits(bits);
      const int blk = (n0 + wave * WN) / 32 + j;
      uint32_t p[4];  // the codes 8 g + 4 hi .. + 3
#pragma unroll
      for (int g = 0; g < 4; g++) {
        p[g] = 0u;
#pragma unroll
        for (int e2 = 0; e2 < 4; e2++) p[g] |= ((uint32_t)min(127, max(-128, (int)rintf(h[4 * g + e2] * idv))) & 0xffu) << (8 * e2);
      }
      // lane half hi takes the eights hi and 2 + hi: its own half of each and the other lane's
      const auto r0 = __builtin_amdgcn_permlane32_swap(p[0], p[1], false, false);
      const auto r1 = __builtin_amdgcn_permlane32_swap(p[2], p[3], false, false);
      const u32x2 o0 = qx_order<WT>(r0[0], r0[1]), o1 = qx_order<WT>(r1[0], r1[1]);
      if (lrow < rows && blk < nblk) {
        *reinterpret_cast<u32x4*>(a.hq + (int64_t)(row0 + lrow) * a.N + blk * 32 + hi * 16) = u32x4{o0.x, o0.y, o1.x, o1.y};
        if (hi == 0) {
          uint16_t* hd = reinterpret_cast<uint16_t*>(a.hd + (int64_t)(row0 + lrow) * KDo);
          hd[blk] = bits;
          if (blk == nblk - 1 && (nblk & 1)) hd[blk + 1] = 0;  // the unused half of the last dword
        }
      }
    }
  }
}


// The same tile for at most SIXTEEN sorted positions: v_mfma_i32_16x16x32_i8 takes a block of 16 channels x 16 rows, so a tile of
// up to 16 rows costs half the matrix time (and half the FMAs) of the 32-row form above, which would pad it to 32.  Same packed
// weights: a lane of the 32-row layout holds, of channel lane % 32, the block's elements 8 hi .. 8 hi + 7 (first dword, or two)
// and 16 + 8 hi .. (second); the 16-row operand wants, in lane (channel c, K group kg), eight elements of channel c [+ 16].
// v_permlane16_swap on the PACKED dwords (first eight as first operand, second as second) leaves in the first the channels 0..15
// and in the second the channels 16..31, each with the K groups (hi 0, first), (hi 0, second), (hi 1, first), (hi 1, second): bytes
// 8 kg .. 8 kg + 7 of the stored activation block.  The products that meet are the same and every sum is the same exact integer.
// Same scale products, same FMAs per block, same order of blocks: the same bits as the 32-row form row by row.
template <int WT, int NW, int TN>
__device__ __forceinline__ void qx_tile16(const QXArgs& a, const int e, const int row0, const int rows, const int n0,
                                          unsigned char* smem) {
  constexpr int BK = 64, LDK = BK + 16;
  constexpr int BM = 16, WN = TN * 32;
  constexpr int STAGE = BM * LDK + BM * 4;
  constexpr int QW = WT == MLLM_HIP_Q4_0 ? 1 : 2;
  constexpr int ST = QX_ST16(WT);  // K steps of weights in flight per wave

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lrow = lane & 31;                 // channel of this lane in the packed layout
  const int c16 = lane & 15, kg = lane >> 4;  // 16-row operands: channel / row c16, K group kg
  const int Kp = (int)qg_kp(a.K), kbs = Kp / 64, nbs = (int)(qg_np(a.N) / 32), KD = (a.K + 63) / 64;
  const int64_t qbytes = qg_qbytes(WT, a.N, a.K), wbytes = qg_bytes(WT, a.N, a.K);

  const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.xq), 0, (uint32_t)((int64_t)a.a_rows * a.K), 0x00020000);
  const __amdgpu_buffer_rsrc_t rD = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(a.xd), 0, (uint32_t)((int64_t)a.a_rows * KD * 4), 0x00020000);
  __amdgpu_buffer_rsrc_t rW[NW];
  rW[0] = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(a.W0 + (size_t)e * a.wstride), 0, (uint32_t)wbytes, 0x00020000);
  if (NW == 2) rW[NW - 1] = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(a.W1 + (size_t)e * a.wstride), 0, (uint32_t)wbytes, 0x00020000);

  // activations of threads 0 .. 127: tile row tid / 8, eight codes from 8 (tid % 8); scales of a row: threads 0 .. 15.
  // Rows past `rows` repeat the last one (never stored); columns past K read as zeros.
  const bool ldA = tid < BM * 8;
  const int colA = (tid % 8) * 8;
  auto arow_of = [&](int r) -> uint32_t {
    const int pos = row0 + min(r, rows - 1);
    return (uint32_t)(a.a_index ? a.a_index[pos] / a.a_div : pos);
  };
  const uint32_t offA = ldA ? arow_of(tid / 8) * (uint32_t)a.K + colA : 0xffffffffu;
  const uint32_t offD = tid < BM ? arow_of(tid) * (uint32_t)(KD * 4) : 0xffffffffu;
  uint32_t offQ[TN], offS[TN];
#pragma unroll
  for (int j = 0; j < TN; j++) {
    const int nb = min((n0 + wave * WN) / 32 + j, nbs - 1);
    offQ[j] = (uint32_t)((int64_t)nb * kbs * (1024 * QW) + lane * 16);
    offS[j] = (uint32_t)(qbytes + ((int64_t)nb * kbs * 32 + lrow) * 4);
  }
  u32x2 ga[ST] = {};
  uint32_t gd[ST] = {};
  auto loadA = [&](int set, int kt) {  // as far ahead as the weights, as in the 32-row form
    if (ldA) ga[set] = __builtin_amdgcn_raw_buffer_load_b64(rA, kt * BK + colA < a.K ? offA : 0xffffffffu, kt * BK, 0);
    if (tid < BM) gd[set] = __builtin_amdgcn_raw_buffer_load_b32(rD, kt < KD ? offD : 0xffffffffu, kt * 4, 0);
  };
  auto storeA = [&](int set, int buf) {
    if (ldA) *reinterpret_cast<u32x2*>(smem + buf * STAGE + (tid / 8) * LDK + colA) = ga[set];
    if (tid < BM) *reinterpret_cast<uint32_t*>(smem + buf * STAGE + BM * LDK + tid * 4) = gd[set];
  };

  f32x4 acc[NW][TN][2];  // [matrix][column tile][channel half]
#pragma unroll
  for (int w = 0; w < NW; w++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int h = 0; h < 2; h++) acc[w][j][h] = f32x4{0.f, 0.f, 0.f, 0.f};

  u32x4 rq[ST][NW][TN][QW];
  uint32_t rs[ST][NW][TN];
  auto loadW1 = [&](int slot, int kt, int w, int j) {
#pragma unroll
    for (int p = 0; p < QW; p++)
      rq[slot][w][j][p] = __builtin_amdgcn_raw_buffer_load_b128(rW[w], kt < kbs ? offQ[j] : 0xffffffffu, (kt * QW + p) * 1024, 0);
    rs[slot][w][j] = __builtin_amdgcn_raw_buffer_load_b32(rW[w], kt < kbs ? offS[j] : 0xffffffffu, kt * 128, 0);
  };
  // scale operands: the fp16 scale of the step's first block in K slot 0, of its second block in K slot 1, in the lanes of K
  // group 0; everything else zero
  const uint32_t msk0 = kg ? 0u : 0x0000ffffu, msk1 = kg ? 0u : 0xffff0000u;
  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};
  const v4i izero = {};
  const QXConst kc = qx_const();

  // the operands of one (block, matrix, column tile) from the packed registers: codes of the channels 0..15 | 16..31
  auto unpack = [&](const u32x4 (&q)[QW], int b, int64_t (&fw)[2]) {
    u32x2 o[2];
    if (WT == MLLM_HIP_Q4_0) {
      const auto r = __builtin_amdgcn_permlane16_swap(q[0][2 * b], q[0][2 * b + 1], false, false);
#pragma unroll
      for (int h = 0; h < 2; h++) o[h] = u32x2{qx_low(r[h], kc), qx_high(r[h], kc)};
    } else {
      // block b: first eight in dwords 0, 1 of register b, second in 2, 3
      const auto r0 = __builtin_amdgcn_permlane16_swap(q[QW - 1 ? b : 0][0], q[QW - 1 ? b : 0][2], false, false);
      const auto r1 = __builtin_amdgcn_permlane16_swap(q[QW - 1 ? b : 0][1], q[QW - 1 ? b : 0][3], false, false);
#pragma unroll
      for (int h = 0; h < 2; h++) o[h] = u32x2{r0[h], r1[h]};
    }
#pragma unroll
    for (int h = 0; h < 2; h++) fw[h] = __builtin_bit_cast(int64_t, o[h]);
  };
  auto scales = [&](uint32_t s, int b, u32x4 (&sw)[2]) {
    const uint32_t up = __builtin_amdgcn_permlane16_swap(s, s, false, false)[1];  // lanes 0..15 <- lanes 16..31
    const uint32_t m = b ? msk1 : msk0;
    sw[0].x = s & m;
    sw[1].x = up & m;
  };

  constexpr int G = 2 * NW * TN;  // groups per K step: block-major, then matrix, then column tile
  int64_t fw[2][2];               // [current | next group][channel half]
  u32x4 sw[2][2] = {{{0u, 0u, 0u, 0u}, {0u, 0u, 0u, 0u}}, {{0u, 0u, 0u, 0u}, {0u, 0u, 0u, 0u}}};
  u32x4 rec = {0u, 0u, 0u, 0u};
  asm("" : "+v"(sw[0][0]), "+v"(sw[0][1]), "+v"(sw[1][0]), "+v"(sw[1][1]), "+v"(rec));

  const int nsteps = (kbs + ST - 1) / ST * ST;
#pragma unroll
  for (int s = 0; s < ST; s++) {
    loadA(s, s);
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
      for (int j = 0; j < TN; j++) loadW1(s, s, w, j);
  }
  storeA(0, 0);
  unpack(rq[0][0][0], 0, fw[0]);
  scales(rs[0][0][0], 0, sw[0]);
  __syncthreads();

  auto kstep = [&](auto slot_tag, int kt) {
    constexpr int SLOT = decltype(slot_tag)::value;
    constexpr int NSLOT = (SLOT + 1) % ST;
    const int buf = kt & 1;
    loadA(SLOT, kt + ST);
    int64_t fb[2];
#pragma unroll
    for (int b = 0; b < 2; b++) fb[b] = *reinterpret_cast<const int64_t*>(smem + buf * STAGE + c16 * LDK + b * 32 + kg * 8);
    rec.x = *reinterpret_cast<const uint32_t*>(smem + buf * STAGE + BM * LDK + c16 * 4);
#pragma unroll
    for (int g = 0; g < G; g++) {
      const int c = g & 1, n = c ^ 1;  // the register sets alternate (G is even)
      const int b = g / (NW * TN), w = (g / TN) % NW, j = g % TN;
      const bool last = g == G - 1;
      const int gn = last ? 0 : g + 1;
      const int bn = gn / (NW * TN), wn = (gn / TN) % NW, jn = gn % TN;
      v4i D[2];
      f32x4 T[2];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int h = 0; h < 2; h++) D[h] = __builtin_amdgcn_mfma_i32_16x16x32_i8(fw[c][h], fb[b], izero, 0, 0, 0);
#pragma unroll
      for (int h = 0; h < 2; h++) T[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, sw[c][h]), __builtin_bit_cast(f16x8, rec), zero4, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (last) {
        unpack(rq[NSLOT][wn][jn], bn, fw[n]);
        scales(rs[NSLOT][wn][jn], bn, sw[n]);
      } else {
        unpack(rq[SLOT][wn][jn], bn, fw[n]);
        scales(rs[SLOT][wn][jn], bn, sw[n]);
        if (bn == 1) loadW1(SLOT, kt + ST, wn, jn);  // both blocks of (wn, jn) are unpacked
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[w][j][h][r] = fmaf(T[h][r], (float)D[h][r], acc[w][j][h][r]);
      asm volatile("" : "+v"(acc[w][j][0]), "+v"(acc[w][j][1]));
    }
    storeA(NSLOT, buf ^ 1);
    __syncthreads();
  };
  for (int kt = 0; kt < nsteps; kt += ST) {
    kstep(std::integral_constant<int, 0>{}, kt);
    kstep(std::integral_constant<int, 1>{}, kt + 1);
    if constexpr (ST >= 4) {
      kstep(std::integral_constant<int, 2>{}, kt + 2);
      kstep(std::integral_constant<int, 3>{}, kt + 3);
    }
  }

  if (QX_UNIT(WT) != 1.f) {
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int h = 0; h < 2; h++) acc[w][j][h] *= QX_UNIT(WT);
  }
  // acc[w][j][h][e] = result[row0 + c16][n0 + wave*WN + 32j + 16h + 4kg + e]
  if (NW == 1) {
    if (c16 < rows) {
      const int pos = row0 + c16;
      float* orow = a.out + (int64_t)(a.o_index ? a.o_index[pos] : pos) * a.N;
#pragma unroll
      for (int j = 0; j < TN; j++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const int n = n0 + wave * WN + j * 32 + 16 * h + 4 * kg;
          f32x4 v = acc[0][j][h];
          if (n + 3 < a.N && a.N % 4 == 0) {
            if (a.bias) v += *reinterpret_cast<const f32x4*>(a.bias + n);
            *reinterpret_cast<f32x4*>(orow + n) = v;
          } else {
#pragma unroll
            for (int e2 = 0; e2 < 4; e2++)
              if (n + e2 < a.N) orow[n + e2] = a.bias ? v[e2] + a.bias[n + e2] : v[e2];
          }
        }
    }
  } else {
    // h = silu(gate) * up, quantized to Q8_0 over each block of 32 channels (one column tile j: eight channels in each of the
    // four lanes of a row), written in the next Linear's activation format
    const int nblk = a.N / QK, KDo = (a.N + 63) / 64;
#pragma unroll
    for (int j = 0; j < TN; j++) {
      float hv[8];
      float amax = 0.f;
#pragma unroll
      for (int q = 0; q < 8; q++) {
        hv[q] = silu_f(acc[0][j][q >> 2][q & 3]) * acc[NW - 1][j][q >> 2][q & 3];
        amax = fmaxf(amax, fabsf(hv[q]));
      }
      amax = max16(amax);
      amax = max32(amax);
      const float d = amax / 127.f;
      const float idv = (amax != 0.f) ? 127.f / amax : 0.f;
      uint16_t bits = f32_to_f16bits(d);
      if (a.x86_scale) bits = x86_scale_bits(bits);
      const int blk = (n0 + wave * WN) / 32 + j;
      uint32_t p[2];  // the codes 16 h + 4 kg .. + 3
#pragma unroll
      for (int h = 0; h < 2; h++) {
        p[h] = 0u;
#pragma unroll
        for (int e2 = 0; e2 < 4; e2++) p[h] |= ((uint32_t)min(127, max(-128, (int)rintf(hv[4 * h + e2] * idv))) & 0xffu) << (8 * e2);
      }
      // K group kg takes the eight 2 (kg % 2) + kg / 2: its own half and the half of the lane sixteen away
      const auto r = __builtin_amdgcn_permlane16_swap(p[0], p[1], false, false);
      const u32x2 o = qx_order<WT>(r[0], r[1]);
      if (c16 < rows && blk < nblk) {
        *reinterpret_cast<u32x2*>(a.hq + (int64_t)(row0 + c16) * a.N + blk * 32 + (kg >> 1) * 16 + (kg & 1) * 8) = o;
        if (kg == 0) {
          uint16_t* hd = reinterpret_cast<uint16_t*>(a.hd + (int64_t)(row0 + c16) * KDo);
          hd[blk] = bits;
          if (blk == nblk - 1 && (nblk & 1)) hd[blk + 1] = 0;  // the unused half of the last dword
        }
      }
    }
  }
}

constexpr int QX_TILE_H = 32;
constexpr int QX_DOWN_TN = 2;  // column tiles per wave in the one-matrix mode
constexpr int QX_GROUP = 8;    // tiles per group of work items (see qx_kernel)
// MODE 0: one matrix, up to 32 rows x 256 channels per workgroup.  MODE 1: gate and up together, 32 rows x 128 channels.
template <int WT, int MODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void qx_kernel(QXArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  // Work items in groups of QX_GROUP tiles (list order: an expert's tiles are neighbours) x all column blocks, inside a
  // group the tile index fastest.  Workgroup L runs on XCD L % 8, and every XCD has its own L2: XCD x takes a contiguous
  // eighth of the work items, so that the tiles of one expert and column block -- which read the same weights -- and the
  // column blocks of one tile -- which read the same activation rows -- run on one XCD at about the same time.
  // (512 tokens x 8 of 128 experts, whole FFN: column block slowest over the whole list 167.5 us, groups of eight tiles
  // 162.3; 8192 tokens 1352 -> 1330.)
  const int nt = min(a.ntiles[0], (int)gridDim.x), ny = (int)gridDim.y;
  const int L = (int)(blockIdx.x + gridDim.x * blockIdx.y);
  const int nw = nt * ny, base = nw >> 3, rem = nw & 7;  // XCD x takes base + (x < rem) items
  const int xcd = L & 7, seq = L >> 3;
  if (seq >= base + (xcd < rem)) return;
  const int w = xcd * base + min(xcd, rem) + seq;
  const int per = QX_GROUP * ny, g = w / per, r0 = w - g * per;
  const int gt = min(QX_GROUP, nt - g * QX_GROUP);  // tiles in this group (the last one may be short)
  const int by = r0 / gt, t = g * QX_GROUP + (r0 - by * gt);
  const int e = a.tile_expert[t], row0 = a.tile_row0[t], rows = a.tile_rows[t];
  if constexpr (MODE == 1) {
    const int n0 = by * 128;
    if (rows <= 16 && a.half_tiles) qx_tile16<WT, 2, 1>(a, e, row0, rows, n0, smem);
    else qx_tile<WT, 2, 1>(a, e, row0, rows, n0, smem);
  } else {
    const int n0 = by * (128 * QX_DOWN_TN);
    if (rows <= 16 && a.half_tiles) qx_tile16<WT, 1, QX_DOWN_TN>(a, e, row0, rows, n0, smem);
    else qx_tile<WT, 1, QX_DOWN_TN>(a, e, row0, rows, n0, smem);
  }
}



template <int MODE>
static int launch_qx(int wtype, const QXArgs& a, unsigned max_tiles, hipStream_t st) {
  const int wg_n = MODE == 1 ? 128 : 128 * QX_DOWN_TN;
  const dim3 grid(max_tiles, (unsigned)((a.N + wg_n - 1) / wg_n));
  const size_t lds = 2 * (size_t)(QX_TILE_H * (64 + 16) + QX_TILE_H * 4);
  if (wtype == MLLM_HIP_Q4_0) hipLaunchKernelGGL((qx_kernel<MLLM_HIP_Q4_0, MODE>), grid, dim3(256), lds, st, a);
  else hipLaunchKernelGGL((qx_kernel<MLLM_HIP_Q8_0, MODE>), grid, dim3(256), lds, st, a);
  return (int)hipGetLastError();
}

// activations for the kernel above: Q8_0 quantization (bit-exact codes and scale), a block's codes in QX_ORDER, the scales of two
// blocks per dword (the second half of a last, incomplete one is zero)
template <int WT>
__device__ __forceinline__ void qx_act_block(const void* __restrict__ x, int x_dtype, uint8_t* __restrict__ xq, uint32_t* __restrict__ xd,
                                             int64_t i, int nb, int x86_scale) {
  float v[32];
  uint32_t q[8];
  int sum;
  load_block_f32(x, x_dtype, i * QK, v);
  uint16_t bits = quantize_block_q8_0(v, q, sum);
  if (x86_scale) bits = x86_scale_bits(bits);
  u32x4* out = reinterpret_cast<u32x4*>(xq + i * QK);
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const u32x2 lo = qx_order<WT>(q[2 * h], q[2 * h + 1]), hi = qx_order<WT>(q[4 + 2 * h], q[5 + 2 * h]);
    out[h] = u32x4{lo.x, lo.y, hi.x, hi.y};
  }
  const int64_t row = i / nb;
  const int b = (int)(i - row * nb), KD = (nb + 1) / 2;
  uint16_t* rec = reinterpret_cast<uint16_t*>(xd + row * KD);
  rec[b] = bits;
  if (b == nb - 1 && (nb & 1)) rec[b + 1] = 0;
}

// the two independent preparations of the grouped FFN in one launch: workgroup 0 routes, the others quantize x
template <int WT>
__global__ __launch_bounds__(1024) void qx_prepare_kernel(const int32_t* __restrict__ ids, int n, int E, int tile_h, RouteOut o,
                                                          const void* __restrict__ x, int x_dtype, uint8_t* __restrict__ xq,
                                                          uint32_t* __restrict__ xd, int64_t nblocks, int nb, int x86_scale) {
  extern __shared__ int s_route[];
  if (blockIdx.x == 0) {
    moe_route_body<true>(ids, n, E, tile_h, o, s_route);
    return;
  }
  const int64_t i = (int64_t)(blockIdx.x - 1) * 1024 + threadIdx.x;
  if (i < nblocks) qx_act_block<WT>(x, x_dtype, xq, xd, i, nb, x86_scale);
}

// y[t][h] = sum_j per[t*k + j][h] * w[t][j]   (multiply, then add in j order: modeling_qwen3_moe_fa2.hpp:233-236)
__global__ __launch_bounds__(256) void moe_combine_kernel(const float* __restrict__ per, const float* __restrict__ w, const int32_t* __restrict__ ids,
                                                          float* __restrict__ y, int64_t T, int H, int k, int E) {
  // four consecutive channels per thread (H % 4 == 0: H is a multiple of the block size), all k rows requested before the
  // first is used; the sum itself runs in slot order
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= T * H) return;
  const int64_t t = i / H;
  const int h = (int)(i - t * H);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int j0 = 0; j0 < k; j0 += 8) {
    // every load is unconditional (slots past k repeat the last one; the row of a slot without expert was never written
    // but is readable memory): nothing waits on a branch, and what must not count is dropped by a select
    int e[8];
    float wj[8];
    f32x4 v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int64_t s = t * k + min(j0 + u, k - 1);
      e[u] = ids[s];
      wj[u] = w[s];
      v[u] = *reinterpret_cast<const f32x4*>(per + s * H + h);
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const f32x4 nx = acc + v[u] * wj[u];
      const bool ok = j0 + u < k && e[u] >= 0 && e[u] < E;
      acc.x = ok ? nx.x : acc.x;
      acc.y = ok ? nx.y : acc.y;
      acc.z = ok ? nx.z : acc.z;
      acc.w = ok ? nx.w : acc.w;
    }
  }
  *reinterpret_cast<f32x4*>(y + i) = acc;
}

// ---- workspace carving ---------------------------------------------------------------------------------------
struct Carver {
  char* p;
  size_t used = 0;
  explicit Carver(void* base) : p(reinterpret_cast<char*>(base)) {}
  template <typename T>
  T* take(size_t count) {
    T* r = reinterpret_cast<T*>(p ? p + used : nullptr);
    used += align_up(count * sizeof(T), 256);
    return r;
  }
};
static RouteOut carve_route(Carver& c, int E, int64_t entries, int tile_h = TOK_TILE) {
  RouteOut o;
  const size_t max_tiles = (size_t)E + (size_t)(entries / tile_h) + 1;
  o.counts = c.take<int>(E);
  o.offsets = c.take<int>(E + 1);
  o.sorted_idx = c.take<int>(entries);
  o.tile_expert = c.take<int>(max_tiles);
  o.tile_row0 = c.take<int>(max_tiles);
  o.tile_rows = c.take<int>(max_tiles);
  o.ntiles = c.take<int>(1);
  return o;
}

template <int MODE>
static int launch_tiles(int wtype, const QGemmArgs& a, unsigned max_tiles, hipStream_t st) {
  const dim3 grid(max_tiles, (unsigned)((a.N + 127) / 128));
  const size_t lds = (MODE == 1 && SU_BYTES > SA_BYTES + SDX_BYTES) ? (size_t)SU_BYTES : (size_t)(SA_BYTES + SDX_BYTES);
  auto launch = [&](auto kern) -> int {
    if (lds > 64 * 1024)
      HIP_RET(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, grid, dim3(MODE == 1 ? 512 : 256), lds, st, a);
    return (int)hipGetLastError();
  };
  return wtype == MLLM_HIP_Q4_0 ? launch(qgemm_tile_kernel<MLLM_HIP_Q4_0, MODE>) : launch(qgemm_tile_kernel<MLLM_HIP_Q8_0, MODE>);
}

// The gemm-packed matrix as wk_gemm.h reads it: a block is 64 elements, operand d the lane's eight weights of the d-th 16 of them,
// dequantized to fp16 as in qg_tile.
struct QWavesArgs {
  const char* W;
  const uint16_t* xh;  // fp16 [M][K]
  const float* bias;   // [N] or null
  float* y;            // [M][N]
  int M, N, K;
};
template <int WT>
struct QWaves {
  typedef QWavesArgs Args;
  typedef v16f Acc;
  typedef f32x4 Sum4;
  typedef f16x8 X;
  static constexpr int QW = qg_nibbles(WT) ? 1 : 2, SDW = qg_scale_dwords(WT);
  struct W {
    u32x4 q[QW];
    uint32_t s[SDW];
  };
  struct Col {
    uint32_t q, s;
  };
  static __host__ __device__ __forceinline__ int kblocks(const Args& a) { return (a.K + 63) / 64; }
  static __device__ __forceinline__ int row_bytes(const Args& a) { return a.K * 2; }
  static __device__ __forceinline__ const void* activations(const Args& a) { return a.xh; }
  static __device__ __forceinline__ __amdgpu_buffer_rsrc_t weights(const Args& a) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(a.W), 0, (uint32_t)qg_bytes(WT, a.N, a.K), 0x00020000);
  }
  static __device__ __forceinline__ Col col(const Args& a, int nb, int lane) {
    const int64_t kbs = qg_kp(a.K) / 64;
    nb = min(nb, (int)(qg_np(a.N) / 32) - 1);
    return Col{(uint32_t)(nb * kbs * (1024 * QW) + lane * 16), (uint32_t)(qg_qbytes(WT, a.N, a.K) + (nb * kbs * 32 + (lane & 31)) * 4 * SDW)};
  }
  static __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, const Col& c, int kb, W& w) {
#pragma unroll
    for (int p = 0; p < QW; p++) w.q[p] = __builtin_amdgcn_raw_buffer_load_b128(r, kb < 0 ? 0xffffffffu : c.q, (kb * QW + p) * 1024, 0);
    if constexpr (SDW == 1) {
      w.s[0] = __builtin_amdgcn_raw_buffer_load_b32(r, kb < 0 ? 0xffffffffu : c.s, kb * 128, 0);
    } else {
      const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, kb < 0 ? 0xffffffffu : c.s, kb * 256, 0);
      w.s[0] = v.x;
      w.s[1] = v.y;
    }
  }
  static __device__ __forceinline__ X operand(const W& w, int d) {
    const f16x2 dd = qg_scale2<WT>(w.s, d), dm = qg_offset2<WT>(w.s, d);
    uint32_t o[4], lo;
#pragma unroll
    for (int b = 0; b < 4; b++) o[b] = qg_pair<WT, 1>(w.q, d, b, dd, dm, lo);
    return __builtin_bit_cast(f16x8, u32x4{o[0], o[1], o[2], o[3]});
  }
  static __device__ __forceinline__ Acc mma(const X& w, const X& x, const Acc& acc) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(w, x, acc, 0, 0, 0); }
  static __device__ __forceinline__ void store(const Args& a, int m, int n, f32x4 v) {
    float* y = a.y + (int64_t)m * a.N + n;
    if (n + 3 < a.N && a.N % 4 == 0) {
      if (a.bias) v += *reinterpret_cast<const f32x4*>(a.bias + n);
      *reinterpret_cast<f32x4*>(y) = v;
      return;
    }
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (n + e < a.N) y[e] = a.bias ? v[e] + a.bias[n + e] : v[e];
  }
};
template <int WT>
static int launch_q_waves(int form, const QWavesArgs& a, hipStream_t st) {
  switch (form) {
    case 0: return wk_gemm_launch<QWaves<WT>, 1, 1, 8, 2>(a, st);
    case 1: return wk_gemm_launch<QWaves<WT>, 1, 2, 8, 1>(a, st);
    default: return wk_gemm_64x64<QWaves<WT>>(a, st);
  }
}

// y = sum over the K ranges of their partial results (in range order) + bias
__global__ __launch_bounds__(256) void qg_reduce_kernel(const float* __restrict__ partial, int Z, int64_t MN, int N, const float* __restrict__ bias,
                                                        float* __restrict__ y) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;  // N % 4 == 0 on this path
  if (i >= MN) return;
  f32x4 v = *reinterpret_cast<const f32x4*>(partial + i);
  for (int z = 1; z < Z; z++) v += *reinterpret_cast<const f32x4*>(partial + (size_t)z * MN + i);
  if (bias) v += *reinterpret_cast<const f32x4*>(bias + i % N);
  *reinterpret_cast<f32x4*>(y + i) = v;
}

// How a Linear runs.  Up to a few hundred rows its M/128 x N/256 tiles are far fewer than the chip has CUs (gate projection of the
// 4B layer at 128 rows: 38, down: 10), so there is a choice:
//   waves   the waves of a workgroup split K of a small tile (wk_gemm.h; forms 0..2 of launch_q_waves)
//   halves  128 x 256 tiles by eight waves, four for each half of K: two waves per SIMD where a tile has a CU to itself
//   ranges  128 x 256 tiles, K cut into up to eight ranges that run as separate workgroups (of eight waves, halves of a range each, while all have a CU to
//           themselves, q_ranges_in_halves; else of four), leave partial results and are added by a small second kernel in range order; one range: the plain
//           form by four waves, with half-height tiles for a short last round
// 131 x 2560 x 9728 (Q6_K, with the activations' kernel): 33.6 -> 23.2 us, 93 x 6144 x 2048 (Q4_0) 27 -> 14, 700 x 6144 x 2048 43.7 -> 39,
// 2048 x 2048 x 6144 102 -> 80.
struct QLinearPlan {
  int waves;   // form of launch_q_waves, or -1
  int halves;
  int ranges;
};
static int g_q_gemm_form = 0;  // mllm_hip_q_gemm_set_form
static bool q_ranges_exist(int64_t N, int64_t blocks, int z) {  // whole even ranges, none of them empty
  const int64_t per = ((blocks + z - 1) / z + 1) / 2 * 2;
  return z == 1 || (N % 4 == 0 && (blocks + per - 1) / per == z);
}
// What each form is expected to take, in us with the activations' kernel, fitted per format to 340 shapes each (random, 33 to 2048 rows,
// weights of 512 to 9728 either way; the rms errors stand in the table).  Over 1360 such shapes the form chosen takes 1.005 times the best
// form's time on average (19 % more at worst) and is more than 2 % slower than the one range or the ranges by rows and columns alone that
// ran before in 5 of them (595 x 1016 x 8704 Q4_K 37.4 -> 39.3 us at most); from 33 to 4096 rows of up to 151 936 channels 3 of 520 (404 x
// 17776 x 512 Q4_K 29.3 -> 32.9).  The costs of ranges are those of four waves; eight take 0.95 of them.  With one table for all formats, K products and ragged last tiles at a price, a choice was up to 18 %
// slower than those (63 x 9328 x 8704 Q6_K 41.4 -> 48.9, 345 x 1480 x 8704 Q6_K 33.9 -> 39.1, 424 x 6432 x 5376 Q4_K 56.2 -> 63.3).
struct QFormCost {
  float waves[3][6];  // per form: how a partly filled last round counts, fixed, round, round and 64 of K, 1e6 M K (read again by every
  float halves[6];    // column tile), 1e6 M N
  float eight;        // 64 of K less in the third of the waves' forms where it runs by eight waves (fitted to 34 shapes each, 1.3 to 2.6 % rms)
  float ranges[8];    // two workgroups on a CU, part of a last round; fixed, round, round and 64 of K, M K, M N, M N per partial result
};
static const QFormCost& q_form_cost(int wtype) {
  static const QFormCost cost[] = {
      {{{0.75f, 5.194f, 0.7106f, 0.0662f, 3.222f, 0.06239f},
        {0.75f, 5.554f, 0.1751f, 0.1086f, 1.942f, 1.997f},
        {0.5f, 6.718f, 0.f, 0.1817f, 1.876f, 1.659f}},
       {1.f, 8.318f, 0.3028f, 0.6705f, 0.6885f, 1.894f},
       0.0238f,
       {1.5f, 0.5f, 11.4f, 0.005467f, 0.7897f, 1.398f, 0.7408f, 1.058f}},  // Q4_0: 4 / 4 / 5 / 4 / 6 %
      {{{0.75f, 5.465f, 0.4136f, 0.0751f, 3.046f, 1.154f},
        {1.f, 5.928f, 0.f, 0.1192f, 1.86f, 2.248f},
        {0.5f, 7.359f, 0.f, 0.2f, 1.889f, 1.413f}},
       {1.f, 6.389f, 2.611f, 0.6195f, 1.174f, 1.848f},
       0.0234f,
       {1.6f, 0.5f, 11.23f, 0.f, 0.7656f, 1.514f, 0.6784f, 1.075f}},  // Q8_0: 4 / 4 / 5 / 7 / 7 %
      {{{0.75f, 5.412f, 0.5444f, 0.06797f, 3.148f, 0.8011f},
        {1.f, 5.739f, 0.04121f, 0.1086f, 1.952f, 2.302f},
        {0.5f, 7.01f, 0.f, 0.1872f, 1.97f, 1.559f}},
       {1.f, 10.17f, 0.05216f, 0.6293f, 0.906f, 1.662f},
       0.025f,
       {1.5f, 0.75f, 12.58f, 0.f, 0.763f, 1.45f, 0.7756f, 1.005f}},  // Q4_K: 3 / 3 / 5 / 4 / 6 %
      {{{1.f, 4.986f, 0.6891f, 0.08025f, 3.059f, 2.38f},
        {1.f, 6.076f, 0.f, 0.1191f, 1.771f, 2.268f},
        {0.5f, 7.235f, 0.f, 0.2001f, 1.852f, 1.482f}},
       {1.f, 2.535f, 7.217f, 0.6381f, 1.067f, 1.459f},
       0.0193f,
       {1.7f, 0.5f, 12.05f, 0.f, 0.7532f, 1.344f, 0.6954f, 1.035f}},  // Q6_K: 4 / 3 / 5 / 4 / 6 %
  };
  return cost[wtype == MLLM_HIP_Q4_0 ? 0 : wtype == MLLM_HIP_Q8_0 ? 1 : wtype == MLLM_HIP_Q4_K ? 2 : 3];
}
static QLinearPlan q_linear_plan(int wtype, int64_t M, int64_t N, int64_t K, bool ranges_fit) {
  const int64_t blocks = (K + 63) / 64, cols = (N + 255) / 256, tilesM = (M + QG_TILE_H - 1) / QG_TILE_H;
  if (g_q_gemm_form) {
    const int z = g_q_gemm_form - 4;
    return g_q_gemm_form <= 3 ? QLinearPlan{g_q_gemm_form - 1, 0, 1} : z == 0 ? QLinearPlan{-1, 1, 1}
           : QLinearPlan{-1, 0, ranges_fit && q_ranges_exist(N, blocks, z) ? z : 1};
  }
  const QFormCost& c = q_form_cost(wtype);
  const float mk = (float)M * (float)K * 1e-6f, mn = (float)M * (float)N * 1e-6f;
  QLinearPlan best{-1, 0, 1};
  float least = 0.f;
  auto offer = [&](float cost, const QLinearPlan& p) {
    if (least == 0.f || cost < least) {
      least = cost;
      best = p;
    }
  };
  auto whole = [&](const float* f, float full, float part) {  // one workgroup on a CU at a time, or as good as
    const float rounds = f[0] * full + (1.f - f[0]) * std::max(1.f, part);
    return f[1] + rounds * (f[2] + f[3] * (float)blocks) + f[4] * mk + f[5] * mn;
  };
  static const int rows[3] = {32, 32, 64}, chans[3] = {32, 64, 64};
  for (int f = 0; f < 3; f++) {
    const int64_t tiles = ((M + rows[f] - 1) / rows[f]) * ((N + chans[f] - 1) / chans[f]);
    const float cost = whole(c.waves[f], (float)((tiles + 255) / 256), (float)tiles / 256.f);
    // (activation rows that straddle cache lines and lie within 256 bytes of a multiple of 16 KB apart share a few of the caches' sets, twice the lines each: with
    // more than 512 rows 64 x 64 takes up to 1.42 of the time of ranges there, 1287 x 712 x 8160 Q4_0 64.3 us / 45.4; K a multiple of 64 0.87)
    const bool crowded = M > 512 && K % 64 != 0 && (2 * K + 256) % 16384 <= 512;
    const float eight = f == 2 && wk_eight(M, N, blocks) ? c.eight * (float)blocks - (crowded ? 0.4f * cost : 0.f) : 0.f;
    offer(cost - eight, QLinearPlan{f, 0, 1});
    // One tile of rows and long K, where the weights' bytes are the bound: ranges by eight waves are faster than their costs, which are those of four, by 6 %, and the
    // longer K is beyond the 9728 that they were fitted to, the more so: nibbles from there on (63 x 9224 x 15 456 Q4_0 43.1 us on 64 x 64, 35.6), bytes from about
    // 17 000 (47 x 15 080 x 18 976 Q8_0 83.2, 76.1; up to 16 000 64 x 64 is 0.91 of ranges).  A margin of 1.06 for all sizes kept ranges for 1400 shapes that were
    // 1.11 of the time of the eight waves on 64 x 64 (130 x 3544 x 5632 Q6_K 29.1 us, 22.5; 256 x 2560 x 9728 Q4_0 34.8, 33.8); without any, 8 shapes of more rows
    // are 3 to 15 % slower, all of K near 8192 (above).
    if (best.waves == 2 && eight > 0.f && M <= 64 && blocks >= 120) {
      const float margin = qg_nibbles(wtype) ? 1.f + 0.0015f * (float)(blocks - 90) : blocks < 260 ? 1.06f : 1.2f;
      least = std::min(cost, margin * least);
    }
  }
  // a ragged last tile of 128 rows runs as 64 or 32
  const int64_t rest = M % QG_TILE_H;
  const float tiles = ((float)(M / QG_TILE_H) + (rest == 0 ? 0.f : rest > 64 ? 1.f : rest > 32 ? 0.7f : 0.5f)) * (float)cols;
  offer(whole(c.halves, ceilf(tiles / 256.f), tiles / 256.f), QLinearPlan{-1, 1, 1});
  for (int z = 1; z <= 8; z++) {
    if (z > 1 && (!ranges_fit || (float)z * mn > 16.f)) break;  // 64 MB of partial results at most
    if (!q_ranges_exist(N, blocks, z)) continue;
    const int64_t per = ((blocks + z - 1) / z + 1) / 2 * 2, t = tilesM * cols * z;
    const float* f = c.ranges;
    const float rounds = t <= 256 ? 1.f : t <= 512 ? f[0] : f[0] * (f[1] * (float)((t + 511) / 512) + (1.f - f[1]) * (float)t / 512.f);
    offer(f[2] + rounds * (f[3] + f[4] * (float)per) + f[5] * mk + f[6] * mn + (z > 1 ? f[7] * (float)(z + 1) * mn : 0.f), QLinearPlan{-1, 0, z});
  }
  return best;
}
// Ranges whose workgroups have a CU each run by eight waves, halves of a range each: one wave per SIMD dequantizes and multiplies in turns.  0.946 of the time
// over 623 shapes that take ranges; more than 256 workgroups share CUs already.  Codes of a byte (less to unpack) on more than 200 CUs in ranges of fewer
// than sixteen blocks, whose halves are as unequal as eight and six: 0.990, up to 1.04 (984 x 816 x 7040 Q8_0 38.1 -> 39.6 us), so they stay with four.
static bool q_ranges_in_halves(int wtype, int64_t M, int64_t N, int64_t K, int ranges) {
  const int64_t groups = ((M + QG_TILE_H - 1) / QG_TILE_H) * ((N + 255) / 256) * ranges;
  if (ranges < 2 || groups > 256) return false;
  const int64_t blocks = (K + 63) / 64, per = ((blocks + ranges - 1) / ranges + 1) / 2 * 2;
  return qg_nibbles(wtype) || groups <= 200 || per >= 16;
}
size_t qg_partial_bytes(int wtype, int64_t M, int64_t N, int64_t K) {  // the same for both types of a call (their plans may differ)
  const bool kq = wtype == MLLM_HIP_Q4_K || wtype == MLLM_HIP_Q6_K;
  const int z = std::max(q_linear_plan(kq ? MLLM_HIP_Q4_K : MLLM_HIP_Q4_0, M, N, K, true).ranges,
                         q_linear_plan(kq ? MLLM_HIP_Q6_K : MLLM_HIP_Q8_0, M, N, K, true).ranges);
  return z > 1 ? align_up((size_t)z * M * N * 4, 256) : 0;
}

int qg_linear_run(int wtype, const void* gemm_packed, const uint16_t* xh, const float* bias, float* y, int64_t M, int64_t N,
                  int64_t K, void* partial_ws, hipStream_t st) {
  const QLinearPlan plan = q_linear_plan(wtype, M, N, K, partial_ws != nullptr);
  if (plan.waves >= 0) {
    const QWavesArgs w{reinterpret_cast<const char*>(gemm_packed), xh, bias, y, (int)M, (int)N, (int)K};
    switch (wtype) {
      case MLLM_HIP_Q4_0: return launch_q_waves<MLLM_HIP_Q4_0>(plan.waves, w, st);
      case MLLM_HIP_Q8_0: return launch_q_waves<MLLM_HIP_Q8_0>(plan.waves, w, st);
      case MLLM_HIP_Q4_K: return launch_q_waves<MLLM_HIP_Q4_K>(plan.waves, w, st);
      default: return launch_q_waves<MLLM_HIP_Q6_K>(plan.waves, w, st);
    }
  }
  QG2Args a{};
  a.W0 = a.W1 = reinterpret_cast<const char*>(gemm_packed);
  a.wstride = 0;
  a.xh = xh; a.a_index = nullptr; a.a_div = 1; a.a_rows = (int)M;
  a.o_index = nullptr; a.out = y; a.bias = bias;
  a.N = (int)N; a.K = (int)K; a.wtype = wtype; a.x86_scale = 0;
  a.ksplit = plan.ranges;
  a.halves = plan.halves || q_ranges_in_halves(wtype, M, N, K, plan.ranges);
  a.partial = reinterpret_cast<float*>(partial_ws);
  const int64_t tilesM = (M + QG_TILE_H - 1) / QG_TILE_H, cols = (N + 255) / 256, total = tilesM * cols;
  a.big_cols = (int)cols;
  const int64_t last = total % QG_SLOTS;
  if (a.ksplit <= 1 && !a.halves && total > QG_SLOTS && total < 4 * QG_SLOTS && last && last < QG_SLOTS / 4) {
    // A last round that is less than a quarter full: the columns whose full tiles fill whole rounds, the others as half-height tiles (such
    // a tile takes about 0.6 of a full one: it dequantizes the same weights for half the rows).  Over 180 shapes of 513 to 2600 tiles: 0.89
    // to 0.99 of the time there, 1.01 to 1.09 where the last round is fuller, 0.93 to 1.06 from four rounds on.
    a.big_cols = (int)(total / QG_SLOTS * QG_SLOTS / tilesM);
  }
  const int rc = launch_qg<0>(a, (unsigned)tilesM, st);
  if (rc || a.ksplit <= 1) return rc;
  hipLaunchKernelGGL(qg_reduce_kernel, dim3((unsigned)((M * N / 4 + 255) / 256)), dim3(256), 0, st, a.partial, a.ksplit, M * N, (int)N, bias, y);
  return (int)hipGetLastError();
}

}  // namespace mllmhip

using namespace mllmhip;

// =========================================================================================================
// C ABI
// =========================================================================================================
// rows up to which mllm_hip_linear_q runs as passes of the eight-row GEMV
constexpr int64_t LINEAR_Q_GEMV_ROWS = 16;
MLLM_API size_t mllm_hip_linear_q_workspace_bytes(int64_t M, int64_t K) {
  if (M <= 0 || K <= 0 || K % QK) return 0;
  Carver c(nullptr);
  c.take<int8_t>((size_t)M * K);
  c.take<float>((size_t)M * (K / QK));
  carve_route(c, 1, M);
  // short batches run as passes of the decode GEMV, which keeps the quantized image of eight rows here
  const size_t gemv = M <= LINEAR_Q_GEMV_ROWS ? mllm_hip_gemv_workspace_bytes(8, K) : 0;
  return c.used > gemv ? c.used : gemv;
}

MLLM_API int mllm_hip_linear_q(int wtype, const void* packed, const void* x, int x_dtype, const float* bias, float* y,
                               int64_t M, int64_t N, int64_t K, int act_scale_mode, void* workspace, void* stream) {
  if ((wtype != MLLM_HIP_Q4_0 && wtype != MLLM_HIP_Q8_0) || !packed || !x || !y || !workspace || M <= 0 || N <= 0 || K <= 0)
    return MLLM_HIP_E_BADARG;
  if (x_dtype != MLLM_HIP_F32 && x_dtype != MLLM_HIP_BF16) return MLLM_HIP_E_BADARG;
  if (act_scale_mode != MLLM_HIP_SCALE_IEEE && act_scale_mode != MLLM_HIP_SCALE_X86_REF) return MLLM_HIP_E_BADARG;
  if (K % QK || M * K >= ((int64_t)1 << 32) || N > INT32_MAX) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(workspace) % 16 || reinterpret_cast<uintptr_t>(packed) % 16)
    return MLLM_HIP_E_ALIGN;
  hipStream_t st = (hipStream_t)stream;
  if (M <= LINEAR_Q_GEMV_ROWS) {
    // same block arithmetic, the weights streamed once per eight rows: measured against the tile kernel below on the
    // Qwen3-4B projections, 16 rows: 15-22 us against 40-127 (the tile kernel's workgroup is one row tile x 128 channels
    // whatever the row count, and walks all of K alone)
    const mllm_hip_gemv_part part{packed, bias, y, N};
    return mllm_hip_linear_q_gemv_multi_wsn(wtype, 1, &part, x, x_dtype, (int)M, K, act_scale_mode, workspace,
                                            mllm_hip_gemv_workspace_bytes(8, K), stream);
  }
  Carver c(workspace);
  int8_t* aq = c.take<int8_t>((size_t)M * K);
  float* ad = c.take<float>((size_t)M * (K / QK));
  RouteOut ro = carve_route(c, 1, M);
  const int64_t nblocks = M * (K / QK);
  hipLaunchKernelGGL(quant_rows_kernel, dim3((unsigned)((nblocks + 127) / 128)), dim3(128), 0, st, x, x_dtype, aq, ad, nblocks,
                     act_scale_mode == MLLM_HIP_SCALE_X86_REF);
  RC_RET(launch_identity_tiles(M, TOK_TILE, ro, st));
  QGemmArgs a{};
  a.W0 = a.W1 = reinterpret_cast<const char*>(packed);
  a.wstride = 0;
  a.aq = aq; a.ad = ad; a.a_index = nullptr; a.a_div = 1; a.a_rows = (int)M;
  a.o_index = nullptr; a.out = y; a.bias = bias;
  a.tile_expert = ro.tile_expert; a.tile_row0 = ro.tile_row0; a.tile_rows = ro.tile_rows; a.ntiles = ro.ntiles;
  a.N = (int)N; a.K = (int)K; a.x86_scale = act_scale_mode == MLLM_HIP_SCALE_X86_REF;
  return launch_tiles<0>(wtype, a, (unsigned)((M + TOK_TILE - 1) / TOK_TILE), st);
}

// decode path (moe_decode.hip): up to eight tokens as GEMVs, two launches
namespace mllmhip {
size_t moe_decode_workspace_bytes(int64_t T, int64_t I, int k);
bool moe_decode_applies(int64_t T, int64_t H, int64_t I, int E, int k);
int moe_decode_set_tokens(int tokens);
bool moe_rows_applies(int64_t T, int64_t H, int64_t I, int E, int k);
int moe_rows_set_tokens(int tokens);
int moe_rows_tile();
int launch_moe_rows(int wtype, const void* gate, const void* up, const void* down, const void* x, int x_dtype, const int* tile_expert,
                    const int* tile_row0, const int* tile_rows, const int* ntiles, const int* sorted_idx, void* img, float* per,
                    int64_t T, int64_t H, int64_t I, int E, int k, int x86, unsigned max_tiles, hipStream_t st);

// workspace of the row-tile path: images of h, one down result per pair, routing with tiles of moe_rows_tile() rows
struct RowsCarve {
  unsigned char* img;
  float* per;
  RouteOut ro;
};
static RowsCarve carve_rows(Carver& c, int64_t T, int64_t H, int64_t I, int E, int k) {
  RowsCarve r;
  r.img = c.take<unsigned char>(moe_decode_workspace_bytes(T, I, k));
  r.per = c.take<float>((size_t)T * k * H);
  r.ro = carve_route(c, E, T * k, moe_rows_tile());
  return r;
}
int launch_moe_decode(int wtype, const void* gate, const void* up, const void* down, const void* x, int x_dtype, const int32_t* ids,
                      const float* w, float* y, int64_t T, int64_t H, int64_t I, int E, int k, int x86, void* workspace,
                      hipStream_t st);
}  // namespace mllmhip

MLLM_API size_t mllm_hip_moe_workspace_bytes(int64_t T, int64_t H, int64_t I, int E, int k) {
  if (T <= 0 || H <= 0 || I <= 0 || E <= 0 || k <= 0 || H % QK || I % QK) return 0;
  Carver c(nullptr);
  c.take<int8_t>((size_t)T * H);
  c.take<float>((size_t)T * (H / QK));
  c.take<int8_t>((size_t)T * k * I);
  c.take<float>((size_t)T * k * (I / QK));
  c.take<float>((size_t)T * k * H);
  carve_route(c, E, T * k);
  // whichever path the call then takes
  const size_t decode = moe_decode_workspace_bytes(T, I, k);
  Carver cr(nullptr);
  carve_rows(cr, T, H, I, E, k);
  const size_t most = c.used > cr.used ? c.used : cr.used;
  return most > decode ? most : decode;
}

MLLM_API int mllm_hip_moe_set_tuning(int pair_tokens, int row_tokens) {
  if (pair_tokens < 0 || pair_tokens > 4096 || row_tokens < 0 || row_tokens > 65536) return MLLM_HIP_E_BADARG;
  moe_decode_set_tokens(pair_tokens);
  moe_rows_set_tokens(row_tokens);
  return 0;
}

MLLM_API int mllm_hip_moe_route(const int32_t* topk_ids, int64_t T, int E, int k, int32_t* counts, int32_t* offsets,
                                int32_t* sorted_idx, void* workspace, void* stream) {
  if (!topk_ids || !workspace || T <= 0 || E <= 0 || k <= 0) return MLLM_HIP_E_BADARG;
  hipStream_t st = (hipStream_t)stream;
  Carver c(workspace);
  RouteOut ro = carve_route(c, E, T * k);
  RC_RET(launch_route(topk_ids, T * k, E, TOK_TILE, ro, st));
  if (counts) HIP_RET(hipMemcpyAsync(counts, ro.counts, E * sizeof(int), hipMemcpyDeviceToDevice, st));
  if (offsets) HIP_RET(hipMemcpyAsync(offsets, ro.offsets, (E + 1) * sizeof(int), hipMemcpyDeviceToDevice, st));
  if (sorted_idx) HIP_RET(hipMemcpyAsync(sorted_idx, ro.sorted_idx, T * k * sizeof(int), hipMemcpyDeviceToDevice, st));
  return 0;
}

MLLM_API int mllm_hip_moe_ffn_q(int wtype, const void* gate_packed, const void* up_packed, const void* down_packed,
                                const void* x, int x_dtype, const int32_t* topk_ids, const float* topk_w, float* y,
                                int64_t T, int64_t H, int64_t I, int E, int k, int act_scale_mode, void* workspace,
                                void* stream) {
  if ((wtype != MLLM_HIP_Q4_0 && wtype != MLLM_HIP_Q8_0) || !gate_packed || !up_packed || !down_packed || !x || !topk_ids ||
      !topk_w || !y || !workspace || T <= 0 || E <= 0 || k <= 0)
    return MLLM_HIP_E_BADARG;
  if (x_dtype != MLLM_HIP_F32 && x_dtype != MLLM_HIP_BF16) return MLLM_HIP_E_BADARG;
  if (act_scale_mode != MLLM_HIP_SCALE_IEEE && act_scale_mode != MLLM_HIP_SCALE_X86_REF) return MLLM_HIP_E_BADARG;
  if (H <= 0 || I <= 0 || H % QK || I % QK || E > MOE_MAX_EXPERTS) return MLLM_HIP_E_SHAPE;
  if (T * H >= ((int64_t)1 << 32) || T * k * I >= ((int64_t)1 << 32) || T * k > INT32_MAX) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(workspace) % 16 || reinterpret_cast<uintptr_t>(y) % 16) return MLLM_HIP_E_ALIGN;
  hipStream_t st = (hipStream_t)stream;
  const int x86 = act_scale_mode == MLLM_HIP_SCALE_X86_REF;
  // few pairs per expert: every (token, expert) pair is one GEMV row; two launches instead of five
  if (moe_decode_applies(T, H, I, E, k))
    return launch_moe_decode(wtype, gate_packed, up_packed, down_packed, x, x_dtype, topk_ids, topk_w, y, T, H, I, E, k, x86, workspace, st);
  // a few pairs per expert: the pairs sorted by expert, tiles of eight rows that share the expert's weights
  if (moe_rows_applies(T, H, I, E, k)) {
    Carver cr(workspace);
    RowsCarve rc = carve_rows(cr, T, H, I, E, k);
    const unsigned max_tiles = (unsigned)(E + (T * k) / moe_rows_tile() + 1);
    RC_RET(launch_route(topk_ids, T * k, E, moe_rows_tile(), rc.ro, st));
    int r = launch_moe_rows(wtype, gate_packed, up_packed, down_packed, x, x_dtype, rc.ro.tile_expert, rc.ro.tile_row0, rc.ro.tile_rows,
                            rc.ro.ntiles, rc.ro.sorted_idx, rc.img, rc.per, T, H, I, E, k, x86, max_tiles, st);
    if (r) return r;
    const int64_t total = T * H;
    hipLaunchKernelGGL(moe_combine_kernel, dim3((unsigned)((total / 4 + 255) / 256)), dim3(256), 0, st, rc.per, topk_w, topk_ids, y, T,
                       (int)H, k, E);
    return (int)hipGetLastError();
  }
  Carver c(workspace);
  int8_t* xq = c.take<int8_t>((size_t)T * H);
  float* xd = c.take<float>((size_t)T * (H / QK));
  int8_t* hq = c.take<int8_t>((size_t)T * k * I);
  float* hd = c.take<float>((size_t)T * k * (I / QK));
  float* per = c.take<float>((size_t)T * k * H);
  RouteOut ro = carve_route(c, E, T * k);
  const unsigned max_tiles = (unsigned)(E + (T * k) / TOK_TILE + 1);

  RC_RET(launch_route(topk_ids, T * k, E, TOK_TILE, ro, st));
  const int64_t nblocks = T * (H / QK);
  hipLaunchKernelGGL(quant_rows_kernel, dim3((unsigned)((nblocks + 127) / 128)), dim3(128), 0, st, x, x_dtype, xq, xd, nblocks, x86);

  QGemmArgs a{};
  a.tile_expert = ro.tile_expert; a.tile_row0 = ro.tile_row0; a.tile_rows = ro.tile_rows; a.ntiles = ro.ntiles;
  a.x86_scale = x86;
  // gate & up -> silu(g)*u -> Q8_0, rows in expert-sorted order
  a.W0 = reinterpret_cast<const char*>(gate_packed);
  a.W1 = reinterpret_cast<const char*>(up_packed);
  a.wstride = packed_bytes(wtype, I, H);
  a.aq = xq; a.ad = xd; a.a_index = ro.sorted_idx; a.a_div = k; a.a_rows = (int)T;
  a.hq = hq; a.hd = hd;
  a.N = (int)I; a.K = (int)H;
  int rc = launch_tiles<1>(wtype, a, max_tiles, st);
  if (rc) return rc;
  // down -> per-(token, slot) rows
  a.W0 = a.W1 = reinterpret_cast<const char*>(down_packed);
  a.wstride = packed_bytes(wtype, H, I);
  a.aq = hq; a.ad = hd; a.a_index = nullptr; a.a_div = 1; a.a_rows = (int)(T * k);
  a.o_index = ro.sorted_idx; a.out = per; a.bias = nullptr; a.hq = nullptr; a.hd = nullptr;
  a.N = (int)H; a.K = (int)I;
  rc = launch_tiles<0>(wtype, a, max_tiles, st);
  if (rc) return rc;
  const int64_t total = T * H;
  hipLaunchKernelGGL(moe_combine_kernel, dim3((unsigned)((total / 4 + 255) / 256)), dim3(256), 0, st, per, topk_w, topk_ids, y, T,
                     (int)H, k, E);
  return (int)hipGetLastError();
}

// ---- matrix-core path (gemm-packed weights) -------------------------------------------------------------------
MLLM_API size_t mllm_hip_q_gemm_packed_bytes(int wtype, int64_t N, int64_t K) {
  if ((wtype != MLLM_HIP_Q4_0 && wtype != MLLM_HIP_Q8_0) || N <= 0 || K <= 0 || K % QK) return 0;
  return (size_t)qg_bytes(wtype, N, K);
}

MLLM_API int mllm_hip_q_gemm_prepack(int wtype, const void* blocks, int weight_scale_mode, void* packed, int64_t N, int64_t K,
                                     void* stream) {
  if ((wtype != MLLM_HIP_Q4_0 && wtype != MLLM_HIP_Q8_0) || !blocks || !packed || N <= 0 || K <= 0) return MLLM_HIP_E_BADARG;
  if (weight_scale_mode != MLLM_HIP_SCALE_IEEE && weight_scale_mode != MLLM_HIP_SCALE_X86_REF) return MLLM_HIP_E_BADARG;
  if (K % QK || N > INT32_MAX || K > INT32_MAX || qg_bytes(wtype, N, K) >= ((int64_t)1 << 32)) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(packed) % 16) return MLLM_HIP_E_ALIGN;
  hipStream_t st = (hipStream_t)stream;
  const int64_t words = qg_qbytes(wtype, N, K) / 4, count = qg_np(N) * (qg_kp(K) / 64);
  const unsigned char* b = reinterpret_cast<const unsigned char*>(blocks);
  uint32_t* q = reinterpret_cast<uint32_t*>(packed);
  uint32_t* sc = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(packed) + qg_qbytes(wtype, N, K));
  const int x86 = weight_scale_mode == MLLM_HIP_SCALE_X86_REF;
  if (wtype == MLLM_HIP_Q4_0) {
    hipLaunchKernelGGL(qg_prepack_q_kernel<MLLM_HIP_Q4_0>, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, st, b, q, (int)N, (int)K, words);
    hipLaunchKernelGGL(qg_prepack_s_kernel<MLLM_HIP_Q4_0>, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, b, sc, (int)N, (int)K, x86, count);
  } else {
    hipLaunchKernelGGL(qg_prepack_q_kernel<MLLM_HIP_Q8_0>, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, st, b, q, (int)N, (int)K, words);
    hipLaunchKernelGGL(qg_prepack_s_kernel<MLLM_HIP_Q8_0>, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, b, sc, (int)N, (int)K, x86, count);
  }
  return (int)hipGetLastError();
}

MLLM_API int mllm_hip_q_gemm_set_form(int form) {
  if (form < 0 || form > 12) return MLLM_HIP_E_BADARG;
  g_q_gemm_form = form;
  return 0;
}
MLLM_API int mllm_hip_q_gemm_form(int wtype, int64_t M, int64_t N, int64_t K, int short_call) {
  if (wtype != MLLM_HIP_Q4_0 && wtype != MLLM_HIP_Q8_0 && wtype != MLLM_HIP_Q4_K && wtype != MLLM_HIP_Q6_K) return 0;
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const QLinearPlan p = q_linear_plan(wtype, M, N, K, short_call && qg_partial_bytes(wtype, M, N, K));
  return p.waves >= 0 ? 1 + p.waves : p.halves ? 4 : 4 + p.ranges;
}
MLLM_API int mllm_hip_q_gemm_eight(int wtype, int64_t M, int64_t N, int64_t K, int short_call) {
  if (mllm_hip_q_gemm_form(wtype, M, N, K, short_call) == 0) return 0;
  const QLinearPlan p = q_linear_plan(wtype, M, N, K, short_call && qg_partial_bytes(wtype, M, N, K));
  return p.waves >= 0 ? p.waves < 2 || wk_eight(M, N, (K + 63) / 64) : p.halves || q_ranges_in_halves(wtype, M, N, K, p.ranges);
}

MLLM_API size_t mllm_hip_linear_q_gemm_workspace_bytes(int64_t M, int64_t K) {
  if (M <= 0 || K <= 0 || K % QK) return 0;
  Carver c(nullptr);
  c.take<uint16_t>((size_t)M * K);
  return c.used;
}

MLLM_API int mllm_hip_linear_q_gemm(int wtype, const void* gemm_packed, const void* x, int x_dtype, const float* bias,
                                    float* y, int64_t M, int64_t N, int64_t K, int act_scale_mode, void* workspace,
                                    void* stream) {
  if ((wtype != MLLM_HIP_Q4_0 && wtype != MLLM_HIP_Q8_0) || !gemm_packed || !x || !y || !workspace || M <= 0 || N <= 0 || K <= 0)
    return MLLM_HIP_E_BADARG;
  if (x_dtype != MLLM_HIP_F32 && x_dtype != MLLM_HIP_BF16) return MLLM_HIP_E_BADARG;
  if (act_scale_mode != MLLM_HIP_SCALE_IEEE && act_scale_mode != MLLM_HIP_SCALE_X86_REF) return MLLM_HIP_E_BADARG;
  if (K % QK || M * K * 2 >= ((int64_t)1 << 32) || N > INT32_MAX || qg_bytes(wtype, N, K) >= ((int64_t)1 << 32)) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(workspace) % 16 ||
      reinterpret_cast<uintptr_t>(gemm_packed) % 16 || reinterpret_cast<uintptr_t>(y) % 16)
    return MLLM_HIP_E_ALIGN;
  hipStream_t st = (hipStream_t)stream;
  Carver c(workspace);
  uint16_t* xh = c.take<uint16_t>((size_t)M * K);
  const int64_t nblocks = M * (K / QK);
  hipLaunchKernelGGL(qg_act_kernel, dim3((unsigned)((nblocks + 63) / 64)), dim3(256), 0, st, x, x_dtype, xh,
                     (uint16_t*)nullptr, nblocks, act_scale_mode == MLLM_HIP_SCALE_X86_REF);
  return qg_linear_run(wtype, gemm_packed, xh, bias, y, M, N, K, nullptr, st);
}

// the same with room for the partial results of K ranges (behind the activations, on a 256-byte line of their own)
MLLM_API size_t mllm_hip_linear_q_gemm_short_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0 || K % QK) return 0;
  return align_up(mllm_hip_linear_q_gemm_workspace_bytes(M, K), 256) + 256 + qg_partial_bytes(MLLM_HIP_Q4_0, M, N, K);
}
MLLM_API int mllm_hip_linear_q_gemm_short(int wtype, const void* gemm_packed, const void* x, int x_dtype, const float* bias, float* y,
                                          int64_t M, int64_t N, int64_t K, int act_scale_mode, void* workspace, void* stream) {
  if ((wtype != MLLM_HIP_Q4_0 && wtype != MLLM_HIP_Q8_0) || !gemm_packed || !x || !y || !workspace || M <= 0 || N <= 0 || K <= 0)
    return MLLM_HIP_E_BADARG;
  if (x_dtype != MLLM_HIP_F32 && x_dtype != MLLM_HIP_BF16) return MLLM_HIP_E_BADARG;
  if (act_scale_mode != MLLM_HIP_SCALE_IEEE && act_scale_mode != MLLM_HIP_SCALE_X86_REF) return MLLM_HIP_E_BADARG;
  if (K % QK || M * K * 2 >= ((int64_t)1 << 32) || N > INT32_MAX || qg_bytes(wtype, N, K) >= ((int64_t)1 << 32)) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(workspace) % 256 ||
      reinterpret_cast<uintptr_t>(gemm_packed) % 16 || reinterpret_cast<uintptr_t>(y) % 16)
    return MLLM_HIP_E_ALIGN;
  hipStream_t st = (hipStream_t)stream;
  Carver c(workspace);
  uint16_t* xh = c.take<uint16_t>((size_t)M * K);
  const int64_t nblocks = M * (K / QK);
  hipLaunchKernelGGL(qg_act_kernel, dim3((unsigned)((nblocks + 63) / 64)), dim3(256), 0, st, x, x_dtype, xh,
                     (uint16_t*)nullptr, nblocks, act_scale_mode == MLLM_HIP_SCALE_X86_REF);
  void* partial = qg_partial_bytes(MLLM_HIP_Q4_0, M, N, K) ? c.p + align_up(mllm_hip_linear_q_gemm_workspace_bytes(M, K), 256) : nullptr;
  return qg_linear_run(wtype, gemm_packed, xh, bias, y, M, N, K, partial, st);
}

namespace mllmhip {
struct QXCarve {
  uint8_t* xq;
  uint32_t* xd;
  uint8_t* hq;
  uint32_t* hd;
  float* per;
  RouteOut ro;
};
static QXCarve carve_qx(Carver& c, int64_t T, int64_t H, int64_t I, int E, int k) {
  QXCarve r;
  r.xq = c.take<uint8_t>((size_t)T * H);
  r.xd = c.take<uint32_t>((size_t)T * ((H + 63) / 64));
  r.hq = c.take<uint8_t>((size_t)T * k * I);
  r.hd = c.take<uint32_t>((size_t)T * k * ((I + 63) / 64));
  r.per = c.take<float>((size_t)T * k * H);
  r.ro = carve_route(c, E, T * k, QX_TILE_H);
  return r;
}
// 0: exact block sums (qx_kernel); 1: fp16 operands with the block scales folded in (qg_kernel); 2: as 0 with every tile in
// the 32-row form (the comparison for the 16-row form: same bits)
static int g_moe_gemm_path = 0;
}  // namespace mllmhip

MLLM_API int mllm_hip_moe_gemm_set_path(int path) {
  if (path < 0 || path > 2) return MLLM_HIP_E_BADARG;
  g_moe_gemm_path = path;
  return 0;
}

// The grouped expert FFN with the reference's own block arithmetic on the matrix cores (qx_kernel): route, quantize x,
// gate + up + SiLU * up + re-quantization in one launch, down, weighted sum in slot order.
static int moe_ffn_qx(int wtype, const void* gate_packed, const void* up_packed, const void* down_packed, const void* x, int x_dtype,
                      const int32_t* topk_ids, const float* topk_w, float* y, int64_t T, int64_t H, int64_t I, int E, int k, int x86,
                      void* workspace, hipStream_t st) {
  Carver c(workspace);
  QXCarve w = carve_qx(c, T, H, I, E, k);
  const unsigned max_tiles = (unsigned)(E + (T * k) / QX_TILE_H + 1);
  if (E > MOE_MAX_EXPERTS) return MLLM_HIP_E_SHAPE;
  const int64_t nblocks = T * (H / QK);
  const auto prepare = wtype == MLLM_HIP_Q4_0 ? qx_prepare_kernel<MLLM_HIP_Q4_0> : qx_prepare_kernel<MLLM_HIP_Q8_0>;
  hipLaunchKernelGGL(prepare, dim3((unsigned)(1 + (nblocks + 1023) / 1024)), dim3(1024), 5 * (size_t)E * sizeof(int), st,
                     topk_ids, (int)(T * k), E, QX_TILE_H, w.ro, x, x_dtype, w.xq, w.xd, nblocks, (int)(H / QK), x86);
  HIP_RET(hipGetLastError());
  QXArgs a{};
  a.tile_expert = w.ro.tile_expert; a.tile_row0 = w.ro.tile_row0; a.tile_rows = w.ro.tile_rows; a.ntiles = w.ro.ntiles;
  a.x86_scale = x86;
  a.half_tiles = g_moe_gemm_path != 2;
  a.W0 = reinterpret_cast<const char*>(gate_packed);
  a.W1 = reinterpret_cast<const char*>(up_packed);
  a.wstride = (size_t)qg_bytes(wtype, I, H);
  a.xq = w.xq; a.xd = w.xd; a.a_index = w.ro.sorted_idx; a.a_div = k; a.a_rows = (int)T;
  a.hq = w.hq; a.hd = w.hd;
  a.N = (int)I; a.K = (int)H;
  RC_RET(launch_qx<1>(wtype, a, max_tiles, st));
  a.W0 = a.W1 = reinterpret_cast<const char*>(down_packed);
  a.wstride = (size_t)qg_bytes(wtype, H, I);
  a.xq = w.hq; a.xd = w.hd; a.a_index = nullptr; a.a_div = 1; a.a_rows = (int)(T * k);
  a.o_index = w.ro.sorted_idx; a.out = w.per; a.bias = nullptr; a.hq = nullptr; a.hd = nullptr;
  a.N = (int)H; a.K = (int)I;
  RC_RET(launch_qx<0>(wtype, a, max_tiles, st));
  const int64_t total = T * H;
  hipLaunchKernelGGL(moe_combine_kernel, dim3((unsigned)((total / 4 + 255) / 256)), dim3(256), 0, st, w.per, topk_w, topk_ids, y, T,
                     (int)H, k, E);
  return (int)hipGetLastError();
}

MLLM_API size_t mllm_hip_moe_gemm_workspace_bytes(int64_t T, int64_t H, int64_t I, int E, int k) {
  if (T <= 0 || H <= 0 || I <= 0 || E <= 0 || k <= 0 || H % QK || I % QK) return 0;
  Carver c(nullptr);
  c.take<uint16_t>((size_t)T * H);
  c.take<uint16_t>((size_t)T * H);
  c.take<uint16_t>((size_t)T * k * I);
  c.take<float>((size_t)T * k * H);
  carve_route(c, E, T * k);
  // the exact form: codes as fp16 integers + scale pairs for x and for h, the per-pair rows, routing
  Carver cx(nullptr);
  carve_qx(cx, T, H, I, E, k);
  return c.used > cx.used ? c.used : cx.used;
}

MLLM_API int mllm_hip_moe_ffn_q_gemm(int wtype, const void* gate_packed, const void* up_packed, const void* down_packed,
                                     const void* x, int x_dtype, const int32_t* topk_ids, const float* topk_w, float* y,
                                     int64_t T, int64_t H, int64_t I, int E, int k, int act_scale_mode, void* workspace,
                                     void* stream) {
  if ((wtype != MLLM_HIP_Q4_0 && wtype != MLLM_HIP_Q8_0) || !gate_packed || !up_packed || !down_packed || !x || !topk_ids ||
      !topk_w || !y || !workspace || T <= 0 || E <= 0 || k <= 0)
    return MLLM_HIP_E_BADARG;
  if (x_dtype != MLLM_HIP_F32 && x_dtype != MLLM_HIP_BF16) return MLLM_HIP_E_BADARG;
  if (act_scale_mode != MLLM_HIP_SCALE_IEEE && act_scale_mode != MLLM_HIP_SCALE_X86_REF) return MLLM_HIP_E_BADARG;
  if (H <= 0 || I <= 0 || H % QK || I % QK || E > MOE_MAX_EXPERTS) return MLLM_HIP_E_SHAPE;
  if (T * H * 2 >= ((int64_t)1 << 32) || T * k * I * 2 >= ((int64_t)1 << 32) || T * k > INT32_MAX) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(workspace) % 16 || reinterpret_cast<uintptr_t>(y) % 16) return MLLM_HIP_E_ALIGN;
  hipStream_t st = (hipStream_t)stream;
  const int x86 = act_scale_mode == MLLM_HIP_SCALE_X86_REF;
  if (g_moe_gemm_path != 1)
    return moe_ffn_qx(wtype, gate_packed, up_packed, down_packed, x, x_dtype, topk_ids, topk_w, y, T, H, I, E, k, x86, workspace, st);
  Carver c(workspace);
  uint16_t* xh = c.take<uint16_t>((size_t)T * H);
  uint16_t* xl = c.take<uint16_t>((size_t)T * H);
  uint16_t* hh = c.take<uint16_t>((size_t)T * k * I);
  float* per = c.take<float>((size_t)T * k * H);
  RouteOut ro = carve_route(c, E, T * k);
  const unsigned max_tiles = (unsigned)(E + (T * k) / QG_TILE_H + 1);

  RC_RET(launch_route(topk_ids, T * k, E, QG_TILE_H, ro, st));
  const int64_t nblocks = T * (H / QK);
  hipLaunchKernelGGL(qg_act_kernel, dim3((unsigned)((nblocks + 63) / 64)), dim3(256), 0, st, x, x_dtype, xh, xl, nblocks, x86);

  QG2Args a{};
  a.tile_expert = ro.tile_expert; a.tile_row0 = ro.tile_row0; a.tile_rows = ro.tile_rows; a.ntiles = ro.ntiles;
  a.wtype = wtype; a.x86_scale = x86;
  // gate & up -> silu(g)*u -> Q8_0 round trip in fp16, rows in expert-sorted order
  a.W0 = reinterpret_cast<const char*>(gate_packed);
  a.W1 = reinterpret_cast<const char*>(up_packed);
  a.wstride = (size_t)qg_bytes(wtype, I, H);
  a.xh = xh; a.xl = xl; a.a_index = ro.sorted_idx; a.a_div = k; a.a_rows = (int)T;
  a.hh = hh;
  a.N = (int)I; a.K = (int)H;
  int rc = launch_qg<1>(a, max_tiles, st);
  if (rc) return rc;
  // down -> per-(token, slot) rows
  a.W0 = a.W1 = reinterpret_cast<const char*>(down_packed);
  a.wstride = (size_t)qg_bytes(wtype, H, I);
  a.xh = hh; a.xl = nullptr; a.a_index = nullptr; a.a_div = 1; a.a_rows = (int)(T * k);
  a.o_index = ro.sorted_idx; a.out = per; a.bias = nullptr; a.hh = nullptr;
  a.N = (int)H; a.K = (int)I;
  rc = launch_qg<0>(a, max_tiles, st);
  if (rc) return rc;
  const int64_t total = T * H;
  hipLaunchKernelGGL(moe_combine_kernel, dim3((unsigned)((total / 4 + 255) / 256)), dim3(256), 0, st, per, topk_w, topk_ids, y, T,
                     (int)H, k, E);
  return (int)hipGetLastError();
}

// ---- experts in the super-block formats (kquant.hip) ----------------------------------------------------------------------
// The shipped Qwen3-MoE recipe quantizes the experts to Q4_K / Q6_K.  Every (token, expert) pair is one row of the K-quant
// GEMV: gate and up in one launch (the workgroup quantizes the token's x to Q8_K), silu(g) * u, the down GEMV (quantizing h),
// the weighted sum in slot order.  Three or four launches for any T; the weights of an expert are read once per pair that uses it,
// so this is the decode form.  With more than two pairs per expert the pairs are sorted by expert and run as tiles of eight
// rows on the matrix-core kernels instead (the grouped form).
namespace mllmhip {
int kq_moe_gemv(int wtype, int nparts, const void* const* packed0, float* const* ys, int64_t N, int64_t K, const void* x, int x_dtype,
                const float* x2, const int32_t* ids, int E, int slots, int slot_div, int form, hipStream_t st);
bool kq_moe_groups_fit(int wtype, int64_t rows, int64_t K, int slots);
size_t kq_image_bytes(int64_t rows, int64_t K);
int kq_quantize_image(const void* x, int x_dtype, void* image, int64_t rows, int64_t K, hipStream_t st);
bool kq_moe_tiles_fit(int64_t K);
int kq_moe_tiles_gemv(int wtype, int nparts, const void* const* packed0, float* const* ys, int64_t N, int64_t K, const void* image,
                      int64_t img_rows, const int* tile_expert, const int* tile_row0, const int* tile_rows, const int* ntiles,
                      unsigned max_tiles, const int* row_ids, int row_div, const int* out_ids, hipStream_t st);
bool kx_moe_tiles_fit(int wtype, int64_t N, int64_t K);
int kx_tile_rows();
int kx_moe_tiles(int wtype, int nparts, const void* const* packed0, float* const* ys, int64_t N, int64_t K, const void* image,
                 int64_t img_rows, const int* tile_expert, const int* tile_row0, const int* tile_rows, const int* ntiles,
                 unsigned max_tiles, const int* row_ids, int row_div, const int* out_ids, int silu_mul, hipStream_t st);
// 0: by the number of pairs per expert; 1: always pairs as GEMV rows; 2: always tiles of eight rows; 3: always tiles of 32 rows
// (where the format has them)
static int g_moe_kq_path = 0;
constexpr int KQ_MOE_TILE = 8;
struct KqMoeCarve {
  float *g, *u, *h, *per;
  char *ximg, *himg;
  RouteOut ro;
};
static KqMoeCarve carve_kq_moe(Carver& c, int64_t T, int64_t H, int64_t I, int E, int k) {
  KqMoeCarve r;
  const size_t slots = (size_t)T * k;
  r.g = c.take<float>(slots * I);
  r.u = c.take<float>(slots * I);
  r.h = c.take<float>(slots * I);
  r.per = c.take<float>(slots * H);
  r.ximg = c.take<char>(kq_image_bytes(T, H));
  r.himg = c.take<char>(kq_image_bytes((int64_t)slots, I));
  r.ro = carve_route(c, E, (int64_t)slots, KQ_MOE_TILE);
  return r;
}
}  // namespace mllmhip

MLLM_API int mllm_hip_moe_kq_set_path(int path) {
  if (path < 0 || path > 3) return MLLM_HIP_E_BADARG;
  g_moe_kq_path = path;
  return 0;
}

MLLM_API size_t mllm_hip_moe_kq_workspace_bytes(int64_t T, int64_t H, int64_t I, int E, int k) {
  if (T <= 0 || H <= 0 || I <= 0 || E <= 0 || k <= 0 || H % 256 || I % 256) return 0;
  Carver c(nullptr);
  carve_kq_moe(c, T, H, I, E, k);
  return c.used;
}

MLLM_API int mllm_hip_moe_ffn_kq2(int wtype, int wtype_down, const void* gate_packed, const void* up_packed, const void* down_packed,
                                  const void* x, int x_dtype, const int32_t* topk_ids, const float* topk_w, float* y, int64_t T,
                                  int64_t H, int64_t I, int E, int k, void* workspace, void* stream) {
  if ((wtype != MLLM_HIP_Q4_K && wtype != MLLM_HIP_Q6_K) || (wtype_down != MLLM_HIP_Q4_K && wtype_down != MLLM_HIP_Q6_K) || !gate_packed || !up_packed || !down_packed || !x || !topk_ids ||
      !topk_w || !y || !workspace || T <= 0 || E <= 0 || k <= 0)
    return MLLM_HIP_E_BADARG;
  if (x_dtype != MLLM_HIP_F32 && x_dtype != MLLM_HIP_BF16) return MLLM_HIP_E_BADARG;
  if (H <= 0 || I <= 0 || H % 256 || I % 256 || T * k > 65535) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(workspace) % 16 ||
      reinterpret_cast<uintptr_t>(gate_packed) % 16 || reinterpret_cast<uintptr_t>(up_packed) % 16 ||
      reinterpret_cast<uintptr_t>(down_packed) % 16 || reinterpret_cast<uintptr_t>(y) % 16)
    return MLLM_HIP_E_ALIGN;
  hipStream_t st = (hipStream_t)stream;
  const int slots = (int)(T * k);
  Carver c(workspace);
  const KqMoeCarve w = carve_kq_moe(c, T, H, I, E, k);
  float *g = w.g, *u = w.u, *h = w.h, *per = w.per;
  // More than about one pair per expert (Q6_K: half a pair): the pairs are sorted by expert and run as tiles of eight rows on the matrix-core
  // kernels, so an expert's matrices are streamed once per eight pairs instead of once per pair (the grouped form).
  // x and h are quantized to Q8_K once (bit-exact images), the tiles gather their rows from the images.
  const bool tiles_ok = E <= MOE_MAX_EXPERTS && kq_moe_tiles_fit(H) && kq_moe_tiles_fit(I) &&
                        (size_t)E + (size_t)slots / KQ_MOE_TILE + 1 <= 65535;
  const bool many = (wtype == MLLM_HIP_Q4_K && wtype_down == MLLM_HIP_Q4_K) ? slots > E : 2 * slots > E;
  // Four pairs per expert and more: tiles of 32 rows, weights as the second operand of 32 x 32 matrix instructions (one pass
  // over an expert's weights per 32 pairs, one unpacking per 32 rows).  Same integer arithmetic; silu(gate) * up is formed where
  // the two results leave their kernel (six launches).
  const bool tiles32_ok = E <= MOE_MAX_EXPERTS && kx_moe_tiles_fit(wtype, I, H) && kx_moe_tiles_fit(wtype_down, H, I);
  if (tiles32_ok && (g_moe_kq_path == 3 || (g_moe_kq_path == 0 && slots >= 4 * E))) {
    const int th = kx_tile_rows();
    const unsigned max_tiles = (unsigned)(E + slots / th + 1);
    RC_RET(launch_route(topk_ids, slots, E, th, w.ro, st));
    RC_RET(kq_quantize_image(x, x_dtype, w.ximg, T, H, st));
    const void* gu2[2] = {gate_packed, up_packed};
    float* guy2[2] = {h, u};  // silu(gate) * up, rows in expert-sorted order
    RC_RET(kx_moe_tiles(wtype, 2, gu2, guy2, I, H, w.ximg, T, w.ro.tile_expert, w.ro.tile_row0, w.ro.tile_rows, w.ro.ntiles, max_tiles,
                        w.ro.sorted_idx, k, nullptr, 1, st));
    RC_RET(kq_quantize_image(h, MLLM_HIP_F32, w.himg, slots, I, st));
    const void* dn2[1] = {down_packed};
    float* dny2[1] = {per};  // row t * k + j
    RC_RET(kx_moe_tiles(wtype_down, 1, dn2, dny2, H, I, w.himg, slots, w.ro.tile_expert, w.ro.tile_row0, w.ro.tile_rows, w.ro.ntiles,
                        max_tiles, nullptr, 1, w.ro.sorted_idx, 0, st));
    const int64_t total2 = T * H;
    hipLaunchKernelGGL(moe_combine_kernel, dim3((unsigned)((total2 / 4 + 255) / 256)), dim3(256), 0, st, per, topk_w, topk_ids, y, T,
                       (int)H, k, E);
    return (int)hipGetLastError();
  }
  // Such tiles with 16 pairs to less than one pair per expert: the workgroups find an expert's pairs themselves and take up to
  // eight at a time (kquant_rows.h), without a routing launch; same bits.  Q4_K / Q6_K, 128 experts, top-8, us, sorted tiles / this: 2048 x
  // 768 nine tokens 56.6 / 54.4, twelve 62.3 / 61.8, fifteen 67.6 / 68.8; 1024 x 512 nine 31.5 / 27.2, twelve 33.8 / 30.8
  const bool unsorted = g_moe_kq_path == 0 && tiles_ok && many && slots >= 16 && slots < E && slots <= 512;
  if (tiles_ok && (g_moe_kq_path == 2 || ((g_moe_kq_path == 0 || g_moe_kq_path == 3) && many && !unsorted))) {
    const unsigned max_tiles = (unsigned)(E + slots / KQ_MOE_TILE + 1);
    RC_RET(launch_route(topk_ids, slots, E, KQ_MOE_TILE, w.ro, st));
    RC_RET(kq_quantize_image(x, x_dtype, w.ximg, T, H, st));
    const void* gu2[2] = {gate_packed, up_packed};
    float* guy2[2] = {g, u};  // rows in expert-sorted order
    RC_RET(kq_moe_tiles_gemv(wtype, 2, gu2, guy2, I, H, w.ximg, T, w.ro.tile_expert, w.ro.tile_row0, w.ro.tile_rows, w.ro.ntiles,
                             max_tiles, w.ro.sorted_idx, k, nullptr, st));
    // positions past the last valid pair (invalid expert ids) are never written nor read: the tiles cover offsets[E] rows
    RC_RET(mllm_hip_silu_mul(g, u, h, MLLM_HIP_F32, slots, I, nullptr, MLLM_HIP_SCALE_IEEE, stream));
    RC_RET(kq_quantize_image(h, MLLM_HIP_F32, w.himg, slots, I, st));
    const void* dn2[1] = {down_packed};
    float* dny2[1] = {per};  // row t * k + j
    RC_RET(kq_moe_tiles_gemv(wtype_down, 1, dn2, dny2, H, I, w.himg, slots, w.ro.tile_expert, w.ro.tile_row0, w.ro.tile_rows,
                             w.ro.ntiles, max_tiles, nullptr, 1, w.ro.sorted_idx, st));
    const int64_t total2 = T * H;
    hipLaunchKernelGGL(moe_combine_kernel, dim3((unsigned)((total2 / 4 + 255) / 256)), dim3(256), 0, st, per, topk_w, topk_ids, y, T,
                       (int)H, k, E);
    return (int)hipGetLastError();
  }
  const void* gu[2] = {gate_packed, up_packed};
  float* guy[2] = {g, u};
  auto form = [&](int wt, int64_t rows, int64_t K) {
    return unsorted ? KQ_MOE_TILES : g_moe_kq_path == 0 && kq_moe_groups_fit(wt, rows, K, slots) ? KQ_MOE_GROUPS : KQ_MOE_PAIRS;
  };
  const int form_down = form(wtype_down, H, I);
  int rc = kq_moe_gemv(wtype, 2, gu, guy, I, H, x, x_dtype, nullptr, topk_ids, E, slots, k, form(wtype, 2 * I, H), st);
  if (rc) return rc;
  // silu(g) * u: up to 32 pairs it is formed where the down GEMV reads its activations (same fp32 operations; one launch
  // fewer: one token 17.8 -> 16.4 us); with more pairs every down workgroup reading g and u costs more than the elementwise
  // launch (eight tokens 50 against 48 us), where the workgroups share an expert's pairs from about 128 on
  const void* dn[1] = {down_packed};
  float* dny[1] = {per};
  if (slots <= (form_down != KQ_MOE_PAIRS ? 128 : 32)) {
    rc = kq_moe_gemv(wtype_down, 1, dn, dny, H, I, g, MLLM_HIP_F32, u, topk_ids, E, slots, 1, form_down, st);
  } else {
    rc = mllm_hip_silu_mul(g, u, h, MLLM_HIP_F32, slots, I, nullptr, MLLM_HIP_SCALE_IEEE, stream);
    if (rc) return rc;
    rc = kq_moe_gemv(wtype_down, 1, dn, dny, H, I, h, MLLM_HIP_F32, nullptr, topk_ids, E, slots, 1, form_down, st);
  }
  if (rc) return rc;
  const int64_t total = T * H;
  hipLaunchKernelGGL(moe_combine_kernel, dim3((unsigned)((total / 4 + 255) / 256)), dim3(256), 0, st, per, topk_w, topk_ids, y, T,
                     (int)H, k, E);
  return (int)hipGetLastError();
}

MLLM_API int mllm_hip_moe_ffn_kq(int wtype, const void* gate_packed, const void* up_packed, const void* down_packed, const void* x,
                                 int x_dtype, const int32_t* topk_ids, const float* topk_w, float* y, int64_t T, int64_t H,
                                 int64_t I, int E, int k, void* workspace, void* stream) {
  return mllm_hip_moe_ffn_kq2(wtype, wtype, gate_packed, up_packed, down_packed, x, x_dtype, topk_ids, topk_w, y, T, H, I, E, k, workspace,
                              stream);
}

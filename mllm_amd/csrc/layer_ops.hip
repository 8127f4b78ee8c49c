// The operators either side of a quantized Linear in a decoder layer, for gfx950: RMSNorm, SiLU, elementwise add / mul,
// SiLU(gate) * up, softmax, top-k and the whole MoE gate (logits -> softmax -> top-k -> normalise).
//
// Arithmetic follows the reference's x86 CPU kernels:
//   RMSNorm   mllm/backends/cpu/kernels/x86/rmsnorm.cpp:17-52      y = x * (w * rms), rms = 1 / sqrt(mean(x^2) + eps)
//   SiLU      mllm/backends/cpu/kernels/x86/silu.cpp:16-27         x * (1 / (1 + exp_poly(-x)))
//   exp_poly  mllm/backends/cpu/kernels/x86/math.hpp:19-72         Cephes polynomial
//   softmax   mllm/backends/cpu/kernels/x86/softmax.cpp:18-76      exp_poly(x - max) * (1 / sum); expf for len <= 16
//   top-k     mllm/backends/cpu/ops/TopKOp.cpp:20-72               k extreme values, by value or by index
//   MoE gate  mllm/models/qwen3_moe/modeling_qwen3_moe_fa2.hpp:121-139
// Sums run in a different order than the CPU's vector lanes; everything elementwise is the same fp32 operation
// sequence.
//
// All of these are HBM- or latency-bound.  What they add for this GPU: the kernels that produce the input of a decode
// GEMV (RMSNorm, SiLU*up) can also write that input's Q8_0 image in the form the GEMV kernel copies into LDS, so the
// GEMV of every workgroup skips the quantization.
#include "qcommon.h"

namespace mllmhip {

// `accurate` replaces the polynomial (whose argument reduction, as written in the reference, leaves a relative error of
// about 2.1e-4 per unit of the binary exponent of the result) by expf.
__device__ __forceinline__ float silu_ref(float x, bool accurate) { return x * (1.0f / (1.0f + (accurate ? expf(-x) : exp_poly(-x)))); }

// ---- eight consecutive elements per lane ------------------------------------------------------------------------------
template <int XT>
struct Item8 {
  u32x4 r[XT == MLLM_HIP_F32 ? 2 : 1];
};
template <int XT>
__device__ __forceinline__ void item_load(const void* p, int64_t elem, Item8<XT>& it) {
  if (XT == MLLM_HIP_F32) {
    const u32x4* q = reinterpret_cast<const u32x4*>(reinterpret_cast<const float*>(p) + elem);
    it.r[0] = q[0];
    it.r[XT == MLLM_HIP_F32 ? 1 : 0] = q[1];
  } else {
    it.r[0] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(p) + elem);
  }
}
template <int XT>
__device__ __forceinline__ void item_to_f32(const Item8<XT>& it, float (&v)[8]) {
  if (XT == MLLM_HIP_F32) {
    const u32x4 a = it.r[0], b = it.r[XT == MLLM_HIP_F32 ? 1 : 0];
    v[0] = __uint_as_float(a.x); v[1] = __uint_as_float(a.y); v[2] = __uint_as_float(a.z); v[3] = __uint_as_float(a.w);
    v[4] = __uint_as_float(b.x); v[5] = __uint_as_float(b.y); v[6] = __uint_as_float(b.z); v[7] = __uint_as_float(b.w);
  } else {
    const uint32_t w[4] = {it.r[0].x, it.r[0].y, it.r[0].z, it.r[0].w};
#pragma unroll
    for (int j = 0; j < 4; j++) {
      v[2 * j + 0] = __uint_as_float(w[j] << 16);
      v[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
    }
  }
}
// stores v in the tensor's type and leaves in v what a reader of the tensor will see (bf16: the rounded values)
template <int XT>
__device__ __forceinline__ void item_store(void* p, int64_t elem, float (&v)[8]) {
  if (XT == MLLM_HIP_F32) {
    u32x4* q = reinterpret_cast<u32x4*>(reinterpret_cast<float*>(p) + elem);
    q[0] = u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
    q[1] = u32x4{__float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]), __float_as_uint(v[7])};
  } else {
    u32x4 o = {pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7])};
    *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(p) + elem) = o;
    const uint32_t w[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
    for (int j = 0; j < 4; j++) {
      v[2 * j + 0] = __uint_as_float(w[j] << 16);
      v[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
    }
  }
}

__device__ __forceinline__ float wave_sum(float v) { return group_sum<64>(v); }
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, dpp_f<0xB1>(v));
  v = fmaxf(v, dpp_f<0x4E>(v));
  v = fmaxf(v, dpp_f<0x141>(v));
  v = fmaxf(v, dpp_f<0x140>(v));
  v = max16(v);
  v = max32(v);
  return v;
}

// ---- RMSNorm ----------------------------------------------------------------------------------------------------------
struct RmsArgs {
  const void* x;
  const float* w;
  void* y;
  int64_t rows;
  int D;
  float eps;
  int add_unit_offset;
  QImage img;
};
// One workgroup per row; a lane keeps NI items of eight elements in registers between the two passes.
template <int XT, int NI>
__global__ __launch_bounds__(256) void rmsnorm_kernel(RmsArgs a) {
  __shared__ float s_grp[4 * NI];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t row = blockIdx.x;
  if (row >= a.rows) {  // only launched for the zero rows of an image
    image_zero_row(a.img, (int)row, tid, 256);
    return;
  }
  const int nitems = a.D >> 3;
  Item8<XT> raw[NI];
  Item8<MLLM_HIP_F32> wraw[NI];
#pragma unroll
  for (int k = 0; k < NI; k++) {
    const int it = min(tid + 256 * k, nitems - 1);
    item_load<XT>(a.x, row * a.D + (int64_t)it * 8, raw[k]);
  }
#pragma unroll
  for (int k = 0; k < NI; k++) {
    const int it = min(tid + 256 * k, nitems - 1);
    item_load<MLLM_HIP_F32>(a.w, (int64_t)it * 8, wraw[k]);
  }
  // Sum of squares in a fixed order (per item an fma chain, the 64 items of a group through the wave butterfly, the
  // groups one after the other): a function of the row alone, not of how rows are spread over workgroups.
  float v[NI][8];
#pragma unroll
  for (int k = 0; k < NI; k++) {
    item_to_f32<XT>(raw[k], v[k]);
    float p = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e++) p = fmaf(v[k][e], v[k][e], p);
    p = wave_sum(tid + 256 * k < nitems ? p : 0.f);
    if (lane == 0) s_grp[wave + 4 * k] = p;
  }
  __syncthreads();
  float total = 0.f;  // (groups past the row hold 0)
#pragma unroll
  for (int g = 0; g < 4 * NI; g++) total += s_grp[g];
  const float rms = 1.0f / sqrtf(total / (float)a.D + a.eps);
#pragma unroll
  for (int k = 0; k < NI; k++) {
    const int it = tid + 256 * k;
    const bool valid = it < nitems;
    float wv[8], o[8];
    item_to_f32<MLLM_HIP_F32>(wraw[k], wv);
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float mult = (a.add_unit_offset ? wv[e] + 1.0f : wv[e]) * rms;
      o[e] = valid ? v[k][e] * mult : 0.f;
    }
    if (valid) item_store<XT>(a.y, row * a.D + (int64_t)it * 8, o);
    if (a.img.base) quad_quantize_to_image(o, a.img, (int)row, it >> 2, it & 3, valid);
  }
}

// ---- elementwise: SiLU, SiLU(gate) * up, add, mul ---------------------------------------------------------------------
enum { EW_SILU = 0, EW_SILU_MUL = 1, EW_ADD = 2, EW_MUL = 3 };
struct EwArgs {
  const void* a;
  const void* b;
  void* y;
  int64_t rows;  // image: rows of D elements; without image rows * D is just the element count
  int D;
  int exp_accurate;
  QImage img;
};
template <int XT, int OP>
__device__ __forceinline__ float ew_one(float x, float y, int exp_accurate) {
  if (OP == EW_ADD) return x + y;
  if (OP == EW_MUL) return x * y;
  float s = silu_ref(x, exp_accurate);
  if (OP == EW_SILU) return s;
  // the reference runs SiLU and the product as two operators: the SiLU result is stored in the tensor's type first
  if (XT != MLLM_HIP_F32) s = bf16_to_f32(f32_to_bf16(s));
  return s * y;
}
template <int XT, int OP>
__global__ __launch_bounds__(256) void elementwise_kernel(EwArgs a) {
  const int ipr = a.D >> 3;  // items per row
  const int64_t it = (int64_t)blockIdx.x * 256 + threadIdx.x;
  int64_t row = 0;  // (of an image)
  if (a.img.base) {
    row = it <= 0xffffffffll ? (int64_t)((uint32_t)it / (uint32_t)ipr) : it / ipr;  // (64 bits: 100 instructions)
    if (row >= max((int64_t)a.img.MT, a.rows)) return;  // whole quads leave together: ipr is a multiple of 4 whenever an image is written
  } else if (it >= a.rows * ipr) {
    return;
  }
  const int col = (int)(it - row * ipr);
  float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const bool valid = row < a.rows;
  if (valid) {
    Item8<XT> ra, rb;
    float va[8], vb[8];
    item_load<XT>(a.a, it * 8, ra);
    if (OP != EW_SILU) item_load<XT>(a.b, it * 8, rb);
    item_to_f32<XT>(ra, va);
    if (OP != EW_SILU) item_to_f32<XT>(rb, vb);
#pragma unroll
    for (int e = 0; e < 8; e++) o[e] = ew_one<XT, OP>(va[e], OP == EW_SILU ? 0.f : vb[e], a.exp_accurate);
    item_store<XT>(a.y, it * 8, o);
  }
  if (a.img.base) quad_quantize_to_image(o, a.img, (int)row, col >> 2, col & 3, true);
}

// SiLU of up to EW_PAIRS_ITEMS items: two elements per thread.  Eight are a chain of 330 instructions (exponential, division) in waves that have
// a SIMD to themselves.  SiLU(gate) * up in a graph, eight / two, us: 1 x 9728 fp32 2.5 / 2.0, bf16 2.9 / 2.0, 8 x 9728 2.6 / 2.0, 64 x 9728
// 3.1 / 2.4, 256 x 9728 (311 296 items) 5.3 / 4.6; 1024 x 9728 18.6 / 19.2, bound by memory.
constexpr int64_t EW_PAIRS_ITEMS = 320 * 1024;
template <int XT, int OP>
__global__ __launch_bounds__(256) void elementwise_pairs_kernel(EwArgs a) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= a.rows * (a.D >> 1)) return;
  float x[2], y[2] = {0.f, 0.f};
  auto load = [&](const void* p, float (&v)[2]) {
    if (XT == MLLM_HIP_F32) {
      const f32x2 r = reinterpret_cast<const f32x2*>(p)[i];
      v[0] = r.x, v[1] = r.y;
    } else {
      const uint32_t r = reinterpret_cast<const uint32_t*>(p)[i];
      v[0] = __uint_as_float(r << 16), v[1] = __uint_as_float(r & 0xffff0000u);
    }
  };
  load(a.a, x);
  if (OP != EW_SILU) load(a.b, y);
#pragma unroll
  for (int e = 0; e < 2; e++) x[e] = ew_one<XT, OP>(x[e], y[e], a.exp_accurate);
  if (XT == MLLM_HIP_F32) reinterpret_cast<f32x2*>(a.y)[i] = f32x2{x[0], x[1]};
  else reinterpret_cast<uint32_t*>(a.y)[i] = pack_bf16(x[0], x[1]);
}

// ---- softmax over the last axis, one wave per row ----------------------------------------------------------------------
// rows of at most 16 elements use expf like the reference's short-row branch (softmax.cpp:19-31); in longer rows the
// whole vectors of eight take the polynomial and the len % 8 tail elements expf (softmax.cpp:44-57)
__device__ __forceinline__ float softmax_exp(float x, bool poly) { return poly ? exp_poly(x) : expf(x); }

__global__ __launch_bounds__(256) void softmax_rows_kernel(const float* __restrict__ x, float* __restrict__ y, int64_t rows, int len,
                                                           int exp_accurate) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float* xr = x + row * len;
  float* yr = y + row * len;
  const bool poly = len > 16 && !exp_accurate;
  float mx = -3.402823466e+38f;
  for (int i = lane; i < len; i += 64) mx = fmaxf(mx, xr[i]);
  mx = wave_max(mx);
  float sum = 0.f;
  for (int i = lane; i < len; i += 64) {
    const float e = softmax_exp(xr[i] - mx, poly && i < (len & ~7));
    yr[i] = e;
    sum += e;
  }
  sum = wave_sum(sum);
  const float inv = 1.f / sum;
  for (int i = lane; i < len; i += 64) yr[i] *= inv;  // each lane re-reads what it wrote itself
}

// Rows of up to 64 NR elements: the lane keeps its elements (index lane + 64 j) in registers -- one pass over memory, every
// load requested before the first is used (the loops above are a load per iteration, three times over) -- and sums them in
// the same order: the same bits.  32 rows of 1024 (the attention of a decode token): 11.7 -> 3.6 us.
template <int NR>
__global__ __launch_bounds__(256) void softmax_rows_reg_kernel(const float* __restrict__ x, float* __restrict__ y, int64_t rows, int len,
                                                               int exp_accurate) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float* xr = x + row * len;
  float* yr = y + row * len;
  const bool poly = len > 16 && !exp_accurate;
  float v[NR];
#pragma unroll
  for (int j = 0; j < NR; j++) v[j] = lane + 64 * j < len ? xr[lane + 64 * j] : -3.402823466e+38f;
  float mx = -3.402823466e+38f;
#pragma unroll
  for (int j = 0; j < NR; j++) mx = fmaxf(mx, v[j]);
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < NR; j++) {
    const int i = lane + 64 * j;
    if (i < len) {
      v[j] = softmax_exp(v[j] - mx, poly && i < (len & ~7));
      sum += v[j];
    }
  }
  sum = wave_sum(sum);
  const float inv = 1.f / sum;
#pragma unroll
  for (int j = 0; j < NR; j++)
    if (lane + 64 * j < len) yr[lane + 64 * j] = v[j] * inv;
}
// Long rows (a vocabulary): a workgroup of sixteen waves per row, three passes with eight loads in flight per thread; maxima
// and sums meet in LDS (per thread in index order, then the waves in order).  Eight rows of 151 936: 1993 -> about 60 us.
constexpr int SOFTMAX_WG = 1024;
__global__ __launch_bounds__(SOFTMAX_WG) void softmax_long_rows_kernel(const float* __restrict__ x, float* __restrict__ y, int len,
                                                                      int exp_accurate) {
  __shared__ float s_red[SOFTMAX_WG / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* xr = x + (int64_t)blockIdx.x * len;
  float* yr = y + (int64_t)blockIdx.x * len;
  const bool poly = !exp_accurate;
  constexpr int UB = 8;
  float mx = -3.402823466e+38f;
  for (int i0 = tid; i0 < len; i0 += SOFTMAX_WG * UB) {
    float v[UB];
#pragma unroll
    for (int u = 0; u < UB; u++) v[u] = i0 + SOFTMAX_WG * u < len ? xr[i0 + SOFTMAX_WG * u] : -3.402823466e+38f;
#pragma unroll
    for (int u = 0; u < UB; u++) mx = fmaxf(mx, v[u]);
  }
  mx = wave_max(mx);
  if (lane == 0) s_red[wave] = mx;
  __syncthreads();
  mx = s_red[0];
#pragma unroll
  for (int w = 1; w < SOFTMAX_WG / 64; w++) mx = fmaxf(mx, s_red[w]);
  __syncthreads();
  float sum = 0.f;
  for (int i0 = tid; i0 < len; i0 += SOFTMAX_WG * UB) {
    float v[UB];
#pragma unroll
    for (int u = 0; u < UB; u++) v[u] = i0 + SOFTMAX_WG * u < len ? xr[i0 + SOFTMAX_WG * u] : 0.f;
#pragma unroll
    for (int u = 0; u < UB; u++) {
      const int i = i0 + SOFTMAX_WG * u;
      if (i < len) {
        const float e = softmax_exp(v[u] - mx, poly && i < (len & ~7));
        yr[i] = e;
        sum += e;
      }
    }
  }
  sum = wave_sum(sum);
  if (lane == 0) s_red[wave] = sum;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < SOFTMAX_WG / 64; w++) total += s_red[w];
  const float inv = 1.f / total;
  for (int i0 = tid; i0 < len; i0 += SOFTMAX_WG * UB) {  // each thread re-reads what it wrote itself
    float v[UB];
#pragma unroll
    for (int u = 0; u < UB; u++) v[u] = i0 + SOFTMAX_WG * u < len ? yr[i0 + SOFTMAX_WG * u] : 0.f;
#pragma unroll
    for (int u = 0; u < UB; u++)
      if (i0 + SOFTMAX_WG * u < len) yr[i0 + SOFTMAX_WG * u] = v[u] * inv;
  }
}

// Few long rows spread over the chip (mllm_hip_softmax_ws): a row is cut into pieces of SOFTMAX_PIECE elements with a
// workgroup each, and the row's maximum and sum meet in the caller's workspace, so the operator is three launches: maxima of
// the pieces, sums of the pieces (which need the row's maximum: the reference's polynomial is not exp(a) exp(b) = exp(a + b)
// to fp32), results -- or two, see STAGE 3 below.  A workgroup per row is bound by what one CU can load and by its vector ALU: eight rows of
// 151 936 take 49 us there and 9.7 here (one row 47 -> 8.0; a launch costs about 2.5 us whatever it does).  A piece inside the polynomial's
// range has no branch per element, so that its exponentials overlap (with the branches: 14.8 and 13.5); pieces of 2048 elements
// are no faster.
constexpr int SOFTMAX_PIECE = 4096;
// In a graph, us, a workgroup per row / pieces (which do not get slower below their limits: the limits are not where the two meet):
//   1 to 16 rows of 8192: 7.1 / 9.0, 16 384: 13.4 / 9.3, 20 480: 9.0 / 9.4, 32 000: 12.0 / 10.4, 40 960: 14.7 / 9.6, 64 000: 21.4 / 10.2
//   256 rows of 20 480: 16.6 / 17.4, 40 960: 32.0 / 33.4, 64 000: 48.5 / 46.1;  512 rows of 24 576: 36.6 / 38.0, 40 960: 60.4 / 56.1, 64 000: 101 /
//   83, 151 936: 308 / 231;  1024 rows of 40 960: 131 / 106, 151 936: 603 / 455
// Up to 16 rows the pieces win from about 22 000 elements on (and from 12 288 to 16 384, where one workgroup holds the row in registers),
// with 256 rows from about 50 000: 193 to 256 rows are one whole round of the chip for the form of a workgroup per row, which stays up to
// there (233 x 46 120: 33.8 / 35.7; 192 x 50 000 30.7 / 30.9, 256 x 50 000 39.1 / 39.0, 256 x 56 000 43.1 / 42.3, 320 x 40 968 43.1 / 40.0).
// The other limit dates from pieces with a branch per element (32 000: 13.9) and lies late for few rows.
constexpr int SOFTMAX_LONG = 40960;
constexpr int SOFTMAX_LONG_ROUND = 50000;  // with 193 to 256 rows
constexpr int SOFTMAX_SPLIT_ROWS = 512;
__device__ __forceinline__ float block_max_256(float v, float* s_red) {
  v = wave_max(v);
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = v;
  __syncthreads();
  v = fmaxf(fmaxf(s_red[0], s_red[1]), fmaxf(s_red[2], s_red[3]));
  __syncthreads();
  return v;
}
__device__ __forceinline__ float block_sum_256(float v, float* s_red) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = v;
  __syncthreads();
  v = ((s_red[0] + s_red[1]) + s_red[2]) + s_red[3];
  __syncthreads();
  return v;
}
// STAGE 0: pmax[row][piece], and psum[row][piece] = SOFTMAX_NO_SUM;  1: psum[row][piece];  2: y;  3: both in one launch.  ws: pmax, then psum, of
// rows * pieces floats each.
// STAGE 3: a workgroup keeps its exponentials in registers, publishes their sum and reads the other pieces' as they appear (the value is its
// own flag; stores and loads of device scope, since every XCD has an L2 of its own).  It runs for up to SOFTMAX_WAIT workgroups, a quarter of what
// the chip holds at once, so they run together.  Where they should not (other work on the chip), a workgroup gives up after `polls` looks
// and adds up the row by itself: the wait is bounded, the bits are the same.  In a graph, us, stages 1 and 2 / 3 (with more workgroups, or more
// pieces to look at, the looks cost more than a launch): 1 x 50 000 8.9 / 7.2, 4 x 64 000 9.7 / 7.9, 8 x 151 936 10.6 / 9.7, 16 x 151 936 (608)
// 12.0 / 12.4, 512 x 151 936 225 / 255, 1 x 1 000 000 (245 pieces) 9.9 / 11.4; a launch less for the host.
constexpr uint32_t SOFTMAX_NO_SUM = 0xffffffffu;
constexpr int SOFTMAX_WAIT = 512, SOFTMAX_WAIT_PIECES = 64;
// Looks: sixteen were too few in some of the runs of 8 x 151 936 and 13 x 151 931, 32 and more in none.  64 take about 30 us, less than to
// add up the row (50 to 90 us with no wait: 8 x 151 936, 1 x 262 144), so that a workgroup whose row is not on the chip all at once gives its
// place up soon.
constexpr int SOFTMAX_LOOKS = 64;
static int g_softmax_polls = SOFTMAX_LOOKS;  // mllm_hip_softmax_set_wait
template <int STAGE>
__global__ __launch_bounds__(256) void softmax_pieces_kernel(const float* __restrict__ x, float* __restrict__ y, float* __restrict__ ws,
                                                             int len, int exp_accurate, int polls) {
  __shared__ float s_red[4];
  constexpr int R = SOFTMAX_PIECE / 256;
  const int tid = threadIdx.x, piece = blockIdx.x, pieces = gridDim.x;
  const int64_t row = blockIdx.y;
  float* pmax = ws + row * pieces;
  float* psum = ws + ((int64_t)gridDim.y + row) * pieces;
  const float* xr = x + row * len;
  float v[R];
  auto load = [&](int i0) {
#pragma unroll
    for (int j = 0; j < R; j++) v[j] = i0 + 256 * j < len ? xr[i0 + 256 * j] : -3.402823466e+38f;
  };
  const int i0 = piece * SOFTMAX_PIECE + tid;
  load(i0);
  if (STAGE == 0) {
    float mx = v[0];
#pragma unroll
    for (int j = 1; j < R; j++) mx = fmaxf(mx, v[j]);
    mx = block_max_256(mx, s_red);
    if (tid == 0) {
      pmax[piece] = mx;
      psum[piece] = __uint_as_float(SOFTMAX_NO_SUM);
    }
    return;
  }
  const bool poly = !exp_accurate;
  float mx = -3.402823466e+38f;
  for (int p = tid; p < pieces; p += 256) mx = fmaxf(mx, pmax[p]);
  float total = 0.f;
  if (STAGE == 2)
    for (int p = tid; p < pieces; p += 256) total += psum[p];
  mx = block_max_256(mx, s_red);
  auto exponentials = [&](int p, int i0) {  // of piece p, in v; returns the thread's sum
    float sum = 0.f;
    if (poly && (int64_t)(p + 1) * SOFTMAX_PIECE <= (len & ~7)) {  // (uniform) the whole piece takes the polynomial
#pragma unroll
      for (int j = 0; j < R; j++) {
        v[j] = exp_poly(v[j] - mx);
        sum += v[j];
      }
    } else {
#pragma unroll
      for (int j = 0; j < R; j++) {
        const int i = i0 + 256 * j;
        if (i < len) {
          v[j] = softmax_exp(v[j] - mx, poly && i < (len & ~7));
          sum += v[j];
        }
      }
    }
    return sum;
  };
  float sum = exponentials(piece, i0);
  if (STAGE == 1 || STAGE == 3) {
    sum = block_sum_256(sum, s_red);
    if (tid == 0) {
      if (STAGE == 1) psum[piece] = sum;
      else __hip_atomic_store(&psum[piece], sum == sum ? sum : __uint_as_float(0x7fc00000u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (STAGE == 1) return;
    bool missing = tid < pieces;  // (at most 64 pieces)
    for (int n = 0; missing && n <= polls; n++) {
      total = __hip_atomic_load(&psum[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      missing = __float_as_uint(total) == SOFTMAX_NO_SUM;
    }
    if (__syncthreads_or(missing)) {
      total = 0.f;
      for (int p = 0; p < pieces; p++) {
        load(p * SOFTMAX_PIECE + tid);
        const float s = block_sum_256(exponentials(p, p * SOFTMAX_PIECE + tid), s_red);
        if (tid == p) total += s;
      }
      load(i0);
      exponentials(piece, i0);
    }
  }
  const float inv = 1.f / block_sum_256(total, s_red);
  float* yr = y + row * len;
#pragma unroll
  for (int j = 0; j < R; j++)
    if (i0 + 256 * j < len) yr[i0 + 256 * j] = v[j] * inv;
}

// Rows between the two (2049 to 16 384 elements: the keys of an attention row): a workgroup of four waves per row, the row in
// registers (16, 32 or 64 elements per thread), one pass over memory; maxima and sums meet in LDS.
template <int R>
__global__ __launch_bounds__(256) void softmax_wg_rows_kernel(const float* __restrict__ x, float* __restrict__ y, int len, int exp_accurate) {
  __shared__ float s_red[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* xr = x + (int64_t)blockIdx.x * len;
  float* yr = y + (int64_t)blockIdx.x * len;
  const bool poly = !exp_accurate;
  float v[R];
#pragma unroll
  for (int j = 0; j < R; j++) v[j] = tid + 256 * j < len ? xr[tid + 256 * j] : -3.402823466e+38f;
  float mx = v[0];
#pragma unroll
  for (int j = 1; j < R; j++) mx = fmaxf(mx, v[j]);
  mx = wave_max(mx);
  if (lane == 0) s_red[wave] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(s_red[0], s_red[1]), fmaxf(s_red[2], s_red[3]));
  __syncthreads();
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < R; j++) {
    const int i = tid + 256 * j;
    if (i < len) {
      v[j] = softmax_exp(v[j] - mx, poly && i < (len & ~7));
      sum += v[j];
    }
  }
  sum = wave_sum(sum);
  if (lane == 0) s_red[wave] = sum;
  __syncthreads();
  const float inv = 1.f / (((s_red[0] + s_red[1]) + s_red[2]) + s_red[3]);
#pragma unroll
  for (int j = 0; j < R; j++)
    if (tid + 256 * j < len) yr[tid + 256 * j] = v[j] * inv;
}

// ---- top-k over the last axis, one wave per row -------------------------------------------------------------------------
// Selection by repeated wave-wide extreme: round r takes the best element that comes after the one taken in round r-1
// in the order (value descending [ascending for smallest], index ascending).  Equal values are taken lowest index
// first (the reference's order among equal values is whatever its heap and std::sort leave).
struct KeyIdx {
  float v;
  int i;
};
__device__ __forceinline__ bool comes_before(float va, int ia, float vb, int ib, bool largest) {
  if (va != vb) return largest ? va > vb : va < vb;
  return ia < ib;
}
__device__ __forceinline__ KeyIdx wave_best(KeyIdx k, bool largest) {
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const float ov = __shfl_xor(k.v, off, 64);
    const int oi = __shfl_xor(k.i, off, 64);
    if (oi >= 0 && (k.i < 0 || comes_before(ov, oi, k.v, k.i, largest))) {
      k.v = ov;
      k.i = oi;
    }
  }
  return k;
}
// rows of `vals` may live in global memory or in LDS; out arrays are written by lane 0.  sorted == 0: by index.
__device__ __forceinline__ void wave_topk(const float* vals, int len, int k, bool largest, bool sorted, float* out_v, int* out_i,
                                          int lane) {
  float pv = 0.f;
  int pi = -1;  // previous pick
  for (int r = 0; r < k; r++) {
    KeyIdx best{0.f, -1};
    for (int i = lane; i < len; i += 64) {
      const float v = vals[i];
      const bool after_prev = pi < 0 || comes_before(pv, pi, v, i, largest);
      if (after_prev && (best.i < 0 || comes_before(v, i, best.v, best.i, largest))) {
        best.v = v;
        best.i = i;
      }
    }
    best = wave_best(best, largest);
    pv = best.v;
    pi = best.i;
    if (lane == 0) {
      out_v[r] = best.v;
      out_i[r] = best.i;
    }
  }
  if (!sorted && lane == 0) {  // by index: insertion sort of k entries
    for (int a = 1; a < k; a++) {
      const float v = out_v[a];
      const int i = out_i[a];
      int b = a - 1;
      while (b >= 0 && out_i[b] > i) {
        out_v[b + 1] = out_v[b];
        out_i[b + 1] = out_i[b];
        b--;
      }
      out_v[b + 1] = v;
      out_i[b + 1] = i;
    }
  }
}

// The same selection for a row of up to 64 R elements in LDS, by rank: a lane keeps its R elements (index lane + 64 j) and counts,
// over one pass of broadcast reads, how many elements of the row come before each of them in the order above; the elements
// of rank < k are the selection, rank = place by value, and the place by index is a count over ballots.  One pass instead of
// k rounds of wave-wide extremes (each six exchanges through the LDS pipe): the gate's 8 of 128 take a fifth of the time.
// (value, index) as one unsigned key, larger = earlier in that order: the float's bits made monotonic (-0 counts as +0, as it
// compares equal), inverted for "smallest first"; below it the inverted index, so that equal values go lowest index first
__device__ __forceinline__ unsigned long long order_key(float v, int i, bool largest) {
  uint32_t b = __float_as_uint(v + 0.f);
  b = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
  if (!largest) b = ~b;
  return ((unsigned long long)b << 32) | (uint32_t)~(uint32_t)i;
}
template <int R>
__device__ __forceinline__ void wave_topk_ranked(const float* vals, int len, int k, bool largest, bool sorted, float* out_v, int* out_i,
                                                 int lane) {
  float v[R];
  unsigned long long key[R];
  int rank[R];
#pragma unroll
  for (int j = 0; j < R; j++) {
    v[j] = lane + 64 * j < len ? vals[lane + 64 * j] : 0.f;
    key[j] = order_key(v[j], lane + 64 * j, largest);
    rank[j] = 0;
  }
#pragma unroll 8
  for (int o = 0; o < len; o++) {  // (eight reads in flight: one at a time, their latency is the whole cost)
    const unsigned long long ok = order_key(vals[o], o, largest);  // every lane the same address
#pragma unroll
    for (int j = 0; j < R; j++) rank[j] += ok > key[j] ? 1 : 0;
  }
  unsigned long long m[R];
#pragma unroll
  for (int j = 0; j < R; j++) m[j] = __ballot(lane + 64 * j < len && rank[j] < k);
  int before = 0;  // selected elements of the lower sixty-fours
#pragma unroll
  for (int j = 0; j < R; j++) {
    if (lane + 64 * j < len && rank[j] < k) {
      const int pos = sorted ? rank[j] : before + __popcll(m[j] & ((1ull << lane) - 1ull));
      out_v[pos] = v[j];
      out_i[pos] = lane + 64 * j;
    }
    before += __popcll(m[j]);
  }
}

__global__ __launch_bounds__(256) void topk_rows_kernel(const float* __restrict__ x, float* __restrict__ values, int32_t* __restrict__ indices,
                                                        int64_t rows, int len, int k, int largest, int sorted) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;  // (no workgroup barrier below)
  if (len <= 256) {  // short rows -- the experts of an MoE gate -- by rank in one pass over a copy of the row in LDS
    __shared__ float s_row[4][256];
    float* sr = s_row[threadIdx.x >> 6];
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = lane + 64 * j < len ? x[row * len + lane + 64 * j] : 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) sr[lane + 64 * j] = v[j];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (len <= 128) wave_topk_ranked<2>(sr, len, k, largest != 0, sorted != 0, values + row * k, indices + row * k, lane);
    else wave_topk_ranked<4>(sr, len, k, largest != 0, sorted != 0, values + row * k, indices + row * k, lane);
    return;
  }
  wave_topk(x + row * len, len, k, largest != 0, sorted != 0, values + row * k, indices + row * k, lane);
}

// Long rows (a vocabulary): a workgroup of sixteen waves per row runs the same k rounds, every thread scanning its share of
// the row with eight loads in flight, the waves' candidates meeting in LDS.  20 of 151 936: 11.3 ms with one wave -> 0.2 ms.
constexpr int TOPK_WG = 1024;
__global__ __launch_bounds__(TOPK_WG) void topk_long_rows_kernel(const float* __restrict__ x, float* __restrict__ values,
                                                                int32_t* __restrict__ indices, int len, int k, int largest, int sorted) {
  __shared__ float s_v[TOPK_WG / 64];
  __shared__ int s_i[TOPK_WG / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t row = blockIdx.x;
  const float* xr = x + row * len;
  float* out_v = values + row * k;
  int32_t* out_i = indices + row * k;
  const bool lg = largest != 0;
  float pv = 0.f;
  int pi = -1;  // previous pick
  constexpr int UB = 8;
  for (int r = 0; r < k; r++) {
    KeyIdx best{0.f, -1};
    for (int i0 = tid; i0 < len; i0 += TOPK_WG * UB) {
      float v[UB];
#pragma unroll
      for (int u = 0; u < UB; u++) v[u] = i0 + TOPK_WG * u < len ? xr[i0 + TOPK_WG * u] : 0.f;
#pragma unroll
      for (int u = 0; u < UB; u++) {
        const int i = i0 + TOPK_WG * u;
        if (i < len) {
          const bool after_prev = pi < 0 || comes_before(pv, pi, v[u], i, lg);
          if (after_prev && (best.i < 0 || comes_before(v[u], i, best.v, best.i, lg))) {
            best.v = v[u];
            best.i = i;
          }
        }
      }
    }
    best = wave_best(best, lg);
    if (lane == 0) {
      s_v[wave] = best.v;
      s_i[wave] = best.i;
    }
    __syncthreads();
    best = KeyIdx{s_v[0], s_i[0]};
#pragma unroll
    for (int w = 1; w < TOPK_WG / 64; w++) {
      const float ov = s_v[w];
      const int oi = s_i[w];
      if (oi >= 0 && (best.i < 0 || comes_before(ov, oi, best.v, best.i, lg))) best = KeyIdx{ov, oi};
    }
    __syncthreads();
    pv = best.v;
    pi = best.i;
    if (tid == 0) {
      out_v[r] = best.v;
      out_i[r] = best.i;
    }
  }
  if (!sorted && tid == 0) {  // by index: insertion sort of k entries (thread 0 wrote them itself)
    for (int a = 1; a < k; a++) {
      const float v = out_v[a];
      const int i = out_i[a];
      int b = a - 1;
      while (b >= 0 && out_i[b] > i) {
        out_v[b + 1] = out_v[b];
        out_i[b + 1] = out_i[b];
        b--;
      }
      out_v[b + 1] = v;
      out_i[b + 1] = i;
    }
  }
}

// Rows longer than 256 elements, k up to TOPK_SEL_MAX: radix select.  (value, index) pairs are ordered by order_key(); the
// key of the k-th pair is found a digit at a time (four bytes, or 12, 12 and 8 bits), highest first: a histogram of that digit
// over the elements that agree with the digits found so far (LDS counters; lanes of a wave that hold the same digit add once),
// then the bin in which the k-th falls.  These counting passes give the value's key; where more elements share that value
// than are still wanted, as many again over the inverted index choose the lowest indices among them.  Every pair at or above the k-th key is then collected
// in LDS and placed by its rank among the k.  The passes read the row again (eight 16-byte loads in flight per thread) or,
// for rows of up to eight such loads per thread, keep the keys in registers.  The cost does not depend on k.
constexpr int TOPK_SEL_MAX = 2048;
#ifndef TOPK_LEADERS
#define TOPK_LEADERS 2
#endif
template <int VEC> struct TopkVec;
template <> struct TopkVec<1> { typedef float T; };
template <> struct TopkVec<4> { typedef float4 T; };
template <int NT, int VEC, int R, bool WIDE>
__global__ __launch_bounds__(NT) void topk_select_rows_kernel(const float* __restrict__ x, float* __restrict__ values,
                                                              int32_t* __restrict__ indices, int len, int k, int largest, int sorted) {
  typedef typename TopkVec<VEC>::T VT;
  __shared__ unsigned s_hist[WIDE ? 4096 : 256];
  __shared__ unsigned s_pick[4];  // chosen digit, pairs still wanted inside its bin, the bin's count; [3]: pairs collected
  __shared__ unsigned long long s_sel[TOPK_SEL_MAX];
  const int tid = threadIdx.x, lane = tid & 63;
  const int64_t row = blockIdx.x;
  const float* xr = x + row * len;
  const bool lg = largest != 0;
  const int nunits = len / VEC;  // (VEC divides len)
  const bool inreg = nunits <= NT * R;
  uint32_t kreg[R][VEC];
  auto vkey = [&](float v) {
    uint32_t b = __float_as_uint(v + 0.f);
    b = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
    return lg ? b : ~b;
  };
  auto load_keys = [&](int base, uint32_t (&kk)[R][VEC]) {
    VT v[R];
#pragma unroll
    for (int j = 0; j < R; j++) {
      const int u = base + tid + NT * j;
      if (u < nunits) v[j] = reinterpret_cast<const VT*>(xr)[u];
      else v[j] = VT{};
    }
#pragma unroll
    for (int j = 0; j < R; j++) {
      const float* f = reinterpret_cast<const float*>(&v[j]);
#pragma unroll
      for (int e = 0; e < VEC; e++) kk[j][e] = vkey(f[e]);
    }
  };
  if (inreg) load_keys(0, kreg);
  // f(key, index, valid) for every element of the row, by all lanes of every wave together (f holds wave-wide operations)
  auto scan = [&](auto&& f) {
    if (inreg) {
#pragma unroll
      for (int j = 0; j < R; j++) {
        const int u = tid + NT * j;
#pragma unroll
        for (int e = 0; e < VEC; e++) f(kreg[j][e], u * VEC + e, u < nunits);
      }
    } else {
      for (int base = 0; base < nunits; base += NT * R) {
        uint32_t kk[R][VEC];
        load_keys(base, kk);
#pragma unroll
        for (int j = 0; j < R; j++) {
          const int u = base + tid + NT * j;
#pragma unroll
          for (int e = 0; e < VEC; e++) f(kk[j][e], u * VEC + e, u < nunits);
        }
      }
    }
  };
  auto hist_add = [&](bool match, uint32_t digit) {
    unsigned long long m = __ballot(match);
    for (int it = 0; it < TOPK_LEADERS && m; it++) {  // (m is the same in every lane)
      const int leader = __ffsll((long long)m) - 1;
      const uint32_t d0 = (uint32_t)__builtin_amdgcn_readlane((int)digit, leader);
      const bool mine = match && digit == d0;
      const unsigned long long same = __ballot(mine);
      if (lane == leader) atomicAdd(&s_hist[d0], (unsigned)__popcll(same));
      match = match && !mine;
      m &= ~same;
    }
    if (match) atomicAdd(&s_hist[digit], 1u);
  };
  // the bin of the `need`-th largest digit among nb bins: wave 0, a lane per nb / 64 bins
  auto pick = [&](uint32_t need, int nb) {
    if (tid < 64) {
      const int per = nb >> 6, b0 = lane * per;
      uint32_t tot = 0;
      for (int q = 0; q < per; q++) tot += s_hist[b0 + ((q + lane) & (per - 1))];  // (the lanes on different banks)
      uint32_t incl = tot;  // this lane's bins and all higher ones
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const uint32_t o = (uint32_t)__shfl_down((int)incl, off, 64);
        if (lane + off < 64) incl += o;
      }
      uint32_t a = incl - tot;
      if (a < need && need <= incl) {
        for (int q = per - 1; q >= 0; q--) {
          const uint32_t c = s_hist[b0 + q];
          if (a + c >= need) {
            s_pick[0] = (uint32_t)(b0 + q);
            s_pick[1] = need - a;
            s_pick[2] = c;
            break;
          }
          a += c;
        }
      }
    }
  };
  // one counting pass over the digit of `bits` bits at `shift`: keyof(key, index, valid, &k32) says whether the element still
  // agrees with the digits found so far and gives the 32 bits the digit is taken from
  auto count_pass = [&](int shift, int bits, uint32_t need, auto&& keyof) {
    const int nb = 1 << bits;
    for (int b = tid; b < nb; b += NT) s_hist[b] = 0;
    __syncthreads();
    scan([&](uint32_t key, int idx, bool ok) {
      uint32_t k32;
      const bool mt = keyof(key, idx, ok, k32);
      hist_add(mt, (k32 >> shift) & (uint32_t)(nb - 1));
    });
    __syncthreads();
    pick(need, nb);
    __syncthreads();
  };
  // rows read again per pass: 12 + 12 + 8 bits (a pass over memory less); rows in registers: four bytes (256 counters to clear
  // and to walk per pass instead of 4096)
  constexpr int NPASS = WIDE ? 3 : 4;
  const int p_shift[4] = {WIDE ? 20 : 24, WIDE ? 8 : 16, WIDE ? 0 : 8, 0}, p_bits[4] = {WIDE ? 12 : 8, WIDE ? 12 : 8, 8, 8};
  uint32_t need = (uint32_t)k, t_val = 0, mask = 0, ties = 0;
  if (tid == 0) s_pick[3] = 0;
#pragma unroll
  for (int p = 0; p < NPASS; p++) {
    count_pass(p_shift[p], p_bits[p], need, [&](uint32_t key, int, bool ok, uint32_t& k32) {
      k32 = key;
      return ok && (key & mask) == t_val;
    });
    t_val |= s_pick[0] << p_shift[p];
    mask |= ((1u << p_bits[p]) - 1u) << p_shift[p];
    need = s_pick[1];
    ties = s_pick[2];
  }
  uint32_t t_idx = 0;  // pairs of the k-th value are taken down to this inverted index
  if (ties != need) {   // (the same in every thread)
    mask = 0;
#pragma unroll
    for (int p = 0; p < NPASS; p++) {
      count_pass(p_shift[p], p_bits[p], need, [&](uint32_t key, int idx, bool ok, uint32_t& k32) {
        k32 = ~(uint32_t)idx;
        return ok && key == t_val && (k32 & mask) == t_idx;
      });
      t_idx |= s_pick[0] << p_shift[p];
      mask |= ((1u << p_bits[p]) - 1u) << p_shift[p];
      need = s_pick[1];
    }
  }
  scan([&](uint32_t key, int idx, bool ok) {
    const uint32_t ni = ~(uint32_t)idx;
    if (ok && (key > t_val || (key == t_val && ni >= t_idx))) {
      const unsigned pos = atomicAdd(&s_pick[3], 1u);
      if (pos < (unsigned)TOPK_SEL_MAX) s_sel[pos] = ((unsigned long long)key << 32) | ni;
    }
  });
  __syncthreads();
  const bool by_value = sorted != 0;
  for (int t = tid; t < k; t += NT) {
    const unsigned long long my = s_sel[t];
    const unsigned long long mc = by_value ? my : (my << 32);  // by index: the inverted index alone, larger = earlier
    int rank = 0;
    for (int j = 0; j < k; j++) {
      const unsigned long long o = s_sel[j];
      rank += (by_value ? o : (o << 32)) > mc ? 1 : 0;
    }
    const int idx = (int)~(uint32_t)my;
    values[row * k + rank] = xr[idx];
    indices[row * k + rank] = idx;
  }
}

// Few long rows spread over the chip (mllm_hip_topk_ws), k up to 128: a row is cut into equal pieces of at most TOPK_PIECE elements, a
// workgroup selects the k largest keys of its piece into the caller's workspace, and a second launch selects among the
// pieces' keys.  A workgroup per row is bound by what one CU loads per pass over the row: 20 of eight rows of 151 936 take
// 110 us there and 9.5 here, 64 of them 111 and 12.5.
//
// Selection inside a workgroup: keys are unique (value, inverted index).  The k-th largest of the threads' own maxima (found a
// bit at a time by counting, every wave on its own) is at most the k-th largest value, so the keys at or above it contain the
// selection, and of keys that are spread over the threads in any order they are few more than k (about 180 at k = 128).  They
// are collected in LDS and placed by rank, up to 64 of them in the registers of one wave; should they be more than TOPK_CAND
// (many equal values, or one thread's keys all larger than the other threads'), the k-th key itself is found a bit at a time.  The bound
// is taken as soon as at most twelve maxima more than k reach it, and the second launch takes values from the keys: with the exact bound and
// the values read again 8 x 151 936 took 10.8 us for the largest 20 (9.7 now), 8.85 for one (7.3), 8 x 32 000 12.8 for 64 (10.3).
// Equal pieces, so that every thread has elements: a last piece of 432 (12 720 cut at 4096s) gave 108 threads four each, all of them
// candidates for the largest 128 (256 rows of 12 720: 37.8 us, 19.7 in equal pieces, 20.3 as a workgroup per row).
// Limits, in a graph, us, a workgroup per row / pieces (with the exact bound, 0.4 to 2 us more than now), the largest 1 | 50 | 128: 8 rows of 4100: 17.6 / 8.6 | 19.1 / 12.9 | 21.3 / 13.9 (up to
// 4096 a row is one piece, and the second launch has nothing to merge), of 151 936: 109 / 9.3 | 111 / 15.0 | 113 / 23.5; 512 rows of 4100: 19.0 /
// 11.7 | 20.9 / 16.8 | 24.1 / 19.4, of 151 936: 256 / 76 | 260 / 101 | 264 / 143.  Pieces win on either side of 512 rows (1024 rows of 4100:
// 38.2 / 23.5, of 151 936: 511 / 187, the largest 50); the limits bound the workspace, 512 x 38 pieces x 128 keys of 8 bytes: 20 MB.
constexpr int TOPK_PIECE = 4096;
constexpr int TOPK_CAND = 1024;
constexpr int TOPK_SPLIT_K = 128;
constexpr int TOPK_SPLIT_LEN = 4096;
constexpr int TOPK_SPLIT_ROWS = 512;
constexpr int TOPK_MERGE_R = 20;  // keys per thread of the second launch, at most
struct TopkShared {
  unsigned long long top[256];  // the selection by value
  unsigned long long cand[TOPK_CAND];
  uint32_t maxima[256];
  unsigned count, hits[4];
};
__device__ __forceinline__ unsigned long long lane_u64(unsigned long long v, int lane) {  // (lane: the same in every lane)
  return ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), lane) << 32) |
         (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
}
// the k largest non-zero keys of the workgroup's 256 R keys (zero = no element), largest first, in sh.top; returns how many there are
template <int R>
__device__ __forceinline__ int block_topk_256(const unsigned long long (&key)[R], int k, TopkShared& sh) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  unsigned long long mine = key[0];
#pragma unroll
  for (int j = 1; j < R; j++) mine = key[j] > mine ? key[j] : mine;
  if (tid == 0) sh.count = 0;
  sh.maxima[tid] = (uint32_t)(mine >> 32);
  __syncthreads();
  const u32x4 m4 = *reinterpret_cast<const u32x4*>(&sh.maxima[4 * lane]);  // every wave on its own, four maxima per lane
  // a bit costs about 100 clocks (four ballots and their counts); it need not be the k-th largest exactly: enough once few are left.  Four bits
  // between two looks at that: with a branch per bit equal values, which take all 32, were up to 16 % slower than without any (largest 20 of 2 x 48 496 with
  // ten values: 12.6 us without, 14.5 with, 12.8 now; normal ones, 8 x 151 936: 10.9, 9.7, 9.5)
  uint32_t b32 = 0;
  int reach = 256;  // maxima at or above b32
  for (int bit = 31; bit >= 0 && reach > k + 12; bit -= 4) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t t = b32 | (1u << (bit - i));
      const int c = __popcll(__ballot(m4.x >= t)) + __popcll(__ballot(m4.y >= t)) + __popcll(__ballot(m4.z >= t)) + __popcll(__ballot(m4.w >= t));
      b32 = c >= k ? t : b32;
      reach = c >= k ? c : reach;
    }
  }
  unsigned long long bound = (unsigned long long)b32 << 32;
  if (bound == 0) bound = 1;  // fewer than k threads hold an element: every element is wanted
  auto collect = [&]() {
#pragma unroll
    for (int j = 0; j < R; j++)
      if (key[j] >= bound) {
        const unsigned pos = atomicAdd(&sh.count, 1u);
        if (pos < (unsigned)TOPK_CAND) sh.cand[pos] = key[j];
      }
    __syncthreads();
  };
  collect();
  if (sh.count > (unsigned)TOPK_CAND) {  // (the same in every thread)
    unsigned long long kth = 0;
    for (int bit = 63; bit >= 0; bit--) {
      const unsigned long long t = kth | (1ull << bit);
      unsigned c = 0;
#pragma unroll
      for (int j = 0; j < R; j++) c += (unsigned)__popcll(__ballot(key[j] >= t));
      if (lane == 0) sh.hits[wave] = c;
      __syncthreads();
      if (sh.hits[0] + sh.hits[1] + sh.hits[2] + sh.hits[3] >= (unsigned)k) kth = t;
      __syncthreads();
    }
    bound = kth;
    if (tid == 0) sh.count = 0;
    __syncthreads();
    collect();  // exactly k
  }
  const int n = (int)sh.count;
  if (n <= 64) {
    if (wave == 0) {
      const unsigned long long my = lane < n ? sh.cand[lane] : 0ull;
      int r = 0;
      for (int j = 0; j < n; j++) r += lane_u64(my, j) > my ? 1 : 0;
      if (lane < n && r < k) sh.top[r] = my;
    }
  } else {
    for (int i = tid; i < n; i += 256) {
      const unsigned long long my = sh.cand[i];
      int r = 0;
#pragma unroll 8
      for (int j = 0; j < n; j++) r += sh.cand[j] > my ? 1 : 0;
      if (r < k) sh.top[r] = my;
    }
  }
  __syncthreads();
  return n < k ? n : k;
}
template <int VEC>
__global__ __launch_bounds__(256) void topk_pieces_kernel(const float* __restrict__ x, unsigned long long* __restrict__ ws, int len, int per, int k,
                                                          int largest) {
  typedef typename TopkVec<VEC>::T VT;
  __shared__ TopkShared sh;
  constexpr int R = TOPK_PIECE / 256, RV = R / VEC;
  const int tid = threadIdx.x, piece = blockIdx.x;
  const int64_t row = blockIdx.y;
  const VT* xr = reinterpret_cast<const VT*>(x + row * len);
  const int u0 = piece * per + tid, end = min(len / VEC, (piece + 1) * per);  // per: vectors of a piece (VEC divides len)
  VT v[RV];
#pragma unroll
  for (int j = 0; j < RV; j++) v[j] = u0 + 256 * j < end ? xr[u0 + 256 * j] : VT{};
  unsigned long long key[R];
#pragma unroll
  for (int j = 0; j < RV; j++) {
    const float* f = reinterpret_cast<const float*>(&v[j]);
#pragma unroll
    for (int e = 0; e < VEC; e++)
      key[j * VEC + e] = u0 + 256 * j < end ? order_key(f[e], (u0 + 256 * j) * VEC + e, largest != 0) : 0ull;
  }
  const int n = block_topk_256<R>(key, k, sh);
  // the pieces' largest keys first, then their second largest ...: the large ones spread over the threads of the next launch
  unsigned long long* out = ws + row * gridDim.x * k + piece;
  for (int t = tid; t < k; t += 256) out[(int64_t)t * gridDim.x] = t < n ? sh.top[t] : 0ull;
}
template <int R>
__global__ __launch_bounds__(256) void topk_merge_kernel(const float* __restrict__ x, const unsigned long long* __restrict__ ws,
                                                         float* __restrict__ values, int32_t* __restrict__ indices, int len, int n, int k,
                                                         int largest, int sorted) {
  __shared__ TopkShared sh;
  const int tid = threadIdx.x;
  const int64_t row = blockIdx.x;
  unsigned long long key[R];
#pragma unroll
  for (int j = 0; j < R; j++) key[j] = tid + 256 * j < n ? ws[row * n + tid + 256 * j] : 0ull;
  block_topk_256<R>(key, k, sh);  // (k keys: the row has that many elements)
  for (int t = tid; t < k; t += 256) {
    const unsigned long long my = sh.top[t];
    int r = t;
    if (!sorted) {
      r = 0;
      for (int j = 0; j < k; j++) r += (uint32_t)sh.top[j] > (uint32_t)my ? 1 : 0;  // the inverted index: larger = earlier
    }
    const int idx = (int)~(uint32_t)my;
    uint32_t b = (uint32_t)(my >> 32);  // order_key undone: not for zeros (of either sign) and NaN, which are read again
    if (!largest) b = ~b;
    float v = __uint_as_float(b & 0x80000000u ? b ^ 0x80000000u : ~b);
    if (v == 0.f || v != v) v = x[row * len + idx];
    values[row * k + r] = v;
    indices[row * k + r] = idx;
  }
}

// ---- MoE gate: logits = x . W^T (fp32), softmax, top-k, optional normalisation ------------------------------------------
// A workgroup of sixteen waves takes four tokens: the tokens' activations sit in LDS, every wave walks a sixteenth of the
// experts (16-byte loads along H, the tokens share each weight load), then wave t finishes token t.
// A lane requests eight pieces of an expert's row before it multiplies the first (a row of 2048 elements is one such batch,
// a round trip to memory per expert instead of one per piece), and only the workgroup's real tokens are multiplied.  One
// decode token of a 128-expert layer (1 MB of gate weights through one workgroup): 109 us with four waves and a load per
// iteration, an order of magnitude less this way; the sums run in the same order per lane (same logits bit for bit).
struct GateArgs {
  const void* x;
  const float* w;  // [E, H]
  int32_t* ids;    // [M, k]
  float* weights;  // [M, k]
  float* scores;   // [M, E] or null
  int64_t M;
  int H, E, k, norm, exp_accurate;
};
constexpr int GATE_TOK = 4;
constexpr int GATE_WAVES = 16;
// x of the workgroup's ntok tokens -> fp32 in LDS
template <int XT>
__device__ __forceinline__ void gate_stage_x(const GateArgs& a, int64_t tok0, int ntok, float* s_x, int tid, int nthreads) {
  const int ipr = a.H >> 3, nitems = ntok * ipr;
  for (int it = tid; it < nitems; it += nthreads) {  // (four tokens of 2048 elements, 1024 threads: one item per thread)
    const int t = it / ipr, c = it - t * ipr;
    float v[8];
    Item8<XT> r;
    item_load<XT>(a.x, (tok0 + t) * a.H + (int64_t)c * 8, r);
    item_to_f32<XT>(r, v);
    f32x4* dst = reinterpret_cast<f32x4*>(s_x + (size_t)t * a.H + c * 8);
    dst[0] = f32x4{v[0], v[1], v[2], v[3]};
    dst[1] = f32x4{v[4], v[5], v[6], v[7]};
  }
}
constexpr int GATE_CB = 8;  // pieces of a row a lane requests before it multiplies the first
struct GatePieces {
  f32x4 v[GATE_CB];
};
__device__ __forceinline__ void gate_request(const GateArgs& a, int e, int c0, GatePieces& p) {
  const f32x4* wr = reinterpret_cast<const f32x4*>(a.w + (size_t)min(e, a.E - 1) * a.H);
  const int last = (a.H >> 2) - 1;
#pragma unroll
  for (int u = 0; u < GATE_CB; u++) p.v[u] = wr[min(c0 + 64 * u, last)];
}
// logits of experts e0 + wave, e0 + wave + nwaves, ... < e1 for the ntok tokens in s_x; out[t * ostride + e].  AHEAD: first holds the first of the
// pieces, requested before x was staged
template <bool AHEAD>
__device__ __forceinline__ void gate_logits(const GateArgs& a, const float* s_x, int ntok, int e0, int e1, int wave, int nwaves, int lane,
                                            const GatePieces& first, float* out, size_t ostride) {
  constexpr int CB = GATE_CB;
  const int nc = a.H >> 2;
  GatePieces w = first;
  f32x4(&wv)[CB] = w.v;
  bool have = AHEAD;
  for (int e = e0 + wave; e < e1; e += nwaves) {
    float acc[GATE_TOK] = {0.f, 0.f, 0.f, 0.f};
    for (int c0 = lane; c0 < nc; c0 += 64 * CB) {
      if (!have) gate_request(a, e, c0, w);  // (uniform)
      have = false;
#pragma unroll
      for (int u = 0; u < CB; u++) {
        const int c = c0 + 64 * u;
        if (c < nc) {
#pragma unroll
          for (int t = 0; t < GATE_TOK; t++) {
            if (t < ntok) {  // uniform
              const f32x4 xv = reinterpret_cast<const f32x4*>(s_x + (size_t)t * a.H)[c];
              acc[t] = fmaf(xv.x, wv[u].x, acc[t]);
              acc[t] = fmaf(xv.y, wv[u].y, acc[t]);
              acc[t] = fmaf(xv.z, wv[u].z, acc[t]);
              acc[t] = fmaf(xv.w, wv[u].w, acc[t]);
            }
          }
        }
      }
    }
#pragma unroll
    for (int t = 0; t < GATE_TOK; t++) {
      if (t < ntok) {
        const float s = wave_sum(acc[t]);
        if (lane == 0) out[t * ostride + e] = s;
      }
    }
  }
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, true));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, true));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, true));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xf, 0xf, true));
  const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = max((uint32_t)a[0], (uint32_t)a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return max((uint32_t)b[0], (uint32_t)b[1]);
}
// The same for up to 64 R experts, of which k is at most GATE_ROUNDS, without LDS but for the k selected: the lane keeps the logits of experts
// lane + 64 j, and a round takes the largest of what is left (a butterfly within the wave and a ballot, some 120 clocks; by rank the token's
// 128 scores were compared with every lane's through LDS, 3 us).  Same sums, selection and weights bit for bit.
constexpr int GATE_ROUNDS = 16;
template <int R>
__device__ __forceinline__ void gate_select_rounds(const GateArgs& a, float (&v)[R], int64_t tok, float* tv, int* ti, int lane) {
  const bool poly = a.E > 16 && !a.exp_accurate;
  float mx = -3.402823466e+38f;
#pragma unroll
  for (int j = 0; j < R; j++)
    if (lane + 64 * j < a.E) mx = fmaxf(mx, v[j]);
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < R; j++) {
    const int i = lane + 64 * j;
    if (i < a.E) {
      v[j] = softmax_exp(v[j] - mx, poly && i < (a.E & ~7));
      sum += v[j];
    }
  }
  sum = wave_sum(sum);
  const float inv = 1.f / sum;
  uint32_t key[R];
  unsigned long long taken[R];
#pragma unroll
  for (int j = 0; j < R; j++) {
    const int i = lane + 64 * j;
    v[j] *= inv;
    if (a.scores && i < a.E) a.scores[tok * a.E + i] = v[j];
    key[j] = i < a.E ? max((uint32_t)(order_key(v[j], 0, true) >> 32), 1u) : 0u;
    taken[j] = 0;
  }
  for (int r = 0; r < a.k; r++) {
    uint32_t m = key[0];
#pragma unroll
    for (int j = 1; j < R; j++) m = max(m, key[j]);
    m = wave_max_u32(m);
    bool found = false;  // (uniform) the lowest index among equal ones
#pragma unroll
    for (int j = 0; j < R; j++) {
      const unsigned long long at = __ballot(key[j] == m);
      if (!found && at) {
        const unsigned long long one = at & (0ull - at);
        taken[j] |= one;
        if ((one >> lane) & 1) key[j] = 0u;
        found = true;
      }
    }
  }
  int before = 0;
#pragma unroll
  for (int j = 0; j < R; j++) {
    if ((taken[j] >> lane) & 1) {
      const int pos = before + __popcll(taken[j] & ((1ull << lane) - 1ull));
      tv[pos] = v[j];
      ti[pos] = lane + 64 * j;
    }
    before += __popcll(taken[j]);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  float tsum = 0.f;
  for (int r = 0; r < a.k; r++) tsum += tv[r];
  if (lane < a.k) {
    const float wv = tv[lane];
    a.weights[tok * a.k + lane] = a.norm ? wv / tsum : wv;
    a.ids[tok * a.k + lane] = ti[lane];
  }
}
// one wave finishes one token: softmax over its E logits in lg (LDS, overwritten), the k largest in index order, weights
__device__ __forceinline__ void gate_select(const GateArgs& a, float* lg, int64_t tok, float* tv, int* ti, int lane) {
  const bool poly = a.E > 16 && !a.exp_accurate;
  float mx = -3.402823466e+38f;
  for (int i = lane; i < a.E; i += 64) mx = fmaxf(mx, lg[i]);
  mx = wave_max(mx);
  float sum = 0.f;
  for (int i = lane; i < a.E; i += 64) {
    const float ex = softmax_exp(lg[i] - mx, poly && i < (a.E & ~7));
    lg[i] = ex;
    sum += ex;
  }
  sum = wave_sum(sum);
  const float inv = 1.f / sum;
  for (int i = lane; i < a.E; i += 64) {
    const float p = lg[i] * inv;
    lg[i] = p;
    if (a.scores) a.scores[tok * a.E + i] = p;
  }
  // LDS writes of this wave are read back by other lanes of the same wave only
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  if (a.E <= 128) wave_topk_ranked<2>(lg, a.E, a.k, true, false, tv, ti, lane);
  else if (a.E <= 256) wave_topk_ranked<4>(lg, a.E, a.k, true, false, tv, ti, lane);
  else wave_topk(lg, a.E, a.k, true, false, tv, ti, lane);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  // topk(..., largest = true, sorted = false): by index; then weight / sum(weights) in index order
  float tsum = 0.f;
  for (int r = 0; r < a.k; r++) tsum += tv[r];
  for (int r = lane; r < a.k; r += 64) {
    const float wv = tv[r];
    a.weights[tok * a.k + r] = a.norm ? wv / tsum : wv;
    a.ids[tok * a.k + r] = ti[r];
  }
}
// the logits of a token, in LDS or in memory -> its experts; lg: LDS for them
__device__ __forceinline__ void gate_finish(const GateArgs& a, const float* logits, float* lg, int64_t tok, float* tv, int* ti, int lane) {
  auto rounds = [&](auto held) {
    float(&v)[sizeof(held) / sizeof(float)] = held.v;
#pragma unroll
    for (int j = 0; j < (int)(sizeof(held) / sizeof(float)); j++) v[j] = lane + 64 * j < a.E ? logits[lane + 64 * j] : 0.f;
    gate_select_rounds(a, v, tok, tv, ti, lane);
  };
  struct Two { float v[2]; };
  struct Four { float v[4]; };
  if (a.k <= GATE_ROUNDS && a.E <= 128) return rounds(Two{});
  if (a.k <= GATE_ROUNDS && a.E <= 256) return rounds(Four{});
  if (logits != lg) {
    for (int i = lane; i < a.E; i += 64) lg[i] = logits[i];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  gate_select(a, lg, tok, tv, ti, lane);
}
// everything in one launch: a workgroup per four tokens (callers that pass no scores buffer)
template <int XT, bool AHEAD>
__global__ __launch_bounds__(GATE_WAVES * 64) void moe_gate_kernel(GateArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  float* s_x = reinterpret_cast<float*>(smem);     // [GATE_TOK][H]
  float* s_logit = s_x + (size_t)GATE_TOK * a.H;   // [GATE_TOK][E]
  float* s_tv = s_logit + (size_t)GATE_TOK * a.E;  // [GATE_TOK][k]
  int* s_ti = reinterpret_cast<int*>(s_tv + (size_t)GATE_TOK * a.k);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t tok0 = (int64_t)blockIdx.x * GATE_TOK;
  const int ntok = (int)min((int64_t)GATE_TOK, a.M - tok0);  // uniform
  GatePieces first;
  if (AHEAD) gate_request(a, wave, lane, first);
  gate_stage_x<XT>(a, tok0, ntok, s_x, tid, GATE_WAVES * 64);
  __syncthreads();
  gate_logits<AHEAD>(a, s_x, ntok, 0, a.E, wave, GATE_WAVES, lane, first, s_logit, (size_t)a.E);
  __syncthreads();
  if (wave >= ntok) return;
  gate_finish(a, s_logit + wave * a.E, s_logit + wave * a.E, tok0 + wave, s_tv + wave * a.k, s_ti + wave * a.k, lane);
}
// The same in two launches for callers that pass a scores buffer, which holds the logits in between: with few tokens one
// workgroup per four tokens leaves the chip to one CU (a decode token: 1 MB of gate weights through one workgroup), so the
// experts are spread over the grid's y -- epg experts and as many waves per workgroup -- and a second, small launch
// finishes each token.  Same logits, same selection.
template <int XT, bool AHEAD>
__global__ __launch_bounds__(GATE_WAVES * 64) void moe_gate_logits_kernel(GateArgs a, int epg) {
  extern __shared__ __align__(16) unsigned char smem[];
  float* s_x = reinterpret_cast<float*>(smem);  // [GATE_TOK][H]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nthreads = blockDim.x;
  const int64_t tok0 = (int64_t)blockIdx.x * GATE_TOK;
  const int ntok = (int)min((int64_t)GATE_TOK, a.M - tok0);  // uniform
  const int e0 = (int)blockIdx.y * epg;
  GatePieces first;
  if (AHEAD) gate_request(a, e0 + wave, lane, first);
  gate_stage_x<XT>(a, tok0, ntok, s_x, tid, nthreads);
  __syncthreads();
  gate_logits<AHEAD>(a, s_x, ntok, e0, min(a.E, e0 + epg), wave, nthreads >> 6, lane, first, a.scores + tok0 * a.E, (size_t)a.E);
}
__global__ __launch_bounds__(GATE_TOK * 64) void moe_gate_select_kernel(GateArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  float* s_logit = reinterpret_cast<float*>(smem);  // [GATE_TOK][E]
  float* s_tv = s_logit + (size_t)GATE_TOK * a.E;   // [GATE_TOK][k]
  int* s_ti = reinterpret_cast<int*>(s_tv + (size_t)GATE_TOK * a.k);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t tok = (int64_t)blockIdx.x * GATE_TOK + wave;
  if (tok >= a.M) return;  // (no workgroup barrier below)
  gate_finish(a, a.scores + tok * a.E, s_logit + wave * a.E, tok, s_tv + wave * a.k, s_ti + wave * a.k, lane);
}

}  // namespace mllmhip

using namespace mllmhip;

static int g_exp_accurate = 0;
namespace mllmhip {
int exp_mode_accurate() { return g_exp_accurate; }
}
MLLM_API int mllm_hip_set_exp_mode(int accurate) {
  if (accurate != 0 && accurate != 1) return MLLM_HIP_E_BADARG;
  g_exp_accurate = accurate;
  return 0;
}

static bool dtype_ok(int t) { return t == MLLM_HIP_F32 || t == MLLM_HIP_BF16; }
static bool al16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// image argument checks shared by the producers: rows <= 8, D a multiple of 32
static int make_image(void* q_image, int64_t rows, int64_t D, int act_scale_mode, QImage& q) {
  q = QImage{nullptr, 0, 0, 0};
  if (!q_image) return 0;
  if (act_scale_mode != MLLM_HIP_SCALE_IEEE && act_scale_mode != MLLM_HIP_SCALE_X86_REF) return MLLM_HIP_E_BADARG;
  if (rows < 1 || rows > 8 || D % QK) return MLLM_HIP_E_SHAPE;
  if (!al16(q_image)) return MLLM_HIP_E_ALIGN;
  q.base = reinterpret_cast<unsigned char*>(q_image);
  q.MT = rows <= 1 ? 1 : (rows <= 2 ? 2 : (rows <= 4 ? 4 : 8));
  q.nb = (int)(D / QK);
  q.x86_scale = act_scale_mode == MLLM_HIP_SCALE_X86_REF;
  return 0;
}

MLLM_API int mllm_hip_rmsnorm(const void* x, int dtype, const float* weight, void* y, int64_t rows, int64_t D, float epsilon,
                              int add_unit_offset, void* q_image, int act_scale_mode, void* stream) {
  if (!x || !weight || !y || !dtype_ok(dtype) || rows <= 0 || D <= 0) return MLLM_HIP_E_BADARG;
  if (D % 8 || D > 8 * 256 * 8 || rows > 0x7fffffff) return MLLM_HIP_E_SHAPE;
  if (!al16(x) || !al16(y) || !al16(weight)) return MLLM_HIP_E_ALIGN;
  RmsArgs a{x, weight, y, rows, (int)D, epsilon, add_unit_offset, {}};
  int rc = make_image(q_image, rows, D, act_scale_mode, a.img);
  if (rc) return rc;
  const unsigned grid = (unsigned)(a.img.base ? a.img.MT : rows);
  const int ni = (int)((D / 8 + 255) / 256);
  hipStream_t st = (hipStream_t)stream;
#define RMS(XT_, NI_) hipLaunchKernelGGL((rmsnorm_kernel<XT_, NI_>), dim3(grid), dim3(256), 0, st, a)
#define RMS_T(XT_)        \
  if (ni <= 1) RMS(XT_, 1); \
  else if (ni <= 2) RMS(XT_, 2); \
  else if (ni <= 4) RMS(XT_, 4); \
  else RMS(XT_, 8)
  if (dtype == MLLM_HIP_F32) {
    RMS_T(MLLM_HIP_F32);
  } else {
    RMS_T(MLLM_HIP_BF16);
  }
#undef RMS_T
#undef RMS
  return (int)hipGetLastError();
}

template <int OP>
static int launch_elementwise(const void* a_, const void* b_, void* y, int dtype, int64_t rows, int64_t D, void* q_image,
                              int act_scale_mode, void* stream) {
  if (!a_ || (OP != EW_SILU && !b_) || !y || !dtype_ok(dtype) || rows <= 0 || D <= 0) return MLLM_HIP_E_BADARG;
  if (D % 8 || D > 0x7fffffff) return MLLM_HIP_E_SHAPE;
  if (!al16(a_) || !al16(b_) || !al16(y)) return MLLM_HIP_E_ALIGN;
  EwArgs a{a_, b_, y, rows, (int)D, g_exp_accurate, {}};
  int rc = make_image(q_image, rows, D, act_scale_mode, a.img);
  if (rc) return rc;
  const int64_t total_rows = a.img.base ? a.img.MT : rows;
  const int64_t items = total_rows * (D / 8);
  if ((items + 255) / 256 > 0x7fffffff) return MLLM_HIP_E_SHAPE;
  const unsigned grid = (unsigned)((items + 255) / 256);
  hipStream_t st = (hipStream_t)stream;
  if constexpr (OP == EW_SILU || OP == EW_SILU_MUL) {
    if (!a.img.base && items <= EW_PAIRS_ITEMS) {
      const dim3 pairs((unsigned)((items * 4 + 255) / 256));
      if (dtype == MLLM_HIP_F32) hipLaunchKernelGGL((elementwise_pairs_kernel<MLLM_HIP_F32, OP>), pairs, dim3(256), 0, st, a);
      else hipLaunchKernelGGL((elementwise_pairs_kernel<MLLM_HIP_BF16, OP>), pairs, dim3(256), 0, st, a);
      return (int)hipGetLastError();
    }
  }
  if (dtype == MLLM_HIP_F32)
    hipLaunchKernelGGL((elementwise_kernel<MLLM_HIP_F32, OP>), dim3(grid), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((elementwise_kernel<MLLM_HIP_BF16, OP>), dim3(grid), dim3(256), 0, st, a);
  return (int)hipGetLastError();
}

MLLM_API int mllm_hip_silu(const void* x, void* y, int dtype, int64_t n, void* stream) {
  if (n <= 0 || n % 8) return n <= 0 ? MLLM_HIP_E_BADARG : MLLM_HIP_E_SHAPE;
  return launch_elementwise<EW_SILU>(x, nullptr, y, dtype, n / 8, 8, nullptr, 0, stream);
}
MLLM_API int mllm_hip_add(const void* a, const void* b, void* y, int dtype, int64_t rows, int64_t D, void* q_image,
                          int act_scale_mode, void* stream) {
  return launch_elementwise<EW_ADD>(a, b, y, dtype, rows, D, q_image, act_scale_mode, stream);
}
MLLM_API int mllm_hip_mul(const void* a, const void* b, void* y, int dtype, int64_t rows, int64_t D, void* q_image,
                          int act_scale_mode, void* stream) {
  return launch_elementwise<EW_MUL>(a, b, y, dtype, rows, D, q_image, act_scale_mode, stream);
}
MLLM_API int mllm_hip_silu_mul(const void* gate, const void* up, void* y, int dtype, int64_t rows, int64_t D, void* q_image,
                               int act_scale_mode, void* stream) {
  return launch_elementwise<EW_SILU_MUL>(gate, up, y, dtype, rows, D, q_image, act_scale_mode, stream);
}

MLLM_API int mllm_hip_softmax(const float* x, float* y, int64_t rows, int64_t len, void* stream) {
  if (!x || !y || rows <= 0 || len <= 0) return MLLM_HIP_E_BADARG;
  if (len > 0x7fffffff || (rows + 3) / 4 > 0x7fffffff) return MLLM_HIP_E_SHAPE;
  const dim3 grid4((unsigned)((rows + 3) / 4));
  hipStream_t st = (hipStream_t)stream;
  if (len <= 256) hipLaunchKernelGGL(softmax_rows_reg_kernel<4>, grid4, dim3(256), 0, st, x, y, rows, (int)len, g_exp_accurate);
  else if (len <= 1024) hipLaunchKernelGGL(softmax_rows_reg_kernel<16>, grid4, dim3(256), 0, st, x, y, rows, (int)len, g_exp_accurate);
  else if (len <= 2048) hipLaunchKernelGGL(softmax_rows_reg_kernel<32>, grid4, dim3(256), 0, st, x, y, rows, (int)len, g_exp_accurate);
  else if (len <= 4096 && rows <= 0x7fffffff) hipLaunchKernelGGL(softmax_wg_rows_kernel<16>, dim3((unsigned)rows), dim3(256), 0, st, x, y, (int)len, g_exp_accurate);
  else if (len <= 8192 && rows <= 0x7fffffff) hipLaunchKernelGGL(softmax_wg_rows_kernel<32>, dim3((unsigned)rows), dim3(256), 0, st, x, y, (int)len, g_exp_accurate);
  else if (len <= 16384 && rows <= 0x7fffffff) hipLaunchKernelGGL(softmax_wg_rows_kernel<64>, dim3((unsigned)rows), dim3(256), 0, st, x, y, (int)len, g_exp_accurate);
  else if (len >= 16384 && rows <= 0x7fffffff) hipLaunchKernelGGL(softmax_long_rows_kernel, dim3((unsigned)rows), dim3(SOFTMAX_WG), 0, st, x, y, (int)len, g_exp_accurate);
  else hipLaunchKernelGGL(softmax_rows_kernel, grid4, dim3(256), 0, st, x, y, rows, (int)len, g_exp_accurate);
  return (int)hipGetLastError();
}

MLLM_API int mllm_hip_topk(const float* x, float* values, int32_t* indices, int64_t rows, int64_t len, int k, int largest,
                           int sorted, void* stream) {
  if (!x || !values || !indices || rows <= 0 || len <= 0) return MLLM_HIP_E_BADARG;
  if (k < 1 || k > len || len > 0x7fffffff || (rows + 3) / 4 > 0x7fffffff) return MLLM_HIP_E_SHAPE;
  if (len > 256 && k <= TOPK_SEL_MAX && rows <= 0x7fffffff) {
    const bool vec = len % 4 == 0 && ((uintptr_t)x & 15) == 0;
    const int64_t units = vec ? len / 4 : len;
    const dim3 grid((unsigned)rows);
    hipStream_t st = (hipStream_t)stream;
#define TOPK_SELECT(NT, R, WIDE) \
  do { \
    if (vec) hipLaunchKernelGGL((topk_select_rows_kernel<NT, 4, R, WIDE>), grid, dim3(NT), 0, st, x, values, indices, (int)len, k, largest, sorted); \
    else hipLaunchKernelGGL((topk_select_rows_kernel<NT, 1, R, WIDE>), grid, dim3(NT), 0, st, x, values, indices, (int)len, k, largest, sorted); \
  } while (0)
    if (units <= 256) TOPK_SELECT(256, 1, false);  // (loads per thread that hold the row: no empty slots to step over)
    else if (units <= 512) TOPK_SELECT(256, 2, false);
    else if (units <= 1024) TOPK_SELECT(256, 4, false);
    else if (units <= 2048) TOPK_SELECT(256, 8, false);
    else if (units <= 4096) TOPK_SELECT(1024, 4, false);
    else if (units <= 8192) TOPK_SELECT(1024, 8, false);
    else TOPK_SELECT(1024, 8, true);
#undef TOPK_SELECT
  } else if (len >= 8192 && rows <= 0x7fffffff)
    hipLaunchKernelGGL(topk_long_rows_kernel, dim3((unsigned)rows), dim3(TOPK_WG), 0, (hipStream_t)stream, x, values, indices, (int)len, k,
                       largest, sorted);
  else
    hipLaunchKernelGGL(topk_rows_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, (hipStream_t)stream, x, values, indices, rows,
                       (int)len, k, largest, sorted);
  return (int)hipGetLastError();
}

// Pieces of a row that few long rows are cut into, 0 where a workgroup per row is the better form
static int softmax_pieces(int64_t rows, int64_t len) {
  return len > (rows > 192 && rows <= 256 ? SOFTMAX_LONG_ROUND : SOFTMAX_LONG) && rows <= SOFTMAX_SPLIT_ROWS && len <= 0x7fffffff ? (int)((len + SOFTMAX_PIECE - 1) / SOFTMAX_PIECE) : 0;
}
MLLM_API size_t mllm_hip_softmax_workspace_bytes(int64_t rows, int64_t len) {
  if (rows <= 0 || len <= 0) return 0;
  return (size_t)rows * softmax_pieces(rows, len) * 2 * sizeof(float);
}
MLLM_API int mllm_hip_softmax_set_wait(int polls) {
  if (polls < -1) return MLLM_HIP_E_BADARG;
  g_softmax_polls = std::min(polls, SOFTMAX_LOOKS);
  return 0;
}
MLLM_API int mllm_hip_softmax_wait(void) { return g_softmax_polls; }
MLLM_API int mllm_hip_softmax_ws(const float* x, float* y, int64_t rows, int64_t len, void* workspace, void* stream) {
  const int pieces = workspace && rows > 0 && len > 0 ? softmax_pieces(rows, len) : 0;
  if (!pieces) return mllm_hip_softmax(x, y, rows, len, stream);
  if (!x || !y) return MLLM_HIP_E_BADARG;
  if (reinterpret_cast<uintptr_t>(workspace) % 4) return MLLM_HIP_E_ALIGN;
  const dim3 grid((unsigned)pieces, (unsigned)rows);
  hipStream_t st = (hipStream_t)stream;
  float* ws = reinterpret_cast<float*>(workspace);
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, x, y, ws, (int)len, g_exp_accurate, g_softmax_polls); };
  go(softmax_pieces_kernel<0>);
  // results over the input: a workgroup that adds up the row by itself would read what another one has written already
  const uintptr_t xa = reinterpret_cast<uintptr_t>(x), ya = reinterpret_cast<uintptr_t>(y), bytes = (uintptr_t)rows * (uintptr_t)len * 4;
  const bool apart = xa + bytes <= ya || ya + bytes <= xa;
  if (apart && pieces <= SOFTMAX_WAIT_PIECES && pieces * rows <= SOFTMAX_WAIT && g_softmax_polls >= 0) {
    go(softmax_pieces_kernel<3>);
  } else {
    go(softmax_pieces_kernel<1>);
    go(softmax_pieces_kernel<2>);
  }
  return (int)hipGetLastError();
}

// Pieces of a row, 0 where a workgroup per row is the better form.  vec: rows of whole aligned 16-byte vectors.  The largest 50, us, a
// workgroup per row / pieces: 8 rows of 4100 elements 20.9 / 14.8, of 8192 26.0 / 15.0, of 151 936 113 / 16.6; 512 rows of 8192 29.0 / 18.8.
// Element by element the pieces load slower than the row's workgroup, which holds up to 8192 elements in registers: 8 rows of 4097
// 12.6 / 16.6, of 8191 14.1 / 15.5, of 8193 26.7 / 15.3; where the rows need a second round of workgroups pieces pay there too (300
// rows of 4097: 0.87 of the time).
static int topk_pieces(int64_t rows, int64_t len, int k, bool vec) {
  if (len <= TOPK_SPLIT_LEN || rows > TOPK_SPLIT_ROWS || k < 1 || k > TOPK_SPLIT_K || len > 0x7fffffff) return 0;
  if (!vec && len <= 8192 && rows <= 256) return 0;
  const int64_t pieces = (len + TOPK_PIECE - 1) / TOPK_PIECE;
  return pieces * k <= 256 * TOPK_MERGE_R ? (int)pieces : 0;
}
MLLM_API size_t mllm_hip_topk_workspace_bytes(int64_t rows, int64_t len, int k) {
  if (rows <= 0 || len <= 0) return 0;
  return (size_t)rows * topk_pieces(rows, len, k, len % 4 == 0) * (k > 0 ? k : 0) * sizeof(unsigned long long);
}
MLLM_API int mllm_hip_topk_ws(const float* x, float* values, int32_t* indices, int64_t rows, int64_t len, int k, int largest, int sorted,
                              void* workspace, void* stream) {
  const bool vec = len % 4 == 0 && ((uintptr_t)x & 15) == 0;
  const int pieces = workspace && rows > 0 && len > 0 ? topk_pieces(rows, len, k, vec) : 0;
  if (!pieces) return mllm_hip_topk(x, values, indices, rows, len, k, largest, sorted, stream);
  if (!x || !values || !indices) return MLLM_HIP_E_BADARG;
  if (reinterpret_cast<uintptr_t>(workspace) % 8) return MLLM_HIP_E_ALIGN;
  const dim3 grid((unsigned)pieces, (unsigned)rows);
  hipStream_t st = (hipStream_t)stream;
  unsigned long long* ws = reinterpret_cast<unsigned long long*>(workspace);
  const int units = (int)(vec ? len / 4 : len), per = (units + pieces - 1) / pieces;  // (at most TOPK_PIECE elements)
  if (vec) hipLaunchKernelGGL(topk_pieces_kernel<4>, grid, dim3(256), 0, st, x, ws, (int)len, per, k, largest);
  else hipLaunchKernelGGL(topk_pieces_kernel<1>, grid, dim3(256), 0, st, x, ws, (int)len, per, k, largest);
  if (pieces * k <= 1024) hipLaunchKernelGGL(topk_merge_kernel<4>, dim3((unsigned)rows), dim3(256), 0, st, x, ws, values, indices, (int)len, pieces * k, k, largest, sorted);
  else hipLaunchKernelGGL(topk_merge_kernel<TOPK_MERGE_R>, dim3((unsigned)rows), dim3(256), 0, st, x, ws, values, indices, (int)len, pieces * k, k, largest, sorted);
  return (int)hipGetLastError();
}

static int g_gate_two_launches = 1;  // 0: the one-launch form also where a scores buffer is given (comparison runs and tests)
MLLM_API int mllm_hip_moe_gate_set_form(int two_launches) {
  if (two_launches != 0 && two_launches != 1) return MLLM_HIP_E_BADARG;
  g_gate_two_launches = two_launches;
  return 0;
}

MLLM_API int mllm_hip_moe_gate(const void* x, int x_dtype, const float* gate_weight, int32_t* topk_ids, float* topk_weights,
                               float* scores, int64_t M, int64_t H, int64_t E, int k, int norm_topk_prob, void* stream) {
  if (!x || !gate_weight || !topk_ids || !topk_weights || !dtype_ok(x_dtype) || M <= 0 || H <= 0 || E <= 0) return MLLM_HIP_E_BADARG;
  if (k < 1 || k > E || H % 8 || (M + GATE_TOK - 1) / GATE_TOK > 0x7fffffff) return MLLM_HIP_E_SHAPE;
  if (!al16(x) || !al16(gate_weight)) return MLLM_HIP_E_ALIGN;
  const size_t lds = ((size_t)GATE_TOK * H + (size_t)GATE_TOK * E + (size_t)2 * GATE_TOK * k) * 4;
  if (lds > 160 * 1024) return MLLM_HIP_E_SHAPE;
  GateArgs a{x, gate_weight, topk_ids, topk_weights, scores, M, (int)H, (int)E, k, norm_topk_prob, g_exp_accurate};
  const unsigned grid = (unsigned)((M + GATE_TOK - 1) / GATE_TOK);
  hipStream_t st = (hipStream_t)stream;
  if (scores && g_gate_two_launches) {
    // experts per workgroup: four (one per wave) while the token groups alone do not fill the chip, else sixteen
    const int epg = grid >= 64 ? 16 : 4;
    const size_t lds1 = (size_t)GATE_TOK * H * 4, lds2 = ((size_t)GATE_TOK * E + (size_t)2 * GATE_TOK * k) * 4;
    auto go = [&](auto kern) -> int {
      if (lds1 > 64 * 1024)
        HIP_RET(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds1));
      hipLaunchKernelGGL(kern, dim3(grid, (unsigned)((E + epg - 1) / epg)), dim3(64 * epg), lds1, st, a, epg);
      return (int)hipGetLastError();
    };
    // weights ahead of x: 78 registers, so that a CU holds one workgroup of sixteen waves instead of two.  us without / with: 512 tokens, 128 experts of 2048
    // 16.2 / 20.9, 2048 tokens 45 / 65, 512 tokens, 300 experts 50 / 62; in one round 7.4 / 7.4 (256 tokens, 64 of 1024).  Workgroups of four waves do not
    // mind: 8 tokens 8.4 / 8.3, 192 13.2 / 13.6
    const bool ahead = epg == 4;
    RC_RET(x_dtype == MLLM_HIP_F32 ? ahead ? go(moe_gate_logits_kernel<MLLM_HIP_F32, true>) : go(moe_gate_logits_kernel<MLLM_HIP_F32, false>)
           : ahead                 ? go(moe_gate_logits_kernel<MLLM_HIP_BF16, true>)
                                   : go(moe_gate_logits_kernel<MLLM_HIP_BF16, false>));
    if (lds2 > 64 * 1024)
      HIP_RET(hipFuncSetAttribute(reinterpret_cast<const void*>(moe_gate_select_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds2));
    hipLaunchKernelGGL(moe_gate_select_kernel, dim3(grid), dim3(GATE_TOK * 64), lds2, st, a);
    return (int)hipGetLastError();
  }
  auto launch = [&](auto kern) -> int {
    if (lds > 64 * 1024)
      HIP_RET(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3(grid), dim3(GATE_WAVES * 64), lds, st, a);
    return (int)hipGetLastError();
  };
  // weights ahead of x while there is one workgroup per CU at most (84 registers, see above): 128 experts of 2048, us without / with: 8 tokens 23.8 / 22.1,
  // 1024 24.6 / 23.8, 2048 37 / 43
  const bool ahead = grid <= 256;
  return x_dtype == MLLM_HIP_F32 ? ahead ? launch(moe_gate_kernel<MLLM_HIP_F32, true>) : launch(moe_gate_kernel<MLLM_HIP_F32, false>)
         : ahead                 ? launch(moe_gate_kernel<MLLM_HIP_BF16, true>)
                                 : launch(moe_gate_kernel<MLLM_HIP_BF16, false>);
}

// Q4_K / Q6_K Linear for gfx950: super-block formats of 256 weights with Q8_K activations (the formats the shipped
// Qwen3-MoE recipe quantizes to).  Decode GEMV for up to eight activation rows; more rows run as groups of eight.
//
// Arithmetic follows the reference's x86 CPU path:
//   activation quantization  quantize_row_q8_K_reference   mllm/backends/cpu/kernels/common/ggml/quantize/quantize_q8.cpp:215-248
//   Q4_K dot                 vec_dot_q4_K_q8_K (AVX2)       mllm/backends/cpu/kernels/common/ggml/vec_dot.cpp:498-560
//   Q6_K dot                 vec_dot_q6_K_q8_K (AVX2)       mllm/backends/cpu/kernels/common/ggml/vec_dot.cpp:955-1044
//   dequantization probes    dequantize_row_q4_K / _q6_K    quantize_q4.cpp:284-312, quantize_q6.cpp:108-133
//   call site                ggml::mat_mul generic branch    mllm/backends/cpu/kernels/common/ggml/matmul.cpp:147-189,300-360
// The integer work (codes, sums of 16, sub-block-scaled dot products per super-block) is exact; the fp32 accumulation
// runs per lane and is reduced over the lanes of a row, a different order than the CPU's eight lanes.
//
// HBM-bound like the Q4_0 / Q8_0 GEMV: a launch streams 144 (Q4_K) or 210 (Q6_K) bytes per 256 weights once, as 16-byte
// loads that are contiguous across the lanes of a group.  The reference's array-of-structures blocks (210 is not even a
// multiple of 4) are split at load time into planes of 16-byte records.
#include <initializer_list>

#include "qcommon.h"
#include "qgemm_layout.h"

#include "kquant_layout.h"

namespace mllmhip {

// what an fp16 field reads as: the IEEE pattern itself, or (files of the x86 build) the number stored there taken as
// the pattern
__device__ __forceinline__ uint16_t field_bits(const uint8_t* p, int x86) {
  const uint16_t raw = (uint16_t)p[0] | ((uint16_t)p[1] << 8);
  if (!x86) return raw;
  const float num = f16bits_to_f32(raw);
  return (num >= 0.f && num < 65536.f) ? (uint16_t)(uint32_t)num : (uint16_t)0;
}
__device__ __forceinline__ uint32_t bytes_u32(const uint8_t* p) {
  return (uint32_t)p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16) | ((uint32_t)p[3] << 24);
}

// ---- scale decoding ----------------------------------------------------------------------------------------------------
// the 6-bit scales and mins of a Q4_K super-block as bytes: sc[0..7] in (lo, hi) of `sc`, mins likewise
// (get_scale_min_k4, quantize.hpp; the same bit shuffle as vec_dot.cpp:507-512)
struct K4Scales {
  uint32_t sc0, sc1, mn0, mn1;
};
__device__ __forceinline__ K4Scales k4_scales(uint32_t u0, uint32_t u1, uint32_t u2) {
  K4Scales r;
  r.mn1 = ((u2 >> 4) & 0x0f0f0f0fu) | (((u1 >> 6) & 0x03030303u) << 4);
  r.mn0 = u1 & 0x3f3f3f3fu;
  r.sc1 = (u2 & 0x0f0f0f0fu) | (((u0 >> 6) & 0x03030303u) << 4);
  r.sc0 = u0 & 0x3f3f3f3fu;
  return r;
}
__device__ __forceinline__ int byte_of(uint32_t lo, uint32_t hi, int k) {  // k = 0..7
  return (int)(((k < 4 ? lo : hi) >> (8 * (k & 3))) & 0xffu);
}

// one thread per 16-byte record of plane A (Q4_K: 8 per super-block; Q6_K: 8 per super-block); thread 0 of a super-block
// also writes the small planes
__global__ void kq_prepack_kernel(int wtype, const uint8_t* __restrict__ blocks, int x86, KView v, int64_t nsb_total) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t sb = i >> 3;
  const int c = (int)(i & 7);
  if (sb >= nsb_total) return;
  u32x4* A = const_cast<u32x4*>(v.a);
  u32x4* S = const_cast<u32x4*>(v.s);
  if (wtype == MLLM_HIP_Q4_K) {
    const uint8_t* b = blocks + sb * 144;
    const uint8_t* q = b + 16 + 16 * c;
    A[sb * 8 + c] = u32x4{bytes_u32(q), bytes_u32(q + 4), bytes_u32(q + 8), bytes_u32(q + 12)};
    if (c == 0) {
      const K4Scales k = k4_scales(bytes_u32(b + 4), bytes_u32(b + 8), bytes_u32(b + 12));
      uint32_t rec[4];
#pragma unroll
      for (int p = 0; p < 4; p++)
        rec[p] = (uint32_t)byte_of(k.sc0, k.sc1, 2 * p) | ((uint32_t)byte_of(k.sc0, k.sc1, 2 * p + 1) << 8) |
                 ((uint32_t)byte_of(k.mn0, k.mn1, 2 * p) << 16) | ((uint32_t)byte_of(k.mn0, k.mn1, 2 * p + 1) << 24);
      S[sb] = u32x4{rec[0], rec[1], rec[2], rec[3]};
      reinterpret_cast<uint32_t*>(const_cast<uint16_t*>(v.d))[sb] = (uint32_t)field_bits(b, x86) | ((uint32_t)field_bits(b + 2, x86) << 16);
    }
  } else {
    const uint8_t* b = blocks + sb * 210;
    const uint8_t* q = b + 16 * c;
    A[sb * 8 + c] = u32x4{bytes_u32(q), bytes_u32(q + 4), bytes_u32(q + 8), bytes_u32(q + 12)};
    if (c < 4) {
      const uint8_t* hq = b + 128 + 16 * c;
      const_cast<u32x4*>(v.h)[sb * 4 + c] = u32x4{bytes_u32(hq), bytes_u32(hq + 4), bytes_u32(hq + 8), bytes_u32(hq + 12)};
    }
    if (c == 0) {
      const uint8_t* s = b + 192;
      S[sb] = u32x4{bytes_u32(s), bytes_u32(s + 4), bytes_u32(s + 8), bytes_u32(s + 12)};
      const_cast<uint16_t*>(v.d)[sb] = field_bits(b + 208, x86);
    }
  }
}

// ---- dequantization probe ------------------------------------------------------------------------------------------------
__global__ void kq_dequantize_kernel(int wtype, KView v, float* __restrict__ w, int64_t nsb_total) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // one thread per element
  const int64_t sb = i >> 8;
  const int e = (int)(i & 255);
  if (sb >= nsb_total) return;
  const uint8_t* A = reinterpret_cast<const uint8_t*>(v.a) + sb * 128;
  if (wtype == MLLM_HIP_Q4_K) {
    const uint32_t dd = reinterpret_cast<const uint32_t*>(v.d)[sb];
    const float d = f16bits_to_f32((uint16_t)(dd & 0xffff)), mn = f16bits_to_f32((uint16_t)(dd >> 16));
    const int j = e >> 5, l = e & 31;  // sub-block, element
    const uint32_t rec = reinterpret_cast<const uint32_t*>(v.s)[sb * 4 + (j >> 1)];
    const int q = (j & 1) ? (A[32 * (j >> 1) + l] >> 4) : (A[32 * (j >> 1) + l] & 0xF);
    const float d1 = d * (float)((rec >> (8 * (j & 1))) & 0xffu), m1 = mn * (float)((rec >> (16 + 8 * (j & 1))) & 0xffu);
    w[i] = d1 * (float)q - m1;
  } else {
    const uint8_t* H = reinterpret_cast<const uint8_t*>(v.h) + sb * 64;
    const int8_t* sc = reinterpret_cast<const int8_t*>(v.s) + sb * 16;
    const int n = e >> 7, r = e & 127, g = r >> 5, l = r & 31;
    int lo = A[64 * n + ((g & 1) ? 32 : 0) + l];
    lo = (g >= 2) ? (lo >> 4) : (lo & 0xF);
    const int hi = (H[32 * n + l] >> (2 * g)) & 3;
    const int q = (int)(int8_t)(lo | (hi << 4)) - 32;
    const float d = f16bits_to_f32(v.d[sb]);
    w[i] = d * (float)sc[e >> 4] * (float)q;
  }
}

// ---- Q8_K quantization of activations ---------------------------------------------------------------------------------------
// 32 neighbouring lanes (half a wave) hold one super-block, eight consecutive elements per lane; both halves of the wave
// must be active or idle as a whole.  The reference takes the element of largest magnitude WITH its sign, the first one
// when several are equal.  Bit patterns as signed integers have the largest positive element as their maximum, as unsigned ones the
// negative one of largest magnitude: two butterflies give both, and only where they are equal in magnitude the first element is looked
// for (the lowest set bit of a ballot over the lanes that hold one, and in that lane its first; a search in every block was a third of
// the instructions).  Quotients: a reciprocal estimate and one Newton step are the correctly rounded 1 / amax for every amax in the
// range (checked for all of its floats), -128 times that is exact, and so is its reciprocal, from amax / 128 in the estimate's place; outside the range
// IEEE divisions.  Codes: the product is
// rounded to fp32, then adding 1.5 * 2^23 rounds to nearest-even as rintf does and leaves the two's-complement code in the
// low byte; the clamp to 127 is an integer min on the bits of that (positive) sum.  Outputs of a lane: its eight codes (two dwords), the sum of its
// eight codes, the block scale.
struct Q8KItem {
  uint32_t q0, q1;
  int sum8;
  float d;
};
__device__ __forceinline__ Q8KItem quantize_q8k_item(const float (&v)[8], int lane) {
  int pos = (int)__float_as_uint(v[0]);
  uint32_t neg = __float_as_uint(v[0]);
#pragma unroll
  for (int e = 1; e < 8; e++) {
    pos = max(pos, (int)__float_as_uint(v[e]));
    neg = max(neg, __float_as_uint(v[e]));
  }
#define Q8K_STEP(ctrl)                                                                                    \
  pos = max(pos, __builtin_amdgcn_update_dpp((int)0x80000000u, pos, ctrl, 0xf, 0xf, false));              \
  neg = max(neg, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)neg, ctrl, 0xf, 0xf, false));
  Q8K_STEP(0xB1)   // lane ^ 1
  Q8K_STEP(0x4E)   // lane ^ 2
  Q8K_STEP(0x141)  // half-row mirror
  Q8K_STEP(0x140)  // row mirror
#undef Q8K_STEP
  const auto p16 = __builtin_amdgcn_permlane16_swap((uint32_t)pos, (uint32_t)pos, false, false);  // lane ^ 16
  const auto n16 = __builtin_amdgcn_permlane16_swap(neg, neg, false, false);
  pos = max((int)p16[0], (int)p16[1]);
  neg = max(n16[0], n16[1]);
  // (no positive element: pos is negative, and neg's magnitude the larger one; no negative one: neg == pos)
  const uint32_t nmag = neg & 0x7fffffffu, am = max((uint32_t)max(pos, 0), nmag);
  bool negative = neg != (uint32_t)pos ? pos < (int)nmag : pos < 0;
  if (__any(pos == (int)nmag && neg != (uint32_t)pos)) {
    float sel = 0.f;  // the lane's first element of that magnitude
#pragma unroll
    for (int e = 7; e >= 0; e--) sel = ((__float_as_uint(v[e]) & 0x7fffffffu) == am) ? v[e] : sel;
    const bool hit = (__float_as_uint(sel) & 0x7fffffffu) == am, below = (__float_as_uint(sel) >> 31) != 0u;
    const unsigned long long mh = __ballot(hit), mn = __ballot(hit && below);
    const uint32_t h32 = (lane & 32) ? (uint32_t)(mh >> 32) : (uint32_t)mh;
    const uint32_t n32 = (lane & 32) ? (uint32_t)(mn >> 32) : (uint32_t)mn;
    negative = (n32 & (h32 & (0u - h32))) != 0u;
  }
  const float amax = __uint_as_float(am);
  Q8KItem r{0u, 0u, 0, 0.f};
  const bool usual = am - 0x1f800000u < 0x40000000u;  // 2^-64 <= amax < 2^64
  float iscale;
  if (__all(usual)) {
    const float y = __builtin_amdgcn_rcpf(amax);
    iscale = fmaf(fmaf(-amax, y, 1.f), y, y) * (negative ? 128.f : -128.f);
    const float w = amax * (negative ? 0x1p-7f : -0x1p-7f);
    r.d = fmaf(fmaf(-iscale, w, 1.f), w, w);
  } else {
    if (amax == 0.f) return r;
    iscale = -128.f / (negative ? -amax : amax);
    r.d = 1.f / iscale;
  }
  uint32_t b[8];
#pragma unroll
  for (int e = 0; e < 8; e++) b[e] = (uint32_t)min((int)__float_as_uint(iscale * v[e] + 12582912.0f), 0x4B40007F);  // bits of 1.5 * 2^23 + 127
  r.q0 = __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u) | __builtin_amdgcn_perm(b[3], b[2], 0x04000c0cu);
  r.q1 = __builtin_amdgcn_perm(b[5], b[4], 0x0c0c0400u) | __builtin_amdgcn_perm(b[7], b[6], 0x04000c0cu);
  r.sum8 = __builtin_amdgcn_sdot4((int)r.q1, 0x01010101, __builtin_amdgcn_sdot4((int)r.q0, 0x01010101, 0, false), false);
  return r;
}

template <int XT>
__device__ __forceinline__ void load8(const void* x, int64_t elem, float (&v)[8]) {
  if (XT == MLLM_HIP_F32) {
    const f32x4* p = reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(x) + elem);
    const f32x4 a = p[0], b = p[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
    const u32x4 r = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(x) + elem);
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int j = 0; j < 4; j++) {
      v[2 * j + 0] = __uint_as_float(w[j] << 16);
      v[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
    }
  }
}

// stand-alone form: codes int8 [rows][K], d fp32 [rows][K/256], sums of 16 int16 [rows][K/16]; items from `valid` on
// (rows beyond the real ones) are written as zeros.  Used as parity probe and, with the three arrays back to back, to
// write the image the GEMV copies into LDS.
constexpr int KQ_IMAGE = 2;  // activation "type": the quantized image instead of activations
__global__ __launch_bounds__(256) void quantize_q8k_kernel(const void* __restrict__ x, int x_dtype, int8_t* __restrict__ codes,
                                                           float* __restrict__ d, int16_t* __restrict__ bsums, int64_t nitems,
                                                           int64_t valid) {
  const int64_t it = (int64_t)blockIdx.x * 256 + threadIdx.x;  // nitems is a multiple of 32: whole half-waves
  if (it >= nitems) return;
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (it < valid) {
    if (x_dtype == MLLM_HIP_F32) load8<MLLM_HIP_F32>(x, it * 8, v);
    else load8<MLLM_HIP_BF16>(x, it * 8, v);
  }
  const Q8KItem r = quantize_q8k_item(v, threadIdx.x & 63);
  *reinterpret_cast<u32x2*>(codes + it * 8) = u32x2{r.q0, r.q1};
  const int s16 = r.sum8 + __builtin_amdgcn_update_dpp(0, r.sum8, 0xB1, 0xf, 0xf, true);  // with the neighbouring lane
  if ((it & 1) == 0) bsums[it >> 1] = (int16_t)s16;
  if ((it & 31) == 0) d[it >> 5] = r.d;
}

// ---- GEMV -------------------------------------------------------------------------------------------------------------
// One launch serves up to four weight matrices that share the activations and K (sibling projections): workgroups
// [wg_start[p], wg_start[p + 1]) belong to part p.
constexpr int KQ_MAX_PARTS = 4;
struct KGemvPart {
  KView w;
  const float* bias;
  float* y;
  int N;
};
struct KGemvArgs {
  KGemvPart part[KQ_MAX_PARTS];
  int wg_start[KQ_MAX_PARTS + 1];
  int nparts;
  const void* x;
  int M, nsb;  // nsb = K / 256
  // MoE slots (M = 1 only): blockIdx.y = slot; its expert's matrices lie slot_ids[slot] * estride bytes further in every plane,
  // its activation row is slot / slot_div, its output row is the slot.  slot_ids == null: a plain Linear.
  const int32_t* slot_ids;
  const float* x2;       // slots with fp32 x only: the activation is silu(x) * x2 (the MLP's product folded into the down GEMV)
  int silu_accurate;     // expf instead of the reference's polynomial (mllm_hip_set_exp_mode)
  int slot_E, slot_div, slot_div_slots;  // experts, pairs per activation row, number of slots (grid y)
  size_t estride;
  // MoE row tiles (matrix-core kernels, quantized image as input): blockIdx.y = a tile of up to eight expert-sorted positions
  // that share an expert.  The image holds img_rows rows; tile row m reads image row row_ids[row0 + m] / row_div (row_ids
  // null: row0 + m) and writes output row out_ids[row0 + m] (null: row0 + m).  tile_expert == null: a plain Linear.
  const int* tile_expert;
  const int* tile_row0;
  const int* tile_rows;
  const int* ntiles;
  const int* row_ids;
  const int* out_ids;
  int row_div;
  int img_rows;  // rows of the image (0: the kernel's row tile MT)
};
// the tile of this workgroup: how many rows it has, where they start, where the expert's matrices lie
struct KTile {
  int rows, row0;
  size_t eoff;
  bool active;
};
__device__ __forceinline__ KTile kq_tile(const KGemvArgs& a) {
  KTile t{a.M, 0, 0, true};
  if (a.tile_expert) {
    const int ti = blockIdx.y;
    if (ti >= min(a.ntiles[0], (int)gridDim.y)) {
      t.active = false;
      return t;
    }
    t.rows = a.tile_rows[ti];
    t.row0 = a.tile_row0[ti];
    t.eoff = (size_t)a.tile_expert[ti] * a.estride;
  }
  return t;
}
__device__ __forceinline__ int kq_tile_in_row(const KGemvArgs& a, const KTile& t, int m) {
  if (!a.tile_expert) return m;
  const int pos = t.row0 + min(m, t.rows - 1);  // rows past the tile repeat its last row; their results are dropped
  return a.row_ids ? a.row_ids[pos] / a.row_div : pos;
}
__device__ __forceinline__ int kq_tile_out_row(const KGemvArgs& a, const KTile& t, int m) {
  if (!a.tile_expert) return m;
  return a.out_ids ? a.out_ids[t.row0 + m] : t.row0 + m;
}
template <typename T>
__device__ __forceinline__ const T* kq_at(const T* p, size_t byte_offset) {
  return reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + byte_offset);
}
#define KBUF_OOB 0xffffffffu
#define KBUF_NT 2

// A unit = what one lane takes per step.  Q4_K: one 16-byte chunk of nibbles = 32 weights (eight units per super-block).
// Q6_K: one 16-byte chunk of high bits with its two chunks of low nibbles = 64 weights (four units per super-block).
template <int WT>
struct KUnit {
  u32x4 a, b, h, s;
  uint16_t d;
};
struct KRsrc {
  __amdgpu_buffer_rsrc_t a, h, s, d;
};

// byte offsets of a lane's first unit in a row; units that are a multiple of eight further on lie a multiple of these steps on
struct KOff {
  uint32_t a, h, s, d;
};
template <int WT>
__device__ __forceinline__ KOff unit_offsets(uint32_t sb_base, int unit) {
  KOff o{};
  if (WT == MLLM_HIP_Q4_K) {
    const uint32_t sb = sb_base + (uint32_t)(unit >> 3);
    o.a = (sb * 8u + (uint32_t)(unit & 7)) * 16u;
    o.s = sb * 16u + (uint32_t)((unit >> 1) & 3) * 4u;  // its pair's scales
    o.d = sb * 4u;
  } else {
    const uint32_t sb = sb_base + (uint32_t)(unit >> 2);
    const uint32_t n = (uint32_t)(unit >> 1) & 1u, t = (uint32_t)unit & 1u;
    o.a = (sb * 8u + 4u * n + t) * 16u;
    o.h = (sb * 4u + 2u * n + t) * 16u;
    o.s = sb * 16u;
    o.d = sb * 2u;
  }
  return o;
}
// the unit `ahead` (uniform) units behind that of o; one that is not there fetches nothing
template <int WT>
__device__ __forceinline__ void load_unit(KUnit<WT>& u, const KRsrc& r, const KOff& o, int ahead, bool ok) {
  if (WT == MLLM_HIP_Q4_K) {
    u.a = __builtin_amdgcn_raw_buffer_load_b128(r.a, ok ? o.a : KBUF_OOB, ahead * 16, KBUF_NT);
    u.s.x = __builtin_amdgcn_raw_buffer_load_b32(r.s, ok ? o.s : KBUF_OOB, ahead * 2, KBUF_NT);
    u.s.y = __builtin_amdgcn_raw_buffer_load_b32(r.d, ok ? o.d : KBUF_OOB, ahead / 2, KBUF_NT);  // d, dmin
  } else {
    u.a = __builtin_amdgcn_raw_buffer_load_b128(r.a, ok ? o.a : KBUF_OOB, ahead * 32, KBUF_NT);
    u.b = __builtin_amdgcn_raw_buffer_load_b128(r.a, ok ? o.a : KBUF_OOB, ahead * 32 + 32, KBUF_NT);
    u.h = __builtin_amdgcn_raw_buffer_load_b128(r.h, ok ? o.h : KBUF_OOB, ahead * 16, KBUF_NT);
    u.s = __builtin_amdgcn_raw_buffer_load_b128(r.s, ok ? o.s : KBUF_OOB, ahead * 4, KBUF_NT);
    u.d = __builtin_amdgcn_raw_buffer_load_b16(r.d, ok ? o.d : KBUF_OOB, ahead / 2, KBUF_NT);
  }
}

__device__ __forceinline__ int dot16(const u32x4& w, const u32x4& x) {
  int acc = __builtin_amdgcn_sdot4((int)w.x, (int)x.x, 0, false);
  acc = __builtin_amdgcn_sdot4((int)w.y, (int)x.y, acc, false);
  acc = __builtin_amdgcn_sdot4((int)w.z, (int)x.z, acc, false);
  acc = __builtin_amdgcn_sdot4((int)w.w, (int)x.w, acc, false);
  return acc;
}
__device__ __forceinline__ int half16(uint32_t pair, int hi) { return (int)(int16_t)(hi ? (pair >> 16) : (pair & 0xffffu)); }

__device__ __forceinline__ void silu_mul8(float (&v)[8], const float* u, bool accurate) {
  const f32x4 a = reinterpret_cast<const f32x4*>(u)[0], b = reinterpret_cast<const f32x4*>(u)[1];
  const float uu[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
  for (int e = 0; e < 8; e++) v[e] = v[e] * (1.0f / (1.0f + (accurate ? expf(-v[e]) : exp_poly(-v[e])))) * uu[e];
}

// Workgroup = NW waves; a wave is cut into 64 / G groups of G lanes; a group owns R consecutive weight rows and its lanes
// stride over the row's units.  x is quantized to Q8_K once per workgroup into LDS: codes [MT][K], scales [MT][nsb], sums
// of 16 as int16 [MT][nsb][16].
// U = units a lane keeps in flight per row: a ring, a unit's registers take the one U further on as soon as it is multiplied.  (A second set
// of registers for a whole next trip, copied over, took 220 registers for Q6_K with two units of two rows, 152 now; 2 x 9728 x 2560 at two rows, with the
// offsets below and 24-bit products of sums and scales: Q4_K 11.2 -> 10.5 us, Q6_K 14.9 -> 13.9.)
// ONE: the row's units fit one trip (units <= G U): nothing to refill.
// AHEAD: a second set for the whole next trip, requested before this one is multiplied: its requests leave together, where the ring's leave one by one behind
// the products (two trips of four units each, one row per group: the second trip comes 0.6 to 1.4 us later).
template <int WT, int XT, int MT, int G, int R, int U, int LB = 256, bool ONE = false, bool AHEAD = false>
__global__ __launch_bounds__(LB) void kq_gemv_kernel(KGemvArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int nsb = a.nsb;
  const int K = nsb * QK_K;
  u32x4* s_q = reinterpret_cast<u32x4*>(smem);                         // [MT][K / 16]
  uint32_t* s_bs = reinterpret_cast<uint32_t*>(smem + (size_t)MT * K);  // [MT][nsb][8] pairs of int16 (sums of 16)
  float* s_d = reinterpret_cast<float*>(s_bs + (size_t)MT * nsb * 8);   // [MT][nsb]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int GROUPS = 64 / G;
  const int grp = lane / G, c0 = lane % G;
  const int nthreads = blockDim.x;  // 64 .. LB
  int pidx = 0;  // uniform: which matrix this workgroup works on
#pragma unroll
  for (int p = 1; p < KQ_MAX_PARTS; p++)
    if (p < a.nparts && (int)blockIdx.x >= a.wg_start[p]) pidx = p;
  const KGemvPart& pt = a.part[pidx];
  const int64_t row0 = ((int64_t)(blockIdx.x - a.wg_start[pidx]) * (nthreads >> 6) + wave) * (GROUPS * R) + (int64_t)grp * R;
  constexpr int UPS = WT == MLLM_HIP_Q4_K ? 8 : 4;  // units per super-block
  const int units = nsb * UPS;

  // MoE slot (uniform): expert offset of the weight planes, activation row, output row.  A slot whose expert id is outside
  // [0, E) computes with expert 0 and its row is never read (the combine pass skips it).
  size_t eoff = 0;
  int64_t xrow = 0, yrow = 0;
  if (MT == 1 && a.slot_ids) {
    const int slot = blockIdx.y;
    const int e = a.slot_ids[slot];
    eoff = (size_t)((e >= 0 && e < a.slot_E) ? e : 0) * a.estride;
    xrow = slot / a.slot_div;
    yrow = slot;
  }
  const char* xp = reinterpret_cast<const char*>(a.x) + xrow * K * (XT == MLLM_HIP_BF16 ? 2 : 4);
  const float* x2p = (XT == MLLM_HIP_F32 && MT == 1 && a.x2) ? a.x2 + xrow * K : nullptr;  // uniform
  KRsrc rs;
  {
    const uint32_t sbt = (uint32_t)pt.N * (uint32_t)nsb;
    auto at = [&](const void* base) { return const_cast<char*>(reinterpret_cast<const char*>(base) + eoff); };
    rs.a = __builtin_amdgcn_make_buffer_rsrc(at(pt.w.a), 0, sbt * 128u, 0x00020000);
    rs.h = __builtin_amdgcn_make_buffer_rsrc(at(WT == MLLM_HIP_Q6_K ? pt.w.h : pt.w.a), 0, sbt * 64u, 0x00020000);
    rs.s = __builtin_amdgcn_make_buffer_rsrc(at(pt.w.s), 0, sbt * 16u, 0x00020000);
    rs.d = __builtin_amdgcn_make_buffer_rsrc(at(pt.w.d), 0, sbt * (WT == MLLM_HIP_Q4_K ? 4u : 2u), 0x00020000);
  }
  // Memory requests return in order: the activations a thread will quantize (its first two items) are requested first,
  // then the first trip of weights, so that the quantization runs while the weights are still on their way.
  const int nitems = MT * (K >> 3);
  const int valid = a.M * (K >> 3);
  constexpr int XL = XT == KQ_IMAGE ? MLLM_HIP_F32 : XT;
  // (two rows: four items, or rows of 2560 elements leave half an item per thread to the loop further down, where it comes
  // back behind the weights)
  constexpr int NPRE = MT == 2 ? 4 : 2;
  u32x4 raw[NPRE][XL == MLLM_HIP_F32 ? 2 : 1];
  u32x4 raw2[2][2];
  if (XT != KQ_IMAGE) {
#pragma unroll
    for (int k = 0; k < NPRE; k++) {
      const int it = min(tid + k * nthreads, valid - 1);
      if (XL == MLLM_HIP_F32) {
        const u32x4* p = reinterpret_cast<const u32x4*>(reinterpret_cast<const float*>(xp) + (int64_t)it * 8);
        raw[k][0] = p[0];
        raw[k][XL == MLLM_HIP_F32 ? 1 : 0] = p[1];
      } else {
        raw[k][0] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(xp) + (int64_t)it * 8);
      }
    }
    if (XT == MLLM_HIP_F32 && MT == 1 && x2p) {  // the second factor with the first (ahead of the weights: requests return in order)
#pragma unroll
      for (int k = 0; k < 2; k++) {
        const u32x4* p = reinterpret_cast<const u32x4*>(x2p + (int64_t)min(tid + k * nthreads, valid - 1) * 8);
        raw2[k][0] = p[0];
        raw2[k][1] = p[1];
      }
    }
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }
  KOff off[R];
  bool row_ok[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    off[r] = unit_offsets<WT>((uint32_t)((row0 + r) * nsb), c0);
    row_ok[r] = row0 + r < pt.N;
  }
  KUnit<WT> cur[U][R];
#pragma unroll
  for (int uu = 0; uu < U; uu++)
#pragma unroll
    for (int r = 0; r < R; r++) load_unit<WT>(cur[uu][r], rs, off[r], uu * G, row_ok[r] && uu * G + c0 < units);

  __asm__ volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  // ---- activations -> Q8_K in LDS (rows m >= M are zero) ----
  if (XT == KQ_IMAGE) {  // codes | sums | scales, written by quantize_q8k_kernel in exactly this layout
    const int n16 = MT * (K >> 4), n4 = MT * nsb * 9;
    for (int c = tid; c < n16; c += nthreads) s_q[c] = reinterpret_cast<const u32x4*>(a.x)[c];
    const uint32_t* tail = reinterpret_cast<const uint32_t*>(a.x) + (size_t)n16 * 4;
    for (int c = tid; c < n4; c += nthreads) s_bs[c] = tail[c];
  }
  auto quantize_to_lds = [&](int it, const float (&v)[8]) {
    const Q8KItem q = quantize_q8k_item(v, lane);
    reinterpret_cast<u32x2*>(s_q)[it] = u32x2{q.q0, q.q1};
    const int s16 = q.sum8 + __builtin_amdgcn_update_dpp(0, q.sum8, 0xB1, 0xf, 0xf, true);
    const int s16b = __builtin_amdgcn_update_dpp(0, s16, 0x4E, 0xf, 0xf, true);  // the other pair of the quad
    if ((it & 3) == 0) s_bs[it >> 2] = ((uint32_t)s16 & 0xffffu) | ((uint32_t)s16b << 16);
    if ((it & 31) == 0) s_d[it >> 5] = q.d;
  };
  if (XT != KQ_IMAGE) {
#pragma unroll
    for (int k = 0; k < NPRE; k++) {  // whole half-waves: nitems is a multiple of 32
      const int it = tid + k * nthreads;
      if (it < nitems) {
        float v[8];
        if (XL == MLLM_HIP_F32) {
          const u32x4 p = raw[k][0], q = raw[k][XL == MLLM_HIP_F32 ? 1 : 0];
          v[0] = __uint_as_float(p.x); v[1] = __uint_as_float(p.y); v[2] = __uint_as_float(p.z); v[3] = __uint_as_float(p.w);
          v[4] = __uint_as_float(q.x); v[5] = __uint_as_float(q.y); v[6] = __uint_as_float(q.z); v[7] = __uint_as_float(q.w);
        } else {
          const uint32_t w[4] = {raw[k][0].x, raw[k][0].y, raw[k][0].z, raw[k][0].w};
#pragma unroll
          for (int j = 0; j < 4; j++) {
            v[2 * j + 0] = __uint_as_float(w[j] << 16);
            v[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
          }
        }
        if (it >= valid) {
#pragma unroll
          for (int e = 0; e < 8; e++) v[e] = 0.f;
        }
        if (XT == MLLM_HIP_F32 && MT == 1 && x2p) silu_mul8(v, reinterpret_cast<const float*>(&raw2[k < 2 ? k : 0][0]), a.silu_accurate);
        quantize_to_lds(it, v);
      }
    }
    for (int it = tid + NPRE * nthreads; it < nitems; it += nthreads) {
      float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (it < valid) load8<XL>(xp, (int64_t)it * 8, v);
      if (XT == MLLM_HIP_F32 && MT == 1 && x2p) silu_mul8(v, x2p + (int64_t)min(it, valid - 1) * 8, a.silu_accurate);
      quantize_to_lds(it, v);
    }
  }
  __syncthreads();

  float acc[R][MT];
#pragma unroll
  for (int r = 0; r < R; r++)
#pragma unroll
    for (int m = 0; m < MT; m++) acc[r][m] = 0.f;

  for (int u0 = 0; u0 < units; u0 += G * U) {
    const bool more = !ONE && u0 + G * U < units;  // uniform
    KUnit<WT> nxt[AHEAD ? U : 1][R];
    if (AHEAD && more) {
#pragma unroll
      for (int uu = 0; uu < U; uu++)
#pragma unroll
        for (int r = 0; r < R; r++)
          load_unit<WT>(nxt[AHEAD ? uu : 0][r], rs, off[r], u0 + G * U + uu * G, row_ok[r] && u0 + G * U + uu * G + c0 < units);
    }
#pragma unroll
    for (int uu = 0; uu < U; uu++) {
    const KUnit<WT>(&cu)[R] = cur[uu];
    const int unit = u0 + uu * G + c0;
    if (unit < units) {
      if (WT == MLLM_HIP_Q4_K) {
        const int sb = unit >> 3, c = unit & 7, jp = c >> 1, hh = c & 1;
        int sc_lo[R], sc_hi[R], mn_lo[R], mn_hi[R];
        float dw[R], dmw[R];
        u32x4 wlo[R], whi[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
          const uint32_t rec = cu[r].s.x;  // {sc[2jp], sc[2jp+1], m[2jp], m[2jp+1]}
          sc_lo[r] = (int)(rec & 0xffu);
          sc_hi[r] = (int)((rec >> 8) & 0xffu);
          mn_lo[r] = (int)((rec >> 16) & 0xffu);
          mn_hi[r] = (int)(rec >> 24);
          dw[r] = f16bits_to_f32((uint16_t)(cu[r].s.y & 0xffffu));
          dmw[r] = f16bits_to_f32((uint16_t)(cu[r].s.y >> 16));
          const uint32_t m4 = 0x0f0f0f0fu;
          wlo[r] = u32x4{cu[r].a.x & m4, cu[r].a.y & m4, cu[r].a.z & m4, cu[r].a.w & m4};
          whi[r] = u32x4{(cu[r].a.x >> 4) & m4, (cu[r].a.y >> 4) & m4, (cu[r].a.z >> 4) & m4, (cu[r].a.w >> 4) & m4};
        }
#pragma unroll
        for (int m = 0; m < MT; m++) {
          const int qb = m * (K >> 4) + sb * 16 + 4 * jp + hh;  // 16-byte chunk of the sub-block pair's low half
          const u32x4 xlo = s_q[qb], xhi = s_q[qb + 2];
          const float yd = s_d[m * nsb + sb];
          const u32x2 bp = reinterpret_cast<const u32x2*>(s_bs)[(m * nsb + sb) * 4 + jp];  // sums 4jp..4jp+3
          const int bs_lo = half16(bp.x, hh), bs_hi = half16(bp.y, hh);
#pragma unroll
          for (int r = 0; r < R; r++) {
            // (24-bit factors: one instruction instead of four times one)
            const int isum = __mul24(sc_lo[r], dot16(wlo[r], xlo)) + __mul24(sc_hi[r], dot16(whi[r], xhi));
            const int msum = __mul24(mn_lo[r], bs_lo) + __mul24(mn_hi[r], bs_hi);
            acc[r][m] = fmaf(yd * dw[r], (float)isum, acc[r][m]);
            acc[r][m] = fmaf(-yd * dmw[r], (float)msum, acc[r][m]);
          }
        }
      } else {
        const int sb = unit >> 2, n = (unit >> 1) & 1, t = unit & 1;
        u32x4 wv[R][4];
        int sc[R][4];
        float dw[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
          dw[r] = f16bits_to_f32(cu[r].d);
          const uint32_t sw[4] = {cu[r].s.x, cu[r].s.y, cu[r].s.z, cu[r].s.w};
#pragma unroll
          for (int g = 0; g < 4; g++) {
            const u32x4& src = (g & 1) ? cu[r].b : cu[r].a;
            const int sh = (g >= 2) ? 4 : 0;
            const uint32_t m4 = 0x0f0f0f0fu, m2 = 0x03030303u;
            wv[r][g] = u32x4{((src.x >> sh) & m4) | (((cu[r].h.x >> (2 * g)) & m2) << 4), ((src.y >> sh) & m4) | (((cu[r].h.y >> (2 * g)) & m2) << 4),
                             ((src.z >> sh) & m4) | (((cu[r].h.z >> (2 * g)) & m2) << 4), ((src.w >> sh) & m4) | (((cu[r].h.w >> (2 * g)) & m2) << 4)};
            const int si = 8 * n + 2 * g + t;  // scale of these 16 weights
            sc[r][g] = (int)(int8_t)((sw[si >> 2] >> (8 * (si & 3))) & 0xffu);
          }
        }
#pragma unroll
        for (int m = 0; m < MT; m++) {
          const float yd = s_d[m * nsb + sb];
          const u32x4 bq = reinterpret_cast<const u32x4*>(s_bs)[(m * nsb + sb) * 2 + n];  // sums 8n..8n+7
          const uint32_t bw[4] = {bq.x, bq.y, bq.z, bq.w};
          int tot[R];
#pragma unroll
          for (int r = 0; r < R; r++) tot[r] = 0;
#pragma unroll
          for (int g = 0; g < 4; g++) {
            const u32x4 xq = s_q[m * (K >> 4) + sb * 16 + 8 * n + 2 * g + t];
            const int bs = half16(bw[g], t);
#pragma unroll
            for (int r = 0; r < R; r++) tot[r] += __mul24(sc[r][g], dot16(wv[r][g], xq) - 32 * bs);
          }
#pragma unroll
          for (int r = 0; r < R; r++) acc[r][m] = fmaf(yd * dw[r], (float)tot[r], acc[r][m]);
        }
      }
    }
    if (!AHEAD && more) {  // the next trip's unit into the registers of this one
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < R; r++) load_unit<WT>(cur[uu][r], rs, off[r], u0 + G * U + uu * G, row_ok[r] && u0 + G * U + uu * G + c0 < units);
      __builtin_amdgcn_sched_barrier(0);
    }
    }
    if (AHEAD && more) {
#pragma unroll
      for (int uu = 0; uu < U; uu++)
#pragma unroll
        for (int r = 0; r < R; r++) cur[uu][r] = nxt[AHEAD ? uu : 0][r];
    }
  }

#pragma unroll
  for (int r = 0; r < R; r++)
#pragma unroll
    for (int m = 0; m < MT; m++) {
      const float v = group_sum<G>(acc[r][m]);
      const int64_t row = row0 + r;
      if (c0 == 0 && row < pt.N && m < a.M) pt.y[(yrow + m) * pt.N + row] = pt.bias ? v + pt.bias[row] : v;
    }
}

static int g_kq_G = 0, g_kq_NW = 0, g_kq_U = 0;  // tuning overrides (0 = heuristic)

// R1: one weight row per lane group and up to 16 waves per workgroup (few rows of many units: o_proj, down_proj).  The
// quantization of x is the long part of such a workgroup, so it is shared by as many rows as still fill the CUs.
template <int WT, int XT, int MT, int G, int U, bool R1 = false, bool ONE = false, bool AHEAD = false>
static int launch_kq_u(const KGemvArgs& a_in, int NW, hipStream_t st) {
  constexpr int R = R1 ? 1 : (WT == MLLM_HIP_Q4_K && MT >= 4) ? 4 : 2;  // wider row tiles reuse every LDS read for more weight rows
  constexpr int LB = R1 ? 1024 : 256;
  if (NW < 1 || NW * 64 > LB) return MLLM_HIP_E_BADARG;  // the kernel is compiled for at most LB threads
  const int rows_per_wg = NW * (64 / G) * R;
  const int K = a_in.nsb * QK_K;
  const size_t lds = (size_t)MT * K + (size_t)MT * a_in.nsb * 4 + (size_t)MT * a_in.nsb * 32;
  if (lds > 160 * 1024) return MLLM_HIP_E_SHAPE;
  KGemvArgs a = a_in;
  unsigned grid = 0;
  for (int p = 0; p < a.nparts; p++) {
    a.wg_start[p] = (int)grid;
    grid += (unsigned)((a.part[p].N + rows_per_wg - 1) / rows_per_wg);
  }
  a.wg_start[a.nparts] = (int)grid;
  if (ONE && a_in.nsb * (WT == MLLM_HIP_Q4_K ? 8 : 4) > G * U) return MLLM_HIP_E_BADARG;
  auto kern = kq_gemv_kernel<WT, XT, MT, G, R, U, LB, ONE, AHEAD>;
  if (lds > 64 * 1024)
    HIP_RET(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  const unsigned slots = (MT == 1 && a.slot_ids) ? (unsigned)a.slot_div_slots : 1u;
  hipLaunchKernelGGL(kern, dim3(grid, slots), dim3(NW * 64), lds, st, a);
  return (int)hipGetLastError();
}
template <int WT, int XT, int MT, int G>
static int launch_kq_g(const KGemvArgs& a, int NW, int U, bool r1, hipStream_t st) {
  // Q4_K, one or two rows, 32 lanes per weight row: a row of up to 96 (128 in the large workgroups) units is requested whole
  // before the quantization of x, three (four) units per lane, instead of one trip ahead of the dot loop -- time stamps put
  // a round trip to memory into every further trip (2560-element rows: 2.0 to 2.9 us of loop for three trips)
  if constexpr (WT == MLLM_HIP_Q4_K && MT <= 2 && G == 32) {
    const int units = a.nsb * 8;
    if (!g_kq_U) {  // (a tuning override of the units in flight keeps the trips)
      if (r1 && units <= 4 * G) return launch_kq_u<WT, XT, MT, G, 4, true, true>(a, NW, st);
      // (one row only: with two, no gain.  117 registers = four waves per SIMD, so the 1216 workgroups of gate + up come in
      // two rounds; asking the compiler for five waves, 96 registers, measured slower: gate + up 8.7 -> 9.1 us, q+k+v 5.35 -> 5.65)
      if constexpr (MT == 1)
        if (!r1 && units > 2 * G && units <= 3 * G) return launch_kq_u<WT, XT, MT, G, 3, false, true>(a, NW, st);
    }
  }
  // MoE slots: the row's units at once where two per lane hold them (Q4_K rows of up to 1024 elements, Q6_K of up to 2048), Q4_K four at a time up to 2048.  us of a
  // layer of 128 experts of 2048 x 768, top-8, two at a time with a second set of registers for the next trip / this: Q4_K / Q6_K one token 15.1 / 14.3, four
  // 26.4 / 25.4, eight 40.8 / 39.8 (three at a time 44.4), Q6_K eight 53.5 / 47.2.  Longer rows of Q4_K keep the second set: over 900 layers of 2304 to 7168 elements,
  // of the time before there was a ring, mean (most): four at a time by the ring 1.00 (1.09), the second set 0.97 (1.04); one token of 2560 x 3072, eight
  // experts 31.2 / 34.0 / 30.9 us
  if constexpr (MT == 1 && G == 16) {
    const int units = a.nsb * (WT == MLLM_HIP_Q4_K ? 8 : 4);
    if (a.slot_ids && U == 2 && !g_kq_U) {
      if (units <= G) return launch_kq_u<WT, XT, MT, G, 1, false, true>(a, NW, st);
      if (units <= 2 * G) return launch_kq_u<WT, XT, MT, G, 2, false, true>(a, NW, st);
      if constexpr (WT == MLLM_HIP_Q4_K) {
        if (units <= 4 * G) return launch_kq_u<WT, XT, MT, G, 4>(a, NW, st);
        return launch_kq_u<WT, XT, MT, G, 2, false, false, true>(a, NW, st);
      }
    }
  }
  // Q4_K in the large workgroups, beyond one trip: a second set of registers, but for rows that want one unit more of a lane at most, whose request leaves first
  // either way.  Without the offsets, 24-bit products and ring / ring / second set, us, one row: 1552 x 7936 6.9 / 8.1 / 6.8, 880 x 14 592 8.5 / 9.7 / 8.4; over 1500
  // shapes by how far the last trip is filled, of the first: up to a quarter 0.94 / 0.98, a half 0.99 / 0.98, three quarters 1.04 / 0.98, more 1.06 / 0.98
  if constexpr (WT == MLLM_HIP_Q4_K && MT <= 2 && G >= 32) {
    const int units = a.nsb * 8;
    if (r1 && !g_kq_U && (units <= 4 * G || units > 5 * G)) return launch_kq_u<WT, XT, MT, G, 4, true, false, true>(a, NW, st);
  }
  if (r1 && MT <= 2 && G >= 32) return launch_kq_u<WT, XT, MT, G, (MT <= 2 && G >= 32 && WT == MLLM_HIP_Q4_K) ? 4 : 1, (MT <= 2 && G >= 32)>(a, NW, st);
  if (WT == MLLM_HIP_Q4_K && U >= 4 && MT <= 2) return launch_kq_u<WT, XT, MT, G, (WT == MLLM_HIP_Q4_K && MT <= 2) ? 4 : 1>(a, NW, st);
  if (U >= 2 && MT <= 2) return launch_kq_u<WT, XT, MT, G, MT <= 2 ? 2 : 1>(a, NW, st);
  return launch_kq_u<WT, XT, MT, G, 1>(a, NW, st);
}
template <int WT, int XT, int MT>
static int launch_kq_m(const KGemvArgs& a, hipStream_t st) {
  // Measured on MI355X over the Qwen3-4B projection shapes (lanes per row x waves x units in flight swept): Q4_K rows want 32
  // lanes, Q6_K rows (units twice as heavy) the whole wave; four waves per workgroup share the activation quantization;
  // a grid of about one workgroup per CU keeps four units per lane in flight, a larger grid gets its bytes in flight
  // from occupancy and keeps one.
  const int units = a.nsb * (WT == MLLM_HIP_Q4_K ? 8 : 4);
  int best = WT == MLLM_HIP_Q4_K ? 32 : 64;
  while (best > 8 && best / 2 >= units) best >>= 1;
  int NW = 4;
  int64_t rows = 0;
  for (int p = 0; p < a.nparts; p++) rows += a.part[p].N;
  // (MoE slots multiply the grid: the shape rules below look at the whole launch)
  const int grid = (int)((rows + NW * (64 / best) * 2 - 1) / (NW * (64 / best) * 2)) * ((MT == 1 && a.slot_ids) ? a.slot_div_slots : 1);
  int U = 1;  // (four units in flight only in the large workgroups below: the 384-workgroup q/k/v launch measured 5.8 us with
              // one unit against 6.4 us with four)
  // few rows of many units (o_proj, down_proj): large workgroups of one row per lane group, the whole wave on a row when it is
  // long enough to keep 64 lanes busy for a trip
  // (only with at least 32 lanes per row: the narrower shapes have no such variant and keep their 256-thread workgroups)
  const bool r1 = MT <= 2 && grid < (WT == MLLM_HIP_Q4_K ? 256 : 512) && best >= 32 && !g_kq_NW && !g_kq_G;
  if (r1) {
    if (units >= 64 * 4) best = 64;
    NW = best == 64 ? 16 : 8;  // 16 rows per workgroup either way
    // ... or fewer, so that the grid is about one workgroup per CU (the Q4_0 kernel's finding: 2560 rows of 9728 elements
    // as 160 workgroups of 16 waves or as 256 of 10)
    const int rpw = 64 / best;  // rows per wave
    const int want = (int)((rows / rpw + 255) / 256);
    if (want >= 4 && want < NW) NW = want;
  }  // (many rows, K = 2560: eight waves per workgroup measured slower than four, 11.0 against 9.6 us for gate + up)
  // Q6_K rows whose units leave most of a 64-lane trip idle (K = 2560: 40 units): 16 lanes per row, two waves, where that still
  // makes a thousand workgroups (gate + up 15.8 -> 13.5 us; the smaller q/k/v launch stays faster with the whole wave)
  if (WT == MLLM_HIP_Q6_K && MT <= 2 && !r1 && !g_kq_G && !g_kq_NW && best == 64 && rows / 16 >= 1024 &&
      2 * ((units + 15) / 16 * 16 - units) < (units + 63) / 64 * 64 - units) {
    best = 16;
    NW = 2;
  }
  // MoE slots (thousands of small workgroups, each quantizing its token's x): 16 lanes per row make the workgroups twice as
  // tall, two units in flight (Qwen3-30B-A3B experts, eight tokens: 54.6 -> 45.1 us for the layer)
  if (MT == 1 && a.slot_ids && a.slot_div_slots > 1 && best >= 16 && !r1) {
    best = 16;
    U = 2;
  }
  if (g_kq_G) best = g_kq_G;
  if (g_kq_NW) NW = g_kq_NW;
  if (g_kq_U) U = g_kq_U;
  if (best == 64) return launch_kq_g<WT, XT, MT, 64>(a, NW, U, r1, st);
  if (best == 32) return launch_kq_g<WT, XT, MT, 32>(a, NW, U, r1, st);
  if (best == 16) return launch_kq_g<WT, XT, MT, 16>(a, NW, U, r1, st);
  return launch_kq_g<WT, XT, MT, 8>(a, NW, U, r1, st);
}
template <int WT, int XT>
static int launch_kq(const KGemvArgs& a, hipStream_t st) {
  if (a.M <= 1) return launch_kq_m<WT, XT, 1>(a, st);
  if (a.M <= 2) return launch_kq_m<WT, XT, 2>(a, st);
  if (a.M <= 4) return launch_kq_m<WT, XT, 4>(a, st);
  return launch_kq_m<WT, XT, 8>(a, st);
}


typedef int kv4i __attribute__((ext_vector_type(4)));
#include "kquant_rows.h"

static int g_kq_path = 0;  // 1: always the dot4 kernel (comparison runs and tests); 0 and 2: the matrix-core kernel wherever it fits


// ---- many rows: the matrix-core GEMM of the block formats (moe.hip, qg_kernel) with these weights -------------------------
// Same scheme as for Q4_0 / Q8_0: both operands as fp16 with their scales folded in, fp32 accumulation in
// v_mfma_f32_32x32x16_f16.  Activations: the Q8_K round trip xh = fp16(d * q) (codes and d bit-exact, the product rounded
// once).  Weights: Q4_K as 4-bit codes q with the sub-block's fp16(d * sc) and fp16(dmin * m), value = fma(q, ds, -dm)
// rounded once; Q6_K as int8 codes q - 32 with fp16(d * sc) per 16 elements.  Within about 5e-4 relative L2 of the
// reference's integer / fp32 arithmetic.
//
// code area, Q4_K: one output dword per thread, in the order of the Q4_0 gemm layout
template <int WT>
__global__ __launch_bounds__(256) void kqg_prepack_q_kernel(const uint8_t* __restrict__ blocks, uint32_t* __restrict__ P, int N, int K,
                                                            int64_t words) {
  const int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (w >= words) return;
  const int kbs = K / 64, nsb = K / QK_K;
  uint32_t v = 0;
  if (WT == MLLM_HIP_Q4_K) {
    const int d = (int)(w % 4), l = (int)((w / 4) % 64);
    const int64_t blk = w / 256;
    const int kb = (int)(blk % kbs), nb = (int)(blk / kbs);
    const int n = nb * 32 + (l & 31), k0 = kb * 64 + d * 16 + (l >> 5) * 8;
    if (n < N) {
      const uint8_t* qs = blocks + ((int64_t)n * nsb + k0 / QK_K) * 144 + 16;
      const int e = k0 % QK_K, c = e >> 6, p = e & 63;  // 64-element chunk, position: low nibbles first, then high
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const uint32_t byte = qs[32 * c + (p & 31) + i];
        const uint32_t q = p < 32 ? (byte & 15u) : (byte >> 4);
        v |= q << (4 * ((i >> 1) + 4 * (i & 1)));
      }
    }
  } else {
    const int x = (int)(w % 4), l = (int)((w / 4) % 64), pl = (int)((w / 256) % 2);
    const int64_t blk = w / 512;
    const int kb = (int)(blk % kbs), nb = (int)(blk / kbs);
    const int d = 2 * pl + x / 2;
    const int n = nb * 32 + (l & 31), k0 = kb * 64 + d * 16 + (l >> 5) * 8 + 4 * (x % 2);
    if (n < N) {
      const uint8_t* b = blocks + ((int64_t)n * nsb + k0 / QK_K) * 210;
      uint32_t c[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {  // dequantize_row_q6_K's element order: halves of 128, quarters of 32
        const int e = k0 % QK_K + i, h = e >> 7, r = e & 127, g = r >> 5, ll = r & 31;
        int lo = b[64 * h + ((g & 1) ? 32 : 0) + ll];
        lo = g >= 2 ? (lo >> 4) : (lo & 15);
        const int hi = (b[128 + 32 * h + ll] >> (2 * g)) & 3;
        c[i] = (uint32_t)((lo | (hi << 4)) - 32) & 0xffu;
      }
      v = c[0] | (c[2] << 8) | (c[1] << 16) | (c[3] << 24);
    }
  }
  P[w] = v;
}
// scale records: one thread per (32-row group, 64-element step, row)
template <int WT>
__global__ __launch_bounds__(256) void kqg_prepack_s_kernel(const uint8_t* __restrict__ blocks, u32x2* __restrict__ S, int N, int K, int x86,
                                                            int64_t count) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  const int kbs = K / 64, nsb = K / QK_K;
  const int row = (int)(i % 32), kb = (int)((i / 32) % kbs), nb = (int)(i / 32 / kbs);
  const int n = nb * 32 + row;
  u32x2 v{0u, 0u};
  if (n < N) {
    if (WT == MLLM_HIP_Q4_K) {
      const uint8_t* b = blocks + ((int64_t)n * nsb + kb / 4) * 144;
      const float d = f16bits_to_f32(field_bits(b, x86)), dmin = f16bits_to_f32(field_bits(b + 2, x86));
      const K4Scales k = k4_scales(bytes_u32(b + 4), bytes_u32(b + 8), bytes_u32(b + 12));
      const int j = 2 * (kb % 4);
      v.x = (uint32_t)f32_to_f16bits(d * (float)byte_of(k.sc0, k.sc1, j)) | ((uint32_t)f32_to_f16bits(d * (float)byte_of(k.sc0, k.sc1, j + 1)) << 16);
      v.y = (uint32_t)f32_to_f16bits(dmin * (float)byte_of(k.mn0, k.mn1, j)) | ((uint32_t)f32_to_f16bits(dmin * (float)byte_of(k.mn0, k.mn1, j + 1)) << 16);
    } else {
      const uint8_t* b = blocks + ((int64_t)n * nsb + kb / 4) * 210;
      const float d = f16bits_to_f32(field_bits(b + 208, x86));
      const int8_t* sc = reinterpret_cast<const int8_t*>(b + 192) + 4 * (kb % 4);
      v.x = (uint32_t)f32_to_f16bits(d * (float)sc[0]) | ((uint32_t)f32_to_f16bits(d * (float)sc[1]) << 16);
      v.y = (uint32_t)f32_to_f16bits(d * (float)sc[2]) | ((uint32_t)f32_to_f16bits(d * (float)sc[3]) << 16);
    }
  }
  S[i] = v;
}
// activations: Q8_K quantization and back to fp16 in one pass, xh[rows][K]
__global__ __launch_bounds__(256) void kq_act_f16_kernel(const void* __restrict__ x, int x_dtype, uint16_t* __restrict__ xh, int64_t nitems) {
  const int64_t it = (int64_t)blockIdx.x * 256 + threadIdx.x;  // nitems is a multiple of 32: whole half-waves
  if (it >= nitems) return;
  float v[8];
  if (x_dtype == MLLM_HIP_F32) load8<MLLM_HIP_F32>(x, it * 8, v);
  else load8<MLLM_HIP_BF16>(x, it * 8, v);
  const Q8KItem r = quantize_q8k_item(v, threadIdx.x & 63);
  uint32_t o[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const uint32_t word = j < 2 ? r.q0 : r.q1;
    const float a = r.d * (float)(int8_t)(word >> (16 * (j & 1)));
    const float b = r.d * (float)(int8_t)(word >> (16 * (j & 1) + 8));
    o[j] = (uint32_t)f32_to_f16bits(a) | ((uint32_t)f32_to_f16bits(b) << 16);
  }
  *reinterpret_cast<u32x4*>(xh + it * 8) = u32x4{o[0], o[1], o[2], o[3]};
}

}  // namespace mllmhip

using namespace mllmhip;

static int kq_check(int wtype, const void* packed, int64_t N, int64_t K) {
  if (wtype != MLLM_HIP_Q4_K && wtype != MLLM_HIP_Q6_K) return MLLM_HIP_E_BADARG;
  if (!packed || N <= 0 || K <= 0) return MLLM_HIP_E_BADARG;
  if (K % QK_K) return MLLM_HIP_E_SHAPE;
  if (N > INT32_MAX || N * (K / QK_K) * 128 >= ((int64_t)1 << 32)) return MLLM_HIP_E_SHAPE;  // 32-bit buffer offsets
  if (reinterpret_cast<uintptr_t>(packed) % 256) return MLLM_HIP_E_ALIGN;
  return 0;
}

MLLM_API int mllm_hip_kq_set_path(int path) {
  if (path != 0 && path != 1 && path != 2) return MLLM_HIP_E_BADARG;
  g_kq_path = path;
  return 0;
}
MLLM_API int mllm_hip_kq_set_slice_meeting(int mode, int waves_per_wg) {
  if (mode < -1 || mode > 1 || (waves_per_wg != 0 && (waves_per_wg < 1 || waves_per_wg > 8))) return MLLM_HIP_E_BADARG;
  return 0;
}

MLLM_API int mllm_hip_kq_set_rows_shape(int tiles, int waves) {
  const bool off = tiles == 0 && waves == 0;
  if (!off && (tiles < 1 || tiles > 8 || waves < 1 || tiles * waves > 16)) return MLLM_HIP_E_BADARG;
  g_kr_shape = KrShape{tiles, waves};
  return 0;
}

MLLM_API int mllm_hip_kq_rows_shape(int wtype, int64_t M, int64_t N, int64_t K, int row_tiles) {
  if ((wtype != MLLM_HIP_Q4_K && wtype != MLLM_HIP_Q6_K) || M < 3 || M > 8 || N <= 0 || N > 0x7fffffff || K <= 0 || K % QK_K || !kr_fits((int)(K / QK_K)) || row_tiles < 0 || row_tiles > 65535) return 0;
  const int id = 0;
  KGemvArgs a{};
  if (row_tiles) a.tile_expert = &id;
  a.M = (int)M;
  a.nsb = (int)(K / QK_K);
  a.nparts = 1;
  a.part[0].N = (int)N;
  const KrShape s = kr_shape(wtype == MLLM_HIP_Q4_K, a, row_tiles ? (unsigned)row_tiles : 1u);
  return s.tiles * 16 + s.waves;
}

MLLM_API int mllm_hip_kq_set_tuning(int lanes_per_row, int waves_per_wg, int units_in_flight) {
  auto ok = [](int v, std::initializer_list<int> allowed) {
    for (int x : allowed)
      if (v == x) return true;
    return false;
  };
  if (!ok(lanes_per_row, {0, 8, 16, 32, 64}) || !ok(waves_per_wg, {0, 1, 2, 4}) || !ok(units_in_flight, {0, 1, 2, 4})) return MLLM_HIP_E_BADARG;
  g_kq_G = lanes_per_row;
  g_kq_NW = waves_per_wg;
  g_kq_U = units_in_flight;
  return 0;
}

MLLM_API size_t mllm_hip_kq_packed_bytes(int wtype, int64_t N, int64_t K) {
  if ((wtype != MLLM_HIP_Q4_K && wtype != MLLM_HIP_Q6_K) || N <= 0 || K <= 0 || K % QK_K) return 0;
  return kq_packed_bytes(wtype, N, K);
}

MLLM_API int mllm_hip_kq_prepack(int wtype, const void* blocks, int weight_scale_mode, void* packed, int64_t N, int64_t K, void* stream) {
  int rc = kq_check(wtype, packed, N, K);
  if (rc) return rc;
  if (!blocks || (weight_scale_mode != MLLM_HIP_SCALE_IEEE && weight_scale_mode != MLLM_HIP_SCALE_X86_REF)) return MLLM_HIP_E_BADARG;
  const int64_t nsb = N * (K / QK_K);
  hipLaunchKernelGGL(kq_prepack_kernel, dim3((unsigned)((nsb * 8 + 255) / 256)), dim3(256), 0, (hipStream_t)stream, wtype,
                     (const uint8_t*)blocks, weight_scale_mode == MLLM_HIP_SCALE_X86_REF, kq_view(wtype, packed, N, K), nsb);
  return (int)hipGetLastError();
}

MLLM_API int mllm_hip_kq_dequantize(int wtype, const void* packed, float* w, int64_t N, int64_t K, void* stream) {
  int rc = kq_check(wtype, packed, N, K);
  if (rc) return rc;
  if (!w) return MLLM_HIP_E_BADARG;
  const int64_t nsb = N * (K / QK_K);
  hipLaunchKernelGGL(kq_dequantize_kernel, dim3((unsigned)nsb), dim3(256), 0, (hipStream_t)stream, wtype, kq_view(wtype, packed, N, K), w, nsb);
  return (int)hipGetLastError();
}

MLLM_API int mllm_hip_quantize_q8_K(const void* x, int x_dtype, int8_t* codes, float* d, int16_t* bsums, int64_t M, int64_t K, void* stream) {
  if (!x || !codes || !d || !bsums || M <= 0 || K <= 0 || (x_dtype != MLLM_HIP_F32 && x_dtype != MLLM_HIP_BF16)) return MLLM_HIP_E_BADARG;
  if (K % QK_K) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(codes) % 8) return MLLM_HIP_E_ALIGN;
  const int64_t nitems = M * K / 8;
  hipLaunchKernelGGL(quantize_q8k_kernel, dim3((unsigned)((nitems + 255) / 256)), dim3(256), 0, (hipStream_t)stream, x, x_dtype, codes, d,
                     bsums, nitems, nitems);
  return (int)hipGetLastError();
}

MLLM_API size_t mllm_hip_kq_workspace_bytes(int64_t M, int64_t K) {
  if (M <= 0 || K <= 0 || K % QK_K) return 0;
  return (size_t)8 * K + (size_t)8 * (K / QK_K) * 36;  // one group of eight rows: codes, sums of 16, scales
}

MLLM_API size_t mllm_hip_kq_workspace_bytes_n(int64_t M, int64_t K, int64_t N_total) {
  (void)N_total;  // (the K slices of a tile meet in LDS)
  return mllm_hip_kq_workspace_bytes(M, K);
}

MLLM_API int mllm_hip_linear_kq_multi(int wtype, int nparts, const mllm_hip_gemv_part* parts, const void* x, int x_dtype, int64_t M,
                                      int64_t K, void* workspace, void* stream) {
  return mllm_hip_linear_kq_multi_ws(wtype, nparts, parts, x, x_dtype, M, K, workspace, workspace ? mllm_hip_kq_workspace_bytes(M, K) : 0,
                                     stream);
}

MLLM_API int mllm_hip_linear_kq_multi_ws(int wtype, int nparts, const mllm_hip_gemv_part* parts, const void* x, int x_dtype, int64_t M,
                                         int64_t K, void* workspace, size_t workspace_bytes, void* stream) {
  if (nparts < 1 || nparts > KQ_MAX_PARTS || !parts) return MLLM_HIP_E_BADARG;
  if (!x || M <= 0 || (x_dtype != MLLM_HIP_F32 && x_dtype != MLLM_HIP_BF16)) return MLLM_HIP_E_BADARG;
  if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(workspace) % 16) return MLLM_HIP_E_ALIGN;
  for (int p = 0; p < nparts; p++) {
    int rc = kq_check(wtype, parts[p].packed, parts[p].N, K);
    if (rc) return rc;
    if (!parts[p].y) return MLLM_HIP_E_BADARG;
  }
  const size_t xrow = (size_t)K * (x_dtype == MLLM_HIP_F32 ? 4 : 2);
  const int nsb = (int)(K / QK_K);
  hipStream_t st = (hipStream_t)stream;
  int rc = 0;
  if (workspace && workspace_bytes < mllm_hip_kq_workspace_bytes(M, K)) return MLLM_HIP_E_BADARG;
  for (int64_t m0 = 0; m0 < M; m0 += 8) {  // more than eight rows: groups of eight (each streams the weights again)
    const int rows = (int)(M - m0 < 8 ? M - m0 : 8);
    const void* xg = reinterpret_cast<const char*>(x) + m0 * xrow;
    KGemvArgs a{};
    for (int p = 0; p < nparts; p++)
      a.part[p] = KGemvPart{kq_view(wtype, parts[p].packed, parts[p].N, K), parts[p].bias, parts[p].y + m0 * parts[p].N, (int)parts[p].N};
    a.nparts = nparts;
    a.x = xg;
    a.M = rows;
    a.nsb = nsb;
    // From three rows on the matrix cores, while the rows' codes fit the LDS.  The rule looks at the number of rows and the row
    // length only: a projection gives the same bits alone and as a part of a launch.
    if (rows >= 3 && g_kq_path != 1 && kr_fits(nsb)) {
      if (workspace && kr_image(wtype, a)) {
        hipLaunchKernelGGL(kr_image_kernel, dim3((unsigned)((nsb * 32 + 255) / 256), (unsigned)rows), dim3(256), 0, st, xg, x_dtype,
                           reinterpret_cast<unsigned char*>(workspace), nsb, rows);
        a.x = workspace;
        rc = launch_kq_rows_any<KQ_IMAGE>(wtype, a, st);
      } else {
        rc = x_dtype == MLLM_HIP_F32 ? launch_kq_rows_any<MLLM_HIP_F32>(wtype, a, st) : launch_kq_rows_any<MLLM_HIP_BF16>(wtype, a, st);
      }
    } else if (workspace && rows >= 3) {
      // several rows: quantize once for all workgroups; the GEMV then copies the image instead of quantizing
      const int MT = rows <= 4 ? 4 : 8;
      int8_t* img = reinterpret_cast<int8_t*>(workspace);
      const int64_t nitems = (int64_t)MT * K / 8;
      hipLaunchKernelGGL(quantize_q8k_kernel, dim3((unsigned)((nitems + 255) / 256)), dim3(256), 0, st, xg, x_dtype, img,
                         reinterpret_cast<float*>(img + (size_t)MT * K + (size_t)MT * nsb * 32),
                         reinterpret_cast<int16_t*>(img + (size_t)MT * K), nitems, (int64_t)rows * K / 8);
      a.x = img;
      rc = wtype == MLLM_HIP_Q4_K ? launch_kq<MLLM_HIP_Q4_K, KQ_IMAGE>(a, st) : launch_kq<MLLM_HIP_Q6_K, KQ_IMAGE>(a, st);
    } else if (wtype == MLLM_HIP_Q4_K) {
      rc = x_dtype == MLLM_HIP_F32 ? launch_kq<MLLM_HIP_Q4_K, MLLM_HIP_F32>(a, st) : launch_kq<MLLM_HIP_Q4_K, MLLM_HIP_BF16>(a, st);
    } else {
      rc = x_dtype == MLLM_HIP_F32 ? launch_kq<MLLM_HIP_Q6_K, MLLM_HIP_F32>(a, st) : launch_kq<MLLM_HIP_Q6_K, MLLM_HIP_BF16>(a, st);
    }
    if (rc) return rc;
  }
  return 0;
}

MLLM_API int mllm_hip_linear_kq(int wtype, const void* packed, const void* x, int x_dtype, const float* bias, float* y, int64_t M,
                                int64_t N, int64_t K, void* workspace, void* stream) {
  if (!y) return MLLM_HIP_E_BADARG;
  mllm_hip_gemv_part part{packed, bias, y, N};
  return mllm_hip_linear_kq_multi(wtype, 1, &part, x, x_dtype, M, K, workspace, stream);
}

// ---- MoE slots: one GEMV row per (token, expert) pair ---------------------------------------------------------------------------
// nparts sibling matrices per expert (gate and up, or down alone), packed0[p] = expert 0's matrix of part p, the experts'
// matrices mllm_hip_kq_packed_bytes(wtype, N, K) apart; slot s multiplies activation row s / slot_div by the matrices of
// expert ids[s] and writes row s of ys[p] ([slots][N]).  x2 (fp32, same rows as x): the activation is silu(x) * x2.
// form: KQ_MOE_PAIRS one by one; KQ_MOE_GROUPS the workgroups find the pairs that share an expert, same bits (kq_moe_groups_fit);
// KQ_MOE_TILES they find them too, up to eight, with the sums of the sorted tiles.
namespace mllmhip {
int exp_mode_accurate();  // layer_ops.hip: the setting of mllm_hip_set_exp_mode
int kq_moe_gemv(int wtype, int nparts, const void* const* packed0, float* const* ys, int64_t N, int64_t K, const void* x, int x_dtype,
                const float* x2, const int32_t* ids, int E, int slots, int slot_div, int form, hipStream_t st) {
  if (x2 && x_dtype != MLLM_HIP_F32) return MLLM_HIP_E_BADARG;
  if (nparts < 1 || nparts > KQ_MAX_PARTS || slots < 1 || slots > 65535) return MLLM_HIP_E_SHAPE;
  KGemvArgs a{};
  for (int p = 0; p < nparts; p++) a.part[p] = KGemvPart{kq_view(wtype, packed0[p], N, K), nullptr, ys[p], (int)N};
  a.nparts = nparts;
  a.x = x;
  a.M = 1;
  a.nsb = (int)(K / QK_K);
  a.slot_ids = ids;
  a.x2 = x2;
  a.silu_accurate = exp_mode_accurate();
  a.slot_E = E;
  a.slot_div = slot_div;
  a.slot_div_slots = slots;
  a.estride = kq_packed_bytes(wtype, N, K);
  if (form == KQ_MOE_GROUPS) {
    if (wtype != MLLM_HIP_Q6_K) return MLLM_HIP_E_BADARG;
    a.M = 4;
    return x_dtype == MLLM_HIP_F32 ? launch_kq_rows<MLLM_HIP_Q6_K, MLLM_HIP_F32, 1, KR_PAIRS>(a, st, (unsigned)slots)
                                   : launch_kq_rows<MLLM_HIP_Q6_K, MLLM_HIP_BF16, 1, KR_PAIRS>(a, st, (unsigned)slots);
  }
  if (form == KQ_MOE_TILES) {
    a.M = 8;
    return x_dtype == MLLM_HIP_F32 ? launch_kq_rows_any<MLLM_HIP_F32, KR_TILES>(wtype, a, st, (unsigned)slots)
                                   : launch_kq_rows_any<MLLM_HIP_BF16, KR_TILES>(wtype, a, st, (unsigned)slots);
  }
  if (wtype == MLLM_HIP_Q4_K)
    return x_dtype == MLLM_HIP_F32 ? launch_kq<MLLM_HIP_Q4_K, MLLM_HIP_F32>(a, st) : launch_kq<MLLM_HIP_Q4_K, MLLM_HIP_BF16>(a, st);
  return x_dtype == MLLM_HIP_F32 ? launch_kq<MLLM_HIP_Q6_K, MLLM_HIP_F32>(a, st) : launch_kq<MLLM_HIP_Q6_K, MLLM_HIP_BF16>(a, st);
}

// Groups of pairs pay for Q6_K rows of three to six super-blocks (the dot4 kernel's sixteen lanes then hold a row in one or two
// trips and wait for each) from about 32 k rows of weights in the launch on.  128 to 512 experts, us of the layer, pairs one by one / in
// groups: down 2048 x 768 at 16 / 24 / 64 pairs 0.91 / 0.83 / 0.76 of the time, 4096 x 1024 0.90 / 0.90 / 0.78, 1024 x 1024 1.05 /
// 0.98 / 0.82; two super-blocks 1.01 to 1.15, eight 0.96 to 1.14 of it; gate + up of 2 x 512 x 1024 1.07 / 0.99 / 0.81, of 2 x 768 x 2048
// 1.01 to 1.15.  (Q4_K: 0.95 to 1.2 over the same sizes.)  The search walks the slots, hence at most 512.
bool kq_moe_groups_fit(int wtype, int64_t rows, int64_t K, int slots) {
  const int64_t nsb = K / QK_K;
  return wtype == MLLM_HIP_Q6_K && nsb >= 3 && nsb <= 6 && slots >= 16 && slots <= 512 && rows * slots >= 32768 && !g_kq_G && !g_kq_NW && !g_kq_U;
}

// The Q8_K image of `rows` activation rows (codes [rows][K], sums of 16 [rows][K/16] int16, scales
// [rows][K/256]) at `image`: what the matrix-core kernels copy into LDS.
size_t kq_image_bytes(int64_t rows, int64_t K) { return (size_t)rows * K + (size_t)rows * (K / 16) * 2 + (size_t)rows * (K / QK_K) * 4; }
int kq_quantize_image(const void* x, int x_dtype, void* image, int64_t rows, int64_t K, hipStream_t st) {
  const int64_t nitems = rows * K / 8;
  int8_t* codes = reinterpret_cast<int8_t*>(image);
  int16_t* bsums = reinterpret_cast<int16_t*>(codes + rows * K);
  float* d = reinterpret_cast<float*>(codes + rows * K + rows * (K / 16) * 2);
  hipLaunchKernelGGL(quantize_q8k_kernel, dim3((unsigned)((nitems + 255) / 256)), dim3(256), 0, st, x, x_dtype, codes, d, bsums, nitems,
                     nitems);
  return (int)hipGetLastError();
}
bool kq_moe_tiles_fit(int64_t K) {
  return kr_fits((int)(K / QK_K));
}
// MoE row tiles on the matrix-core kernels: tile t (blockIdx.y) = up to eight expert-sorted positions of expert tile_expert[t];
// its rows read image rows row_ids[pos] / row_div (null: pos) and write rows out_ids[pos] (null: pos) of ys[p].
int kq_moe_tiles_gemv(int wtype, int nparts, const void* const* packed0, float* const* ys, int64_t N, int64_t K, const void* image,
                      int64_t img_rows, const int* tile_expert, const int* tile_row0, const int* tile_rows, const int* ntiles,
                      unsigned max_tiles, const int* row_ids, int row_div, const int* out_ids, hipStream_t st) {
  if (nparts < 1 || nparts > KQ_MAX_PARTS || max_tiles < 1 || max_tiles > 65535) return MLLM_HIP_E_SHAPE;
  KGemvArgs a{};
  for (int p = 0; p < nparts; p++) a.part[p] = KGemvPart{kq_view(wtype, packed0[p], N, K), nullptr, ys[p], (int)N};
  a.nparts = nparts;
  a.x = image;
  a.M = 8;
  a.nsb = (int)(K / QK_K);
  a.estride = kq_packed_bytes(wtype, N, K);
  a.tile_expert = tile_expert; a.tile_row0 = tile_row0; a.tile_rows = tile_rows; a.ntiles = ntiles;
  a.row_ids = row_ids; a.out_ids = out_ids; a.row_div = row_div > 0 ? row_div : 1;
  a.img_rows = (int)img_rows;
  return launch_kq_rows_any<KQ_IMAGE, KR_TILES>(wtype, a, st, max_tiles);
}
}  // namespace mllmhip

// ---- many rows on the matrix cores ------------------------------------------------------------------------------------------
static bool kq_type(int wtype) { return wtype == MLLM_HIP_Q4_K || wtype == MLLM_HIP_Q6_K; }
MLLM_API size_t mllm_hip_kq_gemm_packed_bytes(int wtype, int64_t N, int64_t K) {
  if (!kq_type(wtype) || N <= 0 || K <= 0 || K % QK_K) return 0;
  return (size_t)qg_bytes(wtype, N, K);
}
MLLM_API int mllm_hip_kq_gemm_prepack(int wtype, const void* blocks, int weight_scale_mode, void* gemm_packed, int64_t N, int64_t K,
                                      void* stream) {
  if (!kq_type(wtype) || !blocks || !gemm_packed || N <= 0 || K <= 0) return MLLM_HIP_E_BADARG;
  if (weight_scale_mode != MLLM_HIP_SCALE_IEEE && weight_scale_mode != MLLM_HIP_SCALE_X86_REF) return MLLM_HIP_E_BADARG;
  if (K % QK_K || N > INT32_MAX || K > INT32_MAX || qg_bytes(wtype, N, K) >= ((int64_t)1 << 32)) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(gemm_packed) % 16) return MLLM_HIP_E_ALIGN;
  hipStream_t st = (hipStream_t)stream;
  const int64_t words = qg_qbytes(wtype, N, K) / 4, count = qg_np(N) * (K / 64);
  const uint8_t* b = reinterpret_cast<const uint8_t*>(blocks);
  uint32_t* q = reinterpret_cast<uint32_t*>(gemm_packed);
  u32x2* sc = reinterpret_cast<u32x2*>(reinterpret_cast<char*>(gemm_packed) + qg_qbytes(wtype, N, K));
  const int x86 = weight_scale_mode == MLLM_HIP_SCALE_X86_REF;
  const dim3 gq((unsigned)((words + 255) / 256)), gs((unsigned)((count + 255) / 256));
  if (wtype == MLLM_HIP_Q4_K) {
    hipLaunchKernelGGL(kqg_prepack_q_kernel<MLLM_HIP_Q4_K>, gq, dim3(256), 0, st, b, q, (int)N, (int)K, words);
    hipLaunchKernelGGL(kqg_prepack_s_kernel<MLLM_HIP_Q4_K>, gs, dim3(256), 0, st, b, sc, (int)N, (int)K, x86, count);
  } else {
    hipLaunchKernelGGL(kqg_prepack_q_kernel<MLLM_HIP_Q6_K>, gq, dim3(256), 0, st, b, q, (int)N, (int)K, words);
    hipLaunchKernelGGL(kqg_prepack_s_kernel<MLLM_HIP_Q6_K>, gs, dim3(256), 0, st, b, sc, (int)N, (int)K, x86, count);
  }
  return (int)hipGetLastError();
}
MLLM_API size_t mllm_hip_linear_kq_gemm_workspace_bytes(int64_t M, int64_t K) {
  if (M <= 0 || K <= 0 || K % QK_K) return 0;
  return align_up((size_t)M * K * 2, 256);
}
MLLM_API int mllm_hip_linear_kq_gemm(int wtype, const void* gemm_packed, const void* x, int x_dtype, const float* bias, float* y, int64_t M,
                                     int64_t N, int64_t K, void* workspace, void* stream) {
  if (!kq_type(wtype) || !gemm_packed || !x || !y || !workspace || M <= 0 || N <= 0 || K <= 0) return MLLM_HIP_E_BADARG;
  if (x_dtype != MLLM_HIP_F32 && x_dtype != MLLM_HIP_BF16) return MLLM_HIP_E_BADARG;
  if (K % QK_K || M * K * 2 >= ((int64_t)1 << 32) || N > INT32_MAX || qg_bytes(wtype, N, K) >= ((int64_t)1 << 32)) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(workspace) % 16 || reinterpret_cast<uintptr_t>(gemm_packed) % 16 ||
      reinterpret_cast<uintptr_t>(y) % 16)
    return MLLM_HIP_E_ALIGN;
  hipStream_t st = (hipStream_t)stream;
  uint16_t* xh = reinterpret_cast<uint16_t*>(workspace);
  const int64_t nitems = M * K / 8;
  hipLaunchKernelGGL(kq_act_f16_kernel, dim3((unsigned)((nitems + 255) / 256)), dim3(256), 0, st, x, x_dtype, xh, nitems);
  return qg_linear_run(wtype, gemm_packed, xh, bias, y, M, N, K, nullptr, st);
}

// the same with room for the partial results of K ranges that run as separate workgroups
MLLM_API size_t mllm_hip_linear_kq_gemm_short_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0 || K % QK_K) return 0;
  return mllm_hip_linear_kq_gemm_workspace_bytes(M, K) + 256 + qg_partial_bytes(MLLM_HIP_Q4_K, M, N, K);
}
MLLM_API int mllm_hip_linear_kq_gemm_short(int wtype, const void* gemm_packed, const void* x, int x_dtype, const float* bias, float* y,
                                           int64_t M, int64_t N, int64_t K, void* workspace, void* stream) {
  if (!kq_type(wtype) || !gemm_packed || !x || !y || !workspace || M <= 0 || N <= 0 || K <= 0) return MLLM_HIP_E_BADARG;
  if (x_dtype != MLLM_HIP_F32 && x_dtype != MLLM_HIP_BF16) return MLLM_HIP_E_BADARG;
  if (K % QK_K || M * K * 2 >= ((int64_t)1 << 32) || N > INT32_MAX || qg_bytes(wtype, N, K) >= ((int64_t)1 << 32)) return MLLM_HIP_E_SHAPE;
  if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(workspace) % 256 || reinterpret_cast<uintptr_t>(gemm_packed) % 16 ||
      reinterpret_cast<uintptr_t>(y) % 16)
    return MLLM_HIP_E_ALIGN;
  hipStream_t st = (hipStream_t)stream;
  uint16_t* xh = reinterpret_cast<uint16_t*>(workspace);
  const int64_t nitems = M * K / 8;
  hipLaunchKernelGGL(kq_act_f16_kernel, dim3((unsigned)((nitems + 255) / 256)), dim3(256), 0, st, x, x_dtype, xh, nitems);
  char* base = reinterpret_cast<char*>(workspace);
  void* partial = qg_partial_bytes(MLLM_HIP_Q4_K, M, N, K) ? base + mllm_hip_linear_kq_gemm_workspace_bytes(M, K) : nullptr;
  return qg_linear_run(wtype, gemm_packed, xh, bias, y, M, N, K, partial, st);
}

MLLM_API int mllm_hip_kq_moe_pair_tiles(int nparts, int64_t N, int64_t K, int slots) {
  if (nparts < 1 || nparts > KQ_MAX_PARTS || slots < 1 || slots > 65535 || N <= 0 || N > 0x7fffffff || K <= 0 || !kq_moe_groups_fit(MLLM_HIP_Q6_K, nparts * N, K, slots)) return 0;
  const int id = 0;
  KGemvArgs a{};
  a.slot_ids = &id;
  a.M = 4;
  a.nsb = (int)(K / QK_K);
  a.nparts = nparts;
  for (int p = 0; p < nparts; p++) a.part[p].N = (int)N;
  return kr_pair_tiles(a, (unsigned)slots, kr_shape(false, a, (unsigned)slots, true, true).tiles);
}

MLLM_API int mllm_hip_kq_rows_image(int wtype, int64_t M, int64_t N, int64_t K) {
  if (!mllm_hip_kq_rows_shape(wtype, M, N, K, 0)) return 0;
  KGemvArgs a{};
  a.M = (int)M;
  a.nsb = (int)(K / QK_K);
  a.nparts = 1;
  a.part[0].N = (int)N;
  return kr_image(wtype, a);
}

// Q4_K / Q6_K weights x three to eight activation rows (or the rows of an MoE expert) on the matrix cores.  Included by
// kquant.hip behind KGemvArgs, the Q8_K quantizer and load8.
//
// A tile is sixteen weight rows (channels) x up to eight activation rows x all of K.  The weights are the SECOND operand of
// v_mfma_i32_16x16x64_i8, so that a lane owns ONE channel and the scales it needs are bytes of its own channel's record:
// no table of scales in LDS, one byte extract per scale.  The instruction sums over K = 64 and every 32 (Q4_K) or 16 (Q6_K) elements
// have a scale of their own, so the ACTIVATION operand keeps them apart: its sixteen rows are (sub-block pair member q, row m)
// resp. (unit q of four, four of the rows), with zeros outside the lane group(s) that hold sub-block q.
//   Q4_K  lane (channel c = l % 16, g = l / 16) holds record 4 j + g of its channel's super-block: the low-nibble instruction
//         sees sub-block 4 j in groups 0, 1 and 4 j + 2 in groups 2, 3 (high nibbles one further); its four results are rows
//         4 (g % 2) .. + 3 of the sub-block of q = g / 2.  I += sc * D; the minimum term accumulates in the matrix pipe: the same
//         activation operand against the byte m in all sixteen places (one v_perm) sums m * code.
//   Q6_K  group g's record is exactly one unit of 16 elements: D = sum over unit g of (code - 32) * x for four rows (the
//         -32 is a first instruction against a constant operand), I += sc * D.  Five to eight rows: a second instruction.
// Per super-block acc = fma(fp32(d * dx), float(I), acc) (and the minimum term): the reference's vec_dot (integer sums per
// super-block, then d * dx) with the sums of a super-block split over two (Q4_K) or four lanes.
//
// What bounds it (time stamps written by the kernel, gate + up of 9728 x 2560 at five rows, us after the start): the codes back
// 2.2, all waves past the barrier 3.8, the last wave's loop done 7.9, end 8.4 -- the weights, 28 MB, flow from 1.5 on; with a quantizer of
// twice the instructions, whose third item per thread came back behind the weights: 0.4 more.  Kept
// short by spreading K over the waves of a workgroup (one tile's waves meet in LDS, not in memory), by requests for activations ahead
// of every wave's weights, and by loading whole lines: with weights loaded in the operand's own order (sixteen rows per instruction) the
// L1's tags were the bottleneck and the last wave passed the barrier at 10.7.  Five rows, us with the quantization (before: K slices as
// workgroups that met in memory, or scale tables in LDS): q+k+v 9.9 -> 7.4, o 9.6 -> 7.6, gate+up 14.7 -> 10.7, down (Q6_K, 2560 x
// 9728) 17.3 -> 12.6; 20 MB of the last take 4 us at the copy rate of the card.
// K is cut into slices of KR_SPS super-blocks whatever the launch shape; a slice is summed in one chain and the slices are added in
// order, by one wave or over several: the bits depend on the weight type and K alone.
//
// MoE layers quantize twice more behind these sums, and the router of the next layer picks by them: a last bit that moves one code of h
// or x over a rounding edge is 1e-4 to 1e-3 of a token's output.  A form that serves an MoE layer therefore keeps the fp32 order of the
// form it stands in for (the integer sums are the same in all):
//   KR_TILES  eight rows of an expert.  Every sub-block (Q6_K: unit of 16) is scaled on its own, acc = fma((d * sc) * dx, D, acc), Q4_K's
//             minimum behind it, acc = fma(-((dmin * m) * dx), sum of the codes, acc); a lane group's chain runs over the slice
//             (kr_moe_slice), the lane groups meet pairwise (0 + 1) + (2 + 3), then the slices in order.
//   KR_PAIRS  Q6_K pairs in groups of four, in the order of the dot4 kernel on sixteen lanes per weight row: units of 64 elements
//             (scaled int sum, then acc = fma(dx * d, sum, acc)) in sixteen chains, unit modulo 16, added as a binary tree.
//             Bound by the weights of the experts in use; a Q4_K / Q6_K layer of 128 experts of 2048 x 768, top-8, two / four / eight tokens:
//             22.5 / 35.1 / 59.7 -> 19.9 / 27.7 / 43.7 us against one dot4 row per pair.
#pragma once

constexpr int KR_SPS = 2;                      // super-blocks per slice
constexpr int KR_SB_LDS = 16 * 8 * 16;         // codes of a super-block, at most: [unit of 16][rows] 16 bytes
constexpr size_t KR_LDS_MAX = 160 * 1024;
// the image in memory: codes [super-block][unit][rows][16], then scales [super-block][8]
static int kr_slices(int nsb) { return (nsb + KR_SPS - 1) / KR_SPS; }
// super-blocks of a slice in MoE layers: up to five while there are at most eight slices
__host__ __device__ __forceinline__ int kr_moe_slice(int nsb) {
  int s = 1;
  while (s < 8 && nsb > 5 * s) s *= 2;
  return (nsb + s - 1) / s;
}
// super-blocks of weights a wave has in flight: two, one where the registers of a second set would spill (more in flight, four, measured
// slower: every wave then queues its requests for weights ahead of other waves' activations)
constexpr int kr_depth(bool q4, int th) { return q4 || th == 1 ? 2 : 1; }
constexpr int kr_stage_bytes(bool q4) { return q4 ? 2048 + 1024 + 256 : 2048 + 1024 + 1024 + 128; }  // per wave: codes [, bit pairs], scales, d
static size_t kr_lds_bytes(bool q4, int nsb, int tiles, int waves_per_tile) {
  return (size_t)(nsb + 1) * KR_SB_LDS + (size_t)nsb * 32 + 64 + (size_t)tiles * waves_per_tile * kr_stage_bytes(q4) +
         (waves_per_tile > 1 ? (size_t)tiles * kr_slices(nsb) * 512 : 0);
}
static bool kr_fits(int nsb) { return kr_lds_bytes(false, nsb, 1, 4) <= KR_LDS_MAX; }

// the activation rows -> the image
__global__ __launch_bounds__(256) void kr_image_kernel(const void* __restrict__ x, int x_dtype, unsigned char* __restrict__ image, int nsb, int rows) {
  const int it = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;  // item (eight elements) of row m; whole half-waves
  if (it >= nsb * 32) return;
  float v[8];
  const int64_t e = ((int64_t)m * nsb * 32 + it) * 8;
  if (x_dtype == MLLM_HIP_F32) load8<MLLM_HIP_F32>(x, e, v);
  else load8<MLLM_HIP_BF16>(x, e, v);
  const Q8KItem r = quantize_q8k_item(v, threadIdx.x & 63);
  reinterpret_cast<u32x2*>(image)[((it >> 1) * rows + m) * 2 + (it & 1)] = u32x2{r.q0, r.q1};
  if ((it & 31) == 0) reinterpret_cast<float*>(image + (size_t)nsb * 256 * rows)[(it >> 5) * 8 + m] = r.d;
}

// sum over lane bit 5 (permlane32) / bit 4 (permlane16) of two values at once: lanes with the bit clear keep a's, the others b's
__device__ __forceinline__ float kr_fold32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ int kr_fold32i(int a, int b) {
  const auto r = __builtin_amdgcn_permlane32_swap((uint32_t)a, (uint32_t)b, false, false);
  return (int)(r[0] + r[1]);
}
__device__ __forceinline__ float kr_fold16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// a trip's weights on their way: whole 128-byte lines (lanes 8 r .. 8 r + 7 hold row r's super-block; one row per lane, the operand's own
// order, would touch 64 lines per instruction and was bound by the L1's tag rate)
template <int WT, int DEPTH>
struct KrWeights {
  u32x4 a[DEPTH][2], s;                             // rows l / 8 and 8 + l / 8, piece l % 8; scale record of (row l / 4, super-block l % 4)
  u32x4 h[WT == MLLM_HIP_Q4_K ? 1 : DEPTH];         // Q6_K: row l / 4, piece l % 4
  uint32_t d;                                         // as s
};

// blockDim = tiles per workgroup * P waves (wave = tile * P + p); XT: fp32 / bf16 activations, quantized by the workgroup, or the
// image (KQ_IMAGE: of these eight rows; MoE row tiles: codes [rows][K], sums, scales of all rows, gathered).
// TH = groups of four rows (Q4_K: always two).  ORDER: the sums, see above; pairs: one wave per tile.
enum { KR_LINEAR, KR_TILES, KR_PAIRS };
template <int WT, int XT, int TH, int ORDER>
__global__ __launch_bounds__(1024) void kq_rows_kernel(KGemvArgs a, int P_or_T) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr bool Q4 = WT == MLLM_HIP_Q4_K;
  constexpr bool TILES = ORDER == KR_TILES, PAIRS = ORDER == KR_PAIRS;
  const int P = PAIRS ? 1 : P_or_T, T = PAIRS ? P_or_T : 1;  // waves per tile; tiles per wave
  static_assert(!PAIRS || (!Q4 && TH == 1), "pairs in groups: Q6_K, groups of four");
  constexpr int DEPTH = kr_depth(Q4, PAIRS ? 2 : TH);  // (pairs: sixteen accumulators)
  const int nsb = a.nsb, K = nsb * QK_K;
  const int tid = threadIdx.x, lane = tid & 63, nthreads = blockDim.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles_wg = (nthreads >> 6) / P, tl = wave / P, p = wave - tl * P;
  int pidx = 0;
#pragma unroll
  for (int i = 1; i < KQ_MAX_PARTS; i++)
    if (i < a.nparts && (int)blockIdx.x >= a.wg_start[i]) pidx = i;
  const KGemvPart& pt = a.part[pidx];
  const int N = pt.N;

  u32x4* xc = reinterpret_cast<u32x4*>(smem);                                 // [unit][R rows] 16 codes
  unsigned char* zblk = smem + (size_t)nsb * KR_SB_LDS;                       // one super-block of zeros
  float* dxs = reinterpret_cast<float*>(zblk + KR_SB_LDS);                    // [super-block][8]
  int* s_rows = reinterpret_cast<int*>(dxs + (size_t)nsb * 8);                // [8] MoE pairs: the tile's slots; [8]: how many
  // a wave's own stage, where lines become operands: pieces of 16 bytes, conflict-free both ways (one wave's LDS operations execute in order)
  unsigned char* stage = reinterpret_cast<unsigned char*>(s_rows) + 64 + (size_t)wave * kr_stage_bytes(Q4);
  f32x2* part = reinterpret_cast<f32x2*>(reinterpret_cast<unsigned char*>(s_rows) + 64 + (size_t)(nthreads >> 6) * kr_stage_bytes(Q4));  // [tile][slice][lane]

  constexpr int GROUP = Q4 ? 8 : 4 * TH;
  // ---- which rows -----------------------------------------------------------------------------------------------------------
  KTile mt = kq_tile(a);
  if (!mt.active) return;  // uniform, ahead of every barrier
  if (a.slot_ids) {
    // MoE pairs: the pairs of one expert are found by the workgroups themselves.  Slot blockIdx.y works if it is the first of
    // its expert's slots, or the one after a group of GROUP, ...; it takes the next GROUP.  No routing launch, weights read once per expert.
    const int mine = blockIdx.y, e = a.slot_ids[mine];
    if (e < 0 || e >= a.slot_E) return;
    int before = 0, total = 0;
    for (int c = 0; c < a.slot_div_slots; c += 64) {
      const int s = c + lane;
      const bool same = s < a.slot_div_slots && a.slot_ids[min(s, a.slot_div_slots - 1)] == e;
      const unsigned long long b = __ballot(same);
      const int ahead = total + __popcll(b & ((1ull << lane) - 1ull));  // this expert's slots ahead of s
      if (mine >= c) before += __popcll(mine - c >= 64 ? b : b & ((1ull << (mine - c)) - 1ull));
      // (mine's own rank is known once its chunk has been seen; slots behind it only count from then on)
      if (same && s >= mine && ahead - before < GROUP) {
        if (wave == 0) s_rows[ahead - before] = s;
      }
      total += __popcll(b);
    }
    if (before % GROUP) return;  // uniform
    mt.rows = min(GROUP, total - before);
    mt.eoff = (size_t)e * a.estride;
    __syncthreads();
  }
  const int R = mt.rows;
  auto in_row = [&](int m) -> int64_t { return a.slot_ids ? (int64_t)(s_rows[m] / a.slot_div) : (int64_t)kq_tile_in_row(a, mt, m); };

  // ---- 1. activations requested, then the wave's first super-blocks of weights (memory requests return in order) ------------
  const int c = lane & 15, g = lane >> 4;
  int row0 = (((int)blockIdx.x - a.wg_start[pidx]) * tiles_wg + tl) * T * 16;
  const uint32_t sbt = (uint32_t)N * (uint32_t)nsb;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<u32x4*>(kq_at(pt.w.a, mt.eoff)), 0, sbt * 128u, 0x00020000);
  const __amdgpu_buffer_rsrc_t rh = __builtin_amdgcn_make_buffer_rsrc(const_cast<u32x4*>(kq_at(Q4 ? pt.w.a : pt.w.h, mt.eoff)), 0, sbt * 64u, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsc = __builtin_amdgcn_make_buffer_rsrc(const_cast<u32x4*>(kq_at(pt.w.s, mt.eoff)), 0, sbt * 16u, 0x00020000);
  const __amdgpu_buffer_rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(kq_at(pt.w.d, mt.eoff)), 0, sbt * (Q4 ? 4u : 2u), 0x00020000);
  const int sps = PAIRS ? nsb : TILES ? kr_moe_slice(nsb) : KR_SPS;
  const int S = (nsb + sps - 1) / sps;
  const int sl0 = p * S / P, sl1 = (p + 1) * S / P;                // this wave's slices
  const int sb0 = sl0 * sps, sb1 = min(nsb, sl1 * sps);            // and super-blocks
  uint32_t rb8, rb4;
  bool ok8[2], ok4;
  auto rows_of = [&](int r) {  // the rows that weights are requested of
    rb8 = (uint32_t)(r + (lane >> 3)) * (uint32_t)nsb, rb4 = (uint32_t)(r + (lane >> 2)) * (uint32_t)nsb;
    ok8[0] = r + (lane >> 3) < N, ok8[1] = r + 8 + (lane >> 3) < N, ok4 = r + (lane >> 2) < N;
  };
  rows_of(row0);
  KrWeights<WT, DEPTH> w;
  auto load_sb = [&](int i, int sb) {
#pragma unroll
    for (int t = 0; t < 2; t++)
      w.a[i][t] = __builtin_amdgcn_raw_buffer_load_b128(
          ra, ok8[t] && sb < sb1 ? (rb8 + (uint32_t)(8 * t * nsb + sb)) * 128u + (uint32_t)(lane & 7) * 16u : KBUF_OOB, 0, KBUF_NT);
    if constexpr (!Q4)
      w.h[i] = __builtin_amdgcn_raw_buffer_load_b128(rh, ok4 && sb < sb1 ? (rb4 + (uint32_t)sb) * 64u + (uint32_t)(lane & 3) * 16u : KBUF_OOB, 0, KBUF_NT);
  };
  auto load_scales = [&](int sb) {
    const int si = sb + (lane & 3);
    const bool ok = ok4 && (lane & 3) < DEPTH && si < sb1;
    w.s = __builtin_amdgcn_raw_buffer_load_b128(rsc, ok ? (rb4 + (uint32_t)si) * 16u : KBUF_OOB, 0, KBUF_NT);
    if constexpr (Q4) w.d = __builtin_amdgcn_raw_buffer_load_b32(rd, ok ? (rb4 + (uint32_t)si) * 4u : KBUF_OOB, 0, KBUF_NT);
    else w.d = __builtin_amdgcn_raw_buffer_load_b16(rd, ok ? (rb4 + (uint32_t)si) * 2u : KBUF_OOB, 0, KBUF_NT);
  };
  // (behind a barrier, so that the requests for activations of ALL waves are ahead of any weights: the L1 answers in order)
  auto load_first = [&]() {
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    load_scales(sb0);
#pragma unroll
    for (int i = 0; i < DEPTH; i++) load_sb(i, sb0 + i);
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  for (int i = tid; i < KR_SB_LDS / 16; i += nthreads) reinterpret_cast<u32x4*>(zblk)[i] = u32x4{0u, 0u, 0u, 0u};
  if (XT == KQ_IMAGE && !a.tile_expert) {
    const u32x4* src = reinterpret_cast<const u32x4*>(a.x);
    const int n16 = nsb * 16 * R;
    constexpr int U = 6;
    u32x4 v[U];
    float dv = 0.f;
    if (tid < nsb * 8) dv = reinterpret_cast<const float*>(src + n16)[tid];
#pragma unroll
    for (int u = 0; u < U; u++)
      if (tid + u * nthreads < n16) v[u] = src[tid + u * nthreads];
    load_first();
    if (tid < nsb * 8) dxs[tid] = dv;
#pragma unroll
    for (int u = 0; u < U; u++)
      if (tid + u * nthreads < n16) xc[tid + u * nthreads] = v[u];
    for (int i = tid + U * nthreads; i < n16; i += nthreads) xc[i] = src[i];
    for (int i = tid + nthreads; i < nsb * 8; i += nthreads) dxs[i] = reinterpret_cast<const float*>(src + n16)[i];
  } else if (XT == KQ_IMAGE) {  // rows gathered from codes [R][K], sums of 16 [R][K/16], scales [R][nsb]
    const size_t RI = (size_t)a.img_rows;
    const u32x4* codes = reinterpret_cast<const u32x4*>(a.x);
    const float* dd = reinterpret_cast<const float*>(reinterpret_cast<const char*>(a.x) + RI * K + RI * nsb * 32);
    const int m = tid & 7, p0 = tid >> 3, pstep = nthreads >> 3, nu = m < R ? nsb * 16 : 0;
    const size_t src = (size_t)kq_tile_in_row(a, mt, m) * (size_t)nsb;  // in super-blocks
    constexpr int U = 4;
    u32x4 v[U];
    float dv = 0.f;
    if (p0 < nsb) dv = dd[src + p0];
#pragma unroll
    for (int u = 0; u < U; u++)
      if (p0 + u * pstep < nu) v[u] = codes[src * 16 + p0 + u * pstep];
    load_first();
    if (p0 < nsb) dxs[p0 * 8 + m] = dv;
#pragma unroll
    for (int u = 0; u < U; u++)
      if (p0 + u * pstep < nu) xc[(p0 + u * pstep) * R + m] = v[u];
    for (int u = p0 + U * pstep; u < nu; u += pstep) xc[u * R + m] = codes[src * 16 + u];
    for (int sb = p0 + pstep; sb < nsb; sb += pstep) dxs[sb * 8 + m] = dd[src + sb];
  } else {
    // quantized here: items of eight elements, 32 consecutive ones = a super-block; rows past the tile's are left as they are
    // (a row's results depend on its own codes only, and theirs are dropped)
    constexpr int XL = XT == KQ_IMAGE ? MLLM_HIP_F32 : XT;
    const int ipr = nsb * 32, nitems = mt.rows * ipr;
    const float inv = 1.0f / (float)ipr;
    constexpr int U = 4;  // items a thread requests ahead of the weights: as many as there are in a plain Linear
    const bool prod = XT == MLLM_HIP_F32 && a.x2 != nullptr;  // uniform
    auto fetch = [&](int it, float (&v)[8], float (&f)[8]) {
      const int m = (int)(((float)it + 0.5f) * inv), i = it - m * ipr;  // it / ipr: far from rounding trouble
      const int64_t e = (in_row(m) * ipr + i) * 8;
      load8<XL>(a.x, e, v);
      if (prod) load8<MLLM_HIP_F32>(a.x2, e, f);
    };
    auto put = [&](int it, float (&v)[8], const float (&f)[8]) {
      const int m = (int)(((float)it + 0.5f) * inv), i = it - m * ipr;
      if (prod) silu_mul8(v, f, a.silu_accurate);
      const Q8KItem q = quantize_q8k_item(v, lane);
      reinterpret_cast<u32x2*>(xc)[((i >> 1) * R + m) * 2 + (i & 1)] = u32x2{q.q0, q.q1};
      if ((i & 31) == 0) dxs[(i >> 5) * 8 + m] = q.d;
    };
    float v[U][8] = {}, f[U][8] = {};
#pragma unroll
    for (int u = 0; u < U; u++)
      if (tid + u * nthreads < nitems) fetch(tid + u * nthreads, v[u], f[u]);
    load_first();
#pragma unroll
    for (int u = 0; u < U; u++)
      if (tid + u * nthreads < nitems) put(tid + u * nthreads, v[u], f[u]);  // whole half-waves
    for (int it = tid + U * nthreads; it < nitems; it += nthreads) {
      float v1[8], f1[8] = {};
      fetch(it, v1, f1);
      put(it, v1, f1);
    }
  }
  __syncthreads();

  // ---- 2. a super-block: sums on the matrix cores, scales as integers ---------------------------------------------------------
  const int i16 = lane & 15;                      // the activation operand's row
  const int q = Q4 ? i16 >> 3 : i16 >> 2;          // sub-block (unit) it belongs to
  const int im = Q4 ? i16 & 7 : i16 & 3;           // and its row (Q6_K: of the first four)
  // the lane groups that supply its codes; the others read zeros
  const bool act = Q4 ? (g >> 1) == q : g == q;
  const int u0 = Q4 ? 4 * q + (g & 1) : q, R16 = R * 16;
  const unsigned char* xb[Q4 ? 1 : TH];
  uint32_t xstep[Q4 ? 1 : TH];
#pragma unroll
  for (int h = 0; h < (Q4 ? 1 : TH); h++) {
    const bool on = act && im + 4 * h < R;
    xb[h] = on ? smem + u0 * R16 + (im + 4 * h) * 16 : zblk;
    xstep[h] = on ? (uint32_t)(16 * R16) : 0u;
  }
  const float* dxl = dxs + (Q4 ? 4 * (g & 1) : 0);
  constexpr int NA = PAIRS ? 16 : Q4 ? 4 : 4 * TH;  // accumulators (pairs: super-block modulo 4, half, row)
  float acc[NA], tot[2] = {0.f, 0.f};
#pragma unroll
  for (int r = 0; r < NA; r++) acc[r] = 0.f;
  const uint32_t bsel = (uint32_t)g * 8u;
  const kv4i zero = {0, 0, 0, 0}, m32 = {(int)0xe0e0e0e0u, (int)0xe0e0e0e0u, (int)0xe0e0e0e0u, (int)0xe0e0e0e0u},
             ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
  u32x4* st_a = reinterpret_cast<u32x4*>(stage);                   // [16 rows][8] piece ^ (row / 2 % 8)
  u32x4* st_s = st_a + 128;                                        // [16 rows][4] super-block ^ (row / 4)
  u32x4* st_h = st_s + 64;                                         // Q6_K: [16 rows][4] piece ^ (row / 4)
  uint32_t* st_d = reinterpret_cast<uint32_t*>(stage + 3072);      // Q4_K: [16 rows][4]
  uint16_t* st_d6 = reinterpret_cast<uint16_t*>(stage + 4096);     // Q6_K: [16 rows][4]
  const int wra = (lane >> 3) * 8 + ((lane & 7) ^ ((lane >> 4) & 7)), wrb = wra ^ 4;  // rows l / 8 and 8 + l / 8
  const int wr4 = (lane & ~3) + ((lane & 3) ^ (lane >> 4));                           // row l / 4: (row / 4) = l / 16
  auto put_scales = [&]() {
    st_s[wr4] = w.s;
    if constexpr (Q4) st_d[lane] = w.d;
    else st_d6[lane] = (uint16_t)w.d;
  };
  auto put_sb = [&](int i) {
    st_a[wra] = w.a[i][0];
    st_a[64 + wrb] = w.a[i][1];
    if constexpr (!Q4) st_h[wr4] = w.h[i];
  };
  struct {
    u32x4 a[2], h[2], s4;
    uint32_t s[2], d;
  } u;
  auto take_sb = [&](int i) {
#pragma unroll
    for (int j = 0; j < 2; j++) {
      u.a[j] = st_a[c * 8 + ((4 * j + g) ^ (c >> 1))];
      if constexpr (Q4) u.s[j] = reinterpret_cast<const uint32_t*>(st_s + c * 4 + (i ^ (c >> 2)))[2 * j + (g >> 1)];
      else u.h[j] = st_h[c * 4 + ((2 * j + (g & 1)) ^ (c >> 2))];
    }
    if constexpr (Q4) {
      u.d = st_d[c * 4 + i];
    } else {
      u.s4 = st_s[c * 4 + (i ^ (c >> 2))];
      u.d = st_d6[c * 4 + i];
    }
  };
  // (part: the super-block modulo 4, a constant; used by pairs only)
  auto compute = [&](int sb, int part) {
    if constexpr (Q4 && TILES) {
      const float d = f16bits_to_f32((uint16_t)(u.d & 0xffffu)), dmin = f16bits_to_f32((uint16_t)(u.d >> 16));
      const f32x4 dx = *reinterpret_cast<const f32x4*>(dxl + sb * 8);
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const unsigned char* x = xb[0] + (uint32_t)sb * xstep[0] + 8 * j * R16;
#pragma unroll
        for (int h = 0; h < 2; h++) {  // sub-blocks 4 j + 2 q (low nibbles) and the next one (high nibbles)
          const kv4i xv = *reinterpret_cast<const kv4i*>(x + 2 * h * R16);
          kv4i wv;
#pragma unroll
          for (int e = 0; e < 4; e++) wv[e] = (int)((u.a[j][e] >> (4 * h)) & 0x0f0f0f0fu);
          const kv4i D = __builtin_amdgcn_mfma_i32_16x16x64_i8(xv, wv, zero, 0, 0, 0);
          const kv4i X = __builtin_amdgcn_mfma_i32_16x16x64_i8(xv, ones, zero, 0, 0, 0);  // sums of the codes
          const float ds = d * (float)((u.s[j] >> (8 * h)) & 0xffu), dm = dmin * (float)((u.s[j] >> (16 + 8 * h)) & 0xffu);
#pragma unroll
          for (int r = 0; r < 4; r++) {
            acc[r] = fmaf(ds * dx[r], (float)D[r], acc[r]);
            acc[r] = fmaf(-(dm * dx[r]), (float)X[r], acc[r]);
          }
        }
      }
    } else if constexpr (Q4) {
      int I[4] = {0, 0, 0, 0};
      kv4i mn = zero;
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const unsigned char* x = xb[0] + (uint32_t)sb * xstep[0] + 8 * j * R16;
        const kv4i xl = *reinterpret_cast<const kv4i*>(x), xh = *reinterpret_cast<const kv4i*>(x + 2 * R16);
        kv4i wl, wh;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          wl[e] = (int)(u.a[j][e] & 0x0f0f0f0fu);
          wh[e] = (int)((u.a[j][e] >> 4) & 0x0f0f0f0fu);
        }
        const int ml = (int)__builtin_amdgcn_perm(0u, u.s[j], 0x02020202u), mh = (int)__builtin_amdgcn_perm(0u, u.s[j], 0x03030303u);
        const kv4i dl = __builtin_amdgcn_mfma_i32_16x16x64_i8(xl, wl, zero, 0, 0, 0);
        const kv4i dh = __builtin_amdgcn_mfma_i32_16x16x64_i8(xh, wh, zero, 0, 0, 0);
        mn = __builtin_amdgcn_mfma_i32_16x16x64_i8(xl, kv4i{ml, ml, ml, ml}, mn, 0, 0, 0);
        mn = __builtin_amdgcn_mfma_i32_16x16x64_i8(xh, kv4i{mh, mh, mh, mh}, mn, 0, 0, 0);
        const int sl = (int)(u.s[j] & 0xffu), sh = (int)((u.s[j] >> 8) & 0xffu);
#pragma unroll
        for (int r = 0; r < 4; r++) I[r] += __mul24(sl, dl[r]) + __mul24(sh, dh[r]);
      }
      const float d = f16bits_to_f32((uint16_t)(u.d & 0xffffu)), dmin = f16bits_to_f32((uint16_t)(u.d >> 16));
      const f32x4 dx = *reinterpret_cast<const f32x4*>(dxl + sb * 8);
#pragma unroll
      for (int r = 0; r < 4; r++) {
        acc[r] = fmaf(dx[r] * d, (float)I[r], acc[r]);
        acc[r] = fmaf(-(dx[r] * dmin), (float)mn[r], acc[r]);
      }
    } else {
      int I[4 * TH];
#pragma unroll
      for (int r = 0; r < 4 * TH; r++) I[r] = 0;
      const float d = f16bits_to_f32((uint16_t)u.d);
      f32x4 dx[TH];
#pragma unroll
      for (int h = 0; h < TH; h++) dx[h] = *reinterpret_cast<const f32x4*>(dxl + sb * 8 + 4 * h);
      const uint32_t shl = 2u * (uint32_t)(g >> 1);  // low-nibble units of this group take bit pair g / 2, high-nibble units g / 2 + 2
#pragma unroll
      for (int j = 0; j < 2; j++) {
        kv4i wl, wh;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const uint32_t hs = u.h[j][e] >> shl;
          wl[e] = (int)((u.a[j][e] & 0x0f0f0f0fu) | ((hs & 0x03030303u) << 4));
          wh[e] = (int)(((u.a[j][e] >> 4) & 0x0f0f0f0fu) | (hs & 0x30303030u));
        }
        const int sl = (int)(u.s4[2 * j] << (24 - bsel)) >> 24, sh = (int)(u.s4[2 * j + 1] << (24 - bsel)) >> 24;
        const float dsl = d * (float)sl, dsh = d * (float)sh;
        int U[4 * TH];  // pairs: this lane's share of a unit's sum
#pragma unroll
        for (int h = 0; h < TH; h++) {
          const unsigned char* x = xb[h] + (uint32_t)sb * xstep[h] + 8 * j * R16;
          const kv4i xl = *reinterpret_cast<const kv4i*>(x), xh = *reinterpret_cast<const kv4i*>(x + 4 * R16);
          kv4i dl = __builtin_amdgcn_mfma_i32_16x16x64_i8(xl, m32, zero, 0, 0, 0);
          kv4i dh = __builtin_amdgcn_mfma_i32_16x16x64_i8(xh, m32, zero, 0, 0, 0);
          dl = __builtin_amdgcn_mfma_i32_16x16x64_i8(xl, wl, dl, 0, 0, 0);
          dh = __builtin_amdgcn_mfma_i32_16x16x64_i8(xh, wh, dh, 0, 0, 0);
#pragma unroll
          for (int r = 0; r < 4; r++) {
            if constexpr (TILES) {
              acc[4 * h + r] = fmaf(dsl * dx[h][r], (float)dl[r], acc[4 * h + r]);
              acc[4 * h + r] = fmaf(dsh * dx[h][r], (float)dh[r], acc[4 * h + r]);
            } else if constexpr (PAIRS) {
              U[r] = __mul24(sl, dl[r]) + __mul24(sh, dh[r]);
            } else {
              I[4 * h + r] += __mul24(sl, dl[r]) + __mul24(sh, dh[r]);
            }
          }
        }
        if constexpr (PAIRS) {  // records g and g + 2 make one unit of 64: lane groups 0, 1 keep rows 0, 2, groups 2, 3 rows 1, 3
          const int s01 = kr_fold32i(U[0], U[1]), s23 = kr_fold32i(U[2], U[3]);
          acc[4 * part + 2 * j] = fmaf((g >> 1 ? dx[0][1] : dx[0][0]) * d, (float)s01, acc[4 * part + 2 * j]);
          acc[4 * part + 2 * j + 1] = fmaf((g >> 1 ? dx[0][3] : dx[0][2]) * d, (float)s23, acc[4 * part + 2 * j + 1]);
        }
      }
      if constexpr (ORDER == KR_LINEAR) {
#pragma unroll
        for (int h = 0; h < TH; h++)
#pragma unroll
          for (int r = 0; r < 4; r++) acc[4 * h + r] = fmaf(dx[h][r] * d, (float)I[4 * h + r], acc[4 * h + r]);
      }
    }
  };
  // the end of a slice: the lanes of a channel meet.  Afterwards lane (c, g) holds two rows of channel c:
  //   Q4_K 4 (g % 2) + g / 2 and that + 2;  Q6_K 2 (g % 2) + g / 2 and that + 4 (tiles: g and that + 4)
  //   pairs: the row 2 (g % 2) + g / 2
  int slice = sl0, left = sps;  // left: super-blocks up to the end of the slice
  auto flush = [&]() {
    f32x2 v;
    if constexpr (PAIRS) {
      float s[8];
#pragma unroll
      for (int i = 0; i < 8; i++) s[i] = kr_fold16(acc[2 * i], acc[2 * i + 1]);
      v = f32x2{((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7])), 0.f};
    } else if constexpr (Q4) {
      v = f32x2{kr_fold32(acc[0], acc[1]), kr_fold32(acc[2], acc[3])};
    } else if constexpr (TILES) {  // (units 0, 1 and 2, 3 first)
      v.x = kr_fold32(kr_fold16(acc[0], acc[1]), kr_fold16(acc[2], acc[3]));
      v.y = TH == 2 ? kr_fold32(kr_fold16(acc[NA - 4], acc[NA - 3]), kr_fold16(acc[NA - 2], acc[NA - 1])) : 0.f;
    } else {
      v.x = kr_fold16(kr_fold32(acc[0], acc[1]), kr_fold32(acc[2], acc[3]));
      v.y = TH == 2 ? kr_fold16(kr_fold32(acc[NA - 4], acc[NA - 3]), kr_fold32(acc[NA - 2], acc[NA - 1])) : 0.f;
    }
#pragma unroll
    for (int r = 0; r < NA; r++) acc[r] = 0.f;
    if (P > 1) {
      part[(tl * S + slice) * 64 + lane] = v;
    } else if (slice == 0) {
      tot[0] = v.x;
      tot[1] = v.y;
    } else {
      tot[0] += v.x;
      tot[1] += v.y;
    }
    slice++;
    left = sps;
  };
  const auto bias_of = [&](int n) { return pt.bias ? pt.bias[n] : 0.f; };
  auto write = [&]() {
    const int n = row0 + c;
    if (n >= N) return;
    const float bias = bias_of(n);
#pragma unroll
    for (int k = 0; k < (PAIRS ? 1 : 2); k++) {
      const int m = Q4 ? 4 * (g & 1) + (g >> 1) + 2 * k : (TILES ? g : 2 * (g & 1) + (g >> 1)) + 4 * k;
      if (m >= mt.rows) continue;
      const int64_t orow = a.slot_ids ? (int64_t)s_rows[m] : (int64_t)kq_tile_out_row(a, mt, m);
      pt.y[orow * N + n] = pt.bias ? tot[k] + bias : tot[k];
    }
  };
  if constexpr (PAIRS) {  // the wave's tiles one after the other; the next one's first super-block is requested with this one's last
    for (int t = 0; t < T; t++) {
#pragma unroll 1
      for (int s4 = 0; s4 < nsb; s4 += 4) {
#pragma unroll
        for (int i = 0; i < 4; i++) {  // (the super-block modulo 4 is a constant)
          const int sb = s4 + i;
          if (sb >= nsb) break;  // uniform
          const bool last = sb + 1 == nsb;
          int next = sb + 1;  // (past the wave's last one: fetches nothing)
          if (last && t + 1 < T) {
            rows_of(row0 + 16);
            next = 0;
          }
          put_scales();
          load_scales(next);
          put_sb(0);
          __builtin_amdgcn_wave_barrier();
          take_sb(0);
          __builtin_amdgcn_wave_barrier();
          load_sb(0, next);
          __builtin_amdgcn_sched_barrier(0);
          compute(sb, i);
          if (last) flush();
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      write();
      row0 += 16;
      slice = 0;
    }
    return;
  }
  for (int sb = sb0; sb < sb1; sb += DEPTH) {
    put_scales();
    load_scales(sb + DEPTH);  // (past the wave's last one: fetches nothing)
#pragma unroll
    for (int i = 0; i < DEPTH; i++) {
      if (sb + i < sb1) {  // uniform
        put_sb(i);
        __builtin_amdgcn_wave_barrier();
        take_sb(i);
        __builtin_amdgcn_wave_barrier();
      }
      load_sb(i, sb + DEPTH + i);
      __builtin_amdgcn_sched_barrier(0);
      if (sb + i < sb1) {
        compute(sb + i, i);
        if (--left == 0 || sb + i + 1 == nsb) flush();
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // ---- 3. slices in order, bias ----------------------------------------------------------------------------------------------
  if (P > 1) {
    __syncthreads();
    if (p != 0) return;
    const f32x2 v0 = part[tl * S * 64 + lane];
    tot[0] = v0.x;
    tot[1] = v0.y;
#pragma unroll 4
    for (int s = 1; s < S; s++) {
      const f32x2 v = part[(tl * S + s) * 64 + lane];
      tot[0] += v.x;
      tot[1] += v.y;
    }
  }
  write();
}

// Tiles per workgroup and waves per tile.  A plain Linear: about one workgroup per CU, up to sixteen waves in it, none with more
// slices than needed (2560 x 9728: one tile of ten waves 12.6 us, two tiles of eight 18; 2 x 9728 x 2560 in tiles x waves: 5 x 2
// 12.0, 8 x 1 12.6, 2 x 8 17.2).  MoE: thousands of workgroups, small ones that share a CU (48 us with 4 x 1 for eight tokens,
// 60 with 8 x 1, 65 with 2 x 2).  Tiles of rows of more than ten super-blocks (four slices or more) or with few tiles spread the slices over
// waves, or one wave's walk along K is what the layer waits for.  Experts, us of the layer, tiles x 1 / this: 8 x 512 x 3584, 5 and 28 tokens
// Q4_K / Q6_K 33.5 / 26.4, 36.6 / 28.2; 8 x 4096 x 768 Q4_K, 5 tokens 31.8 / 27.6; 32 x 4096 x 1536 Q4_K, 18 tokens 73.5 / 70.1 (2 x 4: 74.7),
// Q6_K 103.6 / 95.4 (4 x 2: 110.9); 4 x 2048 x 2048 Q6_K, 4 tokens 31.2 / 28.2.  Six to ten super-blocks and many tiles: 0.83 to 1.07 of the time.
struct KrShape {
  int tiles, waves;
};
static KrShape g_kr_shape{0, 0};  // mllm_hip_kq_set_rows_shape
static KrShape kr_shape(bool q4, const KGemvArgs& a, unsigned grid_y, bool quantizes = false, bool pairs = false) {
  int64_t tiles = 0;
  for (int i = 0; i < a.nparts; i++) tiles += (a.part[i].N + 15) / 16;
  const int S = kr_slices(a.nsb);
  const bool moe = a.slot_ids || a.tile_expert;
  int tw = (int)std::min<int64_t>(moe ? 4 : 8, (tiles * grid_y + 255) / 256);
  int P = moe ? 1 : std::min(S, tw >= 5 ? 10 / tw : 16 / tw);
  while (P > 1 && (S + P - 2) / (P - 1) == (S + P - 1) / P) P--;
  // One tile per workgroup and more than twelve slices: waves with two slices each, up to six rows and where x is quantized ahead (13 to
  // 16 waves with one slice each have nothing in flight beside it and start later; fewer waves also make the image pay from three rows
  // on).  13 to 16 slices, 128 to 4096 channels, us, a slice / two per wave: 3 x 2048 x 8192 Q4_K 10.1 / 8.8, Q6_K 10.8 / 9.5; 6 x 1024 x
  // 7168 8.84 / 8.67, 10.1 / 9.9; eight rows 8.96 / 9.26, 10.2 / 10.5; with twelve slices 8.36 / 8.46, 9.1 / 9.9.
  if (!quantizes && !moe && tw == 1 && P > 12 && P == S && a.M <= 6) P = (S + 1) / 2;
  // one tile per workgroup that quantizes x itself: waves without a slice share that, two items per thread of the four that it requests ahead (up to eight waves; 1024 x 1024
  // Q6_K at three / four / eight rows 5.8 / 6.3 / 8.9 -> 5.2 / 5.3 / 6.5 us, Q4_K at eight 8.3 -> 6.0; with more tiles the added waves cost
  // more than they take over, 6144 x 2048 Q6_K at eight rows 8.4 -> 9.5)
  if (quantizes && !moe && tw == 1) P = std::max(P, std::min(8, (a.M * a.nsb * 32 + 127) / 128));
  if (moe && !pairs) {
    const int slices = (a.nsb + kr_moe_slice(a.nsb) - 1) / kr_moe_slice(a.nsb);
    if (slices >= 4) {
      P = q4 && tw == 4 ? 2 : 4;
      tw = q4 && tw == 4 ? 4 : std::min(tw, 2);
    } else if (slices == 2 && tw < 4) {
      P = 2;
      tw = std::min(tw, 2);
    }
  }
  if (g_kr_shape.tiles && !moe) tw = g_kr_shape.tiles, P = g_kr_shape.waves;
  while (P > 1 && kr_lds_bytes(q4, a.nsb, 1, P) > KR_LDS_MAX) P--;
  while (tw > 1 && kr_lds_bytes(q4, a.nsb, tw, P) > KR_LDS_MAX) tw--;
  return KrShape{tw, P};
}
// Whether three to eight rows are quantized once, by a launch of its own (given a workspace): where every workgroup would have more than four items of
// eight elements per thread to quantize, as many as a thread requests ahead of the weights (own launch / in the workgroups, us: q+k+v of 2560 elements,
// three rows 8.2 / 7.0, five 8.2 / 7.4, eight (four items) 8.2 / 8.3; gate+up 12.0 / 10.2, 11.9 / 10.7, 11.9 / 11.6; o of 4096, four rows 7.5 / 7.1,
// five (five items) 7.6 / 7.8, eight 7.6 / 9.3; 2048 x 6144 Q6_K at four 9.8 / 9.2, at five (five items) 10.1 / 10.4; 1024 x 1024 at three 6.3 / 4.8, at
// eight 6.5 / 5.5).  And where the launch lets waves take two slices each (thirteen and more, kr_shape): three rows of 2560 x 7168 Q4_K 8.3 / 8.6, Q6_K
// 8.9 / 9.5, four 8.5 / 9.4, 9.1 / 10.1; 4096 x 6656 Q6_K 8.9 / 9.5, 9.0 / 10.1.  Same bits.
static bool kr_image(int wtype, const KGemvArgs& a) {
  const bool q4 = wtype == MLLM_HIP_Q4_K;
  const KrShape with = kr_shape(q4, a, 1), without = kr_shape(q4, a, 1, true);
  const int slices = kr_slices(a.nsb);
  return a.M * a.nsb * 32 > 4 * without.tiles * without.waves * 64 || (with.tiles == 1 && slices > 12 && with.waves == (slices + 1) / 2);
}
// Pairs: tiles per wave.  Two save the second round of workgroups, which repeat the search for the pairs and the quantization, but a wave waits for
// twice the weights.  us of a layer of 128 experts, top-8 (top-4 for 768 x 2048), one tile / two (workgroups of the launch with one, all parts; the chip holds 1024 by their registers):
// down of 768 elements, 2048 rows: 30.4 / 32.0 (1280), 33.7 / 34.4 (1536), 42.1 / 41.4 (2048), 49.7 / 48.4 (2560), 57.2 / 57.4 (4096); gate + up of
// 768 elements, 2 x 2048 rows: 26.0 / 25.9 (1536), 29.8 / 28.4 (2048), 34.5 / 33.2 (2560), 44.8 / 45.5 (4096).  Longer rows gain nothing: 1024 elements 41.3 / 42.2
// (1536), 51.5 / 52.4 (2048), 60.5 / 60.7 (3072), 1536 elements 57.9 / 60.2, 73.7 / 75.9, 84.4 / 84.3.  (N is a multiple of 256 here: whole tiles.)
static int kr_pair_tiles(const KGemvArgs& a, unsigned grid_y, int tw) {
  int64_t workgroups = 0;
  for (int i = 0; i < a.nparts; i++) workgroups += (int64_t)grid_y * (((a.part[i].N + 15) / 16 + tw - 1) / tw);
  return a.nsb <= 3 && workgroups >= 2048 ? 2 : 1;
}
template <int WT, int XT, int TH, int ORDER>
static int launch_kq_rows(const KGemvArgs& a_in, hipStream_t st, unsigned grid_y = 1) {
  KGemvArgs a = a_in;
  const KrShape shape = kr_shape(WT == MLLM_HIP_Q4_K, a, grid_y, XT != KQ_IMAGE, ORDER == KR_PAIRS);
  const int tw = shape.tiles, P = shape.waves;
  const size_t lds = kr_lds_bytes(WT == MLLM_HIP_Q4_K, a.nsb, tw, P);
  if (lds > KR_LDS_MAX) return MLLM_HIP_E_SHAPE;
  unsigned grid = 0;
  const int T = ORDER == KR_PAIRS ? kr_pair_tiles(a, grid_y, tw) : 1;
  for (int i = 0; i < a.nparts; i++) {
    a.wg_start[i] = (int)grid;
    grid += (unsigned)(((a.part[i].N + 15) / 16 + tw * T - 1) / (tw * T));
  }
  a.wg_start[a.nparts] = (int)grid;
  auto kern = kq_rows_kernel<WT, XT, TH, ORDER>;
  if (lds > 64 * 1024)
    HIP_RET(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(kern, dim3(grid, grid_y), dim3(tw * P * 64), lds, st, a, ORDER == KR_PAIRS ? T : P);
  return (int)hipGetLastError();
}
template <int XT, int ORDER = KR_LINEAR>
static int launch_kq_rows_any(int wtype, const KGemvArgs& a, hipStream_t st, unsigned grid_y = 1) {
  if (wtype == MLLM_HIP_Q4_K) return launch_kq_rows<MLLM_HIP_Q4_K, XT, 2, ORDER>(a, st, grid_y);
  return a.M <= 4 ? launch_kq_rows<MLLM_HIP_Q6_K, XT, 1, ORDER>(a, st, grid_y) : launch_kq_rows<MLLM_HIP_Q6_K, XT, 2, ORDER>(a, st, grid_y);
}

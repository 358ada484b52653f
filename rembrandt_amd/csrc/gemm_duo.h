// fp32 contractions on the fp16 matrix instructions: every operand value, scaled by a power of two, is the sum of two fp16 values.
//
// a 2^e = a1 + a2 2^-11 with a1 = fp16(a 2^e) and a2 = fp16((a 2^e - a1) 2^11); e is one exponent for a row of the operand (for
// the image of a convolution: for all pixels of an image) and takes its largest value to [2^14, 2^15).  The product of two fp16
// values is exact in fp32, and of the four products of a pair the one of two second parts (2^-22 of it) is left out: three
// v_mfma_f32_32x32x16_f16 do the work for which the exact sum of three bf16 values (gemm_tri.h) needs six.  (Two halves, the second held
// 2^11 times as large, three products and sums kept outside the matrix unit are a published scheme: Ootomo and Yokota, "Recovering single
// precision accuracy from Tensor Cores while surpassing the FP32 theoretical peak performance", 2022.  The exponents by row and what is
// done about values out of range are this library's.)
//
// Precision.  Two parts hold 22 to 24 of a value's 24 bits: three values of four exactly, the fourth is off by its last bit
// (relative error 4.3e-8, rms; with the product left out 7.5e-8 a product, N(0,1) data).  What a sum of many products loses, the
// rounding of its accumulator, is kept shorter than gemm_tri.h keeps it: the chain of large products ends every kDuoChain K steps
// and is added to a sum of its own, in the gradients' passes with what that addition rounds off kept for the next chain (KEEP).
// Relative error against 64 bits at 36, 72, 144 and 216 K steps, half of one operand zeros as behind a ReLU: forward 1.15, 1.2,
// 1.3 and 1.45e-7, data gradient 1.1e-7 at all four; three bf16 parts 1.04, 1.5, 2.2 and 2.8e-7, the fp32 instruction and Winograd 2.3 to
// 3.5e-7.  So it is for long contractions (duo_replaces, conv_common.h).  KEEP costs 5 % of the kernel's time and takes the data
// gradient of AlexNet's conv5, whose deltas are zeros for the most part, from 1.21 to 0.94e-7 (three parts 1.04).
//
// Range.  A value keeps its 22 bits down to 2^-29 of the largest of its row; below that a product with b loses up to 2^-35 b (scaled).  A
// result in which that could be seen is not finite and formed again from the operands themselves on the fp32 instruction (tri_redo), as
// is one with an operand that is no finite number.
// * An image's small value is marked by a NaN in the first part, unless the other seven of its group (eight channels of a pixel, which
//   every result with one of them has, met by eight channels of one tap of a filter) make up for it: ratio is the least one, over the
//   filters, of a value to the largest of its group, so if the group's largest, times it, is n 2^-14 at least, there is a product of
//   n 2^-14 b beside the n 2^-35 b that n small values lose.  Of AlexNet's, NIN's and ResNet-18's activations none was marked, nor of
//   AlexNet's and NIN's deltas.  Behind a batch norm all deltas are small beside the few that a ReLU let through: in ResNet-18 up to 1250 of a
//   tensor are under 2^-29, some of them marked in one call of 25, which takes 0.1 to 0.5 ms longer.
// * A filter's small values (one in 1e8 of normal weights) are counted.  They cost a result 2^-20 each at most, so its sum, before it is
//   scaled back, has to be four times their number: 2^27 is usual.  (A mark would have the filter's whole plane formed again.)
// * In the filter gradient, where the eight of a group are images and zeros of the other operand say nothing of the sum, every small value
//   is marked, and one such value makes it a call in three parts (TriRest; AlexNet's at 26 batches one call in 39, of
//   NIN's the 5x5 layer's 16 of 17, of its 3x3 layers' 7 of 15).
//   Formed again, a block of 32 x 32 results is bound by the latency of its loads, 32 of them in flight (one by one 384 -> 384 3x3 13x13
//   b256 forward took 3.0 ms longer for one value): 330 us, with one value in x 930, with one in every group 3.9 ms (three parts 550 us,
//   1.4 and 2.9 ms); 5x5 of 96 channels 0.6, 0.9 and 12 ms, 1x1 at 128 images 54, 93 and 260 us.  In the filter gradient, whose loads are
//   of 32 channels a plane apart, 350 us, 3.9 and 9.3 ms.
#pragma once
#include "gemm_tri.h"

namespace rh {

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2_t;

constexpr int kDuoChain = 8;         // K steps in a chain of large products (even)
constexpr float kDuoLow = 2048.0f;   // the second part is held 2^11 times as large
constexpr float kDuoBeside = 6.103515625e-5f;   // 2^-14

// The exponent for a row whose largest finite magnitude is `top`.
__device__ __forceinline__ int duo_exponent(float top) {
  const int e = (int)(__builtin_bit_cast(uint32_t, top) >> 23);
  return 141 - (e > 0 ? e : 1);
}

// The bits of the smallest magnitude, in a row with exponent e, of which two parts hold 22 bits: 2^-14 scaled.
__device__ __forceinline__ uint32_t duo_least(int e) {
  const int b = 113 - e;
  return b > 0 ? (uint32_t)b << 23 : b > -23 ? 1u << (22 + b) : 0u;
}

// Eight values (one group) of a row with exponent e; returns how many of them are, but not 0, under duo_least or no finite numbers.
// mark(most, n) says whether the n small ones are marked, most being the group's largest scaled value.
template <class MARK>
__device__ __forceinline__ int duo_pack8(const float (&v)[8], int e, MARK mark, uint4 (&o)[2]) {
  uint32_t w[2][4];
  uint32_t top = 0, low = 0xffffffffu;   // the largest magnitude, and one under the smallest that is not 0
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float x = __builtin_amdgcn_ldexpf(v[2 * i], e), y = __builtin_amdgcn_ldexpf(v[2 * i + 1], e);
    const f16x2_t h = {(_Float16)x, (_Float16)y};
    const f16x2_t l = {(_Float16)((x - (float)h.x) * kDuoLow), (_Float16)((y - (float)h.y) * kDuoLow)};
    w[0][i] = __builtin_bit_cast(uint32_t, h);
    w[1][i] = __builtin_bit_cast(uint32_t, l);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const uint32_t bits = __builtin_bit_cast(uint32_t, v[2 * i + k]) & 0x7fffffffu;
      top = bits > top ? bits : top;
      low = bits - 1u < low ? bits - 1u : low;
    }
  }
  const uint32_t least = duo_least(e), under = least > 0 ? least - 1u : 0u;
  int lost = 0;
  if ((low < under) | (top >= 0x7f800000u)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) lost += (__builtin_bit_cast(uint32_t, v[i]) & 0x7fffffffu) - 1u < under;
    const bool small = mark(__builtin_amdgcn_ldexpf(__builtin_bit_cast(float, top), e), lost);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t bits = __builtin_bit_cast(uint32_t, v[2 * i + h]) & 0x7fffffffu;
        lost += bits >= 0x7f800000u;
        if (bits >= 0x7f800000u || (small && bits - 1u < under)) {
          const uint32_t keep = h ? 0xffffu : 0xffff0000u;
          w[0][i] = (w[0][i] & keep) | (0x7e00u << (16 * h));
          w[1][i] &= keep;
        }
      }
    }
  }
#pragma unroll
  for (int p = 0; p < 2; ++p) o[p] = make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]);
  return lost;
}

// An operand of this form: TriParams with two parts, the exponents of its rows: row m has exps[m / ediv % emod], and the counts of their
// small values (of A, nullptr in the filter gradient).
struct DuoParams {
  TriParams t;
  const int *exps, *lost;
  int ediv, emod;
};

// The operands themselves, for results that are formed again (and for nothing else: index arithmetic in full).
struct DuoSource {
  int pass;                 // RH_CONV_*
  const float *a, *b;       // forward: filter, image; backward-data: filter, dy; backward-filter: dy, image
  int N, C, H, W;           // of the tensor b
  int rows, R, S, st, halo, P, Q;
  // eight values `stride` floats apart, the first n of them there
  static __device__ __forceinline__ void load8(const float* p, size_t stride, int n, float (&v)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float x = p[e < n ? e * stride : 0];
      v[e] = e < n ? x : 0.0f;
    }
  }
  // row, or column, m of the operand; its eight values of group g
  __device__ __forceinline__ void load_a(int m, int g, float (&v)[8]) const {
    if (pass == RH_CONV_BWD_FILTER) {
      const int PQ = P * Q, n8 = g / PQ, pq = g - n8 * PQ;
      return load8(a + ((size_t)n8 * 8 * rows + m) * PQ + pq, (size_t)rows * PQ, N - n8 * 8, v);
    }
    int rs, c0;
    tap(g, rs, c0);
    const int RS = R * S;
    if (pass == RH_CONV_BWD_DATA) load8(a + ((size_t)c0 * rows + m) * RS + (RS - 1 - rs), (size_t)rows * RS, 8, v);
    else load8(a + ((size_t)m * C + c0) * RS + rs, RS, 8, v);
  }
  __device__ __forceinline__ void load_b(int m, int g, float (&v)[8]) const {
    if (pass == RH_CONV_BWD_FILTER) {   // m = (r, s, c)
      const int PQ = P * Q, n8 = g / PQ, pq = g - n8 * PQ, p = pq / Q, q = pq - p * Q;
      const int rs = m / C, c = m - rs * C, r = rs / S, h = p * st + r - halo, w = q * st + (rs - r * S) - halo;
      if ((unsigned)h >= (unsigned)H || (unsigned)w >= (unsigned)W) return;
      return load8(b + (((size_t)n8 * 8 * C + c) * H + h) * W + w, (size_t)C * H * W, N - n8 * 8, v);
    }
    int rs, c0;
    tap(g, rs, c0);
    const int PQ = P * Q, n = m / PQ, pq = m - n * PQ, p = pq / Q, q = pq - p * Q, r = rs / S;
    const int h = p * st + r - halo, w = q * st + (rs - r * S) - halo;
    if (n >= N || (unsigned)h >= (unsigned)H || (unsigned)w >= (unsigned)W) return;
    load8(b + (((size_t)n * C + c0) * H + h) * W + w, (size_t)H * W, 8, v);
  }
  // the tap and the first channel of group g (tri_filter_body's order)
  __device__ __forceinline__ void tap(int g, int& rs, int& c0) const {
    const int RS = R * S, pairs = C / 16 * RS, step = g >> 1;
    if (step < pairs) {
      rs = step % RS;
      c0 = step / RS * 16 + (g & 1) * 8;
    } else {
      rs = g - 2 * pairs;
      c0 = C - 8;
    }
  }
};

// Brings one K step (16 k = two groups, two parts) of both operands to LDS with direct loads: four a block of 64 rows.  Each wave
// brings one block; of a fifth block (the last of B) each wave brings one (part, group).
template <int RA, int RB>
struct DmaDuo {
  static constexpr int NB = (RA + RB) / 64;
  static_assert(RA % 64 == 0 && RB % 64 == 0 && (NB == 4 || NB == 5), "a block of rows for every wave");
  static constexpr int CNT = NB;
  typedef const __attribute__((address_space(4))) int* ctab_t;
  u32x4 rsrc, xrsrc;
  const int* tab;
  uint32_t vbase, lds, lds_slab, xvbase, xlds;
  int plane, gstride, xplane, xhalf;
  bool linear;
  int so[2], xso;

  static __device__ __forceinline__ u32x4 resource(const RowV8Params& p) {
    const uint64_t a = reinterpret_cast<uint64_t>(p.ptr);
    u32x4 r;
    r.x = __builtin_amdgcn_readfirstlane((uint32_t)a);
    r.y = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32) & 0xffffu);
    r.z = __builtin_amdgcn_readfirstlane(p.bytes);
    r.w = 0x00020000u;
    return r;
  }
  static __device__ __forceinline__ uint32_t row_offset(const RowV8Params& p, int m) {
    if (m >= p.M) return 0x80000000u;
    const int n = m / p.inner, rem = m - n * p.inner, a2 = rem / p.innerW, b2 = rem - a2 * p.innerW;
    return (uint32_t)(n * p.img_stride + a2 * p.a_stride + b2 * p.b_stride);
  }
  __device__ __forceinline__ void init(const DuoParams& ap, const DuoParams& bp, int m0, int n0, int wave, int lane) {
    const bool is_a = wave < RA / 64;
    const TriParams& t = is_a ? ap.t : bp.t;
    rsrc = resource(t.v);
    tab = bp.t.v.soff;
    plane = __builtin_amdgcn_readfirstlane(t.plane);
    gstride = __builtin_amdgcn_readfirstlane(t.v.group_stride);
    linear = is_a;
    const int rb = is_a ? wave : wave - RA / 64;
    lds = (uint32_t)(((is_a ? 0 : 4 * RA) + rb * 64) * 16);
    lds_slab = (uint32_t)((is_a ? RA : RB) * 16);
    vbase = row_offset(t.v, (is_a ? m0 : n0) + rb * 64 + lane);
    if (NB == 5) {
      xrsrc = resource(bp.t.v);
      xhalf = wave >> 1;
      xplane = __builtin_amdgcn_readfirstlane((wave & 1) * bp.t.plane);
      xlds = (uint32_t)((4 * RA + RB - 64 + ((wave & 1) * 2 + xhalf) * RB) * 16);
      xvbase = row_offset(bp.t.v, n0 + RB - 64 + lane);
    }
  }
  // (scalar loads, which the hand-counted vmcnt of the direct loads does not see)
  __device__ __forceinline__ void prep(int step) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int g = 2 * step + h;
      const int t = ((ctab_t)(uintptr_t)tab)[g];
      so[h] = linear ? g * gstride : t;
      if (NB == 5 && h == xhalf) xso = t;
    }
  }
  __device__ __forceinline__ void issue(uint32_t base, int i) const {   // i = part + 2 group; 4: the share of the fifth block
    if (i < 4) dma_load16(rsrc, base + lds + (uint32_t)((i & 1) * 2 + i / 2) * lds_slab, vbase, (uint32_t)(so[i / 2] + (i & 1) * plane));
    else dma_load16(xrsrc, base + xlds, xvbase, (uint32_t)(xso + xplane));
  }
};

// The ring: a step of four blocks of 64 rows is 16 KB, of five 20 KB; two blocks share a CU's 160 KB.
template <class T>
struct DuoShape {
  static constexpr int RA = (T::BM + 63) / 64 * 64, RB = (T::BN + 63) / 64 * 64, STEP = 4 * (RA + RB), R = 80 * 1024 / (16 * STEP), LDS = R * STEP * 16;
  static_assert(T::NT == 4 * kWave && T::BK == 16 && R >= 4, "four waves, 16 k a step");
};

// K steps [s_begin, s_end) of the tile at (m0, n0).  Three MFMAs for each 32 x 32 block of a wave and step: a2 b1, a1 b2 (accumulators
// of their own, 2^11 times as large) and a1 b1.  a2 and b2 of the next step are read over this step's once their product has been
// issued, a1 and b1 into a second set: 64 x 64 of a 128 x 128 tile are 192 accumulators in three sets and 48 registers of operands, two
// waves to a SIMD.  Step `it` of a wave issues the loads of step it + R - 1 into the buffer that step it - 1 left, so they
// have R - 2 steps to land.  Bound by the power that the MFMAs draw: 384 -> 384 3x3 13x13 b256 forward takes 270 us = 425 TFLOP/s of fp32
// multiply-adds (three bf16 parts 470 us; from registers alone three products reach 530 to 573 TFLOP/s with N(0,1) operands, 580 to 622 where
// half of one are zeros, from box to box).  In AlexNet's step at 256 images the matrix pipes are busy 64 to 69 % of the time forward, at
// 1.6 to 1.9 GHz, and 58 to 63 % in the gradients, at 1.8 to 2.1 GHz, where the ends of chains (KEEP) and their sums are 4.0 to 4.5 VALU
// instructions an MFMA for 2.5.  A barrier every second step, or a raised wave priority, changes nothing.
template <class T, bool NCHW, bool KEEP>
__device__ __forceinline__ void duo_block(const DuoParams& ap, const DuoParams& bp, const DuoSource& src, const EpiParams& ep, int m0,
                                          int n0, int s_begin, int s_end, int groups, int dst_split) {
  typedef DuoShape<T> D;
  constexpr int TM = T::TM, TN = T::TN, Q = TM * TN, R = D::R, RA = D::RA, RBn = D::RB;
  typedef DmaDuo<RA, RBn> Loader;
  constexpr int SA = 4 * RA, SB = 4 * RBn;   // 16-byte pieces of a step
  extern __shared__ float lds_dyn[];
  uint4* const sm = reinterpret_cast<uint4*>(lds_dyn);   // [R][A: part, group, row; B]
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)sm;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % T::WM, wn = wave / T::WM;
  const int nk = s_end - s_begin;

  Loader ld;
  ld.init(ap, bp, m0, n0, wave, lane);

  f32x16 zero;
#pragma unroll
  for (int v = 0; v < 16; ++v) zero[v] = 0.0f;
  f32x16 acc[TM][TN], low[TM][TN], sum[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = low[i][j] = sum[i][j] = zero;

#pragma unroll
  for (int s = 0; s < R - 1; ++s)
    if (s < nk) {
      ld.prep(s_begin + s);
#pragma unroll
      for (int i = 0; i < Loader::CNT; ++i) ld.issue(lds0 + (uint32_t)(s * (SA + SB)) * 16u, i);
    }
  int lost_here = 0;   // small values in the wave's rows (looked at once the first steps have landed)
  if (ap.lost)
#pragma unroll
    for (int r = 0; r < TM * 32; r += 64)
      if (r + lane < TM * 32) lost_here |= ap.lost[m0 + wm * (TM * 32) + r + lane];
  ld.prep(s_begin + (R - 1 < nk ? R - 1 : nk - 1));
  wait_vmcnt<0>();
  __syncthreads();
  const bool any_lost = __any(lost_here != 0);

  const uint4* const pa0 = sm + (lane >> 5) * RA + wm * (TM * 32) + (lane & 31);
  const uint4* const pb0 = sm + SA + (lane >> 5) * RBn + wn * (TN * 32) + (lane & 31);
  uint4 a1[2][TM], b1[2][TN], a2[TM], b2[TN];
#pragma unroll
  for (int i = 0; i < TM; ++i) { a1[0][i] = pa0[i * 32]; a2[i] = pa0[2 * RA + i * 32]; }
#pragma unroll
  for (int j = 0; j < TN; ++j) { b1[0][j] = pb0[j * 32]; b2[j] = pb0[2 * RBn + j * 32]; }

  // element x of a wave's chains to its sum; KEEP: what that rounds off is where the next chain begins
  auto end_chain = [&](int x) {
    f32x16& d = sum[x / 16 / TN][x / 16 % TN];
    f32x16& c = acc[x / 16 / TN][x / 16 % TN];
    const float s = d[x % 16] + c[x % 16];
    if constexpr (KEEP) c[x % 16] -= s - d[x % 16];
    d[x % 16] = s;
    if constexpr (!KEEP)
      if (x % 16 == 15) asm volatile("" : "+v"(d));   // (formed here, not where it is used next)
  };

  int rd = 0;   // buffer of the current step
  auto step = [&](int it, auto c_tag, auto more_tag, auto first_tag) {
    constexpr int c = decltype(c_tag)::value, n = c ^ 1;
    constexpr bool MORE = decltype(more_tag)::value;     // this step issues the loads of step it + R - 1
    constexpr bool FIRST = decltype(first_tag)::value;   // of a chain: the one that ended goes to the sum
    __builtin_amdgcn_sched_barrier(0);
    if (MORE) wait_vmcnt<(R - 3) * Loader::CNT>();
    else wait_vmcnt<0>();
    __syncthreads();
    const int nx = rd + 1 == R ? 0 : rd + 1, past = rd == 0 ? R - 1 : rd - 1;
    const uint4* const pa = pa0 + nx * (SA + SB);
    const uint4* const pb = pb0 + nx * (SA + SB);
    const uint32_t base = lds0 + (uint32_t)(past * (SA + SB)) * 16u;
    rd = nx;
    constexpr int kA1 = TM, kB1 = kA1 + TN, kA2 = kB1 + TM, kB2 = kA2 + TN;
    auto read = [&](int s) {
      if (s < kA1) a1[n][s] = pa[s * 32];
      else if (s < kB1) b1[n][s - kA1] = pb[(s - kA1) * 32];
      else if (s < kA2) a2[s - kB1] = pa[2 * RA + (s - kB1) * 32];
      else if (s < kB2) b2[s - kA2] = pb[2 * RBn + (s - kA2) * 32];
    };
    int slot = 0, load = 0, moved = 0;
#pragma unroll
    for (int m = 0; m < 3 * Q; ++m) {
      const int p = m / Q, t = m % Q, i = t / TN, j = t % TN;
      if (p < 2)
        low[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, p ? a1[c][i] : a2[i]),
                                                           __builtin_bit_cast(f16x8_t, p ? b2[j] : b1[c][j]), low[i][j], 0, 0, 0);
      else
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a1[c][i]), __builtin_bit_cast(f16x8_t, b1[c][j]),
                                                           FIRST && !KEEP ? zero : acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (FIRST) {
#pragma unroll
        for (; moved < 16 * Q && moved < (m + 1) * 8; ++moved) end_chain(moved);
      }
      // a1 and b1 at any time, a2 behind the first product, b2 behind the second
      const int upto = m < Q ? (m + 1) * kB1 / Q : m < 2 * Q ? kB1 + (m + 1 - Q) * TM / Q : m + 1 - 2 * Q < TN ? kA2 + m + 1 - 2 * Q : kB2;
#pragma unroll
      for (; slot < upto; ++slot) read(slot);
      if (MORE) {
#pragma unroll
        for (; load < Loader::CNT && load < (m + 1) * Loader::CNT / (3 * Q - 2); ++load) ld.issue(base, load);
        if (m == 3 * Q - 1) ld.prep(s_begin + (it + R < nk ? it + R : nk - 1));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  const std::integral_constant<int, 0> c0;
  const std::integral_constant<int, 1> c1;
  const std::true_type yes;
  const std::false_type no;
  int it = 0;
  for (; it + kDuoChain + R - 2 < nk; it += kDuoChain) {
    step(it, c0, yes, yes);
#pragma unroll 1
    for (int u = 1; u + 1 < kDuoChain; u += 2) {
      step(it + u, c1, yes, no);
      step(it + u + 1, c0, yes, no);
    }
    step(it + kDuoChain - 1, c1, yes, no);
  }
  if (it > 0) {
#pragma unroll
    for (int x = 0; x < 16 * Q; ++x) {
      end_chain(x);
      if (!KEEP) acc[x / 16 / TN][x / 16 % TN][x % 16] = 0.0f;
    }
  }
  for (; it + R < nk; it += 2) {
    step(it, c0, yes, no);
    step(it + 1, c1, yes, no);
  }
  if (it + R - 1 < nk) {
    step(it, c0, yes, no);
    step(it + 1, c1, no, no);
    it += 2;
  }
  while (it < nk) {
    step(it++, c0, no, no);
    if (it >= nk) break;
    step(it++, c1, no, no);
  }

  if (any_lost) {   // (sums in which small values could be seen)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const float least = 4.0f * (float)ap.lost[m0 + wm * (TM * 32) + i * 32 + (lane >> 5) * 4 + (v >> 2) * 8 + (v & 3)];
#pragma unroll
        for (int j = 0; j < TN; ++j)
          if (fabsf(sum[i][j][v] + fmaf(low[i][j][v], 1.0f / kDuoLow, acc[i][j][v])) < least) sum[i][j][v] = __builtin_nanf("");
      }
  }

  // the sums, scaled back by the row's and the column's exponent
  int eb[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int col = n0 + wn * (TN * 32) + j * 32 + (lane & 31);
    eb[j] = col < bp.t.v.M ? bp.exps[col / bp.ediv % bp.emod] : 0;
  }
  float finite = 0.0f;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int row = m0 + wm * (TM * 32) + i * 32 + (lane >> 5) * 4;   // (the exponents are there up to a multiple of 128 rows)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int4 ea = *reinterpret_cast<const int4*>(ap.exps + row + 8 * q);
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int v = 4 * q + u, e = u == 0 ? ea.x : u == 1 ? ea.y : u == 2 ? ea.z : ea.w;
          const float d = sum[i][j][v] + fmaf(low[i][j][v], 1.0f / kDuoLow, acc[i][j][v]);
          acc[i][j][v] = __builtin_amdgcn_ldexpf(d, -(e + eb[j]));
          finite = fmaf(acc[i][j][v], 0.0f, finite);
        }
    }
  }
  if (__any(!(finite == 0.0f))) {
    const int g0 = 2 * s_begin, g1 = 2 * s_end < groups ? 2 * s_end : groups;
#pragma unroll 1
    for (int t = 0; t < Q; ++t) {
      f32x16 d = acc[0][0];
#pragma unroll
      for (int u = 1; u < Q; ++u)
        if (t == u) d = acc[u / TN][u % TN];
      const int row0 = m0 + wm * (TM * 32) + t / TN * 32, col0 = n0 + wn * (TN * 32) + t % TN * 32;
      const int ra = row0 + (lane & 31) < ep.rows ? row0 + (lane & 31) : 0, cb = col0 + (lane & 31) < ep.cols ? col0 + (lane & 31) : 0;
      tri_redo(d, ep.rows - row0, ep.cols - col0, lane, g0, g1, [&](int g, float (&v)[8]) { src.load_a(ra, g, v); },
               [&](int g, float (&v)[8]) { src.load_b(cb, g, v); });
#pragma unroll
      for (int u = 0; u < Q; ++u)
        if (t == u) acc[u / TN][u % TN] = d;
    }
  }
  store_tile<T, NCHW>(acc, ep, m0, n0, wm, wn, lane, dst_split);
}

template <class T, bool NCHW, class PASS>
__global__ __launch_bounds__(T::NT, T::OCC) void mfma_gemm_duo_kernel(DuoParams ap, DuoParams bp, DuoSource src, EpiParams ep,
                                                                      int tiles_m, int k_steps, int steps_per_split, int groups, TriRest rest) {
  if constexpr (std::is_same<PASS, PassConvBwdFilter>::value) {
    if (rest.any && *rest.any != 0) {
      tri_rest_blocks<typename std::conditional<T::BM == 64, T64x192t, T>::type>(rest, ep);
      return;
    }
  }
  int slice, logical, dst_split;   // as in mfma_gemm_kernel
  if (ep.tail_tiles > 0) {
    const int b = blockIdx.x;
    if (b < ep.full_tiles) {
      logical = xcd_remap(b, ep.full_tiles);
      slice = 0;
      dst_split = -1;
    } else {
      const int r = xcd_remap(b - ep.full_tiles, ep.tail_tiles * ep.tail_splits);
      slice = r / ep.tail_tiles;
      logical = ep.full_tiles + (r - slice * ep.tail_tiles);
      dst_split = slice;
    }
  } else {
    const int tiles = gridDim.x;
    const int linear = xcd_remap(blockIdx.y * tiles + blockIdx.x, tiles * gridDim.y);
    slice = linear / tiles;
    logical = linear - slice * tiles;
    dst_split = ep.split_stride != 0 ? slice : -1;
  }
  slice = __builtin_amdgcn_readfirstlane(slice);
  logical = __builtin_amdgcn_readfirstlane(logical);
  dst_split = __builtin_amdgcn_readfirstlane(dst_split);
  const int tile_m = logical % tiles_m, tile_n = logical / tiles_m;
  const bool whole = ep.tail_tiles > 0 && dst_split < 0;
  const int s_begin = whole ? 0 : slice * steps_per_split;
  int s_end = whole ? k_steps : s_begin + steps_per_split;
  if (s_end > k_steps) s_end = k_steps;
  duo_block<T, NCHW, !std::is_same<PASS, PassConvFwd>::value>(ap, bp, src, ep, tile_m * T::BM, tile_n * T::BN, s_begin, s_end, groups, dst_split);
}

}  // namespace rh

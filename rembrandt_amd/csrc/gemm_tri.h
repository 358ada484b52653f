// fp32 contractions on the bf16 matrix instructions: every operand value is the sum of three bf16 values.
//
// v_mfma_f32_32x32x2_f32 executes 256 FLOP per cycle and SIMD, v_mfma_f32_32x32x16_bf16 sixteen times that.  An fp32
// value a is exactly a1 + a2 + a3 with a1 = bf16(a), a2 = bf16(a - a1), a3 = a - a1 - a2 (8 + 8 + 8 significand bits; for
// all values but those below), the product of two bf16 values is exact in fp32, and of the
// nine products of a pair the three below 2^-24 of it (a2 b3, a3 b2, a3 b3) are left out: six MFMAs do the work of
// eight times 16 / 2 fp32 ones in 6/16 of their time.  Registers only, six products on random data: 302 TFLOP/s of fp32
// multiply-adds (1.81 PFLOP/s of bf16 at the clock it settles at) where the fp32 instruction reaches 154.
//
// Precision.  The five small products of a pair have accumulators of their own, added to the large product's behind the
// loop: one rounding at the size of the sum per 16 terms instead of one per two.  Relative error of chains of 256, 1152 and
// 3456 terms against 64 bits, N(0,1) data: 0.9e-7, 2.0e-7 and 3.6e-7, the fp32 instruction 2.9e-7, 6.1e-7 and 10.4e-7 (with
// one set of accumulators 2.4e-7, 5.2e-7 and 9.2e-7, and above the fp32 instruction where half of one operand is zero).  Operands of
// one sign, uniform [0, 1), chains of 576, 1152, 2304 and 6400 terms: 1.2e-7, 1.7e-7, 2.3e-7 and 4.2e-7, the fp32 instruction at 6400 11e-7.
// Operands whose small values share a sign beside few large ones are what the wide form is for.
//
// Values without such a sum: infinities and NaNs, the floats that round to an infinity in bf16, and below 2^-110 those whose
// last bits lie under bf16's smallest value, 2^-133 (their parts would lose 2^-14 of them at 2^-120, all of them under 2^-134).
// Their first part is a NaN and the other two hold their bits, so every result that has one among its operands comes out as
// a NaN, and a result that is not finite is formed again from the operands' values on the fp32 instruction (tri_redo).
#pragma once
#include "gemm_core.h"

namespace rh {

// An operand of this form: RowV8Params' packed bf16 layout (eight consecutive k of a row are 16 bytes) three times over, the
// parts `plane` bytes apart.  All of it within 2 GiB.
struct TriParams {
  RowV8Params v;
  int plane;
};

// Eight values (one group) into the three parts' groups: pair() for each of the four pairs, then fix().
constexpr uint32_t kTriNoSum = 0x7fc0u;   // first part of a value that is no sum of three
constexpr int kTriWide = 6;              // (the wide form, below)
struct TriPack8 {
  uint32_t w[3][4];
  uint32_t rest = 0;
  __device__ __forceinline__ void pair(const float (&v)[8], int e) {
    float x = v[2 * e], y = v[2 * e + 1];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      w[i][e] = pack_bf16(x, y);
      x -= __builtin_bit_cast(float, w[i][e] << 16);
      y -= __builtin_bit_cast(float, w[i][e] & 0xffff0000u);
    }
    rest |= __builtin_bit_cast(uint32_t, x) | __builtin_bit_cast(uint32_t, y);   // (+0 where the parts add up to the value)
  }
  __device__ __forceinline__ void fix(const float (&v)[8]) {
    if (rest == 0) return;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t bits = __builtin_bit_cast(uint32_t, v[2 * e + h]);
        const uint32_t keep = h ? 0xffffu : 0xffff0000u, sh = 16 * h;
        float x = v[2 * e + h];
#pragma unroll
        for (int i = 0; i < 3; ++i) x -= __builtin_bit_cast(float, h ? w[i][e] & 0xffff0000u : w[i][e] << 16);
        if (__builtin_bit_cast(uint32_t, x) == 0) continue;
        w[0][e] = (w[0][e] & keep) | (kTriNoSum << sh);
        w[1][e] = (w[1][e] & keep) | ((bits >> 16) << sh);
        w[2][e] = (w[2][e] & keep) | ((bits & 0xffffu) << sh);
      }
    }
  }
  // For the wide form, behind fix(): the third part's last bit, 0 for every value from 2^-108 on (what two parts leave of 24 bits),
  // says that a value is under 2^-kTriWide of the group's largest.  A smaller value that needs the bit is made one without a sum.
  __device__ __forceinline__ void rank(const float (&v)[8]) {
    uint32_t top = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t mag = __builtin_bit_cast(uint32_t, v[e]) & 0x7fffffffu;
      if (mag > top) top = mag;
    }
    const uint32_t limit = top > ((uint32_t)kTriWide << 23) ? top - ((uint32_t)kTriWide << 23) : 0u;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t bits = __builtin_bit_cast(uint32_t, v[2 * e + h]);
        const uint32_t keep = h ? 0xffffu : 0xffff0000u, sh = 16 * h;
        if ((w[0][e] >> sh & 0xffffu) == kTriNoSum) continue;
        if (w[2][e] >> sh & 1u) {
          w[0][e] = (w[0][e] & keep) | (kTriNoSum << sh);
          w[1][e] = (w[1][e] & keep) | ((bits >> 16) << sh);
          w[2][e] = (w[2][e] & keep) | ((bits & 0xffffu) << sh);
        } else if ((bits & 0x7fffffffu) < limit) {
          w[2][e] |= 1u << sh;
        }
      }
    }
  }
  __device__ __forceinline__ uint4 part(int i) const { return make_uint4(w[i][0], w[i][1], w[i][2], w[i][3]); }
};
// The value again: p, q, r its parts.
template <bool WIDE>
__device__ __forceinline__ float tri_value(uint32_t p, uint32_t q, uint32_t r) {
  if (WIDE && p != kTriNoSum) r &= ~1u;
  const float sum = __builtin_bit_cast(float, p << 16) + (__builtin_bit_cast(float, q << 16) + __builtin_bit_cast(float, r << 16));
  return p == kTriNoSum ? __builtin_bit_cast(float, q << 16 | r) : sum;
}
__device__ __forceinline__ void tri_pack8(const float (&v)[8], uint4 (&o)[3], bool wide = false) {
  TriPack8 t;
#pragma unroll
  for (int e = 0; e < 4; ++e) t.pair(v, e);
  t.fix(v);
  if (wide) t.rank(v);
#pragma unroll
  for (int i = 0; i < 3; ++i) o[i] = t.part(i);
}

// Brings one K step (16 k = two groups, three parts) of both operands to LDS with direct loads.  A tile has four blocks of
// 64 rows, A's first, and each of the four waves brings one of them: six loads.
template <int RA, int RB, bool B_LINEAR>
struct DmaTri {
  static_assert(RA % 64 == 0 && RB % 64 == 0 && RA + RB == 256, "a block of rows for every wave");
  static constexpr int CNT = 6;
  typedef const __attribute__((address_space(4))) int* ctab_t;
  u32x4 rsrc;
  const int* tab;
  uint32_t vbase, lds, lds_slab;   // of a step's LDS: this wave's block, and from a (part, group) to the next
  int plane, gstride;
  bool linear;
  int so[2];

  __device__ __forceinline__ void init(const TriParams& ap, const TriParams& bp, int m0, int n0, int wave, int lane) {
    const bool is_a = wave < RA / 64;
    const TriParams& t = is_a ? ap : bp;
    const RowV8Params& p = t.v;
    const uint64_t a = reinterpret_cast<uint64_t>(p.ptr);
    rsrc.x = __builtin_amdgcn_readfirstlane((uint32_t)a);
    rsrc.y = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32) & 0xffffu);
    rsrc.z = __builtin_amdgcn_readfirstlane(p.bytes);
    rsrc.w = 0x00020000u;
    tab = bp.v.soff;
    plane = __builtin_amdgcn_readfirstlane(t.plane);
    gstride = __builtin_amdgcn_readfirstlane(p.group_stride);
    linear = is_a || B_LINEAR;
    const int rb = is_a ? wave : wave - RA / 64;
    lds = (uint32_t)(((is_a ? 0 : 6 * RA) + rb * 64) * 16);
    lds_slab = (uint32_t)((is_a ? RA : RB) * 16);
    const int m = (is_a ? m0 : n0) + rb * 64 + lane;
    const bool valid = m < p.M;
    const int mm = valid ? m : 0;
    const int n = mm / p.inner, rem = mm - n * p.inner;
    const int a2 = rem / p.innerW, b2 = rem - a2 * p.innerW;
    vbase = valid ? (uint32_t)(n * p.img_stride + a2 * p.a_stride + b2 * p.b_stride) : 0x80000000u;
  }
  // (scalar loads, which the hand-counted vmcnt of the direct loads does not see)
  __device__ __forceinline__ void prep(int step) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int g = 2 * step + h;
      so[h] = g * gstride;
      if (!B_LINEAR) {
        const int t = ((ctab_t)(uintptr_t)tab)[g];
        if (!linear) so[h] = t;
      }
    }
  }
  __device__ __forceinline__ void issue(uint32_t base, int i) const {   // i = part + 3 group
    dma_load16(rsrc, base + lds + (uint32_t)((i % 3) * 2 + i / 3) * lds_slab, vbase, (uint32_t)(so[i / 3] + (i % 3) * plane));
  }
};

// The block d of 32 x 32 results with its elements that are not finite and lie in the result formed again over groups
// [g0, g1) on the fp32 instruction: load_a(g, v) and load_b(g, v) give this lane's row (lane % 32) and column their eight values of
// group g.  Two levels of sums, 128 terms each, as the chains of K steps may be longer than fp32's rounding allows.  The whole wave
// takes part whether one element or all of them are formed.  Bound by the latency of its own loads, so a call with one such value takes
// 50 to 1100 us longer, one with one in every group 3 to 8 times as long (96 -> 256 5x5 27x27 b256 forward 1000 us, with one such value
// 1180, with one in every group 5190).
template <class LA, class LB>
__device__ __forceinline__ void tri_redo(f32x16& d, int rows_left, int cols_left, int lane, int g0, int g1, LA load_a, LB load_b) {
  bool any = false;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const bool in = (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3) < rows_left && (lane & 31) < cols_left;
    any |= in && !(fabsf(d[v]) < INFINITY);
  }
  if (!__any(any)) return;
  f32x16 sum;
#pragma unroll
  for (int v = 0; v < 16; ++v) sum[v] = 0.0f;
#pragma unroll 1
  for (int top = g0; top < g1; top += 16) {
    f32x16 part;
#pragma unroll
    for (int v = 0; v < 16; ++v) part[v] = 0.0f;
#pragma unroll 1
    for (int g = top; g < top + 16 && g < g1; g += 4) {   // (the loads of four groups in flight)
      float a[2][8], b[2][8];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int mine = g + 2 * u + (lane >> 5);   // k 0 and 1 of an MFMA: of this group and of the next
#pragma unroll
        for (int e = 0; e < 8; ++e) a[u][e] = b[u][e] = 0.0f;
        if (mine < g1) {
          load_a(mine, a[u]);
          load_b(mine, b[u]);
        }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) part = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u][e], b[u][e], part, 0, 0, 0);
    }
    sum += part;
  }
#pragma unroll
  for (int v = 0; v < 16; ++v)
    if (!(fabsf(d[v]) < INFINITY)) d[v] = sum[v];
}

// Row (or column) m of an operand of three parts: its eight values of the group `at` bytes into it.
struct TriRow {
  const char* base;
  int plane;
  __device__ __forceinline__ TriRow(const TriParams& t, int m) : plane(t.plane) {
    const RowV8Params& p = t.v;
    const int mm = m < p.M ? m : 0;
    const int n = mm / p.inner, rem = mm - n * p.inner, a2 = rem / p.innerW, b2 = rem - a2 * p.innerW;
    base = static_cast<const char*>(p.ptr) + (uint32_t)(n * p.img_stride + a2 * p.a_stride + b2 * p.b_stride);
  }
  template <bool WIDE>
  __device__ __forceinline__ void load(size_t at, float (&v)[8]) const {
    uint32_t w[3][4];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const uint4 p = *reinterpret_cast<const uint4*>(base + at + (size_t)i * plane);
      w[i][0] = p.x; w[i][1] = p.y; w[i][2] = p.z; w[i][3] = p.w;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[2 * e] = tri_value<WIDE>(w[0][e] & 0xffffu, w[1][e] & 0xffffu, w[2][e] & 0xffffu);
      v[2 * e + 1] = tri_value<WIDE>(w[0][e] >> 16, w[1][e] >> 16, w[2][e] >> 16);
    }
  }
};

// A block's tile in a ring of R buffers of one K step each.  Step `it` of a wave: its operands are in registers (read a step
// ago); once all waves are there, buffer `it` is free and buffer it+1 complete; between its MFMAs, one to a slot, it reads
// the operands of step it+1 and issues the loads of step it+R into buffer `it`, which then have R - 1 steps to land.
// A wave is 64 x 64 of a 128 x 128 tile (128 accumulators in two sets, twice 48 registers of operands: two waves to a SIMD,
// two blocks to a CU): 12 operand reads of 1 KB for 24 MFMAs, half of what the LDS delivers, and 24 KB of fill, half of what
// the L2 does.
constexpr int kTriRing = 3;
constexpr int kTriLdsBytes = kTriRing * 6 * 16 * 256;

// The wide form.  The instruction adds eight products at a time (k 0 to 7, then 8 to 15) and cuts each of them toward zero at 2^-24 of
// the largest of the eight; the sum of the eight is rounded to nearest where it joins the accumulator (a probe of the builtin).  Where
// A has a small value of one sign almost everywhere beside a few large ones, as a batch norm's backward leaves behind a ReLU, and B is
// positive, what is cut off the small values' products has one sign and adds up over the sum, in slices or not.  So the first parts
// of A's values under 2^-kTriWide of their group's largest, which the copy marks, are multiplied apart from the others': seven
// MFMAs, and five VALU instructions a register of A between MFMAs that do not wait for them.  64 -> 64 channels 3x3 56x56, 48 images, x
// 1.48 +- 0.6, one delta in ten from N(0, 10), each channel's mean taken off: error against 64 bits 7.6e-7, 9.5e-6 with six MFMAs, 1.4e-6 on
// the fp32 instruction; ResNet-18's filter gradients, 8 to 200 images, relative to the form replaced: 0.43 in the geometric mean of 218
// calls, 0.69 at most; with six MFMAs up to 5.1.  Time, 140 layers and batches of ResNet-18: 1.071 of six MFMAs' in the geometric mean, 64 -> 64 56x56
// b256 509 -> 533 us, 512 -> 512 7x7 b256 296 -> 332; the forms replaced take 754 and 376.
//
// K steps [s_begin, s_end) of the tile at (m0, n0).
template <class T, bool B_LINEAR, bool NCHW, bool WIDE>
__device__ __forceinline__ void tri_block(const TriParams& ap, const TriParams& bp, const EpiParams& ep, int m0, int n0, int s_begin,
                                          int s_end, int groups, int dst_split) {
  constexpr int TM = T::TM, TN = T::TN, R = kTriRing, RA = (T::BM + 63) / 64 * 64, RBn = (T::BN + 63) / 64 * 64;
  static_assert(T::NT == 4 * kWave && T::BK == 16, "four waves, 16 k a step");
  typedef DmaTri<RA, RBn, B_LINEAR> Loader;
  constexpr int SA = 6 * RA, SB = 6 * RBn;   // 16-byte pieces of a step
  extern __shared__ float lds_dyn[];
  uint4* const sm = reinterpret_cast<uint4*>(lds_dyn);   // [R][A: part, group, row; B]
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)sm;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % T::WM, wn = wave / T::WM;

  const int nk = s_end - s_begin;

  Loader ld;
  ld.init(ap, bp, m0, n0, wave, lane);

  f32x16 acc[TM][TN], low[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = low[i][j][v] = 0.0f;

#pragma unroll
  for (int s = 0; s < R; ++s)
    if (s < nk) {
      ld.prep(s_begin + s);
#pragma unroll
      for (int i = 0; i < Loader::CNT; ++i) ld.issue(lds0 + (uint32_t)(s * (SA + SB)) * 16u, i);
    }
  if (nk > R) ld.prep(s_begin + R);
  wait_vmcnt<0>();
  __syncthreads();

  const uint4* const pa0 = sm + (lane >> 5) * RA + wm * (TM * 32) + (lane & 31);
  const uint4* const pb0 = sm + SA + (lane >> 5) * RBn + wn * (TN * 32) + (lane & 31);
  uint4 a[2][3][TM], b[2][3][TN];
#pragma unroll
  for (int p = 0; p < 3; ++p) {
#pragma unroll
    for (int i = 0; i < TM; ++i) a[0][p][i] = pa0[p * 2 * RA + i * 32];
#pragma unroll
    for (int j = 0; j < TN; ++j) b[0][p][j] = pb0[p * 2 * RBn + j * 32];
  }

  int rd = 0;   // buffer of the current step
  auto step = [&](int it, auto c_tag, auto more_tag) {
    constexpr int c = decltype(c_tag)::value, n = c ^ 1;
    constexpr bool MORE = decltype(more_tag)::value;   // this step issues the loads of step it+R
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): this step's operands, asked for a step ago
    if (MORE) wait_vmcnt<(R - 2) * Loader::CNT>();
    else wait_vmcnt<0>();
    __syncthreads();
    const int nx = rd + 1 == R ? 0 : rd + 1;
    const uint4* pa = pa0 + nx * (SA + SB);
    const uint4* pb = pb0 + nx * (SA + SB);
    const uint32_t base = lds0 + (uint32_t)(rd * (SA + SB)) * 16u;
    rd = nx;
    // slots behind the MFMAs: the operand reads first (the next step waits for them), then the loads, then the offsets of
    // the loads that the next step issues
    constexpr int kReads = 3 * (TM + TN), kLoads = Loader::CNT;
    // (the wide form's fourth part of A: the small first parts; its first: those and the large ones, later the large ones alone)
    constexpr int PRODUCTS = WIDE ? 7 : 6;
    constexpr int PA[7] = {0, WIDE ? 0 : 2, 1, WIDE ? 1 : 0, WIDE ? 2 : 1, WIDE ? 3 : 0, 0};
    constexpr int PB[7] = {2, WIDE ? 1 : 0, 1, WIDE ? 0 : 1, 0, 0, 0};
    uint4 small[TM];
    auto apart = [&](int r) {   // register r of A: the marks out of the third part, the small first parts out of the first one
      uint32_t* const a1 = &a[c][0][r >> 2].x + (r & 3);
      uint32_t* const a3 = &a[c][2][r >> 2].x + (r & 3);
      uint32_t* const sm1 = &small[r >> 2].x + (r & 3);
      const uint32_t marks = *a3 & 0x00010001u;
      *a3 ^= marks;
      *sm1 = *a1 & __umul24(marks, 0xffffu);
    };
    auto large = [&](int r) { (&a[c][0][r >> 2].x)[r & 3] ^= (&small[r >> 2].x)[r & 3]; };
    int slot = 0;
    auto fill = [&](int s) {
      if (s < kReads) {
        const int p = s / (TM + TN), x = s % (TM + TN);
        if (x < TM) a[n][p][x] = pa[p * 2 * RA + x * 32];
        else b[n][p][x - TM] = pb[p * 2 * RBn + (x - TM) * 32];
      } else if (MORE && s < kReads + kLoads) {
        ld.issue(base, s - kReads);
      } else if (MORE && s == kReads + kLoads) {
        const int f = it + R + 1 < nk ? it + R + 1 : nk - 1;
        ld.prep(s_begin + f);
      }
    };
    constexpr int kSlots = kReads + kLoads + 1, kMfma = PRODUCTS * TM * TN, kRegs = 4 * TM;
    int taken = 0, left = 0;   // registers of A taken apart, and whose first part is the large ones'
#pragma unroll
    for (int m = 0; m < kMfma; ++m) {
      const int p = m / (TM * TN), t = m % (TM * TN), i = t / TN, j = t % TN;
      f32x16& d = p == PRODUCTS - 1 ? acc[i][j] : low[i][j];
      d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, PA[p] == 3 ? small[i] : a[c][PA[p] % 3][i]),
                                                  __builtin_bit_cast(bf16x8_t, b[c][PB[p]][j]), d, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (WIDE) {   // (the third part and the small ones are used from the fifth product on, the whole first part in the first two)
#pragma unroll
        for (; taken < kRegs && taken < (m + 1) * kRegs / (2 * TM * TN); ++taken) apart(taken);
#pragma unroll
        for (; left < kRegs && left < (m + 1 - 2 * TM * TN) * kRegs / (2 * TM * TN); ++left) large(left);
      }
#pragma unroll
      for (; slot < (m + 1) * kSlots / kMfma || (m + 1 == kMfma && slot < kSlots); ++slot) fill(slot);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  const std::integral_constant<int, 0> c0;
  const std::integral_constant<int, 1> c1;
  int it = 0;
  for (; it + 1 + R < nk; it += 2) {
    step(it, c0, std::true_type());
    step(it + 1, c1, std::true_type());
  }
  if (it + R < nk) {
    step(it, c0, std::true_type());
    step(it + 1, c1, std::false_type());
    it += 2;
  }
  while (it < nk) {
    step(it++, c0, std::false_type());
    if (it >= nk) break;
    step(it++, c1, std::false_type());
  }

  float finite = 0.0f;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      acc[i][j] += low[i][j];
#pragma unroll
      for (int v = 0; v < 16; ++v) finite = fmaf(acc[i][j][v], 0.0f, finite);
    }
  if (__any(!(finite == 0.0f))) {
    const int g0 = 2 * s_begin, g1 = 2 * s_end < groups ? 2 * s_end : groups;
#pragma unroll 1
    for (int t = 0; t < TM * TN; ++t) {
      f32x16 d = acc[0][0];
#pragma unroll
      for (int u = 1; u < TM * TN; ++u)
        if (t == u) d = acc[u / TN][u % TN];
      const int row0 = m0 + wm * (TM * 32) + t / TN * 32, col0 = n0 + wn * (TN * 32) + t % TN * 32;
      const TriRow ra(ap, row0 + (lane & 31)), rb(bp, col0 + (lane & 31));
      tri_redo(d, ep.rows - row0, ep.cols - col0, lane, g0, g1,
               [&](int g, float (&v)[8]) { ra.template load<WIDE>((size_t)g * ap.v.group_stride, v); },
               [&](int g, float (&v)[8]) { rb.template load<false>(B_LINEAR ? (size_t)g * bp.v.group_stride : (size_t)bp.v.soff[g], v); });
#pragma unroll
      for (int u = 0; u < TM * TN; ++u)
        if (t == u) acc[u / TN][u % TN] = d;
    }
  }
  store_tile<T, NCHW>(acc, ep, m0, n0, wm, wn, lane, dst_split);
}

template <class T, bool B_LINEAR, bool NCHW, class PASS, bool WIDE = false>
__global__ __launch_bounds__(T::NT, T::OCC) void mfma_gemm_tri_kernel(TriParams ap, TriParams bp, EpiParams ep, int tiles_m,
                                                                      int k_steps, int steps_per_split, int groups) {
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
  const int m0 = tile_m * T::BM, n0 = tile_n * T::BN;
  const bool whole = ep.tail_tiles > 0 && dst_split < 0;
  const int s_begin = whole ? 0 : slice * steps_per_split;
  int s_end = whole ? k_steps : s_begin + steps_per_split;
  if (s_end > k_steps) s_end = k_steps;
  tri_block<T, B_LINEAR, NCHW, WIDE>(ap, bp, ep, m0, n0, s_begin, s_end, groups, dst_split);
}

// A filter gradient in three parts for operands that two fp16 parts cannot hold: *any is set where their copies met a value with too few
// bits there.  Its copies are a launch of a few blocks, its contraction the work of the blocks of the one in two parts (gemm_duo.h),
// so that where it is not wanted it costs one short launch.
struct TriRest {
  const int* any;   // nullptr: no such form
  TriParams ap, bp;
  int tiles_m, tiles, splits, k_steps, steps_per_split, groups;
};
int launch_tri_rest_copies(const ConvDims& d, const TriFilterPlan& p, const float* x, const float* dy, void* ws, const int* any,
                           hipStream_t stream, TriRest* rest);
template <class T>
__device__ __forceinline__ void tri_rest_blocks(const TriRest& r, const EpiParams& ep) {
  const int blocks = (int)(gridDim.x * gridDim.y), total = r.tiles * r.splits;
  for (int b = (int)(blockIdx.y * gridDim.x + blockIdx.x); b < total; b += blocks) {
    const int slice = __builtin_amdgcn_readfirstlane(b / r.tiles), logical = __builtin_amdgcn_readfirstlane(b - slice * r.tiles);
    const int s0 = slice * r.steps_per_split, s1 = s0 + r.steps_per_split < r.k_steps ? s0 + r.steps_per_split : r.k_steps;
    tri_block<T, false, false, false>(r.ap, r.bp, ep, logical % r.tiles_m * T::BM, logical / r.tiles_m * T::BN, s0, s1, r.groups,
                                      ep.split_stride != 0 ? slice : -1);
    __syncthreads();   // (the ring is the next tile's)
  }
}

// Backward-data of stride 2 to 4 (conv_common.h: residue classes): the classes' contractions in one launch, the longest first, so that
// the short ones fill the last round (launched one by one the classes of 64 -> 128 56x56 b24 are 98 tiles each on 256 CUs).  Bound by
// the MFMAs as above and by the classes' results, which a second pass interleaves.
struct TriClass {
  int first_tile, steps, groups_true;
  int tiles, slice_steps;    // of a slice: its tiles, and K steps at most
  int cols, inner, innerW;   // n U V, U V, V
  uint32_t wt_at, img_at;    // bytes into the operand copies: the class's filter, its first pixel at its first tap
  int soff_at;
  long long out_at;          // floats
};
struct TriClasses { int count, tiles_m; long long slab; TriClass c[16]; };   // slab: floats from a slice's results to the next's
template <class T>
__global__ __launch_bounds__(T::NT, T::OCC) void mfma_gemm_tri_classes_kernel(TriParams ap, TriParams bp, EpiParams ep, TriClasses t) {
  const int block = blockIdx.x;
  int i = 0;
  while (i + 1 < t.count && block >= t.c[i + 1].first_tile) ++i;
  i = __builtin_amdgcn_readfirstlane(i);
  const TriClass c = t.c[i];
  const int blocks = (i + 1 < t.count ? t.c[i + 1].first_tile : (int)gridDim.x) - c.first_tile;
  const int linear = __builtin_amdgcn_readfirstlane(xcd_remap(block - c.first_tile, blocks));
  const int slice = linear / c.tiles, logical = linear - slice * c.tiles;
  const int s0 = slice * c.slice_steps, s1 = s0 + c.slice_steps < c.steps ? s0 + c.slice_steps : c.steps;
  ap.v.ptr = static_cast<const char*>(ap.v.ptr) + c.wt_at;
  ap.plane = c.steps * 2 * ap.v.M * 16;
  ap.v.bytes = (uint32_t)(3 * ap.plane);
  bp.v.ptr = static_cast<const char*>(bp.v.ptr) + c.img_at;
  bp.v.bytes -= c.img_at;
  bp.v.M = c.cols; bp.v.inner = c.inner; bp.v.innerW = c.innerW;
  bp.v.soff += c.soff_at;
  ep.out += c.out_at + slice * t.slab;
  ep.cols = c.cols; ep.inner = c.inner;
  tri_block<T, false, true, false>(ap, bp, ep, logical % t.tiles_m * T::BM, logical / t.tiles_m * T::BN, s0, s1, c.groups_true, -1);
}

}  // namespace rh

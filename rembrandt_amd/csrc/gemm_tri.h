// fp32 contractions on the bf16 matrix instructions: every operand value is the sum of three bf16 values.
//
// v_mfma_f32_32x32x2_f32 executes 256 FLOP per cycle and SIMD, v_mfma_f32_32x32x16_bf16 sixteen times that.  An fp32
// value a is exactly a1 + a2 + a3 with a1 = bf16(a), a2 = bf16(a - a1), a3 = a - a1 - a2 (8 + 8 + 8 significand bits;
// bf16 has the exponent range of fp32, so nothing is scaled), the product of two bf16 values is exact in fp32, and of the
// nine products of a pair the three below 2^-24 of it (a2 b3, a3 b2, a3 b3) are left out: six MFMAs do the work of
// eight times 16 / 2 fp32 ones in 6/16 of their time.  Registers only, six products on random data: 302 TFLOP/s of fp32
// multiply-adds (1.81 PFLOP/s of bf16 at the clock it settles at) where the fp32 instruction reaches 154.
//
// Precision.  The five small products of a pair have accumulators of their own, added to the large product's behind the
// loop: one rounding at the size of the sum per 16 terms instead of one per two.  Relative error of chains of 256, 1152 and
// 3456 terms against 64 bits, N(0,1) data: 0.9e-7, 2.0e-7 and 3.6e-7, the fp32 instruction 2.9e-7, 6.1e-7 and 10.4e-7 (with
// one set of accumulators 2.4e-7, 5.2e-7 and 9.2e-7, and above the fp32 instruction where half of one operand is zero).
//
// Infinities.  The parts of an infinity are (inf, 0, 0), and inf * 0 makes a NaN where fp32 multiplication has none.  So a
// result that is not finite is computed again from the parts (whose sum is the operand), term by term in fp32.
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
struct TriPack8 {
  uint32_t w[3][4];
  float rest = 0.0f;
  __device__ __forceinline__ void pair(const float (&v)[8], int e) {
    float x = v[2 * e], y = v[2 * e + 1];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      w[i][e] = pack_bf16(x, y);
      x -= __builtin_bit_cast(float, w[i][e] << 16);
      y -= __builtin_bit_cast(float, w[i][e] & 0xffff0000u);
    }
    rest += x + y;   // zeros, or a NaN where a first part is no number
  }
  __device__ __forceinline__ void fix(const float (&v)[8]) {
    if (rest == 0.0f) return;
    // infinities and NaNs have no further parts; the largest floats, which round to an infinity, are cut off instead
#pragma unroll
    for (int e = 0; e < 4; ++e) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const float x = v[2 * e + h];
        const uint32_t bits = __builtin_bit_cast(uint32_t, x), mag = bits & 0x7fffffffu;
        if (mag <= 0x7f7f7fffu) continue;
        uint32_t p = bits >> 16, q = 0, r = 0;
        if (mag > 0x7f800000u) p |= 0x40u;
        if (mag < 0x7f800000u) {
          const float t = x - __builtin_bit_cast(float, p << 16);
          q = pack_bf16(t, 0.0f) & 0xffffu;
          r = pack_bf16(t - __builtin_bit_cast(float, q << 16), 0.0f) & 0xffffu;
        }
        const uint32_t keep = h ? 0xffffu : 0xffff0000u, sh = 16 * h;
        w[0][e] = (w[0][e] & keep) | (p << sh);
        w[1][e] = (w[1][e] & keep) | (q << sh);
        w[2][e] = (w[2][e] & keep) | (r << sh);
      }
    }
  }
  __device__ __forceinline__ uint4 part(int i) const { return make_uint4(w[i][0], w[i][1], w[i][2], w[i][3]); }
};
__device__ __forceinline__ void tri_pack8(const float (&v)[8], uint4 (&o)[3]) {
  TriPack8 t;
#pragma unroll
  for (int e = 0; e < 4; ++e) t.pair(v, e);
  t.fix(v);
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

// Element (row, col) over groups [g0, g1), from the operands' parts, in fp32.
template <bool B_LINEAR>
__device__ __forceinline__ float tri_dot(const TriParams& a, const TriParams& b, int row, int col, int g0, int g1) {
  auto base = [](const RowV8Params& p, int m) {
    const int n = m / p.inner, rem = m - n * p.inner, a2 = rem / p.innerW, b2 = rem - a2 * p.innerW;
    return static_cast<const char*>(p.ptr) + (uint32_t)(n * p.img_stride + a2 * p.a_stride + b2 * p.b_stride);
  };
  const char* pa = base(a.v, row);
  const char* pb = base(b.v, col);
  float sum = 0.0f;
  for (int g = g0; g < g1 && sum == sum; ++g) {   // (a NaN stays one)
    const uint16_t* qa = reinterpret_cast<const uint16_t*>(pa + g * a.v.group_stride);
    const uint16_t* qb = reinterpret_cast<const uint16_t*>(pb + (B_LINEAR ? g * b.v.group_stride : b.v.soff[g]));
    auto value = [](const uint16_t* q, int plane, int e) {
      auto part = [&](int i) { return __builtin_bit_cast(float, (uint32_t)q[(size_t)i * (plane / 2) + e] << 16); };
      return part(0) + (part(1) + part(2));   // (exact; the largest floats' first two parts add up to 2^128)
    };
    for (int e = 0; e < 8; ++e) sum = fmaf(value(qa, a.plane, e), value(qb, b.plane, e), sum);
  }
  return sum;
}

// A block's tile in a ring of R buffers of one K step each.  Step `it` of a wave: its operands are in registers (read a step
// ago); once all waves are there, buffer `it` is free and buffer it+1 complete; between its MFMAs, one to a slot, it reads
// the operands of step it+1 and issues the loads of step it+R into buffer `it`, which then have R - 1 steps to land.
// A wave is 64 x 64 of a 128 x 128 tile (128 accumulators in two sets, twice 48 registers of operands: two waves to a SIMD,
// two blocks to a CU): 12 operand reads of 1 KB for 24 MFMAs, half of what the LDS delivers, and 24 KB of fill, half of what
// the L2 does.
constexpr int kTriRing = 3;
constexpr int kTriLdsBytes = kTriRing * 6 * 16 * 256;

// K steps [s_begin, s_end) of the tile at (m0, n0).
template <class T, bool B_LINEAR, bool NCHW>
__device__ __forceinline__ void tri_block(const TriParams& ap, const TriParams& bp, const EpiParams& ep, int m0, int n0, int s_begin,
                                          int s_end, int groups, int dst_split) {
  constexpr int TM = T::TM, TN = T::TN, R = kTriRing, RA = (T::BM + 63) / 64 * 64, RBn = (T::BN + 63) / 64 * 64;
  static_assert(T::NT == 4 * kWave && T::BK == 16, "four waves, 16 k a step");
  static_assert(kTriLdsBytes >= TN * 16 * 4 * kWave * 4, "a row of blocks fits the ring");
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
    constexpr int PA[6] = {0, 2, 1, 0, 1, 0}, PB[6] = {2, 0, 1, 1, 0, 0};
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
    constexpr int kSlots = kReads + kLoads + 1, kMfma = 6 * TM * TN;
#pragma unroll
    for (int m = 0; m < kMfma; ++m) {
      const int p = m / (TM * TN), t = m % (TM * TN), i = t / TN, j = t % TN;
      f32x16& d = p == 5 ? acc[i][j] : low[i][j];
      d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a[c][PA[p]][i]),
                                                  __builtin_bit_cast(bf16x8_t, b[c][PB[p]][j]), d, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
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
  __syncthreads();   // the ring has been read for the last time
  if (__any(!(finite == 0.0f))) {
    float* const mine = lds_dyn + wave * (TN * 16 * kWave) + lane;   // [value][lane]
    const int g0 = 2 * s_begin, g1 = 2 * s_end < groups ? 2 * s_end : groups;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) mine[(j * 16 + v) * kWave] = acc[i][j][v];
#pragma unroll 1
      for (int e = 0; e < TN * 16; ++e) {
        const int v = e & 15, j = e >> 4;
        const int row = m0 + wm * (TM * 32) + i * 32 + (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3);
        const int col = n0 + wn * (TN * 32) + j * 32 + (lane & 31);
        if (!(fabsf(mine[e * kWave]) < INFINITY) && row < ep.rows && col < ep.cols)
          mine[e * kWave] = tri_dot<B_LINEAR>(ap, bp, row, col, g0, g1);
      }
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = mine[(j * 16 + v) * kWave];
    }
  }
  store_tile<T, NCHW>(acc, ep, m0, n0, wm, wn, lane, dst_split);
}

template <class T, bool B_LINEAR, bool NCHW, class PASS>
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
  tri_block<T, B_LINEAR, NCHW>(ap, bp, ep, m0, n0, s_begin, s_end, groups, dst_split);
}

// Backward-data of stride 2 to 4 (conv_common.h: residue classes): the classes' contractions in one launch, the longest first, so that
// the short ones fill the last round (launched one by one the classes of 64 -> 128 56x56 b24 are 98 tiles each on 256 CUs).  Bound by
// the MFMAs as above and by the classes' results, which a second pass interleaves.
struct TriClass {
  int first_tile, steps, groups_true;
  int cols, inner, innerW;   // n U V, U V, V
  uint32_t wt_at, img_at;    // bytes into the operand copies: the class's filter, its first pixel at its first tap
  int soff_at;
  long long out_at;          // floats
};
struct TriClasses { int count, tiles_m; TriClass c[16]; };
template <class T>
__global__ __launch_bounds__(T::NT, T::OCC) void mfma_gemm_tri_classes_kernel(TriParams ap, TriParams bp, EpiParams ep, TriClasses t) {
  const int block = blockIdx.x;
  int i = 0;
  while (i + 1 < t.count && block >= t.c[i + 1].first_tile) ++i;
  i = __builtin_amdgcn_readfirstlane(i);
  const TriClass c = t.c[i];
  const int tiles = (i + 1 < t.count ? t.c[i + 1].first_tile : (int)gridDim.x) - c.first_tile;
  const int logical = __builtin_amdgcn_readfirstlane(xcd_remap(block - c.first_tile, tiles));
  ap.v.ptr = static_cast<const char*>(ap.v.ptr) + c.wt_at;
  ap.plane = c.steps * 2 * ap.v.M * 16;
  ap.v.bytes = (uint32_t)(3 * ap.plane);
  bp.v.ptr = static_cast<const char*>(bp.v.ptr) + c.img_at;
  bp.v.bytes -= c.img_at;
  bp.v.M = c.cols; bp.v.inner = c.inner; bp.v.innerW = c.innerW;
  bp.v.soff += c.soff_at;
  ep.out += c.out_at;
  ep.cols = c.cols; ep.inner = c.inner;
  tri_block<T, false, true>(ap, bp, ep, logical % t.tiles_m * T::BM, logical / t.tiles_m * T::BN, 0, c.steps, c.groups_true, -1);
}

}  // namespace rh

// Column-major SGEMM on the bf16 matrix instructions with exactly split operands (gemm_tri.h), for the products of large affine
// layers.  As in sgemm.hip D[jn][im] = sum_l opB(l, jn) * opA(im, l): rows jn, columns im.
//
//   forward (A transposed) and data gradient (neither): A is the weights, far the larger operand and read once.  A split copy of
//     it would cost 10 bytes a value where the product reads 4, so the kernel below brings it to LDS as it lies and splits it in
//     registers; B, the activations or deltas of a batch, gets a split copy in front (a launch of 3 to 6 us).
//   filter gradient (B transposed): both operands are of batch size and the result is the large tensor: split copies of both, and
//     the kernel of the convolutions.
#include "conv_common.h"
#include "gemm_tri.h"
#include "sgemm_tri.h"

namespace rh {

// A dense operand into [k/8][row][8] in three parts, groups past the last k as zeros.
struct TriDenseArgs {
  const float* src; uint4* dst;
  int rows, K, groups;
  long long sk, sr;   // floats from a k and from a row to the next
  int vec;            // k contiguous, whole groups, 16-byte aligned
};
__device__ __forceinline__ void tri_dense_body(const TriDenseArgs& a, long long i) {
  const long long total = (long long)a.groups * a.rows;
  if (i >= total) return;
  const int g = (int)(i / a.rows), row = (int)(i - (long long)g * a.rows);
  const float* src = a.src + (long long)g * 8 * a.sk + row * a.sr;
  float v[8];
  if (a.vec && g * 8 < a.K) {
    const float4 lo = reinterpret_cast<const float4*>(src)[0], hi = reinterpret_cast<const float4*>(src)[1];
    v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w;
    v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = g * 8 + e < a.K ? src[e * a.sk] : 0.0f;
  }
  uint4 o[3];
  tri_pack8(v, o);
#pragma unroll
  for (int p = 0; p < 3; ++p) a.dst[i + p * total] = o[p];
}
__global__ __launch_bounds__(256) void tri_dense_kernel(TriDenseArgs a, TriDenseArgs b, int a_blocks) {
  if ((int)blockIdx.x < a_blocks) tri_dense_body(a, (long long)blockIdx.x * 256 + threadIdx.x);
  else tri_dense_body(b, (long long)(blockIdx.x - a_blocks) * 256 + threadIdx.x);
}

// 32 TM rows x 128 columns a block, 32 TM x 32 a wave, one K step (16 k) a ring buffer: the rows' parts, shared by the waves, and
// the wave's own columns as fp32 values.  Step `it` of a wave: its column parts and its first row block are in registers;
// between its MFMAs it reads the next row block and the columns of step it+1, and splits those, a pair of values to a slot (a
// wave splits 8 values a lane and step, 17 VALU instructions a pair, against 6 TM MFMAs of 32 cycles).
// Two blocks to a CU: at 128 rows the MFMAs bound it as in the convolutions' kernel, at 64 and 32 the reading of the weights.
// 9216 -> 4096 forward, whole calls: 256 images 164 -> 112 us (172 TFLOP/s of fp32 multiply-adds), 37 images 63 -> 38 us (4 TB/s of
// weights, the split copy and the slices' reduction included), 8 images 40 -> 33 us.
template <class T> struct TriStream {
  static constexpr int RA = T::BM, A_UNITS = 6 * RA / 64, NA = (A_UNITS + 3) / 4, CNT = NA + 2;
  static constexpr int A_PIECES = 6 * RA, PIECES = A_PIECES + 4 * 128;
  static constexpr int R = 80 * 1024 / (16 * PIECES);   // 4, 5 and 7 steps
  static constexpr int LDS = R * PIECES * 16;
};

template <class T, bool K_CONTIG>
__global__ __launch_bounds__(T::NT, T::OCC) void mfma_gemm_tri_stream_kernel(TriParams ap, DenseParams rows32, DenseParams bp, EpiParams ep,
                                                                             int tiles_m, int k_steps, int steps_per_split) {
  typedef TriStream<T> S;
  constexpr int TM = T::TM, RA = S::RA, R = S::R, CNT = S::CNT;
  static_assert(T::TN == 1 && T::WM == 1 && T::WN == 4 && T::BK == 16 && R >= 4 && (TM == 1 || TM % 2 == 0), "block shape");
  extern __shared__ float lds_dyn[];
  uint4* const sm = reinterpret_cast<uint4*>(lds_dyn);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)sm;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  // row tiles fastest: blocks that read the same weights follow one another on an XCD
  const int tiles = gridDim.x;
  const int linear = xcd_remap(blockIdx.y * tiles + blockIdx.x, tiles * gridDim.y);
  const int slice = __builtin_amdgcn_readfirstlane(linear / tiles);
  const int logical = __builtin_amdgcn_readfirstlane(linear - slice * tiles);
  const int m0 = logical % tiles_m * T::BM, n0 = logical / tiles_m * T::BN;
  const int s_begin = slice * steps_per_split;
  const int s_end = s_begin + steps_per_split < k_steps ? s_begin + steps_per_split : k_steps;
  const int nk = s_end - s_begin;

  auto rsrc_of = [](const void* ptr, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(ptr);
    u32x4 r;
    r.x = __builtin_amdgcn_readfirstlane((uint32_t)a);
    r.y = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32) & 0xffffu);
    r.z = __builtin_amdgcn_readfirstlane(bytes);
    r.w = 0x00020000u;
    return r;
  };
  const u32x4 ra = rsrc_of(ap.v.ptr, ap.v.bytes), rb = rsrc_of(bp.ptr, bp.bytes);
  // pieces of 16 bytes, 64 to a load; the waves past the last unit of rows bring it again (the same bytes to the same place)
  uint32_t va[S::NA], la[S::NA], vb[2];
#pragma unroll
  for (int i = 0; i < S::NA; ++i) {
    const int u = wave + 4 * i < S::A_UNITS ? wave + 4 * i : S::A_UNITS - 1;
    const int x = u * 64 + lane, part = x / (2 * RA), grp = x / RA & 1, row = m0 + x % RA;
    va[i] = row < ap.v.M ? (uint32_t)(part * ap.plane + grp * ap.v.group_stride + row * 16) : 0x80000000u;
    la[i] = (uint32_t)u * 1024u;
  }
  const uint32_t lb = (uint32_t)(S::A_PIECES + wave * 128) * 16u;
  const uint32_t bstep = K_CONTIG ? 64u : 64u * (uint32_t)bp.ld;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    if (K_CONTIG) {   // column r's quarter q of 16 k at piece 4 r + (q ^ r / 4 % 4): a read of 64 pieces touches all banks alike
      const int r = u * 16 + (lane >> 2), q = (lane & 3) ^ (r >> 2 & 3), col = n0 + wave * 32 + r;
      vb[u] = col < bp.rows ? 4u * ((uint32_t)col * (uint32_t)bp.ld + (uint32_t)(s_begin * 16 + q * 4)) : 0x80000000u;
    } else {          // [k][32 columns]; the k past the last lie outside the buffer's range
      const int k = s_begin * 16 + u * 8 + (lane >> 3), col = n0 + wave * 32 + (lane & 7) * 4;
      vb[u] = col < bp.rows ? 4u * ((uint32_t)k * (uint32_t)bp.ld + (uint32_t)col) : 0x80000000u;
    }
  }
  // step s (of this block) into the buffer at `base`; the steps are issued in order
  auto issue = [&](uint32_t base, int s, int i) {
    if (i < 2) {
      dma_load16(rb, base + lb + (uint32_t)i * 1024u, vb[i], 0u);
      if (K_CONTIG || vb[i] < 0x80000000u) vb[i] += bstep;
    } else {
      dma_load16(ra, base + la[i - 2], va[i - 2], (uint32_t)((s_begin + s) * 2 * ap.v.group_stride));
    }
  };

  f32x16 acc[TM][1], low[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[i][0][v] = low[i][v] = 0.0f;

#pragma unroll
  for (int s = 0; s < R - 1; ++s)
    if (s < nk) {
#pragma unroll
      for (int i = 0; i < CNT; ++i) issue(lds0 + (uint32_t)(s * S::PIECES) * 16u, s, i);
    }
  wait_vmcnt<0>();
  __syncthreads();

  uint4 a[2][3], b[2][3];
  float raw[8];
  auto read_a = [&](int buf, int i, uint4 (&d)[3]) {
    const uint4* p = sm + buf * S::PIECES + (lane >> 5) * RA + i * 32 + (lane & 31);
#pragma unroll
    for (int q = 0; q < 3; ++q) d[q] = p[q * 2 * RA];
  };
  auto read_b = [&](int buf) {
    const uint4* p = sm + buf * S::PIECES + S::A_PIECES + wave * 128;
    const int r = lane & 31, h = lane >> 5;
    if (K_CONTIG) {
      const float4* f = reinterpret_cast<const float4*>(p) + r * 4;
      const float4 lo = f[(2 * h) ^ (r >> 2 & 3)], hi = f[(2 * h + 1) ^ (r >> 2 & 3)];
      raw[0] = lo.x; raw[1] = lo.y; raw[2] = lo.z; raw[3] = lo.w;
      raw[4] = hi.x; raw[5] = hi.y; raw[6] = hi.z; raw[7] = hi.w;
    } else {
      const float* f = reinterpret_cast<const float*>(p) + h * 8 * 32 + r;
#pragma unroll
      for (int e = 0; e < 8; ++e) raw[e] = f[e * 32];
    }
  };
  read_b(0);
  tri_pack8(raw, b[0]);
  read_a(0, 0, a[0]);

  int rd = 0;   // buffer of the current step
  auto step = [&](int it, auto c_tag, auto more_tag) {
    constexpr int c = decltype(c_tag)::value;
    constexpr bool MORE = decltype(more_tag)::value;   // this step issues the loads of step it+R-1
    if (MORE) wait_vmcnt<(R - 3) * CNT>();             // step it+1 is there, this wave's share of it
    else wait_vmcnt<0>();
    __syncthreads();                                   // all of it, and step it-1 has been read
    const int nx = rd + 1 == R ? 0 : rd + 1;
    const uint32_t base = lds0 + (uint32_t)((rd == 0 ? R - 1 : rd - 1) * S::PIECES) * 16u;
    TriPack8 t;
    constexpr int kMfma = 6 * TM, kFirst = kMfma / 3;
    constexpr int PA[6] = {0, 2, 1, 0, 1, 0}, PB[6] = {2, 0, 1, 1, 0, 0};
    int pairs = 0, loads = 0;
#pragma unroll
    for (int m = 0; m < kMfma; ++m) {
      const int i = m / 6, p = m % 6, par = TM == 1 ? c : i & 1;
      if (p == 0) {
        if (m == 0) read_b(nx);
        if (i + 1 < TM) read_a(rd, i + 1, a[par ^ 1]);
        else read_a(nx, 0, a[par ^ 1]);
      }
      f32x16& d = p == 5 ? acc[i][0] : low[i];
      d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a[par][PA[p]]), __builtin_bit_cast(bf16x8_t, b[c][PB[p]]),
                                                  d, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      for (; MORE && loads < CNT && loads < (m + 1) * CNT / kFirst; ++loads) issue(base, it + R - 1, loads);
      for (; m >= kFirst && pairs < 4 && pairs < (m + 1 - kFirst) * 4 / (kMfma - kFirst); ++pairs) t.pair(raw, pairs);
      __builtin_amdgcn_sched_barrier(0);
    }
    t.fix(raw);
#pragma unroll
    for (int q = 0; q < 3; ++q) b[c ^ 1][q] = t.part(q);
    rd = nx;
  };
  const std::integral_constant<int, 0> c0;
  const std::integral_constant<int, 1> c1;
  int it = 0;
  for (; it + R < nk; it += 2) {
    step(it, c0, std::true_type());
    step(it + 1, c1, std::true_type());
  }
  if (it + R - 1 < nk) {
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
  for (int i = 0; i < TM; ++i) {
    acc[i][0] += low[i];
#pragma unroll
    for (int v = 0; v < 16; ++v) finite = fmaf(acc[i][0][v], 0.0f, finite);
  }
  if (__any(!(finite == 0.0f))) {   // as in tri_block, from the operands themselves
    const int col0 = n0 + wave * 32, col = col0 + (lane & 31) < bp.rows ? col0 + (lane & 31) : 0;
    const float* const pb = bp.ptr + (K_CONTIG ? (size_t)col * bp.ld : (size_t)col);
    const int k1 = s_end * 16 < bp.K ? s_end * 16 : bp.K;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int row0 = m0 + i * 32, row = row0 + (lane & 31) < rows32.rows ? row0 + (lane & 31) : 0;
      const float* const pa = rows32.ptr + (size_t)row * rows32.ld;
      auto load = [&](const float* p, size_t step, int g, float (&v)[8]) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (g * 8 + e < k1) v[e] = p[(size_t)(g * 8 + e) * step];
      };
      tri_redo(acc[i][0], ep.rows - row0, ep.cols - col0, lane, s_begin * 2, (k1 + 7) / 8,
               [&](int g, float (&v)[8]) { load(pa, 1, g, v); },
               [&](int g, float (&v)[8]) { load(pb, K_CONTIG ? 1 : (size_t)bp.ld, g, v); });
    }
  }
  store_tile<T, false>(acc, ep, m0, n0, 0, wave, lane, ep.split_stride != 0 ? slice : -1);
}

typedef Tile<128, 128, 16, 1, 4, 2> T128x128s;
typedef Tile<64, 128, 16, 1, 4, 2> T64x128s;
typedef Tile<32, 128, 16, 1, 4, 2> T32x128s;

SgemmTriPlan plan_sgemm_tri(bool a_trans, bool b_trans, int m, int n, int k) {
  SgemmTriPlan p = {};
  if ((a_trans && b_trans) || m <= 0 || n <= 0 || k <= 0 || m % 4 != 0 || (a_trans && k % 16 != 0)) return p;
  p.groups = round_up(cdiv(k, 8), 2);
  const int steps = p.groups / 2;
  const size_t rows_bytes = 48 * (size_t)p.groups * n, cols_bytes = b_trans ? 48 * (size_t)p.groups * m : 0;
  if (rows_bytes > kMaxBufferBytes || cols_bytes > kMaxBufferBytes) return p;
  p.rows_bytes = align256(rows_bytes);
  p.cols_bytes = align256(cols_bytes);
  p.bm = b_trans || n > 64 ? 128 : n > 32 ? 64 : 32;
  const long long tiles = (long long)cdiv(n, p.bm) * cdiv(m, 128);
  const double out_mb = 4e-6 * (double)m * (double)n, w_mb = b_trans ? 0.0 : 4e-6 * (double)m * (double)k * cdiv(n, p.bm);
  // slices: the longer of the MFMAs (as in plan_tri) and the weights' bytes at the rate of a copy, for which two blocks have to be
  // on a CU, and behind it their sums
  p.splits = 1;
  double best = 1e30;
  for (int want = 1; want <= 64 && (want == 1 || (!b_trans && want * 8 <= steps && tiles * want <= 1024)); ++want) {
    const int len = cdiv(steps, want), S = cdiv(steps, len);
    if (S != want) continue;
    const long long each = cdiv<long long>(tiles * S, 256);
    const double mfma = (each == 1 ? 0.415 : 0.456 * (double)each) * len * p.bm / 128.0;
    const double mem = w_mb / 4.7 * (tiles * S < 512 ? 512.0 / (double)(tiles * S) : 1.0);
    const double us = fmax(mfma, mem) + (S > 1 ? 4.0 + out_mb * (2 * S + 1) / 5.0 : out_mb / 4.2);
    if (us < best) { best = us; p.splits = S; }
  }
  p.part_bytes = p.splits > 1 ? align256(sizeof(float) * (size_t)p.splits * m * n) : 0;
  p.ok = true;
  return p;
}

template <class T, bool K_CONTIG>
static int launch_stream(const TriParams& ap, const DenseParams& rows32, const DenseParams& bp, const EpiParams& ep, int steps, int splits,
                         int* used, double flops, hipStream_t stream, const char* tag) {
  const int tiles_m = cdiv(ep.rows, T::BM), tiles_n = cdiv(ep.cols, T::BN), sps = cdiv(steps, splits);
  *used = cdiv(steps, sps);
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&mfma_gemm_tri_stream_kernel<T, K_CONTIG>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, TriStream<T>::LDS);
  if (attr != hipSuccess) return (int)attr;
  ProfScope prof(tag, flops, stream);
  hipLaunchKernelGGL((mfma_gemm_tri_stream_kernel<T, K_CONTIG>), dim3((unsigned)(tiles_m * tiles_n), (unsigned)*used), dim3(T::NT),
                     TriStream<T>::LDS, stream, ap, rows32, bp, ep, tiles_m, steps, sps);
  return launch_status();
}

int launch_sgemm_tri(const SgemmTriPlan& p, bool a_trans, bool b_trans, const DenseParams& rows, const DenseParams& cols, EpiParams ep,
                     void* ws, hipStream_t stream, int* used) {
  char* base = static_cast<char*>(ws);
  const int k = rows.K, n = rows.rows, m = cols.rows, steps = p.groups / 2;
  auto dense = [&](const DenseParams& d, bool rows_contiguous, char* dst) {
    TriDenseArgs a;
    a.src = d.ptr; a.dst = reinterpret_cast<uint4*>(dst); a.rows = d.rows; a.K = k; a.groups = p.groups;
    a.sk = rows_contiguous ? d.ld : 1; a.sr = rows_contiguous ? 1 : d.ld;
    a.vec = !rows_contiguous && k % 8 == 0 && d.ld % 4 == 0 && (reinterpret_cast<uintptr_t>(d.ptr) & 15) == 0;
    return a;
  };
  auto packed = [&](int count, char* at) {
    TriParams t;
    t.v.ptr = at; t.v.bytes = (uint32_t)(48 * (size_t)p.groups * count); t.v.M = count; t.v.inner = 1; t.v.innerW = 1;
    t.v.img_stride = 16; t.v.a_stride = 0; t.v.b_stride = 0; t.v.soff = nullptr; t.v.group_stride = count * 16;
    t.plane = (int)(16 * (size_t)p.groups * count);
    return t;
  };
  const TriDenseArgs da = dense(rows, b_trans, base), db = b_trans ? dense(cols, true, base + p.rows_bytes) : da;
  const unsigned a_blocks = (unsigned)cdiv<long long>((long long)p.groups * n, 256);
  const unsigned b_blocks = b_trans ? (unsigned)cdiv<long long>((long long)p.groups * m, 256) : 0;
  {
    ProfScope prof("tri_dense", 80.0 * (double)p.groups * (n + (b_trans ? m : 0)), stream);
    hipLaunchKernelGGL(tri_dense_kernel, dim3(a_blocks + b_blocks), dim3(256), 0, stream, da, db, (int)a_blocks);
  }
  if (int e = launch_status()) return e;
  const double flops = 12.0 * (double)m * n * k;
  const TriParams ap = packed(n, base);
  if (b_trans) {
    typedef Tile<128, 128, 16, 2, 2, 2> T;
    const TriParams bp = packed(m, base + p.rows_bytes);
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&mfma_gemm_tri_kernel<T, true, false, PassSgemm>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, kTriLdsBytes);
    if (attr != hipSuccess) return (int)attr;
    *used = 1;
    ProfScope prof("sgemm_tri_128x128", flops, stream);
    hipLaunchKernelGGL((mfma_gemm_tri_kernel<T, true, false, PassSgemm>), dim3((unsigned)(cdiv(n, T::BM) * cdiv(m, T::BN))), dim3(T::NT),
                       kTriLdsBytes, stream, ap, bp, ep, cdiv(n, T::BM), steps, steps, p.groups);
    return launch_status();
  }
#define RH_STREAM(TILE, TAG)                                                                                          \
  (a_trans ? launch_stream<TILE, true>(ap, rows, cols, ep, steps, p.splits, used, flops, stream, "sgemm_tri_stream_" TAG) \
           : launch_stream<TILE, false>(ap, rows, cols, ep, steps, p.splits, used, flops, stream, "sgemm_tri_stream_" TAG))
  switch (p.bm) {
    case 128: return RH_STREAM(T128x128s, "128x128");
    case 64: return RH_STREAM(T64x128s, "64x128");
    default: return RH_STREAM(T32x128s, "32x128");
  }
#undef RH_STREAM
}

}  // namespace rh

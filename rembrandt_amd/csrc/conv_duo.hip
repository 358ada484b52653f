// fp32 convolutions on the fp16 matrix instructions with operands of two scaled parts (gemm_duo.h): forward, stride-1
// backward-data and backward-filter.
//
// Three launches in front of the reduction of slices: the largest magnitudes (and the filters' ratios), the operand copies in two fp16 parts (4
// bytes a value, in the orders of conv_tri.hip), the contraction; in the filter gradient a fourth before the contraction, which copies in
// three parts where a value asks for them (TriRest).  The exponents are the filter's by row and the image's by image, and in the filter
// gradient both operands' by channel.
#include "conv_common.h"
#include "gemm_duo.h"

namespace rh {

// The largest finite magnitude of each row r of a tensor [O][R][I], in `parts` parts of the O I values of a row, part[r][parts].  Bound by
// its reads: a block has eight loads a thread in flight.
struct DuoMaxJob {
  const float* src; float* part;
  int* zero; int zeros;        // with the first block: counts to begin with
  int R, parts, blocks, vec;   // vec: by four values, I a multiple of 4 and src 16-byte aligned
  unsigned I, total, len;      // of a row, in units of four values where vec: I, O I and those of a part
  FastDiv dI;
};
static DuoMaxJob duo_max_job(const float* src, float* part, int O, int R, int I, int parts, int* zero = nullptr, int zeros = 0) {
  DuoMaxJob j;
  j.zero = zero; j.zeros = zeros;
  j.src = src; j.part = part; j.R = R; j.parts = parts; j.blocks = R * parts;
  j.vec = I % 4 == 0 && (reinterpret_cast<uintptr_t>(src) & 15) == 0;
  j.I = (unsigned)(j.vec ? I / 4 : I);
  j.total = (unsigned)O * j.I;
  j.len = cdiv(j.total, (unsigned)parts);
  j.dI = FastDiv(j.I);
  return j;
}
template <class V>
__device__ __forceinline__ uint32_t duo_max_range(const DuoMaxJob& j, int r, unsigned f0, unsigned f1) {
  const V* const src = reinterpret_cast<const V*>(j.src);
  uint32_t top = 0;
  for (unsigned f = f0 + threadIdx.x; f < f1; f += 256 * 8) {
    V v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const unsigned at = f + 256 * u;
      uint32_t o, i;
      j.dI.divmod(at < f1 ? at : f, o, i);
      v[u] = src[((size_t)o * j.R + r) * j.I + i];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (unsigned c = 0; c < sizeof(V) / 4; ++c) {
        const uint32_t bits = __builtin_bit_cast(uint32_t, reinterpret_cast<const float*>(&v[u])[c]) & 0x7fffffffu;
        if (bits < 0x7f800000u && bits > top) top = bits;
      }
  }
  return top;
}
__device__ __forceinline__ void duo_max_body(const DuoMaxJob& j, int b, uint32_t (&wave_top)[4]) {
  const int r = b / j.parts, q = b - r * j.parts;
  if (b == 0)
    for (int i = threadIdx.x; i < j.zeros; i += 256) j.zero[i] = 0;
  const unsigned f0 = (unsigned)q * j.len, f1 = f0 + j.len < j.total ? f0 + j.len : j.total;
  uint32_t top = j.vec ? duo_max_range<float4>(j, r, f0, f1) : duo_max_range<float>(j, r, f0, f1);
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    const uint32_t other = __shfl_xor(top, d);
    top = other > top ? other : top;
  }
  if ((threadIdx.x & 63) == 0) wave_top[threadIdx.x >> 6] = top;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < 4; ++w) top = wave_top[w] > top ? wave_top[w] : top;
    j.part[b] = __builtin_bit_cast(float, top);
  }
}
// For each group of eight channels of a filter tensor (Ck / 8 of them) the least ratio, over rows and taps, of a value to the largest of
// its eight (0: a zero beside others), in kDuoRatioParts parts.
constexpr int kDuoRatioParts = 8;
struct DuoRatioJob {
  const float* w; float* part;
  int rows, Ck, RS, bwd;
  FastDiv dRS;
};
__device__ __forceinline__ void duo_ratio_body(const DuoRatioJob& j, int b, uint32_t (&wave_least)[4]) {
  const int cg = b / kDuoRatioParts, q = b - cg * kDuoRatioParts;
  float least = 1.0f;
  for (unsigned i = (unsigned)q * 256 + threadIdx.x; i < (unsigned)j.rows * (unsigned)j.RS; i += kDuoRatioParts * 256) {
    uint32_t row, rs;
    j.dRS.divmod(i, row, rs);
    const float* const w = j.bwd ? j.w + ((size_t)cg * 8 * j.rows + row) * j.RS + rs : j.w + ((size_t)row * j.Ck + cg * 8) * j.RS + rs;
    const size_t stride = j.bwd ? (size_t)j.rows * j.RS : (size_t)j.RS;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = fabsf(w[e * stride]);
    float lo = v[0], hi = v[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) { lo = fminf(lo, v[e]); hi = fmaxf(hi, v[e]); }
    if (hi > 0.0f) least = fminf(least, lo / hi);
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) least = fminf(least, __shfl_xor(least, d));
  if ((threadIdx.x & 63) == 0) wave_least[threadIdx.x >> 6] = __builtin_bit_cast(uint32_t, least);
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < 4; ++w) least = fminf(least, __builtin_bit_cast(float, wave_least[w]));
    j.part[b] = least;
  }
}
__global__ __launch_bounds__(256) void duo_max_kernel(DuoMaxJob a, DuoMaxJob b, DuoRatioJob c) {
  __shared__ uint32_t wave_top[4];
  const int at = (int)blockIdx.x - a.blocks;
  if (at < 0) duo_max_body(a, blockIdx.x, wave_top);
  else if (at < b.blocks) duo_max_body(b, at, wave_top);
  else duo_ratio_body(c, at - b.blocks, wave_top);
}

template <class MARK>
__device__ __forceinline__ int duo_store(uint4* dst, size_t at, size_t plane, const float (&v)[8], int e, MARK mark) {
  uint4 o[2];
  const int lost = duo_pack8(v, e, mark, o);
#pragma unroll
  for (int p = 0; p < 2; ++p) dst[at + p * plane] = o[p];
  return lost;
}

// Filter copy, its rows' exponents and the table of the image's group offsets; tri_filter_body's items and order.
struct DuoFilterArgs {
  const float* w; uint4* wt; int* soff;
  const float* top; int *exps, *lost;   // of a row
  int groups, groups_true, rows, Ck, RS, S, Wp, bwd;
};
__device__ __forceinline__ void duo_filter_body(const DuoFilterArgs& a, long long i) {
  const long long total = (long long)a.groups * a.rows;
  if (i >= total) return;
  const int g = (int)(i / a.rows), row = (int)(i - (long long)g * a.rows);
  const int pairs = a.Ck / 16 * a.RS, step = g >> 1;
  int rs, c0;
  if (step < pairs) {
    rs = step % a.RS;
    c0 = step / a.RS * 16 + (g & 1) * 8;
  } else {
    rs = g - 2 * pairs;
    c0 = a.Ck - 8;
  }
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    v[e] = 0.0f;
    if (g < a.groups_true)
      v[e] = a.bwd ? a.w[((size_t)(c0 + e) * a.rows + row) * a.RS + (a.RS - 1 - rs)] : a.w[((size_t)row * a.Ck + c0 + e) * a.RS + rs];
  }
  const int e = duo_exponent(a.top[row]);
  const int lost = duo_store(a.wt, (size_t)i, (size_t)total, v, e, [](float, int) { return false; });
  if (lost > 0) atomicAdd(a.lost + row, lost);
  if (g == 0) a.exps[row] = e;
  if (row == 0) {
    const int r = rs / a.S, s2 = rs - r * a.S;
    a.soff[g] = g < a.groups_true ? ((r * (a.Ck / 8) + c0 / 8) * a.Wp + s2) * 16 : 0;
  }
}

// x [n][C][H][W] -> [n][Hp][C/8][Wp][8], a thread per group, the images' exponents from `parts` maxima each, and behind it the
// filter copy.
__global__ __launch_bounds__(256) void duo_image_kernel(const float* __restrict__ x, uint4* __restrict__ xt, unsigned total, int H,
                                                        int W, FastDiv dWp, FastDiv dCg, FastDiv dHp, int halo, int img_blocks,
                                                        const float4* __restrict__ top, int parts, int* __restrict__ exps,
                                                        const float4* __restrict__ ratio, DuoFilterArgs f) {
  if ((int)blockIdx.x >= img_blocks) {
    duo_filter_body(f, (long long)(blockIdx.x - img_blocks) * 256 + threadIdx.x);
    return;
  }
  const unsigned i = (unsigned)xcd_remap(blockIdx.x, img_blocks) * 256u + threadIdx.x;
  if (i >= total) return;
  uint32_t t, wp, cg, hp, n;
  dWp.divmod(i, t, wp);
  dCg.divmod(t, t, cg);
  dHp.divmod(t, n, hp);
  const int h = (int)hp - halo, wc = (int)wp - halo;
  float v[8];
  if ((unsigned)h < (unsigned)H && (unsigned)wc < (unsigned)W) {
    const size_t plane = (size_t)H * W;
    const float* src = x + ((size_t)n * dCg.div * 8 + cg * 8) * plane + (size_t)h * W + wc;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = src[e * plane];
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 0.0f;
  }
  float m = 0.0f;
  const float4* const tn = top + (size_t)n * (parts / 4);
  for (int q = 0; q < parts / 4; ++q) {
    const float4 p = tn[q];
    m = fmaxf(m, fmaxf(fmaxf(p.x, p.y), fmaxf(p.z, p.w)));
  }
  const int e = duo_exponent(m);
  duo_store(xt, i, total, v, e, [&](float most, int n) {
    const float4* const r = ratio + (size_t)cg * (kDuoRatioParts / 4);
    float least = 1.0f;
#pragma unroll
    for (int q = 0; q < kDuoRatioParts / 4; ++q) least = fminf(least, fminf(fminf(r[q].x, r[q].y), fminf(r[q].z, r[q].w)));
    return !(most * least >= (float)n * kDuoBeside);
  });
  if (wp == 0 && cg == 0 && hp == 0) exps[n] = e;
}

// x [N][C][H][W] -> [n/8][Hp][Wp][C][8 n], as tri_batch_body: a block moves 32 pixels x 32 channels of eight images through LDS, and
// may leave the sums of its pixels and images for the bias gradient.
constexpr int kDuoPix = 32, kDuoCh = 32;
struct DuoBatchArgs {
  const float* x; uint4* xt;
  const float* top; int parts;   // [C][parts]
  int* exps;
  int* any;                      // set where a value has too few bits: it is marked, and TriRest's form may take over
  int N, C, H, W, halo, HpWp;
  FastDiv dWp;
  size_t plane;
  int px, cx, blocks;
  float* sums;
};
__device__ __forceinline__ void duo_batch_body(const DuoBatchArgs& a, int b, float (&tile)[8][kDuoCh][kDuoPix + 1], float (&tops)[8][kDuoCh]) {
  const int bx = b % a.px, t = b / a.px, by = t % a.cx, bz = t / a.cx;
  const int pix0 = bx * kDuoPix, c0 = by * kDuoCh, n0 = bz * 8;
  {
    const int pl = threadIdx.x & 31, pix = pix0 + pl;
    uint32_t hp, wp;
    a.dWp.divmod((uint32_t)pix, hp, wp);
    const int h = (int)hp - a.halo, w = (int)wp - a.halo;
    const bool in = pix < a.HpWp && (unsigned)h < (unsigned)a.H && (unsigned)w < (unsigned)a.W;
    const size_t hw = (size_t)a.H * a.W;
    const float* src = a.x + (size_t)(in ? h * a.W + w : 0);
    const int c_first = threadIdx.x >> 5;
    float v[8][kDuoCh / 8];
#pragma unroll
    for (int n = 0; n < 8; ++n)
#pragma unroll
      for (int i = 0; i < kDuoCh / 8; ++i) {
        const int c = c0 + c_first + 8 * i;
        v[n][i] = in && c < a.C && n0 + n < a.N ? src[((size_t)(n0 + n) * a.C + c) * hw] : 0.0f;
      }
    float m = 0.0f;
    const int cm = c0 + (threadIdx.x & 31);
    if (cm < a.C)
      for (int q = threadIdx.x >> 5; q < a.parts; q += 8) m = fmaxf(m, a.top[(size_t)cm * a.parts + q]);
    tops[threadIdx.x >> 5][threadIdx.x & 31] = m;
#pragma unroll
    for (int n = 0; n < 8; ++n)
#pragma unroll
      for (int i = 0; i < kDuoCh / 8; ++i) tile[n][c_first + 8 * i][pl] = v[n][i];
  }
  __syncthreads();
  const int cl = threadIdx.x & 31, c = c0 + cl;
  float m = 0.0f;
#pragma unroll
  for (int q = 0; q < 8; ++q) m = fmaxf(m, tops[q][cl]);
  const int ex = duo_exponent(m);
  if (bx == 0 && bz == 0 && threadIdx.x < kDuoCh && c < a.C) a.exps[c] = ex;
  float sum = 0.0f;
  int lost = 0;
#pragma unroll
  for (int i = 0; i < kDuoPix / 8; ++i) {
    const int pl = (threadIdx.x >> 5) + 8 * i, pix = pix0 + pl;
    float v[8];
#pragma unroll
    for (int n = 0; n < 8; ++n) v[n] = tile[n][cl][pl];
    if (a.sums) sum += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    if (pix < a.HpWp && c < a.C) lost |= duo_store(a.xt, ((size_t)bz * a.HpWp + pix) * a.C + c, a.plane, v, ex, [](float, int) { return true; });
  }
  if (lost != 0) *a.any = 1;
  if (a.sums) {
    __syncthreads();
    float* const part = &tile[0][0][0];
    part[threadIdx.x] = sum;
    __syncthreads();
    if (threadIdx.x < kDuoCh && c < a.C) {
      float s = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) s += part[i * 32 + cl];
      a.sums[((size_t)bz * a.px + bx) * a.C + c] = s;
    }
  }
}

// Both operands of a filter gradient and soff[g], the place of group g = (n/8, p, q) in x's copy; the groups past the last
// are zeros of dy.
__global__ __launch_bounds__(256) void duo_batch_kernel(DuoBatchArgs dy, DuoBatchArgs x, int* __restrict__ soff, int groups,
                                                        int groups_true, int PQ, int Q, int st, int Wp) {
  __shared__ float tile[8][kDuoCh][kDuoPix + 1];
  __shared__ float tops[8][kDuoCh];
  int b = blockIdx.x;
  if (b < dy.blocks) { duo_batch_body(dy, xcd_remap(b, dy.blocks), tile, tops); return; }
  b -= dy.blocks;
  if (b < x.blocks) { duo_batch_body(x, xcd_remap(b, x.blocks), tile, tops); return; }
  b -= x.blocks;
  if (groups > groups_true)   // (one group: every block of the table writes a share)
    for (int i = b * 256 + threadIdx.x; i < 2 * dy.C; i += (int)(gridDim.x - dy.blocks - x.blocks) * 256)
      dy.xt[(size_t)(i / dy.C) * dy.plane + (size_t)groups_true * dy.C + i % dy.C] = make_uint4(0, 0, 0, 0);
  const int g = b * 256 + threadIdx.x;
  if (g >= groups) return;
  int off = 0;
  if (g < groups_true) {
    const int n8 = g / PQ, pq = g - n8 * PQ, p = pq / Q, q = pq - p * Q;
    off = (n8 * x.HpWp + p * st * Wp + q * st) * x.C * 16;
  }
  soff[g] = off;
}

template <class T, bool NCHW, class PASS>
static int launch_duo(const DuoParams& ap, const DuoParams& bp, const DuoSource& src, const EpiParams& ep, int k_steps, int groups,
                      int splits, int* used, double flops, hipStream_t stream, const char* tag, const TriRest& rest = TriRest{}) {
  const int tiles_m = cdiv(ep.rows, T::BM), tiles_n = cdiv(ep.cols, T::BN);
  if (ep.tail_tiles > 0) splits = ep.tail_splits;
  const int sps = cdiv(k_steps, splits < 1 ? 1 : splits);
  const int n_split = cdiv(k_steps, sps);
  if (used) *used = n_split;
  dim3 grid((unsigned)(tiles_m * tiles_n), (unsigned)n_split);
  if (ep.tail_tiles > 0) {
    if (n_split != ep.tail_splits || ep.full_tiles + ep.tail_tiles != tiles_m * tiles_n) return RH_E_INVALID;
    grid = dim3((unsigned)(ep.full_tiles + ep.tail_tiles * ep.tail_splits), 1u);
  }
  constexpr size_t lds = DuoShape<T>::LDS;
  static_assert(2 * lds <= 160 * 1024 && lds >= kTriLdsBytes, "two blocks share a CU");
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&mfma_gemm_duo_kernel<T, NCHW, PASS>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (attr != hipSuccess) return (int)attr;
  ProfScope prof(tag, flops, stream);
  hipLaunchKernelGGL((mfma_gemm_duo_kernel<T, NCHW, PASS>), grid, dim3(T::NT), lds, stream, ap, bp, src, ep, tiles_m, k_steps, sps, groups, rest);
  return launch_status();
}

// What a contraction takes: a block alone on a CU, or two at a time, in us a K step and a block.
struct DuoRates { double one, one_block, two, two_block; };
static double duo_run_us(const DuoRates& r, long long blocks, int steps) {
  const long long k = cdiv<long long>(blocks, 256);
  return k <= 1 ? r.one_block + steps * r.one : (double)k * (r.two_block + steps * r.two);
}

// Parts of an image whose maxima are taken one by one: enough blocks for the CUs.
static int duo_image_parts(int N) { return N >= 128 ? 8 : N >= 32 ? 16 : 32; }
static int duo_channel_parts(int C) { const int p = round_up(cdiv(2048, C), 8); return p < 64 ? p : 64; }

// Rows of a table that the tiles read whole.
static int duo_rows(int rows) { return round_up(rows, 128); }

// The constants are a fit to 1561 timed calls (12 layers at 10 batches, slices of 1 to 24 and tails of 2 to 6; rms error 6 %); the
// slices chosen by it are 0.5 % slower than the best of them on average.
static const DuoRates kDuo128 = {0.285, 2.4, 0.262, 0.7}, kDuo96 = {0.22, 10.2, 0.224, 0.9}, kDuo64 = {0.107, 6.9, 0.269, 0.6};
TriPlan plan_duo(int N, int Ci, int Hi, int Wi, int rows, int R, int S, int st, int halo, int P, int Q) {
  TriPlan p = {};
  p.N = N; p.Ci = Ci; p.Hi = Hi; p.Wi = Wi; p.rows = rows; p.R = R; p.S = S; p.st = st; p.halo = halo; p.P = P; p.Q = Q;
  if (Ci % 8 != 0 || halo < 0 || P <= 0 || Q <= 0) return p;
  p.Hp = Hi + 2 * halo; p.Wp = Wi + 2 * halo;
  p.groups_true = Ci / 8 * R * S;
  p.groups = round_up(p.groups_true, 2);
  p.tab_bytes = align256(sizeof(int) * (size_t)p.groups) + align256(sizeof(int) * (2 * (size_t)duo_rows(rows) + N)) +
                align256(sizeof(float) * ((size_t)N * duo_image_parts(N) + round_up(rows, 4) + Ci / 8 * kDuoRatioParts));
  const size_t w_part = 16 * (size_t)p.groups * rows, img_part = 2 * (size_t)N * Ci * p.Hp * p.Wp;
  if (2 * w_part > kMaxBufferBytes || 2 * img_part > kMaxBufferBytes) return p;
  p.wt_bytes = align256(2 * w_part);
  p.img_bytes = align256(2 * img_part);
  p.bm = pick_bm(rows);
  if (p.bm == 32) p.bm = 64;
  p.bn = p.bm == 64 ? 256 : 128;
  const long long cols = (long long)N * P * Q, tiles = (long long)cdiv(rows, p.bm) * cdiv<long long>(cols, p.bn);
  const int steps = p.groups / 2, tm = cdiv(rows, p.bm);
  const double out_us = 4.0 * (double)rows * (double)cols / 1e6;   // at 1 TB/s
  p.splits = 1;
  p.tail = TailSplit{0, 0, 1, 0};
  const DuoRates& rate = p.bm == 128 ? kDuo128 : p.bm == 96 ? kDuo96 : kDuo64;
  p.us = duo_run_us(rate, tiles, steps);
  for (int want = 2; want <= 24 && want * 6 <= steps && tiles * want <= 2048; ++want) {
    const int n = cdiv(steps, want), S2 = cdiv(steps, n);
    if (S2 != want || (double)S2 * out_us > 256.0) continue;
    const double us = duo_run_us(rate, tiles * S2, n) + 1.6 + 0.136 * out_us * (2 * S2 + 1);
    if (us < 0.97 * p.us) { p.us = us; p.splits = S2; }
  }
  const long long full_cols = tiles / 256 * 256 / tm, full = full_cols * tm, tail = tiles - full;
  for (int S2 = 2; S2 <= 12 && S2 * 6 <= steps && full > 0 && tail > 0; ++S2) {
    const int n = cdiv(steps, S2);
    if (cdiv(steps, n) != S2) continue;
    const double us = duo_run_us(rate, full, steps) + (double)cdiv<long long>(tail * S2, 256) * (n * rate.two + rate.two_block) + 1.6 +
                      0.136 * out_us * (double)tail / (double)tiles * (2 * S2 + 1);
    if (us < 0.97 * p.us) { p.us = us; p.splits = 1; p.tail.splits = S2; }
  }
  if (p.tail.splits > 1) {
    p.tail.full_tiles = (int)full; p.tail.tail_tiles = (int)tail; p.tail.col0 = full_cols * p.bn;
  }
  // the maxima and the copies (more slowly past what the Infinity Cache holds), and the result
  const double in_mb = 4e-6 * (double)N * Ci * Hi * Wi;
  p.us += 13.8 + 0.466 * in_mb + 5e-6 * (double)rows * Ci * R * S + 0.154 * out_us + 0.2 * fmax(0.0, 2.0 * in_mb + out_us - 300.0);
  const long long total = (long long)rows * cols;
  p.part_bytes = p.splits > 1 ? align256(sizeof(float) * (size_t)p.splits * (size_t)total)
                 : p.tail.splits > 1 ? align256(sizeof(float) * (size_t)p.tail.splits * (size_t)(total - tail_first_elem(p.tail, (long long)P * Q, rows))) : 0;
  p.ok = true;
  return p;
}

int launch_conv_duo(const TriPlan& p, bool bwd, const float* in, const float* w, float* out, float alpha, float beta,
                    const float* bias, int relu, const float* mask, void* ws, hipStream_t stream, BnInferJob* bn) {
  char* base = static_cast<char*>(ws);
  int* soff = reinterpret_cast<int*>(base);
  int* exps_a = reinterpret_cast<int*>(base + align256(sizeof(int) * (size_t)p.groups));
  int* lost = exps_a + duo_rows(p.rows);
  int* exps_b = lost + duo_rows(p.rows);
  float* top_b = reinterpret_cast<float*>(reinterpret_cast<char*>(exps_a) + align256(sizeof(int) * (2 * (size_t)duo_rows(p.rows) + p.N)));
  const int parts = duo_image_parts(p.N);
  float* top_a = top_b + (size_t)p.N * parts;
  float* ratio = top_a + round_up(p.rows, 4);
  uint4* wt = reinterpret_cast<uint4*>(base + p.tab_bytes);
  uint4* xt = reinterpret_cast<uint4*>(base + p.tab_bytes + p.wt_bytes);
  float* part = reinterpret_cast<float*>(base + p.tab_bytes + p.wt_bytes + p.img_bytes);
  const size_t w_plane = (size_t)p.groups * p.rows, img_groups = (size_t)p.N * (p.Ci / 8) * p.Hp * p.Wp;
  const int RS = p.R * p.S;
  {
    const DuoMaxJob ji = duo_max_job(in, top_b, 1, p.N, p.Ci * p.Hi * p.Wi, parts);
    const DuoMaxJob jw = bwd ? duo_max_job(w, top_a, p.Ci, p.rows, RS, 1, lost, duo_rows(p.rows)) : duo_max_job(w, top_a, 1, p.rows, p.Ci * RS, 1, lost, duo_rows(p.rows));
    DuoRatioJob jr;
    jr.w = w; jr.part = ratio; jr.rows = p.rows; jr.Ck = p.Ci; jr.RS = RS; jr.bwd = bwd ? 1 : 0; jr.dRS = FastDiv((uint32_t)RS);
    ProfScope prof("duo_max", 4.0 * ((double)p.N * p.Ci * p.Hi * p.Wi + 2.0 * p.rows * p.Ci * RS), stream);
    hipLaunchKernelGGL(duo_max_kernel, dim3((unsigned)(ji.blocks + jw.blocks + p.Ci / 8 * kDuoRatioParts)), dim3(256), 0, stream, ji, jw, jr);
  }
  if (int e = launch_status()) return e;
  {
    DuoFilterArgs f;
    f.w = w; f.wt = wt; f.soff = soff; f.top = top_a; f.exps = exps_a; f.lost = lost; f.groups = p.groups; f.groups_true = p.groups_true; f.rows = p.rows;
    f.Ck = p.Ci; f.RS = RS; f.S = p.S; f.Wp = p.Wp; f.bwd = bwd ? 1 : 0;
    const unsigned img_blocks = (unsigned)cdiv<size_t>(img_groups, 256);
    ProfScope prof("duo_image", 4.0 * (double)p.N * p.Ci * p.Hi * p.Wi + 32.0 * (double)img_groups + 64.0 * (double)w_plane, stream);
    hipLaunchKernelGGL(duo_image_kernel, dim3(img_blocks + (unsigned)cdiv<size_t>(w_plane, 256)), dim3(256), 0, stream, in, xt,
                       (unsigned)img_groups, p.Hi, p.Wi, FastDiv((uint32_t)p.Wp), FastDiv((uint32_t)(p.Ci / 8)), FastDiv((uint32_t)p.Hp),
                       p.halo, (int)img_blocks, reinterpret_cast<const float4*>(top_b), parts, exps_b,
                       reinterpret_cast<const float4*>(ratio), f);
  }
  if (int e = launch_status()) return e;
  DuoParams ap, bp;
  ap.t.v.ptr = wt; ap.t.plane = (int)(16 * w_plane); ap.t.v.bytes = (uint32_t)(32 * w_plane);
  ap.t.v.M = p.rows; ap.t.v.inner = 1; ap.t.v.innerW = 1; ap.t.v.img_stride = 16; ap.t.v.a_stride = 0; ap.t.v.b_stride = 0;
  ap.t.v.soff = nullptr; ap.t.v.group_stride = p.rows * 16;
  ap.exps = exps_a; ap.lost = lost; ap.ediv = 1; ap.emod = p.rows;
  bp.t.v.ptr = xt; bp.t.plane = (int)(16 * img_groups); bp.t.v.bytes = (uint32_t)(32 * img_groups);
  bp.t.v.M = p.N * p.P * p.Q; bp.t.v.inner = p.P * p.Q; bp.t.v.innerW = p.Q;
  bp.t.v.img_stride = p.Hp * p.Wp * p.Ci * 2; bp.t.v.a_stride = p.st * (p.Ci / 8) * p.Wp * 16; bp.t.v.b_stride = p.st * 16;
  bp.t.v.soff = soff; bp.t.v.group_stride = 0;
  bp.exps = exps_b; bp.lost = nullptr; bp.ediv = p.P * p.Q; bp.emod = p.N;
  DuoSource src;
  src.pass = bwd ? RH_CONV_BWD_DATA : RH_CONV_FWD; src.a = w; src.b = in; src.N = p.N; src.C = p.Ci; src.H = p.Hi; src.W = p.Wi;
  src.rows = p.rows; src.R = p.R; src.S = p.S; src.st = p.st; src.halo = p.halo; src.P = p.P; src.Q = p.Q;
  EpiParams ep;
  ep.out = out; ep.bias = bias; ep.alpha = alpha; ep.beta = beta;
  ep.rows = p.rows; ep.cols = bp.t.v.M; ep.inner = p.P * p.Q; ep.ld = 0; ep.relu = relu; ep.split_stride = 0; ep.mask = mask;
  const long long total = (long long)ep.rows * ep.cols;
  const EpiParams fin = ep;
  const long long first = p.splits > 1 ? 0 : tail_first_elem(p.tail, ep.inner, ep.rows);
  if (p.splits > 1) {
    ep.out = part; ep.split_stride = total;
  } else if (p.tail.splits > 1) {
    ep.part = part; ep.part_first = first; ep.split_stride = total - first;
    ep.full_tiles = p.tail.full_tiles; ep.tail_tiles = p.tail.tail_tiles; ep.tail_splits = p.tail.splits;
  }
  const double flops = 6.0 * (double)total * p.Ci * RS;
  const int steps = p.groups / 2;
  int used = 1, e;
#define RH_DUO(TILE, TAG)                                                                                                           \
  (bwd ? launch_duo<TILE, true, PassConvBwdData>(ap, bp, src, ep, steps, p.groups_true, p.splits, &used, flops, stream,             \
                                                 "conv_bwd_data_duo_" TAG)                                                          \
       : launch_duo<TILE, true, PassConvFwd>(ap, bp, src, ep, steps, p.groups_true, p.splits, &used, flops, stream, "conv_fwd_duo_" TAG))
  switch (p.bm) {
    case 128: e = RH_DUO(T128x128t, "128x128"); break;
    case 96: e = RH_DUO(T96x128t, "96x128"); break;
    default: e = RH_DUO(T64x256t, "64x256"); break;
  }
#undef RH_DUO
  if (e) return e;
  if (p.splits > 1 || p.tail.splits > 1)
    launch_split_reduce_nchw(part, used, total - first, fin.out, total, fin.inner, fin.rows, fin.alpha, fin.beta, fin.bias, fin.relu,
                             stream, p.splits > 1 ? 0 : p.tail.col0, fin.mask, bn);
  return launch_status();
}

// (1355 timed calls of 13 layers, slices of 1 to 128: rms error 9 %, the slices chosen 0.6 % slower than the best of them.)
static const DuoRates kDuoFilter128 = {0.279, 2.9, 0.233, 0.0}, kDuoFilter96 = {0.267, 9.4, 0.482, 0.0}, kDuoFilter64 = {0.282, 0.8, 0.24, 1.9};
TriFilterPlan plan_duo_bwd_filter(const ConvDims& d) {
  TriFilterPlan p = {};
  if (d.P <= 0 || d.Q <= 0) return p;
  p.Hp = d.H + 2 * d.pad; p.Wp = d.W + 2 * d.pad;
  p.n8 = cdiv(d.N, 8);
  const long long groups = (long long)p.n8 * d.P * d.Q;
  p.groups_true = (int)groups;
  p.groups = round_up(p.groups_true, 2);
  const size_t dy_part = 16 * (size_t)p.groups * d.K, x_part = 16 * (size_t)p.n8 * p.Hp * p.Wp * d.C;
  if (2 * dy_part > kMaxBufferBytes || 2 * x_part > kMaxBufferBytes) return p;
  p.tab_bytes = align256(sizeof(int) * (size_t)p.groups) + align256(sizeof(int) * ((size_t)duo_rows(d.K) + d.C + 1)) +
                align256(sizeof(float) * ((size_t)d.K * duo_channel_parts(d.K) + (size_t)d.C * duo_channel_parts(d.C)));
  p.dyt_bytes = align256(2 * dy_part);
  p.xt_bytes = align256(2 * x_part);
  p.bm = pick_bm(d.K);
  if (p.bm == 32) p.bm = 64;
  p.bn = p.bm == 64 ? 256 : 128;
  const int CRS = d.C * d.R * d.S, tiles = cdiv(d.K, p.bm) * cdiv(CRS, p.bn), steps = p.groups / 2;
  p.us = 1e30;
  const DuoRates& rate = p.bm == 128 ? kDuoFilter128 : p.bm == 96 ? kDuoFilter96 : kDuoFilter64;
  // (more slices take 0.45 us each at least)
  for (int want = 1; want <= 256 && 0.45 * want < p.us && (want == 1 || (want * 6 <= steps && (long long)tiles * want <= 2048)); ++want) {
    const int n = cdiv(steps, want), S = cdiv(steps, n);
    if (S != want || 4.0 * (double)S * (double)d.w_elems > 256e6) continue;
    const double us = duo_run_us(rate, (long long)tiles * S, n) + 0.45 * S + 1.6e-6 * (double)d.w_elems * (S + 1);
    if (us < p.us) { p.us = us; p.splits = S; }
  }
  if (p.splits == 0) p.splits = 1;   // (as plan_tri_bwd_filter)
  p.us += kDuoFilterCopies + 2e-6 * (double)(d.x_elems + d.y_elems);
  p.part_bytes = align256(sizeof(float) * (size_t)p.splits * (size_t)d.w_elems);
  p.sum_rows = p.n8 * cdiv(d.P * d.Q, kDuoPix);
  p.sum_bytes = align256(sizeof(float) * (size_t)p.sum_rows * d.K);
  p.ok = true;
  return p;
}

int launch_conv_duo_bwd_filter(const ConvDims& d, const TriFilterPlan& p, const float* x, const float* dy, float* sums, void* ws,
                               hipStream_t stream, float** parts, int* used, const TriFilterPlan* three, OrThree* or_three) {
  char* base = static_cast<char*>(ws);
  int* soff = reinterpret_cast<int*>(base);
  int* exps_a = reinterpret_cast<int*>(base + align256(sizeof(int) * (size_t)p.groups));
  int *exps_b = exps_a + duo_rows(d.K), *any = exps_b + d.C;
  float* top_a = reinterpret_cast<float*>(reinterpret_cast<char*>(exps_a) + align256(sizeof(int) * ((size_t)duo_rows(d.K) + d.C + 1)));
  const int parts_a = duo_channel_parts(d.K), parts_b = duo_channel_parts(d.C);
  float* top_b = top_a + (size_t)d.K * parts_a;
  uint4* dyt = reinterpret_cast<uint4*>(base + p.tab_bytes);
  uint4* xt = reinterpret_cast<uint4*>(base + p.tab_bytes + p.dyt_bytes);
  *parts = reinterpret_cast<float*>(base + p.tab_bytes + p.dyt_bytes + p.xt_bytes);
  const size_t dy_plane = (size_t)p.groups * d.K, x_plane = (size_t)p.n8 * p.Hp * p.Wp * d.C;
  {
    const DuoMaxJob ja = duo_max_job(dy, top_a, d.N, d.K, d.P * d.Q, parts_a, any, 1), jb = duo_max_job(x, top_b, d.N, d.C, d.H * d.W, parts_b);
    ProfScope prof("duo_max", 4.0 * (double)(d.y_elems + d.x_elems), stream);
    hipLaunchKernelGGL(duo_max_kernel, dim3((unsigned)(ja.blocks + jb.blocks)), dim3(256), 0, stream, ja, jb, DuoRatioJob{});
  }
  if (int e = launch_status()) return e;
  {
    DuoBatchArgs a, b;
    a.x = dy; a.xt = dyt; a.top = top_a; a.parts = parts_a; a.exps = exps_a; a.any = any; a.N = d.N; a.C = d.K; a.H = d.P; a.W = d.Q; a.halo = 0;
    a.HpWp = d.P * d.Q; a.dWp = FastDiv((uint32_t)d.Q); a.plane = dy_plane; a.px = cdiv(a.HpWp, kDuoPix); a.cx = cdiv(a.C, kDuoCh);
    a.blocks = a.px * a.cx * p.n8; a.sums = sums;
    b.x = x; b.xt = xt; b.top = top_b; b.parts = parts_b; b.exps = exps_b; b.any = any; b.N = d.N; b.C = d.C; b.H = d.H; b.W = d.W; b.halo = d.pad;
    b.HpWp = p.Hp * p.Wp; b.dWp = FastDiv((uint32_t)p.Wp); b.plane = x_plane; b.px = cdiv(b.HpWp, kDuoPix); b.cx = cdiv(b.C, kDuoCh);
    b.blocks = b.px * b.cx * p.n8; b.sums = nullptr;
    ProfScope prof("duo_batch", 4.0 * (double)(d.y_elems + d.x_elems) + 32.0 * (double)(dy_plane + x_plane), stream);
    hipLaunchKernelGGL(duo_batch_kernel, dim3((unsigned)(a.blocks + b.blocks + cdiv(p.groups, 256))), dim3(256), 0, stream, a, b, soff,
                       p.groups, p.groups_true, d.P * d.Q, d.Q, d.st, p.Wp);
  }
  if (int e = launch_status()) return e;
  TriRest rest = {};
  if (three) {
    if (int e = launch_tri_rest_copies(d, *three, x, dy, base + p.tab_bytes, any, stream, &rest)) return e;
    or_three->any = any; or_three->splits = rest.splits;
  }
  const int CRS = d.C * d.R * d.S;
  DuoParams ap, bp;
  ap.t.v.ptr = dyt; ap.t.plane = (int)(16 * dy_plane); ap.t.v.bytes = (uint32_t)(32 * dy_plane);
  ap.t.v.M = d.K; ap.t.v.inner = 1; ap.t.v.innerW = 1; ap.t.v.img_stride = 16; ap.t.v.a_stride = 0; ap.t.v.b_stride = 0;
  ap.t.v.soff = nullptr; ap.t.v.group_stride = d.K * 16;
  ap.exps = exps_a; ap.lost = nullptr; ap.ediv = 1; ap.emod = d.K;
  bp.t.v.ptr = xt; bp.t.plane = (int)(16 * x_plane); bp.t.v.bytes = (uint32_t)(32 * x_plane);
  bp.t.v.M = CRS; bp.t.v.inner = d.S * d.C; bp.t.v.innerW = d.C;   // columns j = (r, s, c)
  bp.t.v.img_stride = p.Wp * d.C * 16; bp.t.v.a_stride = d.C * 16; bp.t.v.b_stride = 16;
  bp.t.v.soff = soff; bp.t.v.group_stride = 0;
  bp.exps = exps_b; bp.lost = nullptr; bp.ediv = 1; bp.emod = d.C;
  DuoSource src;
  src.pass = RH_CONV_BWD_FILTER; src.a = dy; src.b = x; src.N = d.N; src.C = d.C; src.H = d.H; src.W = d.W;
  src.rows = d.K; src.R = d.R; src.S = d.S; src.st = d.st; src.halo = d.pad; src.P = d.P; src.Q = d.Q;
  EpiParams ep;
  ep.out = *parts; ep.bias = nullptr; ep.alpha = 1.0f; ep.beta = 0.0f;
  ep.rows = d.K; ep.cols = CRS; ep.inner = 0; ep.ld = CRS; ep.relu = 0; ep.split_stride = (long long)d.K * CRS;
  const double flops = 6.0 * (double)d.w_elems * d.N * d.P * d.Q;
  const int steps = p.groups / 2;
#define RH_DUO(TILE, TAG) \
  launch_duo<TILE, false, PassConvBwdFilter>(ap, bp, src, ep, steps, p.groups_true, p.splits, used, flops, stream, "conv_bwd_filter_duo_" TAG, rest)
  switch (p.bm) {
    case 128: return RH_DUO(T128x128t, "128x128");
    case 96: return RH_DUO(T96x128t, "96x128");
    default: return RH_DUO(T64x256t, "64x256");
  }
#undef RH_DUO
}

}  // namespace rh

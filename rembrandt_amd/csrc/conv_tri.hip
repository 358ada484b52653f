// fp32 convolutions on the bf16 matrix instructions with exactly split operands (gemm_tri.h): forward, stride-1
// backward-data and backward-filter.
//
// Operand copies, each in three bf16 parts (6 bytes a value, written once per call):
//   forward        filter [k/8][ko][8], image [n][Hp][c/8][Wp][8] with its zero border; k = (c/16, r, s, c % 16)
//   backward-data  the same of the flipped, transposed filter and of dy
//   backward-filter  dy [n/8][p][q][ko][8 n] and x [n/8][Hp][Wp][c][8 n]; k = (n/8, p, q) and the image of a group of eight:
//     a group of eight k is one pixel of eight images, so a filter tap is a constant displacement of the group, whatever its
//     parity, and rows (filters, channels) are neighbouring 16-byte pieces
#include "conv_common.h"
#include "gemm_tri.h"

namespace rh {

// part i of the group at `at` (16-byte pieces), parts `plane` pieces apart
__device__ __forceinline__ void tri_store(uint4* dst, size_t at, size_t plane, const float (&v)[8], bool wide = false) {
  uint4 o[3];
  tri_pack8(v, o, wide);
#pragma unroll
  for (int i = 0; i < 3; ++i) dst[at + i * plane] = o[i];
}

// Filter copy and the table of the image's group offsets; an item is a (group, row).  bwd: rows are input channels, the
// contraction runs over filters and the taps are flipped.
struct TriFilterArgs {
  const float* w; uint4* wt; int* soff;
  int groups, groups_true, rows, Ck, RS, S, Wp, bwd;
};
__device__ __forceinline__ void tri_filter_body(const TriFilterArgs& a, long long i) {
  const long long total = (long long)a.groups * a.rows;
  if (i >= total) return;
  const int g = (int)(i / a.rows), row = (int)(i - (long long)g * a.rows);
  // all taps of sixteen channels, two groups a tap, then of the next sixteen: the pixels that a block reads for one tap it
  // reads for the others soon after, from the L2 (of eight channels that are left over one group a tap)
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
  tri_store(a.wt, (size_t)i, (size_t)total, v);
  if (row == 0) {
    const int r = rs / a.S, s2 = rs - r * a.S;
    a.soff[g] = g < a.groups_true ? ((r * (a.Ck / 8) + c0 / 8) * a.Wp + s2) * 16 : 0;
  }
}

// The sub-filters of all residue classes one behind the other, [class][k/8][c][8] in three parts each, and their tables; k order and
// taps as above, a class's taps (i, j) being the filter's (a + st i, b + st j).
struct TriClassFilter { int first, groups, groups_true, a, b, Ra, Sb; };   // groups of all classes before; of this one
struct TriClassFilterArgs {
  const float* w; uint4* wt; int* soff;
  int groups, C, K, R, S, st, Wp, count;
  TriClassFilter c[16];
};
__device__ __forceinline__ void tri_class_filter_body(const TriClassFilterArgs& f, long long i) {
  if (i >= (long long)f.groups * f.C) return;
  const int all = (int)(i / f.C), row = (int)(i - (long long)all * f.C);
  int q = 0;
  while (q + 1 < f.count && all >= f.c[q + 1].first) ++q;
  const TriClassFilter c = f.c[q];
  const int g = all - c.first, taps = c.Ra * c.Sb, pairs = f.K / 16 * taps, step = g >> 1;
  int t, k0;
  if (step < pairs) {
    t = step % taps;
    k0 = step / taps * 16 + (g & 1) * 8;
  } else {
    t = g - 2 * pairs;
    k0 = f.K - 8;
  }
  const bool live = g < c.groups_true;
  const int ti = live ? t / c.Sb : 0, tj = live ? t - ti * c.Sb : 0;
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e)
    v[e] = live ? f.w[(((size_t)(k0 + e) * f.C + row) * f.R + (c.a + f.st * ti)) * f.S + (c.b + f.st * tj)] : 0.0f;
  tri_store(f.wt + (size_t)c.first * 3 * f.C, (size_t)g * f.C + row, (size_t)c.groups * f.C, v);
  if (row == 0) f.soff[all] = live ? (((c.Ra - 1 - ti) * (f.K / 8) + k0 / 8) * f.Wp + (c.Sb - 1 - tj)) * 16 : 0;
}
__global__ __launch_bounds__(256) void tri_class_filter_kernel(TriClassFilterArgs f) {
  tri_class_filter_body(f, (long long)blockIdx.x * 256 + threadIdx.x);
}

// x [n][C][H][W] -> [n][Hp][C/8][Wp][8], a thread per group, and behind it the filter copy, which is independent of it: one
// launch less in front of the contraction.  Blocks that follow one another stay on an XCD: their reads share cache lines.
__global__ __launch_bounds__(256) void tri_image_kernel(const float* __restrict__ x, uint4* __restrict__ xt, unsigned total, int H,
                                                        int W, FastDiv dWp, FastDiv dCg, FastDiv dHp, int halo, int img_blocks,
                                                        TriFilterArgs f) {
  if ((int)blockIdx.x >= img_blocks) {
    tri_filter_body(f, (long long)(blockIdx.x - img_blocks) * 256 + threadIdx.x);
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
  tri_store(xt, i, total, v);
}

// x [N][C][H][W] -> [n/8][Hp][Wp][C][8 n]: a block moves 32 pixels x 32 channels of eight images through LDS, and may leave
// the sums of its pixels and images, a row of C values, for the bias gradient.
constexpr int kTriPix = 32, kTriCh = 32;
struct TriBatchArgs {
  const float* x; uint4* xt;
  int N, C, H, W, halo, HpWp;
  FastDiv dWp;
  size_t plane;         // 16-byte pieces of a part
  int px, cx, blocks;   // blocks along the pixels and the channels; all of them
  float* sums;          // [n/8][pixel block][C], or nullptr
  bool wide;            // mark for the wide form
};
__device__ __forceinline__ void tri_batch_body(const TriBatchArgs& a, int b, float (&tile)[8][kTriCh][kTriPix + 1]) {
  const int bx = b % a.px, t = b / a.px, by = t % a.cx, bz = t / a.cx;
  const int pix0 = bx * kTriPix, c0 = by * kTriCh, n0 = bz * 8;
  {
    const int pl = threadIdx.x & 31, pix = pix0 + pl;
    uint32_t hp, wp;
    a.dWp.divmod((uint32_t)pix, hp, wp);
    const int h = (int)hp - a.halo, w = (int)wp - a.halo;
    const bool in = pix < a.HpWp && (unsigned)h < (unsigned)a.H && (unsigned)w < (unsigned)a.W;
    const size_t hw = (size_t)a.H * a.W;
    const float* src = a.x + (size_t)(in ? h * a.W + w : 0);
    const int c_first = threadIdx.x >> 5;   // eight channels at a time
    float v[8][kTriCh / 8];
#pragma unroll
    for (int n = 0; n < 8; ++n)
#pragma unroll
      for (int i = 0; i < kTriCh / 8; ++i) {
        const int c = c0 + c_first + 8 * i;
        v[n][i] = in && c < a.C && n0 + n < a.N ? src[((size_t)(n0 + n) * a.C + c) * hw] : 0.0f;
      }
#pragma unroll
    for (int n = 0; n < 8; ++n)
#pragma unroll
      for (int i = 0; i < kTriCh / 8; ++i) tile[n][c_first + 8 * i][pl] = v[n][i];
  }
  __syncthreads();
  const int cl = threadIdx.x & 31, c = c0 + cl;
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < kTriPix / 8; ++i) {
    const int pl = (threadIdx.x >> 5) + 8 * i, pix = pix0 + pl;
    float v[8];
#pragma unroll
    for (int n = 0; n < 8; ++n) v[n] = tile[n][cl][pl];
    if (a.sums) sum += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    if (pix < a.HpWp && c < a.C) tri_store(a.xt, ((size_t)bz * a.HpWp + pix) * a.C + c, a.plane, v, a.wide);
  }
  if (a.sums) {
    __syncthreads();
    float* const part = &tile[0][0][0];
    part[threadIdx.x] = sum;
    __syncthreads();
    if (threadIdx.x < kTriCh && c < a.C) {
      float s = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) s += part[i * 32 + cl];
      a.sums[((size_t)bz * a.px + bx) * a.C + c] = s;
    }
  }
}

// The same for x of a first layer, up to kTriFew channels, where 29 of the 32 channels above would be none: a thread a pixel, all its
// channels and images, past LDS.  Bound by its bytes.  Copies of both operands, 3 channels, us: 96 filters 11x11 stride 4 at 50 and 256 images 80 -> 51
// and 343 -> 238, 64 filters 7x7 stride 2 at 24 and 256 50 -> 41 and 608 -> 487.
constexpr int kTriFew = 4, kTriFewPix = 256;
__device__ __forceinline__ void tri_few_body(const TriBatchArgs& a, int b) {
  const int bx = b % a.px, bz = b / a.px, pix = bx * kTriFewPix + (int)threadIdx.x, n0 = bz * 8;
  if (pix >= a.HpWp) return;
  uint32_t hp, wp;
  a.dWp.divmod((uint32_t)pix, hp, wp);
  const int h = (int)hp - a.halo, w = (int)wp - a.halo;
  const bool in = (unsigned)h < (unsigned)a.H && (unsigned)w < (unsigned)a.W;
  const size_t hw = (size_t)a.H * a.W;
  const float* const src = a.x + (size_t)(in ? h * a.W + w : 0);
  float v[kTriFew][8];
#pragma unroll
  for (int c = 0; c < kTriFew; ++c)
#pragma unroll
    for (int n = 0; n < 8; ++n) v[c][n] = in && c < a.C && n0 + n < a.N ? src[((size_t)(n0 + n) * a.C + c) * hw] : 0.0f;
#pragma unroll
  for (int c = 0; c < kTriFew; ++c)
    if (c < a.C) tri_store(a.xt, ((size_t)bz * a.HpWp + pix) * a.C + c, a.plane, v[c], false);
}

// Both operands of a filter gradient and soff[g], the place of group g = (n/8, p, q) in x's copy; the groups past the last
// are zeros of dy.
struct TriTableArgs { int* soff; int groups, groups_true, PQ, Q, st, Wp, blocks; };
__device__ __forceinline__ void tri_batch_block(const TriBatchArgs& dy, const TriBatchArgs& x, const TriTableArgs& t, int b,
                                                float (&tile)[8][kTriCh][kTriPix + 1]) {
  if (b < dy.blocks) { tri_batch_body(dy, xcd_remap(b, dy.blocks), tile); return; }
  b -= dy.blocks;
  if (b < x.blocks) {
    if (x.C <= kTriFew) tri_few_body(x, xcd_remap(b, x.blocks));
    else tri_batch_body(x, xcd_remap(b, x.blocks), tile);
    return;
  }
  b -= x.blocks;
  if (t.groups > t.groups_true)   // (one group: every block of the table writes a share)
    for (int i = b * 256 + threadIdx.x; i < 3 * dy.C; i += t.blocks * 256)
      dy.xt[(size_t)(i / dy.C) * dy.plane + (size_t)t.groups_true * dy.C + i % dy.C] = make_uint4(0, 0, 0, 0);
  const int g = b * 256 + threadIdx.x;
  if (g >= t.groups) return;
  int off = 0;
  if (g < t.groups_true) {
    const int n8 = g / t.PQ, pq = g - n8 * t.PQ, p = pq / t.Q, q = pq - p * t.Q;
    off = (n8 * x.HpWp + p * t.st * t.Wp + q * t.st) * x.C * 16;
  }
  t.soff[g] = off;
}
__global__ __launch_bounds__(256) void tri_batch_kernel(TriBatchArgs dy, TriBatchArgs x, TriTableArgs t) {
  __shared__ float tile[8][kTriCh][kTriPix + 1];
  tri_batch_block(dy, x, t, blockIdx.x, tile);
}
// The same by a few blocks, and only where it is wanted (TriRest): a launch of as many blocks as there is work for would wait, beside
// another stream's, for a place for each of them before it could end (AlexNet b256: 77 us on average, 12 so).
__global__ __launch_bounds__(256) void tri_rest_batch_kernel(TriBatchArgs dy, TriBatchArgs x, TriTableArgs t, const int* __restrict__ any) {
  __shared__ float tile[8][kTriCh][kTriPix + 1];
  if (*any == 0) return;
  for (int b = blockIdx.x; b < dy.blocks + x.blocks + t.blocks; b += (int)gridDim.x) {
    tri_batch_block(dy, x, t, b, tile);
    __syncthreads();   // (the tile is the next block's)
  }
}

template <class T, bool B_LINEAR, bool NCHW, class PASS, bool WIDE = false>
static int launch_tri(const TriParams& ap, const TriParams& bp, const EpiParams& ep, int k_steps, int groups, int splits, int* used,
                      double flops, hipStream_t stream, const char* tag) {
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
  constexpr size_t lds = kTriLdsBytes;
  static_assert(2 * lds <= 160 * 1024, "two blocks share a CU");
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&mfma_gemm_tri_kernel<T, B_LINEAR, NCHW, PASS, WIDE>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (attr != hipSuccess) return (int)attr;
  ProfScope prof(tag, flops, stream);
  hipLaunchKernelGGL((mfma_gemm_tri_kernel<T, B_LINEAR, NCHW, PASS, WIDE>), grid, dim3(T::NT), lds, stream, ap, bp, ep, tiles_m,
                     k_steps, sps, groups);
  return launch_status();
}

// Slices of the contraction, of all tiles or of those past a multiple of 256, and the time a call is expected to take: two
// blocks to a CU, a K step of a block at a time each (0.456 us on 128 x 128: 294 TFLOP/s of fp32 multiply-adds on all CUs), a
// block alone on its CU 0.415 us.  The constants are a fit to 2138 timed calls (22 layers at 14 batches, slices of 1 to 24 and
// tails of 2 to 12; rms error 6 %); the slices chosen by it are 0.9 % slower than the best of them on average.
TriPlan plan_tri(int N, int Ci, int Hi, int Wi, int rows, int R, int S, int st, int halo, int P, int Q, int max_chain) {
  TriPlan p = {};
  p.N = N; p.Ci = Ci; p.Hi = Hi; p.Wi = Wi; p.rows = rows; p.R = R; p.S = S; p.st = st; p.halo = halo; p.P = P; p.Q = Q;
  if (Ci % 8 != 0 || halo < 0 || P <= 0 || Q <= 0) return p;
  p.Hp = Hi + 2 * halo; p.Wp = Wi + 2 * halo;
  p.groups_true = Ci / 8 * R * S;
  p.groups = round_up(p.groups_true, 2);
  p.tab_bytes = align256(sizeof(int) * (size_t)p.groups);
  const size_t w_part = 16 * (size_t)p.groups * rows, img_part = 2 * (size_t)N * Ci * p.Hp * p.Wp;
  if (3 * w_part > kMaxBufferBytes || 3 * img_part > kMaxBufferBytes) return p;
  p.wt_bytes = align256(3 * w_part);
  p.img_bytes = align256(3 * img_part);
  p.bm = pick_bm(rows);
  if (p.bm == 32) p.bm = 64;
  p.bn = p.bm == 64 ? 192 : 128;
  const long long cols = (long long)N * P * Q, tiles = (long long)cdiv(rows, p.bm) * cdiv<long long>(cols, p.bn);
  const int steps = p.groups / 2, tm = cdiv(rows, p.bm);
  const double out_us = 4.0 * (double)rows * (double)cols / 1e6;   // at 1 TB/s
  p.splits = 1;
  p.tail = TailSplit{0, 0, 1, 0};
  auto run_us = [&](long long blocks, int n) {
    const long long k = cdiv<long long>(blocks, 256);
    return k <= 1 ? n * (p.bm == 128 ? 0.415 : 0.34) : (double)k * n * (p.bm == 128 ? 0.456 : p.bm == 96 ? 0.377 : 0.366);
  };
  const int chain = max_chain > 0 ? max_chain : steps;
  p.us = steps <= chain ? run_us(tiles, steps) : 1e30;
  for (int want = 2; want <= 24 && want * 4 <= steps && (tiles * want <= 1024 || tiles * 2 <= 512 || steps > chain); ++want) {
    const int n = cdiv(steps, want), S = cdiv(steps, n);
    if (S != want || n > chain || (double)S * out_us > 256.0) continue;
    const double us = run_us(tiles * S, n) + 4.0 + out_us * (2 * S + 1) / 7.7;
    if (us < 0.97 * p.us) { p.us = us; p.splits = S; }
  }
  const long long full_cols = tiles / 256 * 256 / tm, full = full_cols * tm, tail = tiles - full;
  for (int S = 2; S <= 12 && S * 4 <= steps && full > 0 && tail > 0 && steps <= chain; ++S) {
    const int n = cdiv(steps, S);
    if (cdiv(steps, n) != S) continue;
    const double us = run_us(full, steps) + (double)cdiv<long long>(tail * S, 256) * n * (p.bm == 128 ? 0.456 : 0.37) + 4.0 +
                      out_us * (double)tail / (double)tiles * (2 * S + 1) / 7.7;
    if (us < 0.97 * p.us) { p.us = us; p.splits = 1; p.tail.splits = S; }
  }
  if (p.us >= 1e30) return p;   // (no such chains)
  if (p.tail.splits > 1) {
    p.tail.full_tiles = (int)full; p.tail.tail_tiles = (int)tail; p.tail.col0 = full_cols * p.bn;
  }
  // the copies (more slowly past what the Infinity Cache holds), and the result
  const double copy = 4.0 * (double)N * Ci * Hi * Wi + 3.0 * (double)img_part;
  p.us += 9.9 + copy / 6.4e6 + 0.12e-6 * fmax(0.0, copy + 1e6 * out_us - 300e6) + 10.0 * (double)rows * Ci * R * S / 2.2e6 + out_us / 4.2;
  const long long total = (long long)rows * cols;
  p.part_bytes = p.splits > 1 ? align256(sizeof(float) * (size_t)p.splits * (size_t)total)
                 : p.tail.splits > 1 ? align256(sizeof(float) * (size_t)p.tail.splits * (size_t)(total - tail_first_elem(p.tail, (long long)P * Q, rows))) : 0;
  p.ok = true;
  return p;
}

int launch_conv_tri(const TriPlan& p, bool bwd, const float* in, const float* w, float* out, float alpha, float beta,
                    const float* bias, int relu, const float* mask, void* ws, hipStream_t stream, BnInferJob* bn) {
  char* base = static_cast<char*>(ws);
  int* soff = reinterpret_cast<int*>(base);
  uint4* wt = reinterpret_cast<uint4*>(base + p.tab_bytes);
  uint4* xt = reinterpret_cast<uint4*>(base + p.tab_bytes + p.wt_bytes);
  float* part = reinterpret_cast<float*>(base + p.tab_bytes + p.wt_bytes + p.img_bytes);
  const size_t w_plane = (size_t)p.groups * p.rows, img_groups = (size_t)p.N * (p.Ci / 8) * p.Hp * p.Wp;
  {
    TriFilterArgs f;
    f.w = w; f.wt = wt; f.soff = soff; f.groups = p.groups; f.groups_true = p.groups_true; f.rows = p.rows; f.Ck = p.Ci;
    f.RS = p.R * p.S; f.S = p.S; f.Wp = p.Wp; f.bwd = bwd ? 1 : 0;
    const unsigned img_blocks = (unsigned)cdiv<size_t>(img_groups, 256);
    ProfScope prof("tri_image", 4.0 * (double)p.N * p.Ci * p.Hi * p.Wi + 48.0 * (double)img_groups + 80.0 * (double)w_plane, stream);
    hipLaunchKernelGGL(tri_image_kernel, dim3(img_blocks + (unsigned)cdiv<size_t>(w_plane, 256)), dim3(256), 0, stream, in, xt,
                       (unsigned)img_groups, p.Hi, p.Wi, FastDiv((uint32_t)p.Wp), FastDiv((uint32_t)(p.Ci / 8)), FastDiv((uint32_t)p.Hp),
                       p.halo, (int)img_blocks, f);
  }
  if (int e = launch_status()) return e;
  TriParams ap, bp;
  ap.v.ptr = wt; ap.plane = (int)(16 * w_plane); ap.v.bytes = (uint32_t)(48 * w_plane);
  ap.v.M = p.rows; ap.v.inner = 1; ap.v.innerW = 1; ap.v.img_stride = 16; ap.v.a_stride = 0; ap.v.b_stride = 0;
  ap.v.soff = nullptr; ap.v.group_stride = p.rows * 16;
  bp.v.ptr = xt; bp.plane = (int)(16 * img_groups); bp.v.bytes = (uint32_t)(48 * img_groups);
  bp.v.M = p.N * p.P * p.Q; bp.v.inner = p.P * p.Q; bp.v.innerW = p.Q;
  bp.v.img_stride = p.Hp * p.Wp * p.Ci * 2; bp.v.a_stride = p.st * (p.Ci / 8) * p.Wp * 16; bp.v.b_stride = p.st * 16;
  bp.v.soff = soff; bp.v.group_stride = 0;
  EpiParams ep;
  ep.out = out; ep.bias = bias; ep.alpha = alpha; ep.beta = beta;
  ep.rows = p.rows; ep.cols = bp.v.M; ep.inner = p.P * p.Q; ep.ld = 0; ep.relu = relu; ep.split_stride = 0; ep.mask = mask;
  const long long total = (long long)ep.rows * ep.cols;
  const EpiParams fin = ep;
  const long long first = p.splits > 1 ? 0 : tail_first_elem(p.tail, ep.inner, ep.rows);
  if (p.splits > 1) {
    ep.out = part; ep.split_stride = total;
  } else if (p.tail.splits > 1) {
    ep.part = part; ep.part_first = first; ep.split_stride = total - first;
    ep.full_tiles = p.tail.full_tiles; ep.tail_tiles = p.tail.tail_tiles; ep.tail_splits = p.tail.splits;
  }
  const double flops = 12.0 * (double)total * p.Ci * p.R * p.S;
  const int steps = p.groups / 2;
  int used = 1, e;
#define RH_TRI(TILE, TAG)                                                                                             \
  (bwd ? launch_tri<TILE, false, true, PassConvBwdData>(ap, bp, ep, steps, p.groups_true, p.splits, &used, flops, stream, \
                                                              "conv_bwd_data_tri_" TAG)                                      \
       : launch_tri<TILE, false, true, PassConvFwd>(ap, bp, ep, steps, p.groups_true, p.splits, &used, flops, stream,  \
                                                          "conv_fwd_tri_" TAG))
  switch (p.bm) {
    case 128: e = RH_TRI(T128x128t, "128x128"); break;
    case 96: e = RH_TRI(T96x128t, "96x128"); break;
    default: e = RH_TRI(T64x192t, "64x192"); break;
  }
#undef RH_TRI
  if (e) return e;
  if (p.splits > 1 || p.tail.splits > 1)
    launch_split_reduce_nchw(part, used, total - first, fin.out, total, fin.inner, fin.rows, fin.alpha, fin.beta, fin.bias, fin.relu,
                             stream, p.splits > 1 ? 0 : p.tail.col0, fin.mask, bn);
  return launch_status();
}

int launch_conv_tri_phases(const ConvDims& d, const PhasePlan& pp, const TriPhasePlan& p, const float* w, const float* dy, void* ws,
                           hipStream_t stream, float** sub) {
  char* base = static_cast<char*>(ws);
  int* soff = reinterpret_cast<int*>(base);
  uint4* wt = reinterpret_cast<uint4*>(base + p.tab_bytes);
  uint4* xt = reinterpret_cast<uint4*>(base + p.tab_bytes + p.wt_bytes);
  *sub = reinterpret_cast<float*>(base + p.tab_bytes + p.wt_bytes + p.img_bytes);
  const int order_max = d.st * d.st;
  int order[16], count = 0;
  for (int i = 0; i < order_max; ++i) {
    const PhaseGeom& g = pp.ph[i];
    if (g.Ra * g.Sb == 0 || g.U <= 0 || g.V <= 0) continue;
    int at = count++;   // longest first
    for (; at > 0 && pp.ph[order[at - 1]].Ra * pp.ph[order[at - 1]].Sb < g.Ra * g.Sb; --at) order[at] = order[at - 1];
    order[at] = i;
  }
  const int tm = p.bm, tn = p.bm == 64 ? 192 : 128;
  TriClassFilterArgs f;
  TriClasses t;
  f.w = w; f.wt = wt; f.soff = soff; f.groups = p.groups; f.C = d.C; f.K = d.K; f.R = d.R; f.S = d.S; f.st = d.st; f.Wp = pp.Wp; f.count = count;
  t.count = count; t.tiles_m = cdiv(d.C, tm); t.slab = (long long)(pp.sub_bytes / sizeof(float));
  int groups = 0, tiles = 0;
  double flops = 0.0;
  for (int q = 0; q < count; ++q) {
    const PhaseGeom& g = pp.ph[order[q]];
    TriClassFilter& c = f.c[q];
    c.first = groups; c.groups_true = d.K / 8 * g.Ra * g.Sb; c.groups = round_up(c.groups_true, 2);
    c.a = order[q] / d.st; c.b = order[q] % d.st; c.Ra = g.Ra; c.Sb = g.Sb;
    TriClass& k = t.c[q];
    k.first_tile = tiles; k.steps = c.groups / 2; k.groups_true = c.groups_true;
    k.inner = g.U * g.V; k.innerW = g.V; k.cols = d.N * k.inner;
    k.wt_at = (uint32_t)(48 * (size_t)groups * d.C);
    k.img_at = (uint32_t)(16 * ((size_t)(g.u0 + pp.L - (g.Ra - 1)) * (d.K / 8) * pp.Wp + (size_t)(g.v0 + pp.L - (g.Sb - 1))));
    k.soff_at = groups;
    k.out_at = g.sub_off;
    groups += c.groups;
    k.tiles = t.tiles_m * cdiv(k.cols, tn);
    k.slice_steps = cdiv(k.steps, p.slices[order[q]]);
    tiles += k.tiles * cdiv(k.steps, k.slice_steps);
    flops += 12.0 * (double)d.C * k.cols * d.K * g.Ra * g.Sb;
  }
  if (groups != p.groups) return RH_E_INVALID;
  const size_t img_groups = (size_t)d.N * (d.K / 8) * pp.Hp * pp.Wp;
  {
    const unsigned img_blocks = (unsigned)cdiv<size_t>(img_groups, 256);
    ProfScope prof("tri_image", 4.0 * (double)d.y_elems + 48.0 * (double)img_groups, stream);
    hipLaunchKernelGGL(tri_image_kernel, dim3(img_blocks), dim3(256), 0, stream, dy, xt, (unsigned)img_groups, d.P, d.Q,
                       FastDiv((uint32_t)pp.Wp), FastDiv((uint32_t)(d.K / 8)), FastDiv((uint32_t)pp.Hp), pp.L, (int)img_blocks, TriFilterArgs{});
  }
  if (int e = launch_status()) return e;
  hipLaunchKernelGGL(tri_class_filter_kernel, dim3((unsigned)cdiv<long long>((long long)groups * d.C, 256)), dim3(256), 0, stream, f);
  if (int e = launch_status()) return e;
  TriParams ap, bp;
  ap.v.ptr = wt; ap.plane = 0; ap.v.bytes = 0;   // (a class's)
  ap.v.M = d.C; ap.v.inner = 1; ap.v.innerW = 1; ap.v.img_stride = 16; ap.v.a_stride = 0; ap.v.b_stride = 0;
  ap.v.soff = nullptr; ap.v.group_stride = d.C * 16;
  bp.v.ptr = xt; bp.plane = (int)(16 * img_groups); bp.v.bytes = (uint32_t)(48 * img_groups);
  bp.v.M = 0; bp.v.inner = 1; bp.v.innerW = 1;
  bp.v.img_stride = pp.Hp * pp.Wp * d.K * 2; bp.v.a_stride = (d.K / 8) * pp.Wp * 16; bp.v.b_stride = 16;
  bp.v.soff = soff; bp.v.group_stride = 0;
  EpiParams ep;
  ep.out = *sub; ep.bias = nullptr; ep.alpha = 1.0f; ep.beta = 0.0f;
  ep.rows = d.C; ep.cols = 0; ep.inner = 1; ep.ld = 0; ep.relu = 0; ep.split_stride = 0;
  auto launch = [&](auto* tag, auto tile) -> int {
    typedef decltype(tile) T;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&mfma_gemm_tri_classes_kernel<T>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, kTriLdsBytes);
    if (attr != hipSuccess) return (int)attr;
    ProfScope prof(tag, flops, stream);
    hipLaunchKernelGGL((mfma_gemm_tri_classes_kernel<T>), dim3((unsigned)tiles), dim3(T::NT), kTriLdsBytes, stream, ap, bp, ep, t);
    return launch_status();
  };
  switch (p.bm) {
    case 128: return launch("conv_bwd_data_tri_128x128", T128x128t());
    case 96: return launch("conv_bwd_data_tri_96x128", T96x128t());
    default: return launch("conv_bwd_data_tri_64x192", T64x192t());
  }
}

TriFilterPlan plan_tri_bwd_filter(const ConvDims& d, bool wide) {
  TriFilterPlan p = {};
  p.wide = wide;
  if (d.P <= 0 || d.Q <= 0) return p;
  p.Hp = d.H + 2 * d.pad; p.Wp = d.W + 2 * d.pad;
  p.n8 = cdiv(d.N, 8);
  const long long groups = (long long)p.n8 * d.P * d.Q;
  p.groups_true = (int)groups;
  p.groups = round_up(p.groups_true, 2);
  const size_t dy_part = 16 * (size_t)p.groups * d.K, x_part = 16 * (size_t)p.n8 * p.Hp * p.Wp * d.C;
  if (3 * dy_part > kMaxBufferBytes || 3 * x_part > kMaxBufferBytes) return p;
  p.tab_bytes = align256(sizeof(int) * (size_t)p.groups);
  p.dyt_bytes = align256(3 * dy_part);
  p.xt_bytes = align256(3 * x_part);
  p.bm = pick_bm(d.K);
  if (p.bm == 32) p.bm = 64;
  p.bn = p.bm == 64 ? 192 : 128;
  const int CRS = d.C * d.R * d.S, tiles = cdiv(d.K, p.bm) * cdiv(CRS, p.bn), steps = p.groups / 2;
  // slices: two blocks to a CU where there are (0.445 us a K step of 128 x 128), their partial sums written and read (a fit to
  // 1859 timed calls; 11664 steps of 38 tiles: 13 slices 1031 us, 6, which leave 28 CUs idle, 1171)
  // (the wide form's K steps take 1.07 and 1.14 times as long, 64-row and other tiles; priced as plain ones, since with those factors
  // 64 -> 128 56x56 stride 2 at batch 32 and 50 go to a form of 76 and 109 us where this one takes 57 and 81; of 83 calls of
  // ResNet-18's layers that come here four are slower than the form replaced: 256 -> 256 14x14 at 90, 128 and 256 images by 0 to 6 %,
  // 256 -> 512 at one image 34 -> 36 us)
  p.us = 1e30;
  for (int want = 1; want <= 256 && (want == 1 || (want * 8 <= steps && (long long)tiles * want <= 1024)); ++want) {
    const int n = cdiv(steps, want), S = cdiv(steps, n);
    if (S != want || 4.0 * (double)S * (double)d.w_elems > 256e6) continue;
    const long long k = cdiv<long long>((long long)tiles * S, 256);
    const double us = (k == 1 ? n * (p.bm == 128 ? 0.47 : 0.38) : (double)k * n * (p.bm == 128 ? 0.445 : 0.375)) + 0.065 * S +
                      4.0 * (double)d.w_elems * (S + 1) / 2.2e6;
    if (us < p.us) { p.us = us; p.splits = S; }
  }
  if (p.splits == 0) p.splits = 1;   // (one slab is past the limit: not taken by itself, but whole where the flags ask for it)
  p.us += 15.0 + (4.0 * (double)(d.x_elems + d.y_elems) + 3.0 * (double)(dy_part + x_part)) / 5.3e6;
  p.part_bytes = align256(sizeof(float) * (size_t)p.splits * (size_t)d.w_elems);
  p.sum_rows = p.n8 * cdiv(d.P * d.Q, kTriPix);
  p.sum_bytes = align256(sizeof(float) * (size_t)p.sum_rows * d.K);
  p.ok = true;
  return p;
}

// What the copies of a filter gradient's operands are made from, and the operands that they are.
struct TriFilterSetup {
  TriBatchArgs dy, x;
  TriTableArgs table;
  TriParams ap, bp;
  float* parts;
};
static TriFilterSetup tri_filter_setup(const ConvDims& d, const TriFilterPlan& p, const float* x, const float* dy, float* sums, void* ws) {
  TriFilterSetup s;
  char* base = static_cast<char*>(ws);
  uint4* dyt = reinterpret_cast<uint4*>(base + p.tab_bytes);
  uint4* xt = reinterpret_cast<uint4*>(base + p.tab_bytes + p.dyt_bytes);
  s.parts = reinterpret_cast<float*>(base + p.tab_bytes + p.dyt_bytes + p.xt_bytes);
  const size_t dy_plane = (size_t)p.groups * d.K, x_plane = (size_t)p.n8 * p.Hp * p.Wp * d.C;
  TriBatchArgs &a = s.dy, &b = s.x;
  a.x = dy; a.xt = dyt; a.N = d.N; a.C = d.K; a.H = d.P; a.W = d.Q; a.halo = 0; a.HpWp = d.P * d.Q; a.dWp = FastDiv((uint32_t)d.Q);
  a.plane = dy_plane; a.px = cdiv(a.HpWp, kTriPix); a.cx = cdiv(a.C, kTriCh); a.blocks = a.px * a.cx * p.n8; a.sums = sums; a.wide = p.wide;
  b.x = x; b.xt = xt; b.N = d.N; b.C = d.C; b.H = d.H; b.W = d.W; b.halo = d.pad; b.HpWp = p.Hp * p.Wp; b.dWp = FastDiv((uint32_t)p.Wp);
  b.plane = x_plane; b.px = cdiv(b.HpWp, d.C <= kTriFew ? kTriFewPix : kTriPix); b.cx = cdiv(b.C, kTriCh); b.blocks = b.px * b.cx * p.n8; b.sums = nullptr; b.wide = false;
  s.table = TriTableArgs{reinterpret_cast<int*>(base), p.groups, p.groups_true, d.P * d.Q, d.Q, d.st, p.Wp, cdiv(p.groups, 256)};
  TriParams &ap = s.ap, &bp = s.bp;
  ap.v.ptr = dyt; ap.plane = (int)(16 * dy_plane); ap.v.bytes = (uint32_t)(48 * dy_plane);
  ap.v.M = d.K; ap.v.inner = 1; ap.v.innerW = 1; ap.v.img_stride = 16; ap.v.a_stride = 0; ap.v.b_stride = 0;
  ap.v.soff = nullptr; ap.v.group_stride = d.K * 16;
  bp.v.ptr = xt; bp.plane = (int)(16 * x_plane); bp.v.bytes = (uint32_t)(48 * x_plane);
  bp.v.M = d.C * d.R * d.S; bp.v.inner = d.S * d.C; bp.v.innerW = d.C;   // rows j = (r, s, c)
  bp.v.img_stride = p.Wp * d.C * 16; bp.v.a_stride = d.C * 16; bp.v.b_stride = 16;
  bp.v.soff = s.table.soff; bp.v.group_stride = 0;
  return s;
}

int launch_tri_rest_copies(const ConvDims& d, const TriFilterPlan& p, const float* x, const float* dy, void* ws, const int* any,
                           hipStream_t stream, TriRest* rest) {
  const TriFilterSetup s = tri_filter_setup(d, p, x, dy, nullptr, ws);
  const int bm = p.bm == 128 ? 128 : p.bm == 96 ? 96 : 64, bn = bm == 64 ? 192 : 128, blocks = s.dy.blocks + s.x.blocks + s.table.blocks;
  rest->any = any; rest->ap = s.ap; rest->bp = s.bp;
  rest->tiles_m = cdiv(d.K, bm);
  rest->tiles = rest->tiles_m * cdiv(d.C * d.R * d.S, bn);
  rest->k_steps = p.groups / 2;
  rest->steps_per_split = cdiv(rest->k_steps, p.splits);
  rest->splits = cdiv(rest->k_steps, rest->steps_per_split);
  rest->groups = p.groups_true;
  ProfScope prof("tri_rest", 0.0, stream);
  hipLaunchKernelGGL(tri_rest_batch_kernel, dim3((unsigned)(blocks < 512 ? blocks : 512)), dim3(256), 0, stream, s.dy, s.x, s.table, any);
  return launch_status();
}

int launch_conv_tri_bwd_filter(const ConvDims& d, const TriFilterPlan& p, const float* x, const float* dy, float* sums, void* ws,
                               hipStream_t stream, float** parts, int* used) {
  const TriFilterSetup s = tri_filter_setup(d, p, x, dy, sums, ws);
  *parts = s.parts;
  {
    ProfScope prof("tri_batch", 4.0 * (double)(d.y_elems + d.x_elems) + 48.0 * (double)(s.dy.plane + s.x.plane), stream);
    hipLaunchKernelGGL(tri_batch_kernel, dim3((unsigned)(s.dy.blocks + s.x.blocks + s.table.blocks)), dim3(256), 0, stream, s.dy, s.x, s.table);
  }
  if (int e = launch_status()) return e;
  const TriParams &ap = s.ap, &bp = s.bp;
  const int CRS = d.C * d.R * d.S;
  EpiParams ep;
  ep.out = *parts; ep.bias = nullptr; ep.alpha = 1.0f; ep.beta = 0.0f;
  ep.rows = d.K; ep.cols = CRS; ep.inner = 0; ep.ld = CRS; ep.relu = 0; ep.split_stride = (long long)d.K * CRS;
  const double flops = (p.wide ? 14.0 : 12.0) * (double)d.w_elems * d.N * d.P * d.Q;
  const int steps = p.groups / 2;
#define RH_TRI(TILE, TAG)                                                                                              \
  (p.wide ? launch_tri<TILE, false, false, PassConvBwdFilter, true>(ap, bp, ep, steps, p.groups_true, p.splits, used, flops, stream, \
                                                                    "conv_bwd_filter_tri_wide_" TAG)                                 \
          : launch_tri<TILE, false, false, PassConvBwdFilter>(ap, bp, ep, steps, p.groups_true, p.splits, used, flops, stream,       \
                                                              "conv_bwd_filter_tri_" TAG))
  switch (p.bm) {
    case 128: return RH_TRI(T128x128t, "128x128");
    case 96: return RH_TRI(T96x128t, "96x128");
    default: return RH_TRI(T64x192t, "64x192");
  }
#undef RH_TRI
}

}  // namespace rh

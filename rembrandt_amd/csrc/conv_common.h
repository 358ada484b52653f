// Host-side helpers shared by the three convolution passes.
#pragma once
#include <math.h>
#include <stdlib.h>

#include "gemm_core.h"

namespace rh {

inline int conv_out_dim(int in, int size, int stride, int pad) {
  int t = in + 2 * pad - size + stride;
  if (t < 0) t = 0;
  return t / stride;
}

inline size_t align256(size_t v) { return (v + 255) & ~size_t(255); }
inline int round_up(int v, int m) { return (v + m - 1) / m * m; }

// Contraction tables are padded to a multiple of this many entries (>= every BK in use).
constexpr int kTabPad = 64;
// Readable bytes kept after an operand that LoadRow4 reads: its last group of four rows may begin at the last valid row.
constexpr size_t kRow4Slack = 16;

struct ConvDims {
  int N, C, H, W, K, R, S, st, pad, P, Q;
  long long x_elems, w_elems, y_elems;
};

inline int conv_dims(const rh_conv_geom* g, ConvDims* d) {
  if (!g) return RH_E_INVALID;
  if (g->N <= 0 || g->C <= 0 || g->H <= 0 || g->W <= 0 || g->K <= 0 || g->R <= 0 || g->S <= 0 ||
      g->stride <= 0 || g->pad < 0)
    return RH_E_INVALID;
  d->N = g->N; d->C = g->C; d->H = g->H; d->W = g->W; d->K = g->K; d->R = g->R; d->S = g->S;
  d->st = g->stride; d->pad = g->pad;
  d->P = conv_out_dim(g->H, g->R, g->stride, g->pad);
  d->Q = conv_out_dim(g->W, g->S, g->stride, g->pad);
  d->x_elems = (long long)g->N * g->C * g->H * g->W;
  d->w_elems = (long long)g->K * g->C * g->R * g->S;
  d->y_elems = (long long)g->N * g->K * d->P * d->Q;
  if ((size_t)d->x_elems * 4 > kMaxBufferBytes || (size_t)d->y_elems * 4 > kMaxBufferBytes ||
      (size_t)d->w_elems * 4 > kMaxBufferBytes)
    return RH_E_LIMIT;
  return 0;
}

// Row-tile height with the least zero padding for `rows` result rows; ties go to the taller tile.
inline int pick_bm(int rows) {
  const int cand[4] = {128, 96, 64, 32};
  int best = 128;
  long long best_pad = -1;
  for (int i = 0; i < 4; ++i) {
    const long long padded = (long long)round_up(rows, cand[i]);
    if (best_pad < 0 || padded < best_pad) { best_pad = padded; best = cand[i]; }
  }
  return best;
}

template <class T, class AL, class BL, bool NCHW, class PASS>
inline int launch_mfma_gemm(const typename AL::Params& ap, const typename BL::Params& bp,
                            const EpiParams& ep, int K, int splits, int* splits_used,
                            hipStream_t stream, const char* tag, int k_algorithmic = 0) {
  const int tiles_m = cdiv(ep.rows, T::BM), tiles_n = cdiv(ep.cols, T::BN);
  const int k_chunks = cdiv(K, T::BK);
  if (ep.tail_tiles > 0) splits = ep.tail_splits;  // tail form: the slices apply to the last tail_tiles tiles only
  if (splits < 1) splits = 1;
  const int cps = cdiv(k_chunks, splits) > 0 ? cdiv(k_chunks, splits) : 1;
  const int used = cdiv(k_chunks, cps) > 0 ? cdiv(k_chunks, cps) : 1;
  if (splits_used) *splits_used = used;
  dim3 grid((unsigned)(tiles_m * tiles_n), (unsigned)used);
  if (ep.tail_tiles > 0) {
    if (used != ep.tail_splits || ep.full_tiles + ep.tail_tiles != tiles_m * tiles_n) return RH_E_INVALID;
    grid = dim3((unsigned)(ep.full_tiles + ep.tail_tiles * ep.tail_splits), 1u);
  }
  constexpr size_t lds_bytes = sizeof(float) * 2 * T::BK * (AL::LD + BL::LD);
  static_assert(lds_bytes <= 160 * 1024, "tile does not fit the 160 KB LDS of a CU");
  if (lds_bytes > 48 * 1024) {
    // opt in to more than the default dynamic LDS limit, once per kernel instantiation
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void*>(&mfma_gemm_kernel<T, AL, BL, NCHW, PASS>),
        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
    if (attr != hipSuccess) return (int)attr;
  }
  ProfScope prof(tag, 2.0 * (double)ep.rows * (double)ep.cols * (double)(k_algorithmic > 0 ? k_algorithmic : K), stream);
  hipLaunchKernelGGL((mfma_gemm_kernel<T, AL, BL, NCHW, PASS>), grid, dim3(T::NT), lds_bytes, stream, ap, bp, ep,
                     tiles_m, k_chunks, cps);
  return launch_status();
}

// Same grid and split logic for the bf16-operand kernel.  FLOPs are counted as for fp32.
template <class T, class AL, class BL, bool NCHW, class PASS>
inline int launch_mfma_gemm_bf16(const typename AL::Params& ap, const typename BL::Params& bp,
                                 const EpiParams& ep, int K, int splits, int* splits_used,
                                 hipStream_t stream, const char* tag, int k_algorithmic = 0) {
  const int tiles_m = cdiv(ep.rows, T::BM), tiles_n = cdiv(ep.cols, T::BN);
  const int k_chunks = cdiv(K, T::BK);
  if (splits < 1) splits = 1;
  const int cps = cdiv(k_chunks, splits) > 0 ? cdiv(k_chunks, splits) : 1;
  const int used = cdiv(k_chunks, cps) > 0 ? cdiv(k_chunks, cps) : 1;
  if (splits_used) *splits_used = used;
  dim3 grid((unsigned)(tiles_m * tiles_n), (unsigned)used);
  constexpr size_t lds_bytes = 16 * 2 * (T::BK / 8) * (T::BM + T::BN);
  static_assert(lds_bytes <= 160 * 1024, "tile does not fit the 160 KB LDS of a CU");
  if (lds_bytes > 48 * 1024) {
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void*>(&mfma_gemm_bf16_kernel<T, AL, BL, NCHW, PASS>),
        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
    if (attr != hipSuccess) return (int)attr;
  }
  ProfScope prof(tag, 2.0 * (double)ep.rows * (double)ep.cols * (double)(k_algorithmic > 0 ? k_algorithmic : K), stream);
  hipLaunchKernelGGL((mfma_gemm_bf16_kernel<T, AL, BL, NCHW, PASS>), grid, dim3(T::NT), lds_bytes, stream, ap, bp, ep,
                     tiles_m, k_chunks, cps);
  return launch_status();
}

// The direct-to-LDS form for packed operands (one pass over the whole contraction).
template <class T, bool A_LINEAR, bool B_LINEAR, bool NCHW, class PASS, bool PK = false, int R = 4, int KS = 1>
inline int launch_mfma_gemm_bf16_dma(const RowV8Params& ap, const RowV8Params& bp, const EpiParams& ep, int K,
                                     hipStream_t stream, const char* tag, int k_algorithmic = 0,
                                     const PackedOut& pk = PackedOut()) {
  const int tiles_m = cdiv(ep.rows, T::BM), tiles_n = cdiv(ep.cols, T::BN);
  if (K <= 0 || K % T::BK != 0) return RH_E_INVALID;
  constexpr size_t lds_bytes = bf16_dma_lds_bytes(T::BM, T::BN, T::BK, R, KS);
  static_assert(lds_bytes * T::OCC * 4 / (T::NT / kWave * KS) <= 160 * 1024, "the blocks meant to share a CU do not fit its 160 KB of LDS");
  if (lds_bytes > 48 * 1024) {
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void*>(&mfma_gemm_bf16_dma_kernel<T, A_LINEAR, B_LINEAR, NCHW, PASS, PK, R, KS>),
        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
    if (attr != hipSuccess) return (int)attr;
  }
  ProfScope prof(tag, 2.0 * (double)ep.rows * (double)ep.cols * (double)(k_algorithmic > 0 ? k_algorithmic : K), stream);
  if (PK && !pk.ptr) return RH_E_INVALID;
  hipLaunchKernelGGL((mfma_gemm_bf16_dma_kernel<T, A_LINEAR, B_LINEAR, NCHW, PASS, PK, R, KS>), dim3((unsigned)(tiles_m * tiles_n)),
                     dim3(T::NT * KS), lds_bytes, stream, ap, bp, ep, tiles_m, K / T::BK, pk);
  return launch_status();
}

#ifndef RH_OCC_128
#define RH_OCC_128 4
#endif
// Tile shapes in use.  rows x cols x k, waves as WM x WN.
typedef Tile<128, 128, 16, 2, 2, RH_OCC_128> T128x128;
typedef Tile<96, 256, 16, 1, 4> T96x256;
typedef Tile<96, 128, 16, 1, 4, 4> T96x128;
typedef Tile<96, 96, 16, 1, 3, 4> T96x96;   // three waves: a 96 x 96 result (1x1 layer, 96 -> 96 channels) without a quarter of dead columns
#ifndef RH_BF16_BK
#define RH_BF16_BK 32
#endif
#ifndef RH_BF16_OCC
#define RH_BF16_OCC 3
#endif
// bf16-operand kernel: a deeper K step keeps more operand loads in flight per wave (its MFMAs are 16x shorter)
typedef Tile<128, 128, RH_BF16_BK, 2, 2, RH_BF16_OCC> T128x128bf;
// Tile of the direct-to-LDS bf16 kernel: eight waves of 128x64 each, one block per CU, four 32-k LDS buffers.
typedef Tile<256, 256, 32, 2, 4, 1> T256x256bf;
typedef Tile<256, 128, 32, 2, 2, 2> T256x128bf;   // direct-to-LDS form with a ring of three: two blocks of four waves share a CU
typedef Tile<128, 256, 32, 2, 2, 2> T128x256bf;   // the same for filter counts that would waste rows of a 256-row tile
// The same loop for grids of few tiles (see bf16_small_form): smaller tiles, and groups of waves that share a tile's K steps.
typedef Tile<128, 128, 32, 2, 2, 3> T128x128bd;   // ring of three, three blocks per CU
typedef Tile<128, 128, 32, 2, 2, 2> T128x128bd2;  // two groups, one block per CU
typedef Tile<64, 128, 32, 2, 2, 4> T64x128bf;     // ring of three, four blocks per CU: up to 64 filters
typedef Tile<64, 64, 32, 2, 2, 4> T64x64bf;       // ring of four, two groups (two blocks per CU) or four (one)
typedef Tile<64, 256, 16, 1, 4, 3> T64x256;
typedef Tile<32, 256, 16, 1, 4, 3> T32x256;
// few result columns as well (a first layer's filter gradient: 20 x 25, 32 x 75): narrower tiles, fewer dead columns
typedef Tile<32, 128, 16, 1, 4, 4> T32x128;
typedef Tile<32, 64, 16, 1, 2, 4> T32x64;
typedef Tile<128, 64, 16, 2, 2, 4> T128x64;   // sliced forward contractions (small images late in a network)
typedef Tile<64, 128, 16, 1, 4, 4> T64x128;   // sliced forward / backward-data contractions of small layers
// Half the K step: 20 KB of LDS, so a CU holds 4 blocks instead of 3.  For grids that need a second round of
// blocks at 3 per CU but fit in one at 4 (e.g. 64 output channels over 64 x 56 x 56 pixels: 784 tiles).
typedef Tile<64, 256, 8, 1, 4, 4> T64x256k8;
// The kernel of gemm_tri.h: two blocks of four waves to a CU.
typedef Tile<128, 128, 16, 2, 2, 2> T128x128t;
typedef Tile<96, 128, 16, 1, 4, 2> T96x128t;
typedef Tile<64, 192, 16, 2, 2, 2> T64x192t;
typedef Tile<64, 256, 16, 1, 4, 2> T64x256t;   // gemm_duo.h
inline bool prefer_k8_64(long long cols) {
  const long long tiles = cdiv<long long>(cols, 256);
  return cdiv<long long>(tiles, 1024) < cdiv<long long>(tiles, 768);
}

// Columns of a block that adds up the rows of an [N][K] matrix: 64-byte reads, or of 32 where the rows are many.
__host__ __device__ constexpr int bias_rows_cols(int N) { return N > 512 ? 8 : 16; }

// Second pass of a split contraction: out[i*ld + j] = alpha * sum_s part[s][i*cols + j] + beta*out.
// A bias gradient that rides in a reduction's launch, in blocks of its own behind the reduction's (small layers are
// bound by the number of dependent launches): db[k] = alpha * sum over n and the plane of src[(n K + k) plane + i] +
// beta * db[k]; plane == 1: src is an [N][K] matrix (an affine layer's delta, or per-image plane sums).
struct BiasJob {
  const float* src = nullptr;
  float* db = nullptr;           // nullptr: no job
  int N = 0, K = 0, plane = 0;
  float alpha = 1.0f, beta = 0.0f;
  unsigned first = 0;            // the job's first block (filled in by the launcher)
  unsigned blocks() const { return !db ? 0u : plane == 1 ? (unsigned)cdiv(K, bias_rows_cols(N)) : (unsigned)K; }
};
void launch_split_reduce(const float* part, int splits, long long split_stride, float* out, int rows, int cols,
                         int ld, float alpha, float beta, hipStream_t stream, const float* bias_col = nullptr, int relu = 0,
                         const BiasJob* bias_job = nullptr);

// Tail form of a forward / backward-data launch (see EpiParams): when the tile count is not close to a multiple of
// the 256 CUs, the column tiles beyond the last multiple are cut into `splits` slices so that every CU ends up with
// nearly the same work, whether the CUs hold all tiles at once or take them in rounds.  splits == 1: not worth it.
struct TailSplit {
  int full_tiles, tail_tiles, splits;
  long long col0;  // first column of the tail
};
inline TailSplit plan_tail_split(int rows, long long cols, int n_k, int bn_force = 0) {
  TailSplit t = {0, 0, 1, 0};
  const int bm = pick_bm(rows), bn = bn_force ? bn_force : bm >= 96 ? 128 : 256;
  const int tiles_m = cdiv(rows, bm);
  const long long tiles_n = cdiv<long long>(cols, bn), T = tiles_m * tiles_n;
  const bool k8 = bm == 64 && tiles_m == 1 && prefer_k8_64(cols);  // the 64x256 tile with the halved K step: 4 per CU
  const long long slots = 256 * (bm >= 96 || k8 ? 4 : 3);
  if (T * 3 <= slots) return t;  // the whole-result split applies
  const long long full_cols = (T / 256 * 256) / tiles_m, full = full_cols * tiles_m, tail = T - full;
  if (tail == 0 || full == 0) return t;
  // Busiest CU in units of one tile's time: whole tiles + its pieces + the partial-sum traffic of those pieces
  // (a tile alone on a CU at ~0.47 TFLOP/s; a piece's slab written and read at a CU's share of ~4 TB/s).
  const double tile_us = 2.0 * bm * bn * (double)n_k / 0.47e6, piece_us = 8.0 * bm * bn / 15.6e3;
  const int k_chunks = n_k / 16;
  double best = (double)cdiv<long long>(T, 256);
  // modelled gain asked for: 7 % when all tiles are resident at once, 2.5 % when the CUs take tiles in several rounds
  // (measured: 1568 tiles 0.511 -> 0.454 ms, 2916 tiles 1.94 -> 1.87 ms, 3136 tiles 0.505 -> 0.478 ms)
  const double need = (T > slots ? 0.975 : 0.93) * best;
  for (int S = 2; S <= 16 && S * 8 <= k_chunks; ++S) {
    if (k_chunks % S != 0) continue;  // equal slices, for the 16- and the 8-deep K step alike
    const long long pieces = cdiv<long long>(tail * S, 256);
    const double cost = (double)cdiv<long long>(full, 256) + (double)pieces / S + pieces * piece_us / tile_us;
    if (cost < best && cost <= need) { best = cost; t.splits = S; }
  }
  if (t.splits > 1) { t.full_tiles = (int)full; t.tail_tiles = (int)tail; t.col0 = full_cols * bn; }
  return t;
}
// First element of the NCHW result that a tail column can touch: the start of the image that holds column col0.
// The partial slabs of the tail form hold the result from there on.
inline long long tail_first_elem(const TailSplit& t, long long inner, long long rows) {
  return t.splits > 1 && inner > 0 ? (t.col0 / inner) * rows * inner : 0;
}

// Scratch layout of the scalar-offset forward / backward-data paths:
//   [k -> byte offset table : n_k ints][transposed filter : n_k x rows floats][padded image copy]
struct SoffPlan {
  int n_k;         // contraction length rounded up to kTabPad
  int Hp, Wp;      // padded image extent
  int halo;        // zeros added on each side
  size_t tab_bytes, wt_bytes, img_bytes;  // img_bytes == 0: the image is used in place
  int splits;      // > 1: the contraction is cut into this many slices, partial results in part_bytes of scratch
  TailSplit tail;  // tail.splits > 1: only the last tiles are cut (splits == 1 then)
  bool narrow128 = false;  // forward, 128-row tiles: the 128 x 64 tile, planned as such
  size_t part_bytes;
  bool ok;         // false: fall back to the per-element gather path
  size_t total() const { return tab_bytes + wt_bytes + img_bytes + part_bytes; }
};

// A forward / backward-data launch whose tiles would occupy under half of the block slots the GPU holds at a time
// (small images late in a network, small batches) cuts the contraction into slices so that the slots fill; every
// slice keeps at least 16 K steps.  Partial results go to scratch slabs shaped like the output and are added in a
// fixed order by split_reduce_nchw.  Returns the slice count (1: no split).
// How many slices the depth of a contraction allows: every slice keeps `normal_min` K steps, so that prologue and
// partial-sum traffic stay small next to it.  Where even that many slices leave three quarters of the block slots
// empty (the layers of a small network at a small batch) a block's chain of K steps, each a memory round trip, is
// what the kernel takes, and the slices go down to `small_min` steps.
inline long long slices_by_depth(long long k_steps, long long tiles, long long slots, int normal_min, int small_min) {
  long long by = k_steps / normal_min;
  if (by < 1) by = 1;
  if (tiles * by * 4 <= slots) by = k_steps / small_min;
  return by < 1 ? 1 : by;
}

inline int plan_k_split(int rows, long long cols, int n_k, int bn_force = 0) {
  const int bm = pick_bm(rows), bn = bn_force ? bn_force : bm >= 96 ? 128 : 256;
  const long long slots = 256 * (bm >= 96 ? 4 : 3);
  const long long tiles = (long long)cdiv(rows, bm) * cdiv<long long>(cols, bn);
  if (tiles == 0 || tiles * 2 > slots) return 1;
  long long want = slots / tiles;
  const long long by_depth = slices_by_depth(n_k / 16, tiles, slots, 16, 4);
  if (want > by_depth) want = by_depth;
  if (want > 16) want = tiles * 64 <= slots ? (want > 32 ? 32 : want) : 16;
  return want < 3 ? 1 : (int)want;   // two slices only trade one round of blocks for the partial-sum traffic
}

// A batch norm at inference behind a forward pass: y = relu?((x - mean[k]) scale[k] ivar[k] + bias[k] + beta old), by the expressions of
// bn_infer_kernel.  A pass whose whole result comes out of the reduction of slices has it formed there and says so in `done`: the
// result x is written as without it.
struct BnInfer {
  const float *mean, *ivar, *scale, *bias, *old;
  float* y;
  float alpha, beta;
  int relu;
};
struct BnInferJob { BnInfer bn; bool done; };

// out[i] = alpha * sum_s part[s*stride + i] + beta*out[i] (+ bias[channel], ReLU) over an NCHW tensor of `total`
// elements, channel = (i / inner) % rows; only elements whose column (image * inner + pixel) is >= col0.
void launch_split_reduce_nchw(const float* part, int splits, long long stride, float* out, long long total, int inner,
                              int rows, float alpha, float beta, const float* bias, int relu, hipStream_t stream,
                              long long col0 = 0, const float* mask = nullptr, BnInferJob* bn = nullptr);


// Slices that the direct form cuts the contraction of a forward / stride-1 backward-data call into.
inline int soff_splits_fwd(const ConvDims& d, int n_k) {
  const long long cols = (long long)d.N * d.P * d.Q;
  const int s = plan_k_split(d.K, cols, n_k);
  return pick_bm(d.K) == 128 && s > 1 ? plan_k_split(d.K, cols, n_k, 64) : s;
}
inline int soff_splits_bwd_data(const ConvDims& d, int n_k) {
  const long long cols = (long long)d.N * d.H * d.W;
  const int s = plan_k_split(d.C, cols, n_k);
  return pick_bm(d.C) == 128 && s > 1 && plan_k_split(d.C, cols, n_k, 64) == 1 ? 1 : s;
}

inline SoffPlan plan_soff_fwd(const ConvDims& d) {
  SoffPlan p;
  p.n_k = round_up(d.C * d.R * d.S, kTabPad);
  p.halo = d.pad;
  p.Hp = d.H + 2 * d.pad;
  p.Wp = d.W + 2 * d.pad;
  p.tab_bytes = align256(sizeof(int) * (size_t)p.n_k);
  p.wt_bytes = align256(sizeof(float) * (size_t)p.n_k * d.K + kRow4Slack);
  const size_t img = sizeof(float) * (size_t)d.N * d.C * p.Hp * p.Wp;
  p.img_bytes = d.pad > 0 ? align256(img) : 0;
  p.ok = img <= kMaxBufferBytes && d.P > 0 && d.Q > 0;
  p.splits = soff_splits_fwd(d, p.n_k);
  p.tail = plan_tail_split(d.K, (long long)d.N * d.P * d.Q, p.n_k);
  if (pick_bm(d.K) == 128 && plan_k_split(d.K, (long long)d.N * d.P * d.Q, p.n_k) > 1) {
    // Few 128 x 128 tiles (small images late in a network): the half-width tile, planned as such.  Twice the tiles often
    // need no slices any more, only a cut of the tiles past the last multiple of 256 (NIN's 1024-channel layers on
    // 6 x 6: 576 tiles = 512 + 64 in eight slices, instead of 288 x 3 with a reduction over the whole result).
    p.narrow128 = true;
    p.tail = plan_tail_split(d.K, (long long)d.N * d.P * d.Q, p.n_k, 64);
  }
  const size_t tail_elems_f = (size_t)(d.y_elems - tail_first_elem(p.tail, (long long)d.P * d.Q, d.K));
  p.part_bytes = p.splits > 1 ? align256(sizeof(float) * (size_t)p.splits * (size_t)d.y_elems)
               : p.tail.splits > 1 ? align256(sizeof(float) * (size_t)p.tail.splits * tail_elems_f) : 0;
  return p;
}

// Backward-data with stride 1: dx[n,c,h,w] = sum dyp[n,ko,h+R-1-r,w+S-1-s] * w[ko,c,r,s] on dy padded
// by R-1-pad zeros per side.
// Backward-data as a stride-1 correlation of the flipped filter with dy.  For stride > 1 the padded copy of dy is
// also dilated (dy[p][q] lands on [halo + st*p][halo + st*q], zeros between): the contraction then multiplies
// (st^2 - 1)/st^2 zeros, but runs on the scalar-offset loaders; the copy is (H + R - 1) x (W + S - 1) per plane.
inline SoffPlan plan_soff_bwd_data(const ConvDims& d) {
  SoffPlan p;
  p.n_k = round_up(d.K * d.R * d.S, kTabPad);
  p.halo = d.R - 1 - d.pad;
  p.Hp = d.H + d.R - 1;   // = P + 2*halo when the stride is 1
  p.Wp = d.W + d.S - 1;
  p.tab_bytes = align256(sizeof(int) * (size_t)p.n_k);
  p.wt_bytes = align256(sizeof(float) * (size_t)p.n_k * d.C);
  const size_t img = p.halo >= 0 ? sizeof(float) * (size_t)d.N * d.K * p.Hp * p.Wp : 0;
  p.img_bytes = (p.halo > 0 || d.st > 1 || p.Hp != d.P || p.Wp != d.Q) ? align256(img) : 0;
  p.ok = p.halo >= 0 && d.R == d.S && img <= kMaxBufferBytes && d.P > 0 && d.Q > 0;
  p.splits = soff_splits_bwd_data(d, p.n_k);
  p.tail = plan_tail_split(d.C, (long long)d.N * d.H * d.W, p.n_k);
  if (pick_bm(d.C) == 128 && p.splits == 1 && plan_k_split(d.C, (long long)d.N * d.H * d.W, p.n_k) > 1) {
    // As in the forward pass, where 128 x 64 tiles need no slices (NIN's 1024-channel 1x1 layers: 0.120 -> 0.098 ms).
    // Where they would still be sliced the 128 x 128 tile stays (a 384-channel 3x3 layer on 6 x 6 lost 9 %).
    p.narrow128 = true;
    p.tail = plan_tail_split(d.C, (long long)d.N * d.H * d.W, p.n_k, 64);
  }
  if (d.st > 1) p.tail.splits = 1;  // the zero-dilated form is a fallback only
  const size_t tail_elems_b = (size_t)(d.x_elems - tail_first_elem(p.tail, (long long)d.H * d.W, d.C));
  p.part_bytes = p.splits > 1 ? align256(sizeof(float) * (size_t)p.splits * (size_t)d.x_elems)
               : p.tail.splits > 1 ? align256(sizeof(float) * (size_t)p.tail.splits * tail_elems_b) : 0;
  return p;
}

// Winograd F(2x2, 3x3) form of a 3x3 stride-1 layer (conv_wino.hip), written as a forward convolution: an input of
// (N, Ci, Hi, Wi) with `halo` zeros around it, Ko filters, a result of (N, Ko, P, Q).  Backward-data is the same over dy
// with halo 2 - pad.  Scratch: [U: transformed filter][V: transformed image patches].
constexpr int kWinoBM = 128, kWinoBM2 = 64, kWinoBN = 32, kWinoR = 3;
struct WinoGeom {
  int N, Ci, Hi, Wi, Ko, halo, P, Q, TP, TQ;
  int Cg;                     // groups of four input channels
  int bm;                     // rows of a tile: kWinoBM (one block per CU) or kWinoBM2 (two)
  int slots() const { return bm == kWinoBM ? 256 : 512; }
  int rows_p;                 // Ko rounded up to whole row tiles
  long long tiles, tiles_p;   // 2x2 output tiles; rounded up to whole column tiles
  size_t u_bytes, v_bytes;
  bool ok;
  bool fine;                  // no call of it loses more bits than the direct form's slices would (see wino_stages_at_most)
  double us;                  // what a call is expected to take
  double whole_us;            // the same with the tail form left out
  // (RH_ALGO_SHARED_GPU: other kernels fill the CUs that a last round leaves idle.  A grid under one round stays sliced:
  // its slices are how long the call is, with or without neighbours.)
  void beside_others() {
    if (full_tiles > 0) { tail_S = 1; us = whole_us; }
  }
  // Tail form (V made in the kernel only): the blocks past the last multiple of 256 (all of them where there are fewer) are cut into tail_S slices of the
  // channel loop, tail_L stages each, whose untransformed-blend partial results go to slabs of scratch that hold the
  // result from element part_first on (the first image a tail block touches); tail_S == 1: not worth it.
  int full_tiles, tail_S, tail_L;
  int chains;                 // into which the stages of a slice are divided, see wino_gemm_fused_kernel
  long long part_first, slab_elems;
  size_t part_bytes;
  // 5x5 forward (wino_geom_fwd5): the filter, extended with zeros to 6x6, is four 3x3 filters at offsets (3 bi, 3 bj);
  // the layer is the sum of their four 3x3 layers over shifted inputs, added in the transform domain: the same 16
  // products over 4 C "channels" (channel 4 c + 2 bi + bj = input channel c read 3 bi rows and 3 bj columns further
  // on): 64 multiply-adds per 2x2 outputs, filter and channel instead of 100.  Ci = 4 C here; the input is read from a
  // zero-bordered copy of Hp x Wp a plane (pad zeros in front, the rest behind), made in img_bytes of scratch.
  int blk5 = 0, C5 = 0, H5 = 0, W5 = 0, pad5 = 0;
  size_t img_bytes = 0;
  size_t total() const { return u_bytes + v_bytes + img_bytes + part_bytes; }
};
// 64-row tiles where 128-row ones would execute an eighth more rows at least (64 filters, 192, 320): row for row they are a
// tenth slower (384 -> 384 13x13 b256 601 us against 532), with half of the rows empty the larger tile takes 655 us on
// 64 -> 64 56x56 b256 where the smaller takes 382 and the direct form 572.
inline int wino_bm(int Ci, int Ko, int blk5) {
  return Ci % 4 == 0 && !blk5 && round_up(Ko, kWinoBM2) * 9 <= round_up(Ko, kWinoBM) * 8 ? kWinoBM2 : kWinoBM;
}
// Stages in a chain of which the form's error against 64 bits is the direct form's at `splits` slices, for a result of
// P x Q with `halo` zeros around the input.  The form's relative rms error, squared, is 1.35 + 0.351 L in units of 1e-14 (L
// stages of four channels in a chain: 2.6e-7 at 16, 3.5e-7 at 32, 5.9e-7 at 96), the direct form's 0.0335 a term that lies on
// the image (2.8e-7 at 256, 4.2e-7 at 576 on 13 x 13).  A direct form that is not sliced has the longer chain at any size.
// Terms on the border add nothing to the result nor to the direct form's error, but the transforms mix them in: with even
// extents, whose tiles end with the result, 0.173 + 0.176 over the share of live terms a stage (0.354 on 28 x 28, 0.392 on
// 6 x 6).  (Without that share 384 -> 1024 6x6 batch 40 took one chain of 48 stages, 4.50e-7 against 4.34e-7 in the direct
// form's five slices; in two chains 3.3e-7, for 2 % of its time.)
inline int wino_stages_at_most(int Ci, int splits, int P, int Q, int halo) {
  if (splits <= 1 || P <= 0 || Q <= 0) return cdiv(Ci, 4);
  const double dead = halo * (halo + 1) / 3.0, live = (1.0 - dead / P) * (1.0 - dead / Q);
  const double stage = P % 2 == 0 || Q % 2 == 0 ? 0.173 + 0.176 / fmax(live, 0.1) : 0.351;
  return (int)((0.0335 * live * 9.0 * Ci / splits - 1.35) / stage);
}
// max_L: the stages in a chain up to which a call counts as fine; it is made of such chains where that can be.
WinoGeom wino_geom(int N, int Ci, int Hi, int Wi, int Ko, int halo, int max_L, int blk5 = 0);
inline bool wino_shape(const ConvDims& d) { return d.R == 3 && d.S == 3 && d.st == 1 && d.pad <= 2; }
inline bool wino_shape5(const ConvDims& d) { return d.R == 5 && d.S == 5 && d.st == 1 && d.pad <= 4 && d.P > 0 && d.Q > 0; }
// (5x5: 5.3e-7 unsliced on 96 channels, 5.0e-7 with a tail of six slices, the unsliced direct form 8.5e-7, three slices 4.9e-7)
inline WinoGeom wino_geom_fwd5(const ConvDims& d) {
  return wino_geom(d.N, d.C, d.H, d.W, d.K, d.pad, soff_splits_fwd(d, round_up(d.C * 25, kTabPad)) <= 1 ? 4 * d.C : 0, 1);
}
inline WinoGeom wino_geom_fwd(const ConvDims& d) {
  return wino_geom(d.N, d.C, d.H, d.W, d.K, d.pad, wino_stages_at_most(d.C, soff_splits_fwd(d, round_up(d.C * 9, kTabPad)), d.P, d.Q, d.pad));
}
inline WinoGeom wino_geom_bwd_data(const ConvDims& d) {
  return wino_geom(d.N, d.K, d.P, d.Q, d.C, 2 - d.pad, wino_stages_at_most(d.K, soff_splits_bwd_data(d, round_up(d.K * 9, kTabPad)), d.H, d.W, 2 - d.pad));
}
// Filter gradient in the same form: zero-bordered copies of x and dy, S slices of the tiles, their partial sums.
struct WinoFilterPlan {
  bool ok;
  int TP, TQ, Kp, Cp, S, stages;   // S slices of `stages` tile groups (of four tiles) each
  long long tiles, TGs;            // tiles; tile groups over all slices
  size_t vt_bytes, dyt_bytes, part_bytes;
  size_t total() const { return vt_bytes + dyt_bytes + part_bytes; }
};
WinoFilterPlan plan_wino_bwd_filter(const ConvDims& d);
// Where the library takes it by itself: as for the other two passes, and few enough slices for their traffic not to matter.
inline bool wino_filter_pays(const ConvDims& d, const WinoFilterPlan& p) {
  return p.ok && d.C >= 64 && d.K >= 64 && 4 * d.K >= 3 * p.Kp && 4 * d.C >= 3 * p.Cp && p.tiles >= 4096 &&
         (long long)(p.Kp / kWinoBM) * (p.Cp / kWinoBN) * p.S >= 192;
}
int launch_conv_wino_bwd_filter(const ConvDims& d, const WinoFilterPlan& p, const float* x, const float* dy, float* dw, float alpha,
                                float beta, void* ws, hipStream_t stream);
int launch_conv_wino(const WinoGeom& g, bool bwd, const float* in, const float* w, float* out, float alpha, float beta,
                     const float* bias, int relu, const float* mask, void* ws, hipStream_t stream, const char* tag);

// Stride-1 layers with both operands staged in LDS as they lie in memory (conv_lds.hip), forward and backward-data.
constexpr int kLdsShapeCount = 6;
// Partial sums of a sliced call are at most this large (more would take longer than the slices save: 16 MB are 8 us), so
// that the workspace of a call is known without choosing its plan.
constexpr size_t kLdsMaxPart = size_t(16) << 20;
constexpr int kLdsMaxSlices = 32;
inline size_t lds_part_bytes(int R, int S, int st, long long out_elems) {
  if (R != S || (R != 3 && R != 5) || st != 1) return 0;
  const size_t most = kLdsMaxSlices * sizeof(float) * (size_t)out_elems;
  return align256(most < kLdsMaxPart ? most : kLdsMaxPart);
}
struct LdsConvPlan {
  bool ok;
  int shape, npos;       // tile shape; staged positions per channel
  int qps, splits;       // channel quads per slice of the contraction; slices
  double us;             // what a call is expected to take
};
// N images of Ci channels, `rows` result channels of P x Q.
LdsConvPlan plan_conv_lds(int N, int Ci, int rows, int P, int Q, int R, int S, int st);
// (Loads of the channels that a last stage has too many, fifteen at most, are out of range by the top bit of their offset:
// their planes have to lie below it too, or the offset would wrap into the first planes, whose infinities times the zero
// filter are no zeros.)
inline bool lds_fits(long long in_elems, int H, int W) { return (in_elems + 15ll * H * W) * 4 < (1ll << 31); }
inline LdsConvPlan plan_lds_fwd(const ConvDims& d) {
  LdsConvPlan p = plan_conv_lds(d.N, d.C, d.K, d.P, d.Q, d.R, d.S, d.st);
  p.ok = p.ok && lds_fits(d.x_elems, d.H, d.W);
  return p;
}
inline LdsConvPlan plan_lds_bwd_data(const ConvDims& d) {   // (halo R - 1 - pad)
  LdsConvPlan p = plan_conv_lds(d.N, d.K, d.C, d.H, d.W, d.R, d.S, d.st);
  p.ok = p.ok && d.pad <= d.R - 1 && lds_fits(d.y_elems, d.P, d.Q);
  return p;
}
// What the engine's forward and backward-data forms take on a stride-1 layer of `rows` result channels and `cols` pixels, in
// microseconds: the copies in front (none in the gather form), rounds of the blocks a CU holds at a time, each K step of a
// block taking its share of the matrix pipes or, with few blocks, its MFMAs and 0.43 us of waiting, and the reduction of
// the slices.  Where only the tiles past a multiple of 256 are sliced, the others' whole chains are the shortest a call can
// be: 1.0 to 1.8 tiles a CU took 15 to 19 % longer than their share of the matrix pipes (212 timings of 60 layers, rms error
// 15 %, 7 % with the chain), and the staged form 6 to 45 % less than they (16 images of 96 -> 256 5x5 27x27 152 us, 123).  A fit to 1582 timings of 792 layers (14 of the benchmark networks at 28 batches, 400 of random sizes; rms
// error 11 %; by FLOPs alone it is 32 % and too short by a third where tiles are mostly empty).
inline double engine_us(const SoffPlan& p, int rows, long long cols, size_t w_elems, bool gather) {
  if (!p.ok) return 1e30;
  const int bm = pick_bm(rows), splits = gather ? 1 : p.splits;
  const bool k8 = bm == 64 && rows <= 64 && prefer_k8_64(cols);
  int bn = bm >= 96 ? 128 : splits > 1 && !gather && !k8 ? 128 : 256;
  if (bm == 128 && p.narrow128 && !gather) bn = 64;
  if (bm == 96 && gather) bn = 256;
  const double out_bytes = 4.0 * (double)rows * (double)cols, steps = p.n_k / 16.0;
  const double step_us = bm * bn * 16 / 128.0 / 2300.0;   // MFMAs of a step of a block, alone on a CU
  const double busy_us = step_us * (bm == 128 ? 1.09 : bm == 96 ? 1.17 : bm == 64 ? 1.15 : 1.28) * (gather ? 1.1 : 1.0);
  const long long tiles = (long long)cdiv(rows, bm) * cdiv<long long>(cols, bn), held = bm >= 96 || k8 ? 4 : 3;
  double us;
  if (splits == 1 && !gather && p.tail.splits > 1) {
    us = steps * fmax(busy_us * (double)tiles / 256.0, step_us + 0.43);
  } else {
    const long long per_cu = cdiv<long long>(tiles * splits, 256), rem = per_cu % held;
    auto round_us = [&](long long k) { return steps / splits * fmax((double)k * busy_us, step_us + 0.43); };
    us = (double)(per_cu / held) * round_us(held) + (rem ? round_us(rem) : 0.0);
  }
  us = fmax(us, out_bytes / 4.0e6);
  us += gather ? 5.8 : 6.1 + fmax(2.0 * (double)p.img_bytes / 3.7e6, 8.0 * (double)w_elems / 1.5e6);
  if (splits > 1) us += 4.1 + out_bytes * (2 * splits + 1) / 6.0e6;
  else if (!gather && p.tail.splits > 1) us += 4.1 + 2.0 * (double)p.part_bytes / 6.0e6;
  return us;
}
// A contraction that fits two K steps goes to the gather form of the forward pass, which needs no launch in front of it
// (a 5x5 layer on one channel).
inline bool fwd_gathers(const ConvDims& d) { return d.C * d.R * d.S <= 32; }

// The direct forms of a 3x3 or 5x5 stride-1 layer and which of them is taken: the staged one where its estimate is below
// the engine's by a twentieth at least (on those timings the choice is then 0.35 % slower than the better one on average,
// 0.31 % with the plain comparison, but in 8 instead of 4 of them 8 % slower than the engine or more; by FLOPs alone 4.4 %).
struct DirectForms {
  SoffPlan soff;
  LdsConvPlan lds;
  bool staged;
  double us;   // what the one taken is expected to take
};
inline bool has_staged_form(const ConvDims& d) { return d.R == d.S && (d.R == 3 || d.R == 5) && d.st == 1; }
inline DirectForms pick_direct(const SoffPlan& soff, const LdsConvPlan& lds, double engine) {
  DirectForms f = {soff, lds, lds.ok && lds.us < 0.95 * engine, engine};
  if (f.staged) f.us = lds.us;
  return f;
}
inline DirectForms direct_fwd(const ConvDims& d) {
  const SoffPlan p = plan_soff_fwd(d);
  return pick_direct(p, plan_lds_fwd(d), engine_us(p, d.K, (long long)d.N * d.P * d.Q, d.w_elems, fwd_gathers(d)));
}
inline DirectForms direct_bwd_data(const ConvDims& d) {
  const SoffPlan p = plan_soff_bwd_data(d);
  return pick_direct(p, plan_lds_bwd_data(d), engine_us(p, d.C, (long long)d.N * d.H * d.W, d.w_elems, false));
}

// Where the library takes the Winograd form by itself: enough channels on both sides for the 16 products to be worth their
// transforms, and either a grid that fills the GPU, or a call expected to take less time than the direct form's: from 8 to
// 22 images on for 128 channels and more (256 -> 384, 13 x 13: 8, 256 -> 256, 14 x 14: 11, 384 -> 1024, 6 x 6: 22).  Rounds
// of blocks make either form the shorter one again for a batch or two (512 -> 512, 7 x 7: 16, 21 to 24, from 27 on).
// A plain comparison of the estimates: against the best of the forms, on the timings above, 0.3 % slower on average;
// asking an eighth of the Winograd form 1.6 % (and ResNet-18 on 9 images takes 436 us with it plain, 442 with the eighth).
inline bool wino_fastest(const WinoGeom& g, const DirectForms& f) { return g.fine && g.Ci % 4 == 0 && g.us < f.us; }
inline bool wino_pays(const WinoGeom& g, const DirectForms& f) {
  if (!g.ok || g.Ci < 64 || g.Ko < 64) return false;
  const long long blocks = (long long)(g.rows_p / g.bm) * (g.tiles_p / kWinoBN);
  // 64-row tiles, two to a CU: from a whole round of blocks on, or from three quarters of the CUs on where it is expected
  // to be the fastest (64 -> 64 56x56: batch 24, 588 blocks 53 us against 57 direct; 64 98 against 144)
  if (g.bm == kWinoBM2) return 4 * g.Ko >= 3 * g.rows_p && ((blocks >= 512 && g.fine) || (blocks >= 192 && wino_fastest(g, f)));
  // (rows: 128-row tiles at least three quarters full: 64 filters in one would execute as much as the direct form)
  if (4 * g.Ko >= 3 * g.rows_p && blocks >= 192) return true;
  return wino_fastest(g, f);
}
// The 5x5 forward form executes 64 % of the direct form's multiply-adds (a little more where the 2x2 tiles overhang
// the result) at a lower rate than the direct kernels reach, 18 % less time on 96 -> 256 channels, 27 x 27, batch 256:
// taken for full row tiles, a channel loop long next to a block's prologue and epilogue, and several rounds of blocks, or
// for several row tiles (which share the patches a block reads four times over) from one round on where it is expected to be
// the fastest (the same layer at batch 24: 151 us against 204 on the engine and 200 staged; below one round, at batch
// 16, 122 against 124 staged: not worth its scratch).
inline bool wino_pays5(const WinoGeom& g, const DirectForms& f) {
  if (!g.ok || !g.blk5 || g.C5 < 64 || g.Ko < 64 || 8 * g.Ko < 7 * g.rows_p) return false;
  const long long blocks = (long long)(g.rows_p / kWinoBM) * (g.tiles_p / kWinoBN);
  return blocks >= 512 || (blocks >= 256 && g.rows_p > kWinoBM && wino_fastest(g, f));
}

// The fp32 contraction on bf16 matrix instructions with exactly split operands (conv_tri.hip).  Forward, and backward-data of
// stride 1 as a forward convolution of dy with halo R - 1 - pad; scratch: [group offsets][filter][image][partial sums].
struct TriPlan {
  int N, Ci, Hi, Wi, rows, R, S, st, halo, P, Q;
  int Hp, Wp;
  int groups_true, groups;   // groups of eight k; rounded up to whole K steps
  int bm, bn, splits;
  TailSplit tail;            // as in SoffPlan
  double us;                 // what a call is expected to take
  size_t tab_bytes, wt_bytes, img_bytes, part_bytes;
  bool ok;
  size_t total() const { return tab_bytes + wt_bytes + img_bytes + part_bytes; }
};
// max_chain: the most K steps that a sum may be one chain of (0: any); not ok where slices cannot make it so.
TriPlan plan_tri(int N, int Ci, int Hi, int Wi, int rows, int R, int S, int st, int halo, int P, int Q, int max_chain);
inline TriPlan plan_tri_fwd(const ConvDims& d, int max_chain = 0) {
  return plan_tri(d.N, d.C, d.H, d.W, d.K, d.R, d.S, d.st, d.pad, d.P, d.Q, max_chain);
}
inline TriPlan plan_tri_bwd_data(const ConvDims& d, int max_chain = 0) {
  if (d.st != 1 || d.R != d.S) return TriPlan{};
  return plan_tri(d.N, d.K, d.P, d.Q, d.C, d.R, d.S, 1, d.R - 1 - d.pad, d.H, d.W, max_chain);
}
int launch_conv_tri(const TriPlan& p, bool bwd, const float* in, const float* w, float* out, float alpha, float beta,
                    const float* bias, int relu, const float* mask, void* ws, hipStream_t stream, BnInferJob* bn = nullptr);
// The same with operands of two scaled fp16 parts (conv_duo.hip): scratch [group offsets, exponents, maxima][filter][image][partial sums].
TriPlan plan_duo(int N, int Ci, int Hi, int Wi, int rows, int R, int S, int st, int halo, int P, int Q);
inline TriPlan plan_duo_pass(const ConvDims& d, bool bwd) {
  if (!bwd) return plan_duo(d.N, d.C, d.H, d.W, d.K, d.R, d.S, d.st, d.pad, d.P, d.Q);
  if (d.st != 1 || d.R != d.S) return TriPlan{};
  return plan_duo(d.N, d.K, d.P, d.Q, d.C, d.R, d.S, 1, d.R - 1 - d.pad, d.H, d.W);
}
int launch_conv_duo(const TriPlan& p, bool bwd, const float* in, const float* w, float* out, float alpha, float beta,
                    const float* bias, int relu, const float* mask, void* ws, hipStream_t stream, BnInferJob* bn = nullptr);
struct TriFilterPlan {
  int Hp, Wp, n8, groups_true, groups, bm, bn, splits;
  int sum_rows;   // rows of K partial sums of dy that the copy can leave for the bias gradient
  double us;      // what a call is expected to take
  bool wide;      // the wide form (gemm_tri.h)
  size_t tab_bytes, dyt_bytes, xt_bytes, part_bytes, sum_bytes;
  bool ok;
  size_t sums_at() const { return tab_bytes + dyt_bytes + xt_bytes + part_bytes; }
  size_t total() const { return sums_at() + sum_bytes; }
};
TriFilterPlan plan_tri_bwd_filter(const ConvDims& d, bool wide);
// Leaves `used` slices of dw in (ko, r, s, c) order in *parts, and in `sums`, if given, rows whose sum is dy's over images and
// pixels.
int launch_conv_tri_bwd_filter(const ConvDims& d, const TriFilterPlan& p, const float* x, const float* dy, float* sums, void* ws,
                               hipStream_t stream, float** parts, int* used);
constexpr double kDuoFilterCopies = 22.8;   // us of a call besides its bytes, slices and product
TriFilterPlan plan_duo_bwd_filter(const ConvDims& d);
// three: the plan of three parts for operands that two cannot hold (SplitFilterPick); then there are or_three->splits slices where
// *or_three->any, on the device, is set.
struct OrThree { const int* any; int splits; };
int launch_conv_duo_bwd_filter(const ConvDims& d, const TriFilterPlan& p, const float* x, const float* dy, float* sums, void* ws,
                               hipStream_t stream, float** parts, int* used, const TriFilterPlan* three, OrThree* or_three);

bool conv1x1_stream_applies(const ConvDims& d);

// Where a caller that allows it (RH_ALGO_BF16X3) gets the form of exactly split operands: where its expected time is below
// that of the form taken otherwise.  The engine's estimate was fitted to 3x3 and 5x5 stride-1 layers and is 10 to 25 % short on
// others, hence the tenth.  Over 308 timed forward calls (22 layers at 14 batches) the forms chosen so are 1.27 times as fast as
// without it, geometric mean; of 900 calls of all passes the slowest beside the form replaced are 384 -> 1024 3x3 6x6 data gradients
// (batch 24 56 -> 60 us, 90 129 -> 137) and 256 -> 384 13x13 b256 (355 -> 370).  1x1 layers of up to 128 channels keep the streaming kernels, which
// read their operands where they lie (96 -> 96 54x54 b128 82 us against 158).  Winograd -> this form on one row tile of filters:
// 64 -> 128 5x5 24x24 b128 forward 198 -> 141 us, 128 -> 128 3x3 28x28 filter gradient b37, 64, 256 98 -> 64, 139 -> 92, 466 -> 349.
inline bool tri_allowed(int flags) {
  return (flags & RH_ALGO_BF16X3) && !(flags & (RH_MATH_BF16_MFMA_FP32ACC | RH_ALGO_GATHER | RH_ALGO_SCALAR_OFFSET | RH_ALGO_WINOGRAD));
}
inline bool tri_wide(int flags) { return (flags & RH_ALGO_BF16X3_WIDE) != 0; }
inline bool tri_forced(int flags) { return tri_allowed(flags) && (flags & RH_ALGO_DIRECT); }
inline bool duo_allowed(int flags) {
  return (flags & RH_ALGO_F16X2) && !(flags & (RH_MATH_BF16_MFMA_FP32ACC | RH_ALGO_GATHER | RH_ALGO_SCALAR_OFFSET | RH_ALGO_WINOGRAD));
}
inline bool duo_forced(int flags) { return duo_allowed(flags) && (flags & RH_ALGO_DIRECT) && !tri_allowed(flags); }
// Squared relative error against 64 bits, in units of 1e-14, N(0,1) operands: of this form 0.0525 a K step in a chain (1.34e-7
// at 36, 1.95e-7 at 72), of the engine 0.0335 a term, of the Winograd form as in wino_stages_at_most, of the staged form
// 0.032 a term of its two chains and four more (0.09 2^-48: a rounding's variance).  The chain allowed is the one with three
// quarters of the other form's: half zeros, as behind a ReLU, spare the shorter chains more roundings (1.2 on the square).
// Measured where the form is taken, relative to the other form's error, on the networks' own activations, filters and deltas (forward,
// data and filter gradient; geometric mean and largest): AlexNet 0.77, 0.53, 0.47 and 0.98, NIN 0.54, 0.58, 0.51 and 1.01, ResNet-18 0.49,
// 0.69, 0.43 and 1.00 (its filter gradients in the wide form), CIFAR-10's and LeNet's filter gradients 0.44 and 0.65 (882 calls).  Sums of operands of
// one sign on both sides are another matter, slices make them more exact than their chains alone: uniform [0, 1) on all sides
// 0.8 to 0.9 in the geometric mean of 137 calls, but up to 1.9 beside a form of many slices, 3e-7 and less in all.
inline int tri_max_chain(double other) { const double n = 0.75 * other / 0.0525; return n < 1.0 ? 1 : n < 1e6 ? (int)n : 1000000; }
inline double engine_err(const SoffPlan& p, int terms) { return 0.0335 * terms / p.splits; }
inline double staged_err(const LdsConvPlan& p, int R) {
  const double chain = R == 3 ? 36.0 : 52.0, terms = 4.0 * p.qps * R * R;
  return 0.032 * (chain + terms / chain + 4.0);
}
inline double wino_err(const WinoGeom& g) {
  const int stages = g.full_tiles > 0 || g.tail_S <= 1 ? g.Cg : g.tail_L;
  return 1.35 + 0.351 * cdiv(stages, g.chains > 0 ? g.chains : 1);
}
// The form that a call takes without the bit, [1] with RH_ALGO_SHARED_GPU beside it: its expected time and its error.
struct TriRival { double us, err; };
inline void tri_rivals(const ConvDims& d, bool bwd, TriRival (&r)[2]) {
  const int terms = (bwd ? d.K : d.C) * d.R * d.S;
  if (!has_staged_form(d)) {
    const SoffPlan sp = bwd ? plan_soff_bwd_data(d) : plan_soff_fwd(d);
    r[0].us = 1.1 * engine_us(sp, bwd ? d.C : d.K, (long long)d.N * (bwd ? d.H * d.W : d.P * d.Q), d.w_elems, false);
    r[0].err = engine_err(sp, terms);
    r[1] = r[0];
    return;
  }
  const DirectForms f = bwd ? direct_bwd_data(d) : direct_fwd(d);
  r[0].us = f.us;
  r[0].err = f.staged ? staged_err(f.lds, d.R) : engine_err(f.soff, terms);
  r[1] = r[0];
  const bool five = !bwd && wino_shape5(d);
  if (!wino_shape(d) && !five) return;
  WinoGeom wg = five ? wino_geom_fwd5(d) : bwd ? wino_geom_bwd_data(d) : wino_geom_fwd(d);
  for (int shared = 0; shared < 2; ++shared) {
    if (shared) wg.beside_others();
    if (five ? wino_pays5(wg, f) : wino_pays(wg, f)) r[shared] = TriRival{wg.us, wino_err(wg)};
  }
}
inline bool tri_shape(const ConvDims& d, bool bwd) {
  return (bwd ? d.st == 1 && d.K % 8 == 0 : d.C % 8 == 0 && !fwd_gathers(d)) && !conv1x1_stream_applies(d);
}
inline TriPlan plan_tri_pass(const ConvDims& d, bool bwd, int max_chain) {
  return bwd ? plan_tri_bwd_data(d, max_chain) : plan_tri_fwd(d, max_chain);
}
// The form of split operands that a call takes, if any: 3 or 2 parts.  Two parts where they are expected to be faster than what the
// call takes otherwise, and no further from 64 bits.
// What a result is summed from, over all tiles: K steps in a chain, and slices beyond the first (a sliced tail has short chains).
struct MeanChain { double steps, slices; };
inline MeanChain mean_chain(const TriPlan& p) {
  const double n = cdiv(p.groups / 2, p.splits);
  if (p.tail.splits <= 1) return MeanChain{n, p.splits - 1.0};
  const double tail = (double)p.tail.tail_tiles / (p.tail.full_tiles + p.tail.tail_tiles);
  return MeanChain{(1.0 - tail) * n + tail * cdiv(p.groups / 2, p.tail.splits), tail * (p.tail.splits - 1)};
}
// What two parts lose that three do not, 2^-23 of a value, is the same at every length; what three round grows with the chain, and with the
// deltas that are not zeros, of which few are left behind a max-pool.  Squared error in units of 1e-14, a fit to 118 layers and batches of
// N(0,1) operands (0.87 to 1.16 of its square root measured): forward, half of the image zeros, three parts 0.0327 a step and
// 0.012 a slice, two 1.25, 0.004 and 0.027; data gradient, nine deltas in ten zeros, 0.06, 0.0066 and 0.028, two 1.0 and 0.035 a slice.  So
// taken, the error is 0.59 of three parts' forward (geometric mean; 0.93 at most) and 0.78 backward (0.96, and 1.02 at the line); with half
// of the deltas 0.38, with one in twenty 1.04 (1.3 at most).  dense: the caller says that there are deltas almost everywhere (RH_ALGO_BF16X3_WIDE), where three parts have
// 0.0526 a step: 0.33 over 311 data gradients of ResNet-18 (0.45 at most).
inline bool duo_replaces_tri(bool bwd, bool dense, const TriPlan& tri, const TriPlan& duo) {
  const MeanChain a = mean_chain(tri), b = mean_chain(duo);
  if (bwd && dense) return cdiv(tri.groups / 2, tri.splits) >= 130;
  return bwd ? 0.0066 * a.steps + 0.028 * a.slices >= 0.92 + 0.035 * b.slices
             : 0.0327 * a.steps + 0.012 * a.slices >= 1.56 + 0.005 * b.steps + 0.034 * b.slices;
}
// The others' errors are in tri_max_chain's units, N(0,1).  Over 539 timed calls (18 layers at 11 batches, all passes, half zeros) two parts
// are taken in a quarter, 1.34 times as fast in the geometric mean, none slower, with 0.50 of the error of the form replaced, 0.87 at most; on
// the networks' own activations, filters and deltas at 67 batches (2423 calls; forward, data gradient, filter gradient) AlexNet 0.55, 0.46 and
// 0.55, NIN 0.59, 0.39 and 0.73 (most of its filter gradients end in three parts), ResNet-18 0.52 and 0.33; 0.89, 0.94 and 0.98 at most.
inline bool duo_replaces(double err, int duo_steps) { return 2.5 + 0.008 * duo_steps <= err; }
struct SplitPick {
  int parts;
  TriPlan plan;
};
// (the estimates of three and two parts have an error of 6 % each; a twenty-fifth keeps the choice from changing for nothing)
inline bool duo_pays(const TriPlan& p, bool bwd, int flags, const TriPlan* tri, const TriRival& other) {
  if (!p.ok || p.us >= 0.96 * (tri ? tri->us : other.us)) return false;
  return tri ? duo_replaces_tri(bwd, tri_wide(flags), *tri, p) : duo_replaces(other.err, cdiv(p.groups / 2, p.splits));
}
inline SplitPick pick_split(const ConvDims& d, bool bwd, int flags, size_t ws_bytes) {
  SplitPick s = {};
  if (tri_forced(flags) || duo_forced(flags)) {
    s.parts = tri_forced(flags) ? 3 : 2;
    s.plan = s.parts == 3 ? plan_tri_pass(d, bwd, 0) : plan_duo_pass(d, bwd);
    return s;
  }
  if ((!tri_allowed(flags) && !duo_allowed(flags)) || !tri_shape(d, bwd)) return s;
  TriRival r[2];
  tri_rivals(d, bwd, r);
  const TriRival& other = r[flags & RH_ALGO_SHARED_GPU ? 1 : 0];
  if (tri_allowed(flags)) {
    const TriPlan p = plan_tri_pass(d, bwd, tri_max_chain(other.err));
    if (p.ok && p.us < other.us && p.total() <= ws_bytes) s = SplitPick{3, p};
  }
  if (duo_allowed(flags)) {
    const TriPlan p = plan_duo_pass(d, bwd);
    if (p.total() <= ws_bytes && duo_pays(p, bwd, flags, s.parts ? &s.plan : nullptr, other)) s = SplitPick{2, p};
  }
  return s;
}
// Scratch of these forms where they pay, with the hint or without (three parts' also where two are taken: with less scratch a call
// takes those); 0 also where it cannot be more than `floor`: sized for every batch up to a capacity from the largest down, many
// batches end there.
inline size_t split_bytes(const ConvDims& d, bool bwd, int flags, size_t floor) {
  if (!tri_shape(d, bwd)) return 0;
  // (the copies of three parts, and 24 slices of all tiles, of 256 MB together, or 12 of up to 255 tiles and of an image that they share;
  // exponents, maxima and ratios)
  const int halo = bwd ? d.R - 1 - d.pad : d.pad, rows = bwd ? d.C : d.K, Ci = bwd ? d.K : d.C;
  const double img = 6.0 * d.N * Ci * ((bwd ? d.P : d.H) + 2 * halo) * ((bwd ? d.Q : d.W) + 2 * halo);
  const double out = 4.0 * (double)(bwd ? d.x_elems : d.y_elems);
  const double parts = fmin(24.0 * out, 12.0 * ((256.0 + rows / 64) * 128 * 192 * 4 + out / d.N));
  if (img + (6.5 * Ci * d.R * d.S + 64.0) * rows + parts + 160.0 * d.N + 4.0 * Ci + 8192.0 < (double)floor) return 0;
  TriRival r[2];
  tri_rivals(d, bwd, r);
  size_t need = 0;
  TriPlan p = {}, q = {};
  if (duo_allowed(flags)) q = plan_duo_pass(d, bwd);
  int chain = 0;
  for (const TriRival& other : r) {
    bool tri = false;
    if (tri_allowed(flags)) {
      const int c = tri_max_chain(other.err);
      if (c != chain) p = plan_tri_pass(d, bwd, c);
      chain = c;
      tri = p.ok && p.us < other.us;
      if (tri && p.total() > need) need = p.total();
    }
    if (duo_pays(q, bwd, flags, tri ? &p : nullptr, other) && q.total() > need) need = q.total();
  }
  return need;
}
// Filter gradient: the other forms take about 15 us, their multiply-adds at 50 (32-row tiles), 60 or 100 TFLOP/s, a quarter more
// where taps are gathered or transformed, and 11 us a million weights of partial sums (fitted by hand to 308 timed calls, of
// which this form is then chosen in 188, 1.53 times as fast in the geometric mean).  1x1 layers need 384 channels or so to be
// worth two split copies.  Its slices are short enough for the chain limit almost everywhere: it turns down 4 of 5493 calls (30
// layers at every batch up to 256), of one to four images.
// (or_three: beside a plan of two parts, the one for operands that two cannot hold; at plan.tab_bytes of its scratch, its slabs in the
// same place)
struct SplitFilterPick {
  int parts;
  TriFilterPlan plan, or_three;
};
SplitFilterPick pick_split_bwd_filter(const ConvDims& d, int flags, size_t ws_bytes, size_t* need = nullptr);

int launch_conv_lds(const LdsConvPlan& pl, bool bwd, int N, int Ci, int H, int W, int rows, int P, int Q, int R, int halo,
                    const float* in, const float* w, float* out, float alpha, float beta, const float* bias, int relu,
                    const float* mask, void* ws, hipStream_t stream, BnInferJob* bn = nullptr);

// Forward with packed bf16 operands (RH_MATH_BF16_MFMA_FP32ACC, input channels a multiple of 8): the contraction runs
// over k = (r, s, c) with c fastest, the image is copied once to bf16 as [n][hp][c/8][wp][8] with its zero border,
// the filter to bf16 as [k/8][ko][8] (zero past C*R*S), so that eight consecutive k of one row are 16 contiguous
// bytes of either operand and neighbouring rows are neighbouring 16-byte pieces.
// Scratch: table of byte offsets per group of eight k | filter copy | image copy.
struct Bf16FwdPlan {
  int n_k, Hp, Wp;
  int s_groups;  // 0: groups of eight channels; > 0: groups of eight filter columns, this many per filter row
  size_t tab_bytes, wt_bytes, img_bytes;
  bool ok;
  size_t total() const { return tab_bytes + wt_bytes + img_bytes; }
};

// Channel counts that are not a multiple of 8 (first layers: 3 channels) with an even stride group the contraction
// by filter columns instead: k = (c, r, s) with s padded to a multiple of 8, the image copied to bf16 in its own
// NCHW order with its zero border (rows widened by the padding of s, to an even width), so that the eight s of a
// group are 16 contiguous bytes starting at an even element (4-byte aligned, as a vector load needs) and
// neighbouring pixels are `stride` elements apart.  An 11x11 filter pads to 16 columns (1.45x the contraction; with
// channels padded 3 -> 8 it would be 2.7x), a 7x7 to 8.
inline Bf16FwdPlan plan_bf16_fwd(const ConvDims& d) {
  Bf16FwdPlan p;
  p.Hp = d.H + 2 * d.pad;
  if (d.C % 8 == 0) {
    p.s_groups = 0;
    p.n_k = round_up(d.C * d.R * d.S, kTabPad);
    p.Wp = d.W + 2 * d.pad;
  } else {
    p.s_groups = cdiv(d.S, 8);
    p.n_k = round_up(d.C * d.R * p.s_groups * 8, kTabPad);
    p.Wp = round_up(d.W + 2 * d.pad + p.s_groups * 8 - d.S, 2);
  }
  p.tab_bytes = align256(sizeof(int) * (size_t)(p.n_k / 8));
  p.wt_bytes = align256(2 * (size_t)p.n_k * d.K);
  const size_t img = 2 * (size_t)d.N * d.C * p.Hp * p.Wp;
  p.img_bytes = align256(img);
  p.ok = (d.C % 8 == 0 || d.st % 2 == 0) && img <= kMaxBufferBytes && d.P > 0 && d.Q > 0 &&
         (long long)p.Hp * p.Wp < (1ll << 31) / 64;
  return p;
}

// Backward-data with stride st > 1, decomposed by the residue (a, b) of (h + pad, w + pad) modulo st: an input pixel
// with h + pad = st*u + a only meets the filter rows r = a + st*i, and then through dy row p = u - i.  Each of the
// st*st classes is therefore a stride-1 correlation of dy with the sub-filter w[ko][c][a + st*i][b + st*j] over the
// sub-grid (u, v) of that class, with no wasted products.  Scratch: one padded copy of dy shared by all classes
// (halo L = ceil(R/st) - 1 on top / left, zeros below / right up to the largest u any class reaches), the transposed
// sub-filter and offset table of the class at hand, and the dense per-class results, which one pass interleaves into dx.
constexpr int kMaxPhaseStride = 4;
struct PhaseGeom {
  int Ra, Sb;          // filter rows / columns of the class (0: the class receives nothing)
  int u0, U, v0, V;    // first u, v of the class inside the image and how many
  long long sub_off;   // where the class's dense [n][c][U][V] result starts in the scratch, in floats
  int splits;          // slices of the class's contraction (plan_k_split)
};
struct PhasePlan {
  bool ok;
  int L, Hp, Wp, n_k;  // n_k: the largest padded contraction length among the classes
  size_t tab_bytes, wt_bytes, img_bytes, sub_bytes, part_bytes;
  PhaseGeom ph[kMaxPhaseStride * kMaxPhaseStride];
  size_t total() const { return tab_bytes + wt_bytes + img_bytes + sub_bytes + part_bytes; }
};

inline void phase_axis(int a, int st, int pad, int extent, int taps, int* n_taps, int* first, int* count) {
  *n_taps = a < taps ? (taps - a + st - 1) / st : 0;
  const int lo = pad > a ? (pad - a + st - 1) / st : 0;
  const int top = extent - 1 + pad - a;
  const int hi = top >= 0 ? top / st + 1 : 0;
  *first = lo;
  *count = hi > lo ? hi - lo : 0;
}

inline PhasePlan plan_phase_bwd_data(const ConvDims& d) {
  PhasePlan p;
  p.ok = false;
  p.L = p.Hp = p.Wp = p.n_k = 0;
  p.tab_bytes = p.wt_bytes = p.img_bytes = p.sub_bytes = p.part_bytes = 0;
  if (d.st < 2 || d.st > kMaxPhaseStride || d.P <= 0 || d.Q <= 0) return p;
  const int st = d.st;
  p.L = (d.R > d.S ? d.R : d.S);
  p.L = (p.L + st - 1) / st - 1;
  const int umax = (d.H - 1 + d.pad) / st + 1, vmax = (d.W - 1 + d.pad) / st + 1;
  p.Hp = p.L + (d.P > umax ? d.P : umax);
  p.Wp = p.L + (d.Q > vmax ? d.Q : vmax);
  long long off = 0;
  int max_taps = 0;
  for (int a = 0; a < st; ++a)
    for (int b = 0; b < st; ++b) {
      PhaseGeom& g = p.ph[a * st + b];
      phase_axis(a, st, d.pad, d.H, d.R, &g.Ra, &g.u0, &g.U);
      phase_axis(b, st, d.pad, d.W, d.S, &g.Sb, &g.v0, &g.V);
      g.sub_off = off;
      const long long elems = (long long)d.N * d.C * g.U * g.V;
      off += elems;
      if (g.Ra * g.Sb > max_taps) max_taps = g.Ra * g.Sb;
      g.splits = 1;
      if (g.Ra * g.Sb > 0 && elems > 0) {
        g.splits = plan_k_split(d.C, (long long)d.N * g.U * g.V, round_up(d.K * g.Ra * g.Sb, kTabPad));
        const size_t part = g.splits > 1 ? align256(sizeof(float) * (size_t)g.splits * (size_t)elems) : 0;
        if (part > p.part_bytes) p.part_bytes = part;
      }
    }
  p.n_k = round_up(d.K * (max_taps > 0 ? max_taps : 1), kTabPad);
  p.tab_bytes = align256(sizeof(int) * (size_t)p.n_k);
  p.wt_bytes = align256(sizeof(float) * (size_t)p.n_k * d.C);
  const size_t img = sizeof(float) * (size_t)d.N * d.K * p.Hp * p.Wp;
  p.img_bytes = (p.L > 0 || p.Hp != d.P || p.Wp != d.Q) ? align256(img) : 0;
  p.sub_bytes = align256(sizeof(float) * (size_t)off);
  p.ok = img <= kMaxBufferBytes && (size_t)off * 4 <= kMaxBufferBytes;
  return p;
}

// The residue classes with exactly split operands (conv_tri.hip): one copy of dy, the sub-filters of all classes, one launch for
// all contractions.  ok where it is expected to pay and where no class has a longer chain of sums than tri_max_chain allows.
struct TriPhasePlan {
  bool ok;
  int bm, groups;   // groups of eight k of all classes, each a whole number of K steps
  int slices[kMaxPhaseStride * kMaxPhaseStride], most;   // of a class's contraction; the largest count: slabs of all classes' results
  size_t tab_bytes, wt_bytes, img_bytes, sub_bytes;
  size_t total() const { return tab_bytes + wt_bytes + img_bytes + sub_bytes; }
};
// The other form is a preparation, a product and mostly a reduction for each class, about 10 us and its multiply-adds at 100 TFLOP/s;
// this one copies once and launches once, so it gains most on few pixels.  3x3, stride 2, us: 64 -> 128 56x56 at 8, 24, 64, 128,
// 256 images 93 -> 39, 124 -> 50, 176 -> 99, 274 -> 181, 521 -> 355; 128 -> 256 28x28 at 64, 128, 256 images 176 -> 78, 272 -> 121,
// 405 -> 230; 256 -> 512 14x14 at 256 403 -> 194.
// Below those batches the other form's slices had the smaller error, so here the long classes go in slices too, as many as the error asks
// for or the time: the pass that interleaves the classes adds them up.  128 -> 256 28x28 at 1, 8, 24, 36 images 83 -> 33, 88 -> 39, 125 -> 50,
// 134 -> 58, 256 -> 512 14x14 at 8, 24, 64, 128 94 -> 40, 129 -> 50, 184 -> 79, 253 -> 113, 96 -> 64 5x5 27x27 at 8 and 64 75 -> 32, 133 -> 56;
// 44 layers and batches have 0.45 to 0.83 of the other form's error against 64 bits.
inline TriPhasePlan plan_tri_phases(const ConvDims& d, const PhasePlan& pp) {
  TriPhasePlan p = {};
  if (!pp.ok || d.K % 8 != 0 || d.x_elems == 0 || d.R * d.S == 1) return p;
  p.bm = pick_bm(d.C);
  if (p.bm == 32) return p;
  const int bn = p.bm == 64 ? 192 : 128;
  double other = 30.0;
  int steps[kMaxPhaseStride * kMaxPhaseStride] = {}, least[kMaxPhaseStride * kMaxPhaseStride] = {}, longest = 0;
  for (int i = 0; i < d.st * d.st; ++i) {
    const PhaseGeom& g = pp.ph[i];
    const long long cols = (long long)d.N * g.U * g.V;
    if (g.Ra * g.Sb == 0 || cols == 0) continue;
    const int k_true = d.K * g.Ra * g.Sb, n = round_up(k_true / 8, 2) / 2;
    // (the engine's slices, and a rounding for each slice added to those before)
    const double err = 0.0335 * k_true / g.splits + (g.splits > 1 ? 0.016 * g.splits : 0.0);
    int S = 1;
    while (S <= 8 && cdiv(n, S) > tri_max_chain(err - (S > 1 ? 0.021 * S : 0.0))) ++S;
    if (S > 8) return p;
    steps[i] = n; least[i] = S;
    p.groups += 2 * n;
    if (n > longest) longest = n;
    other += 10.0 + 2.0 * (double)d.C * (double)cols * k_true / 100e6;
  }
  const size_t img = 6 * (size_t)d.N * d.K * pp.Hp * pp.Wp, wt = 48 * (size_t)p.groups * d.C;
  if (p.groups == 0 || img > kMaxBufferBytes || wt > kMaxBufferBytes) return p;
  const double step_us = p.bm == 128 ? 0.456 : 0.377;
  double run = 1e30;
  for (int want = 1; want <= 8; ++want) {
    const int cap = cdiv(longest, want);
    double all = 0.0, slabs = 0.0;
    int chain = 0, most = 1, slices[kMaxPhaseStride * kMaxPhaseStride] = {};
    for (int i = 0; i < d.st * d.st; ++i) {
      if (steps[i] == 0) continue;
      const int S = max(least[i], cdiv(steps[i], cap)), n = cdiv(steps[i], S);
      const long long cols = (long long)d.N * pp.ph[i].U * pp.ph[i].V;
      slices[i] = cdiv(steps[i], n);
      all += (double)steps[i] * cdiv(d.C, p.bm) * (double)cdiv<long long>(cols, bn);
      slabs += 8.0 * (slices[i] - 1) * (double)d.C * (double)cols / 3e6;
      chain = max(chain, n);
      most = max(most, slices[i]);
    }
    if (most > 8) continue;
    const double t = fmax(chain * step_us, all / 256.0 * step_us) + slabs;
    if (t >= 0.95 * run) continue;
    run = t;
    p.most = most;
    for (int i = 0; i < d.st * d.st; ++i) p.slices[i] = slices[i];
  }
  const double us = 20.0 + run + (4.0 * (double)d.y_elems + (double)img) / 5.3e6 + 12.0 * (double)d.x_elems / 5.3e6 +
        10.0 * (double)d.w_elems / 2.2e6;
  if (us >= other) return p;
  p.tab_bytes = align256(sizeof(int) * (size_t)p.groups);
  p.wt_bytes = align256(wt);
  p.img_bytes = align256(img);
  p.sub_bytes = pp.sub_bytes * (size_t)p.most;
  if (p.sub_bytes > kMaxBufferBytes) return p;
  p.ok = true;
  return p;
}
// Leaves the classes' results at *sub, PhaseGeom::sub_off apart.
int launch_conv_tri_phases(const ConvDims& d, const PhasePlan& pp, const TriPhasePlan& p, const float* w, const float* dy, void* ws,
                           hipStream_t stream, float** sub);

// 1x1 / stride 1 / no padding layers with at most this many channels on both sides run on the register-resident
// streaming kernel (conv1x1.hip) in forward and backward-data.
constexpr int kConv1x1MaxChannels = 128;
bool conv1x1_stream_applies(const ConvDims& d);
int launch_conv1x1_stream(const ConvDims& d, int pass, const float* w, const float* src, float* out, float alpha, float beta,
                          const float* bias, int relu, hipStream_t stream, const float* mask = nullptr);

// The same for packed bf16 activations on both sides (conv1x1_bf16.hip): channels in multiples of 32, at most 128.
bool conv1x1_bf16_stream_applies(const ConvDims& d);   // the layers it is chosen for
bool conv1x1_bf16_stream_runs(const ConvDims& d);      // the layers it can run (RH_ALGO_SCALAR_OFFSET forces it on those)
int launch_conv1x1_bf16_stream(const ConvDims& d, const void* xp, const void* wb, const float* bias, int relu,
                               const PackedOut& pk, hipStream_t stream);

// dst[n][c][halo + dil*h][halo + dil*w] = src[n][c][h][w], zeros elsewhere; dst is planes x Hp x Wp.
void launch_pad_image(const float* src, float* dst, long long planes, int H, int W, int Hp, int Wp, int halo,
                      hipStream_t stream, int dil = 1);

// Filter-side scratch of the scalar-offset paths: wT[k][row] and the byte-offset table soff[k] into the padded copy
// (bwd = 0: forward, k = (c,r,s), rows = output channels; bwd = 1: stride-1 backward-data, k = (ko,r,s) with the
// filter flipped, rows = input channels), alone or in one launch with the padded copy of the image (no dilation).
void launch_prep_soff(const float* w, float* wT, int* soff, int n_k, int k_true, int rows, int R, int S, int HpWp, int Wp,
                      int bwd, hipStream_t stream);
void launch_pad_image_prep_soff(const float* src, float* dst, long long planes, int H, int W, int Hp, int Wp, int halo,
                                const float* w, float* wT, int* soff, int n_k, int k_true, int rows, int R, int S, int bwd,
                                hipStream_t stream);

void launch_build_fwd_tab(int4* tab, int n_entries, int CRS, int R, int S, int HW, int W,
                          hipStream_t stream);

}  // namespace rh

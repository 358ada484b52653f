// Spatial batch normalisation over NCHW fp32 tensors: one mean / inverse standard deviation per channel, taken
// over the N*H*W values of that channel.  Stands where the reference calls CudnnBatchNormOp in Spatial mode
// (src/operator/conv.rs:493-535 forward, :594-607 backward).  All three passes are bandwidth bound:
//
//   forward (training)   reduce: read x once            apply: read x (+ y when blending), write y
//   backward             reduce: read x, dy once        apply: read x, dy (+ dx when blending), write dx
//
// A channel of up to 20480 values (kBnChannelMax) takes one launch (bn_channel_kernel): a block brings the whole channel
// into its registers, reduces it and writes the result.  Larger channels take three: a reduce launch of C x G blocks, where
// wave (g, w) of channel c adds work units u = 4g + w, 4g + w + 4G, ... (a unit is one 2048-value piece of one image's
// plane) and leaves one partial per block; a finish launch (16 threads to a channel) that adds the G partials in double
// precision; and an apply launch that sweeps the tensor.  Every order of addition is fixed, so results do not depend on
// scheduling.  The variance is accumulated around the channel's first value as a shift, which keeps the one-pass
// E[d^2] - E[d]^2 form free of the cancellation a zero shift would have for a large mean.
#include "common.h"

namespace rh {

constexpr int kBnChunk = 2048;  // values of one plane a wave adds per work unit

struct BnPlan {
  int chunks;        // pieces per plane
  long long units;   // N * chunks, per channel
  int G;             // blocks per channel
};

inline BnPlan bn_plan(int N, int C, int plane) {
  BnPlan p;
  p.chunks = cdiv(plane, kBnChunk);
  p.units = (long long)N * p.chunks;
  long long g = cdiv<long long>(2048, C);
  const long long most = cdiv<long long>(p.units, 4);
  if (g > most) g = most;
  if (g < 1) g = 1;
  p.G = (int)g;
  return p;
}

__device__ __forceinline__ float wave_sum(float v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  return v;
}

struct BnMask { const float* scale; const float* ivar; const float* bias; };

// MODE 0: (sum d, sum d*d) with d = x - x[first value of the channel].
// MODE 1: (sum dy, sum dy*(x - mean[c])).
// VEC (plane % 4 == 0, 16-byte aligned tensors): a lane reads 16 bytes at a time, two such loads in flight per operand.
// MASK (MODE 1): dy counts only where the forward pass's ReLU let the value through, i.e. where
// bn_affine(x, mean, scale*ivar, bias) > 0, recomputed here exactly as the forward pass computed it.
template <int MODE, bool VEC, bool MASK = false>
__global__ __launch_bounds__(256) void bn_reduce_kernel(const float* __restrict__ x, const float* __restrict__ dy,
                                                        const float* __restrict__ mean, int C, int plane, int chunks,
                                                        long long units, float2* __restrict__ part, BnMask mk) {
  const int c = blockIdx.x, g = blockIdx.y, G = gridDim.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float shift = MODE == 0 ? x[(size_t)c * plane] : mean[c];
  const float m_si = MASK ? mk.scale[c] * mk.ivar[c] : 0.0f, m_bias = MASK ? mk.bias[c] : 0.0f;
  float s0a = 0.0f, s0b = 0.0f, s1a = 0.0f, s1b = 0.0f;
  for (long long u = (long long)g * 4 + wave; u < units; u += (long long)G * 4) {
    const int n = (int)(u / chunks), ch = (int)(u - (long long)n * chunks);
    const size_t base = ((size_t)n * C + c) * plane;
    const int p0 = ch * kBnChunk, p1 = min(plane, p0 + kBnChunk);
    if (VEC) {
      auto add4 = [&](const float4 xv, const float4 gv, float& t0, float& t1) {
        const float d[4] = {xv.x - shift, xv.y - shift, xv.z - shift, xv.w - shift};
        float gg[4] = {gv.x, gv.y, gv.z, gv.w};
        if (MASK) {
          const float xs[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
          for (int e = 0; e < 4; ++e) gg[e] = bn_affine(xs[e], shift, m_si, m_bias) > 0.0f ? gg[e] : 0.0f;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (MODE == 0) { t0 += d[e]; t1 = fmaf(d[e], d[e], t1); }
          else { t0 += gg[e]; t1 = fmaf(gg[e], d[e], t1); }
        }
      };
      const float4* x4 = reinterpret_cast<const float4*>(x + base);
      const float4* g4 = reinterpret_cast<const float4*>((MODE == 1 ? dy : x) + base);
      const int q1 = p1 >> 2;
      int q = (p0 >> 2) + lane;
      for (; q + 64 < q1; q += 128) {
        const float4 xa = x4[q], xb = x4[q + 64];
        const float4 ga = MODE == 1 ? g4[q] : xa, gb = MODE == 1 ? g4[q + 64] : xb;
        add4(xa, ga, s0a, s1a);
        add4(xb, gb, s0b, s1b);
      }
      if (q < q1) {
        const float4 xa = x4[q];
        add4(xa, MODE == 1 ? g4[q] : xa, s0a, s1a);
      }
      continue;
    }
    int i = p0 + lane;
    for (; i + 64 < p1; i += 128) {
      const float d0 = x[base + i] - shift, d1 = x[base + i + 64] - shift;
      if (MODE == 0) {
        s0a += d0; s0b += d1;
        s1a = fmaf(d0, d0, s1a); s1b = fmaf(d1, d1, s1b);
      } else {
        float g0 = dy[base + i], g1 = dy[base + i + 64];
        if (MASK) {
          g0 = bn_affine(x[base + i], shift, m_si, m_bias) > 0.0f ? g0 : 0.0f;
          g1 = bn_affine(x[base + i + 64], shift, m_si, m_bias) > 0.0f ? g1 : 0.0f;
        }
        s0a += g0; s0b += g1;
        s1a = fmaf(g0, d0, s1a); s1b = fmaf(g1, d1, s1b);
      }
    }
    if (i < p1) {
      const float d0 = x[base + i] - shift;
      if (MODE == 0) {
        s0a += d0;
        s1a = fmaf(d0, d0, s1a);
      } else {
        float g0 = dy[base + i];
        if (MASK) g0 = bn_affine(x[base + i], shift, m_si, m_bias) > 0.0f ? g0 : 0.0f;
        s0a += g0;
        s1a = fmaf(g0, d0, s1a);
      }
    }
  }
  const float s0 = wave_sum(s0a + s0b), s1 = wave_sum(s1a + s1b);
  __shared__ float2 sm[4];
  if (lane == 0) sm[wave] = make_float2(s0, s1);
  __syncthreads();
  if (threadIdx.x == 0)
    part[(size_t)g * C + c] = make_float2((sm[0].x + sm[1].x) + (sm[2].x + sm[3].x), (sm[0].y + sm[1].y) + (sm[2].y + sm[3].y));
}

// What a channel's statistics are formed from and written to.
struct BnFwdStats {
  double count, ema, epsilon;
  const float* scale; const float* bias;
  float* running_mean; float* running_ivar; float* cached_mean; float* cached_ivar;
};
struct BnBwdStats {
  double count;
  float alpha, beta;  // of the parameter gradients
  const float* scale;
  float* dscale; float* dbias;
  const float* cached_mean; const float* cached_ivar;
};

// Sums of a channel -> (mean, scale*ivar, bias, unused); the statistics are stored by the one thread that says so.
__device__ __forceinline__ float4 bn_finish(const BnFwdStats& a, int c, float shift, double s0, double s1, bool store) {
  const double md = s0 / a.count;
  double var = s1 / a.count - md * md;
  if (var < 0.0) var = 0.0;
  const float mean = (float)((double)shift + md);
  const float ivar = (float)(1.0 / sqrt(var + a.epsilon));
  if (store) {
    a.cached_mean[c] = mean;
    a.cached_ivar[c] = ivar;
    a.running_mean[c] = (float)((1.0 - a.ema) * (double)a.running_mean[c] + a.ema * (double)mean);
    a.running_ivar[c] = (float)((1.0 - a.ema) * (double)a.running_ivar[c] + a.ema * (double)ivar);
  }
  return make_float4(mean, a.scale[c] * ivar, a.bias[c], 0.0f);
}

// -> (mean, scale*ivar, sum(dy)/m, ivar^2 * sum(dy*(x-mean))/m)
__device__ __forceinline__ float4 bn_finish(const BnBwdStats& a, int c, float, double s0, double s1, bool store) {
  const double ivar = (double)a.cached_ivar[c];
  if (store) {
    const float ds = (float)(s1 * ivar), db = (float)s0;
    a.dscale[c] = a.beta != 0.0f ? fmaf(a.beta, a.dscale[c], a.alpha * ds) : a.alpha * ds;
    a.dbias[c] = a.beta != 0.0f ? fmaf(a.beta, a.dbias[c], a.alpha * db) : a.alpha * db;
  }
  return make_float4(a.cached_mean[c], a.scale[c] * (float)ivar, (float)(s0 / a.count), (float)(s1 * ivar * ivar / a.count));
}

// coef[c] = what the G partials of channel c give.  A launch of its own between two passes over the tensor, bound by the latency of its
// reads, hence 16 threads to a channel's partials.  (x: its first value is the shift of the sums.)  With a thread to a channel 8.4 us forward
// and 7.3 backward on ResNet-18's layers at 256 images, now 5.0 and 4.7.
constexpr int kBnFinishChans = 16, kBnFinishSubs = 16;
template <class Stats>
__global__ __launch_bounds__(kBnFinishChans * kBnFinishSubs) void bn_finish_kernel(Stats stats, const float* __restrict__ x,
                                                                                  const float2* __restrict__ part, int G, int C, int plane,
                                                                                  float4* __restrict__ coef) {
  __shared__ double2 sums[kBnFinishSubs][kBnFinishChans];
  const int cl = threadIdx.x % kBnFinishChans, sub = threadIdx.x / kBnFinishChans, c = blockIdx.x * kBnFinishChans + cl;
  double s0 = 0.0, s1 = 0.0;
  if (c < C)
    for (int g = sub; g < G; g += kBnFinishSubs) {
      const float2 p = part[(size_t)g * C + c];
      s0 += (double)p.x;
      s1 += (double)p.y;
    }
  const float shift = sub == 0 && c < C ? x[(size_t)c * plane] : 0.0f;
  sums[sub][cl] = make_double2(s0, s1);
  __syncthreads();
  if (sub != 0 || c >= C) return;
#pragma unroll
  for (int i = 1; i < kBnFinishSubs; ++i) {
    s0 += sums[i][cl].x;
    s1 += sums[i][cl].y;
  }
  coef[c] = bn_finish(stats, c, shift, s0, s1, true);
}

// Forward:  out = alpha * f((x - mean)*a + b) + beta*old, f = identity or max(., 0) applied after the blend when RELU.
// (old: out itself, or the tensor a residual unit adds.  Read where it lies, 5 residual units need no copy of their input in
// front of this pass: 46 us each for 256 x 64 x 56 x 56, 3 to 5 us for a few images.)
// Backward: out = alpha * a*(dy - c2 - (x - mean)*c3) + beta*old.
// MASK (backward only): dy is taken as 0 where the forward ReLU clamped, see bn_reduce_kernel; mb = the layer's bias.
template <bool BWD, bool RELU, bool MASK>
__device__ __forceinline__ float bn_one(float xv, float gv, float ov, const float4 k, float mb, float alpha, float beta) {
  float v;
  if (MASK) gv = bn_affine(xv, k.x, k.y, mb) > 0.0f ? gv : 0.0f;
  if (BWD) v = k.y * (gv - k.z - (xv - k.x) * k.w);
  else v = bn_affine(xv, k.x, k.y, k.z);
  v *= alpha;
  if (beta != 0.0f) v = fmaf(beta, ov, v);
  if (RELU) v = v > 0.0f ? v : 0.0f;
  return v;
}
template <bool BWD, bool RELU, bool MASK>
__device__ __forceinline__ float4 bn_one(float4 x, float4 g, float4 o, const float4 k, float mb, float alpha, float beta) {
  return make_float4(bn_one<BWD, RELU, MASK>(x.x, g.x, o.x, k, mb, alpha, beta), bn_one<BWD, RELU, MASK>(x.y, g.y, o.y, k, mb, alpha, beta),
                     bn_one<BWD, RELU, MASK>(x.z, g.z, o.z, k, mb, alpha, beta), bn_one<BWD, RELU, MASK>(x.w, g.w, o.w, k, mb, alpha, beta));
}

// One value into a channel's two sums: (d, d*d) forward, (dy, dy*(x - mean)) backward with shift = mean.
template <bool BWD, bool MASK>
__device__ __forceinline__ void bn_add(float xv, float gv, float shift, float m_si, float mb, float& t0, float& t1) {
  const float d = xv - shift;
  if (MASK) gv = bn_affine(xv, shift, m_si, mb) > 0.0f ? gv : 0.0f;
  t0 += BWD ? gv : d;
  t1 = fmaf(BWD ? gv : d, d, t1);
}
template <bool BWD, bool MASK>
__device__ __forceinline__ void bn_add(float4 x, float4 g, float shift, float m_si, float mb, float& t0, float& t1) {
  bn_add<BWD, MASK>(x.x, g.x, shift, m_si, mb, t0, t1);
  bn_add<BWD, MASK>(x.y, g.y, shift, m_si, mb, t0, t1);
  bn_add<BWD, MASK>(x.z, g.z, shift, m_si, mb, t0, t1);
  bn_add<BWD, MASK>(x.w, g.w, shift, m_si, mb, t0, t1);
}

__device__ __forceinline__ void bn_zero(float& v) { v = 0.0f; }
__device__ __forceinline__ void bn_zero(float4& v) { v = make_float4(0.0f, 0.0f, 0.0f, 0.0f); }

// Where unit i (a value, or four) of channel c lies: a channel is N planes of `pu` units, C planes apart.
struct BnUnits {
  uint32_t C, pu;
  FastDiv by_plane;
  __device__ __forceinline__ size_t at(uint32_t c, uint32_t i) const {
    const uint32_t n = by_plane.quot(i);
    return ((size_t)n * C + c) * pu + (i - n * pu);
  }
};

// A channel's whole pass in one block: the values stay in registers between the sums and the result.  Small tensors are
// bound by the dependent launches, not by bytes: 24 x 256 x 14 x 14 backward 12 + 6 + 10 us in three, 9 us in this one;
// a ResNet-18 training step of 24 samples 4.52 -> 4.25 ms.  256 x 512 x 7 x 7 forward (12544 single values
// a channel; the most are 20480) 41 -> 24 us.
// T = float4 (plane % 4 == 0 and 16-byte aligned tensors, so a unit never crosses a plane) or float.
template <class T, bool BWD, bool RELU, bool MASK, int THREADS, int U, class Stats>
__global__ __launch_bounds__(THREADS) void bn_channel_kernel(const T* x, const T* dy, const T* old, T* out, Stats stats, BnUnits un,
                                                             uint32_t units, float alpha, float beta, const float* mask_bias) {
  const uint32_t c = blockIdx.x, t = threadIdx.x;
  T xv[U], gv[U], ov[U];
#pragma unroll
  for (int k = 0; k < U; ++k) {
    const uint32_t i = t + k * THREADS;
    bn_zero(xv[k]); bn_zero(gv[k]); bn_zero(ov[k]);
    if (i < units) {
      const size_t at = un.at(c, i);
      xv[k] = x[at];
      if constexpr (BWD) gv[k] = dy[at];
      if (beta != 0.0f) ov[k] = old[at];
    }
  }
  float shift, m_si = 0.0f, mb = 0.0f;
  if constexpr (BWD) shift = stats.cached_mean[c];
  else shift = reinterpret_cast<const float*>(x)[(size_t)c * un.pu * (sizeof(T) / 4)];
  if constexpr (MASK) { m_si = stats.scale[c] * stats.cached_ivar[c]; mb = mask_bias[c]; }
  float t0 = 0.0f, t1 = 0.0f;
#pragma unroll
  for (int k = 0; k < U; ++k)
    if (t + k * THREADS < units) bn_add<BWD, MASK>(xv[k], gv[k], shift, m_si, mb, t0, t1);
  t0 = wave_sum(t0);
  t1 = wave_sum(t1);
  constexpr int kWaves = THREADS / 64;
  __shared__ float2 sm[kWaves];
  if ((t & 63) == 0) sm[t >> 6] = make_float2(t0, t1);
  __syncthreads();  // also: the shift has been read by everyone before anyone writes an aliased x
  double s0 = 0.0, s1 = 0.0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) { s0 += (double)sm[w].x; s1 += (double)sm[w].y; }
  const float4 k4 = bn_finish(stats, c, shift, s0, s1, t == 0);
#pragma unroll
  for (int k = 0; k < U; ++k) {
    const uint32_t i = t + k * THREADS;
    if (i < units) out[un.at(c, i)] = bn_one<BWD, RELU, MASK>(xv[k], gv[k], ov[k], k4, mb, alpha, beta);
  }
}

// T = float4 or float as above.  (Forming the coefficients here, each wave adding its channel's partials, saved the finish
// launch of 9 us and cost this kernel 15: 94 -> 109 us backward on 256 x 64 x 56 x 56.)
template <class T, bool BWD, bool RELU, bool MASK>
__global__ __launch_bounds__(256) void bn_apply_kernel(const T* x, const T* dy, const T* old, T* out, const float4* __restrict__ coef,
                                                       uint32_t groups, FastDiv plane_groups, FastDiv chans, float alpha,
                                                       float beta, const float* __restrict__ mask_bias) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= groups) return;
  const uint32_t row = plane_groups.quot(i);  // n*C + c
  const uint32_t c = row - chans.quot(row) * chans.div;
  const float4 k = coef[c];
  const float mb = MASK ? mask_bias[c] : 0.0f;
  T gv, ov;
  bn_zero(gv); bn_zero(ov);
  const T xv = x[i];
  if constexpr (BWD) gv = dy[i];
  if (beta != 0.0f) ov = old[i];
  out[i] = bn_one<BWD, RELU, MASK>(xv, gv, ov, k, mb, alpha, beta);
}

// Inference: the coefficients are a handful of cached loads per thread.
template <class T, bool RELU>
__global__ __launch_bounds__(256) void bn_infer_kernel(const T* x, const T* old, T* out, const float* __restrict__ scale,
                                                       const float* __restrict__ bias, const float* __restrict__ running_mean,
                                                       const float* __restrict__ running_ivar, uint32_t groups, FastDiv plane_groups,
                                                       FastDiv chans, float alpha, float beta) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= groups) return;
  T ov;
  bn_zero(ov);
  if (beta != 0.0f) ov = old[i];
  const T xv = x[i];
  const uint32_t row = plane_groups.quot(i);  // n*C + c
  const uint32_t c = row - chans.quot(row) * chans.div;
  const float4 k = make_float4(running_mean[c], scale[c] * running_ivar[c], bias[c], 0.0f);
  out[i] = bn_one<false, RELU, false>(xv, xv, ov, k, 0.0f, alpha, beta);
}

inline bool bn_vec(int plane, const void* a, const void* b, const void* c, const void* d = nullptr) {
  return plane % 4 == 0 && ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) | reinterpret_cast<uintptr_t>(c) |
                             reinterpret_cast<uintptr_t>(d)) & 15) == 0;
}

template <class T, bool BWD, bool RELU, bool MASK, int THREADS, int U, class Stats>
void launch_bn_channel(const float* x, const float* dy, const float* old, float* out, const Stats& stats, const BnUnits& un, uint32_t units,
                       float alpha, float beta, const float* mask_bias, hipStream_t st) {
  hipLaunchKernelGGL((bn_channel_kernel<T, BWD, RELU, MASK, THREADS, U, Stats>), dim3(un.C), dim3(THREADS), 0, st,
                     reinterpret_cast<const T*>(x), reinterpret_cast<const T*>(dy), reinterpret_cast<const T*>(old), reinterpret_cast<T*>(out), stats, un, units,
                     alpha, beta, mask_bias);
}

// Values of a channel a block of 1024 threads holds: five 16-byte units a thread, or 20 single values where a plane is no
// multiple of four (two operands and the old result of a blend of those are more than its registers).
constexpr long long kBnChannelMax = 20480, kBnChannelMaxBwd1 = 6144;

// Whether the whole pass goes in one launch.
inline bool bn_whole(bool bwd, bool vec, int N, int plane) {
  return (long long)N * plane <= (bwd && !vec ? kBnChannelMaxBwd1 : kBnChannelMax);
}

template <bool BWD, bool RELU, bool MASK, class Stats>
void launch_bn_whole(const float* x, const float* dy, const float* old, float* out, const Stats& stats, int N, int C, int plane, float alpha,
                     float beta, const float* mask_bias, hipStream_t st) {
  const long long values = (long long)N * plane;
  BnUnits un;
  un.C = (uint32_t)C;
  if (bn_vec(plane, x, dy, out, old)) {
    un.pu = (uint32_t)(plane / 4);
    un.by_plane = FastDiv(un.pu);
    const uint32_t units = (uint32_t)(values / 4);
    if (units <= 256 * 2) launch_bn_channel<float4, BWD, RELU, MASK, 256, 2>(x, dy, old, out, stats, un, units, alpha, beta, mask_bias, st);
    else if (units <= 512 * 4) launch_bn_channel<float4, BWD, RELU, MASK, 512, 4>(x, dy, old, out, stats, un, units, alpha, beta, mask_bias, st);
    else launch_bn_channel<float4, BWD, RELU, MASK, 1024, 5>(x, dy, old, out, stats, un, units, alpha, beta, mask_bias, st);
  } else {
    un.pu = (uint32_t)plane;
    un.by_plane = FastDiv(un.pu);
    const uint32_t units = (uint32_t)values;
    if (units <= 256 * 6) launch_bn_channel<float, BWD, RELU, MASK, 256, 6>(x, dy, old, out, stats, un, units, alpha, beta, mask_bias, st);
    else if (units <= 1024 * 6) launch_bn_channel<float, BWD, RELU, MASK, 1024, 6>(x, dy, old, out, stats, un, units, alpha, beta, mask_bias, st);
    else if constexpr (!BWD) launch_bn_channel<float, BWD, RELU, MASK, 1024, 20>(x, dy, old, out, stats, un, units, alpha, beta, mask_bias, st);
  }
}

template <bool BWD, bool RELU, bool MASK>
void launch_bn_apply(const float* x, const float* dy, const float* old, float* out, const float4* coef, int N, int C, int plane, float alpha,
                     float beta, const float* mask_bias, hipStream_t st) {
  auto go = [&](auto zero, int width) {
    using T = decltype(zero);
    const uint32_t groups = (uint32_t)((long long)N * C * plane / width);
    hipLaunchKernelGGL((bn_apply_kernel<T, BWD, RELU, MASK>), dim3(cdiv(groups, 256u)), dim3(256), 0, st,
                       reinterpret_cast<const T*>(x), reinterpret_cast<const T*>(dy), reinterpret_cast<const T*>(old), reinterpret_cast<T*>(out), coef, groups,
                       FastDiv((uint32_t)(plane / width)), FastDiv((uint32_t)C), alpha, beta, mask_bias);
  };
  if (bn_vec(plane, x, dy, out, old)) go(float4(), 4);
  else go(0.0f, 1);
}

template <bool RELU>
void launch_bn_infer(const float* x, const float* old, float* out, const float* scale, const float* bias, const float* running_mean,
                     const float* running_ivar, long long total, int C, int plane, float alpha, float beta, hipStream_t st) {
  auto go = [&](auto zero, int width) {
    using T = decltype(zero);
    const uint32_t groups = (uint32_t)(total / width);
    hipLaunchKernelGGL((bn_infer_kernel<T, RELU>), dim3(cdiv(groups, 256u)), dim3(256), 0, st, reinterpret_cast<const T*>(x),
                       reinterpret_cast<const T*>(old), reinterpret_cast<T*>(out), scale, bias, running_mean, running_ivar, groups,
                       FastDiv((uint32_t)(plane / width)), FastDiv((uint32_t)C), alpha, beta);
  };
  if (bn_vec(plane, x, out, old)) go(float4(), 4);
  else go(0.0f, 1);
}

template <int MODE, bool MASK>
void launch_bn_reduce(const float* x, const float* dy, const float* mean, int C, int plane, const BnPlan& p, float2* part,
                      const BnMask& mk, hipStream_t st) {
  const dim3 grid(C, p.G);
  if (bn_vec(plane, x, dy, nullptr))
    hipLaunchKernelGGL((bn_reduce_kernel<MODE, true, MASK>), grid, dim3(256), 0, st, x, dy, mean, C, plane, p.chunks, p.units, part, mk);
  else
    hipLaunchKernelGGL((bn_reduce_kernel<MODE, false, MASK>), grid, dim3(256), 0, st, x, dy, mean, C, plane, p.chunks, p.units, part, mk);
}

inline size_t bn_part_bytes(const BnPlan& p, int C) { return ((size_t)p.G * C * sizeof(float2) + 255) & ~(size_t)255; }

int bn_check(int N, int C, int plane, long long* total) {
  if (N < 0 || C < 0 || plane < 0) return RH_E_INVALID;
  *total = (long long)N * C * plane;
  if (*total >= (1ll << 31)) return RH_E_LIMIT;
  return 0;
}

}  // namespace rh

using namespace rh;

extern "C" size_t rh_bnorm_workspace_bytes(int N, int C, int plane) {
  if (N <= 0 || C <= 0 || plane <= 0) return 256;
  const BnPlan p = bn_plan(N, C, plane);
  return bn_part_bytes(p, C) + (((size_t)C * sizeof(float4) + 255) & ~(size_t)255);
}

extern "C" size_t rh_bnorm_workspace_bytes_upto(int N, int C, int plane) {
  size_t need = 256;
  for (int n = N; n >= 1; --n) {
    const size_t b = rh_bnorm_workspace_bytes(n, C, plane);
    if (b > need) need = b;
  }
  return need;
}

template <bool RELU>
static void bn_fwd_train(int N, int C, int plane, float alpha, const float* x, float beta, const float* y0, float* y, const BnFwdStats& stats,
                         void* ws, hipStream_t st) {
  const double total = (double)N * C * plane;
  if (bn_whole(false, bn_vec(plane, x, y, y0), N, plane)) {
    ProfScope prof("bnorm_fwd", (beta != 0.0f ? 12.0 : 8.0) * total, st);
    return launch_bn_whole<false, RELU, false>(x, nullptr, y0, y, stats, N, C, plane, alpha, beta, nullptr, st);
  }
  const BnPlan p = bn_plan(N, C, plane);
  float2* part = static_cast<float2*>(ws);
  float4* coef = reinterpret_cast<float4*>(static_cast<char*>(ws) + bn_part_bytes(p, C));
  {
    ProfScope prof("bnorm_fwd_reduce", 4.0 * total, st);
    launch_bn_reduce<0, false>(x, nullptr, nullptr, C, plane, p, part, BnMask(), st);
    hipLaunchKernelGGL(bn_finish_kernel<BnFwdStats>, dim3(cdiv(C, kBnFinishChans)), dim3(kBnFinishChans * kBnFinishSubs), 0, st, stats, x, part, p.G, C, plane, coef);
  }
  ProfScope prof("bnorm_fwd_apply", (beta != 0.0f ? 12.0 : 8.0) * total, st);
  launch_bn_apply<false, RELU, false>(x, nullptr, y0, y, coef, N, C, plane, alpha, beta, nullptr, st);
}

extern "C" int rh_bnorm_fwd_train_add(int N, int C, int plane, float alpha, const float* x, float beta, const float* y0, float* y,
                                  double ema_factor, double epsilon, const float* scale, const float* bias,
                                  float* running_mean, float* running_ivar, float* cached_mean, float* cached_ivar,
                                  void* ws, size_t ws_bytes, int flags, rh_stream_t stream) {
  long long total;
  if (int e = bn_check(N, C, plane, &total)) return e;
  if (total == 0) return 0;
  if (!x || !y0 || !y || !scale || !bias || !running_mean || !running_ivar || !cached_mean || !cached_ivar || !ws) return RH_E_INVALID;
  if (flags & ~RH_FUSE_RELU) return RH_E_UNSUPPORTED;
  if (ws_bytes < rh_bnorm_workspace_bytes(N, C, plane)) return RH_E_WORKSPACE;
  const BnFwdStats stats = {(double)N * (double)plane, ema_factor, epsilon, scale, bias,
                            running_mean, running_ivar, cached_mean, cached_ivar};
  if (flags & RH_FUSE_RELU) bn_fwd_train<true>(N, C, plane, alpha, x, beta, y0, y, stats, ws, to_stream(stream));
  else bn_fwd_train<false>(N, C, plane, alpha, x, beta, y0, y, stats, ws, to_stream(stream));
  return launch_status();
}

extern "C" int rh_bnorm_fwd_train(int N, int C, int plane, float alpha, const float* x, float beta, float* y,
                                  double ema_factor, double epsilon, const float* scale, const float* bias,
                                  float* running_mean, float* running_ivar, float* cached_mean, float* cached_ivar,
                                  void* ws, size_t ws_bytes, int flags, rh_stream_t stream) {
  return rh_bnorm_fwd_train_add(N, C, plane, alpha, x, beta, y, y, ema_factor, epsilon, scale, bias, running_mean, running_ivar,
                                cached_mean, cached_ivar, ws, ws_bytes, flags, stream);
}

extern "C" int rh_bnorm_fwd_infer_add(int N, int C, int plane, float alpha, const float* x, float beta, const float* y0, float* y,
                                  double epsilon, const float* scale, const float* bias, const float* running_mean,
                                  const float* running_ivar, void* ws, size_t ws_bytes, int flags, rh_stream_t stream) {
  (void)epsilon;  // already inside the stored inverse standard deviation
  long long total;
  if (int e = bn_check(N, C, plane, &total)) return e;
  if (total == 0) return 0;
  if (!x || !y0 || !y || !scale || !bias || !running_mean || !running_ivar || !ws) return RH_E_INVALID;
  if (flags & ~RH_FUSE_RELU) return RH_E_UNSUPPORTED;
  if (ws_bytes < rh_bnorm_workspace_bytes(N, C, plane)) return RH_E_WORKSPACE;
  hipStream_t st = to_stream(stream);
  ProfScope prof("bnorm_fwd_apply", (beta != 0.0f ? 12.0 : 8.0) * (double)total, st);
  if (flags & RH_FUSE_RELU) launch_bn_infer<true>(x, y0, y, scale, bias, running_mean, running_ivar, total, C, plane, alpha, beta, st);
  else launch_bn_infer<false>(x, y0, y, scale, bias, running_mean, running_ivar, total, C, plane, alpha, beta, st);
  return launch_status();
}

extern "C" int rh_bnorm_fwd_infer(int N, int C, int plane, float alpha, const float* x, float beta, float* y, double epsilon,
                                  const float* scale, const float* bias, const float* running_mean,
                                  const float* running_ivar, void* ws, size_t ws_bytes, int flags, rh_stream_t stream) {
  return rh_bnorm_fwd_infer_add(N, C, plane, alpha, x, beta, y, y, epsilon, scale, bias, running_mean, running_ivar, ws, ws_bytes,
                                flags, stream);
}

template <bool MASK>
static void bn_bwd(int N, int C, int plane, float alpha, const float* x, const float* dy, float beta, float* dx,
                   const BnBwdStats& stats, const float* relu_bias, void* ws, hipStream_t st) {
  const double total = (double)N * C * plane;
  if (bn_whole(true, bn_vec(plane, x, dy, dx), N, plane)) {
    ProfScope prof("bnorm_bwd", (beta != 0.0f ? 16.0 : 12.0) * total, st);
    return launch_bn_whole<true, false, MASK>(x, dy, dx, dx, stats, N, C, plane, alpha, beta, relu_bias, st);
  }
  const BnPlan p = bn_plan(N, C, plane);
  float2* part = static_cast<float2*>(ws);
  float4* coef = reinterpret_cast<float4*>(static_cast<char*>(ws) + bn_part_bytes(p, C));
  {
    ProfScope prof("bnorm_bwd_reduce", 8.0 * total, st);
    const BnMask mk = {stats.scale, stats.cached_ivar, relu_bias};
    launch_bn_reduce<1, MASK>(x, dy, stats.cached_mean, C, plane, p, part, mk, st);
    hipLaunchKernelGGL(bn_finish_kernel<BnBwdStats>, dim3(cdiv(C, kBnFinishChans)), dim3(kBnFinishChans * kBnFinishSubs), 0, st, stats, x, part, p.G, C, plane, coef);
  }
  ProfScope prof("bnorm_bwd_apply", (beta != 0.0f ? 16.0 : 12.0) * total, st);
  launch_bn_apply<true, false, MASK>(x, dy, dx, dx, coef, N, C, plane, alpha, beta, relu_bias, st);
}

static int bnorm_bwd(int N, int C, int plane, float alpha_data, float beta_data, const float* x, const float* dy, float* dx,
                     float alpha_param, float beta_param, const float* scale, float* dscale, float* dbias,
                     const float* cached_mean, const float* cached_ivar, void* ws, size_t ws_bytes, const float* relu_bias,
                     rh_stream_t stream) {
  long long total;
  if (int e = bn_check(N, C, plane, &total)) return e;
  if (total == 0) return 0;
  if (!x || !dy || !dx || !scale || !dscale || !dbias || !cached_mean || !cached_ivar || !ws) return RH_E_INVALID;
  if (ws_bytes < rh_bnorm_workspace_bytes(N, C, plane)) return RH_E_WORKSPACE;
  const BnBwdStats stats = {(double)N * (double)plane, alpha_param, beta_param, scale, dscale, dbias, cached_mean, cached_ivar};
  if (relu_bias) bn_bwd<true>(N, C, plane, alpha_data, x, dy, beta_data, dx, stats, relu_bias, ws, to_stream(stream));
  else bn_bwd<false>(N, C, plane, alpha_data, x, dy, beta_data, dx, stats, nullptr, ws, to_stream(stream));
  return launch_status();
}

extern "C" int rh_bnorm_bwd(int N, int C, int plane, float alpha_data, float beta_data, const float* x, const float* dy,
                            float* dx, float alpha_param, float beta_param, double epsilon, const float* scale, float* dscale,
                            float* dbias, const float* cached_mean, const float* cached_ivar, void* ws, size_t ws_bytes,
                            rh_stream_t stream) {
  (void)epsilon;  // the cached inverse standard deviation of the forward pass is used
  return bnorm_bwd(N, C, plane, alpha_data, beta_data, x, dy, dx, alpha_param, beta_param, scale, dscale, dbias, cached_mean,
                   cached_ivar, ws, ws_bytes, nullptr, stream);
}

extern "C" int rh_bnorm_bwd_relu(int N, int C, int plane, float alpha_data, float beta_data, const float* x, const float* dy,
                                 float* dx, float alpha_param, float beta_param, double epsilon, const float* scale,
                                 const float* bias, float* dscale, float* dbias, const float* cached_mean,
                                 const float* cached_ivar, void* ws, size_t ws_bytes, rh_stream_t stream) {
  (void)epsilon;
  if (!bias) return RH_E_INVALID;
  return bnorm_bwd(N, C, plane, alpha_data, beta_data, x, dy, dx, alpha_param, beta_param, scale, dscale, dbias, cached_mean,
                   cached_ivar, ws, ws_bytes, bias, stream);
}

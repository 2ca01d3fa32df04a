// Batch normalisation over the rows of a (rows, C) feature matrix with the ReLU that follows
// it in every conv-bn-relu block fused in: training statistics, the normalise (+ ReLU) pass,
// and the gradient.  Everything here is HBM-bound; the point of the fusion is the number of
// passes over the tensor (forward 2 reads + 1 write, backward 4 reads + 1 write, the ReLU
// costs none; a residual one more read, and backward one more write and bits) and 16-byte accesses on
// channels-last rows.  Reductions are two-level with a fixed order (per-workgroup partial sums,
// then one thread per channel in fp64): no atomics, bit-reproducible.
//
// The sums walk the rows from the first to the last, all workgroups side by side, and the elementwise pass that
// reads the same tensors again walks them back: what was read last is in the memory-side cache (256 MB).  With a range
// of rows per workgroup in both, 1.1 M x 96 fp16 took 135 + 236 us forward + backward, now 131 + 209; 900 k x 96 with a
// residual 139 + 238, now 129 + 212; 40 k rows the same.
#include <algorithm>
#include <mutex>
#include <type_traits>
#include <utility>
#include <vector>

#include "common.hpp"
#include "host_api.hpp"

namespace ocnn {

constexpr int kBnMaxBlocks = 512;     // workgroups of a reduction (their partial sums are added by one more kernel)
constexpr int kBnApplyBlocks = 2048;  // workgroups of an elementwise pass, at most (fewer where the device holds fewer at once)

template <typename T, int VEC> struct alignas(sizeof(T) * VEC) BnVec { T v[VEC]; };

// element c of a per-channel parameter held as f32 / f16 / bf16 (p == nullptr: dflt)
__device__ __forceinline__ float bn_param(const void* p, int dtype, int c, float dflt) {
  if (!p) return dflt;
  if (dtype == OCNN_F32) return ((const float*)p)[c];
  if (dtype == OCNN_F16) return to_f32(((const f16*)p)[c]);
  return to_f32(((const bf16*)p)[c]);
}

// gamma and beta of the channels c0 .. c0 + VEC - 1 (1 and 0 where the pointer is null).  The raw
// values of both are requested before either is converted, so that a workgroup waits for one
// round trip to memory and not for one per channel.
template <int VEC>
__device__ __forceinline__ void bn_params(const void* __restrict__ gamma, const void* __restrict__ beta, int dtype,
                                          int c0, float (&ga)[VEC], float (&be)[VEC]) {
  if (dtype == OCNN_F32) {
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      ga[v] = gamma ? ((const float*)gamma)[c0 + v] : 1.f;
      be[v] = beta ? ((const float*)beta)[c0 + v] : 0.f;
    }
    return;
  }
  // f16: 1.0 = 0x3c00; bf16: 1.0 = 0x3f80
  unsigned short rg[VEC], rb[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
    rg[v] = gamma ? ((const unsigned short*)gamma)[c0 + v] : (unsigned short)(dtype == OCNN_F16 ? 0x3c00 : 0x3f80);
    rb[v] = beta ? ((const unsigned short*)beta)[c0 + v] : (unsigned short)0;
  }
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
    if (dtype == OCNN_F16) {
      ga[v] = to_f32(__builtin_bit_cast(f16, rg[v]));
      be[v] = to_f32(__builtin_bit_cast(f16, rb[v]));
    } else {
      ga[v] = __uint_as_float((uint32_t)rg[v] << 16);
      be[v] = __uint_as_float((uint32_t)rb[v] << 16);
    }
  }
}

__device__ __forceinline__ void bn_store(void* p, int dtype, int c, float v) {
  if (dtype == OCNN_F32) ((float*)p)[c] = v;
  else if (dtype == OCNN_F16) ((f16*)p)[c] = from_f32<f16>(v);
  else ((bf16*)p)[c] = from_f32<bf16>(v);
}

// partial[blk][0][c] = sum_r (x[r][c] - x[0][c]),  partial[blk][1][c] = sum_r (x[r][c] - x[0][c])^2
// over the rows of the workgroup, blocks of 4 rpp of them gridDim.x apart (shifting by the first row keeps the variance free of
// cancellation when the mean is large against the spread).  Thread: VEC channels of every
// rpp-th row.
template <typename T, int VEC>
__global__ __launch_bounds__(256) void bn_stats_kernel(const T* __restrict__ x, int64_t rows, int C, float* __restrict__ partial) {
  typedef BnVec<T, VEC> V;
  __shared__ float s_a[256 * VEC], s_b[256 * VEC];
  const int lpr = C / VEC, rpp = 256 / lpr;
  const int tid = threadIdx.x, rl = tid / lpr, cl = tid - rl * lpr;
  float s1[VEC], s2[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) s1[v] = s2[v] = 0.f;
  if (rl < rpp) {
    const V k = *(const V*)(x + cl * VEC);
    // four rows in flight per thread (rows past the end repeat row 0, whose shifted value is 0)
    for (int64_t r = (int64_t)blockIdx.x * (4 * rpp) + rl; r < rows; r += (int64_t)gridDim.x * (4 * rpp)) {
      V a[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t ru = r + (int64_t)u * rpp;
        a[u] = *(const V*)(x + (ru < rows ? ru * C : 0) + cl * VEC);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < VEC; ++v) {
          const float d = to_f32(a[u].v[v]) - to_f32(k.v[v]);
          s1[v] += d;
          s2[v] += d * d;
        }
    }
  }
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
    s_a[tid * VEC + v] = s1[v];
    s_b[tid * VEC + v] = s2[v];
  }
  __syncthreads();
  if (tid < lpr) {
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      float a = 0.f, b = 0.f;
      for (int g = 0; g < rpp; ++g) {
        a += s_a[(g * lpr + tid) * VEC + v];
        b += s_b[(g * lpr + tid) * VEC + v];
      }
      partial[((int64_t)blockIdx.x * 2 + 0) * C + tid * VEC + v] = a;
      partial[((int64_t)blockIdx.x * 2 + 1) * C + tid * VEC + v] = b;
    }
  }
}

// Sum of the per-workgroup partial sums of a channel, in a fixed order and in fp64: 1024 threads = 256
// lanes x 4 channels, lane l adds the partials l and l + 256 (kBnMaxBlocks is 512), then the 16 lanes of a wave, then
// the waves.  Bound by latency: every partial is requested at once (with 64 lanes, two dependent rounds of
// loads and a chain of 64 LDS reads the launches of an fp16 U-Net step took 8.3 and 7.4 us, now 5.3 and 4.8).
// More workgroups in the reduction do not pay: with 1024 of them 40 k x 256 in fp16 took 22 us instead of 16.
// Returns the channel for the threads that hold a result, -1 for the others.
constexpr int kBnFinishThreads = 1024;
__device__ __forceinline__ int bn_sum_partials(const float* __restrict__ partial, int nblk, int C, double& a,
                                               double& b) {
  constexpr int kLanes = kBnFinishThreads / 4, kEach = kBnMaxBlocks / kLanes;
  __shared__ double s_pa[kBnFinishThreads / 16], s_pb[kBnFinishThreads / 16];
  const int tid = threadIdx.x, l = tid >> 2;
  const int c = blockIdx.x * 4 + (tid & 3);
  float va[kEach], vb[kEach];
#pragma unroll
  for (int u = 0; u < kEach; ++u) {
    const int i = l + kLanes * u;
    const bool in = c < C && i < nblk;
    va[u] = in ? partial[((int64_t)i * 2 + 0) * C + c] : 0.f;
    vb[u] = in ? partial[((int64_t)i * 2 + 1) * C + c] : 0.f;
  }
  double sa = 0.0, sb = 0.0;
#pragma unroll
  for (int u = 0; u < kEach; ++u) {
    sa += (double)va[u];
    sb += (double)vb[u];
  }
#pragma unroll
  for (int o = 4; o < 64; o <<= 1) {
    sa += __shfl_xor(sa, o);
    sb += __shfl_xor(sb, o);
  }
  if ((tid & 63) < 4) {
    s_pa[(tid >> 6) * 4 + (tid & 3)] = sa;
    s_pb[(tid >> 6) * 4 + (tid & 3)] = sb;
  }
  __syncthreads();
  if (l != 0 || c >= C) return -1;
  a = 0.0;
  b = 0.0;
#pragma unroll
  for (int k = 0; k < kBnFinishThreads / 64; ++k) {
    a += s_pa[4 * k + tid];
    b += s_pb[4 * k + tid];
  }
  return c;
}

// mean, biased variance and 1 / sqrt(var + eps) per channel from the partial sums
// running_mean / running_var (dtype rdtype), when given, move towards the batch statistics by
// `factor` (the running variance towards the unbiased one), as torch.nn.functional.batch_norm.
template <typename T>
__global__ __launch_bounds__(kBnFinishThreads) void bn_stats_finish_kernel(
    const float* __restrict__ partial, int nblk, const T* __restrict__ x, int64_t rows, int C, float eps,
    float* __restrict__ mean, float* __restrict__ var, float* __restrict__ invstd, void* running_mean, void* running_var,
    int rdtype, float factor, long long* batches_tracked) {
  // (the module's count of training batches, kept here to spare a launch of its own)
  if (batches_tracked != nullptr && blockIdx.x == 0 && threadIdx.x == 0) *batches_tracked += 1;
  double a, b;
  const int c = bn_sum_partials(partial, nblk, C, a, b);
  if (c < 0) return;
  const double m = a / (double)rows;
  const double v = fmax(b / (double)rows - m * m, 0.0);
  mean[c] = (float)((double)to_f32(x[c]) + m);
  var[c] = (float)v;
  invstd[c] = (float)(1.0 / sqrt(v + (double)eps));
  if (running_mean) {
    const float unbiased = (float)(v * ((double)rows / (double)max(rows - 1, (int64_t)1)));
    bn_store(running_mean, rdtype, c, (1.f - factor) * bn_param(running_mean, rdtype, c, 0.f) + factor * mean[c]);
    bn_store(running_var, rdtype, c, (1.f - factor) * bn_param(running_var, rdtype, c, 0.f) + factor * unbiased);
  }
}

// y = (x - mean) * (invstd * gamma) + beta (+ res), then max(., 0) when relu.  A thread keeps the
// constants of its VEC channels in registers and walks the rows back to the first, four rows in flight.
// run_mean, run_var (dtype rdtype), when given, take the place of mean and invstd: a module's running statistics as it holds
// them, the reciprocal formed here (made into mean and invstd by passes of their own they were four of the five launches of a
// layer in evaluation).  BITS: the mask of BnMasked is kept.  (A kernel of its own: a mask that may not be there cost the
// others registers, in fp32 a workgroup a CU of six, 250 k x 192 66.7 -> 70.7 us, 700 k x 64 60.7 -> 62.7.)
template <typename T, int VEC, bool BITS>
__global__ __launch_bounds__(256) void bn_apply_kernel(const T* __restrict__ x, int64_t rows, int C,
                                                       const float* __restrict__ mean,
                                                       const float* __restrict__ invstd,
                                                       const void* __restrict__ gamma,
                                                       const void* __restrict__ beta, int pdtype, int relu,
                                                       const T* __restrict__ res, T* __restrict__ y,
                                                       const void* __restrict__ run_mean,
                                                       const void* __restrict__ run_var, int rdtype, float eps,
                                                       uint8_t* __restrict__ mask) {
  typedef BnVec<T, VEC> V;
  const int lpr = C / VEC, rpp = 256 / lpr;
  const int tid = threadIdx.x, rl = tid / lpr, cl = tid - rl * lpr;
  if (rl >= rpp) return;
  float m[VEC], sc[VEC], be[VEC];
  if (run_var) {
    bn_params<VEC>(run_var, run_mean, rdtype, cl * VEC, sc, m);
#pragma unroll
    for (int v = 0; v < VEC; ++v) sc[v] = 1.f / sqrtf(sc[v] + eps);
  } else {
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      m[v] = mean[cl * VEC + v];
      sc[v] = invstd[cl * VEC + v];
    }
  }
  {
    float ga[VEC];
    bn_params<VEC>(gamma, beta, pdtype, cl * VEC, ga, be);
#pragma unroll
    for (int v = 0; v < VEC; ++v) sc[v] *= ga[v];
  }
  const int64_t last = (rows + 4 * rpp - 1) / (4 * rpp) - 1;
  for (int64_t at = last - blockIdx.x; at >= 0; at -= gridDim.x) {
    const int64_t r = at * (4 * rpp) + rl;
    V a[4], b[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t ru = r + (int64_t)u * rpp;
      if (ru < rows) {
        a[u] = *(const V*)(x + ru * C + cl * VEC);
        if (res) b[u] = *(const V*)(res + ru * C + cl * VEC);
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t ru = r + (int64_t)u * rpp;
      if (ru >= rows) continue;
      V o;
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        float t = (to_f32(a[u].v[v]) - m[v]) * sc[v] + be[v];
        if (res) t = to_f32(from_f32<T>(t)) + to_f32(b[u].v[v]);      // (rounded as the separate passes would)
        if (relu) t = fmaxf(t, 0.f);
        o.v[v] = from_f32<T>(t);
      }
      *(V*)(y + ru * C + cl * VEC) = o;
      if constexpr (BITS) {
        uint32_t bits = 0;
#pragma unroll
        for (int v = 0; v < VEC; ++v) bits |= (to_f32(o.v[v]) > 0.f ? 1u : 0u) << v;
        mask[ru * lpr + cl] = (uint8_t)bits;
      }
    }
  }
}

// What the ReLU of the forward pass let through: a function of x alone, or, where a residual was added, its output or a byte
// of bits for each VEC channels.  The bits are 1/16 of the output, which both passes of the backward pass read otherwise;
// forward + backward with a residual, us, from the output / from the bits: fp16 1.11 M x 96 508 / 431, 460 k x 128 284 / 239,
// 200 k x 192 202 / 169, fp32 300 k x 64 171 / 155 (writing them: 1 - 4 of that).  A kernel for each, since the rows of an output
// that may not be there cost the others registers, a wave a SIMD of the elementwise pass: without residual fp16 1.11 M x 96
// 361 / 345, 200 k x 192 151 / 143.
enum BnMask { kBnOfX, kBnOfY, kBnBits };
template <typename T, int VEC, int MASK> struct BnMasked {
  typedef typename std::conditional<MASK == kBnBits, uint8_t, BnVec<T, VEC>>::type V;
  V m;
  __device__ __forceinline__ void load(const void* __restrict__ mask, int64_t vec) {
    if constexpr (MASK != kBnOfX) m = ((const V*)mask)[vec];
  }
  __device__ __forceinline__ bool passed(int v, float of_x) const {
    if constexpr (MASK == kBnOfY) return to_f32(m.v[v]) > 0.f;
    else if constexpr (MASK == kBnBits) return (m >> v) & 1;
    else return of_x > 0.f;
  }
};

// partial[blk][0][c] = sum_r dy'[r][c],  partial[blk][1][c] = sum_r dy'[r][c] * xhat[r][c], with
// xhat = (x - mean) * invstd and dy' = dy where the forward output was positive (relu) or dy.
template <typename T, int VEC, int MASK>
__global__ __launch_bounds__(256) void bn_bwd_stats_kernel(const T* __restrict__ x, const T* __restrict__ dy,
                                                           int64_t rows, int C,
                                                           const float* __restrict__ mean,
                                                           const float* __restrict__ invstd,
                                                           const void* __restrict__ gamma,
                                                           const void* __restrict__ beta, int pdtype, int relu,
                                                           const void* __restrict__ mask,
                                                           float* __restrict__ partial) {
  typedef BnVec<T, VEC> V;
  __shared__ float s_a[256 * VEC], s_b[256 * VEC];
  const int lpr = C / VEC, rpp = 256 / lpr;
  const int tid = threadIdx.x, rl = tid / lpr, cl = tid - rl * lpr;
  float s1[VEC], s2[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) s1[v] = s2[v] = 0.f;
  if (rl < rpp) {
    float m[VEC], is[VEC], ga[VEC], be[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      m[v] = mean[cl * VEC + v];
      is[v] = invstd[cl * VEC + v];
    }
    bn_params<VEC>(gamma, beta, pdtype, cl * VEC, ga, be);
    // (four rows of both tensors in flight)
    for (int64_t r = (int64_t)blockIdx.x * (4 * rpp) + rl; r < rows; r += (int64_t)gridDim.x * (4 * rpp)) {
      V a[4], g[4];
      BnMasked<T, VEC, MASK> pass[4];
      bool ok[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t ru = r + (int64_t)u * rpp;
        ok[u] = ru < rows;
        a[u] = *(const V*)(x + (ok[u] ? ru * C : 0) + cl * VEC);
        g[u] = *(const V*)(dy + (ok[u] ? ru * C : 0) + cl * VEC);
        pass[u].load(mask, (ok[u] ? ru * lpr : 0) + cl);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < VEC; ++v) {
          const float xc = to_f32(a[u].v[v]) - m[v];
          const float xh = xc * is[v];
          float d = ok[u] ? to_f32(g[u].v[v]) : 0.f;
          if (relu && !pass[u].passed(v, xc * (is[v] * ga[v]) + be[v])) d = 0.f;       // the forward pass's expression
          s1[v] += d;
          s2[v] += d * xh;
        }
    }
  }
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
    s_a[tid * VEC + v] = s1[v];
    s_b[tid * VEC + v] = s2[v];
  }
  __syncthreads();
  if (tid < lpr) {
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      float a = 0.f, b = 0.f;
      for (int g = 0; g < rpp; ++g) {
        a += s_a[(g * lpr + tid) * VEC + v];
        b += s_b[(g * lpr + tid) * VEC + v];
      }
      partial[((int64_t)blockIdx.x * 2 + 0) * C + tid * VEC + v] = a;
      partial[((int64_t)blockIdx.x * 2 + 1) * C + tid * VEC + v] = b;
    }
  }
}

// (gw / gb: the same sums in the parameters' dtype, when given)
__global__ __launch_bounds__(kBnFinishThreads) void bn_bwd_finish_kernel(const float* __restrict__ partial, int nblk, int C,
                                     float* __restrict__ dbeta, float* __restrict__ dgamma, void* gw, void* gb,
                                     int pdtype) {
  double a, b;
  const int c = bn_sum_partials(partial, nblk, C, a, b);
  if (c < 0) return;
  dbeta[c] = (float)a;
  dgamma[c] = (float)b;
  if (gw) bn_store(gw, pdtype, c, (float)b);
  if (gb) bn_store(gb, pdtype, c, (float)a);
}

// training: dx = gamma * invstd * (dy' - dbeta / N - xhat * dgamma / N); with fixed statistics
// (evaluation mode): dx = gamma * invstd * dy'.  Thread layout as in bn_apply_kernel.
template <typename T, int VEC, int MASK>
__global__ __launch_bounds__(256) void bn_bwd_apply_kernel(const T* __restrict__ x, const T* __restrict__ dy,
                                                           int64_t rows, int C,
                                                           const float* __restrict__ mean,
                                                           const float* __restrict__ invstd,
                                                           const void* __restrict__ gamma,
                                                           const void* __restrict__ beta, int pdtype, int relu,
                                                           const float* __restrict__ dbeta,
                                                           const float* __restrict__ dgamma, int training,
                                                           const void* __restrict__ mask, T* __restrict__ dres,
                                                           T* __restrict__ dx) {
  typedef BnVec<T, VEC> V;
  const int lpr = C / VEC, rpp = 256 / lpr;
  const int tid = threadIdx.x, rl = tid / lpr, cl = tid - rl * lpr;
  if (rl >= rpp) return;
  const float inv_n = 1.0f / (float)rows;
  float m[VEC], is[VEC], sc[VEC], be[VEC], db[VEC], dg[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
    const int c = cl * VEC + v;
    m[v] = mean[c];
    is[v] = invstd[c];
    db[v] = training ? dbeta[c] * inv_n : 0.f;
    dg[v] = training ? dgamma[c] * inv_n : 0.f;
  }
  bn_params<VEC>(gamma, beta, pdtype, cl * VEC, sc, be);
#pragma unroll
  for (int v = 0; v < VEC; ++v) sc[v] *= is[v];
  const int64_t last = (rows + 2 * rpp - 1) / (2 * rpp) - 1;       // (four rows in flight cost more in occupancy than they gain)
  for (int64_t at = last - blockIdx.x; at >= 0; at -= gridDim.x) {
    const int64_t r = at * (2 * rpp) + rl;
    V a[2], g[2];
    BnMasked<T, VEC, MASK> pass[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t ru = r + (int64_t)u * rpp;
      if (ru < rows) {
        a[u] = *(const V*)(x + ru * C + cl * VEC);
        g[u] = *(const V*)(dy + ru * C + cl * VEC);
        pass[u].load(mask, ru * lpr + cl);
      }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t ru = r + (int64_t)u * rpp;
      if (ru >= rows) continue;
      V o, gr;
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        const float xc = to_f32(a[u].v[v]) - m[v];
        float d = to_f32(g[u].v[v]);
        if (relu && !pass[u].passed(v, xc * sc[v] + be[v])) d = 0.f;
        gr.v[v] = from_f32<T>(d);                                      // the gradient of the residual
        if (training) d = d - db[v] - (xc * is[v]) * dg[v];
        o.v[v] = from_f32<T>(d * sc[v]);
      }
      *(V*)(dx + ru * C + cl * VEC) = o;
      if (dres) *(V*)(dres + ru * C + cl * VEC) = gr;
    }
  }
}

// ---- few rows: one launch, or two ----
//
// At some ten thousand rows and below (the coarse levels of a network, small clouds) a pass is launch latency, and a
// training step's forward and backward pass have three launches each (sums, their sum, the elementwise pass).  Here a
// workgroup of 1024 threads has 64 or 128 bytes of a row (LANES threads) to itself, of all rows or of a range of them:
// * one launch: sums, statistics and the elementwise pass follow each other in the workgroup, the rows come from L2 the
//   second time;
// * two: the sums of every range, and an elementwise pass whose workgroups add the ranges' sums themselves, while their rows are on
//   their way: of so few channels that is nothing (of whole rows it was a launch of its own).
// Forward / backward in us, three launches before, now: fp32 4096 x 128 10.9 / 13.4, 7.8 / 9.1; 20 k x 128 15.4 / 21.7, 9.7 / 17.3;
// 39 k x 96 17.9 / 25.0, 12.8 / 22.3; fp16 2048 x 256 (one launch before) 12.8 / 20.2, 9.5 / 12.5; 20 k x 96 15.8 / 22.5, 11.1 / 15.4;
// 60 k x 128 24.4 / 39.5, 17.5 / 31.8.  The lines:
// * one launch up to 1024 rows: fp32 x 256 800 rows 6.3 / 7.9, two 7.4 / 8.6; 1425 rows 7.7 / 10.1, two 7.2 / 8.8;
// * the three launches, whose workgroups have whole rows, where the elementwise pass is more than a round of workgroups, of
//   which a CU holds one (registers).  Two / three launches: one round, fp32 130 k x 32 forward 14.2 / 19.4, 60 k x 32 backward
//   14.1 / 18.0, 60 k x 40 forward 12.6 / 16.1; fp16 64 k x 120 forward 20.2 / 24.1.  What more rounds are worth hangs on the rows:
//   - of one line of 128 bytes or less, and of channels that leave a workgroup's last part of a row empty, nothing: fp32
//     160 k x 16 17.9 / 17.6, 27.6 / 22.7, 98 k x 32 backward 23.7 / 22.2, 66 k x 40 17.4 / 16.6, 28.8 / 21.7, 36 k x 104 19.9 /
//     18.1, 31.9 / 24.5; fp16 131 k x 64 backward 39.9 / 35.3, 150 k x 64 33.3 / 25.6, 24 k x 200 backward 38.0 / 33.4 (less than
//     a line in two parts backward a little: 84 k x 40 27.3 / 29.4, 90 k x 48 29.7 / 32.9, 84 k x 56 30.8 / 32.3);
//   - forward two rounds in fp32 (66 k x 64 17.4 / 20.0, 131 k x 64 25.0 / 25.8, 33 k x 256 21.0 / 26.4; the third 87 k x 96 26.3 /
//     25.3), in 16 bits of whole 512 bytes (66 k x 256 27.8 / 29.5, 33 k x 512 28.9 / 30.8; 74 k x 128 27.0 / 25.0, 60 k x 192
//     26.6 / 25.5, 40 k x 320 29.2 / 27.1);
//   - backward two (fp16 66 k x 128 36.3 / 40.0, 82 k 46.4 / 42.9, 30 k x 320 44.7 / 41.6; fp32 60 k x 64 23.1 / 25.4, 74 k 29.7 /
//     29.3), of more than 256 bytes in fp32 and of whole 512 bytes in 16 bits two and a half (fp32 37 k x 128 26.0 / 29.2,
//     9.2 k x 512 27.7 / 30.3; fp16 41 k x 256 40.1 / 42.0, 20 k x 512 42.2 / 43.4);
// * 128 bytes of a row, whole lines, from 4 MB on in fp32 (20 k x 128: 9.7 / 17.3, with 64 bytes 11.0 / 23.7), from 12 MB on in 16
//   bits, where they are 64 channels (39 k x 96 15.4 / 28.6, with 64 bytes 13.1 / 20.6; 33 k x 256 21.3 / 37.5, 22.4 / 46.2).
constexpr int kBnSlabThreads = 1024;
constexpr int64_t kBnSmallRows = 1024, kBnRound = 256, kBnWideF32 = 4 << 20, kBnWide16 = 12 << 20;
constexpr int kBnUnrollForward = 4, kBnUnrollBackward = 2;   // passes over the rows that a workgroup of the elementwise pass takes, at most
constexpr int kBnSlabRanges = 64;         // of the sums, at most (more where the channels are few slabs: a workgroup on every CU)

// sums over the workgroup of the 2 VEC values of each thread, per thread of a row: s_out[kind][channel of the
// workgroup], in a fixed order: 2 VEC threads' values in fp64, then those sums one after the other.
template <int VEC, int LANES>
__device__ __forceinline__ void bn_slab_sums(const float (&s1)[VEC], const float (&s2)[VEC], float* s_f, double* s_d,
                                             double* s_out) {
  constexpr int lpr = LANES;
  const int tid = threadIdx.x, cl = tid % lpr, rl = tid / lpr;
  constexpr int pitch = kBnSlabThreads / lpr + 1, sums = 2 * lpr * VEC, segments = kBnSlabThreads / sums;
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
    s_f[(cl * VEC + v) * pitch + rl] = s1[v];
    s_f[((lpr + cl) * VEC + v) * pitch + rl] = s2[v];
  }
  __syncthreads();
  {
    const float* p = s_f + (tid % sums) * pitch + tid / sums * (2 * VEC);
    double a = 0.0;
#pragma unroll
    for (int i = 0; i < 2 * VEC; ++i) a += (double)p[i];
    s_d[tid] = a;
  }
  __syncthreads();
  if (tid < sums) {
    double a = 0.0;
#pragma unroll 8
    for (int i = 0; i < segments; ++i) a += s_d[i * sums + tid];
    s_out[tid] = a;
  }
  __syncthreads();
}

// partial[range][kind][channel] of the workgroup's channels added over the ranges, in their order by segments
template <int VEC, int LANES>
__device__ __forceinline__ void bn_slab_fold(const double* __restrict__ partial, int ranges, int C, double* s_d, double* s_out) {
  constexpr int width = LANES * VEC, sums = 2 * width, segments = kBnSlabThreads / sums;
  const int tid = threadIdx.x, j = tid % sums, seg = tid / sums;
  const int kind = j / width, c = (int)blockIdx.x * width + j % width;
  double a = 0.0;
  if (c < C)
    for (int i = seg; i < ranges; i += segments) a += partial[((int64_t)i * 2 + kind) * C + c];
  s_d[tid] = a;
  __syncthreads();
  if (tid < sums) {
    double t = 0.0;
    for (int i = 0; i < min(ranges, segments); ++i) t += s_d[i * sums + tid];
    s_out[tid] = t;
  }
  __syncthreads();
}

// sums of the rows r0 .. r1 - 1, shifted by row 0 (whose shifted value, 0, stands in for rows past the end)
template <typename T, int VEC, int LANES>
__device__ __forceinline__ void bn_slab_rows(const T* __restrict__ x, int r0, int r1, int C, int c0, float (&s1)[VEC], float (&s2)[VEC]) {
  typedef BnVec<T, VEC> V;
  constexpr int rpp = kBnSlabThreads / LANES;
  const V k = *(const V*)(x + c0);
  for (int r = r0 + (int)threadIdx.x / LANES; r < r1; r += 4 * rpp) {
    V a[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) a[u] = *(const V*)(x + (r + u * rpp < r1 ? (int64_t)(r + u * rpp) * C : 0) + c0);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        const float d = to_f32(a[u].v[v]) - to_f32(k.v[v]);
        s1[v] += d;
        s2[v] += d * d;
      }
  }
}

struct BnStats {                 // where a training pass leaves its statistics
  float eps;
  float *mean, *var, *invstd;
  void *running_mean, *running_var;
  int rdtype;
  float factor;
  long long* batches_tracked;
};

// mean and 1 / sqrt(var + eps) of the workgroup's channels to LDS; `keep`: also to where they are kept
template <typename T, int VEC, int LANES>
__device__ __forceinline__ void bn_slab_finish(const double* s_sum, const T* __restrict__ x, int rows, int C, const BnStats& st,
                                               bool keep, float* s_mean, float* s_is) {
  constexpr int width = LANES * VEC;
  const int tid = threadIdx.x, c = (int)blockIdx.x * width + tid;
  if (keep && st.batches_tracked != nullptr && blockIdx.x == 0 && tid == 0) *st.batches_tracked += 1;
  if (tid < width && c < C) {
    const double m = s_sum[tid] / (double)rows;
    const double va = fmax(s_sum[width + tid] / (double)rows - m * m, 0.0);
    const float mf = (float)((double)to_f32(x[c]) + m), isf = (float)(1.0 / sqrt(va + (double)st.eps));
    s_mean[tid] = mf;
    s_is[tid] = isf;
    if (keep) {
      st.mean[c] = mf;
      st.invstd[c] = isf;
      st.var[c] = (float)va;
      if (st.running_mean) {
        const float unbiased = (float)(va * ((double)rows / (double)max(rows - 1, 1)));
        bn_store(st.running_mean, st.rdtype, c, (1.f - st.factor) * bn_param(st.running_mean, st.rdtype, c, 0.f) + st.factor * mf);
        bn_store(st.running_var, st.rdtype, c, (1.f - st.factor) * bn_param(st.running_var, st.rdtype, c, 0.f) + st.factor * unbiased);
      }
    }
  }
  __syncthreads();
}

// four rows of a thread from row r on (those below r1), requested and normalised
template <typename T, int VEC, int LANES> struct BnRows {
  static constexpr int kPass = kBnSlabThreads / LANES;
  BnVec<T, VEC> a[4], b[4];
  __device__ __forceinline__ void load(const T* __restrict__ x, const T* __restrict__ res, int r, int r1, int C, int c0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t at = (int64_t)(r + u * kPass) * C + c0;
      if (r + u * kPass < r1) {
        a[u] = *(const BnVec<T, VEC>*)(x + at);
        if (res) b[u] = *(const BnVec<T, VEC>*)(res + at);
      }
    }
  }
  __device__ __forceinline__ void apply(const float (&m)[VEC], const float (&sc)[VEC], const float (&be)[VEC], bool with, int relu,
                                        T* __restrict__ y, int r, int r1, int C, int c0) const {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (r + u * kPass >= r1) continue;
      BnVec<T, VEC> o;
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        float t = (to_f32(a[u].v[v]) - m[v]) * sc[v] + be[v];
        if (with) t = to_f32(from_f32<T>(t)) + to_f32(b[u].v[v]);
        if (relu) t = fmaxf(t, 0.f);
        o.v[v] = from_f32<T>(t);
      }
      *(BnVec<T, VEC>*)(y + (int64_t)(r + u * kPass) * C + c0) = o;
    }
  }
};

// ranges = 1, partial null: the whole batch norm.  SUMS: the sums of range blockIdx.y alone, to partial.  Else: rows of range
// blockIdx.y (of `per`) with the sums of `ranges` ranges.
template <typename T, int VEC, int LANES, bool SUMS>
__global__ __launch_bounds__(kBnSlabThreads) void bn_slab_kernel(
    const T* __restrict__ x, int rows, int C, int per, double* __restrict__ partial, int ranges, BnStats st,
    const void* __restrict__ gamma, const void* __restrict__ beta, int pdtype, int relu, const T* __restrict__ res,
    T* __restrict__ y) {
  constexpr int lpr = LANES, rpp = kBnSlabThreads / LANES, width = lpr * VEC;
  __shared__ float s_f[2 * VEC * (kBnSlabThreads + lpr)];
  __shared__ double s_d[kBnSlabThreads], s_sum[2 * width];
  __shared__ float s_mean[width], s_is[width];
  const int tid = threadIdx.x, cl = tid % lpr, rl = tid / lpr;
  const int c0 = (int)blockIdx.x * width + cl * VEC;         // first channel of the thread
  const bool ok = c0 < C;
  const int r0 = (int)blockIdx.y * per, r1 = min(rows, r0 + per);
  BnRows<T, VEC, LANES> first;
  if (!SUMS && partial != nullptr) {
    if (ok) first.load(x, res, r0 + rl, r1, C, c0);          // (on their way under the sums)
    bn_slab_fold<VEC, LANES>(partial, ranges, C, s_d, s_sum);
  } else {
    float s1[VEC], s2[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) s1[v] = s2[v] = 0.f;
    if (ok) bn_slab_rows<T, VEC, LANES>(x, r0, r1, C, c0, s1, s2);
    bn_slab_sums<VEC, LANES>(s1, s2, s_f, s_d, s_sum);
  }
  if constexpr (SUMS) {
    const int c = (int)blockIdx.x * width + tid % width;
    if (tid < 2 * width && c < C) partial[((int64_t)blockIdx.y * 2 + tid / width) * C + c] = s_sum[tid];
  } else {
    bn_slab_finish<T, VEC, LANES>(s_sum, x, rows, C, st, blockIdx.y == 0, s_mean, s_is);
    if (!ok) return;
    float m[VEC], sc[VEC], be[VEC];
    bn_params<VEC>(gamma, beta, pdtype, c0, sc, be);
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      m[v] = s_mean[cl * VEC + v];
      sc[v] = s_is[cl * VEC + v] * sc[v];
    }
    for (int r = r0 + rl; r < r1; r += 4 * rpp) {
      if (partial == nullptr || r != r0 + rl) first.load(x, res, r, r1, C, c0);
      first.apply(m, sc, be, res != nullptr, relu, y, r, r1, C, c0);
    }
  }
}

// two rows of a thread, for the gradient: x, dy and the forward output where it is the mask
template <typename T, int VEC, int LANES> struct BnBwdRows {
  static constexpr int kPass = kBnSlabThreads / LANES;
  BnVec<T, VEC> a[2], g[2], ym[2];
  __device__ __forceinline__ void load(const T* __restrict__ x, const T* __restrict__ dy, const T* __restrict__ ymask, int r,
                                       int r1, int C, int c0) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t at = (r + u * kPass < r1 ? (int64_t)(r + u * kPass) * C : 0) + c0;   // (past the end: row 0)
      a[u] = *(const BnVec<T, VEC>*)(x + at);
      g[u] = *(const BnVec<T, VEC>*)(dy + at);
      ym[u] = a[u];                                          // (defined without a mask, too)
      if (ymask) ym[u] = *(const BnVec<T, VEC>*)(ymask + at);
    }
  }
};

// the gradient, as bn_bwd_stats_kernel, bn_bwd_finish_kernel and bn_bwd_apply_kernel after each other; ranges, partial and
// SUMS as in bn_slab_kernel
template <typename T, int VEC, int LANES, bool SUMS>
__global__ __launch_bounds__(kBnSlabThreads) void bn_bwd_slab_kernel(
    const T* __restrict__ x, const T* __restrict__ dy, int rows, int C, int per, double* __restrict__ partial, int ranges,
    const float* __restrict__ mean, const float* __restrict__ invstd, const void* __restrict__ gamma,
    const void* __restrict__ beta, int pdtype, int relu, int training, const T* __restrict__ ymask, float* __restrict__ dbeta,
    float* __restrict__ dgamma, void* gw, void* gb, T* __restrict__ dres, T* __restrict__ dx) {
  typedef BnVec<T, VEC> V;
  constexpr int lpr = LANES, rpp = kBnSlabThreads / LANES, width = lpr * VEC;
  __shared__ float s_f[2 * VEC * (kBnSlabThreads + lpr)];
  __shared__ double s_d[kBnSlabThreads], s_sum[2 * width];
  const int tid = threadIdx.x, cl = tid % lpr, rl = tid / lpr;
  const int c0 = (int)blockIdx.x * width + cl * VEC;
  const bool ok = c0 < C;
  const int r0 = (int)blockIdx.y * per, r1 = min(rows, r0 + per);
  float m[VEC], is[VEC], ga[VEC], be[VEC];
  BnBwdRows<T, VEC, LANES> v2;
  if (ok) {
    if (!SUMS && partial != nullptr) v2.load(x, dy, ymask, r0 + rl, r1, C, c0);
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      m[v] = mean[c0 + v];
      is[v] = invstd[c0 + v];
    }
    bn_params<VEC>(gamma, beta, pdtype, c0, ga, be);
  }
  // dy' of a value: dy where the forward output was positive (or without the ReLU)
  auto passed = [&](int u, int v, float xc, float scale) {
    const float seen = ymask ? to_f32(v2.ym[u].v[v]) : xc * scale + be[v];
    const bool on = !relu || seen > 0.f;
    return on ? to_f32(v2.g[u].v[v]) : 0.f;
  };
  if (!SUMS && partial != nullptr) {
    bn_slab_fold<VEC, LANES>(partial, ranges, C, s_d, s_sum);
  } else {
    float s1[VEC], s2[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) s1[v] = s2[v] = 0.f;
    if (ok)
      for (int r = r0 + rl; r < r1; r += 2 * rpp) {
        v2.load(x, dy, ymask, r, r1, C, c0);
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int v = 0; v < VEC; ++v) {
            const float xc = to_f32(v2.a[u].v[v]) - m[v];
            const float xh = xc * is[v];
            const float d = r + u * rpp < r1 ? passed(u, v, xc, is[v] * ga[v]) : 0.f;
            s1[v] += d;
            s2[v] += d * xh;
          }
      }
    bn_slab_sums<VEC, LANES>(s1, s2, s_f, s_d, s_sum);
  }
  if constexpr (SUMS) {
    const int c = (int)blockIdx.x * width + tid % width;
    if (tid < 2 * width && c < C) partial[((int64_t)blockIdx.y * 2 + tid / width) * C + c] = s_sum[tid];
  } else {
    if (tid < width && blockIdx.y == 0) {
      const int c = (int)blockIdx.x * width + tid;
      if (c < C) {
        const float a = (float)s_sum[tid], b = (float)s_sum[width + tid];
        dbeta[c] = a;
        dgamma[c] = b;
        if (gw) bn_store(gw, pdtype, c, b);
        if (gb) bn_store(gb, pdtype, c, a);
      }
    }
    if (!ok) return;
    const float inv_n = 1.0f / (float)rows;
    float db[VEC], dg[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      db[v] = training ? (float)s_sum[cl * VEC + v] * inv_n : 0.f;
      dg[v] = training ? (float)s_sum[width + cl * VEC + v] * inv_n : 0.f;
      ga[v] *= is[v];
    }
    for (int r = r0 + rl; r < r1; r += 2 * rpp) {
      if (partial == nullptr || r != r0 + rl) v2.load(x, dy, ymask, r, r1, C, c0);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (r + u * rpp >= r1) continue;
        const int64_t at = (int64_t)(r + u * rpp) * C + c0;
        V o, gr;
#pragma unroll
        for (int v = 0; v < VEC; ++v) {
          const float xc = to_f32(v2.a[u].v[v]) - m[v];
          float d = passed(u, v, xc, ga[v]);
          gr.v[v] = from_f32<T>(d);
          if (training) d = d - db[v] - (xc * is[v]) * dg[v];
          o.v[v] = from_f32<T>(d * ga[v]);
        }
        *(V*)(dx + at) = o;
        if (dres) *(V*)(dres + at) = gr;
      }
    }
  }
}

// How a pass is launched: LANES and, for two launches, the rows of a workgroup of the sums (a range) and of one of the
// elementwise pass: whole passes, as few as give every CU a workgroup, `unroll` of them at most.
struct BnSlabs {
  int lanes, slabs, sums_per, ranges, per, parts;
  bool split;                    // two launches
};
static BnSlabs bn_slabs(int dtype, int64_t rows, int channels, int unroll) {
  BnSlabs s;
  const int vec = dtype == OCNN_F32 ? 4 : 8;
  s.split = rows > kBnSmallRows;
  s.lanes = s.split && rows * channels * 16 / vec >= (dtype == OCNN_F32 ? kBnWideF32 : kBnWide16) ? 8 : 4;
  s.slabs = (int)cdiv(channels, s.lanes * vec);
  if (!s.split) {
    s.sums_per = s.per = (int)rows;
    s.ranges = s.parts = 1;
    return s;
  }
  const int64_t pass = kBnSlabThreads / s.lanes;
  const int64_t some = std::min<int64_t>(unroll, std::max<int64_t>(1, cdiv(rows * s.slabs, kBnRound * pass))) * pass;
  s.sums_per = (int)std::max(some, align_up(cdiv(rows, std::max(kBnSlabRanges, 256 / s.slabs)), pass));
  s.ranges = (int)cdiv(rows, s.sums_per);
  s.per = (int)some;
  s.parts = (int)cdiv(rows, s.per);
  return s;
}

// (three launches for rows of more workgroups than these; the lines above)
static bool bn_slabs_take(int dtype, int64_t rows, int channels, bool backward) {
  if (rows <= kBnSmallRows) return true;
  if (channels < (dtype == OCNN_F32 ? 16 : 32)) return false;
  const int unroll = backward ? kBnUnrollBackward : kBnUnrollForward;
  const BnSlabs s = bn_slabs(dtype, rows, channels, unroll);
  const int vec = dtype == OCNN_F32 ? 4 : 8, row_bytes = channels * 16 / vec;
  const bool wide = dtype == OCNN_F32 || row_bytes % 512 == 0;
  int64_t most = kBnRound;
  if (channels % (s.lanes * vec) == 0 && row_bytes > 128)
    most = backward ? (wide && row_bytes > 256 ? 5 * kBnRound / 2 : 2 * kBnRound) : (wide ? 2 * kBnRound : kBnRound);
  else if (backward && row_bytes < 128 && s.slabs == 2)
    most = 2 * kBnRound;
  return rows * s.slabs <= most * unroll * (kBnSlabThreads / s.lanes);
}

}  // namespace ocnn

using namespace ocnn;

#define OCNN_DISPATCH_DTYPE(dtype, ...)                      \
  do {                                                       \
    if (dtype == OCNN_F32) { typedef float T; __VA_ARGS__; } \
    else if (dtype == OCNN_F16) { typedef f16 T; __VA_ARGS__; } \
    else { typedef bf16 T; __VA_ARGS__; }                    \
  } while (0)

static int bn_vec(int dtype) { return dtype == OCNN_F32 ? 4 : 8; }

extern "C" int ocnn_batch_norm_supported(int dtype, int64_t rows, int channels) {
  if (dtype < 0 || dtype > 2) return 0;
  const int vec = bn_vec(dtype);
  if (channels < vec || channels % vec != 0 || channels / vec > 256) return 0;
  return rows >= 1;
}

// workgroups: one for every four rows a thread, max_blocks at most
static int bn_blocks(int dtype, int64_t rows, int channels, int max_blocks) {
  const int rpp = 256 / (channels / bn_vec(dtype));
  return (int)std::min<int64_t>(max_blocks, cdiv(rows, 4 * rpp));
}

// The backward elementwise pass reads two tensors from where the sums ended, back through the memory-side cache, and writes one or
// two: of more than four workgroups a CU the streams are more than that takes.  fp32, us, seven (with a residual six) a CU / four:
// 250 k x 192 98.6 / 95.7 (132.6 / 128.5), 400 k x 128 104.5 / 101.1 (140.4 / 135.1), 700 k x 64 89.4 / 87.3 (121.4 / 116.1).  (16 bit has
// four by its registers.)
constexpr int kBnBackwardPerCu = 4;

// Workgroups of 256 threads of `kernel` that the device holds at once, `most` a CU and kBnApplyBlocks at most:
// an elementwise pass launched with more runs them in rounds, and the last round leaves CUs idle.
static int bn_resident_blocks(const void* kernel, int most = 8) {
  static std::mutex mu;
  static std::vector<std::pair<const void*, int>> known;
  std::lock_guard<std::mutex> lock(mu);
  for (const auto& k : known)
    if (k.first == kernel) return k.second;
  int per_cu = 0, dev = 0, n_cu = 256;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev);
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 256, 0) != hipSuccess || per_cu < 1) {
    (void)hipGetLastError();
    per_cu = 2;
  }
  const int cap = std::min(kBnApplyBlocks, std::max(1, std::min(per_cu, most) * n_cu));
  known.emplace_back(kernel, cap);
  return cap;
}

extern "C" int64_t ocnn_batch_norm_workspace_bytes(int channels) {
  return align_up((int64_t)kBnMaxBlocks * 2 * channels * 4, 256);
}

extern "C" int ocnn_batch_norm_stats(int dtype, const void* x, int64_t rows, int channels, float eps,
                                     float* mean, float* var, float* invstd, void* running_mean,
                                     void* running_var, int running_dtype, float factor,
                                     int64_t* batches_tracked, void* workspace, int64_t workspace_bytes,
                                     void* stream) {
  OCNN_REQUIRE(ocnn_batch_norm_supported(dtype, rows, channels), "batch_norm_stats: shape not supported");
  OCNN_REQUIRE_PTRS("batch_norm_stats", x, mean, var, invstd, workspace);
  OCNN_REQUIRE(workspace_bytes >= ocnn_batch_norm_workspace_bytes(channels), "batch_norm_stats: workspace too small");
  hipStream_t st = (hipStream_t)stream;
  const int nblk = bn_blocks(dtype, rows, channels, kBnMaxBlocks);
  float* partial = (float*)workspace;
  OCNN_DISPATCH_DTYPE(dtype, {
    constexpr int VEC = 16 / sizeof(T);
    hipLaunchKernelGGL((bn_stats_kernel<T, VEC>), dim3(nblk), dim3(256), 0, st, (const T*)x, rows, channels, partial);
    hipLaunchKernelGGL(bn_stats_finish_kernel<T>, dim3((unsigned)cdiv(channels, 4)), dim3(kBnFinishThreads), 0, st,
                       partial, nblk, (const T*)x, rows, channels, eps, mean, var, invstd, running_mean, running_var, running_dtype,
                       factor, (long long*)batches_tracked);
  });
  return check_launch("batch_norm_stats");
}

static int bn_apply(int dtype, const void* x, int64_t rows, int channels, const float* mean, const float* invstd,
                    const void* gamma, const void* beta, int param_dtype, int relu, const void* residual, void* y,
                    const void* run_mean, const void* run_var, int run_dtype, float eps, uint8_t* mask, hipStream_t st) {
  OCNN_DISPATCH_DTYPE(dtype, {
    constexpr int VEC = 16 / sizeof(T);
    const auto launch = [&](auto kernel) {
      const int nblk = bn_blocks(dtype, rows, channels, bn_resident_blocks((const void*)kernel));
      hipLaunchKernelGGL(kernel, dim3(nblk), dim3(256), 0, st, (const T*)x, rows, channels, mean, invstd, gamma, beta, param_dtype,
                         relu, (const T*)residual, (T*)y, run_mean, run_var, run_dtype, eps, mask);
    };
    if (mask) launch(bn_apply_kernel<T, VEC, true>);
    else launch(bn_apply_kernel<T, VEC, false>);
  });
  return check_launch("batch_norm_apply");
}

extern "C" int ocnn_batch_norm_apply(int dtype, const void* x, int64_t rows, int channels, const float* mean,
                                     const float* invstd, const void* gamma, const void* beta, int param_dtype,
                                     int relu, const void* residual, void* y, void* stream) {
  OCNN_REQUIRE(ocnn_batch_norm_supported(dtype, rows, channels), "batch_norm_apply: shape not supported");
  OCNN_REQUIRE_PTRS("batch_norm_apply", x, mean, invstd, y);
  return bn_apply(dtype, x, rows, channels, mean, invstd, gamma, beta, param_dtype, relu, residual, y, nullptr, nullptr, 0,
                  0.f, nullptr, (hipStream_t)stream);
}

extern "C" int64_t ocnnx_batch_norm_mask_bytes(int dtype, int64_t rows, int channels) {
  if (!ocnn_batch_norm_supported(dtype, rows, channels) || bn_slabs_take(dtype, rows, channels, false) ||
      bn_slabs_take(dtype, rows, channels, true))
    return 0;
  return rows * (channels / bn_vec(dtype));
}

// Training: statistics of the batch (with the running ones moved) and the normalise pass behind them.
extern "C" int ocnnx_batch_norm_training(int dtype, const void* x, int64_t rows, int channels, float eps, float* mean,
                                         float* var, float* invstd, void* running_mean, void* running_var,
                                         int running_dtype, float factor, int64_t* batches_tracked, const void* gamma,
                                         const void* beta, int param_dtype, int relu, const void* residual, void* y,
                                         void* mask, void* workspace, int64_t workspace_bytes, void* stream) {
  OCNN_REQUIRE(ocnn_batch_norm_supported(dtype, rows, channels), "batch_norm_training: shape not supported");
  OCNN_REQUIRE_PTRS("batch_norm_training", x, mean, var, invstd, y, workspace);
  OCNN_REQUIRE(workspace_bytes >= ocnn_batch_norm_workspace_bytes(channels), "batch_norm_training: workspace too small");
  // (in place: not as two launches, of which the second reads row 0, the sums' origin, in every workgroup beside the one that writes it)
  if (!bn_slabs_take(dtype, rows, channels, false) || (y == x && rows > kBnSmallRows)) {
    const int status = ocnn_batch_norm_stats(dtype, x, rows, channels, eps, mean, var, invstd, running_mean, running_var,
                                             running_dtype, factor, batches_tracked, workspace, workspace_bytes, stream);
    if (status != OCNN_OK) return status;
    return bn_apply(dtype, x, rows, channels, mean, invstd, gamma, beta, param_dtype, relu, residual, y, nullptr, nullptr,
                    0, 0.f, (uint8_t*)mask, (hipStream_t)stream);
  }
  OCNN_REQUIRE(!mask, "batch_norm_training: no mask of so few rows");
  const BnStats keep{eps, mean, var, invstd, running_mean, running_var, running_dtype, factor, (long long*)batches_tracked};
  const BnSlabs s = bn_slabs(dtype, rows, channels, kBnUnrollForward);
  double* partial = s.split ? (double*)workspace : nullptr;
  OCNN_DISPATCH_DTYPE(dtype, {
    constexpr int VEC = 16 / sizeof(T);
    auto launch = [&](auto kernel, int parts, int per) {
      hipLaunchKernelGGL(kernel, dim3(s.slabs, parts), dim3(kBnSlabThreads), 0, (hipStream_t)stream, (const T*)x, (int)rows, channels,
                         per, partial, s.ranges, keep, gamma, beta, param_dtype, relu, (const T*)residual, (T*)y);
    };
    if (s.split) launch(s.lanes == 8 ? bn_slab_kernel<T, VEC, 8, true> : bn_slab_kernel<T, VEC, 4, true>, s.ranges, s.sums_per);
    launch(s.lanes == 8 ? bn_slab_kernel<T, VEC, 8, false> : bn_slab_kernel<T, VEC, 4, false>, s.parts, s.per);
  });
  return check_launch("batch_norm_training");
}

extern "C" int ocnnx_batch_norm_running(int dtype, const void* x, int64_t rows, int channels, const void* running_mean,
                                        const void* running_var, int running_dtype, float eps, const void* gamma,
                                        const void* beta, int param_dtype, int relu, const void* residual, void* y,
                                        void* stream) {
  OCNN_REQUIRE(ocnn_batch_norm_supported(dtype, rows, channels), "batch_norm_running: shape not supported");
  OCNN_REQUIRE_PTRS("batch_norm_running", x, running_mean, running_var, y);
  return bn_apply(dtype, x, rows, channels, nullptr, nullptr, gamma, beta, param_dtype, relu, residual, y, running_mean,
                  running_var, running_dtype, eps, nullptr, (hipStream_t)stream);
}

extern "C" int ocnn_batch_norm_backward(int dtype, const void* x, const void* dy, int64_t rows, int channels,
                                        const float* mean, const float* invstd, const void* gamma,
                                        const void* beta, int param_dtype, int relu, int training,
                                        const void* y, void* dx, void* d_residual, float* dgamma, float* dbeta,
                                        void* grad_gamma, void* grad_beta, void* workspace,
                                        int64_t workspace_bytes, void* stream) {
  return ocnnx_batch_norm_backward(dtype, x, dy, rows, channels, mean, invstd, gamma, beta, param_dtype, relu, training, y,
                                   nullptr, dx, d_residual, dgamma, dbeta, grad_gamma, grad_beta, workspace, workspace_bytes,
                                   stream);
}

extern "C" int ocnnx_batch_norm_backward(int dtype, const void* x, const void* dy, int64_t rows, int channels,
                                         const float* mean, const float* invstd, const void* gamma, const void* beta,
                                         int param_dtype, int relu, int training, const void* y, const void* mask, void* dx,
                                         void* d_residual, float* dgamma, float* dbeta, void* grad_gamma, void* grad_beta,
                                         void* workspace, int64_t workspace_bytes, void* stream) {
  OCNN_REQUIRE(!d_residual || dx, "batch_norm_backward: d_residual needs dx");
  OCNN_REQUIRE(ocnn_batch_norm_supported(dtype, rows, channels), "batch_norm_backward: shape not supported");
  OCNN_REQUIRE_PTRS("batch_norm_backward", x, dy, mean, invstd, dgamma, dbeta, workspace);
  OCNN_REQUIRE(workspace_bytes >= ocnn_batch_norm_workspace_bytes(channels),
               "batch_norm_backward: workspace too small");
  hipStream_t st = (hipStream_t)stream;
  if (dx && !mask && bn_slabs_take(dtype, rows, channels, true)) {
    const BnSlabs s = bn_slabs(dtype, rows, channels, kBnUnrollBackward);
    double* partial = s.split ? (double*)workspace : nullptr;
    OCNN_DISPATCH_DTYPE(dtype, {
      constexpr int VEC = 16 / sizeof(T);
      auto launch = [&](auto kernel, int parts, int per) {
        hipLaunchKernelGGL(kernel, dim3(s.slabs, parts), dim3(kBnSlabThreads), 0, st, (const T*)x, (const T*)dy, (int)rows, channels,
                           per, partial, s.ranges, mean, invstd, gamma, beta, param_dtype, relu, training, (const T*)y, dbeta,
                           dgamma, grad_gamma, grad_beta, (T*)d_residual, (T*)dx);
      };
      if (s.split) launch(s.lanes == 8 ? bn_bwd_slab_kernel<T, VEC, 8, true> : bn_bwd_slab_kernel<T, VEC, 4, true>, s.ranges, s.sums_per);
      launch(s.lanes == 8 ? bn_bwd_slab_kernel<T, VEC, 8, false> : bn_bwd_slab_kernel<T, VEC, 4, false>, s.parts, s.per);
    });
    return check_launch("batch_norm_backward");
  }
  const int nblk = bn_blocks(dtype, rows, channels, kBnMaxBlocks);
  float* partial = (float*)workspace;
  OCNN_DISPATCH_DTYPE(dtype, {
    constexpr int VEC = 16 / sizeof(T);
    const auto launch = [&](auto sums, auto apply, const void* passed) {
      const int nblk_a = bn_blocks(dtype, rows, channels, bn_resident_blocks((const void*)apply, kBnBackwardPerCu));
      hipLaunchKernelGGL(sums, dim3(nblk), dim3(256), 0, st, (const T*)x, (const T*)dy, rows, channels, mean, invstd, gamma, beta,
                         param_dtype, relu, passed, partial);
      hipLaunchKernelGGL(bn_bwd_finish_kernel, dim3((unsigned)cdiv(channels, 4)), dim3(kBnFinishThreads), 0, st, partial, nblk,
                         channels, dbeta, dgamma, grad_gamma, grad_beta, param_dtype);
      if (dx)
        hipLaunchKernelGGL(apply, dim3(nblk_a), dim3(256), 0, st, (const T*)x, (const T*)dy, rows, channels, mean, invstd, gamma,
                           beta, param_dtype, relu, dbeta, dgamma, training, passed, (T*)d_residual, (T*)dx);
    };
    if (mask) launch(bn_bwd_stats_kernel<T, VEC, kBnBits>, bn_bwd_apply_kernel<T, VEC, kBnBits>, mask);
    else if (y) launch(bn_bwd_stats_kernel<T, VEC, kBnOfY>, bn_bwd_apply_kernel<T, VEC, kBnOfY>, y);
    else launch(bn_bwd_stats_kernel<T, VEC, kBnOfX>, bn_bwd_apply_kernel<T, VEC, kBnOfX>, nullptr);
  });
  return check_launch("batch_norm_backward");
}

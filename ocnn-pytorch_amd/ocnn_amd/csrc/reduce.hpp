// Second pass of every two-pass reduction in the library.
#pragma once
#include "common.hpp"

namespace ocnn {

// fixed-order reduction over the splits; writes (K, ca, cb) or (K, cb, ca)
template <typename T>
__global__ void wgrad_reduce_kernel(const float* __restrict__ partial, int splits, int K, int ca,
                                    int cb, int out_transposed, T* __restrict__ out) {
  int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t per = (int64_t)K * ca * cb;
  if (e >= per) return;
  float acc = 0.f;
  for (int s = 0; s < splits; ++s) acc += partial[(int64_t)s * per + e];
  int64_t o = e;
  if (out_transposed) {
    int b = (int)(e % cb);
    int a = (int)((e / cb) % ca);
    int64_t k = e / ((int64_t)ca * cb);
    o = (k * cb + b) * ca + a;
  }
  out[o] = from_f32<T>(acc);
}

// The same for cb % 4 == 0: 16 bytes per thread, LANES lanes of a workgroup share a column: lane i
// adds the splits i, i + LANES, .. (eight loads in flight), the lanes' sums are added in lane order: a
// fixed order again.  A 32 x 32 layer is 6912 such columns of 256 - 384 splits: with one thread a column
// the launch was 108 waves in a chain of dependent loads (36 us for 42 MB), with 8 lanes it is bound by the bytes.
// With ca > 0 the output is (K, cb, ca): the four sums of a thread (consecutive b) go to
// four rows of the transposed block.
template <typename T, int LANES>
__device__ __forceinline__ void wgrad_reduce4(const float* __restrict__ partial, int splits, int64_t per,
                                              T* __restrict__ out, int ca, int cb, uint32_t block, float* s_sums) {
  typedef __attribute__((ext_vector_type(4))) float v4;
  constexpr int COLS = 256 / LANES;
  v4* s_sum = (v4*)s_sums;                                   // 256 of them (LANES > 1)
  const int col = threadIdx.x % COLS, l = threadIdx.x / COLS;
  const int64_t e = ((int64_t)block * COLS + col) * 4;
  v4 acc = v4{0.f, 0.f, 0.f, 0.f};
  if (e < per) {
    int s = l;
    for (; s + 7 * LANES < splits; s += 8 * LANES) {
      v4 v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = *(const v4*)(partial + (int64_t)(s + i * LANES) * per + e);
#pragma unroll
      for (int i = 0; i < 8; ++i) acc += v[i];
    }
    for (; s < splits; s += LANES) acc += *(const v4*)(partial + (int64_t)s * per + e);
  }
  if constexpr (LANES > 1) {
    s_sum[threadIdx.x] = acc;
    __syncthreads();
    if (l > 0) return;
#pragma unroll
    for (int i = 1; i < LANES; ++i) acc += s_sum[i * COLS + col];
  }
  if (e >= per) return;
  if (ca > 0) {
    const int b = (int)(e % cb);
    const int a = (int)((e / cb) % ca);
    const int64_t k = e / ((int64_t)ca * cb);
#pragma unroll
    for (int i = 0; i < 4; ++i) out[(k * cb + b + i) * ca + a] = from_f32<T>(acc[i]);
  } else {
    typedef __attribute__((ext_vector_type(4))) T t4;
    t4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = from_f32<T>(acc[i]);
    *(t4*)(out + e) = o;
  }
}

template <typename T, int LANES>
__global__ __launch_bounds__(256) void wgrad_reduce4_kernel(const float* __restrict__ partial, int splits, int64_t per,
                                                            T* __restrict__ out, int ca, int cb) {
  __shared__ __attribute__((aligned(16))) float s_sums[LANES > 1 ? 1024 : 4];
  wgrad_reduce4<T, LANES>(partial, splits, per, out, ca, cb, blockIdx.x, s_sums);
}

// lanes a column: as many as leave the launch a few waves a SIMD
inline int wgrad_reduce_lanes(int splits, int64_t per) { return splits >= 16 && per / 4 < 65536 ? 8 : 1; }

// fp32 values as two bf16 pieces: x = hi + lo (+ 2^-17 |x|); a product of two such values is
// hi_a hi_b + hi_a lo_b + lo_a hi_b to about 1e-5 relative.  Two tensors (x, then g) in one launch,
// eight values a thread (counts are multiples of 8).
static __device__ __forceinline__ void split2(const float* __restrict__ x, int64_t nx, bf16* __restrict__ xh,
                                              bf16* __restrict__ xl, const float* __restrict__ g, int64_t ng,
                                              bf16* __restrict__ gh, bf16* __restrict__ gl, uint32_t block) {
  typedef __attribute__((ext_vector_type(4))) float v4;
  typedef __attribute__((ext_vector_type(8))) bf16 b8;
  int64_t e = ((int64_t)block * 256 + threadIdx.x) * 8;
  const float* src = x;
  bf16 *hi = xh, *lo = xl;
  if (e >= nx) {
    e -= nx;
    if (e >= ng) return;
    src = g, hi = gh, lo = gl;
  }
  const v4 a = *(const v4*)(src + e), b = *(const v4*)(src + e + 4);
  b8 h, l;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float v = i < 4 ? a[i] : b[i - 4];
    h[i] = (bf16)v;
    l[i] = (bf16)(v - (float)h[i]);
  }
  *(b8*)(hi + e) = h;
  *(b8*)(lo + e) = l;
}

static __global__ __launch_bounds__(256) void split2_kernel(const float* __restrict__ x, int64_t nx, bf16* __restrict__ xh,
                                                            bf16* __restrict__ xl, const float* __restrict__ g, int64_t ng,
                                                            bf16* __restrict__ gh, bf16* __restrict__ gl) {
  split2(x, nx, xh, xl, g, ng, gh, gl, blockIdx.x);
}

inline void launch_split2(const void* x, int64_t nx, bf16* xh, bf16* xl, const void* g, int64_t ng, bf16* gh, bf16* gl,
                          hipStream_t st) {
  if (nx + ng > 0)
    hipLaunchKernelGGL(split2_kernel, dim3((unsigned)cdiv((nx + ng) / 8, 256)), dim3(256), 0, st, (const float*)x, nx, xh,
                       xl, (const float*)g, ng, gh, gl);
}

// launches the reduction that fits
template <typename T>
inline void launch_wgrad_reduce(const float* partial, int splits, int K, int ca, int cb,
                                int out_transposed, T* out, hipStream_t st) {
  const int64_t per = (int64_t)K * ca * cb;
  if (cb % 4 == 0 && ((uintptr_t)partial % 16) == 0) {
    const int64_t cols = per / 4;
    const int ot = out_transposed ? ca : 0;
    if (wgrad_reduce_lanes(splits, per) == 8)
      hipLaunchKernelGGL((wgrad_reduce4_kernel<T, 8>), dim3((unsigned)cdiv(cols, 32)), dim3(256), 0, st, partial, splits,
                         per, out, ot, cb);
    else
      hipLaunchKernelGGL((wgrad_reduce4_kernel<T, 1>), dim3((unsigned)cdiv(cols, 256)), dim3(256), 0, st, partial, splits,
                         per, out, ot, cb);
  } else {
    hipLaunchKernelGGL(wgrad_reduce_kernel<T>, dim3((unsigned)cdiv(per, 256)), dim3(256), 0, st, partial,
                       splits, K, ca, cb, out_transposed, out);
  }
}

}  // namespace ocnn

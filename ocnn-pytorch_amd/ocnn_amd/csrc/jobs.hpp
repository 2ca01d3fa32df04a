// The small launches around the layers' kernels - weights packed into operand order, fp32 operands split into
// bf16 pieces, column sums, sums of parts and of ranges - as jobs that share a launch.
//
// Each of them is 3 - 8 us of latency on a handful of workgroups, and in a chain they add up: the backward
// pass of a layer had up to seven of them around its two large kernels.  Those that do not depend on each other
// run side by side: jobs_kernel deals its workgroups to up to four jobs.  256 -> 256 bf16 on 4 k rows with bias,
// forward + backward: 104 us as ten launches, 91 as seven.
#pragma once
#include <type_traits>

#include "common.hpp"
#include "host_api.hpp"
#include "mma.hpp"
#include "reduce.hpp"

namespace ocnn {

struct PackTileJob {          // conv_tile.hip: weights in the order of its A operand
  const void* w;
  void* out;
  int K, cin, cout, transposed, reverse, aligned;
};
struct SplitJob {             // reduce.hpp: two fp32 tensors into bf16 pieces
  const float *x, *g;
  bf16 *xh, *xl, *gh, *gl;
  int64_t nx, ng;
};
struct ColsumJob {            // column sums of ranges of rows
  const void* g;
  float* partial;
  int64_t rows, rows_per_split;
  int channels;
};
struct ColsumFinishJob {
  const float* partial;
  void* out;
  int splits, channels;
};
struct TilePartsJob {         // conv_tile.hip: sums of the parts of a split launch and what follows the layer
  const float* partial;
  const void* bias;
  void* out;
  ocnnx_bn bn;
  int64_t rows;
  int parts, cout;
};
struct ReduceJob {            // reduce.hpp: sums of the ranges of a weight gradient
  const float* partial;
  void* out;
  int64_t per;
  int splits, ca, cb, lanes;
};

struct Job {
  enum Kind { kPackTile, kSplit, kColsum, kColsumFinish, kTileParts, kReduce } kind;
  unsigned blocks;            // of 256 threads
  union {
    PackTileJob pack;
    SplitJob split;
    ColsumJob colsum;
    ColsumFinishJob colsum_finish;
    TilePartsJob parts;
    ReduceJob reduce;
  };
};

struct Jobs {
  static constexpr int kMost = 4;
  int n = 0;
  Job job[kMost];
  void add(const Job& j) {
    if (j.blocks > 0) job[n++] = j;
  }
};

// T: the layer's type; its jobs in one launch
template <typename T> void launch_jobs(const Jobs& jobs, hipStream_t st);

inline void launch_jobs(int dtype, const Jobs& jobs, hipStream_t st) {
  if (dtype == OCNN_F32) launch_jobs<float>(jobs, st);
  else if (dtype == OCNN_F16) launch_jobs<f16>(jobs, st);
  else launch_jobs<bf16>(jobs, st);
}

Job pack_tile_job(int dtype, const void* w, void* out, int K, int cin, int cout, int transposed, int reverse);
Job tile_parts_job(const float* partial, int parts, int64_t rows, int cout, const void* bias, const ocnnx_bn& bn, void* out);

// A pass between its jobs: those in front of its kernel, those behind it.
struct Pass {
  Jobs before, after;
  virtual int main() = 0;     // launches the kernel itself
  virtual ~Pass() {}
};

int tile_pass(int dtype, const ocnnx_gather_args& args, hipStream_t st, Pass** pass);
int wgrad_planned_pass(int dtype, const ocnnx_wgrad_args& args, hipStream_t st, Pass** pass);
// column sums as jobs; false (and none added) for channels in odd pieces, which ocnn_colsum takes
bool colsum_jobs(int dtype, const void* g, int64_t rows, int channels, void* out, void* ws, int64_t ws_bytes, Jobs& before,
                 Jobs& after);

// N consecutive values of a per-channel array (f32 / f16 / bf16; null: dflt), N a multiple of 4
template <int N>
__device__ __forceinline__ void load_channels(const void* p, int dtype, int c0, float dflt, float (&v)[N]) {
  if (!p) {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = dflt;
  } else if (dtype == OCNN_F32) {
#pragma unroll
    for (int i = 0; i < N; i += 4) {
      const f32x4 q = *(const f32x4*)((const float*)p + c0 + i);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[i + j] = q[j];
    }
  } else {
    unsigned short r[N];
#pragma unroll
    for (int i = 0; i < N; i += 4) {
      const u32x2 q = *(const u32x2*)((const unsigned short*)p + c0 + i);
      r[i] = (unsigned short)q[0], r[i + 1] = (unsigned short)(q[0] >> 16);
      r[i + 2] = (unsigned short)q[1], r[i + 3] = (unsigned short)(q[1] >> 16);
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
      v[i] = dtype == OCNN_F16 ? to_f32(__builtin_bit_cast(f16, r[i])) : __uint_as_float((uint32_t)r[i] << 16);
  }
}

// What is added to N channels of a row's sums and what they are multiplied with: bias alone, or the batch
// norm behind the layer with its running statistics, ((sum + bias) - mean) * sc + beta = sum * sc + sh.
template <typename O, int N>
__device__ __forceinline__ void layer_tail(const O* bias, const ocnnx_bn& bn, int c0, float (&sc)[N], float (&sh)[N]) {
  load_channels<N>(bias, std::is_same<O, float>::value ? OCNN_F32 : (std::is_same<O, f16>::value ? OCNN_F16 : OCNN_BF16), c0,
                   0.f, sh);
#pragma unroll
  for (int i = 0; i < N; ++i) sc[i] = 1.f;
  if (bn.mean) {
    float m[N], be[N], ga[N];
    load_channels<N>(bn.var, bn.stat_dtype, c0, 1.f, sc);
    load_channels<N>(bn.mean, bn.stat_dtype, c0, 0.f, m);
    load_channels<N>(bn.gamma, bn.param_dtype, c0, 1.f, ga);
    load_channels<N>(bn.beta, bn.param_dtype, c0, 0.f, be);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      sc[i] = ga[i] / sqrtf(sc[i] + bn.eps);
      sh[i] = (sh[i] - m[i]) * sc[i] + be[i];
    }
  }
}

}  // namespace ocnn

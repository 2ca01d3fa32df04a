// Jobs that share a launch (jobs.hpp), and the backward pass of a layer with its small launches merged.
#include <algorithm>
#include <type_traits>

#include "jobs.hpp"

namespace ocnn {

// Packed weights: [input-channel chunk cc][slot k][32 output channels cg][step s][lane][8].
// v_mfma_f32_32x32x16 A operand: lane l holds A[l % 32][8 * (l / 32) + j];
// D: lane l, register r holds D[8 * (r / 4) + 4 * (l / 32) + r % 4][l % 32].
//   output channel = 32 cg + perm(lane % 32), perm(8a + 4q + b) = 16 q + 4 a + b,
// so that a lane ends with 16 consecutive output channels per M tile.
//   16-bit: input channel = 64 cc + 16 s + 8 (lane / 32) + j
//   fp32:   input channel = 32 cc + 16 (s / 2) + 8 (lane / 32) + j, s % 2 = 0: high piece, 1: low
// Input channels are padded to whole chunks with zero weights.
//
// Bound by latency (a layer's weights are 0.1 - 7 MB): few, wide loads a thread, all in flight together.
// transposed: a thread packs a lane's eight values, consecutive in memory.  Otherwise they are rows of
// cout values apart and a thread packs four lanes of consecutive output channels: eight loads of four
// values, 64 consecutive bytes written.  AL: the weights are 16-byte aligned (a module's are; a view
// into something else may not be, and is read value by value).  fp32 256 -> 256, 27 slots: 8.9 -> 6 us (eight
// 4-byte loads a thread before); the 103 launches of an fp32 U-Net step 0.68 -> 0.52 ms.
template <int N, bool AL, typename I>
__device__ __forceinline__ void load_run(const I* __restrict__ p, I (&v)[N]) {
  if constexpr (AL) {
    constexpr int W = N * sizeof(I) < 16 ? N : 16 / sizeof(I);
    typedef __attribute__((ext_vector_type(W))) I vec;
#pragma unroll
    for (int i = 0; i < N; i += W) {
      const vec x = *(const vec*)(p + i);
#pragma unroll
      for (int j = 0; j < W; ++j) v[i + j] = x[j];
    }
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = p[i];
  }
}

template <typename I, typename T, bool AL>
static __device__ __forceinline__ void pack_tile(const I* __restrict__ w, T* __restrict__ out, int K, int cin, int cout,
                                                 int transposed, int reverse, uint32_t block) {
  constexpr bool F32 = std::is_same<I, float>::value;
  constexpr int CH = F32 ? 32 : 64, STEPS = F32 ? 2 : 4;
  typedef __attribute__((ext_vector_type(8))) T t8;
  const uint32_t e = block * 256 + threadIdx.x;
  const uint32_t t = transposed ? e & 63 : e & 15, step = transposed ? e >> 6 : e >> 4;
  const uint32_t ncc = (uint32_t)(cin + CH - 1) / CH, ncg = (uint32_t)cout >> 5;
  const uint32_t s = step % STEPS, base = step / STEPS;      // base = (cc K + k) ncg + cg
  if (base >= ncc * K * ncg) return;
  const uint32_t cg = base % ncg, k = base / ncg % K, cc = base / ncg / K;
  const uint32_t kk = reverse ? K - 1 - k : k;
  T* dst = out + (int64_t)base * 2048;
  // the eight values of a lane -> its place (both pieces of them)
  auto put = [&](const I (&v)[8], uint32_t lane) {
    t8 hi;
#pragma unroll
    for (int j = 0; j < 8; ++j) hi[j] = (T)v[j];
    if constexpr (F32) {
      t8 lo;
#pragma unroll
      for (int j = 0; j < 8; ++j) lo[j] = (T)(v[j] - (float)hi[j]);
      *(t8*)(dst + (2 * s) * 512 + lane * 8) = hi;
      *(t8*)(dst + (2 * s + 1) * 512 + lane * 8) = lo;
    } else {
      *(t8*)(dst + s * 512 + lane * 8) = hi;
    }
  };
  if (transposed) {
    const uint32_t m = t & 31, chan = CH * cc + 16 * s + 8 * (t >> 5);
    const uint32_t co = 32 * cg + 16 * ((m >> 2) & 1) + 4 * (m >> 3) + (m & 3);
    I v[8] = {};
    if (chan < (uint32_t)cin) load_run<8, AL>(w + ((int64_t)kk * cout + co) * cin + chan, v);
    put(v, t);
  } else {
    const uint32_t m4 = t & 7, chan = CH * cc + 16 * s + 8 * (t >> 3);
    const uint32_t co = 32 * cg + 16 * (m4 & 1) + 4 * (m4 >> 1);
    I v[8][4] = {};
    if (chan < (uint32_t)cin) {
#pragma unroll
      for (int j = 0; j < 8; ++j) load_run<4, AL>(w + ((int64_t)kk * cin + chan + j) * cout + co, v[j]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      I r[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) r[j] = v[j][i];
      put(r, 32 * (t >> 3) + 4 * m4 + i);
    }
  }
}

// out = sum of the parts, in their order, and what follows (layer_tail); four consecutive channels a thread, eight
// threads a row's 32 channels, so that a wave reads 128 bytes of consecutive rows at a time and writes 64 - 128.
template <typename O>
static __device__ __forceinline__ void tile_parts(const float* __restrict__ partial, int parts, int64_t rows, int cout,
                                                  const O* __restrict__ bias, const ocnnx_bn& bn, O* __restrict__ out,
                                                  uint32_t block) {
  const uint32_t groups = (uint32_t)cout >> 5;               // of 32 channels: a block has 32 rows of one
  const int64_t row = (int64_t)(block / groups) * 32 + (threadIdx.x >> 3);
  const int c4 = (int)(block % groups) * 8 + (int)(threadIdx.x & 7);   // four channels
  if (row >= rows) return;
  const int64_t n = rows * cout, e = row * cout + 4 * c4;
  const float* src = partial + ((int64_t)c4 * rows + row) * 4;
  f32x4 acc = *(const f32x4*)src;
  int s = 1;
  for (; s + 4 <= parts; s += 4) {                           // four loads in flight
    f32x4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = *(const f32x4*)(src + (s + u) * n);
#pragma unroll
    for (int u = 0; u < 4; ++u) acc += v[u];
  }
  for (; s < parts; ++s) acc += *(const f32x4*)(src + s * n);
  float mul[4], add[4];
  layer_tail<O, 4>(bias, bn, 4 * c4, mul, add);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    acc[i] = acc[i] * mul[i] + add[i];
    if (bn.residual) acc[i] += to_f32(((const O*)bn.residual)[e + i]);
    if (bn.relu) acc[i] = fmaxf(acc[i], 0.f);
  }
  typedef __attribute__((ext_vector_type(4))) O o4;
  o4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = from_f32<O>(acc[i]);
  *(o4*)(out + e) = o;
}

// Column sums of a range of rows in 16-byte pieces: a thread keeps one piece of the row (8 or 4 channels) and walks
// every (256 / pieces)-th row of the split, four loads in flight; the row lanes meet in LDS and
// are added in lane order.  C % (16 / sizeof(T)) == 0.
template <typename T>
static __device__ __forceinline__ void colsum_rows(const T* __restrict__ g, int64_t rows, int C, int64_t rows_per_split,
                                                   float* __restrict__ partial, uint32_t block, float* s_sums) {
  constexpr int VEC = 16 / sizeof(T);
  struct alignas(16) Piece { T v[VEC]; };
  float(*s_acc)[VEC + 1] = (float(*)[VEC + 1])s_sums;
  const int cpr = C / VEC;
  const int lanes_c = cpr < 256 ? cpr : 256, rpi = 256 / lanes_c;
  const int pc = threadIdx.x % lanes_c, rl = threadIdx.x / lanes_c;
  const int64_t r_begin = (int64_t)block * rows_per_split;
  const int64_t r_end = min(rows, r_begin + rows_per_split);
  for (int p0 = 0; p0 < cpr; p0 += lanes_c) {
    const int piece = p0 + pc;
    float acc[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) acc[v] = 0.f;
    if (rl < rpi && piece < cpr) {
      const Piece* src = reinterpret_cast<const Piece*>(g) + piece;
      int64_t i = r_begin + rl;
      for (; i + 3 * rpi < r_end; i += 4 * rpi) {
        Piece q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = src[(i + u * rpi) * cpr];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int v = 0; v < VEC; ++v) acc[v] += to_f32(q[u].v[v]);
      }
      for (; i < r_end; i += rpi) {
        const Piece q = src[i * cpr];
#pragma unroll
        for (int v = 0; v < VEC; ++v) acc[v] += to_f32(q.v[v]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < VEC; ++v) s_acc[threadIdx.x][v] = acc[v];
    __syncthreads();
    if (rl == 0 && piece < cpr) {
#pragma unroll
      for (int v = 0; v < VEC; ++v) {
        float sum = 0.f;
        for (int r = 0; r < rpi; ++r) sum += s_acc[r * lanes_c + pc][v];
        partial[(int64_t)block * C + piece * VEC + v] = sum;
      }
    }
  }
}

// out[c] = sum over the splits, 16 split lanes a channel, each adding every 16th split in order,
// the lanes then in lane order
template <typename T>
static __device__ __forceinline__ void colsum_finish(const float* __restrict__ partial, int splits, int C,
                                                     T* __restrict__ out, uint32_t block, float* s_sums) {
  float(*s_acc)[16] = (float(*)[16])s_sums;
  const int cl = threadIdx.x & 15, sl = threadIdx.x >> 4;
  const int c = (int)block * 16 + cl;
  float acc = 0.f;
  if (c < C) {
#pragma unroll 8
    for (int s = sl; s < splits; s += 16) acc += partial[(int64_t)s * C + c];
  }
  s_acc[sl][cl] = acc;
  __syncthreads();
  if (sl == 0 && c < C) {
    float sum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) sum += s_acc[r][cl];
    out[c] = from_f32<T>(sum);
  }
}

template <typename T, int KIND>
static __device__ __forceinline__ void run_job(const Job& job, uint32_t block, float* s_sums) {
  typedef typename std::conditional<std::is_same<T, float>::value, bf16, T>::type P;   // type of packed weights
  if constexpr (KIND == Job::kPackTile) {
    const PackTileJob& a = job.pack;
    if (a.aligned) pack_tile<T, P, true>((const T*)a.w, (P*)a.out, a.K, a.cin, a.cout, a.transposed, a.reverse, block);
    else pack_tile<T, P, false>((const T*)a.w, (P*)a.out, a.K, a.cin, a.cout, a.transposed, a.reverse, block);
  } else if constexpr (KIND == Job::kSplit) {
    const SplitJob& a = job.split;
    split2(a.x, a.nx, a.xh, a.xl, a.g, a.ng, a.gh, a.gl, block);
  } else if constexpr (KIND == Job::kColsum) {
    const ColsumJob& a = job.colsum;
    colsum_rows<T>((const T*)a.g, a.rows, a.channels, a.rows_per_split, a.partial, block, s_sums);
  } else if constexpr (KIND == Job::kColsumFinish) {
    const ColsumFinishJob& a = job.colsum_finish;
    colsum_finish<T>(a.partial, a.splits, a.channels, (T*)a.out, block, s_sums);
  } else if constexpr (KIND == Job::kTileParts) {
    const TilePartsJob& a = job.parts;
    tile_parts<T>(a.partial, a.parts, a.rows, a.cout, (const T*)a.bias, a.bn, (T*)a.out, block);
  } else {
    const ReduceJob& a = job.reduce;
    if (a.lanes == 8) wgrad_reduce4<T, 8>(a.partial, a.splits, a.per, (T*)a.out, a.ca, a.cb, block, s_sums);
    else wgrad_reduce4<T, 1>(a.partial, a.splits, a.per, (T*)a.out, a.ca, a.cb, block, s_sums);
  }
}

#define OCNN_JOB_KINDS(DO) \
  DO(Job::kPackTile) DO(Job::kSplit) DO(Job::kColsum) DO(Job::kColsumFinish) DO(Job::kTileParts) DO(Job::kReduce)

template <typename T> constexpr int kJobSums = 256 * (16 / sizeof(T) + 1);   // floats of LDS that a job may use

// Workgroup b: the job whose workgroups b falls among.
template <typename T>
__global__ __launch_bounds__(256) void jobs_kernel(Jobs jobs) {
  __shared__ __attribute__((aligned(16))) float s_sums[kJobSums<T>];
  uint32_t block = blockIdx.x;
  int i = 0;
  while (i + 1 < jobs.n && block >= jobs.job[i].blocks) block -= jobs.job[i++].blocks;
  switch (jobs.job[i].kind) {
#define OCNN_CASE(KIND_) case KIND_: run_job<T, KIND_>(jobs.job[i], block, s_sums); break;
    OCNN_JOB_KINDS(OCNN_CASE)
#undef OCNN_CASE
  }
}

// One job by itself: without the other kinds' code around it the launch is 0.6 us shorter.
template <typename T, int KIND>
__global__ __launch_bounds__(256) void job_kernel(Job job) {
  __shared__ __attribute__((aligned(16))) float s_sums[kJobSums<T>];
  run_job<T, KIND>(job, blockIdx.x, s_sums);
}

// The weights of several layers.  A launch for one layer is bound by its own start (4.2 us; 40 in a network of 32 - 256
// channels in 16 bit: 169 us); up to 12 layers fit the arguments: 6 launches of 9.0 us in the same network.
struct PackJobs {
  int n;
  unsigned blocks[OCNNX_PACK_MOST];
  PackTileJob job[OCNNX_PACK_MOST];
};
template <typename T>
__global__ __launch_bounds__(256) void pack_jobs_kernel(PackJobs jobs) {
  typedef typename std::conditional<std::is_same<T, float>::value, bf16, T>::type P;
  uint32_t block = blockIdx.x;
  int i = 0;
  while (i + 1 < jobs.n && block >= jobs.blocks[i]) block -= jobs.blocks[i++];
  const PackTileJob& a = jobs.job[i];
  if (a.aligned) pack_tile<T, P, true>((const T*)a.w, (P*)a.out, a.K, a.cin, a.cout, a.transposed, a.reverse, block);
  else pack_tile<T, P, false>((const T*)a.w, (P*)a.out, a.K, a.cin, a.cout, a.transposed, a.reverse, block);
}

template <typename T> void launch_jobs(const Jobs& jobs, hipStream_t st) {
  unsigned blocks = 0;
  for (int i = 0; i < jobs.n; ++i) blocks += jobs.job[i].blocks;
  if (jobs.n > 1) hipLaunchKernelGGL(jobs_kernel<T>, dim3(blocks), dim3(256), 0, st, jobs);
  if (jobs.n == 1) switch (jobs.job[0].kind) {
#define OCNN_CASE(KIND_) \
    case KIND_: hipLaunchKernelGGL((job_kernel<T, KIND_>), dim3(blocks), dim3(256), 0, st, jobs.job[0]); break;
    OCNN_JOB_KINDS(OCNN_CASE)
#undef OCNN_CASE
  }
}
template void launch_jobs<float>(const Jobs&, hipStream_t);
template void launch_jobs<f16>(const Jobs&, hipStream_t);
template void launch_jobs<bf16>(const Jobs&, hipStream_t);

Job pack_tile_job(int dtype, const void* w, void* out, int K, int cin, int cout, int transposed, int reverse) {
  const int64_t steps = cdiv(cin, dtype == OCNN_F32 ? 32 : 64) * (int64_t)K * (cout / 32) * (dtype == OCNN_F32 ? 2 : 4);
  Job j{Job::kPackTile, (unsigned)cdiv(steps * (transposed ? 64 : 16), 256), {}};
  j.pack = PackTileJob{w, out, K, cin, cout, transposed, reverse, (uintptr_t)w % 16 == 0};
  return j;
}

Job tile_parts_job(const float* partial, int parts, int64_t rows, int cout, const void* bias, const ocnnx_bn& bn, void* out) {
  Job j{Job::kTileParts, (unsigned)(cdiv(rows, 32) * (cout / 32)), {}};
  j.parts = TilePartsJob{partial, bias, out, bn, rows, parts, cout};
  return j;
}

}  // namespace ocnn

using namespace ocnn;

extern "C" int ocnnx_pack_tiles(int dtype, const ocnnx_pack_item* items, int n, void* stream) {
  OCNN_REQUIRE(dtype >= 0 && dtype <= 2 && n >= 1 && n <= OCNNX_PACK_MOST, "pack_tiles: dtype=%d n=%d", dtype, n);
  OCNN_REQUIRE_PTRS("pack_tiles", items);
  PackJobs jobs;
  jobs.n = n;
  unsigned blocks = 0;
  for (int i = 0; i < n; ++i) {
    const ocnnx_pack_item& it = items[i];
    OCNN_REQUIRE(it.w && it.out, "pack_tiles: a required pointer is NULL");
    OCNN_REQUIRE(ocnnx_gather_tile_supported(dtype, 0, it.K, it.cin, it.cout, 0), "pack_tiles: shape not supported");
    const Job j = pack_tile_job(dtype, it.w, it.out, it.K, it.cin, it.cout, it.transposed, it.reverse_slots);
    jobs.blocks[i] = j.blocks;
    jobs.job[i] = j.pack;
    blocks += j.blocks;
  }
  hipStream_t st = (hipStream_t)stream;
  if (dtype == OCNN_F32) hipLaunchKernelGGL(pack_jobs_kernel<float>, dim3(blocks), dim3(256), 0, st, jobs);
  else if (dtype == OCNN_F16) hipLaunchKernelGGL(pack_jobs_kernel<f16>, dim3(blocks), dim3(256), 0, st, jobs);
  else hipLaunchKernelGGL(pack_jobs_kernel<bf16>, dim3(blocks), dim3(256), 0, st, jobs);
  return check_launch("pack_tiles");
}

// Both passes and the bias gradient: what comes before the kernels in one launch, what comes after them in another.
extern "C" int ocnnx_conv_backward(int dtype, const ocnnx_gather_args* dgrad, const ocnnx_wgrad_args* wgrad, const void* grad,
                                   int64_t grad_rows, int grad_channels, void* bias_grad, void* colsum_workspace,
                                   int64_t colsum_bytes, void* stream) {
  hipStream_t st = (hipStream_t)stream;
  OCNN_REQUIRE_PTRS("conv_backward", dgrad, wgrad);
  Pass *d = nullptr, *w = nullptr;
  int rc = tile_pass(dtype, *dgrad, st, &d);
  if (rc == OCNN_OK) rc = wgrad_planned_pass(dtype, *wgrad, st, &w);
  if (rc == OCNN_OK) {
    Jobs before, after;
    for (const Pass* p : {d, w})
      if (p) {
        for (int i = 0; i < p->before.n; ++i) before.add(p->before.job[i]);
        for (int i = 0; i < p->after.n; ++i) after.add(p->after.job[i]);
      }
    bool sums = bias_grad == nullptr;
    if (!sums) sums = colsum_jobs(dtype, grad, grad_rows, grad_channels, bias_grad, colsum_workspace, colsum_bytes, before, after);
    launch_jobs(dtype, before, st);
    // The data gradient last where that pays: what comes next reads it, and the memory-side cache still holds its end.  First where
    // the launch behind both finishes it from parts, in fp32, and where the gradient is so small that the second kernel finds
    // all of it in the L2s: the weight gradient gains more from that.  us a layer, forward + backward, first / last: 16 bit, 96 -> 96 on
    // 3 MB 77.2 / 78.5, 5 MB 82.1 / 82.7, 128 -> 128 on 6 MB 101.3 / 102.0, 192 -> 192 on 9 MB 200.0 / 199.5, 96 -> 96 on 70 MB 506 / 499, 120 MB
    // 621 / 611; fp32, 64 -> 64 85.7 / 87.1, 539 / 546, 2283 / 2294, 32 -> 32 772 / 780; in parts, 256 -> 256 on one cloud's depth 5 90.6 / 92.1.
    const bool last = d && d->after.n == 0 && dtype != OCNN_F32 && grad_rows * grad_channels >= (4ll << 20);
    Pass* order[2] = {last ? w : d, last ? d : w};
    for (Pass* p : order)
      if (rc == OCNN_OK && p) rc = p->main();
    if (rc == OCNN_OK) {
      launch_jobs(dtype, after, st);
      rc = check_launch("conv_backward");
    }
    if (rc == OCNN_OK && !sums)
      rc = ocnn_colsum(dtype, grad, grad_rows, grad_channels, bias_grad, colsum_workspace, colsum_bytes, stream);
  }
  delete d;
  delete w;
  return rc;
}

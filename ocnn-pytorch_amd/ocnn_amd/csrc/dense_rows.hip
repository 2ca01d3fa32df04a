// Dense rows of few channels (one slot, row i reads row i): a 1x1x1 convolution.
#include <algorithm>

#include "common.hpp"
#include "host_api.hpp"
#include "jobs.hpp"
#include "mma.hpp"
#include "reduce.hpp"

namespace ocnn {

// out = in W (+ bias, + what follows the layer) with all weights in the registers of every wave (cin x cout up to
// 16384: 128 registers a lane).  Bound by HBM: a wave walks 32-row blocks on its own, the next block's rows on
// their way while one is multiplied, straight from memory into the operand registers (a lane reads
// 16 bytes of its row a k step; the steps of a block share the lines in L1): no barrier, and no launch that
// packs weights - a workgroup brings them through LDS into its waves' order once.  Blocks are dealt
// round robin, so that the chip walks the rows front to back.
//
// D = W^T x in^T on 32 x 32 blocks: a lane ends with 16 channels of one row, 32 bytes of it next to those of one
// other lane.  Stored like that, results larger than the memory-side cache cost 0.13 - 0.2 us a MB more than in
// whole lines: the block goes through LDS first and leaves a KiB a store (64 -> 64 on 1.13 M rows
// 79 us before, 49 so; 32 -> 256 200 and 126).
//
// Measured (f16; this kernel / the plan-free one with its packing launch): 128 -> 96 on 1.13 M rows 100 / 251 us
// (4.9 TB/s), 96 -> 128 98 / 150, 64 -> 96 69 / 139, 96 -> 64 69 / 80; 300 k rows 26 / 45, 23 / 37, 17 / 30, 16 / 23; 4096 and
// 16 k rows of any width 5 - 7 / 8 - 9.  256 -> 64 gains nothing (142 / 141) and is left to it.
constexpr int kDrMaxWeights = 16384;

template <int KS, int MB> constexpr int kDrWaves = 4 * KS * MB + 8 * KS + 16 * MB + 40 <= 256 ? 2 : 1;   // a SIMD

template <typename T, int KS, int MB>
__global__ __launch_bounds__(256, (kDrWaves<KS, MB>)) void dense_rows_kernel(
    const T* __restrict__ in, uint32_t in_bytes, const T* __restrict__ w, int transposed, const T* __restrict__ bias,
    ocnnx_bn bn, T* __restrict__ out, uint32_t out_bytes, int64_t rows) {
  constexpr int CI = 16 * KS, CO = 32 * MB;
  typedef __attribute__((ext_vector_type(8))) T t8;
  constexpr int kPitch = CO + 8;                               // of a row in a wave's block on its way out
  __shared__ __attribute__((aligned(16))) T s_w[CI * CO > 128 * kPitch ? CI * CO : 128 * kPitch];
  __shared__ __attribute__((aligned(16))) float s_mul[CO], s_add[CO];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane >> 5, r32 = lane & 31;

  if (((uintptr_t)w & 15) == 0) {
    for (int e = tid * 8; e < CI * CO; e += 2048) *(u32x4*)(s_w + e) = *(const u32x4*)(w + e);
  } else {
    for (int e = tid; e < CI * CO; e += 256) s_w[e] = w[e];
  }
  for (int c = tid * 4; c < CO; c += 1024) {
    float mul[4], add[4];
    layer_tail<T, 4>(bias, bn, c, mul, add);
#pragma unroll
    for (int i = 0; i < 4; ++i) s_mul[c + i] = mul[i], s_add[c + i] = add[i];
  }
  __syncthreads();
  u32x4 wreg[MB][KS];
#pragma unroll
  for (int b = 0; b < MB; ++b)
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int co = 32 * b + 16 * (r32 >> 4) + 8 * ((r32 >> 2) & 1) + 4 * ((r32 >> 3) & 1) + (r32 & 3), chan = 16 * s + 8 * q;
      if (transposed) {
        wreg[b][s] = *(const u32x4*)(s_w + co * CI + chan);
      } else {
        t8 v;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = s_w[(chan + j) * CO + co];
        wreg[b][s] = __builtin_bit_cast(u32x4, v);
      }
    }

  __syncthreads();                                             // the weights' place is the results' from here on
  T* const s_out = s_w + wave * 32 * kPitch;
  const __amdgpu_buffer_rsrc_t rs_in = make_rsrc(in, in_bytes);
  const __amdgpu_buffer_rsrc_t rs_out = make_rsrc(out, out_bytes);
  const bool follows = bn.mean || bias;
  const int64_t blocks = (rows + 31) / 32, step = (int64_t)gridDim.x * 4;
  // (blocks past the end read out of range: zeros)
  auto fetch = [&](int64_t block, u32x4 (&x)[KS]) {
    const uint32_t off = block < blocks ? (uint32_t)(block * 32 + r32) * (CI * 2u) + 16u * q : 0xffffff00u - CI * 2u;
#pragma unroll
    for (int s = 0; s < KS; ++s) x[s] = __builtin_amdgcn_raw_buffer_load_b128(rs_in, off + 32 * s, 0, 0);
  };
  auto finish = [&](int64_t block, const u32x4 (&x)[KS]) {
    const int64_t row = block * 32 + r32;
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      f32x16 acc;
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
      for (int s = 0; s < KS; ++s) acc = Mma32<T>::run(wreg[b][s], x[s], acc);
      const int co = 32 * b + 8 * q;                         // channels co .. + 7 and co + 16 .. + 7
      if (follows) {
#pragma unroll
        for (int i = 0; i < 16; i += 4) {
          const f32x4 mul = *(const f32x4*)(s_mul + co + i + (i & 8)), add = *(const f32x4*)(s_add + co + i + (i & 8));
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[i + j] = acc[i + j] * mul[j] + add[j];
        }
      }
      if (bn.residual && row < rows) {
        const T* res = (const T*)bn.residual + row * CO + co;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] += to_f32(res[i + (i & 8)]);
      }
      if (bn.relu) {
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = fmaxf(acc[i], 0.f);
      }
      unsigned pk[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) pk[i] = pack2<T>(acc[2 * i], acc[2 * i + 1]);
      *(u32x4*)(s_out + r32 * kPitch + co) = u32x4{pk[0], pk[1], pk[2], pk[3]};
      *(u32x4*)(s_out + r32 * kPitch + co + 16) = u32x4{pk[4], pk[5], pk[6], pk[7]};
    }
    // the block leaves in the order of memory, a KiB a store (rows past the end are out of range)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int p = 0; p < 2 * MB; ++p) {
      const int e = (64 * p + lane) * 8, r = e / CO, c = e % CO;
      const u32x4 v = *(const u32x4*)(s_out + r * kPitch + c);
      const bool ok = block * 32 + r < rows;
      __builtin_amdgcn_raw_buffer_store_b128(v, rs_out, ok ? (uint32_t)(block * 32) * (CO * 2u) + 2u * e : 0xffffff00u, 0, 0);
    }
    __builtin_amdgcn_wave_barrier();
  };
  u32x4 xa[KS], xb[KS];
  int64_t block = (int64_t)blockIdx.x * 4 + wave;
  fetch(block, xa);
  for (; block < blocks; block += 2 * step) {
    fetch(block + step, xb);
    finish(block, xa);
    if (block + step >= blocks) break;
    fetch(block + 2 * step, xa);
    finish(block + step, xb);
  }
}

}  // namespace ocnn

using namespace ocnn;

static bool dr_channels(int c) { return c == 32 || c == 64 || c == 96 || c == 128 || c == 192; }

extern "C" int ocnnx_dense_rows_supported(int dtype, int64_t rows, int cin, int cout) {
  if (dtype != OCNN_F16 && dtype != OCNN_BF16) return 0;
  if (!dr_channels(cin) || !(dr_channels(cout) || cout == 256) || cin * cout > kDrMaxWeights) return 0;
  return rows >= 0 && (rows + 32) * std::max(cin, cout) * 2 <= 0xfff00000ll;
}

template <typename T, int KS, int MB>
static int launch_dense_rows(const void* in, int64_t rows, const void* w, int w_transposed, const void* bias,
                             const ocnnx_bn& bn, void* out, hipStream_t st) {
  static const int held = [] {
    int dev = 0, n = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, (const void*)dense_rows_kernel<T, KS, MB>, 256, 0) != hipSuccess) n = 1;
    return std::max(1, n) * prop.multiProcessorCount;
  }();
  OCNN_REQUIRE(held > 0, "dense_rows: cannot query the device");
  const unsigned wgs = (unsigned)std::min<int64_t>(held, cdiv(rows, 128));
  hipLaunchKernelGGL((dense_rows_kernel<T, KS, MB>), dim3(wgs), dim3(256), 0, st, (const T*)in, (uint32_t)(rows * KS * 32),
                     (const T*)w, w_transposed, (const T*)bias, bn, (T*)out, (uint32_t)(rows * MB * 64), rows);
  return check_launch("dense_rows");
}

template <typename T>
static int run_dense_rows(const void* in, int64_t rows, const void* w, int cin, int cout, int w_transposed,
                          const void* bias, const ocnnx_bn& bn, void* out, hipStream_t st) {
#define OCNN_DR(CI, CO) \
  if (cin == CI && cout == CO) return launch_dense_rows<T, CI / 16, CO / 32>(in, rows, w, w_transposed, bias, bn, out, st);
  OCNN_DR(32, 32) OCNN_DR(32, 64) OCNN_DR(32, 96) OCNN_DR(32, 128) OCNN_DR(32, 192) OCNN_DR(32, 256)
  OCNN_DR(64, 32) OCNN_DR(64, 64) OCNN_DR(64, 96) OCNN_DR(64, 128) OCNN_DR(64, 192) OCNN_DR(64, 256)
  OCNN_DR(96, 32) OCNN_DR(96, 64) OCNN_DR(96, 96) OCNN_DR(96, 128)
  OCNN_DR(128, 32) OCNN_DR(128, 64) OCNN_DR(128, 96) OCNN_DR(128, 128)
  OCNN_DR(192, 32) OCNN_DR(192, 64)
#undef OCNN_DR
  set_error("dense_rows: no kernel for %d -> %d channels", cin, cout);
  return OCNN_ERR_ARG;
}

extern "C" int ocnnx_dense_rows(int dtype, const void* in, int64_t rows, const void* w, int cin, int cout,
                                int w_transposed, const void* bias, const ocnnx_bn* bn, void* out, void* stream) {
  OCNN_REQUIRE(ocnnx_dense_rows_supported(dtype, rows, cin, cout), "dense_rows: shape not supported");
  if (rows == 0) return OCNN_OK;
  OCNN_REQUIRE_PTRS("dense_rows", in, w, out);
  const ocnnx_bn after = bn ? *bn : ocnnx_bn{};
  if (dtype == OCNN_F16)
    return run_dense_rows<f16>(in, rows, w, cin, cout, w_transposed, bias, after, out, (hipStream_t)stream);
  return run_dense_rows<bf16>(in, rows, w, cin, cout, w_transposed, bias, after, out, (hipStream_t)stream);
}

namespace ocnn {

// x^T g of fp32 rows with every product and sum in fp32 (v_mfma_f32_32x32x2: two rows an instruction), the weight
// gradient of a 1x1x1 convolution.  A workgroup sums a 64 x 64 block of channel pairs over a range of rows, its waves
// every fourth eight rows, the next eight on their way meanwhile; a lane reads one channel of one row, 32 of them a
// line of 128 bytes, so no LDS until the waves' sums are added.  Ranges of rows fill the chip
// however few blocks there are: the sum over the rows is the long side of this product.  With few channels the launches
// bound it (10 us up to 4096 rows, 16 for 96 -> 64 on 31 k), then the reads (64 -> 13 on 1.13 M rows 117 us), with many the
// instruction: 512 -> 512 on 300 k rows 1381 us, 114 Tflop/s (the library, which splits the rows little: 1585; 96 -> 64 on
// 31 k rows 104, on 1.13 M 1674 / 223).  Its error is the smaller one by 2 - 10 times, the sums being shorter.
constexpr int kRgRows = 32;                                    // rows of a step of a workgroup

__global__ __launch_bounds__(256, 2) void rows_wgrad_f32_kernel(
    const float* __restrict__ x, uint32_t x_bytes, const float* __restrict__ g, uint32_t g_bytes, int64_t rows,
    int64_t rows_per_split, int ca, int cb, int nbb, float* __restrict__ partial) {
  __shared__ __attribute__((aligned(16))) float s_sum[4][64 * 64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, c = lane & 31;
  const int a0 = (int)(blockIdx.y / nbb) * 64, b0 = (int)(blockIdx.y % nbb) * 64;
  const int64_t r_begin = (int64_t)blockIdx.x * rows_per_split, r_end = min(rows, r_begin + rows_per_split);
  const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(x, x_bytes);
  const __amdgpu_buffer_rsrc_t rs_g = make_rsrc(g, g_bytes);
  struct Step { float a[4][2], b[4][2]; };
  // (channels past a row's end belong to the next row: they reach only sums that are not written.  Rows past the
  // end of the range are out of the buffer's range: zeros of both operands)
  auto load = [&](int64_t row0) {
    Step s;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int64_t row = row0 + 2 * t + half;
      const uint32_t xo = row < r_end ? (uint32_t)(row * ca + a0 + c) * 4u : 0xffffff00u;
      const uint32_t go = row < r_end ? (uint32_t)(row * cb + b0 + c) * 4u : 0xffffff00u;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        s.a[t][h] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs_x, xo + 128u * h, 0, 0));
        s.b[t][h] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs_g, go + 128u * h, 0, 0));
      }
    }
    return s;
  };
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  auto add = [&](const Step& s) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(s.a[t][i], s.b[t][j], acc[i][j], 0, 0, 0);
  };
  int64_t row = r_begin + 8 * wave;
  Step s0 = load(row);
  for (; row < r_end; row += 2 * kRgRows) {
    const Step s1 = load(row + kRgRows);
    add(s0);
    s0 = load(row + 2 * kRgRows);
    add(s1);
  }
  // (lane, register r): channels 32 i + 8 (r / 4) + 4 half + r % 4 of x, 32 j + c of g
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) s_sum[wave][(32 * i + 8 * (r >> 2) + 4 * half + (r & 3)) * 64 + 32 * j + c] = acc[i][j][r];
  __syncthreads();
  float* dst = partial + (int64_t)blockIdx.x * ca * cb;
  for (int e = tid; e < 64 * 64; e += 256) {
    const int a = a0 + (e >> 6), b = b0 + (e & 63);
    if (a < ca && b < cb) dst[(int64_t)a * cb + b] = s_sum[0][e] + s_sum[1][e] + s_sum[2][e] + s_sum[3][e];
  }
}

}  // namespace ocnn

// ranges of rows: two workgroups a CU, 256 rows a range at least
static int64_t rg_splits(int64_t rows, int ca, int cb) {
  const int64_t blocks = cdiv(ca, 64) * cdiv(cb, 64);
  return std::max<int64_t>(1, std::min<int64_t>(512 / blocks, cdiv(rows, 256)));
}

extern "C" int ocnnx_rows_wgrad_supported(int dtype, int64_t rows, int ca, int cb) {
  if (dtype != OCNN_F32 || ca < 1 || cb < 1 || ca > 1024 || cb > 1024) return 0;
  return rows >= 0 && (rows + 2) * std::max(ca, cb) * 4 <= 0xfff00000ll;
}

extern "C" int64_t ocnnx_rows_wgrad_workspace_bytes(int64_t rows, int ca, int cb) {
  return align_up(rg_splits(rows, ca, cb) * ca * cb * 4, 256);
}

extern "C" int ocnnx_rows_wgrad(int dtype, const void* x, const void* g, int64_t rows, int ca, int cb, int out_transposed,
                                void* gw, void* workspace, int64_t workspace_bytes, void* stream) {
  OCNN_REQUIRE(ocnnx_rows_wgrad_supported(dtype, rows, ca, cb), "rows_wgrad: shape not supported");
  OCNN_REQUIRE_PTRS("rows_wgrad", gw, workspace);
  if (workspace_bytes < ocnnx_rows_wgrad_workspace_bytes(rows, ca, cb)) {
    set_error("rows_wgrad: workspace too small");
    return OCNN_ERR_WORKSPACE;
  }
  hipStream_t st = (hipStream_t)stream;
  int64_t splits = 0;
  if (rows > 0) {
    OCNN_REQUIRE_PTRS("rows_wgrad", x, g);
    const int64_t per = align_up(cdiv(rows, rg_splits(rows, ca, cb)), kRgRows);
    splits = cdiv(rows, per);
    const int nbb = (int)cdiv(cb, 64);
    hipLaunchKernelGGL(rows_wgrad_f32_kernel, dim3((unsigned)splits, (unsigned)(cdiv(ca, 64) * nbb)), dim3(256), 0, st,
                       (const float*)x, (uint32_t)(rows * ca * 4), (const float*)g, (uint32_t)(rows * cb * 4), rows, per, ca, cb,
                       nbb, (float*)workspace);
    const int rc = check_launch("rows_wgrad");
    if (rc != OCNN_OK) return rc;
  }
  launch_wgrad_reduce<float>((const float*)workspace, (int)splits, 1, ca, cb, out_transposed, (float*)gw, st);
  return check_launch("rows_wgrad (sums)");
}

// What the depth-wise kernels on the tile plan share (dw_planned.hip: any table; dw_siblings.hip: tables of
// whole sibling groups): sizes of a tile's place in LDS, the 4x4x4 matrix instruction, the pipeline from
// global memory to LDS.
#pragma once
#include <algorithm>

#include "common.hpp"
#include "mma.hpp"

namespace ocnn {

constexpr int kDpRows = 128;   // rows per tile (the plan's tile size)
constexpr int kDpCap = 416;    // staged rows; plans with a larger tile use another kernel
constexpr int kDpRowsAlloc = (kDpCap + 8) / 8 * 8;
constexpr int kDpThreads = 512;   // eight waves a workgroup, two a SIMD: one computes while the other waits
constexpr int kDpWaves = kDpThreads / 64;
constexpr int kDpListAlloc = 448;   // entries of a list array in LDS (read in whole pieces of 8 rows a wave)

// (Not in the kernel templates: the arguments of the global->LDS load builtin must not be
// type-dependent expressions.)
static __device__ __forceinline__ void dp_dma16(__amdgpu_buffer_rsrc_t rs, char* dst, uint32_t off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)dst, 16, off, 0, 0, 0);
}

// v_mfma_f32_4x4x4_16b_{f16,bf16}: 16 independent 4x4 products D_b = A_b B_b + C_b.  Lane l = 4 b + i
// holds A_b[i][0..3] and B_b[0..3][i] in its two operand registers (four 16-bit values each) and
// D_b[0..3][i] in its four result registers.  8 cycles an instruction: a depth-wise product costs
// 1/32 of a cycle here against 1/8 on the vector unit (v_dot2c_f32 issues every 8 cycles), with
// three quarters of the multipliers fed zeros.
template <typename T> struct Mma4;
template <> struct Mma4<bf16> {
  static __device__ __forceinline__ f32x4 run(u32x2 a, u32x2 b, f32x4 c) {
    typedef __attribute__((ext_vector_type(4))) short s4;
    return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(s4, a), __builtin_bit_cast(s4, b), c, 0, 0, 0);
  }
};
template <> struct Mma4<f16> {
  static __device__ __forceinline__ f32x4 run(u32x2 a, u32x2 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), c, 0, 0, 0);
  }
};

// s_waitcnt immediates (vmcnt in bits 3:0 and 15:14, no wait on the export and LDS counters).  As an
// instruction of its own, not inline assembly: the compiler's own wait insertion then knows that
// the loads have landed and adds no waits of its own for their registers further down.
constexpr int kDpWaitVm0 = 0x0f70, kDpWaitVm2 = 0x0f72, kDpWaitVm4 = 0x0f74;

static __device__ __forceinline__ void dp_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// What a thread carries from global memory to LDS for the tile after next: its entries of the
// list of distinct rows and its 16-byte pieces of the table positions (as LDS byte offsets).
template <int KT>
struct DpAhead {
  static constexpr int kLoc = (KT * 16 + kDpThreads - 1) / kDpThreads;
  static constexpr int kIds = (kDpRowsAlloc + kDpThreads - 1) / kDpThreads;
  int32_t id[kIds];
  u32x4 lc[kLoc];
};

template <int KT>
static __device__ __forceinline__ void dp_ahead_load(DpAhead<KT>& a, const uint16_t* loc, const int32_t* urows,
                                                     int64_t tile, int32_t p0, int U, int tid) {
#pragma unroll
  for (int r = 0; r < DpAhead<KT>::kIds; ++r) {
    const int i = tid + kDpThreads * r;
    a.id[r] = (i >= 1 && i <= U) ? urows[p0 + i - 1] : -1;
  }
  const u32x4* src = (const u32x4*)(loc + tile * (int64_t)(kDpRows * KT));
#pragma unroll
  for (int r = 0; r < DpAhead<KT>::kLoc; ++r) {
    const int i = tid + kDpThreads * r;
    a.lc[r] = src[min(i, KT * 16 - 1)];
  }
}

// First tile and tile count of workgroup `range` of `ranges` (whole tiles, sizes differ by one).
static __device__ __forceinline__ void dp_tile_range(int64_t tiles, int range, int ranges, int64_t& first, int& n) {
  const int64_t q = tiles / ranges, r = tiles % ranges;
  first = range * q + min<int64_t>(range, r);
  n = (int)(q + (range < r ? 1 : 0));
}

inline int dp_cu_count() {
  static int n_cu = 0;
  if (n_cu == 0) {
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) return 0;
    n_cu = prop.multiProcessorCount;
  }
  return n_cu;
}

inline bool dp_slots_ok(int K) { return K == 27 || K == 9 || K == 8 || K == 3; }

// Tile ranges of the weight gradient: one workgroup per CU over the chunks of the channels.
inline int dp_splits(int C, int n_cu) { return std::min(1024, std::max(1, n_cu / (C / 64))); }

}  // namespace ocnn

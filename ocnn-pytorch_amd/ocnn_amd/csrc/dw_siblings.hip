// Both gradients of a depth-wise 3x3x3 convolution over tables of whole sibling groups: the layers over ALL nodes
// of a level, whose rows 8 g .. 8 g + 7 are the children of one node.
//
//   dx[j][c]    = sum_k g[T[j][k]][c] * w[26-k][c]
//   dw[26-k][c] = sum_j g[T[j][k]][c] * x[j][c]
//
// The 3x3x3 windows of eight siblings make up a block of 4x4x4 cells: 64 rows, not 8 x 27 = 216.  The kernels of
// dw_planned.hip read 216 rows from LDS for a group, once for each sum; here a cell is read once and meets every
// sibling that it is a neighbour of (1, 2, 4 or 8): 64 transposed reads a group for dw, and 96 for dx, where a lane
// keeps the sums of the four siblings of one half.  The rest is as there: the distinct rows of g of a tile staged once in
// LDS for both sums, x as the tile's own 128 rows, products on the 4x4x4 matrix instruction, the next tile's rows in flight.
// 766 k rows of 128 channels: 205 us; both sums from one staging without the cells (dw_planned.hip) 238, a kernel for each
// 290.  180 us with all rows of g in the caches: instructions (the matrix unit is busy for 75 us of them) and the chain of a
// tile.  The output alone is bound by its rows' way into LDS and no faster in this form (126 us either way).
// Tried: four waves with one place for rows, two or three workgroups a CU (211 us, the output 158: a wave alone on its SIMD
// waits for itself); a dword of every row of the tile after next asked for ahead, to have it in L2 (202, 134).
//
// Whether a table is of that kind is found from its plan's positions (plan.hip: tile_siblings_kernel); cell (a, b, c), each
// -1 .. 2, is slot (a - sx, b - sy, c - sz) of sibling (sx, sy, sz) for every sibling that it is a neighbour of.
#include <algorithm>
#include <type_traits>

#include "dw_tile.hpp"
#include "reduce.hpp"

namespace ocnn {

constexpr int kDsK = 27;
constexpr int kDsPitch = 68;     // positions of a group: 64 cells, and 4 more so that 16 groups fall on different banks
constexpr int kDsGroups = kDpRows / 8;

// Staged rows in LDS: row p of the list at row p ^ (bit 3 of p), its 16-byte chunks exchanged by bits 1 and 2:
// c ^ (2 (p3 + p5) + 4 (p2 + p4)).  The lanes of a read want the same cell of 4 or 8 neighbouring groups, which
// lie 4, 8 or 16 list entries apart: 1.45 and 1.6 LDS cycles a read for dx and dw on octrees of spheres and boxes, planes
// and indoor scenes; 2.2 and 3.5 in the order of dw_planned.hip.
// Positions (two per dword, below 512) -> byte offsets; a lane's place in the row is then at offset ^ place.
static __device__ __forceinline__ u32x4 ds_loc_offsets(u32x4 v) {
#pragma unroll
  for (int e = 0; e < 4; ++e)
    v[e] = (v[e] << 7) ^ ((v[e] & 0x00080008u) << 4) ^ ((v[e] & 0x00040004u) << 4) ^ ((v[e] & 0x00100010u) << 2) ^
           ((v[e] & 0x00080008u) << 2) ^ (v[e] & 0x00200020u);
  return v;
}

static __device__ __forceinline__ void ds_stage_rows(__amdgpu_buffer_rsrc_t rs, char* s_rows, const int32_t* s_u,
                                                     int groups, uint32_t pitch, uint32_t coff, int wave, int lane) {
  // LDS row 8 (wave + 8 i) + lane / 8
  const int r = (lane >> 3) ^ (wave & 1);
  const uint32_t st_c = (uint32_t)(((lane & 7) ^ (((r >> 2 ^ wave >> 1) & 1) << 2) ^ (((wave ^ wave >> 2) & 1) << 1)) * 16);
  constexpr int kRowPieces = (kDpCap + 1 + 8 * kDpWaves - 1) / (8 * kDpWaves);
  static_assert(8 * kDpWaves * kRowPieces <= kDpListAlloc, "the list array covers every piece");
  int32_t id[kRowPieces];                                    // all list entries first: one LDS wait
#pragma unroll
  for (int i = 0; i < kRowPieces; ++i) id[i] = s_u[8 * wave + r + 8 * kDpWaves * i];   // -1: out of range, loads zeros
#pragma unroll
  for (int i = 0; i < kRowPieces; ++i) {
    const int g = wave + kDpWaves * i;
    if (g < groups) dp_dma16(rs, s_rows + g * 1024, (uint32_t)id[i] * pitch + (coff + st_c));
  }
}

// The thread's piece of positions is slot tid / 16 of the siblings of group tid % 16: to the cells they name, several siblings
// (and slots) the same one.
static __device__ __forceinline__ void ds_ahead_store(const DpAhead<kDsK>& a, int32_t* s_u, uint16_t* s_cell, int tid) {
  static_assert(DpAhead<kDsK>::kLoc == 1 && DpAhead<kDsK>::kIds == 1, "a piece and an entry a thread");
  if (tid < kDpRowsAlloc) s_u[tid] = a.id[0];
  if (tid < kDsK * kDsGroups) {
    const int k = tid >> 4;
    const u32x4 off = ds_loc_offsets(a.lc[0]);
    uint16_t* dst = s_cell + (tid & 15) * kDsPitch + 16 * (k / 9) + 4 * (k / 3 % 3) + k % 3;
#pragma unroll
    for (int s = 0; s < 8; ++s)
      dst[16 * (s >> 2) + 4 * (s >> 1 & 1) + (s & 1)] = (uint16_t)((s & 1) ? off[s >> 1] >> 16 : off[s >> 1] & 0xffffu);
  }
}

// A workgroup owns a 64-channel chunk and a range of tiles (16 groups each).  Wave v, lane l:
// * dx: half v % 2 (sx) of the groups 4 (v / 2) + l % 4, channels 4 (l / 4) .. + 3; diag(w) of the four
//   channels is operand A, the lane's four channels of the cell operand B, so that its four result registers are the channels of
//   its own row.  The sums of a row are taken in the order of the slots.
// * dw: channels 16 (v % 4) + l % 16 (four lanes of l / 4 % 4 = j share them), groups 4 (l / 16) + j, and the cells with
//   a < 1 (v < 4) or a >= 1; operand A is the cell's row read transposed (a lane: one channel of four groups), operand B the
//   sibling's row of x, contracted over the groups, the diagonal of the result wanted.  Waves of a >= 1 work in the mirror image
//   along x, so that all have the slots -1 and 0 along it (18 of the 27).
// A non-finite x must reach the sums of the slots that have an entry and no others, though an empty cell is a row of
// zeros here: such elements are zeros in operand B and are multiplied one by one with the entries that are there, into
// sums in LDS of their own (infinite or NaN, whatever the order).  (A non-finite g reaches the other three channels of its group of
// four in dx, as in dw_planned.hip.)
template <typename T>
__global__ __launch_bounds__(kDpThreads, 1) void dw_siblings_kernel(
    const T* __restrict__ g, const T* __restrict__ x, uint32_t bytes, const uint16_t* __restrict__ loc,
    const int32_t* __restrict__ uptr, const int32_t* __restrict__ urows, const T* __restrict__ w, T* __restrict__ dx,
    int64_t rows, int C, int64_t tiles, int ranges, int nchunk, float* __restrict__ partial) {
  // (two arrays, not one of two halves: the compiler then knows that the reads of one cannot meet the loads in flight
  // into the other and does not wait for them)
  __shared__ __attribute__((aligned(16))) T s_rows0[kDpRowsAlloc * 64];
  __shared__ __attribute__((aligned(16))) T s_rows1[kDpRowsAlloc * 64];
  __shared__ __attribute__((aligned(16))) T s_x[kDpRows * 64];
  __shared__ __attribute__((aligned(16))) uint16_t s_cell[3][kDsGroups * kDsPitch];
  __shared__ int32_t s_u[2][kDpListAlloc];
  __shared__ float s_odd[kDsK * 64];                         // products of non-finite x

  const int chunk = blockIdx.x % nchunk, range = blockIdx.x / nchunk;
  int64_t t_begin;
  int n;
  dp_tile_range(tiles, range, ranges, t_begin, n);
  if (n <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane & 3;
  for (int i = tid; i < kDsK * 64; i += kDpThreads) s_odd[i] = 0.f;

  // ---- dx ----
  const int half = wave & 1, group = 4 * (wave >> 1) + q, cq = lane >> 2;
  u32x2 wd[kDsK];                                            // the lane's weight of a slot at element q, zeros elsewhere
#pragma unroll
  for (int k = 0; k < kDsK; ++k) {
    const T* wp = w + (int64_t)(kDsK - 1 - k) * C + 64 * chunk + 4 * cq + q;
    const uint32_t v = (uint32_t)__builtin_bit_cast(uint16_t, *wp) << (16 * (q & 1));
    wd[k] = u32x2{(q & 2) ? 0u : v, (q & 2) ? v : 0u};
  }
  const uint32_t cell_dx = 2u * (group * kDsPitch + 16 * half);
  const uint32_t lane_dx = (uint32_t)(cq * 8) * 0x00010001u;

  // ---- dw ----
  const int G = lane >> 4, jj = (lane >> 2) & 3, hx = wave >> 2;
  const int g_dw = 4 * G + jj;
  const uint32_t cell_dw = 2u * (g_dw * kDsPitch + 16 * (hx ? 3 : 0));
  const uint32_t lane_dw = (uint32_t)(32 * (wave & 3) + 8 * q) * 0x00010001u;
  // s_x: row r at row r ^ (bit 3 of r), chunks exchanged by bits 4 and 5 of r: the same sibling of 8 groups on different banks
  const char* x_c = (const char*)s_x + 8 * g_dw * 128 + ((32 * (wave & 3) + 8 * q) ^ (((g_dw >> 1) & 1) << 6) ^ (((g_dw >> 2) & 1) << 5));
  f32x4 acc[18];
#pragma unroll
  for (int k = 0; k < 18; ++k) acc[k] = f32x4{0.f, 0.f, 0.f, 0.f};

  const __amdgpu_buffer_rsrc_t rs_g = make_rsrc(g, bytes);
  const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(x, bytes);
  const __amdgpu_buffer_rsrc_t rs_dx = make_rsrc(dx, bytes);
  const uint32_t pitch = (uint32_t)C * 2u, coff = (uint32_t)chunk * 128u;
  auto stage_x = [&](int64_t tile) {
#pragma unroll
    for (int i = 0; i < kDsGroups / kDpWaves; ++i) {
      const int u = wave + kDpWaves * i;
      const uint32_t cc = (uint32_t)((lane & 7) ^ (((u >> 1) & 1) << 2) ^ (((u >> 2) & 1) << 1));
      const int64_t row = tile * kDpRows + 8 * u + ((lane >> 3) ^ (u & 1));
      const uint32_t off = row < rows ? (uint32_t)row * pitch + (coff + cc * 16u) : 0xfffffff0u;
      dp_dma16(rs_x, (char*)s_x + u * 1024, off);
    }
  };

  // ---- prologue: tile 0 staged, tile 1 on its way to registers, the list range of tile 2 ----
  DpAhead<kDsK> ahead;
  int32_t pa = uptr[t_begin], pb = uptr[t_begin + 1];
  dp_ahead_load<kDsK>(ahead, loc, urows, t_begin, pa, pb - pa, tid);
  ds_ahead_store(ahead, s_u[0], s_cell[0], tid);
  int U_next = pb - pa;
  dp_barrier();
  ds_stage_rows(rs_g, (char*)s_rows0, s_u[0], (U_next + 8) >> 3, pitch, coff, wave, lane);
  stage_x(t_begin);
  if (n > 1) {
    pa = pb;
    pb = uptr[t_begin + 2];
    dp_ahead_load<kDsK>(ahead, loc, urows, t_begin + 1, pa, pb - pa, tid);
    U_next = pb - pa;
  }
  const __amdgpu_buffer_rsrc_t rs_uptr = make_rsrc(uptr, (uint32_t)(tiles + 1) * 4u);
  int32_t pc_v = n > 2 ? uptr[t_begin + 3] : 0;              // (a vector load, whose wait does not hold up LDS reads)
  __builtin_amdgcn_s_waitcnt(kDpWaitVm0);

  int b3 = 0;
  auto tile_step = [&](auto BUF, int i) {
    constexpr int b = decltype(BUF)::value;
    T* rows_cur = b ? s_rows1 : s_rows0;
    T* rows_nxt = b ? s_rows0 : s_rows1;
    const int b3n = b3 == 2 ? 0 : b3 + 1;
    // rows of tile i and the registers for tile i + 1 have arrived; the four stores of the tile before may still be on their way
    __builtin_amdgcn_s_waitcnt(kDpWaitVm4);
    if (i + 1 < n) ds_ahead_store(ahead, s_u[b ^ 1], s_cell[b3n], tid);
    dp_barrier();
    const char* rows_c = (const char*)rows_cur;
    const char* cell_c = (const char*)s_cell[b3];
    u32x2 xf[8];                                             // x of the siblings, in the wave's mirror image
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int row = ((s & 3) | ((s >> 2) ^ hx) << 2) ^ (g_dw & 1);
      xf[s] = Mma<T>::read_tr((const T*)(x_c + row * 128));
    }
    // (a 16-bit value is infinite or NaN iff its low 15 bits plus one in the exponent's last place reach bit 15)
    constexpr uint32_t kOne = std::is_same<T, f16>::value ? 0x04000400u : 0x00800080u;
    uint32_t bad = 0;
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) bad |= (xf[s][h] & 0x7fff7fffu) + kOne;
    if (__builtin_amdgcn_ballot_w64((bad & 0x80008000u) != 0u) != 0ull) {
      if (hx == 0) {
        const int ch = 16 * (wave & 3) + (lane & 15);
#pragma unroll 1
        for (int it = 0; it < 32; ++it) {                  // sibling it / 4 of group 4 G + it % 4
          const int g = 4 * G + (it & 3), s = it >> 2;
          const int at = (8 * g + (s ^ (g & 1))) * 128 + ((2 * ch) ^ (((g >> 1) & 1) << 6) ^ (((g >> 2) & 1) << 5));
          const T v = *(const T*)((const char*)s_x + at);
          if ((((__builtin_bit_cast(uint16_t, v) & 0x7fffu) + kOne) & 0x8000u) == 0u) continue;
#pragma unroll 1
          for (int k = 0; k < kDsK; ++k) {
            const int cell = 16 * ((s >> 2) + k / 9) + 4 * ((s >> 1 & 1) + k / 3 % 3) + (s & 1) + k % 3;
            const uint32_t p = *(const uint16_t*)(cell_c + 2 * (g * kDsPitch + cell));
            if (p != 0u) atomicAdd(&s_odd[k * 64 + ch], to_f32(v) * to_f32(*(const T*)(rows_c + (p ^ (2u * ch)))));
          }
        }
      }
#pragma unroll
      for (int s = 0; s < 8; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const uint32_t m = ((xf[s][h] & 0x7fff7fffu) + kOne) & 0x80008000u;
          xf[s][h] &= ~((m >> 15) * 0xffffu);
        }
    }
    dp_barrier();                                          // s_x is free for the next tile
    if (i + 1 < n) {
      ds_stage_rows(rs_g, (char*)rows_nxt, s_u[b ^ 1], (U_next + 8) >> 3, pitch, coff, wave, lane);
      stage_x(t_begin + i + 1);
    }
    if (i + 2 < n) {
      pa = pb;
      pb = __builtin_amdgcn_readfirstlane(pc_v);
      dp_ahead_load<kDsK>(ahead, loc, urows, t_begin + i + 2, pa, pb - pa, tid);
      U_next = pb - pa;
      if (i + 3 < n) pc_v = __builtin_amdgcn_raw_buffer_load_b32(rs_uptr, (uint32_t)(t_begin + i + 4) * 4u, 0, 0);
    }
    asm volatile("" ::: "memory");

    // Steps of four cells along z (positions: 8 bytes), the rows of the next steps in flight.  Cell iz of a step meets sibling sz in slot
    // iz - sz along z (0 .. 2); the order keeps two instructions that add to the same sums apart.
    constexpr int kIz[6] = {0, 1, 1, 2, 2, 3}, kSz[6] = {0, 1, 0, 1, 0, 1};
    {
      constexpr int STEPS = 8, AHEAD = 2;
      u32x2 pos[STEPS], v[AHEAD + 1][4];
#pragma unroll
      for (int t = 0; t < STEPS; ++t)
        pos[t] = *(const u32x2*)(cell_c + (cell_dw + (t >> 2) * (hx ? -32 : 32)) + (t & 3) * 8);
      auto read_rows = [&](int t) {
        const u32x2 p = pos[t] ^ u32x2{lane_dw, lane_dw};
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[t % (AHEAD + 1)][e] = Mma<T>::read_tr((const T*)(rows_c + ((e & 1) ? p[e >> 1] >> 16 : p[e >> 1] & 0xffffu)));
      };
#pragma unroll
      for (int t = 0; t < AHEAD; ++t) read_rows(t);
#pragma unroll
      for (int t = 0; t < STEPS; ++t) {
        if (t + AHEAD < STEPS) read_rows(t + AHEAD);
        __builtin_amdgcn_sched_barrier(0);
        const int ix = t >> 2, iy = t & 3;
#pragma unroll
        for (int sx = 0; sx <= ix; ++sx)                     // (mirrored: cell ix - 1, slots -1 and 0)
#pragma unroll
          for (int sy = 0; sy < 2; ++sy) {
            if (iy - sy < 0 || iy - sy > 2) continue;
#pragma unroll
            for (int e = 0; e < 6; ++e) {
              const int k = 9 * (ix - sx) + 3 * (iy - sy) + kIz[e] - kSz[e];
              acc[k] = Mma4<T>::run(v[t % (AHEAD + 1)][kIz[e]], xf[4 * sx + 2 * sy + kSz[e]], acc[k]);
            }
          }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    {
      constexpr int STEPS = 12, AHEAD = 2;
      u32x2 pos[STEPS], v[AHEAD + 1][4];
      f32x4 sum[2][2];
#pragma unroll
      for (int j = 0; j < 2; ++j) sum[j][0] = sum[j][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < STEPS; ++t) pos[t] = *(const u32x2*)(cell_c + cell_dx + (t >> 2) * 32 + (t & 3) * 8);
      auto read_rows = [&](int t) {
        const u32x2 p = pos[t] ^ u32x2{lane_dx, lane_dx};
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[t % (AHEAD + 1)][e] = *(const u32x2*)(rows_c + ((e & 1) ? p[e >> 1] >> 16 : p[e >> 1] & 0xffffu));
      };
#pragma unroll
      for (int t = 0; t < AHEAD; ++t) read_rows(t);
#pragma unroll
      for (int t = 0; t < STEPS; ++t) {
        if (t + AHEAD < STEPS) read_rows(t + AHEAD);
        __builtin_amdgcn_sched_barrier(0);
        const int iy = t & 3;
#pragma unroll
        for (int e = 0; e < 6; ++e)
#pragma unroll
          for (int sy = 0; sy < 2; ++sy) {
            if (iy - sy < 0 || iy - sy > 2) continue;
            sum[sy][kSz[e]] = Mma4<T>::run(wd[9 * (t >> 2) + 3 * (iy - sy) + kIz[e] - kSz[e]], v[t % (AHEAD + 1)][kIz[e]], sum[sy][kSz[e]]);
          }
        __builtin_amdgcn_sched_barrier(0);
      }
      const int64_t row0 = (t_begin + i) * kDpRows + 8 * group + 4 * half;
      // (every lane issues its four stores: the wait at the top counts on it; groups past the end are dropped)
      const uint32_t off = row0 < rows ? (uint32_t)row0 * pitch + (coff + (uint32_t)cq * 8u) : 0xffff0000u;
#pragma unroll
      for (int s = 0; s < 4; ++s)
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack2<T>(sum[s >> 1][s & 1][0], sum[s >> 1][s & 1][1]),
                                                    pack2<T>(sum[s >> 1][s & 1][2], sum[s >> 1][s & 1][3])},
                                              rs_dx, row0 < rows ? off + s * pitch : off, 0, 0);
    }
    asm volatile("" ::: "memory");
    b3 = b3n;
  };
  for (int i = 0; i < n; i += 2) {
    tile_step(std::integral_constant<int, 0>{}, i);
    if (i + 1 < n) tile_step(std::integral_constant<int, 1>{}, i + 1);
  }

  // ---- dw: the diagonal elements of a channel's four lanes of groups, then the two halves, in a fixed order ----
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  float* s_red = (float*)s_rows0;                          // [18 slots][half][64 channels]
#pragma unroll
  for (int k = 0; k < 18; ++k) {
    float v = q == 0 ? acc[k][0] : q == 1 ? acc[k][1] : q == 2 ? acc[k][2] : acc[k][3];
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    if (lane < 16) s_red[(k * 2 + hx) * 64 + 16 * (wave & 3) + lane] = v;
  }
  __syncthreads();
  for (int i = tid; i < kDsK * 64; i += kDpThreads) {
    const int k = i >> 6, ch = i & 63, ox = k / 9 - 1, rest = k % 9;
    float v = s_odd[i];
    if (ox <= 0) v += s_red[((9 * (ox + 1) + rest) * 2 + 0) * 64 + ch];
    if (ox >= 0) v += s_red[((9 * (1 - ox) + rest) * 2 + 1) * 64 + ch];
    partial[((int64_t)range * kDsK + (kDsK - 1 - k)) * C + 64 * chunk + ch] = v;
  }
}

}  // namespace ocnn

using namespace ocnn;

// Calls that the kernel takes: f16 / bf16, channels % 64, whole groups, a table of 27 slots whose plan says that it is one of
// sibling groups.
extern "C" int ocnnx_dwconv_siblings_supported(int dtype, int64_t rows, int K, int channels, int plan_max_distinct) {
  return K == kDsK && rows % 8 == 0 && ocnn_dwconv_wgrad_planned_supported(dtype, rows, rows, K, channels, plan_max_distinct);
}

// As ocnnx_dwconv_backward_planned.
extern "C" int ocnnx_dwconv_siblings_backward(int dtype, const void* x, const void* g, const uint16_t* loc, const int32_t* uptr,
                                              const int32_t* urows, int plan_max_distinct, int64_t plan_total, int64_t rows,
                                              int K, const void* w, int channels, void* dx, void* gw, void* workspace,
                                              int64_t workspace_bytes, void* stream) {
  OCNN_REQUIRE(ocnnx_dwconv_siblings_supported(dtype, rows, K, channels, plan_max_distinct),
               "dwconv_siblings_backward: shape not supported");
  OCNN_REQUIRE(rows < (1ll << 31) && plan_total >= 0 && plan_total < (1ll << 29), "dwconv_siblings_backward: rows out of range");
  OCNN_REQUIRE_PTRS("dwconv_siblings_backward", w, gw, workspace);
  OCNN_REQUIRE(rows == 0 || (x && g && loc && uptr && urows && dx),
               "dwconv_siblings_backward: a required pointer is NULL (of x, g, loc, uptr, urows, dx)");
  const int n_cu = dp_cu_count();
  if (n_cu <= 0) {
    set_error("dwconv_siblings_backward: cannot query the device");
    return OCNN_ERR_HIP;
  }
  const int nchunk = channels / 64;
  const int64_t tiles = cdiv(rows, kDpRows);
  const int ranges = (int)std::min<int64_t>(tiles, dp_splits(channels, n_cu));
  if (workspace_bytes < (int64_t)ranges * K * channels * 4) {
    set_error("dwconv_siblings_backward: workspace too small");
    return OCNN_ERR_WORKSPACE;
  }
  hipStream_t st = (hipStream_t)stream;
  auto run = [&](auto t) {
    typedef decltype(t) T;
    if (rows > 0)
      hipLaunchKernelGGL((dw_siblings_kernel<T>), dim3((unsigned)(ranges * nchunk)), dim3(kDpThreads), 0, st, (const T*)g,
                         (const T*)x, (uint32_t)(rows * channels * 2), loc, uptr, urows, (const T*)w, (T*)dx, rows, channels, tiles,
                         ranges, nchunk, (float*)workspace);
    launch_wgrad_reduce<T>((float*)workspace, ranges, K, 1, channels, 0, (T*)gw, st);
  };
  if (dtype == OCNN_F16) run(f16{});
  else run(bf16{});
  return check_launch("dwconv_siblings_backward");
}

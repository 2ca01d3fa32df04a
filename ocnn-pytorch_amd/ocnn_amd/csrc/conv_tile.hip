// Gather-GEMM on the tile plan of the neighbour table, with the weights streamed from L2: the
// layers whose weights do not stay in registers (conv_rw.hip) and, in fp32, the planned layers
// (which of them: select.hip).
//
// A workgroup takes one tile of 128 table rows and 32 .. 256 output channels.  The distinct input
// rows of the tile are staged in LDS 128 bytes at a time (64 channels of f16 / bf16, 32 of fp32);
// the weights stream straight into registers, already in the layout of the MFMA A operand (no LDS
// round trip).  M = output channels, N = rows, v_mfma_f32_32x32x16.  A wave owns 64 or 96 output channels of
// 128 or 64 rows (32 of 128 where a layer has no more): a row read from LDS feeds two or three MFMAs and a weight
// fetched four or two.  Layers of fewer channels than four such waves split the SLOTS over the waves instead, whose
// sums are added in LDS at the end.  (Waves of 32 channels x 128 rows side by side read LDS once per MFMA, as fast
// as its pipe delivers gathered rows: on the non-empty nodes of depth 7, 533 k rows, 128 -> 128 381 us, so 328.)
// Two or three workgroups share a CU: while one waits for its next chunk of channels the others compute.
//
// fp32: x = hi + lo in bf16 pieces, accumulated in fp32 as hi hi + hi lo + lo hi (about 1e-5
// relative).  The rows are read as fp32 and split on their way into LDS, so that a row's 128 bytes
// there are [hi | lo] of 32 channels, and the same pair of LDS reads and of weight loads feeds three
// MFMAs: a third of the reads per MFMA that the layer takes as a bf16 layer of three times the
// channels ([hi | hi | lo] x [hi; lo; hi]), and no passes that write and read the pieces.
//
// Few tiles (the coarse levels of a network, small clouds): 128 rows x 128 channels of 256 -> 256 are
// 50 us of one workgroup's time however many CUs are idle.  The launch then also splits the
// reduction, over chunks of input channels and over the slots; each part writes fp32 sums of its own, and a
// second kernel adds them in the order of the parts.
#include <algorithm>
#include <new>
#include <type_traits>

#include "jobs.hpp"

namespace ocnn {

constexpr int kTgRows = 128;   // rows per tile (the plan's tile size)
constexpr int kTgCap = 416;    // staged rows; plans with a larger tile use another kernel
constexpr int kTgRowsAlloc = (kTgCap + 8) / 8 * 8;   // LDS rows 0..kTgCap in whole 8-row groups
// share of a table's entries that are set up to which the kernel tests for empty (32-row block,
// slot) units: non-empty nodes of coarse levels, where a tenth to a half of the units are empty.  With the test / without,
// f16 and fp32, 64 to 256 channels: 0.83 - 0.93 at 22 % set, 0.84 - 0.95 at 36 %, 0.88 - 1.0 at 38 %, 0.96 - 1.0 at
// 41 - 44 %, 0.99 - 1.03 at 50 - 58 %, 0.99 - 1.03 over all nodes (70 %)
constexpr double kTgSkipMaxOccupancy = 0.45;

// (Not in the kernel template: the arguments of the global->LDS load builtin must not be
// type-dependent expressions.)
static __device__ __forceinline__ void tg_dma16(__amdgpu_buffer_rsrc_t rs, char* dst, uint32_t off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)dst, 16, off, 0, 0, 0);
}

// SKIP: a wave leaves out the MFMAs of a slot and 32-row block of the tile where no row has an entry.  Blocks are the outer
// loop of a slot, so that one branch stands around a block's 4 - 18 MFMAs: with the k-steps outside and a branch
// per MFMA the same tables took 6 - 10 % longer.  The rows of a block are read one block ahead, behind a branch of their own.
//
// order: the tile's rows in an order that leaves fewer blocks with an entry (plan.hip: tile_order_kernel); position i of
// a block is row order[i].  It costs the loop nothing (a lane's row is a register either way), and a row's result is the
// same to the bit (of finite values): it has the same products in every wave, and the waves' sums meet in the same pairs whichever block the row
// is in.  Neither MFMAs nor bytes alone bound the loop on such tables (96 -> 96 on 1.13 M rows, 7 % set: 139 us without any slot,
// 280 with a quarter of the MFMAs, 290 with one fetch of weights a chunk), so a turn of it waits for as little as can be:
// two sets of registers in turn, the live blocks of a slot known beforehand from a byte behind the order, half the weights
// of half a chunk.  In us before / now: f16 1.13 M rows 7 % set 96 -> 96 334 / 293, 947 k 15 % 329 / 292, 533 k 31 % 128 -> 128
// 299 / 264, 160 k 38 % 256 -> 256 383 / 341, 31 k 17 % 96 -> 96 26.7 / 21.9; fp32 132 k 36 % 96 -> 96 153 / 145, 264 k 22 %
// 64 -> 64 132 / 124 (105 with three workgroups a CU: tile_half_waves).  Up to two thousand rows the order's own fetch shows: 1.8 k
// rows 28 % set 128 -> 128 20.5 / 21.5, fp32 96 -> 96 22.5 / 23.5, 32 -> 64 13.7 / 13.1.  Above the line of kTgSkipMaxOccupancy
// it gains where a cloud is flat (1.28 M rows 68 % set 96 -> 96 620 / 576) and loses elsewhere (97 k 52 % 256 -> 256 282 / 292).
//
// The four waves: WC along the output channels (32 MB each), WR along the rows (RB = 4 / WR blocks of 32 rows
// each), KS over the slots (each takes every KS-th; their sums are added in LDS at the end).
template <typename T, bool F32, int MB, int WC, int WR, int KS, bool SKIP>
__global__ __launch_bounds__(256, MB * (4 / WR) <= 4 ? 3 : 2) void conv_gather_tile_kernel(
    const void* __restrict__ in, uint32_t in_bytes, const uint16_t* __restrict__ loc,
    const int32_t* __restrict__ uptr, const int32_t* __restrict__ urows, const uint8_t* __restrict__ order,
    const T* __restrict__ wpk, const void* __restrict__ bias_, ocnnx_bn bn, void* __restrict__ out_, float* __restrict__ partial,
    int64_t rows_out, int K, int cin, int cout, int64_t tiles, int64_t tiles_per_xcd, int sc, int sk, int rows_alloc) {
  typedef typename std::conditional<F32, float, T>::type O;
  constexpr int RB = 4 / WR, RBK = RB / KS, CH = F32 ? 32 : 64;
  static_assert(WC * WR * KS == 4 && RB % KS == 0 && RB % 2 == 0, "four waves; blocks in pairs");
  extern __shared__ __attribute__((aligned(16))) char s_rows[];    // rows_alloc rows, positions, the list
  uint16_t* s_loc = (uint16_t*)(s_rows + rows_alloc * 128);
  int32_t* s_u = (int32_t*)(s_loc + ((K + sk - 1) / sk) * kTgRows);
  uint32_t* s_live = (uint32_t*)(s_u + rows_alloc);                // of a slot: its 32-row blocks with an entry (bits)

  const int64_t tile = tiles_per_xcd > 0 ? xcd_tile(blockIdx.x, tiles_per_xcd) : (int64_t)blockIdx.x;
  if (tile >= tiles) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wc = wave % WC, wr = wave / WC % WR, ks = wave / (WC * WR);
  const int q = lane >> 5, r32 = lane & 31;
  const int ncc = (cin + CH - 1) / CH;
  const int ncg = cout >> 5;
  const int cg0 = ((int)blockIdx.y * WC + wc) * MB;         // first 32-channel group of this wave
  const uint32_t pitch = (uint32_t)cin * (F32 ? 4u : 2u);
  const int zc = (int)blockIdx.z / sk, zk = (int)blockIdx.z - zc * sk;
  const int c0 = ncc * zc / sc, c1 = ncc * (zc + 1) / sc;
  const int k0 = K * zk / sk, k1 = K * (zk + 1) / sk;

  // ---- the tile's list of distinct rows and its table positions -> LDS ----
  // (positions first: they don't wait for the list's place)
  constexpr int LP = 27 * 16 / 256 + 1;
  u32x4 lv[LP];
  uint32_t blocks = 0;                                       // of lane k - k0: the slot's 32-row blocks with an entry (bits)
  if constexpr (SKIP)
    if (order && lane < k1 - k0) blocks = order[tile * OCNNX_TILE_ORDER_BYTES + kTgRows + k0 + lane];
  {
    const u32x4* src = (const u32x4*)(loc + (tile * K + k0) * (int64_t)kTgRows);
#pragma unroll
    for (int i = 0; i < LP; ++i)
      if (tid + 256 * i < (k1 - k0) * 16) lv[i] = src[tid + 256 * i];
  }
  const int32_t p0 = uptr[tile];
  const int U = uptr[tile + 1] - p0;
  for (int i = tid; i < rows_alloc; i += 256)
    s_u[i] = (i >= 1 && i <= U) ? urows[p0 + i - 1] : -1;  // LDS row p holds list entry p - 1; row 0 = zeros
#pragma unroll
  for (int i = 0; i < LP; ++i)
    if (tid + 256 * i < (k1 - k0) * 16) ((u32x4*)s_loc)[tid + 256 * i] = lv[i];
  const int groups = (U + 8) >> 3;                          // 8-row groups of LDS rows 0..U

  const __amdgpu_buffer_rsrc_t rs_in = make_rsrc(in, in_bytes);
  // piece i of a wave: the 8 LDS rows from 8 wave + 32 i on, a lane 16 bytes of one of them.
  // 16-byte chunk c of LDS row p sits at chunk c ^ ((p >> 1) & 7) (bank swizzle)
  const int st_p = 8 * wave + (lane >> 3);                  // LDS row of piece 0; piece i: + 32 i
  const uint32_t st_x = (uint32_t)(((lane >> 4) + 4 * wave) & 7);
  const uint32_t st_c = (uint32_t)(((lane & 7) ^ st_x) * 16);
  const bool half_oob = !F32 && (cin & 63) != 0 && st_c >= 64;      // this lane's piece of a half chunk at the end
  constexpr int kRowPieces = (kTgCap + 1 + 31) / 32;

  f32x16 acc[RB][MB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[rb][mb][r] = 0.f;

  // ---- operands ----
  // A: the weights of a (chunk, slot), four pieces of 16 bytes a lane and M tile
  const uint32_t kstride = (uint32_t)ncg * 4096u;            // bytes between consecutive (chunk, slot)
  const bool active = cg0 < ncg;                             // (wave-uniform)
  auto load_a = [&](int kk, u32x4 (&a)[4][MB], auto STEPS) {
    const char* base = (const char*)wpk + (uint64_t)((uint32_t)kk * kstride);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const char* tile_of = base + (uint32_t)min(cg0 + mb, ncg - 1) * 4096u;   // (uniform: the lanes differ in a 32-bit offset)
#pragma unroll
      for (int s = 0; s < decltype(STEPS)::value; ++s) a[s][mb] = *(const u32x4*)(tile_of + (uint32_t)(lane * 16 + s * 1024));
    }
  };
  // B: a lane reads 16 bytes (8 input channels, or their high or low pieces) of the neighbour row of
  // one of the tile's rows, row at[rb] in block rb.  pv = byte address of the row in s_rows with the swizzle of piece 0 folded in.
  int at[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    at[rb] = 32 * (RB * wr + rb) + r32;
    if constexpr (SKIP)
      if (order) at[rb] = order[tile * OCNNX_TILE_ORDER_BYTES + at[rb]];
  }
  auto load_pos = [&](int k, uint32_t (&pv)[RB]) {
    const uint16_t* p = s_loc + (k - k0) * kTgRows;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      const uint32_t l = p[at[rb]];                          // 0 = empty = the zero row
      pv[rb] = (l << 7) | (((l << 3) & 0x70u) ^ ((uint32_t)q << 4));
    }
  };
  auto read_b = [&](uint32_t pv, u32x4 (&b)[4], auto STEPS) {
#pragma unroll
    for (int s = 0; s < decltype(STEPS)::value; ++s) b[s] = *(const u32x4*)(s_rows + (pv ^ ((uint32_t)s << 5)));
  };
  // a block of 32 rows with everything of a slot: behind one branch
  auto multiply = [&](const u32x4 (&a)[4][MB], const u32x4 (&b)[4], f32x16 (&c)[MB], auto STEPS) {
    constexpr int S = decltype(STEPS)::value;
    auto mma = [&](int i, int j) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) c[mb] = Mma32<T>::run(a[i][mb], b[j], c[mb]);
    };
    if constexpr (F32) {                                     // pieces 0, 1 of a: high, low of k-step 0; 0, 2 of b
      mma(0, 0), mma(0, 2), mma(1, 0);
      mma(2, 1), mma(2, 3), mma(3, 1);
    } else {
#pragma unroll
      for (int s = 0; s < S; ++s) mma(s, s);
    }
  };

  // the distinct rows' channels of chunk cc -> LDS; between(): what is done behind the barrier in front
  __syncthreads();
  auto stage_chunk = [&](int cc, auto between) {
    if constexpr (F32) {
      // fp32 rows through registers, split into their bf16 pieces on the way: a lane's four channels
      // 4 (lane % 8) .. are half a 16-byte chunk of either piece
      constexpr int D = 7;                                   // loads in flight
      f32x4 v[D];
      auto load = [&](int i, f32x4& x) {
        if (wave + 4 * i < groups)
          x = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                     rs_in, (uint32_t)s_u[st_p + 32 * i] * pitch + (uint32_t)cc * 128u + (uint32_t)(lane & 7) * 16u, 0, 0));
      };
#pragma unroll
      for (int i = 0; i < D; ++i) load(i, v[i]);
      __syncthreads();                                       // every wave is done with the chunk before
      between();
      const uint32_t half = (uint32_t)(lane & 1) * 8u, ch = (uint32_t)(lane & 7) >> 1;
#pragma unroll
      for (int i = 0; i < kRowPieces; ++i) {
        if (wave + 4 * i < groups) {
          typedef __attribute__((ext_vector_type(4))) T t4;
          t4 hi, lo;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            hi[j] = (T)v[i % D][j];
            lo[j] = (T)(v[i % D][j] - (float)hi[j]);
          }
          char* row = s_rows + (st_p + 32 * i) * 128;
          *(t4*)(row + (ch ^ st_x) * 16u + half) = hi;
          *(t4*)(row + ((ch | 4u) ^ st_x) * 16u + half) = lo;
        }
        if (i + D < kRowPieces) load(i + D, v[i % D]);
      }
      __syncthreads();
    } else {
      __syncthreads();                                       // every wave is done with the chunk before
      between();
      // (list entries in two halves: registers)
      constexpr int D = (kRowPieces + 1) / 2;
#pragma unroll
      for (int h = 0; h < kRowPieces; h += D) {
        int32_t ids[D];
#pragma unroll
        for (int i = 0; i < D; ++i) ids[i] = s_u[min(st_p + 32 * (h + i), rows_alloc - 1)];   // -1: out of range, loads zeros
#pragma unroll
        for (int i = 0; i < D; ++i) {
          const int g = wave + 4 * (h + i);
          if (h + i < kRowPieces && g < groups) {
            uint32_t off = (uint32_t)ids[i] * pitch + ((uint32_t)cc * 128u + st_c);
            if (cc == ncc - 1 && half_oob) off = 0xffffff00u;  // past the row's channels: zeros, not the next row
            tg_dma16(rs_in, s_rows + g * 1024, off);
          }
        }
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
  };

  // This wave's slots (bit k - k0): every KS-th one, with SKIP those of them that have an entry in its rows.
  // (A slot without any costs the weights' way through L1, the busiest unit with 46 - 62 % on such tables, and a turn of the
  // loop.  Indoor scenes, non-empty nodes: 47 % of a tile's slots at depth 9, 1.13 M rows 96 -> 96 423 us, without them 323;
  // 37 % at depth 8, 947 k rows 380 / 327; 30 % at depth 7, 533 k rows 128 -> 128 332 / 317.)
  uint32_t own = 0;
  bool works = false;
  auto find_live = [&]() {
    if constexpr (SKIP)
      if (!order)
        for (int k = wave; k < k1 - k0; k += 4) {
          const unsigned long long lo = __builtin_amdgcn_ballot_w64(s_loc[k * kTgRows + lane] != 0);
          const unsigned long long hi = __builtin_amdgcn_ballot_w64(s_loc[k * kTgRows + 64 + lane] != 0);
          if (lane == 0)
            s_live[k] = ((uint32_t)lo ? 1u : 0u) | (lo >> 32 ? 2u : 0u) | ((uint32_t)hi ? 4u : 0u) | (hi >> 32 ? 8u : 0u);
        }
  };
  auto deal_slots = [&]() {
    uint32_t live = (1u << (k1 - k0)) - 1u;
    if constexpr (SKIP) {
      if (!order && lane < k1 - k0) blocks = s_live[lane];
      blocks = (blocks >> (RB * wr)) & ((1u << RB) - 1u);    // (of this wave's rows)
      live = (uint32_t)__builtin_amdgcn_ballot_w64(blocks != 0u);
    }
    // (every KS-th slot whether or not it is live: in the table's order the same sums as without SKIP, to the bit.  Dealing the live
    // ones in turn evens the waves out and takes 1.0 - 1.03 x as long)
    own = live & ((KS == 4 ? 0x11111111u : (KS == 2 ? 0x55555555u : 0xffffffffu)) << ks);
    works = active && own != 0u;
    if (own == 0u) own = 1u;                                 // (nothing to do: a turn without products)
  };

  // Two slots in hand: the one whose products run, with its weights A, positions and live blocks, and the next one's on
  // their way.  (Two sets of names, in turn: the copies of one set into the other were 24 - 36 instructions a slot, and the
  // blocks that have an entry are known beforehand, so that no branch waits for the positions.)
  u32x4 A[2][4][MB], B[2][4];
  uint32_t pv[2][RB], nz[2] = {~0u, ~0u};
  auto fetch_slot = [&](int cc, int k, auto P, auto STEPS) {
    constexpr int p = decltype(P)::value;
    load_a(cc * K + k, A[p], STEPS);
    load_pos(k, pv[p]);
    if constexpr (SKIP) nz[p] = (uint32_t)__builtin_amdgcn_readlane((int)blocks, k - k0);
  };
  // set P holds the first slot's when a chunk begins (P = 0)
  auto chunk = [&](int cc, auto STEPS) {
    uint32_t rest = own;
    auto slot = [&](auto P) {
      constexpr int p = decltype(P)::value;
      rest &= rest - 1u;
      // the next slot; behind the last one the first of the next chunk (of this one again behind the last chunk)
      const int kn = k0 + __builtin_ctz(rest ? rest : own);
      fetch_slot(rest ? cc : min(cc + 1, c1 - 1), kn, std::integral_constant<int, 1 - p>{}, STEPS);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        // the next block's rows (past the last slot: rows of this chunk, unused)
        if (rb + 1 < RB) {
          if (!SKIP || (nz[p] & (2u << rb))) read_b(pv[p][rb + 1 < RB ? rb + 1 : 0], B[(rb + 1) & 1], STEPS);
        } else {
          if (!SKIP || (nz[1 - p] & 1u)) read_b(pv[1 - p][0], B[0], STEPS);
        }
        if (works && (!SKIP || (nz[p] & (1u << rb)))) multiply(A[p], B[rb & 1], acc[rb], STEPS);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    read_b(pv[0][0], B[0], STEPS);
    for (;;) {
      slot(std::integral_constant<int, 0>{});
      if (rest == 0u) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int s = 0; s < 4; ++s) A[0][s][mb] = A[1][s][mb];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) pv[0][rb] = pv[1][rb];
        nz[0] = nz[1];
        break;
      }
      slot(std::integral_constant<int, 1>{});
      if (rest == 0u) break;
    }
  };
  find_live();
  auto staged_chunk = [&](int cc, auto STEPS) {
    stage_chunk(cc, [&]() {
      if (cc == c0) {                                        // (the first weights come beside the rows)
        deal_slots();
        fetch_slot(c0, k0 + __builtin_ctz(own), std::integral_constant<int, 0>{}, STEPS);
      }
    });
    chunk(cc, STEPS);
  };
  const int nfull = F32 ? c1 : min(c1, cin >> 6);            // whole chunks up to here
  for (int cc = c0; cc < nfull; ++cc) staged_chunk(cc, std::integral_constant<int, 4>{});
  if constexpr (!F32)
    if (nfull < c1) staged_chunk(nfull, std::integral_constant<int, 2>{});   // half a chunk: its first two k-steps

  // ---- KS > 1: the waves' sums of a block are added by one of them: of two waves, or of four as (0 + 2) + (1 + 3), the
  // same pairs for every block and whichever wave has it ----
  if constexpr (KS > 1) {
    f32x4* ex = (f32x4*)s_rows;
    constexpr int kPart = RBK * MB * 4 * 64;                 // a wave's sums of the blocks of one owner
    auto put = [&](int o, f32x4* dst) {
#pragma unroll
      for (int i = 0; i < RBK; ++i)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            dst[((i * MB + mb) * 4 + r) * 64 + lane] = f32x4{acc[RBK * o + i][mb][4 * r], acc[RBK * o + i][mb][4 * r + 1],
                                                             acc[RBK * o + i][mb][4 * r + 2], acc[RBK * o + i][mb][4 * r + 3]};
    };
    auto take = [&](int o, const f32x4* src) {
#pragma unroll
      for (int i = 0; i < RBK; ++i)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const f32x4 v = src[((i * MB + mb) * 4 + r) * 64 + lane];
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[RBK * o + i][mb][4 * r + j] += v[j];
          }
    };
    if constexpr (KS == 2) {
      // both owners at once
      f32x4 *mine = ex + wave * kPart, *other = ex + (wave ^ (WC * WR)) * kPart;
      __syncthreads();
      if (ks == 0) put(1, mine);
      else put(0, mine);
      __syncthreads();
      if (ks == 0) take(0, other);
      else take(1, other);
    } else {
      // halves of the blocks between waves two apart, then single blocks between neighbours: four barriers and
      // every wave at work, where one owner after the other took eight (f16 32 -> 64 on 264 k rows, 22 % set,
      // 56.2 us, so 52.9, 64 -> 32 on 132 k rows 28.3 / 25.7, fp32 64 -> 64 129.9 / 128.5)
      static_assert(KS != 4 || (WC * WR == 1 && RBK == 1), "a block a wave");
      f32x4 *mine = ex + wave * 2 * kPart, *far = ex + (wave ^ 2) * 2 * kPart, *near = ex + (wave ^ 1) * 2 * kPart;
      __syncthreads();
      if (ks < 2) put(2, mine), put(3, mine + kPart);
      else put(0, mine), put(1, mine + kPart);
      __syncthreads();
      if (ks < 2) take(0, far), take(1, far + kPart);
      else take(2, far), take(3, far + kPart);
      __syncthreads();
      if (ks == 0) put(1, mine);
      else if (ks == 1) put(0, mine);
      else if (ks == 2) put(3, mine);
      else put(2, mine);
      __syncthreads();
      if (ks == 0) take(0, near);
      else if (ks == 1) take(1, near);
      else if (ks == 2) take(2, near);
      else take(3, near);
    }
  }

  // ---- epilogue: a lane holds 16 consecutive output channels of a row per M tile ----
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    if (cg0 + mb >= ncg) continue;
    const int co = 32 * (cg0 + mb) + 16 * q;
    if (partial) {
      // [part][16-channel group][4-channel quarter][row][4]: the lanes of a store are consecutive rows
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        if (KS > 1 && rb / RBK != ks) continue;
        const int64_t row = tile * kTgRows + at[rb];
        if (row >= rows_out) continue;
        float* dst = partial + (((int64_t)blockIdx.z * (cout >> 2) + (co >> 2)) * rows_out + row) * 4;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          *(f32x4*)(dst + r * rows_out * 4) =
              f32x4{acc[rb][mb][4 * r], acc[rb][mb][4 * r + 1], acc[rb][mb][4 * r + 2], acc[rb][mb][4 * r + 3]};
      }
      continue;
    }
    float mul[16], add[16];
    layer_tail<O, 16>((const O*)bias_, bn, co, mul, add);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      if (KS > 1 && rb / RBK != ks) continue;
      const int64_t row = tile * kTgRows + at[rb];
      if (row >= rows_out) continue;
      float v[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) v[r] = acc[rb][mb][r] * mul[r] + add[r];
      if (bn.residual) {
        const O* res = (const O*)bn.residual + row * cout + co;
#pragma unroll
        for (int r = 0; r < 16; ++r) v[r] += to_f32(res[r]);
      }
      if (bn.relu) {
#pragma unroll
        for (int r = 0; r < 16; ++r) v[r] = fmaxf(v[r], 0.f);
      }
      if constexpr (F32) {
        float* dst = (float*)out_ + row * cout + co;
#pragma unroll
        for (int r = 0; r < 16; r += 4) *(f32x4*)(dst + r) = f32x4{v[r], v[r + 1], v[r + 2], v[r + 3]};
      } else {
        unsigned pk[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) pk[r] = pack2<T>(v[2 * r], v[2 * r + 1]);
        T* dst = (T*)out_ + row * cout + co;
        *(u32x4*)(dst) = u32x4{pk[0], pk[1], pk[2], pk[3]};
        *(u32x4*)(dst + 8) = u32x4{pk[4], pk[5], pk[6], pk[7]};
      }
    }
  }
}

struct TileLaunch {
  int mb, wc, wr, ks;          // shape of a wave: 32 mb channels x 128 / wr rows, every ks-th slot; wc waves along the channels
  int gy;                      // blocks of output channels
  int sc, sk;                  // parts of the reduction: chunks x slots
};

// What a launch of few tiles takes, in us, cut into sc x sk parts: rounds of the workgroups that run at once
// (two a CU), each of them its rows' staging and its waves' slots one behind the other, and the parts' sums
// written and read.  A slot takes the longer of its MFMAs (half as long again with a second workgroup on the CU)
// and a round trip for the next slot's weights.  The constants are a fit to 670 timed launches (2 - 324 tiles, seven
// pairs of channels, f16 and fp32, 1 - 32 parts): 7 % off in the mean, and the parts it picks take 1.3 % longer
// than the best ones; a rule by thresholds on units and workgroups took 6 %.
static double tile_cost(const TileLaunch& t, bool f32, int64_t tiles, int K, int ncc, int cout, int sc, int sk) {
  const double kLaunch = 8.8, kParts = 3.8, kPartBytes = 1.8e-7, kChunk = 0.96, kSlot = 0.245, kMfma = 0.0228;
  const int chunks = (int)cdiv(ncc, sc), slots = chunks * (int)cdiv(cdiv(K, sk), t.ks);
  const double mfma = kMfma * t.mb * (4 / t.wr) * (f32 ? 6 : 4);
  auto round = [&](int per_cu) { return chunks * kChunk + slots * std::max(kSlot, mfma * (0.5 + 0.5 * per_cu)); };
  const int64_t groups = tiles * t.gy * sc * sk, rest = groups % 512;
  const double us = kLaunch + (double)(groups / 512) * round(2) + (rest == 0 ? 0.0 : round(rest <= 256 ? 1 : 2));
  return sc * sk == 1 ? us : us + kParts + kPartBytes * sc * sk * (double)tiles * kTgRows * cout * 8;
}

// How a launch is cut up.  256 channels a workgroup stage a tile's rows once for all of them where there are tiles
// enough.  From some 600 workgroups on the last, half-empty round costs less than the sums.
constexpr int kTgPartsGroups = 640;
constexpr int kTgMaxSlotParts = 6;

// Whether the four waves of 64 output channels take 32 channels and half the slots each, three workgroups a CU, in place of
// 64 channels and a quarter of the slots, two a CU.  Four blocks of sums a wave instead of eight leave registers for the third
// workgroup, and a tile ends with one round of exchange instead of two; a row read from LDS feeds half the MFMAs.  So it
// pays where a tile is a chain of waits rather than MFMAs.
// Where empty units are left out, us before / now: 565 k rows 7 % set f16 32 -> 64 80 / 65, 256 -> 64 233 / 203, fp32 32 -> 64
// 114 / 89, 64 -> 64 176 / 144, 128 -> 64 276 / 233; 264 k 22 % fp32 64 -> 64 115 / 105; 593 k 25 % f16 128 -> 64 211 / 193; 267 k
// 31 % fp32 64 -> 64 109 / 102, 256 -> 64 354 / 356; nine slots of 822 k rows 0.79.  The third workgroup has to find LDS (297 k
// rows, 378 distinct a tile: 0.95 - 1.04), and there have to be tiles for one and a half rounds of three a CU (1035 tiles
// 0.93 - 1.08, 1130 0.92 - 1.01, 1240 and 1294 0.87 - 0.98, 20 k - 41 k rows 0.91 - 1.08).
// Elsewhere with one chunk of channels: 0.78 - 0.98 on 656 - 9950 tiles, 61 - 73 % set, 2x2x2 tables; with more chunks 0.97 - 1.03.
constexpr int kTgThirdRows = 352;                            // staged rows with which three workgroups fit: 53760 bytes each at 27 slots
constexpr int64_t kTgThirdTiles = 1152;

static bool tile_half_waves(bool f32, int64_t tiles, int cin, bool skip, int max_distinct) {
  if (skip) return tiles > kTgThirdTiles && max_distinct < kTgThirdRows;
  return tiles > kTgPartsGroups && cin <= (f32 ? 32 : 64);
}

// (skip, max_distinct: the shape of the waves, of launches that are not cut up, hangs on them, nothing else)
static TileLaunch tile_launch(bool f32, int64_t tiles, int K, int cin, int cout, bool skip, int max_distinct) {
  TileLaunch t{1, 1, 1, 4, 1, 1, 1};                         // 32 channels
  if (cout % 256 == 0 && tiles * (cout / 256) > 256) t.mb = 2, t.wc = 4, t.ks = 1;
  else if (cout % 96 == 0) t.mb = 3, t.wr = 2, t.ks = 2;
  else if (cout > 64) t.mb = 2, t.wc = 2, t.ks = 2;
  else if (cout > 32 && tile_half_waves(f32, tiles, cin, skip, max_distinct)) t.wc = 2, t.ks = 2;
  else if (cout > 32) t.mb = 2;
  t.gy = (int)cdiv(cout, 32 * t.mb * t.wc);
  const int ncc = (int)cdiv(cin, f32 ? 32 : 64);
  if (tiles > 0 && tiles * t.gy <= kTgPartsGroups) {
    double best = 0.95 * tile_cost(t, f32, tiles, K, ncc, cout, 1, 1);   // (parts have to be worth it)
    for (int sc = 1; sc <= ncc; ++sc) {
      if (sc > 1 && cdiv(ncc, sc) == cdiv(ncc, sc - 1)) continue;        // (no fewer chunks a part)
      for (int sk = 1; sk <= std::min(K, kTgMaxSlotParts) && tiles * t.gy * sc * sk <= 2048; ++sk) {
        if (sk > 1 && cdiv(cdiv(K, sk), t.ks) == cdiv(cdiv(K, sk - 1), t.ks)) continue;   // (no fewer slots a wave)
        const double us = tile_cost(t, f32, tiles, K, ncc, cout, sc, sk);
        if (us < best) best = us, t.sc = sc, t.sk = sk;
      }
    }
  }
  return t;
}

}  // namespace ocnn

using namespace ocnn;

static int64_t tile_packed_bytes(int dtype, int K, int cin, int cout) {
  return align_up(dtype == OCNN_F32 ? (int64_t)K * align_up(cin, 32) * cout * 4 : (int64_t)K * align_up(cin, 64) * cout * 2,
                  256);
}

extern "C" int ocnnx_gather_tile_supported(int dtype, int64_t rows_in, int K, int cin, int cout, int plan_max_distinct) {
  if (dtype < 0 || dtype > 2) return 0;
  if (cin < 32 || cin % 32 != 0 || cout < 32 || cout % 32 != 0 || cin > 2048 || cout > 2048) return 0;
  if (K < 1 || K > 27) return 0;
  if (plan_max_distinct < 0 || plan_max_distinct > kTgCap) return 0;
  if (rows_in < 0 || rows_in * cin * dtype_size(dtype) > 0xfff00000ll) return 0;
  return 1;
}

extern "C" int64_t ocnnx_gather_tile_packed_bytes(int dtype, int K, int cin, int cout) {
  return dtype < 0 || dtype > 2 || K < 1 || cin < 1 || cout < 1 ? 0 : tile_packed_bytes(dtype, K, cin, cout);
}

// (a 2x2x2 table has an entry in every slot of every 32 rows, whatever its occupancy)
extern "C" int ocnnx_gather_tile_ordered(int K, double plan_occupancy) {
  return K != 8 && plan_occupancy >= 0.0 && plan_occupancy <= kTgSkipMaxOccupancy;
}

extern "C" int64_t ocnnx_gather_tile_workspace_bytes(int dtype, int64_t rows_out, int K, int cin, int cout) {
  const TileLaunch t = tile_launch(dtype == OCNN_F32, cdiv(rows_out, kTgRows), K, cin, cout, false, 0);
  const int64_t parts = t.sc * t.sk;
  return tile_packed_bytes(dtype, K, cin, cout) + (parts > 1 ? parts * rows_out * cout * 4 : 0);
}

template <typename T, bool F32> struct TilePass : Pass {
  ocnnx_gather_args a;
  ocnnx_bn bn;
  TileLaunch t;
  bool skip;
  float* partial;
  hipStream_t st;

  TilePass(const ocnnx_gather_args& args, hipStream_t stream) : a(args), bn(args.bn ? *args.bn : ocnnx_bn{}), st(stream) {
    const int dtype = std::is_same<T, f16>::value ? OCNN_F16 : (F32 ? OCNN_F32 : OCNN_BF16);
    skip = ocnnx_gather_tile_ordered(a.K, a.plan_occupancy) != 0;
    t = tile_launch(F32, cdiv(a.rows_out, kTgRows), a.K, a.cin, a.cout, skip, a.plan_max_distinct);
    if (a.split_c > 0 && a.split_k > 0) {
      t.sc = std::min<int>(a.split_c, (int)cdiv(a.cin, F32 ? 32 : 64));
      t.sk = std::min(a.split_k, a.K);
    }
    const int64_t packed = tile_packed_bytes(dtype, a.K, a.cin, a.cout);
    if (packed + (int64_t)t.sc * t.sk * a.rows_out * a.cout * 4 > a.workspace_bytes) t.sc = t.sk = 1;   // (no room for the parts)
    partial = t.sc * t.sk > 1 ? (float*)((char*)a.workspace + packed) : nullptr;
    if (!a.packed) before.add(pack_tile_job(dtype, a.w, a.workspace, a.K, a.cin, a.cout, a.w_transposed, a.reverse_slots));
    if (partial) after.add(tile_parts_job(partial, t.sc * t.sk, a.rows_out, a.cout, a.bias, bn, a.out));
  }

  int main() override {
    typedef typename std::conditional<F32, float, T>::type O;
    const int64_t tiles = cdiv(a.rows_out, kTgRows);
    // few tiles: in launch order, so that they spread over the XCDs
    const int64_t per_xcd = partial ? 0 : cdiv(tiles, 8);
    const dim3 grid((unsigned)(per_xcd > 0 ? per_xcd * 8 : tiles), (unsigned)t.gy, (unsigned)(t.sc * t.sk));
    const uint32_t in_bytes = (uint32_t)(a.rows_in * a.cin * sizeof(O));
    const int rows_alloc = (a.plan_max_distinct + 8) / 8 * 8;
    // LDS: rows, positions, list; at the end the waves' sums
    const int kmax = (a.K + t.sk - 1) / t.sk;
    const size_t lds = std::max<size_t>((size_t)rows_alloc * 132 + (size_t)kmax * kTgRows * 2 + 128,
                                        (size_t)(t.ks == 4 ? 8 : t.ks == 2 ? 2 : 0) * t.wc * t.wr * (4 / t.wr / t.ks) * t.mb * 4096);
#define OCNN_TILE_LAUNCH(MB_, WC_, WR_, KS_, SKIP_)                                                                      \
  hipLaunchKernelGGL((conv_gather_tile_kernel<T, F32, MB_, WC_, WR_, KS_, SKIP_>), grid, dim3(256), lds, st, a.in,       \
                     in_bytes, a.loc, a.uptr, a.urows, a.order, (const T*)(a.packed ? a.packed : a.workspace), a.bias, bn, a.out, partial, a.rows_out, a.K, \
                     a.cin, a.cout, tiles, per_xcd, t.sc, t.sk, rows_alloc)
#define OCNN_TILE_CASE(MB_, WC_, WR_, KS_)                                   \
  if (t.mb == MB_ && t.wc == WC_ && t.wr == WR_ && t.ks == KS_) {            \
    if (skip) OCNN_TILE_LAUNCH(MB_, WC_, WR_, KS_, true);                    \
    else OCNN_TILE_LAUNCH(MB_, WC_, WR_, KS_, false);                        \
  }
    OCNN_TILE_CASE(1, 1, 1, 4) OCNN_TILE_CASE(2, 1, 1, 4) OCNN_TILE_CASE(3, 1, 2, 2) OCNN_TILE_CASE(2, 2, 1, 2)
    OCNN_TILE_CASE(2, 4, 1, 1) OCNN_TILE_CASE(1, 2, 1, 2)
#undef OCNN_TILE_CASE
#undef OCNN_TILE_LAUNCH
    return check_launch("conv_gather_tile");
  }
};

// The pass for these arguments, to be deleted by the caller; none for no rows.
int ocnn::tile_pass(int dtype, const ocnnx_gather_args& a, hipStream_t st, Pass** pass) {
  *pass = nullptr;
  OCNN_REQUIRE(ocnnx_gather_tile_supported(dtype, a.rows_in, a.K, a.cin, a.cout, a.plan_max_distinct),
               "conv_gather_tile: shape not supported");
  OCNN_REQUIRE(a.rows_out >= 0 && a.rows_out < (1ll << 31) && a.plan_total >= 0 && a.plan_total < (1ll << 29),
               "conv_gather_tile: rows out of range");
  if (a.rows_out == 0) return OCNN_OK;
  OCNN_REQUIRE_PTRS("conv_gather_tile", a.loc, a.uptr, a.urows, a.w, a.out, a.workspace);
  OCNN_REQUIRE(a.rows_in == 0 || a.in, "conv_gather_tile: in is NULL");
  if (a.workspace_bytes < (dtype == OCNN_F32 ? (int64_t)a.K * a.cin * a.cout * 4 : (int64_t)a.K * align_up(a.cin, 64) * a.cout * 2)) {
    set_error("conv_gather_tile: workspace too small");
    return OCNN_ERR_WORKSPACE;
  }
  if (dtype == OCNN_F32) *pass = new (std::nothrow) TilePass<bf16, true>(a, st);
  else if (dtype == OCNN_F16) *pass = new (std::nothrow) TilePass<f16, false>(a, st);
  else *pass = new (std::nothrow) TilePass<bf16, false>(a, st);
  OCNN_REQUIRE(*pass, "conv_gather_tile: out of host memory");
  return OCNN_OK;
}

extern "C" int ocnnx_gather_tile_args(int dtype, const ocnnx_gather_args* args, void* stream) {
  OCNN_REQUIRE_PTRS("conv_gather_tile", args);
  Pass* pass = nullptr;
  int rc = tile_pass(dtype, *args, (hipStream_t)stream, &pass);
  if (pass) {
    launch_jobs(dtype, pass->before, (hipStream_t)stream);
    rc = pass->main();
    if (rc == OCNN_OK) launch_jobs(dtype, pass->after, (hipStream_t)stream);
    delete pass;
  }
  return rc == OCNN_OK ? check_launch("conv_gather_tile") : rc;
}

extern "C" int ocnnx_gather_tile(int dtype, const void* in, int64_t rows_in, const uint16_t* loc, const int32_t* uptr,
                                 const int32_t* urows, int plan_max_distinct, int64_t plan_total, double plan_occupancy,
                                 int64_t rows_out, int K, const void* w, int cin, int cout, int w_transposed,
                                 int reverse_slots, const void* bias, const ocnnx_bn* bn_or_null, void* out,
                                 void* workspace, int64_t workspace_bytes, int split_c, int split_k, void* stream) {
  const ocnnx_gather_args args{in, rows_in, loc, uptr, urows, plan_max_distinct, plan_total, plan_occupancy, rows_out, K, w,
                               cin, cout, w_transposed, reverse_slots, bias, bn_or_null, out, workspace, workspace_bytes,
                               split_c, split_k, nullptr, nullptr};
  return ocnnx_gather_tile_args(dtype, &args, stream);
}

// The public entry point: 16-bit wide layers, in one part: its workspace is that of the packed weights, whatever more
// the caller has (the order of the sums does not hang on it).
extern "C" int ocnn_conv_gather_wide_supported(int dtype, int64_t rows_in, int K, int cin, int cout,
                                               int plan_max_distinct) {
  if (dtype != OCNN_F16 && dtype != OCNN_BF16) return 0;
  if (cin < 64 || cout < 96) return 0;
  return ocnnx_gather_tile_supported(dtype, rows_in, K, cin, cout, plan_max_distinct);
}

extern "C" int ocnn_conv_gather_wide(int dtype, const void* in, int64_t rows_in, const uint16_t* loc,
                                     const int32_t* uptr, const int32_t* urows, int plan_max_distinct,
                                     int64_t plan_total, double plan_occupancy, int64_t rows_out, int K,
                                     const void* w, int cin, int cout, int w_transposed, int reverse_slots,
                                     const void* bias, void* out, void* workspace, int64_t workspace_bytes,
                                     void* stream) {
  OCNN_REQUIRE(ocnn_conv_gather_wide_supported(dtype, rows_in, K, cin, cout, plan_max_distinct),
               "conv_gather_wide: shape not supported");
  return ocnnx_gather_tile(dtype, in, rows_in, loc, uptr, urows, plan_max_distinct, plan_total, plan_occupancy, rows_out,
                           K, w, cin, cout, w_transposed, reverse_slots, bias, nullptr, out, workspace,
                           std::min(workspace_bytes, tile_packed_bytes(dtype, K, cin, cout)), 0, 0, stream);
}

// Weight gradient in fp32 on the tile plan of the neighbour table, for multiples of 32 channels, as three products of
// bf16 pieces: x = hi + lo, g = hi + lo, dW = hi hi + hi lo + lo hi, all into one fp32 sum.
//
//   dW[k][a][b] = sum over table rows r of  x[table[r][k]][a] * g[r][b]
//
// The scheme is that of wgrad_planned.hip: a persistent workgroup (4 waves, one per SIMD) owns a block of channel pairs
// and a range of tiles, every wave keeps the sums of its slots in accumulator registers, both operands come from LDS
// by the transposing read, whose per-lane address gathers the rows of x.  Here the rows arrive as fp32 through registers
// and are split into their pieces on the way into LDS, where a row's two pieces take the places of the two 32-channel halves.
//
// What bounds it: the MFMAs' issue and power.  64 -> 64 on 252 k rows (1972 tiles) 137 us = 1.3 PFLOP/s of issued products, 7.3 us
// for a tile of 336 MFMAs a wave; blocks of 32 x 32 (168 MFMAs, 4.6 us) are bound by LDS: an operand read feeds half as many
// MFMAs.  So a workgroup takes 32 channels of x with 64 of g over all slots: four transposing reads for six MFMAs, and x
// and g staged once for the three products.  Before, the pieces were written by a launch of their own and the three products
// were workgroups of the 16-bit kernel with sums each, one read per MFMA, every row staged three times.  With the launches
// around it, us, so / now: 64 -> 64 on 154 k rows 115 / 94, 592 k 376 / 315, 4 k 25.2 / 21.9; 32 -> 32 154 k 54 / 37; 96 -> 96
// 154 k 338 / 207, 30 k 80 / 51; 128 -> 128 154 k 344 / 284; 256 -> 256 51 k 450 / 380; nine slots 64 -> 64 283 k 113 / 84, eight
// 154 / 112.  Wide layers of few slots still go the other way (wp_takes_pieces): nine slots here are twelve slots' worth of MFMAs.
#include <algorithm>
#include <type_traits>

#include "mma.hpp"
#include "wgrad_f32.hpp"

namespace ocnn {

constexpr int kWfRows = 128;   // rows per tile (the plan's tile size)
constexpr int kWfCap = 415;    // staged distinct rows per tile; position 0 is a row of zeros
constexpr int kWfXPiece = (kWfCap + 1) * 32;                 // elements of one piece of the x rows
constexpr int kWfXLoads = (kWfCap + 1) / 32;                 // loads a wave: 8 rows of 128 bytes each
constexpr int kWfLoc = (kWfRows * 27 * 2 + 1023) / 1024 * 512;   // u16 per buffer, whole KiB

// (Not in the kernel template: the arguments of the global->LDS load builtin must not be type-dependent expressions.)
static __device__ __forceinline__ void wf_dma16(__amdgpu_buffer_rsrc_t rs, void* dst, uint32_t off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)dst, 16, off, 0, 0, 0);
}

typedef __attribute__((ext_vector_type(4))) __bf16 wf_b4;

// four fp32 values -> their pieces, 8 bytes each
static __device__ __forceinline__ void wf_split(f32x4 v, bf16* hi_at, bf16* lo_at) {
  wf_b4 hi, lo;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    hi[j] = (bf16)v[j];
    lo[j] = (bf16)(v[j] - (float)hi[j]);
  }
  *(wf_b4*)hi_at = hi;
  *(wf_b4*)lo_at = lo;
}

// A workgroup sums a 32 x CB block (CB = 64 or 32; the last of a row of 64-channel blocks may be half) over the KK slots, or
// one of GROUPS parts of them, of a range of tiles, NS slots a wave.
//
// LDS: rows of 32 channels at a 64-byte pitch (wgrad_planned.hip).  x double-buffered, both pieces.  g has room for one
// tile and the first 16 rows of the next (CB = 64): a step's 16 rows stand in a place of their own, which is free once
// the step's operands have been read, and the next tile's rows come in behind the barrier in front of the last step.
template <int CB, int KK, int GROUPS>
__global__ __launch_bounds__(256, 1) void conv_wgrad_f32_kernel(
    const float* __restrict__ x, const float* __restrict__ g, const uint16_t* __restrict__ loc, uint32_t loc_bytes,
    const int32_t* __restrict__ uptr, const int32_t* __restrict__ urows, uint32_t urows_bytes, int64_t rows, int64_t tiles,
    int64_t tiles_per_split, int64_t run, int workgroups, int ca, int cb, float* __restrict__ partial) {
  int number = (int)xcd_tile(blockIdx.x, gridDim.x >> 3);
  if (number >= workgroups) return;
  const int grp = number % GROUPS;
  number /= GROUPS;
  const int nbb = (cb + CB - 1) / CB, nblocks = nbb * (ca / 32);
  const int block = __builtin_amdgcn_readfirstlane(number % nblocks);
  const int split = __builtin_amdgcn_readfirstlane(number / nblocks);
  const int blk_a = __builtin_amdgcn_readfirstlane(block / nbb), blk_b = block - blk_a * nbb;

  constexpr int HB = CB / 32, NS = (KK + 4 * GROUPS - 1) / (4 * GROUPS);
  constexpr int NU = NS * HB, NM = 3 * NU;                   // sums of 32 x 32 a wave; MFMAs a step
  constexpr int NL = 2 * NS;                                 // rows of x a lane and step
  constexpr int kSlot = 2 * HB * 512;                        // elements of 16 rows of g: [piece][half][16][32]
  constexpr bool kRing = CB == 64;                           // else two whole buffers of g
  constexpr int kSlots = kRing ? 9 : 16;
  constexpr int kGLoads = kRing ? 8 : 4;                     // loads of g a wave and tile

  __shared__ __attribute__((aligned(16))) bf16 s_x0[2 * kWfXPiece];
  __shared__ __attribute__((aligned(16))) bf16 s_x1[2 * kWfXPiece];
  __shared__ __attribute__((aligned(16))) bf16 s_g[kSlots * kSlot];
  __shared__ __attribute__((aligned(16))) uint16_t s_loc0[kWfLoc];
  __shared__ __attribute__((aligned(16))) uint16_t s_loc1[kWfLoc];
  // lists of distinct rows, from entry 4 on; entry 3 stays 0 ("the row before the first", whose values are not kept)
  __shared__ __attribute__((aligned(16))) int32_t s_u0[4 + 512];
  __shared__ __attribute__((aligned(16))) int32_t s_u1[4 + 512];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t t_begin = (int64_t)split * tiles_per_split;
  const int64_t t_end = min(tiles, t_begin + tiles_per_split);
  if (t_begin >= t_end) return;

  // lane (i16, gq): places 8 q + 4 h + i16 / 4 of a 16-row step, channels 16 (gq & 1) + 4 (i16 & 3) ..; step 2u + p has row
  // 32 u + 16 q + 4 (i16 / 4) + 2 p + h there (wgrad_planned.hip)
  const int i16 = lane & 15, gq = lane >> 4, q = lane >> 5, rs = i16 >> 2;
  const uint32_t byte0 = 32u * (gq & 1) + 8u * (i16 & 3);
  const int slot0 = NS * (4 * grp + wave);
  uint32_t lb[NS];                                           // (a wave's slots can end inside its group of NS)
#pragma unroll
  for (int sl = 0; sl < NS; ++sl) lb[sl] = (uint32_t)(min(slot0 + sl, KK - 1) * kWfRows + 16 * q + 4 * rs) * 2u;
  uint32_t gad[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) gad[h] = (uint32_t)(8 * q + 4 * h + rs) * 64u + byte0;

  if (tid == 0) s_u0[3] = s_u1[3] = 0;

  const __amdgpu_buffer_rsrc_t rs_loc = make_rsrc(loc, loc_bytes);
  const __amdgpu_buffer_rsrc_t rs_u = make_rsrc(urows, urows_bytes);
  const __amdgpu_buffer_rsrc_t rs_p = make_rsrc(uptr, (uint32_t)(tiles + 1) * 4u);

  // ---- staging of a tile ----
  // x: load j of a wave brings the 8 positions from 8 wave + 32 j on, a lane 16 bytes of one.  All kWfXLoads of
  // them, branch-free (a list's end is row 0 again and again, which the caches hold).
  const int xp = 8 * wave + (lane >> 3);                     // position of load 0
  const char* x_at = (const char*)x + (int64_t)blk_a * 128 + (lane & 7) * 16;
  const int64_t x_pitch = (int64_t)ca * 4;
  auto load_x = [&](int32_t id) -> f32x4 { return *(const f32x4*)(x_at + (int64_t)id * x_pitch); };
  auto put_x = [&](int j, f32x4 v, bf16* sx) {
    if (j == 0 && xp == 0) v = f32x4{0.f, 0.f, 0.f, 0.f};    // position 0: the row of zeros
    bf16* at = sx + (xp + 32 * j) * 32 + (lane & 7) * 4;
    wf_split(v, at, at + kWfXPiece);
  };
  // g: CB = 64: load j brings 4 rows of step j, CB = 32: 8 rows of step wave / 2 + 2 j
  const int g_row0 = kRing ? 16 * (wave >> 1) + 4 * (lane >> 4) + (wave & 1)
                           : 16 * (wave & 1) + 4 * ((lane >> 3) & 3) + 2 * (wave >> 1) + (lane >> 5);
  const uint32_t g_pitch = (uint32_t)cb * 4u;
  const uint32_t g_off0 = (uint32_t)g_row0 * g_pitch + (uint32_t)(lane & (kRing ? 15 : 7)) * 16u;
  const int g_half = kRing ? (lane & 15) >> 3 : 0;
  auto g_rsrc = [&](int64_t tile) {                          // the rows of a tile, this block's channels
    const int64_t tc = min(tile, tiles - 1);
    const int64_t n = min(rows - tc * kWfRows, (int64_t)kWfRows);
    return make_rsrc(g + tc * kWfRows * cb + blk_b * CB, (uint32_t)n * g_pitch - (uint32_t)blk_b * CB * 4u);
  };
  auto load_g = [&](int j, __amdgpu_buffer_rsrc_t r) -> f32x4 {
    const uint32_t row = (uint32_t)(kRing ? 32 * (j >> 1) + 2 * (j & 1) : 32 * j);
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, g_off0 + row * g_pitch, 0, 0));
  };
  auto g_place = [&](int buffer, int s) -> bf16* {           // of the 16 rows of step s
    return s_g + (kRing ? (s == 0 ? buffer : s + 1) : 8 * buffer + s) * kSlot;
  };
  auto put_g = [&](int j, f32x4 v, int buffer) {
    bf16* at;
    if constexpr (kRing) at = g_place(buffer, j) + (4 * wave + (lane >> 4)) * 32;
    else at = g_place(buffer, 0) + ((wave + 4 * j) >> 1) * kSlot + (8 * (wave & 1) + (lane >> 3)) * 32;
    at += g_half * 512 + (lane & 7) * 4;
    wf_split(v, at, at + HB * 512);
  };
  auto stage_loc = [&](int64_t tile, uint16_t* sl) {
    constexpr int chunks = (kWfRows * KK * 2 + 1023) >> 10;
    const uint32_t off = (uint32_t)(min(tile, tiles - 1) * kWfRows * KK * 2);
#pragma unroll
    for (int t = 0; t < (chunks + 3) / 4; ++t) {
      const int c = min(wave + 4 * t, chunks - 1);           // (a spare wave repeats the last chunk)
      wf_dma16(rs_loc, (char*)sl + c * 1024, off + (uint32_t)c * 1024u + lane * 16u);
    }
  };
  auto stage_list = [&](int32_t first, int32_t len, int32_t* su) {
    const int e = wave * 256 + lane * 4;
    if (wave < 2) wf_dma16(rs_u, su + 4 + wave * 256, e < len ? (uint32_t)(first + e) * 4u : 0xffffff00u);
  };

  f32x16 acc[NS][HB];

  struct Ops {
    u32x2 a[NS][2][2];    // [slot][piece][rows 0-3 / 4-7 of the lane's 8]
    u32x2 b[HB][2][2];
  } ops[2];
  u32x2 pv[NS];          // positions of the lane's two rows in an even step and the one behind it

  auto pf_loc = [&](int slot, const uint16_t* sl, int sn) {  // (sn even)
    pv[slot] = *(const u32x2*)((const char*)sl + lb[slot] + (uint32_t)(sn * 32));
  };
  auto pf_g = [&](int j, const bf16* place, Ops& on) {       // j = 4 half + 2 piece + h
    const int h = j & 1, p = (j >> 1) & 1, bh = j >> 2;
    on.b[bh][p][h] = Mma<bf16>::read_tr((const bf16*)((const char*)place + gad[h] + (uint32_t)((p * HB + bh) * 1024)));
  };
  auto pf_x = [&](int j, const bf16* sx, int sn, Ops& on) {  // j = 2 slot + h
    const uint32_t two = pv[j >> 1][sn & 1];
    const char* at = (const char*)sx + ((j & 1 ? two >> 16 : two & 0xffffu) << 6) + byte0;
    on.a[j >> 1][0][j & 1] = Mma<bf16>::read_tr((const bf16*)at);
    on.a[j >> 1][1][j & 1] = Mma<bf16>::read_tr((const bf16*)(at + kWfXPiece * 2));
  };
  auto mm = [&](int m, const Ops& oc) {                      // hi hi of every unit, then hi lo, then lo hi
    const int p = m / NU, u = m % NU / HB, bh = m % HB, pa = p == 2, pb = p == 1;
    const u32x4 av = u32x4{oc.a[u][pa][0][0], oc.a[u][pa][0][1], oc.a[u][pa][1][0], oc.a[u][pa][1][1]};
    const u32x4 bv = u32x4{oc.b[bh][pb][0][0], oc.b[bh][pb][0][1], oc.b[bh][pb][1][0], oc.b[bh][pb][1][1]};
    acc[u][bh] = Mma32<bf16>::run(av, bv, acc[u][bh]);
  };
  // One step: the MFMAs of 16 rows on `oc`; between them the operands of the next one (positions and g with the first
  // MFMA, x from MFMA XS on) into `on`, and what between(m) does.
  constexpr int XS = NM > 4 ? 3 : 1, XP = (NL + NM - XS - 1) / (NM - XS);
  auto step = [&](const Ops& oc, Ops& on, const bf16* sx, const bf16* gp, const uint16_t* sl, int sn, auto between) {
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      mm(m, oc);
      if (m == 0) {
#pragma unroll
        for (int t = 0; t < NS; ++t)
          if (sn % 2 == 0) pf_loc(t, sl, sn);
#pragma unroll
        for (int t = 0; t < 4 * HB; ++t) pf_g(t, gp, on);
      }
      if (m >= XS) {
#pragma unroll
        for (int t = (m - XS) * XP; t < (m - XS + 1) * XP && t < NL; ++t) pf_x(t, sx, sn, on);
      }
      between(m);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- prologue: first list, first tile, second list ----
  int32_t p_nxt = uptr[t_begin + 1];
  int32_t p_nx2 = uptr[min(t_begin + 2, tiles)];
  int32_t p_nx3 = uptr[min(t_begin + 3, tiles)];
  {
    const int32_t p_cur = uptr[t_begin];
    stage_list(p_cur, p_nxt - p_cur, s_u0);
    stage_loc(t_begin, s_loc0);
    const __amdgpu_buffer_rsrc_t r = g_rsrc(t_begin);
    f32x4 gv[kGLoads], v[kWfXLoads];
#pragma unroll
    for (int j = 0; j < kGLoads; ++j) gv[j] = load_g(j, r);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kWfXLoads; ++j) v[j] = load_x(s_u0[4 + xp + 32 * j - 1]);
    stage_list(p_nxt, p_nx2 - p_nxt, s_u1);
#pragma unroll
    for (int j = 0; j < kGLoads; ++j) put_g(j, gv[j], 0);
#pragma unroll
    for (int j = 0; j < kWfXLoads; ++j) put_x(j, v[j], s_x0);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NS; ++t) pf_loc(t, s_loc0, 0);
#pragma unroll
    for (int t = 0; t < 4 * HB; ++t) pf_g(t, g_place(0, 0), ops[0]);
#pragma unroll
    for (int t = 0; t < NL; ++t) pf_x(t, s_x0, 0, ops[0]);
  }

  // One tile out of buffer B; the next tile -> the other buffer meanwhile: x loads in steps 0 - 3, put two steps later.  g of the next tile:
  //   CB = 64, one place a step for all tiles, two by turns for step 0: the rows of step 0 are loaded in step 0 and put in step
  //   2, into the place whose last readers were in step 7 two tiles ago; the others are loaded in steps 4 and 5 and put in
  //   step 7, behind the barrier that follows step 6, in which this tile's last rows of g are read.
  //   CB = 32, two whole buffers: loaded in step 4, put in step 6, in front of that barrier: the other buffer's last
  //   reader was step 6 of the tile before, and two barriers lie between.
  // Step 7 reads the next tile's first operands: what the barrier in front of it has seen put, in either case.
  auto tile_body = [&](auto BC, int64_t tile) {
    constexpr int B = decltype(BC)::value;
    const bf16* sx = B ? s_x1 : s_x0;
    bf16* nx = B ? s_x0 : s_x1;
    const uint16_t* sl = B ? s_loc1 : s_loc0;
    uint16_t* nl = B ? s_loc0 : s_loc1;
    const int32_t* su = (B ? s_u0 : s_u1) + 4;
    const int32_t l_first = p_nx2, l_len = p_nx3 - p_nx2;
    const __amdgpu_buffer_rsrc_t gr = g_rsrc(tile + 1);
    // list boundary four tiles ahead, as a vector load: a scalar load would share its counter
    // with the LDS reads and force them to drain where it is used
    const uint32_t p_raw = __builtin_amdgcn_raw_buffer_load_b32(rs_p, (uint32_t)min(tile + 4, tiles) * 4u, 0, 0);
    p_nxt = p_nx2;
    p_nx2 = p_nx3;
    f32x4 v[kWfXLoads], gv[kGLoads];
    int32_t ids[kWfXLoads];
    auto run = [&](auto SC) {
      constexpr int s = decltype(SC)::value;
      constexpr int x0 = 3 * s, xn = s < 3 ? 3 : (s == 3 ? kWfXLoads - 9 : 0);           // x loads of this step
      constexpr int w0 = 3 * (s - 2), wn = s < 2 || s > 5 ? 0 : (s < 5 ? 3 : kWfXLoads - 9);
      constexpr int g0 = kRing ? (s == 0 ? 0 : s == 4 ? 1 : 5) : 0;
      constexpr int gn = kRing ? (s == 0 ? 1 : s == 4 ? 4 : s == 5 ? 3 : 0) : (s == 4 ? 4 : 0);
      auto at = [](int i, int n) { return (i * (NM - 2)) / (n > 0 ? n : 1) + 1 < NM ? (i * (NM - 2)) / (n > 0 ? n : 1) + 1 : NM - 1; };
      step(ops[s & 1], ops[(s + 1) & 1], s < 7 ? sx : nx, s < 7 ? g_place(B, s + 1) : g_place(1 - B, 0), s < 7 ? sl : nl,
           s < 7 ? s + 1 : 0, [&](int m) {
             if (m == 0) {
               if (s == 0) stage_loc(tile + 1, nl), stage_list(l_first, l_len, B ? s_u1 : s_u0);
#pragma unroll
               for (int i = 0; i < xn; ++i) ids[x0 + i] = su[xp + 32 * (x0 + i) - 1];
             }
#pragma unroll
             for (int i = 0; i < wn; ++i)
               if (m == at(i, wn)) put_x(w0 + i, v[w0 + i], nx);
#pragma unroll
             for (int i = 0; i < xn; ++i)
               if (m == at(i, xn)) v[x0 + i] = load_x(ids[x0 + i]);
#pragma unroll
             for (int i = 0; i < gn; ++i)
               if (m == at(i, gn)) gv[g0 + i] = load_g(g0 + i, gr);
             if (kRing) {
               if (s == 2 && m == NM - 1) put_g(0, gv[0], 1 - B);
               if (s == 7) {
#pragma unroll
                 for (int i = 1; i < kGLoads; ++i)
                   if (m == at(i - 1, kGLoads)) put_g(i, gv[i], 1 - B);
               }
             } else if (s == 6) {
#pragma unroll
               for (int i = 0; i < kGLoads; ++i)
                 if (m == at(i, kGLoads)) put_g(i, gv[i], 1 - B);
             }
           });
    };
    run(std::integral_constant<int, 0>{});
    run(std::integral_constant<int, 1>{});
    run(std::integral_constant<int, 2>{});
    run(std::integral_constant<int, 3>{});
    run(std::integral_constant<int, 4>{});
    run(std::integral_constant<int, 5>{});
    run(std::integral_constant<int, 6>{});
    // The next tile has landed, and every wave has read this tile's rows of g
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    p_nx3 = __builtin_amdgcn_readfirstlane((int32_t)p_raw);
    run(std::integral_constant<int, 7>{});
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };

  // ---- sums of every `run` tiles -> partial[tile / run][slot][a][b] ----
  const uint32_t pitch = (uint32_t)cb * 4u;
  const uint32_t at = (uint32_t)(4 * q) * pitch + (uint32_t)(lane & 31) * 4u;
  for (int64_t first = t_begin; first < t_end; first += run) {
    const int64_t last = min(first + run, t_end);
#pragma unroll
    for (int u = 0; u < NS; ++u)
#pragma unroll
      for (int bh = 0; bh < HB; ++bh)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[u][bh][r] = 0.f;
    for (int64_t tile = first; tile < last; tile += 2) {
      tile_body(std::integral_constant<int, 0>{}, tile);
      if (tile + 1 < last) tile_body(std::integral_constant<int, 1>{}, tile + 1);
    }
    const uint32_t sums = (uint32_t)KK * ca * pitch;
    const __amdgpu_buffer_rsrc_t rs_out = make_rsrc((char*)partial + (first / run) * (int64_t)sums, sums);
    const uint32_t block_at = (uint32_t)(blk_a * 32) * pitch + (uint32_t)blk_b * (CB * 4u);
#pragma unroll
    for (int u = 0; u < NS; ++u) {
      const int slot = slot0 + u;
      if (slot >= KK) continue;
#pragma unroll
      for (int bh = 0; bh < HB; ++bh) {
        // (a half block at the end of the channels: what the loads brought in beyond a row only reached these sums)
        if (blk_b * CB + 32 * bh >= cb) continue;
#pragma unroll
        for (int r = 0; r < 16; ++r)
          __builtin_amdgcn_raw_buffer_store_b32(
              __float_as_uint(acc[u][bh][r]), rs_out, at,
              block_at + ((uint32_t)slot * ca + (uint32_t)(8 * (r >> 2) + (r & 3))) * pitch + bh * 128u, 0);
      }
    }
  }
}

// channels of g a workgroup: three blocks of 32 for 96, where the second block of 64 would be half empty
static int wf_block(int cb) { return cb == 32 || cb == 96 ? 32 : 64; }

// workgroups of one range of tiles, the slots in one part or in two
static int wf_range_workgroups(int ca, int cb, int groups) { return groups * (ca / 32) * (int)cdiv(cb, wf_block(cb)); }

// What a workgroup takes for a tile, in us, and besides (lists and the first tile, the sums), what a byte of sums takes to be
// written and read; the ranges for the least of it, as in wgrad_planned.hip.  27 slots in two parts are 8 slots a wave's worth
// of MFMAs for 7 and the staging twice, for half the time of a tile: launches of few tiles.
constexpr double kWfFixedUs = 9.0, kWfSumUs = 5.6e-7;
static double wf_tile_us(int K, int cb, int groups) {
  if (K < 27) return wf_block(cb) == 64 ? 3.5 : 2.2;
  return wf_block(cb) == 64 ? (groups == 1 ? 7.3 : 5.0) : (groups == 1 ? 4.6 : 3.3);
}

// Tiles whose products go into one set of accumulators at most.  An MFMA rounds its sums more coarsely the further they have
// grown, and the small products round them as often as the large ones.  From float64, 1.24 M rows of 96 channels: over 230
// tiles 6.0e-6, 64 channels over 77 4.9e-6, over 20 4.5e-6 (three sets of sums over 230 tiles 4.6e-6), of which 4.4e-6 are the
// pieces'.  Blocks of 32 have half the sums to write.
static int64_t wf_run(int cb) { return wf_block(cb) == 64 ? 24 : 16; }

static WfSplit wf_split_launch(int64_t tiles, int K, int ca, int cb, int n_cu) {
  const int cu_xcd = std::max(1, n_cu / 8);
  const double sums = (double)K * ca * cb * 4 * kWfSumUs;
  tiles = std::max<int64_t>(tiles, 1);
  WfSplit best{tiles, tiles, 1, tiles, 1};
  double least = 1e30;
  for (int groups = 1; groups <= (K == 27 ? 2 : 1); ++groups) {
    const int wgs = wf_range_workgroups(ca, cb, groups);
    const int64_t most = std::min(256, std::max(8, n_cu / wgs)), sets_at = wf_run(cb);
    const double tile_us = wf_tile_us(K, cb, groups);
    int64_t s = 1;
    for (bool more = true; more && s <= most;) {             // (the fewest ranges of as many tiles; then of fewer tiles)
      int64_t per = std::max<int64_t>(1, cdiv(tiles, s));
      more = per > 1;
      if (more) s = cdiv(tiles, per - 1);
      // (several sets a range: of an even number of tiles each, the buffers take turns)
      const int64_t sets = cdiv(per, sets_at), run = sets > 1 ? align_up(cdiv(per, sets), 2) : per;
      if (sets > 1) per = run * cdiv(per, run);
      const int64_t used = cdiv(tiles, per);
      const double us = (double)cdiv(cdiv(used * wgs, 8), cu_xcd) * ((double)per * tile_us + kWfFixedUs) +
                        (double)(sets > 1 ? cdiv(tiles, run) : used) * sums;
      if (us < least) least = us, best = WfSplit{per, run, groups, tiles, cdiv(tiles, run)};
    }
  }
  return best;
}

// The sets of sums grow with the rows: 27 slots of 512 x 512 channels 2.4 GB for every 256 k rows.  Beyond this many bytes the tiles
// are taken in launches of as many as fit, with a reduction into one set behind each.  That costs nothing, the sets of a launch
// are still in the memory-side cache when they are added: 512 -> 512 on 300 k rows 2.7 GB and 9.71 ms in one launch, 0.76 GB
// and 9.54 ms in several, 1024 -> 1024 on 60 k 2.3 GB and 7.83 ms, 0.86 and 7.35, nine slots on 100 k 1.2 and 6.88, 0.76 and 6.55.
// (The sums of a range added to by its workgroup, a read for every further set: the kernel's registers do not hold that beside the
// accumulators, 64 -> 64 on 252 k rows 139 -> 165 us.)
constexpr int64_t kWfSumsBytes = 1ll << 30;
WfSplit wf_split_tiles(int64_t tiles, int K, int ca, int cb, int n_cu) {
  WfSplit s = wf_split_launch(tiles, K, ca, cb, n_cu);
  const int64_t room = kWfSumsBytes / ((int64_t)K * ca * cb * 4), most = std::max<int64_t>(1, room - 2);
  if (s.sets <= std::max<int64_t>(1, room)) return s;
  for (int64_t n = cdiv(tiles, most * wf_run(cb)); s.sets > most && s.launch > 1; n += cdiv(n, 4))
    s = wf_split_launch(cdiv(tiles, n), K, ca, cb, n_cu);
  return s;
}

template <int CB, int KK, int GROUPS> static void launch_wf(const WfArgs& a, hipStream_t st) {
  const int64_t tiles = cdiv(a.rows, kWfRows);
  const int wgs = (int)cdiv(tiles, a.split.per) * wf_range_workgroups(a.ca, a.cb, GROUPS);
  const float* x = a.rows_x > 0 ? a.x : a.partial;           // (no rows: position 0 is loaded from somewhere, and not kept)
  hipLaunchKernelGGL((conv_wgrad_f32_kernel<CB, KK, GROUPS>), dim3(8 * (unsigned)cdiv(wgs, 8)), dim3(256), 0, st, x, a.g, a.loc,
                     (uint32_t)(tiles * kWfRows * KK * 2), a.uptr, a.urows, (uint32_t)(a.plan_total * 4), a.rows, tiles, a.split.per,
                     a.split.run, wgs, a.ca, a.cb, a.partial);
}

void launch_wgrad_f32(const WfArgs& a, hipStream_t st) {
#define OCNN_WF_LAUNCH(KK_, GROUPS_) (wf_block(a.cb) == 64 ? launch_wf<64, KK_, GROUPS_>(a, st) : launch_wf<32, KK_, GROUPS_>(a, st))
  if (a.split.groups == 2) OCNN_WF_LAUNCH(27, 2);
  else if (a.K == 27) OCNN_WF_LAUNCH(27, 1);
  else if (a.K == 9) OCNN_WF_LAUNCH(9, 1);
  else if (a.K == 8) OCNN_WF_LAUNCH(8, 1);
  else OCNN_WF_LAUNCH(3, 1);
#undef OCNN_WF_LAUNCH
}

}  // namespace ocnn

// Weight gradient on the tile plan of the neighbour table, for multiples of 32 channels: 32 x 32, 32 x 64 blocks
// where x has 32 channels, 64 x 64 blocks otherwise.
//
//   dW[k][a][b] = sum over table rows r of  x[table[r][k]][a] * g[r][b]
//
// Per 128-row tile the distinct x rows (through the plan), the g rows and the
// table positions are staged ONCE in LDS with asynchronous global->LDS loads,
// double buffered, so the loads of tile i + 1 run under the MFMAs of tile i.  A
// persistent workgroup (4 waves, one per SIMD) owns a range of tiles and a group
// of kernel slots; each wave keeps the 64 x 64 (or 32 x 64) fp32 sums of its slots
// in accumulator registers for the whole range (v_mfma_f32_32x32x16, M = x
// channels, N = g channels, reduction over 16 rows per instruction).  Both
// operands are read with the transposing LDS load, whose per-lane address does
// the gather of the x rows for free.  Per-range sums go to `partial` and are
// added in range order by a second kernel: no atomics, fixed summation order.
#include <algorithm>
#include <new>
#include <type_traits>

#include "jobs.hpp"
#include "mma.hpp"
#include "reduce.hpp"
#include "wgrad_f32.hpp"

namespace ocnn {

constexpr int kWpRows = 128;   // rows per tile (the plan's tile size)
constexpr int kWpCap = 415;    // staged distinct rows per tile: with the zero row, 26 groups of 16
constexpr int kWpLoc = (kWpRows * 27 * 2 + 1023) / 1024 * 512;   // u16 per buffer, whole KiB
constexpr int kWpCapTwo = 367;   // ... with which two workgroups of 32 x 32 blocks share a CU
constexpr int kWpGHalf = kWpRows * 32;

struct WpOps {
  u32x2 a[7][2];    // [unit][rows 0-3 / 4-7 of the lane's 8]
  u32x2 b[2][2];    // [g-channel half][rows]
};

// What the staging pieces of a tile need.  (Not a local class of the kernel template: the
// arguments of the global->LDS load builtin must not be type-dependent expressions.)
struct WpStage {
  uint32_t g_off;       // byte offset of the tile's first g row
  uint32_t loc_off;     // byte offset of the tile's table positions
  uint32_t list_off;    // byte offset of the list of the tile after it, per lane (or out of range)
  int groups;           // number of 16-row groups of distinct x rows of the tile
  const int32_t* su;    // list of this tile's distinct rows (LDS)
  int32_t* su_out;      // where the next list goes (LDS)
  char* sx;             // destination buffers (LDS)
  char* sg;
  char* sl;
};

// A workgroup sums a CA x CB block (64 x 64, 32 x 64 or 32 x 32) of the channel pairs of one range of tiles, one
// of them when the layer has more channels (BLK; C = 64).  NFULL slots per wave with all
// CA x channels, NHALF (0/1, CA = 64 only) slot shared by two waves (one x-channel half each);
// GROUPS workgroups split the K slots.  The workgroups of a range (slot groups, blocks) are neighbours in
// the numbering, and each XCD takes an eighth of all of them in a row: they stage the same rows, and every
// XCD has the same number however few ranges there are.
//
// LDS layout: the two 32-channel halves of the staged rows live in separate arrays
// of 64-byte rows.  A transposing read of a 16-lane group touches 4 rows x 32 B, a
// half wave 4 rows x 64 B; at a 64-byte pitch four consecutive positions cover all
// 64 banks, and the second half is the first plus a constant.
//
// CAP: distinct rows of a tile at most.  A wave of the 32 x 32 layer has 212 registers, and with 367 rows two workgroups find
// room in a CU's LDS, which hides the waits of one behind the other: us, f16, one / two a CU: 7.57 M rows 468 / 425, 4.74 M 295 / 276, 1.13 M
// (7 % set) 80.7 / 74, 947 k 65 / 59.  Where there are
// ranges for one a CU only (wp_places) this form is ahead by its smaller buffers: 120 k 23.8 / 22.8, 330 k 35.9 / 34.2.
//
// 32 channels of x: blocks of 32 x 64 have as many sums over all 27 slots as 64 x 64 over half of them, so one
// workgroup stages a range's rows for all slots: 32 -> 64 on 1.06 M rows (61 % set) 119 us, in half-empty 64 x 64 blocks of two
// slot groups 201.
template <typename T, int CA, int CB, int KK, int NFULL, int NHALF, int GROUPS, bool BLK, int CAP, bool PIECES>
__global__ __launch_bounds__(256, CAP < kWpCap ? 2 : 1) void conv_wgrad_planned_kernel(
    const T* __restrict__ x, uint32_t x_bytes, const T* __restrict__ g, uint32_t g_bytes,
    const uint16_t* __restrict__ loc, uint32_t loc_bytes, const int32_t* __restrict__ uptr,
    const int32_t* __restrict__ urows, uint32_t urows_bytes, int64_t tiles,
    int64_t tiles_per_split, int workgroups, int ca, int cb, float* __restrict__ partial, const T* __restrict__ x_lo,
    const T* __restrict__ g_lo, int64_t set) {
  int number = (int)xcd_tile(blockIdx.x, gridDim.x >> 3);
  if (number >= workgroups) return;
  const int grp = number % GROUPS;
  number /= GROUPS;
  // a block of a wider layer (channel counts are multiples of 32: the last block may be half)
  const int nbb = BLK ? (cb + CB - 1) / CB : 1, nblocks = BLK ? nbb * ((ca + CA - 1) / CA) : 1;
  const int block = __builtin_amdgcn_readfirstlane(number % nblocks);
  const int split = __builtin_amdgcn_readfirstlane(number / nblocks);
  // PIECES: fp32 data as bf16 pieces: hi hi, hi lo, lo hi, each with sums of its own.  (A product's number is a grid
  // index of its own: out of a division it made the pointers, and every staging load, vectors.)
  if constexpr (PIECES) {
    if (blockIdx.y == 1) g = g_lo;
    if (blockIdx.y == 2) x = x_lo;
    partial += blockIdx.y * set;
  }
  constexpr int HA = CA / 32, HB = CB / 32;   // 32-channel halves of a row of x, of g
  constexpr int NU = HA * NFULL + NHALF;      // 32 x CB accumulator units per wave
  constexpr int NS = NFULL + NHALF;           // distinct slots per wave
  constexpr int SPG = 4 * NFULL + 2 * NHALF;  // slots per group
  constexpr int NL = 2 * NS;                  // rows of x per lane and step
  constexpr int NM = HB * NU;                 // MFMAs per step
  constexpr int kWpXHalf = (CAP + 1) * 32;    // elements of one channel half of the x rows (+ zero row)
  constexpr int XH = kWpXHalf * 2, GH = kWpGHalf * 2;   // byte offsets of the second halves
  // CA = 64: MFMAs between the position reads and their use
  constexpr int PF0 = HA == 1 ? 1 : ((NM - NL) < 4 ? (NM - NL) : 4);
  constexpr int IP = (NS + 4 + PF0 - 1) / PF0;
  // CA = 32: positions and g with the first MFMA, the x reads XP per MFMA from MFMA XS on
  constexpr int XS = NM > 2 ? 2 : NM - 1;
  constexpr int XP = (NL + (NM - XS) - 1) / (NM - XS);
  static_assert((HA == 1 || HA == 2) && HB >= HA && HB <= 2 && NU <= 7 && PF0 >= 1 && (HA == 2 || NHALF == 0), "unit layout");

  // one array per buffer, so that the compiler can tell the buffer being filled
  // from the one being read
  __shared__ __attribute__((aligned(16))) T s_x0[HA * kWpXHalf];
  __shared__ __attribute__((aligned(16))) T s_x1[HA * kWpXHalf];
  __shared__ __attribute__((aligned(16))) T s_g0[HB * kWpGHalf];
  __shared__ __attribute__((aligned(16))) T s_g1[HB * kWpGHalf];
  __shared__ __attribute__((aligned(16))) uint16_t s_loc0[kWpLoc];
  __shared__ __attribute__((aligned(16))) uint16_t s_loc1[kWpLoc];
  // lists of distinct rows, from entry 4 on; entry 3 stays -1 ("the row before the first")
  constexpr int kList = CAP < kWpCap ? 384 : 512;
  __shared__ __attribute__((aligned(16))) int32_t s_u0[4 + kList];
  __shared__ __attribute__((aligned(16))) int32_t s_u1[4 + kList];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t t_begin = (int64_t)split * tiles_per_split;
  const int64_t t_end = min(tiles, t_begin + tiles_per_split);
  if (t_begin >= t_end) return;

  const int k0 = grp * SPG;
  const int slotF = k0 + NFULL * wave;                    // first full slot of this wave
  const int slotH = k0 + 4 * NFULL + (wave >> 1);         // the shared slot
  const int slotF_rd = min(slotF, KK - (NFULL > 0 ? NFULL : 1));   // padded slots read a valid column
  const int slotH_rd = min(slotH, KK - 1);
  const uint32_t ahH = (uint32_t)(wave & 1) * (uint32_t)XH;        // this wave's half of the shared slot

  // lane (i16, gq): places 8 q + 4 h + i16 / 4 of a 16-row step, channels 16 (gq & 1) + 4 (i16 & 3) ..
  // Steps 2u and 2u + 1 share 32 rows of the tile: step 2u + p has row 32 u + 16 q + 4 (i16 / 4) + 2 p + h at that place, so
  // that the positions of a lane's rows in both steps are eight consecutive bytes.  (The g rows are staged in that order.)
  const int i16 = lane & 15, gq = lane >> 4, q = lane >> 5;
  const int rs = i16 >> 2;
  const uint32_t byte0 = 32u * (gq & 1) + 8u * (i16 & 3);
  const uint32_t lbF = (uint32_t)(slotF_rd * kWpRows + 16 * q + 4 * rs) * 2u;   // [slot][row] positions, 2 B each
  const uint32_t lbH = (uint32_t)(slotH_rd * kWpRows + 16 * q + 4 * rs) * 2u;
  // CA = 32: a wave's slots can end inside its group of NFULL (K = 27: slots 21..27), so
  // every slot clamps on its own
  uint32_t lbS[HA == 1 ? NFULL : 1];
  if constexpr (HA == 1) {
#pragma unroll
    for (int sl = 0; sl < NFULL; ++sl)
      lbS[sl] = (uint32_t)(min(slotF + sl, KK - 1) * kWpRows + 16 * q + 4 * rs) * 2u;
  }
  uint32_t gad[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) gad[h] = (uint32_t)(8 * q + 4 * h + rs) * 64u + byte0;

  if (tid == 0) s_u0[3] = s_u1[3] = -1;     // position 0 is the zero row: it is staged from out of range

  const __amdgpu_buffer_rsrc_t rs_x = make_rsrc(x, x_bytes);
  const __amdgpu_buffer_rsrc_t rs_g = make_rsrc(g, g_bytes);
  const __amdgpu_buffer_rsrc_t rs_loc = make_rsrc(loc, loc_bytes);
  const __amdgpu_buffer_rsrc_t rs_u = make_rsrc(urows, urows_bytes);
  const __amdgpu_buffer_rsrc_t rs_p = make_rsrc(uptr, (uint32_t)(tiles + 1) * 4u);

  // ---- staging of one tile, cut into per-wave pieces `t` (one load instruction each, 1 KiB):
  //   NG pieces  g rows: 16 rows of one channel half
  //   2 pieces   table positions
  //   NX pieces  x rows: 16 distinct rows (ids in su) of one channel half
  //   1 piece    the list of distinct rows of the tile after (waves 0 and 1)
  // (CA = CB = 64: 4 + 2 + 13 + 1, a wave takes one half of every second 16-row group;
  //  32: 2 + 2 + 7 + 1, a wave takes every fourth group.)
  // The pieces are branch-free: whatever lies past the end of a list, of the table or of
  // the tile range is an out-of-range offset (loads zeros) or row 0.  A wave has one
  // instruction stream for the MFMAs and everything else, so each instruction saved here
  // is MFMA issue time won.
  constexpr int NG = 2 * HB, GST = 4 / HA, GSG = 4 / HB;   // g pieces; 16-row groups between a wave's pieces of x, of g
  constexpr int NX = ((CAP + 16) / 16 + GST - 1) / GST;
  constexpr int tL = NG, tX = NG + 2, tU = NG + 2 + NX, kPieces = tU + 1;
  static_assert(kPieces <= 20 && (CAP + 1) % 16 == 0, "five steps of four pieces stage a tile");
  constexpr int RSH = 5 + HA, RSG = 5 + HB;                // log2 of the bytes of a CA-channel row, of a CB-channel row
  // a block of a wider layer: rows of ca (cb) channels, this block's start at xb (gb)
  const int blk_a = __builtin_amdgcn_readfirstlane(block / nbb), blk_b = block - blk_a * nbb;
  const uint32_t x_pitch = BLK ? (uint32_t)ca * 2u : (1u << RSH), g_pitch = BLK ? (uint32_t)cb * 2u : (1u << RSG);
  const uint32_t xb = (uint32_t)blk_a << RSH, gb = (uint32_t)blk_b << RSG;
  const int st_half = HA == 2 ? (wave & 1) : 0, st_g16 = HA == 2 ? (wave >> 1) : wave;
  const int sg_half = HB == 2 ? (wave & 1) : 0, sg_g16 = HB == 2 ? (wave >> 1) : wave;
  const uint32_t st_xc = (uint32_t)st_half * 64u + (uint32_t)(lane & 3) * 16u;   // byte within a row
  const int st_pos = st_g16 * 16 + (lane >> 2);            // position / row of piece 0; piece j: + 16 GST j
  const uint32_t sg_c = (uint32_t)sg_half * 64u + (uint32_t)(lane & 3) * 16u;
  const uint32_t sg_pos = (uint32_t)(32 * (sg_g16 >> 1) + 2 * (sg_g16 & 1) + 16 * (lane >> 5) + 4 * ((lane >> 2) & 3) + ((lane >> 4) & 1));
  const uint32_t st_gc = (BLK ? sg_pos * g_pitch + gb : (sg_pos << RSG)) + sg_c;
  const uint32_t st_gstep = BLK ? 16u * GSG * g_pitch : 4096u;   // 16 GSG rows further
  auto make_stage = [&](int64_t tile, int U, int32_t list_first, int32_t list_len, const int32_t* su,
                        int32_t* su_out, T* sx, T* sg, uint16_t* sl) {
    WpStage st;
    const int64_t tc = min(tile, tiles - 1);              // past the range: any valid tile
    st.g_off = BLK ? (uint32_t)(tc * kWpRows) * g_pitch : (uint32_t)(tc * kWpRows) << RSG;
    st.loc_off = (uint32_t)(tc * kWpRows * KK * 2);
    const int e = wave * 256 + lane * 4;                   // the four list entries this lane brings in
    st.list_off = e < list_len ? (uint32_t)(list_first + e) * 4u : 0xffffff00u;
    st.groups = (U + 16) >> 4;                             // positions 0..U
    st.su = su; st.su_out = su_out; st.sx = (char*)sx; st.sg = (char*)sg; st.sl = (char*)sl;
    return st;
  };
  auto stage_id = [&](int t, const WpStage& st) -> int32_t {     // row id a lane needs for piece t
    return (t >= tX && t < tU) ? st.su[st_pos + 16 * GST * (t - tX) - 1] : 0;   // position p holds list entry p - 1
  };
  auto stage_piece = [&](int t, const WpStage& st, int32_t id) {
    if (t < NG) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rs_g, (lds_ptr_t)(st.sg + (sg_half * kWpGHalf + (sg_g16 + GSG * t) * 512) * 2), 16,
          st.g_off + st_gc + (uint32_t)t * st_gstep, 0, 0, 0);
    } else if (t < tX) {
      constexpr int nchunk = (kWpRows * KK * 2 + 1023) >> 10;
      if (4 * (t - tL) < nchunk) {
        const int c = min(wave + 4 * (t - tL), nchunk - 1);     // a spare wave repeats the last chunk
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_loc, (lds_ptr_t)(st.sl + c * 1024), 16,
                                                 st.loc_off + (uint32_t)c * 1024u + lane * 16u, 0, 0, 0);
      }
    } else if (t < tU) {
      if ((st_g16 + GST * (t - tX)) < st.groups)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rs_x, (lds_ptr_t)(st.sx + (st_half * kWpXHalf + (st_g16 + GST * (t - tX)) * 512) * 2), 16,
          BLK ? (uint32_t)id * x_pitch + (xb + st_xc) : (((uint32_t)id << RSH) | st_xc), 0, 0, 0);
    } else if (wave < kList / 256 || (kList % 256 != 0 && wave * 256 + lane * 4 < kList)) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_u, (lds_ptr_t)(st.su_out + wave * 256), 16, st.list_off, 0,
                                               0, 0);
    }
  };

  f32x16 acc[NU][HB];
#pragma unroll
  for (int u = 0; u < NU; ++u)
#pragma unroll
    for (int bh = 0; bh < HB; ++bh)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[u][bh][r] = 0.f;

  WpOps ops[2];
  u32x2 pv[NS];          // positions (0 = empty) of the lane's two rows in an even step and the one behind it, per slot

  // ---- the pieces of one step's operand fetch ----
  auto pf_loc = [&](int sl, const char* lcs, int sn) {      // (sn even)
    uint32_t off;
    if constexpr (HA == 1) off = lbS[sl] + (uint32_t)(sn * 32);
    else off = (sl < NFULL ? lbF + (uint32_t)(sl * kWpRows * 2) : lbH) + (uint32_t)(sn * 32);
    pv[sl] = *(const u32x2*)(lcs + off);
  };
  auto pf_g = [&](int j, const char* gs, int sn, WpOps& on) {   // j = 2 * bh + h
    const int h = j & 1, bh = j >> 1;
    on.b[bh][h] = Mma<T>::read_tr((const T*)(gs + gad[h] + (uint32_t)(bh * GH + sn * 1024)));
  };
  auto pf_x = [&](int j, const char* xs, int sn, WpOps& on) {    // j = 2 * slot + h
    const int sl = j >> 1, h = j & 1;
    const uint32_t two = pv[sl][sn & 1];
    const uint32_t ad = ((h ? two >> 16 : two & 0xffffu) << 6) + byte0;      // position 0 is the zero row
    if (sl < NFULL) {
      on.a[HA * sl][h] = Mma<T>::read_tr((const T*)(xs + ad));
      if constexpr (HA == 2) on.a[2 * sl + 1][h] = Mma<T>::read_tr((const T*)(xs + ad + (uint32_t)XH));
    } else {
      on.a[HA * NFULL][h] = Mma<T>::read_tr((const T*)(xs + ad + ahH));
    }
  };
  auto mm = [&](int m, const WpOps& oc) {
    const int u = m / HB, bh = m % HB;
    const u32x4 av = u32x4{oc.a[u][0][0], oc.a[u][0][1], oc.a[u][1][0], oc.a[u][1][1]};
    const u32x4 bv = u32x4{oc.b[bh][0][0], oc.b[bh][0][1], oc.b[bh][1][0], oc.b[bh][1][1]};
    acc[u][bh] = Mma32<T>::run(av, bv, acc[u][bh]);
  };

  // One step: the MFMAs of 16 rows on `oc`; between them the operand fetch of the
  // following step (rows 16 sn.. of the buffers xs/gs/lcs) into `on`, and four staging
  // pieces t0..t0+3 of the next tile (t0 < 0: none).
  auto step = [&](const WpOps& oc, WpOps& on, const char* xs, const char* gs, const char* lcs, int sn,
                  int t0, const WpStage& sg) {
    int32_t ids[4] = {0, 0, 0, 0};
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      mm(m, oc);
      // operand fetch of the next step: table positions and g first, then the x reads
      // that depend on the positions, PF0 MFMAs later
      if constexpr (HA == 2) {
        if (m < PF0) {
#pragma unroll
          for (int t = m * IP; t < (m + 1) * IP && t < NS + 4; ++t) {
            if (t >= NS) pf_g(t - NS, gs, sn, on);
            else if (sn % 2 == 0) pf_loc(t, lcs, sn);
          }
        } else if (m - PF0 < NL) {
          pf_x(m - PF0, xs, sn, on);
        }
      } else {
        if (m == 0) {
#pragma unroll
          for (int t = 0; t < NS; ++t)
            if (sn % 2 == 0) pf_loc(t, lcs, sn);
#pragma unroll
          for (int t = 0; t < 2 * HB; ++t) pf_g(t, gs, sn, on);
        }
        if (m >= XS) {
#pragma unroll
          for (int t = (m - XS) * XP; t < (m - XS + 1) * XP && t < NL; ++t) pf_x(t, xs, sn, on);
        }
      }
      if (t0 >= 0) {
        if (m == 0) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (t0 + j < kPieces) ids[j] = stage_id(t0 + j, sg);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int mj = (j * NM) / 4 + 1 < NM ? (j * NM) / 4 + 1 : NM - 1;
          if (m == mj && t0 + j < kPieces) {
            stage_piece(t0 + j, sg, ids[j]);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // operand fetch of a tile's first step when there is no previous step to hide it under
  auto first_fetch = [&](const char* xs, const char* gs, const char* lcs, WpOps& on) {
#pragma unroll
    for (int t = 0; t < NS; ++t) pf_loc(t, lcs, 0);
#pragma unroll
    for (int t = 0; t < 2 * HB; ++t) pf_g(t, gs, 0, on);
#pragma unroll
    for (int t = 0; t < NL; ++t) pf_x(t, xs, 0, on);
  };

  // ---- prologue: first list, first tile, second list ----
  int32_t p_nxt = uptr[t_begin + 1];
  int32_t p_nx2 = uptr[min(t_begin + 2, tiles)];
  int32_t p_nx3 = uptr[min(t_begin + 3, tiles)];
  {
    const int32_t p_cur = uptr[t_begin];
    WpStage st = make_stage(t_begin, 0, p_cur, p_nxt - p_cur, s_u0 + 4, s_u0 + 4, s_x0, s_g0, s_loc0);
    stage_piece(tU, st, 0);                                // list of the first tile -> s_u0
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    st = make_stage(t_begin, p_nxt - p_cur, p_nxt, p_nx2 - p_nxt, s_u0 + 4, s_u1 + 4, s_x0, s_g0, s_loc0);
#pragma unroll
    for (int t = 0; t < kPieces; ++t) stage_piece(t, st, stage_id(t, st));     // also: list of the second tile
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    first_fetch((const char*)s_x0, (const char*)s_g0, (const char*)s_loc0, ops[0]);
  }

  // one tile out of buffer B; stages the next tile into buffer 1 - B meanwhile
  auto tile_body = [&](auto BC, int64_t tile) {
    constexpr int B = decltype(BC)::value;
    const char* xs = B ? (const char*)s_x1 : (const char*)s_x0;
    const char* gs = B ? (const char*)s_g1 : (const char*)s_g0;
    const char* lcs = B ? (const char*)s_loc1 : (const char*)s_loc0;
    // next tile -> the other buffers (its list is in the other s_u); list of the tile after
    // it -> this tile's s_u, which has been used up
    const WpStage sg = make_stage(tile + 1, p_nx2 - p_nxt, p_nx2, p_nx3 - p_nx2, B ? s_u0 + 4 : s_u1 + 4,
                                  B ? s_u1 + 4 : s_u0 + 4, B ? s_x0 : s_x1, B ? s_g0 : s_g1,
                                  B ? s_loc0 : s_loc1);
    // list boundary four tiles ahead, as a vector load: a scalar load would share its counter
    // with the LDS reads and force them to drain where it is used
    const uint32_t p_raw = __builtin_amdgcn_raw_buffer_load_b32(
        rs_p, (uint32_t)min(tile + 4, tiles) * 4u, 0, 0);
    p_nxt = p_nx2;
    p_nx2 = p_nx3;
#pragma unroll
    for (int s = 0; s < 7; ++s)
      step(ops[s & 1], ops[(s + 1) & 1], xs, gs, lcs, s + 1, s < 5 ? 4 * s : -1, sg);
    // The next tile has landed: own loads, then everyone's.  The LDS reads in flight belong
    // to this tile's buffers and need not drain, so neither barrier is a __syncthreads().
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    p_nx3 = __builtin_amdgcn_readfirstlane((int32_t)p_raw);
    // last step, with the first operands of the next tile fetched from the other buffer
    step(ops[1], ops[0], sg.sx, sg.sg, sg.sl, 0, -1, sg);
    asm volatile("s_barrier" ::: "memory");  // buffer B may be overwritten now: its last reads fed this step
  };

  for (int64_t tile = t_begin; tile < t_end; tile += 2) {
    tile_body(std::integral_constant<int, 0>{}, tile);
    if (tile + 1 < t_end) tile_body(std::integral_constant<int, 1>{}, tile + 1);
  }

  // ---- per-range sums -> partial[split][slot][a][b] ----
  const int b32 = lane & 31;
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int slot = u < HA * NFULL ? slotF + u / HA : slotH;
    const int ah = u < HA * NFULL ? u % HA : (wave & 1);
    if (slot >= KK) continue;
    const int ldb = BLK ? cb : CB;
    float* dst = BLK ? partial + (((int64_t)split * KK + slot) * ca + blk_a * CA) * cb + blk_b * CB
                     : partial + ((int64_t)split * KK + slot) * (CA * CB);
    // a half block at the end of the channels: what the staging loads brought in beyond a
    // row only reached sums that are not written
    if (BLK && blk_a * CA + 32 * ah >= ca) continue;
#pragma unroll
    for (int bh = 0; bh < HB; ++bh) {
      if (BLK && blk_b * CB + 32 * bh >= cb) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int a = 32 * ah + 8 * (r >> 2) + 4 * q + (r & 3);
        dst[a * ldb + 32 * bh + b32] = acc[u][bh][r];
      }
    }
  }
}

}  // namespace ocnn

using namespace ocnn;

// blocks of channel pairs: 64 x 64 (the last of a side half beyond the channels), but for 32 channels of x, whose 32 x 64
// blocks have room for the sums of all 27 slots in one workgroup, and for the 32 x 32 layer
static bool wp_wide(int ca) { return ca > 32; }

// workgroups of one range of tiles: the slot groups, the blocks of channel pairs
static int wp_range_workgroups(int K, int ca, int cb) {
  const int groups = (K == 27 && wp_wide(ca)) ? 2 : 1;
  return groups * ((ca + 63) / 64) * ((cb + 63) / 64);
}

// ranges of tiles at most: as many as put a workgroup in every place, one a CU by its LDS or two (wp_places)
static int wp_splits(int range_workgroups, int places) { return std::min(512, std::max(8, places / range_workgroups)); }

// Workgroups at once: one a CU, and two of 32 x 32 blocks of tiles with few distinct rows (kWpCapTwo) where a CU has 14 tiles: below, the
// further sets of sums take more than the tiles gain.  us, one a CU / two: 27 slots 250 k rows 30.6 / 32.1, 421 k 40.5 / 41.5, 500 k
// 45.1 / 44.3, 1.5 M 111.6 / 105.1; nine 120 k 16.1 / 18.0, 400 k 23.4 / 23.4, 1 M 41.4 / 37.4; eight 120 k 14.8 / 16.5, 400 k 21.1 / 21.2,
// 1 M 36.8 / 32.5; three 120 k 11.8 / 12.9, 400 k 18.6 / 18.9, 1 M 33.2 / 29.7.
static int wp_places(int64_t tiles, int n_cu, bool two) { return two && tiles >= 14 * n_cu ? 2 * n_cu : n_cu; }

// Tiles of a range, for the least time of
//   rounds of workgroups x (tiles of a range + what a workgroup costs besides: lists and the staging of
//   the first tile, writing the sums) + the sums of all ranges written and read back, in units of one tile's time.
// Measured (fp16, 64 x 64 blocks of 27 slots): 2.45 us a tile and 8 us besides on 33 - 157 tiles a range; the sums
// move at about 3.5 TB/s.  Rounds are counted on an XCD's places (40 workgroups on 32 are two rounds), the sums
// where there are few tiles (256 -> 256: 7 MB a range).  The other blocks and slot counts and 32 x 32 with two workgroups
// a CU have no figures of their own.
constexpr double kWpTileUs = 2.45, kWpFixedUs = 8.085, kWpSumUs = 5.635e-7; // us; us a byte of sums
static int64_t wp_tiles_per_range(int64_t tiles, int wgs, int64_t sums_bytes, int places, int products = 1) {
  const int places_xcd = std::max(1, places / 8);
  int64_t best = std::max<int64_t>(tiles, 1);
  double least = 1e30;
  int64_t s = 1;
  const int64_t most = wp_splits(wgs * products, places);
  for (bool more = true; more && s <= most;) {               // (the fewest ranges of as many tiles; then of fewer tiles)
    const int64_t per = std::max<int64_t>(1, cdiv(tiles, s)), used = s;
    more = per > 1;
    if (more) s = cdiv(tiles, per - 1);
    const double cost = (double)cdiv(cdiv(used * wgs, 8) * products, places_xcd) * ((double)per * kWpTileUs + kWpFixedUs) +
                        (double)used * (double)(sums_bytes * products) * kWpSumUs;
    if (cost < least) least = cost, best = per;
  }
  return best;
}

// fp32: whether the operands are split by a launch of their own, and the products are workgroups of the 16-bit kernel on 64 x 64
// blocks.  With few slots that kernel is ahead where the layer is wide enough to make up for the pieces written and read:
// wgrad_f32.hip stages every row of x once for 64 channels of g, and issues the MFMAs of twelve slots for nine.  us, wgrad_f32.hip /
// so: nine slots 256 -> 256 on 4 k rows 32 / 32, 20 k 87 / 84, 100 k 410 / 360; 512 -> 512 on 20 k 323 / 277; 1024 -> 1024 1322 / 956;
// 224 -> 224 on 40 k 147 / 143, 128 -> 256 99 / 100; eight slots 256 -> 256 on 40 k 138 / 136, 120 k 396 / 385, 256 -> 384 on 40 k 204 / 190,
// 512 -> 512 on 20 k 256 / 242; three 256 -> 256 on 40 k 95 / 99, 120 k 284 / 303, 256 -> 384 145 / 131, 512 -> 512 on 20 k 182 / 166, on 4 k 43 / 48.
// (27 slots: wgrad_f32.hip always.)
static bool wp_takes_pieces(int64_t rows, int K, int ca, int cb) {
  if (K == 27) return false;
  return ca * cb >= (K == 3 ? 150 : 128) * (ca + cb) && rows * ca * cb >= (K == 9 ? 1ll << 30 : 1ll << 31);
}

struct WpPieces {                             // ranges of tiles, and where the pieces end in the workspace
  int64_t per, used, x_bytes, g_bytes;
};
static WpPieces wp_pieces(int64_t rows_x, int64_t rows, int K, int ca, int cb, int n_cu) {
  const int64_t tiles = cdiv(rows, kWpRows);
  const int64_t per = wp_tiles_per_range(tiles, wp_range_workgroups(K, ca, cb), (int64_t)K * ca * cb * 4, n_cu, 3);
  return {per, cdiv(tiles, per), align_up(rows_x * ca * 2, 256), align_up(rows * cb * 2, 256)};
}

static int wp_cu_count() {
  static int n_cu = 0;
  if (n_cu == 0) {
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) return 0;
    n_cu = prop.multiProcessorCount;
  }
  return n_cu;
}

extern "C" int ocnn_conv_wgrad_planned_supported(int dtype, int64_t rows_x, int64_t rows, int K, int ca,
                                                 int cb, int plan_max_distinct) {
  if (dtype != OCNN_F16 && dtype != OCNN_BF16 && dtype != OCNN_F32) return 0;   // (fp32: wgrad_f32.hip)
  if (ca < 32 || cb < 32 || ca % 32 != 0 || cb % 32 != 0 || ca > 1024 || cb > 1024)
    return 0;
  if (K != 27 && K != 9 && K != 8 && K != 3) return 0;
  if (plan_max_distinct < 0 || plan_max_distinct > kWpCap) return 0;
  if (rows_x < 0 || rows < 0) return 0;
  if ((int64_t)rows_x * ca * 2 > 0xfff00000ll || ((int64_t)rows + kWpRows) * cb * 2 > 0xfff00000ll) return 0;
  return 1;
}

extern "C" int64_t ocnn_conv_wgrad_planned_workspace_bytes(int K, int ca, int cb) {
  const int n_cu = wp_cu_count();
  const int64_t splits = n_cu > 0 ? wp_splits(wp_range_workgroups(K, ca, cb), ca == 32 && cb == 32 ? 2 * n_cu : n_cu) : 512;
  return align_up(splits * K * ca * cb * 4, 256);
}

extern "C" int64_t ocnn_conv_wgrad_planned_workspace_bytes_for(int dtype, int64_t rows_x, int64_t rows, int K,
                                                               int ca, int cb) {
  if (dtype != OCNN_F32 || rows_x < 0 || rows < 0) return ocnn_conv_wgrad_planned_workspace_bytes(K, ca, cb);
  const int n_cu = wp_cu_count();
  const int64_t tiles = cdiv(rows, kWpRows);
  if (wp_takes_pieces(rows, K, ca, cb) && n_cu > 0) {
    const WpPieces p = wp_pieces(rows_x, rows, K, ca, cb, n_cu);
    return align_up(2 * p.x_bytes + 2 * p.g_bytes + 3 * p.used * K * ca * cb * 4, 256);
  }
  const int64_t sets = n_cu > 0 ? wf_workspace_sets(wf_split_tiles(tiles, K, ca, cb, n_cu), tiles) : tiles;
  return align_up(sets * K * ca * cb * 4, 256);
}

struct WpArgs {
  const void *x, *g, *x_lo, *g_lo;            // x_lo, g_lo: the low bf16 pieces of fp32 data (else null)
  int64_t rows_x, rows, set, per, plan_total; // set: floats of the sums of one product of pieces
  const uint16_t* loc;
  const int32_t *uptr, *urows;
  int K, ca, cb, used;                        // used: ranges of tiles
  float* partial;
  bool two;                                   // two workgroups fit a CU
};

template <typename T, int CA, int CB, int KK, int NFULL, int NHALF, int GROUPS, bool PIECES>
static void launch_wp(const WpArgs& a, hipStream_t st) {
  const int64_t tiles = cdiv(a.rows, kWpRows);
  const uint32_t xb = (uint32_t)(a.rows_x * a.ca * 2), gb = (uint32_t)(a.rows * a.cb * 2);
  const int wgs = a.used * wp_range_workgroups(a.K, a.ca, a.cb);
  const uint32_t lb = (uint32_t)(tiles * kWpRows * KK * 2), ub = (uint32_t)(a.plan_total * 4);
#define OCNN_WP_KERNEL(BLK_, CAP_)                                                                                   \
  hipLaunchKernelGGL((conv_wgrad_planned_kernel<T, CA, CB, KK, NFULL, NHALF, GROUPS, BLK_, CAP_, PIECES>),                   \
                     dim3(8 * (unsigned)cdiv(wgs, 8), PIECES ? 3 : 1), dim3(256), 0, st, (const T*)a.x, xb, (const T*)a.g, \
                     gb, a.loc, lb, a.uptr, a.urows, ub, tiles, a.per, wgs, a.ca, a.cb, a.partial, (const T*)a.x_lo,       \
                     (const T*)a.g_lo, a.set)
  if (a.ca == CA && a.cb == CB) {
    if (CB == 32 && a.two) OCNN_WP_KERNEL(false, CB == 32 ? kWpCapTwo : kWpCap);
    else OCNN_WP_KERNEL(false, kWpCap);
  } else if constexpr (CB == 64)
    OCNN_WP_KERNEL(true, kWpCap);
#undef OCNN_WP_KERNEL
}

// per-range sums of x^T g into `partial`
template <typename T>
static void launch_wp_sums(const WpArgs& a, hipStream_t st) {
#define OCNN_WP_LAUNCH(CA, CB, KK, NF, NH, GR) launch_wp<T, CA, CB, KK, NF, NH, GR, false>(a, st)
  if (wp_wide(a.ca)) {
    if (a.K == 27) OCNN_WP_LAUNCH(64, 64, 27, 3, 1, 2);
    else if (a.K == 9) OCNN_WP_LAUNCH(64, 64, 9, 2, 1, 1);
    else if (a.K == 8) OCNN_WP_LAUNCH(64, 64, 8, 2, 0, 1);
    else OCNN_WP_LAUNCH(64, 64, 3, 1, 0, 1);
  } else if (a.cb > 32) {
    if (a.K == 27) OCNN_WP_LAUNCH(32, 64, 27, 7, 0, 1);
    else if (a.K == 9) OCNN_WP_LAUNCH(32, 64, 9, 3, 0, 1);
    else if (a.K == 8) OCNN_WP_LAUNCH(32, 64, 8, 2, 0, 1);
    else OCNN_WP_LAUNCH(32, 64, 3, 1, 0, 1);
  } else {
    if (a.K == 27) OCNN_WP_LAUNCH(32, 32, 27, 7, 0, 1);
    else if (a.K == 9) OCNN_WP_LAUNCH(32, 32, 9, 3, 0, 1);
    else if (a.K == 8) OCNN_WP_LAUNCH(32, 32, 8, 2, 0, 1);
    else OCNN_WP_LAUNCH(32, 32, 3, 1, 0, 1);
  }
#undef OCNN_WP_LAUNCH
}

// The same of fp32 as three products of bf16 pieces (wp_takes_pieces), sums of their own for each
static void launch_wp_pieces(const WpArgs& a, hipStream_t st) {
  if (a.K == 9) launch_wp<bf16, 64, 64, 9, 2, 1, 1, true>(a, st);
  else if (a.K == 8) launch_wp<bf16, 64, 64, 8, 2, 0, 1, true>(a, st);
  else launch_wp<bf16, 64, 64, 3, 1, 0, 1, true>(a, st);
}

// T: the type of x, g and gw (float: wgrad_f32.hip, or as pieces)
template <typename T> struct WpPass : Pass {
  static constexpr bool F32 = std::is_same<T, float>::value;
  WpArgs a;
  hipStream_t st;
  WfSplit f32;
  int rc = OCNN_OK, splits = 0, out_transposed = 0;
  float* sums_at = nullptr;
  void* gw = nullptr;         // set: the reduction is launched behind the kernel (sums at an odd address)

  WpPass(const ocnnx_wgrad_args& p, hipStream_t stream) : st(stream) {
    const int n_cu = wp_cu_count();
    if (n_cu <= 0) {
      set_error("conv_wgrad_planned: cannot query the device");
      rc = OCNN_ERR_HIP;
      return;
    }
    const int K = p.K, ca = p.ca, cb = p.cb;
    const int64_t tiles = cdiv(p.rows, kWpRows), sums = (int64_t)K * ca * cb * 4;       // bytes of a range's sums
    a = WpArgs{p.x, p.g, nullptr, nullptr, p.rows_x, p.rows, 0, 0, p.plan_total, p.loc, p.uptr, p.urows, K, ca, cb, 0,
               (float*)p.workspace, ca == 32 && cb == 32 && p.plan_max_distinct <= kWpCapTwo};
    WpPieces pieces{};
    const bool split = F32 && wp_takes_pieces(p.rows, K, ca, cb);
    if (split) {
      pieces = wp_pieces(p.rows_x, p.rows, K, ca, cb, n_cu);
      a.per = pieces.per;
      a.used = (int)pieces.used;
      a.set = pieces.used * K * ca * cb;
    } else if (F32) {
      f32 = wf_split_tiles(tiles, K, ca, cb, n_cu);
      a.used = (int)wf_workspace_sets(f32, tiles);
    } else {
      a.per = wp_tiles_per_range(tiles, wp_range_workgroups(K, ca, cb), sums, wp_places(tiles, n_cu, a.two));
      a.used = (int)cdiv(tiles, a.per);
    }
    const int64_t pieces_bytes = 2 * pieces.x_bytes + 2 * pieces.g_bytes;
    if (p.workspace_bytes < pieces_bytes + (split ? 3 : 1) * a.used * sums) {
      set_error("conv_wgrad_planned: workspace too small");
      rc = OCNN_ERR_WORKSPACE;
      return;
    }
    const int64_t per = (int64_t)K * ca * cb;
    splits = p.rows > 0 ? a.used : 0;
    if (split) {
      char* ws = (char*)p.workspace;
      a.partial = (float*)(ws + pieces_bytes);
      splits *= 3;
      if (p.rows > 0) {
        bf16 *xh = (bf16*)ws, *xl = (bf16*)(ws + pieces.x_bytes), *gh = (bf16*)(ws + 2 * pieces.x_bytes);
        bf16* gl = (bf16*)(ws + 2 * pieces.x_bytes + pieces.g_bytes);
        const int64_t nx = p.rows_x * ca, ng = p.rows * cb;
        Job j{Job::kSplit, (unsigned)cdiv((nx + ng) / 8, 256), {}};
        j.split = SplitJob{(const float*)p.x, (const float*)p.g, xh, xl, gh, gl, nx, ng};
        before.add(j);
        a.x = xh, a.x_lo = xl, a.g = gh, a.g_lo = gl;
      }
    }
    sums_at = a.partial;
    if (F32 && !split && p.rows > 0) {                                 // the reduction behind the last launch
      const WfPart last = part_of((cdiv(tiles, f32.launch) - 1) * f32.launch);
      splits = (int)last.splits, sums_at = last.sums_at;
    }
    if ((uintptr_t)a.partial % 16 != 0) {
      gw = p.gw, out_transposed = p.out_transposed;
      return;
    }
    const int lanes = wgrad_reduce_lanes(splits, per);
    Job j{Job::kReduce, (unsigned)cdiv(per / 4, 256 / lanes), {}};
    j.reduce = ReduceJob{sums_at, p.gw, per, splits, p.out_transposed ? ca : 0, cb, lanes};
    after.add(j);
  }

  // fp32 in several launches: their sets lie at 1 .., and what those before have come to (none before the first) at 0 or behind the
  // last place for a set, where the reduction of the launch before left it; their own goes to the other of the two.
  struct WfPart {
    int64_t first, tiles, splits;               // splits: with the sum of those before
    float *partial, *sums_at, *sum_to;
  };
  WfPart part_of(int64_t first) const {
    const int64_t tiles = cdiv(a.rows, kWpRows), per = (int64_t)a.K * a.ca * a.cb, n = std::min(f32.launch, tiles - first);
    if (f32.launch >= tiles) return {0, tiles, f32.sets, a.partial, a.partial, nullptr};
    const int64_t number = first / f32.launch, sets = cdiv(n, f32.run), end = f32.sets + 1;
    const bool behind = number % 2 == 0 && number > 0;       // the sum of those before lies behind
    const int64_t at = behind ? end - sets : 1;
    return {first, n, sets + (number > 0), a.partial + at * per, a.partial + (number == 0 || behind ? at : 0) * per,
            a.partial + (number % 2 == 0 ? 0 : end) * per};
  }

  int main() override {
    if (a.rows > 0) {
      if (F32 && a.x_lo) {
        launch_wp_pieces(a, st);
      } else if constexpr (F32) {
        const int64_t tiles = cdiv(a.rows, kWpRows);
        for (int64_t first = 0; first < tiles; first += f32.launch) {
          const WfPart p = part_of(first);
          launch_wgrad_f32({(const float*)a.x, (const float*)a.g + first * kWpRows * a.cb, a.rows_x,
                            std::min(p.tiles * kWpRows, a.rows - first * kWpRows), a.plan_total, a.loc + first * kWpRows * a.K,
                            a.uptr + first, a.urows, a.K, a.ca, a.cb, f32, p.partial}, st);
          if (first + p.tiles < tiles) launch_wgrad_reduce<float>(p.sums_at, (int)p.splits, a.K, a.ca, a.cb, 0, p.sum_to, st);
        }
      } else {
        launch_wp_sums<T>(a, st);
      }
    }
    if (gw) launch_wgrad_reduce<T>(sums_at, splits, a.K, a.ca, a.cb, out_transposed, (T*)gw, st);
    return check_launch("conv_wgrad_planned");
  }
};

// The pass for these arguments, to be deleted by the caller.
int ocnn::wgrad_planned_pass(int dtype, const ocnnx_wgrad_args& p, hipStream_t st, Pass** pass) {
  *pass = nullptr;
  OCNN_REQUIRE(ocnn_conv_wgrad_planned_supported(dtype, p.rows_x, p.rows, p.K, p.ca, p.cb, p.plan_max_distinct),
               "conv_wgrad_planned: shape not supported");
  OCNN_REQUIRE(p.rows >= 0 && (int64_t)p.rows * p.K * 2 < 0xfff00000ll && p.plan_total >= 0 && p.plan_total < (1ll << 29),
               "conv_wgrad_planned: rows out of range");
  OCNN_REQUIRE_PTRS("conv_wgrad_planned", p.gw, p.workspace);
  OCNN_REQUIRE(p.rows == 0 || (p.g && p.loc && p.uptr && p.urows && (p.rows_x == 0 || p.x)),
               "conv_wgrad_planned: a required pointer is NULL (of x, g, loc, uptr, urows)");
  auto made = [&](auto* wp) {
    OCNN_REQUIRE(wp, "conv_wgrad_planned: out of host memory");
    *pass = wp;
    return wp->rc;
  };
  if (dtype == OCNN_F32) return made(new (std::nothrow) WpPass<float>(p, st));
  if (dtype == OCNN_F16) return made(new (std::nothrow) WpPass<f16>(p, st));
  return made(new (std::nothrow) WpPass<bf16>(p, st));
}

extern "C" int ocnn_conv_wgrad_planned(int dtype, const void* x, int64_t rows_x, const void* g,
                                       const uint16_t* loc, const int32_t* uptr, const int32_t* urows,
                                       int plan_max_distinct, int64_t plan_total, int64_t rows, int K,
                                       int ca, int cb, int out_transposed, void* gw, void* workspace,
                                       int64_t workspace_bytes, void* stream) {
  Pass* pass = nullptr;
  int rc = wgrad_planned_pass(dtype, {x, rows_x, g, loc, uptr, urows, plan_max_distinct, plan_total, rows, K, ca, cb,
                                      out_transposed, gw, workspace, workspace_bytes}, (hipStream_t)stream, &pass);
  if (rc == OCNN_OK) {
    launch_jobs(dtype, pass->before, (hipStream_t)stream);
    rc = pass->main();
    if (rc == OCNN_OK) launch_jobs(dtype, pass->after, (hipStream_t)stream);
  }
  delete pass;
  return rc == OCNN_OK ? check_launch("conv_wgrad_planned") : rc;
}

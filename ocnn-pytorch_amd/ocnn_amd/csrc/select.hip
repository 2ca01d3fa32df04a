// Which kernel runs a layer: the selection among the gather-GEMM and weight-gradient entry
// points.  ocnn_conv_gather_choose and ocnn_conv_wgrad_choose choose among the entry points of the
// public header, for whoever binds it; this package's own host path calls ocnnx_gather_choose in the
// place of the first, which knows the kernel of conv_tile.hip in its full range as well.
//
// Every *_supported() predicate says whether a kernel takes a shape class; the row ranges that
// its entry point checks on top (32-bit buffer offsets of the output, of the table, of the
// plan) are repeated here, so a choice is always one that the chosen entry point accepts.
#include <algorithm>

#include "common.hpp"
#include "host_api.hpp"

using namespace ocnn;

namespace {

constexpr int64_t kOffsetLimit = 0xfff00000ll;   // what a 32-bit buffer offset may reach
constexpr int kPadMinRows = 16384;               // from here on odd channel counts run zero-padded
constexpr double kSparseMaxOccupancy = 0.3;      // share of table entries set, up to which the pair plan pays
constexpr int64_t kSparseMinRows = 32768;        // (its workgroups load their weights once per launch)

bool rows_ok(int64_t rows_out, int64_t plan_total) {
  return rows_out >= 0 && rows_out < (1ll << 31) && plan_total >= 0 && plan_total < (1ll << 29);
}

}  // namespace

extern "C" int ocnn_conv_gather_choose(int dtype, int64_t rows_in, int64_t rows_out, int K, int cin, int cout,
                                       int identity_table, int has_plan, int plan_max_distinct,
                                       int64_t plan_total, double plan_occupancy, double plan_reuse) {
  const bool known = dtype == OCNN_F32 || dtype == OCNN_F16 || dtype == OCNN_BF16;
  if (rows_out >= kPadMinRows && known && (cin % 32 != 0 || cout % 16 != 0)) return OCNN_GATHER_ZERO_PADDED;
  if (identity_table && K == 1 && rows_out == rows_in) {
    if (ocnn_conv_dense_rw_supported(dtype, rows_out, cin, cout)) return OCNN_GATHER_DENSE_RW;
    // (many input channels into few output channels: the row tile that fits LDS is small and
    // the weights are streamed once per tile; the plan-free kernel is no slower there)
    if (!(cin >= 512 && cout < 256) && ocnn_conv_dense_supported(dtype, rows_out, cin, cout))
      return OCNN_GATHER_DENSE;
  }
  if (has_plan && rows_ok(rows_out, plan_total)) {
    if (ocnn_conv_gather_rw_supported(dtype, rows_in, K, cin, cout, plan_max_distinct) &&
        rows_out * K * 2 < kOffsetLimit && (rows_out + 128) * cout * 2 < kOffsetLimit)
      return OCNN_GATHER_RW;
    // (eight slots - the 2x2x2 tables and their inverses - stream a third of the weights of 27 per
    // tile: there the kernel for wide layers beats the pair plan also at one slot in eight set,
    // 0.84 -> 0.67 ms for 96 -> 96 between depths 9 and 8, and without rows shared inside a tile)
    if (K == 8 && ocnn_conv_gather_wide_supported(dtype, rows_in, K, cin, cout, plan_max_distinct))
      return OCNN_GATHER_WIDE;
    if (plan_occupancy <= kSparseMaxOccupancy && rows_out >= kSparseMinRows &&
        rows_out * cout * 2 <= kOffsetLimit &&
        ocnn_conv_gather_sparse_supported(dtype, rows_in, K, cin, cout, plan_max_distinct))
      return OCNN_GATHER_SPARSE;
    // (staging a tile's distinct rows pays when rows are used more than once per tile)
    if (plan_reuse >= 2.0 && ocnn_conv_gather_wide_supported(dtype, rows_in, K, cin, cout, plan_max_distinct))
      return OCNN_GATHER_WIDE;
    if (plan_reuse >= 2.0 && K <= 27 && ocnn_conv_gather_planned_supported(dtype, rows_in, cin, cout))
      return OCNN_GATHER_PLANNED;
  }
  return OCNN_GATHER_PLAIN;
}

// The same for this package's own host path, which also has the kernel of conv_tile.hip in its full
// range: it takes the wide layers, which it splits where there are few tiles, the multi-pass ones (175
// layer passes 39.6 ms instead of 58.4, slower in none) and most of what would run plan-free on a table with a
// plan.  The plan-free kernel stays (us, tile kernel / plan-free)
//  - for 16-bit layers with little work per row that is staged: on 8 or 9 slots below 4096 channel pairs, on 3
//    below 16384 and, there, below kTileMinProducts products (too few for all CUs, and the weights
//    are half of a pass).  64 -> 32 on 4.9 M rows of a 3x1x1 table 369 / 248; 32 -> 64 on those of 2x2x2 502 / 421;
//    256 -> 256 on three slots of 3826 rows 19 / 14, 128 -> 128 of 100 k rows, 36 % set, 26 / 24, of 235 k rows, 85 %
//    set, 55 / 65; 128 -> 32 on nine slots 1.17 x faster on the tile kernel in the median, 256 -> 64 1.5 x, 27 slots
//    1.1 - 2 x from 32 -> 64 on;
//  - for every data type on 8 or 9 slots of a table of little reuse where rows in tiles too dense for the plan
//    run apart (plan_overflow): the second launch and the copy of its rows cost 10 - 40 us, which pays from
//    kTileMinProductsApart on (fp32: three products a pair).  18.8 k rows of 3x3x1 stride 2: 128 -> 128 39 / 19,
//    fp32 111 / 68; 235 k rows: 106 / 97, fp32 433 / 449 and 64 -> 64 202 / 178.
// It also takes the place of the pair plan (OCNN_GATHER_SPARSE) where the slots or blocks of rows without an entry are
// many: on 8 or 9 slots, and on 27 slots but in the inverse tables of stride 2 (fewer rows read than written), where a
// block of fine rows has something in every slot, and below 6 % set, the least that was measured (us, pair plan / tile kernel,
// f16, 96 -> 96 and 128 -> 128): 1.13 M rows 7 % set 349 / 323, 530 / 457; 822 k rows 14 % set 339 / 339, 611 / 484; 533 k
// rows 20 % set 257 / 221, 482 / 338; stride 2 947 k rows 7 % set 337 / 291, 479 / 409, 593 k rows 9 % set 318 / 308 for 96;
// inverse of stride 2 1.13 M rows 6 % set 329 / 332, 505 / 449, 264 k rows 8 % set 91 / 120, 133 / 160, 593 k rows 9 % set
// 190 / 263, 288 / 386; nine slots of 1.13 M rows 16 % set 311 / 247, 454 / 318, inverse 5 % set 241 / 195, 373 / 242.
// Over 916 bf16 passes (six kernel shapes, strides 1 and 2, all and non-empty nodes, three octrees of 20 k - 1 M
// points, eleven widths): all plan-free 80.1 ms, all on the tile kernel 74.1, by this rule 70.0, the faster of the
// two each time 69.3.  Other fp32 layers gain on every table, 1.04 - 9 x: plan-free reads three copies of their rows.
// Dense rows of few channels run on the kernel of dense_rows.hip at every number of rows.  Over its 22 pairs of channels
// (f16) its time is 0.75 of that of the kernel chosen otherwise on 1.13 M rows, 0.68 on 300 k, 0.67 on 60 k, 0.71 on 16 k and
// on 4096.  Pairs without gain: 192 -> 32 on 1.13 M rows 101 / 105 us, 64 -> 256 on 300 k 34 / 34, and 128 -> 128, whose other
// kernel is the dense one: 110 / 118 on 1.13 M rows, but 29.8 / 28.8 on 300 k, 11.2 / 11.0 on 60 k, 8.1 / 7.1 on 16 k and
// 7.8 / 7.2 on 4096.  (With an index of the rows: the dense kernel.)
constexpr double kTileMinProducts = 3.0e9;
constexpr double kTileMinProductsApart = 1.7e10;
constexpr double kTileMinOccupancy = 0.06, kTileMinOccupancyInverse = 0.12;        // of 27 slots

extern "C" int ocnnx_gather_choose(int dtype, int64_t rows_in, int64_t rows_out, int K, int cin, int cout,
                                   int identity_table, int has_plan, int plan_max_distinct, int64_t plan_total,
                                   double plan_occupancy, double plan_reuse, int plan_overflow) {
  const int pick = ocnn_conv_gather_choose(dtype, rows_in, rows_out, K, cin, cout, identity_table, has_plan,
                                           plan_max_distinct, plan_total, plan_occupancy, plan_reuse);
  if (identity_table && K == 1 && rows_out == rows_in && (pick == OCNN_GATHER_PLAIN || pick == OCNN_GATHER_DENSE_RW) &&
      ocnnx_dense_rows_supported(dtype, rows_out, cin, cout))
    return OCNNX_GATHER_ROWS;
  if (!has_plan || !rows_ok(rows_out, plan_total) ||
      !ocnnx_gather_tile_supported(dtype, rows_in, K, cin, cout, plan_max_distinct))
    return pick;
  if (pick == OCNN_GATHER_PLANNED || pick == OCNN_GATHER_WIDE) return OCNNX_GATHER_TILE;
  if (pick == OCNN_GATHER_SPARSE)
    return (K < 27 ? (int64_t)cin * cout >= 4096
                   : plan_occupancy > (rows_in < rows_out ? kTileMinOccupancyInverse : kTileMinOccupancy))
               ? OCNNX_GATHER_TILE
               : pick;
  if (pick != OCNN_GATHER_PLAIN) return pick;
  const bool half = dtype != OCNN_F32;
  const double products = plan_occupancy * (double)rows_out * K * cin * cout * (half ? 1 : 3);
  if (K < 27) {
    if (plan_reuse < 2.0 && plan_overflow && products < kTileMinProductsApart) return pick;
    if (half && (K >= 8 ? cin * cout < 4096 : cin * cout < 16384 || products < kTileMinProducts)) return pick;
  }
  return OCNNX_GATHER_TILE;
}

extern "C" int ocnn_conv_wgrad_choose(int dtype, int64_t rows_x, int64_t rows, int K, int ca, int cb,
                                      int identity_table, int has_plan, int plan_max_distinct,
                                      int64_t plan_total, double plan_occupancy) {
  const bool known = dtype == OCNN_F32 || dtype == OCNN_F16 || dtype == OCNN_BF16;
  if (rows >= kPadMinRows && known && (ca % 32 != 0 || cb % 32 != 0)) return OCNN_WGRAD_ZERO_PADDED;
  // (below some 8 k channel pairs a workgroup's 128 k-pair block is mostly zeros and the
  // plan-free kernel is as fast)
  if (identity_table && K == 1 && rows_x == rows && (int64_t)ca * cb >= 8192 &&
      ocnn_conv_dense_wgrad_rw_supported(dtype, rows, ca, cb))
    return OCNN_WGRAD_DENSE_RW;
  if (has_plan && rows_ok(rows, plan_total) && rows * K * 2 < kOffsetLimit) {
    // (32 x 32 and 64 x 64 have planned kernels of their own that are faster still; with channel
    // counts that are not multiples of 64 on the table-row side the pair-plan kernel, which sums
    // exactly ca x cb and only over the pairs, beats zero-padded 64 x 64 blocks on dense tables too)
    // (32 channels on one side, pair plan / planned, us, f16.  Of x, whose 32 x 64 blocks hold the sums of all 27 slots: 32 -> 64
    // on 1.13 M rows 7 % set 135 / 127, 947 k 15 % 127 / 100, 264 k 22 % 86 / 47; 32 -> 96 154 / 225, 150 / 193, but 95 / 65, 324 k
    // 70 % 96 / 78, and on many rows sparse and dense 533 k 30 % 101 / 108, 1.06 M 61 % 213 / 216.  Of g, in half-empty 64 x 64
    // blocks: 1.06 M rows 61 % set, 64 -> 32 228 / 197, 128 -> 32 420 / 406, but 96 -> 32 338 / 384.  Nine slots, 1.13 M rows
    // 16 % set, 32 -> 64 290 / 63, 96 -> 32 253 / 166.  On eight slots the planned kernel is the faster one at every width: 32 -> 64
    // on 947 k rows 15 % set 112 / 44, 128 -> 64 242 / 127, on 290 k 22 % set 124 / 70.)
    const bool narrow = ca != cb && std::min(ca, cb) == 32;
    const bool planned = K == 8 || (narrow && K < 27) ||
                         (narrow && ca == 32 && (cb % 64 == 0 || (plan_occupancy > 0.2 && rows < 400000))) ||
                         (narrow && cb == 32 && ca % 64 == 0 && plan_occupancy > kSparseMaxOccupancy);
    if ((plan_occupancy <= kSparseMaxOccupancy || cb % 64 != 0) && rows >= kSparseMinRows &&
        !(ca == cb && (ca == 32 || ca == 64)) &&
        !(planned && ocnn_conv_wgrad_planned_supported(dtype, rows_x, rows, K, ca, cb, plan_max_distinct)) &&
        ocnn_conv_wgrad_sparse_supported(dtype, rows_x, rows, K, ca, cb, plan_max_distinct))
      return OCNN_WGRAD_SPARSE;
    // (against the plan-free kernel, us: f16 32 -> 64 on 1.06 M rows 61 % set 119 / 775, 64 -> 32 197 / 732, 41 k 26 / 31, but 20 k
    // 22 / 19 and 10 k 18 / 16; fp32 32 -> 64 on 2.3 M rows 60 % set 660 / 5495, 39 k 32 / 85, 17 k 25 / 52, 4.9 k 19 / 41; 64 -> 32 756 / 5179,
    // 30 / 80, 22 / 52, 15 / 41)
    if (!(narrow && dtype != OCNN_F32 && rows < kSparseMinRows) &&
        ocnn_conv_wgrad_planned_supported(dtype, rows_x, rows, K, ca, cb, plan_max_distinct))
      return OCNN_WGRAD_PLANNED;
  }
  return OCNN_WGRAD_PLAIN;
}

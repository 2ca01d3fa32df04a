// Entry points of libocnn_hip.so for this package's own host path (csrc/host.cpp): kernels and
// choices that need more than the arguments the public header fixes.  Same conventions as there.
#pragma once
#include <stdint.h>

#include "ocnn_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

// What follows a layer in evaluation, taken in the same pass: y = (x - mean) / sqrt(var + eps) * gamma + beta
// (+ residual), then max(., 0) with relu.  mean null: nothing follows.  Statistics and parameters in
// f32 / f16 / bf16 (gamma, beta, residual may be null).
typedef struct {
  const void *mean, *var;
  int stat_dtype;
  float eps;
  const void *gamma, *beta;
  int param_dtype, relu;
  const void* residual;
} ocnnx_bn;

// Gather-GEMM on the tile plan, any of the three data types, channels in multiples of 32
// (conv_tile.hip).  The workspace holds the packed weights and, where a launch of few tiles splits
// its reduction, the parts' sums; with less room than ..._workspace_bytes() (but the packed
// weights') it runs in one part.  split_c, split_k: parts over chunks of input channels and over the
// slots; 0 = the library decides.
int ocnnx_gather_tile_supported(int dtype, int64_t rows_in, int K, int cin, int cout, int plan_max_distinct);
int64_t ocnnx_gather_tile_workspace_bytes(int dtype, int64_t rows_out, int K, int cin, int cout);
int ocnnx_gather_tile(int dtype, const void* in, int64_t rows_in, const uint16_t* loc, const int32_t* uptr,
                      const int32_t* urows, int plan_max_distinct, int64_t plan_total, double plan_occupancy,
                      int64_t rows_out, int K, const void* w, int cin, int cout, int w_transposed, int reverse_slots,
                      const void* bias, const ocnnx_bn* bn, void* out, void* workspace, int64_t workspace_bytes,
                      int split_c, int split_k, void* stream);

// The backward pass of a layer whose data gradient is ocnnx_gather_tile's and whose weight gradient is
// ocnn_conv_wgrad_planned's, with the bias gradient (column sums of grad; null: none): as the calls one
// behind the other, but the launches around the two kernels merged into one before and one after them.
typedef struct {
  const void* in;
  int64_t rows_in;
  const uint16_t* loc;
  const int32_t *uptr, *urows;
  int plan_max_distinct;
  int64_t plan_total;
  double plan_occupancy;
  int64_t rows_out;
  int K;
  const void* w;
  int cin, cout, w_transposed, reverse_slots;
  const void* bias;
  const ocnnx_bn* bn;
  void *out, *workspace;
  int64_t workspace_bytes;
  int split_c, split_k;
  const uint8_t* order;       // null, or the tiles' rows in the order of ocnnx_plan_order
  const void* packed;         // null, or the weights as ocnnx_pack_tiles leaves them (ocnnx_gather_tile_packed_bytes)
} ocnnx_gather_args;
int ocnnx_gather_tile_ordered(int K, double plan_occupancy);
int ocnnx_gather_tile_args(int dtype, const ocnnx_gather_args* args, void* stream);   // ocnnx_gather_tile

// ocnn_conv_gather_rw with the batch norm (or null) behind the layer.
int ocnnx_conv_gather_rw(int dtype, const void* in, int64_t rows_in, const uint16_t* loc, const int32_t* uptr,
                         const int32_t* urows, int plan_max_distinct, int64_t plan_total, int64_t rows_out, int K, const void* w,
                         int cin, int cout, int w_transposed, int reverse_slots, const void* bias, const ocnnx_bn* bn, void* out,
                         void* workspace, int64_t workspace_bytes, void* stream);

// The weights of n layers in the order in which ocnnx_gather_tile reads them, in one launch.
#define OCNNX_PACK_MOST 12
typedef struct {
  const void* w;
  void* out;
  int K, cin, cout, transposed, reverse_slots;
} ocnnx_pack_item;
int64_t ocnnx_gather_tile_packed_bytes(int dtype, int K, int cin, int cout);
int ocnnx_pack_tiles(int dtype, const ocnnx_pack_item* items, int n, void* stream);
typedef struct {
  const void* x;
  int64_t rows_x;
  const void* g;
  const uint16_t* loc;
  const int32_t *uptr, *urows;
  int plan_max_distinct;
  int64_t plan_total, rows;
  int K, ca, cb, out_transposed;
  void *gw, *workspace;
  int64_t workspace_bytes;
} ocnnx_wgrad_args;
int ocnnx_conv_backward(int dtype, const ocnnx_gather_args* dgrad, const ocnnx_wgrad_args* wgrad, const void* grad,
                        int64_t grad_rows, int grad_channels, void* bias_grad, void* colsum_workspace, int64_t colsum_bytes,
                        void* stream);

// ocnn_conv_gather with row i of the result at row out_index[i] (null: i), and with the room that lets a launch of few
// rows split its reduction (with less, but ocnn_conv_gather_workspace_bytes, it runs in one part).
int64_t ocnnx_conv_gather_workspace_bytes(int dtype, int64_t rows_in, int64_t rows_out, int K, int cin, int cout);
int ocnnx_conv_gather(int dtype, const void* in, int64_t rows_in, const int32_t* table, int64_t rows_out, int K,
                      const void* w, int cin, int cout, int w_transposed, int reverse_slots, const void* bias, void* out,
                      const int64_t* out_index, void* workspace, int64_t workspace_bytes, void* stream);

// Dense rows (row i reads row i) of few channels in f16 / bf16: out = in W (+ bias, + the batch norm behind it).
int ocnnx_dense_rows_supported(int dtype, int64_t rows, int cin, int cout);
int ocnnx_dense_rows(int dtype, const void* in, int64_t rows, const void* w, int cin, int cout, int w_transposed,
                     const void* bias, const ocnnx_bn* bn, void* out, void* stream);

// gw = x^T g of fp32 rows, in fp32 throughout (fixed order); any channel counts up to 1024.
int ocnnx_rows_wgrad_supported(int dtype, int64_t rows, int ca, int cb);
int64_t ocnnx_rows_wgrad_workspace_bytes(int64_t rows, int ca, int cb);
int ocnnx_rows_wgrad(int dtype, const void* x, const void* g, int64_t rows, int ca, int cb, int out_transposed, void* gw,
                     void* workspace, int64_t workspace_bytes, void* stream);

// ocnn_conv_gather_choose with ocnnx_gather_tile and ocnnx_dense_rows among the choices.
#define OCNNX_GATHER_TILE 8
#define OCNNX_GATHER_ROWS 9
int ocnnx_gather_choose(int dtype, int64_t rows_in, int64_t rows_out, int K, int cin, int cout, int identity_table,
                        int has_plan, int plan_max_distinct, int64_t plan_total, double plan_occupancy,
                        double plan_reuse, int plan_overflow);

// ocnn_batch_norm_stats and ocnn_batch_norm_apply after each other: one or two launches where there are few rows.  y may be x.
int ocnnx_batch_norm_training(int dtype, const void* x, int64_t rows, int channels, float eps, float* mean, float* var,
                              float* invstd, void* running_mean, void* running_var, int running_dtype, float factor,
                              int64_t* batches_tracked, const void* gamma, const void* beta, int param_dtype, int relu,
                              const void* residual, void* y, void* mask, void* workspace, int64_t workspace_bytes, void* stream);

// Where both directions run in three launches: the size of what mask (or null) takes above, a bit for each value of y that is
// positive.  Else 0, and mask is null.  With it ocnn_batch_norm_backward reads neither y nor, for its mask, x.
int64_t ocnnx_batch_norm_mask_bytes(int dtype, int64_t rows, int channels);
int ocnnx_batch_norm_backward(int dtype, const void* x, const void* dy, int64_t rows, int channels, const float* mean,
                              const float* invstd, const void* gamma, const void* beta, int param_dtype, int relu, int training,
                              const void* y, const void* mask, void* dx, void* d_residual, float* dgamma, float* dbeta,
                              void* grad_gamma, void* grad_beta, void* workspace, int64_t workspace_bytes, void* stream);

// ocnn_batch_norm_apply with a module's running statistics as it holds them (f32 / f16 / bf16).
int ocnnx_batch_norm_running(int dtype, const void* x, int64_t rows, int channels, const void* running_mean,
                             const void* running_var, int running_dtype, float eps, const void* gamma, const void* beta,
                             int param_dtype, int relu, const void* residual, void* y, void* stream);

// Tile plans of n tables in one pass each over all of them (tile0: the tables' tiles numbered one behind the
// other): counts, positions (loc) and, in `pad` entries a tile, the lists of distinct rows; then the
// offsets uptr and the six sizes of ocnn_tile_plan_offsets per table, on the device and in host memory
// that the device writes.  ocnnx_plan_compact moves the lists to urows (null: not of this table).
typedef struct {
  const int32_t* table;
  uint16_t* loc;
  int32_t *uptr, *urows;
  int64_t rows, tile0;
  int K, groups;              // groups: say whether the table is one of sibling groups (csrc/plan.hip), in the second of the sizes
} ocnnx_plan_item;
int ocnnx_plan_build(const ocnnx_plan_item* items, int n, int cap, int pad, int32_t* ucount, int32_t* tile_nnz,
                     int32_t* lists, int64_t* stats, int64_t* host_stats, void* stream);
int ocnnx_plan_compact(const ocnnx_plan_item* items, int n, int cap, int pad, const int32_t* ucount, const int64_t* stats,
                       const int32_t* lists, void* stream);

// The same of one plan, from its positions: tile_marks[tile], zeros before, is nonzero for the tiles of sibling groups.
int ocnnx_plan_siblings(const uint16_t* loc, int64_t rows, int K, int32_t* tile_marks, void* stream);

// Signals of the leaves side by side, in the order of the bits of `parts`: 1 the normal (3), 2 <offset of the mean point from the
// voxel's centre, normal> (1), 4 that offset (3), 8 the mean point * scale - 1 (3); points, normals: (n, 3), null where none is read.
int ocnnx_input_feature(const float* points, const float* normals, int64_t n, int parts, float scale, float* out, void* stream);

// The rows of the tiles of n plans (tile0: as above), 128 numbers below 128 a tile, in the order in which ocnnx_gather_tile takes
// them where it leaves out what is empty (ocnnx_gather_tile_ordered), and behind them of each slot which of the tile's four blocks
// of 32 rows, in that order, have an entry (bits): OCNNX_TILE_ORDER_BYTES a tile.  loc as ocnnx_plan_compact leaves it.
#define OCNNX_TILE_ORDER_BYTES 160
typedef struct {
  const uint16_t* loc;
  uint8_t* order;
  int64_t tiles, tile0;
  int K;
} ocnnx_order_item;
int ocnnx_plan_order(const ocnnx_order_item* items, int n, void* stream);

// The octree build from the points on: normalised points, keys, sort and node counts (sizes: device,
// levels + 1, as ocnn_octree_build_scan); then keys, children and the indices of the non-empty nodes of
// the layers from the deepest full one on (h_index[d], d >= full_depth) and the leaves' mean points and
// normals (normals, out_normals: may be null; rows: 32 bytes a point, from the scan to the fill); then every neighbour table.
int64_t ocnnx_tree_workspace_bytes(int64_t n, int depth, int full_depth, int batch_bits);
int ocnnx_tree_scan(const float* pts, int64_t n, const float* h_bbmin, float factor, const void* batch, int batch_is_float,
                    int depth, int full_depth, int batch_bits, const float* normals, float* rows, void* workspace,
                    int64_t workspace_bytes, int32_t* perm, int64_t* sizes, void* stream);
int ocnnx_tree_fill(const void* workspace, int64_t n, int depth, int full_depth, int batch_size, int batch_bits,
                    const int64_t* h_sizes, const int32_t* perm, int64_t* const* h_keys, int32_t* const* h_children,
                    int32_t* const* h_index, int64_t* inverse, int32_t* seg_start, const float* rows, float* out_pts,
                    float* out_normals, void* stream);
int ocnnx_neigh_all(int depth, int full_depth, int batch, const int64_t* h_nnum, const int64_t* h_nnum_nempty,
                    const int64_t* const* h_keys, const int32_t* const* h_children,
                    const int32_t* const* h_nempty_index, int32_t* const* h_neigh, void* stream);

#ifdef __cplusplus
}
#endif

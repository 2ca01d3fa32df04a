// Entry points of libocnn_hip.so for this package's own host path (csrc/host.cpp): kernels and
// choices that need more than the arguments the public header fixes.  Same conventions as there.
#pragma once
#include <stdint.h>

#include "ocnn_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

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
                      const void* bias, void* out, void* workspace, int64_t workspace_bytes, int split_c, int split_k,
                      void* stream);

// ocnn_conv_gather_choose with that kernel among the choices.
#define OCNNX_GATHER_TILE 8
int ocnnx_gather_choose(int dtype, int64_t rows_in, int64_t rows_out, int K, int cin, int cout, int identity_table,
                        int has_plan, int plan_max_distinct, int64_t plan_total, double plan_occupancy,
                        double plan_reuse);

// ocnn_batch_norm_apply with a module's running statistics as it holds them (f32 / f16 / bf16).
int ocnnx_batch_norm_running(int dtype, const void* x, int64_t rows, int channels, const void* running_mean,
                             const void* running_var, int running_dtype, float eps, const void* gamma, const void* beta,
                             int param_dtype, int relu, const void* residual, void* y, void* stream);

#ifdef __cplusplus
}
#endif

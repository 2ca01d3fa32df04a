// The weight gradient in fp32 on the tile plan (wgrad_f32.hip), for the pass in wgrad_planned.hip.
#pragma once
#include "common.hpp"

namespace ocnn {

struct WfSplit {
  int64_t per, run;                           // tiles of a range (a workgroup's); of a set of sums: per is a multiple
  int groups;                                 // parts of the slots
};
WfSplit wf_split_tiles(int64_t tiles, int K, int ca, int cb, int n_cu);

struct WfArgs {
  const float *x, *g;
  int64_t rows_x, rows, plan_total;
  const uint16_t* loc;
  const int32_t *uptr, *urows;
  int K, ca, cb;
  WfSplit split;
  float* partial;                             // cdiv(tiles, run) sets of (K, ca, cb)
};
void launch_wgrad_f32(const WfArgs& a, hipStream_t st);

}  // namespace ocnn

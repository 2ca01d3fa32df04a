// The weight gradient in fp32 on the tile plan (wgrad_f32.hip), for the pass in wgrad_planned.hip.
#pragma once
#include "common.hpp"

namespace ocnn {

struct WfSplit {
  int64_t per, run;                           // tiles of a range (a workgroup's); of a set of sums: per is a multiple
  int groups;                                 // parts of the slots
  int64_t launch, sets;                       // tiles of a launch; sets of sums of the largest one
};
WfSplit wf_split_tiles(int64_t tiles, int K, int ca, int cb, int n_cu);

// Sets of sums in the workspace: with several launches also the sums of those before, in two places by turns.
inline int64_t wf_workspace_sets(const WfSplit& s, int64_t tiles) { return s.launch < tiles ? s.sets + 2 : s.sets; }

struct WfArgs {
  const float *x, *g;
  int64_t rows_x, rows, plan_total;
  const uint16_t* loc;
  const int32_t *uptr, *urows;
  int K, ca, cb;
  WfSplit split;
  float* partial;                             // cdiv(tiles, run) sets of (K, ca, cb)
};
// (for a part of the tiles: the rows, g, loc and uptr from its first one on)
void launch_wgrad_f32(const WfArgs& a, hipStream_t st);

}  // namespace ocnn

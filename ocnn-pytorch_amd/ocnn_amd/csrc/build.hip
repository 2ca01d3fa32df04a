// Octree construction: the sort of the point keys, the numbering of every layer's nodes in one
// pass over the sorted points, keys and children of all layers, the per-leaf signal averages, and
// the regrowing of an octree from split decisions.
#include <algorithm>
#include <cstring>

#include <rocprim/rocprim.hpp>

#include "common.hpp"
#include "host_api.hpp"
#include "morton.hpp"

namespace ocnn {

__global__ void leaf_mean_kernel(const float* src, int C, const int32_t* perm,
                                 const int32_t* seg_start, int64_t n_leaf, float* out) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_leaf * C) return;
  int64_t leaf = t / C;
  int c = (int)(t % C);
  int32_t s = seg_start[leaf], e = seg_start[leaf + 1];
  float acc = 0.f;
  for (int32_t q = s; q < e; ++q) acc += src[(int64_t)perm[q] * C + c];   // point order
  out[t] = acc / (float)(e - s);
}

__global__ void leaf_normal_kernel(const float* src, const int32_t* perm,
                                   const int32_t* seg_start, int64_t n_leaf, float* out) {
  int64_t leaf = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (leaf >= n_leaf) return;
  int32_t s = seg_start[leaf], e = seg_start[leaf + 1];
  float ax = 0.f, ay = 0.f, az = 0.f;
  for (int32_t q = s; q < e; ++q) {
    const float* p = src + (int64_t)perm[q] * 3;
    ax += p[0];
    ay += p[1];
    az += p[2];
  }
  float nrm = sqrtf(ax * ax + ay * ay + az * az);
  float d = fmaxf(nrm, 1e-12f);
  out[3 * leaf + 0] = ax / d;
  out[3 * leaf + 1] = ay / d;
  out[3 * leaf + 2] = az / d;
}

// both of them for a cloud with normals: a leaf's points are walked once
__global__ void leaf_points_normals_kernel(const float* __restrict__ pts, const float* __restrict__ nrm,
                                           const int32_t* __restrict__ perm, const int32_t* __restrict__ seg_start,
                                           int64_t n_leaf, float* __restrict__ out_pts, float* __restrict__ out_nrm) {
  int64_t leaf = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (leaf >= n_leaf) return;
  const int32_t s = seg_start[leaf], e = seg_start[leaf + 1];
  float px = 0.f, py = 0.f, pz = 0.f, ax = 0.f, ay = 0.f, az = 0.f;
  for (int32_t q = s; q < e; ++q) {
    const int64_t at = (int64_t)perm[q] * 3;
    const float* p = pts + at;
    const float* v = nrm + at;
    px += p[0];
    py += p[1];
    pz += p[2];
    ax += v[0];
    ay += v[1];
    az += v[2];
  }
  const float cnt = (float)(e - s);
  out_pts[3 * leaf + 0] = px / cnt;
  out_pts[3 * leaf + 1] = py / cnt;
  out_pts[3 * leaf + 2] = pz / cnt;
  const float d = fmaxf(sqrtf(ax * ax + ay * ay + az * az), 1e-12f);
  out_nrm[3 * leaf + 0] = ax / d;
  out_nrm[3 * leaf + 1] = ay / d;
  out_nrm[3 * leaf + 2] = az / d;
}

// ---- regrowing an octree from split decisions (generative decoders) ----------------------
__global__ void split_flag_kernel(const int32_t* split, int64_t n, int32_t* flag) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) flag[i] = split[i] != 0;
}

// rank = inclusive count of the split nodes up to i.  A layer in which nothing is split keeps
// node 0 as its one non-empty node (the reference does, so that the next layer is never empty).
__global__ void split_children_kernel(const int32_t* flag, const int32_t* rank, int64_t n,
                                      int32_t* children, int64_t* count) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int32_t total = rank[n - 1];
  int32_t c = flag[i] ? rank[i] - 1 : -1;
  if (total == 0 && i == 0) c = 0;
  children[i] = c;
  if (i == 0) *count = total == 0 ? 1 : total;
}

// Node 8 p + j of the new layer is child j of the p-th non-empty node of the layer above:
// its key is that node's key with j appended below the batch bits; it is numbered as itself.
__global__ void grow_layer_kernel(const int64_t* key_above, const int32_t* nempty_index, int64_t n_out,
                                  int64_t* keys, int32_t* children) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_out) return;
  const int64_t k = key_above[nempty_index[i >> 3]];
  const int64_t low = k & ((1ll << 48) - 1);
  keys[i] = (k - low) | (low << 3) | (i & 7);
  children[i] = (int32_t)i;
}

// ---- the whole tree above the sorted point keys in one scan and one scatter ---------------
// A sorted point starts a new node l layers above the leaves (l = 0: a new leaf) iff its key
// differs from its predecessor's in a bit at or above 3 l, or in the batch id.  Counting those
// starts for all layers together numbers the nodes of every layer in one scan over the points.
constexpr int kBuildMaxDepth = 16;

constexpr int kBuildThreads = 256;   // four waves, each on a run of consecutive points
// Sorted points per workgroup of the counting and the scatter kernel: a thread's points follow each other, so that a cloud
// too small to fill the chip is cut finer.  The line: counts, offsets and scatter in us, spans of 1024 / 256 points, of a sphere
// 20 k points depth 6 24.2 / 14.9, 65 k depth 7 25.3 / 18.8, 100 k depth 6 31.4 / 19.9, 131 k depth 7 28.5 / 21.4, 262 k depths 7
// and 8 31.0 / 26.6, 29.1 / 27.4, 400 k depth 7 36.0 / 36.1, 524 k depths 7 and 8 40.6 / 42.2, 36.4 / 42.4, 1 M depth 9 57.6 /
// 81.8 (the one workgroup of the offsets has four times the spans to add: 5.2 / 15.7 us of these).
constexpr int kBuildSpan = 1024, kBuildSmallSpan = 256;
constexpr int64_t kBuildSmallPoints = 1 << 18;
static int build_span(int64_t n) { return n <= kBuildSmallPoints ? kBuildSmallSpan : kBuildSpan; }

// number of layers at which sorted point i starts a node, minus one (-1: same leaf as i - 1)
template <typename K>
__device__ inline int start_level(const K* __restrict__ sorted, int64_t i, int key_bits, int levels) {
  if (i == 0) return levels;
  const K x = sorted[i] ^ sorted[i - 1];
  if (x == 0) return -1;
  const int hb = 63 - __builtin_clzll((unsigned long long)x);
  if (hb >= key_bits) return levels;
  const int l = hb / 3;
  return l < levels ? l : levels;
}

__device__ inline uint32_t lanes_below(unsigned long long mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// starts of nodes, by layer, among the points of each workgroup's span: sums[span][N]
template <typename K, int N, int SPAN>
__global__ __launch_bounds__(kBuildThreads) void build_count_kernel(const K* __restrict__ sorted, int64_t n,
                                                                    int key_bits, int levels,
                                                                    uint32_t* __restrict__ sums) {
  __shared__ uint32_t s_cnt[kBuildThreads / 64][N];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t base = (int64_t)blockIdx.x * SPAN + wave * (SPAN / 4);
  uint32_t cnt[N];
#pragma unroll
  for (int l = 0; l < N; ++l) cnt[l] = 0u;
#pragma unroll
  for (int it = 0; it < SPAN / kBuildThreads; ++it) {
    const int64_t q = base + it * 64 + lane;
    const int lv = q < n ? start_level(sorted, q, key_bits, levels) : -1;
#pragma unroll
    for (int l = 0; l < N; ++l) cnt[l] += (uint32_t)__popcll(__ballot(lv >= l));
  }
  if (lane == 0) {
#pragma unroll
    for (int l = 0; l < N; ++l) s_cnt[wave][l] = cnt[l];
  }
  __syncthreads();
  if (threadIdx.x < N) {
    uint32_t c = 0u;
    for (int w = 0; w < kBuildThreads / 64; ++w) c += s_cnt[w][threadIdx.x];
    sums[(int64_t)blockIdx.x * N + threadIdx.x] = c;
  }
}

// offs[span][l] = starts at layer l before the span; sizes[l] = their total.  One workgroup: thread
// (chunk, l) walks a chunk of spans twice, the chunks' totals meet in LDS in between.
template <int N>
__global__ __launch_bounds__(1024) void build_offsets_kernel(const uint32_t* __restrict__ sums, int64_t spans,
                                                             int levels, uint32_t* __restrict__ offs,
                                                             int64_t* __restrict__ sizes) {
  constexpr int kChunks = 1024 / N;
  __shared__ uint32_t s_tot[kChunks][N];
  const int l = threadIdx.x % N, c = threadIdx.x / N;
  const int64_t per = (spans + kChunks - 1) / kChunks;
  const int64_t lo = c * per < spans ? c * per : spans, hi = lo + per < spans ? lo + per : spans;
  uint32_t tot = 0u;
  for (int64_t b = lo; b < hi; ++b) tot += sums[b * N + l];
  s_tot[c][l] = tot;
  __syncthreads();
  uint32_t run = 0u;
  for (int cc = 0; cc < c; ++cc) run += s_tot[cc][l];
  // (host memory in a build from points, whose host side watches for the values)
  if (c == kChunks - 1 && l <= levels)
    __hip_atomic_store(&sizes[l], (int64_t)(run + tot), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  for (int64_t b = lo; b < hi; ++b) {
    offs[b * N + l] = run;
    run += sums[b * N + l];
  }
}

struct BuildTree {
  int64_t* keys[kBuildMaxDepth + 1];
  int32_t* children[kBuildMaxDepth + 1];
  int64_t begin[kBuildMaxDepth + 2];   // running total of the node counts, by depth
  int32_t* index[kBuildMaxDepth + 1];  // (optional) the non-empty nodes of the layers from the deepest full one on
};

// Signals to be averaged over the leaves (or none): a point's 32 bytes are its point and normal, one line of memory to a
// fetch in sorted order where two arrays of 12 bytes are two or four (build of 1 M points at depth 9 192 us, so 172).
struct BuildSignal {
  const float4* rows;
  float *out_pts, *out_nrm;      // (out_nrm may be null)
};

// Full layers, and -1 in the children of every other layer.  Four nodes a thread (the layers below the
// full ones are whole groups of eight, and so are the full ones from layer 1 on).
__global__ void build_init_kernel(BuildTree t, int depth, int full_depth) {
  const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (i >= t.begin[depth + 1] - t.begin[1] + 4 * ((t.begin[1] + 3) / 4)) return;
  const int64_t root = 4 * ((t.begin[1] + 3) / 4);            // layer 0 (a node per octree) padded to groups of four
  if (i < root) {
    for (int64_t j = i; j < i + 4 && j < t.begin[1]; ++j) {
      t.keys[0][j] = j << 48;
      t.children[0][j] = full_depth > 0 ? (int32_t)j : -1;
    }
    return;
  }
  const int64_t at = i - root + t.begin[1];
  int d = 1;
  while (at >= t.begin[d + 1]) ++d;
  const int64_t j = at - t.begin[d];
  int4 c = make_int4(-1, -1, -1, -1);
  if (d <= full_depth) {
#pragma unroll
    for (int u = 0; u < 4; ++u) t.keys[d][j + u] = ((j + u) & ((1ll << (3 * d)) - 1)) | (((j + u) >> (3 * d)) << 48);
    if (d < full_depth) c = make_int4((int)j, (int)j + 1, (int)j + 2, (int)j + 3);
  }
  *(int4*)(t.children[d] + j) = c;
}

struct OpenLeaf {                // a leaf whose points a span does not hold all: its signals' sums so far
  uint64_t key;
  int64_t leaf;
  int count;
  float sum[6];
};

// mean point and normal of a leaf from the sums over its points
__device__ __forceinline__ void leaf_signals(const BuildSignal& sig, int64_t leaf, const float* a, int64_t points) {
  const float cnt = (float)points;
#pragma unroll
  for (int e = 0; e < 3; ++e) sig.out_pts[3 * leaf + e] = a[e] / cnt;
  if (sig.out_nrm) {
    const float len = fmaxf(sqrtf(a[3] * a[3] + a[4] * a[4] + a[5] * a[5]), 1e-12f);
#pragma unroll
    for (int e = 0; e < 3; ++e) sig.out_nrm[3 * leaf + e] = a[3 + e] / len;
  }
}

// Numbers every point's nodes (its span's offsets + the starts before it inside the span, counted
// with wave ballots) and writes what the point starts: a leaf's entry in its parent's children, a
// parent's eight keys, and so on up to the deepest full layer.  With signals, also the leaves' mean points and
// normals: every thread fetches its points' 24 bytes, side by side with everything else, and the thread that starts a
// leaf adds them from LDS in the order of the points (a launch of its own walked a leaf's points one behind the other,
// each from memory: 5.6 us of them for 20 k points at depth 6).  The leaf that goes on in the spans behind is the whole
// workgroup's: one thread walking on from memory waited for key, point number and signals of every point in turn.  Builds in us,
// launch of its own / walked on / now: 1 M points of a cube at depth 2 9100 / 5680 / 570, depth 3 1870 / 1290 / 240, depth 4
// 360 / 285 / 187; of a sphere at depth 5 460 / 428 / 207, depth 6 217 / 220 / 174, 3 M 508 / 600 / 372; 200 k points of one
// cell 30300 / 51400 / 4580, one chain of additions.  (Where the next span starts a leaf, as most do, nothing follows the walk:
// with the further points asked for in every span a build of 1 M points at depth 9 took 6 us more.)
template <typename K, int N, int SPAN>
__global__ __launch_bounds__(kBuildThreads) void build_scatter_kernel(
    const K* __restrict__ sorted, const uint32_t* __restrict__ offs, const int32_t* __restrict__ perm, int64_t n,
    int key_bits, int depth, int full_depth, BuildTree t, BuildSignal sig, int64_t* __restrict__ inverse,
    int32_t* __restrict__ seg_start) {
  __shared__ uint32_t s_cnt[kBuildThreads / 64][N];
  __shared__ __attribute__((aligned(16))) float s_sig[6][SPAN];
  __shared__ uint8_t s_new[SPAN];                            // the point starts a leaf (or is none)
  __shared__ OpenLeaf s_open;
  constexpr int kIt = SPAN / kBuildThreads;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t base = (int64_t)blockIdx.x * SPAN + wave * (SPAN / 4);
  const int levels = depth - full_depth;
  const int64_t behind = ((int64_t)blockIdx.x + 1) * SPAN;
  const bool goes_on = sig.rows && behind < n && sorted[behind] == sorted[behind - 1];   // a leaf does, in the span behind
  if (threadIdx.x == 0) s_open.leaf = -1;
  int lv[kIt], at[kIt];
  uint32_t run[N];
#pragma unroll
  for (int it = 0; it < kIt; ++it) {
    const int64_t q = base + it * 64 + lane;
    at[it] = q < n ? perm[q] : -1;
  }
  float4 v[kIt][2];
#pragma unroll
  for (int it = 0; it < kIt; ++it) {
    v[it][0] = v[it][1] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (at[it] >= 0 && sig.rows) {
      v[it][0] = sig.rows[2 * (int64_t)at[it]];
      if (sig.out_nrm) v[it][1] = sig.rows[2 * (int64_t)at[it] + 1];
    }
  }
#pragma unroll
  for (int l = 0; l < N; ++l) run[l] = 0u;
#pragma unroll
  for (int it = 0; it < kIt; ++it) {
    const int64_t q = base + it * 64 + lane;
    lv[it] = q < n ? start_level(sorted, q, key_bits, levels) : -1;
#pragma unroll
    for (int l = 0; l < N; ++l) run[l] += (uint32_t)__popcll(__ballot(lv[it] >= l));
  }
  if (lane == 0) {
#pragma unroll
    for (int l = 0; l < N; ++l) s_cnt[wave][l] = run[l];
  }
#pragma unroll
  for (int it = 0; it < kIt; ++it) {
    const int j = wave * (SPAN / 4) + it * 64 + lane;
    s_new[j] = at[it] < 0 || lv[it] >= 0 ? 1 : 0;
    s_sig[0][j] = v[it][0].x, s_sig[1][j] = v[it][0].y, s_sig[2][j] = v[it][0].z;
    s_sig[3][j] = v[it][0].w, s_sig[4][j] = v[it][1].x, s_sig[5][j] = v[it][1].y;
  }
  __syncthreads();
#pragma unroll
  for (int l = 0; l < N; ++l) {
    uint32_t r = offs[(int64_t)blockIdx.x * N + l];
    for (int w = 0; w < wave; ++w) r += s_cnt[w][l];
    run[l] = r;
  }
#pragma unroll
  for (int it = 0; it < kIt; ++it) {
    const int64_t q = base + it * 64 + lane;
    uint32_t s[N];                      // inclusive: nodes of layer l started up to and with this point
#pragma unroll
    for (int l = 0; l < N; ++l) {
      const unsigned long long mask = __ballot(lv[it] >= l);
      s[l] = run[l] + lanes_below(mask) + (lv[it] >= l ? 1u : 0u);
      run[l] += (uint32_t)__popcll(mask);
    }
    if (q >= n) continue;
    const int32_t leaf = (int32_t)s[0] - 1;
    inverse[at[it]] = leaf;
    if (q == n - 1) seg_start[leaf + 1] = (int32_t)n;
    if (lv[it] < 0) continue;
    seg_start[leaf] = (int32_t)q;
    const uint64_t c = (uint64_t)sorted[q];
    const int64_t b = (int64_t)(c >> key_bits);
    const int64_t m = (int64_t)(c & ((1ull << key_bits) - 1));
    uint32_t top = 0u;
#pragma unroll
    for (int l = 0; l < N; ++l) {
      if (l == levels) top = s[l];
      if (l < N - 1 && l < levels && l <= lv[it]) {
        const int d = depth - l;
        const int64_t kl = m >> (3 * l);
        const int64_t p = (int64_t)s[l + 1 < N ? l + 1 : l] - 1;
        t.children[d][(p << 3) | (kl & 7)] = (int32_t)s[l] - 1;
        if (t.index[d]) t.index[d][s[l] - 1] = (int32_t)((p << 3) | (kl & 7));
        if (l + 1 <= lv[it]) {
          const int64_t first = (b << 48) | ((kl >> 3) << 3);
          int64_t* dst = t.keys[d] + (p << 3);
#pragma unroll
          for (int j = 0; j < 8; ++j) dst[j] = first + j;
        }
      }
    }
    if (lv[it] >= levels) {
      const int64_t node = (b << (3 * full_depth)) | (m >> (3 * levels));
      if (node < t.begin[full_depth + 1] - t.begin[full_depth]) {    // a batch id beyond batch_size has no node
        t.children[full_depth][node] = (int32_t)top - 1;
        if (t.index[full_depth]) t.index[full_depth][top - 1] = (int32_t)node;
      }
    }
    if (!sig.rows) continue;
    float a[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    int j = wave * (SPAN / 4) + it * 64 + lane;
    const int from = j;
    do {
#pragma unroll
      for (int e = 0; e < 6; ++e) a[e] += s_sig[e][j];
      ++j;
    } while (j < SPAN && !s_new[j]);
    if (j < SPAN || !goes_on) {
      leaf_signals(sig, leaf, a, j - from);
    } else {                                                 // (one leaf of the span at most)
      s_open.key = c;
      s_open.leaf = leaf;
      s_open.count = j - from;
#pragma unroll
      for (int e = 0; e < 6; ++e) s_open.sum[e] = a[e];
    }
  }
  if (!goes_on) return;
  // The leaf whose further points lie in the spans behind: 256 of them at a time to LDS, and six threads add their signals, in
  // the order of the points
  __syncthreads();
  const int64_t leaf = s_open.leaf;
  if (leaf < 0) return;
  const K key = (K)s_open.key;
  int64_t count = s_open.count;
  float a = threadIdx.x < 6 ? s_open.sum[threadIdx.x] : 0.f;
  for (int64_t first = behind;; first += kBuildThreads) {
    const int64_t q = first + threadIdx.x;
    const K k = q < n ? sorted[q] : (K)0;
    const int32_t point = q < n ? perm[q] : 0;               // (beside the key, not behind it)
    const bool mine = q < n && k == key;                     // (the points are sorted: the first so many threads)
    float4 u = make_float4(0.f, 0.f, 0.f, 0.f), w = u;
    if (mine) {
      const float4* row = sig.rows + 2 * (int64_t)point;
      u = row[0];
      if (sig.out_nrm) w = row[1];
    }
    s_sig[0][threadIdx.x] = u.x, s_sig[1][threadIdx.x] = u.y, s_sig[2][threadIdx.x] = u.z;
    s_sig[3][threadIdx.x] = u.w, s_sig[4][threadIdx.x] = w.x, s_sig[5][threadIdx.x] = w.y;
    const int more = __syncthreads_count(mine);
    if (threadIdx.x < 6) {
#pragma unroll 4
      for (int j = 0; j < more; j += 4) {
        const float4 v = *(const float4*)&s_sig[threadIdx.x][j];
        a += v.x;
        if (j + 1 < more) a += v.y;
        if (j + 2 < more) a += v.z;
        if (j + 3 < more) a += v.w;
      }
    }
    count += more;
    __syncthreads();
    if (more < kBuildThreads) break;
  }
  if (threadIdx.x < 6) s_open.sum[threadIdx.x] = a;
  __syncthreads();
  if (threadIdx.x == 0) leaf_signals(sig, leaf, s_open.sum, count);
}

using ForceOnesweep = rocprim::radix_sort_config<rocprim::default_config, rocprim::default_config,
                                                 rocprim::default_config, 0>;

// counts of the spans, and what the scatter does with the points of a span (build_span)
template <typename K, int N>
static void launch_build_count(const K* csorted, int64_t n, int64_t spans, int key_bits, int levels, uint32_t* sums,
                               hipStream_t st) {
  hipLaunchKernelGGL((build_span(n) == kBuildSpan ? build_count_kernel<K, N, kBuildSpan> : build_count_kernel<K, N, kBuildSmallSpan>),
                     dim3((unsigned)spans), dim3(kBuildThreads), 0, st, csorted, n, key_bits, levels, sums);
}

struct BuildLayout {
  int64_t csorted, sums, offs, temp, temp_bytes, total, spans;
};

// batch id packed right above the Morton bits, read straight from the 64-bit keys by the sort
template <typename K>
struct PackKey {
  int key_bits;
  __host__ __device__ K operator()(int64_t key) const {
    const uint64_t k = (uint64_t)key;
    return (K)(((k >> 48) << key_bits) | (k & ((1ull << key_bits) - 1)));
  }
};

template <typename K, int N>
static int build_layout_t(int64_t n, BuildLayout* L) {
  size_t sort_bytes = 0;
  auto kin = rocprim::make_transform_iterator((const int64_t*)nullptr, PackKey<K>{0});
  auto vin = rocprim::make_counting_iterator<int32_t>(0);
  hipError_t e = rocprim::radix_sort_pairs<ForceOnesweep>(nullptr, sort_bytes, kin, (K*)nullptr, vin,
                                                          (int32_t*)nullptr, (size_t)n, 0, 8 * sizeof(K));
  if (e != hipSuccess) return OCNN_ERR_HIP;
  L->spans = cdiv(n, build_span(n));
  int64_t off = 0;
  L->csorted = off; off += align_up(n * (int64_t)sizeof(K), 256);
  L->sums = off;    off += align_up(L->spans * N * 4, 256);
  L->offs = off;    off += align_up(L->spans * N * 4, 256);
  L->temp = off;
  L->temp_bytes = align_up((int64_t)sort_bytes + 256, 256);
  L->total = off + L->temp_bytes;
  return OCNN_OK;
}

template <typename K, int N>
static int build_scan_t(const int64_t* key, int64_t n, int key_bits, int batch_bits, int levels, char* ws,
                        int64_t ws_bytes, int32_t* perm, int64_t* sizes, hipStream_t st) {
  BuildLayout L;
  if (build_layout_t<K, N>(n, &L) != OCNN_OK) { set_error("octree_build_scan: rocprim size query failed"); return OCNN_ERR_HIP; }
  if (ws_bytes < L.total) { set_error("octree_build_scan: workspace %lld < %lld", (long long)ws_bytes, (long long)L.total); return OCNN_ERR_WORKSPACE; }
  K* csorted = (K*)(ws + L.csorted);
  uint32_t* sums = (uint32_t*)(ws + L.sums);
  uint32_t* offs = (uint32_t*)(ws + L.offs);
  size_t tb = (size_t)L.temp_bytes;
  auto kin = rocprim::make_transform_iterator(key, PackKey<K>{key_bits});
  auto vin = rocprim::make_counting_iterator<int32_t>(0);
  hipError_t e = rocprim::radix_sort_pairs<ForceOnesweep>(ws + L.temp, tb, kin, csorted, vin, perm, (size_t)n, 0u,
                                                          (unsigned)(key_bits + batch_bits), st);
  if (e != hipSuccess) { set_error("octree_build_scan: radix sort: %s", hipGetErrorString(e)); return OCNN_ERR_HIP; }
  launch_build_count<K, N>(csorted, n, L.spans, key_bits, levels, sums, st);
  hipLaunchKernelGGL(build_offsets_kernel<N>, dim3(1), dim3(1024), 0, st, sums, L.spans, levels, offs, sizes);
  return check_launch("octree_build_scan");
}

template <typename K, int N>
static int build_fill_t(const char* ws, int64_t n, int key_bits, int depth, int full_depth, const BuildTree& t,
                        const int32_t* perm, const BuildSignal& sig, int64_t* inverse, int32_t* seg_start, hipStream_t st) {
  BuildLayout L;
  if (build_layout_t<K, N>(n, &L) != OCNN_OK) { set_error("octree_build_fill: rocprim size query failed"); return OCNN_ERR_HIP; }
  const K* csorted = (const K*)(ws + L.csorted);
  const uint32_t* offs = (const uint32_t*)(ws + L.offs);
  hipLaunchKernelGGL(build_init_kernel, dim3((unsigned)cdiv(t.begin[depth + 1] + 4, 1024)), dim3(256), 0, st, t, depth,
                     full_depth);
  hipLaunchKernelGGL((build_span(n) == kBuildSpan ? build_scatter_kernel<K, N, kBuildSpan> : build_scatter_kernel<K, N, kBuildSmallSpan>),
                     dim3((unsigned)L.spans), dim3(kBuildThreads), 0, st, csorted, offs, perm, n, key_bits, depth, full_depth, t,
                     sig, inverse, seg_start);
  return check_launch("octree_build_fill");
}

// key type and counter count of a build: 32-bit sort keys when batch id and Morton bits fit
#define OCNN_BUILD_DISPATCH(CALL)                                   \
  do {                                                               \
    const bool narrow = key_bits + batch_bits <= 32;                 \
    if (levels + 1 <= 8) {                                           \
      if (narrow) return CALL(uint32_t, 8); else return CALL(uint64_t, 8);   \
    } else {                                                         \
      if (narrow) return CALL(uint32_t, 16); else return CALL(uint64_t, 16); \
    }                                                                \
  } while (0)

struct LevelLayout {
  int64_t flag, uid, temp, temp_bytes, total;
};

static int level_layout(int64_t n, LevelLayout* L) {
  size_t scan_bytes = 0;
  hipError_t e = rocprim::inclusive_scan(nullptr, scan_bytes, (int32_t*)nullptr,
                                         (int32_t*)nullptr, (size_t)n, rocprim::plus<int32_t>());
  if (e != hipSuccess) return OCNN_ERR_HIP;
  int64_t off = 0;
  L->flag = off; off += align_up(n * 4, 256);
  L->uid = off;  off += align_up(n * 4, 256);
  L->temp = off;
  L->temp_bytes = align_up((int64_t)scan_bytes + 256, 256);
  L->total = off + L->temp_bytes;
  return OCNN_OK;
}

}  // namespace ocnn

using namespace ocnn;

extern "C" int64_t ocnn_build_level_workspace_bytes(int64_t n) {
  if (n <= 0) return 256;
  LevelLayout L;
  if (level_layout(n, &L) != OCNN_OK) return -1;
  return L.total;
}

// A full layer: every node of every octree of the batch exists, in key order.
__global__ void full_layer_kernel(int depth, int64_t total, int32_t child_fill, int64_t* __restrict__ keys,
                                  int32_t* __restrict__ children) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int64_t b = i >> (3 * depth);
  keys[i] = (i & ((1ll << (3 * depth)) - 1)) | (b << 48);
  children[i] = child_fill < 0 ? child_fill : (int32_t)i;
}

extern "C" int ocnn_build_full_layer(int depth, int batch_size, int with_children, int64_t* keys,
                                     int32_t* children, void* stream) {
  OCNN_REQUIRE(depth >= 0 && depth <= 8 && batch_size >= 1 && ((int64_t)batch_size << (3 * depth)) < (1ll << 31),
               "build_full_layer: depth=%d batch_size=%d out of range", depth, batch_size);
  OCNN_REQUIRE_PTRS("build_full_layer", keys, children);
  const int64_t total = (int64_t)batch_size << (3 * depth);
  hipLaunchKernelGGL(full_layer_kernel, dim3((unsigned)cdiv(total, 256)), dim3(256), 0, (hipStream_t)stream, depth,
                     total, with_children ? 0 : -1, keys, children);
  return check_launch("build_full_layer");
}

extern "C" int ocnn_split_children(const int32_t* split, int64_t n, void* workspace, int64_t workspace_bytes,
                                   int32_t* children, int64_t* count, void* stream) {
  OCNN_REQUIRE(n > 0 && n < (1ll << 28), "split_children: n=%lld out of range", (long long)n);
  OCNN_REQUIRE_PTRS("split_children", split, workspace, children, count);
  LevelLayout L;
  if (level_layout(n, &L) != OCNN_OK) { set_error("split_children: rocprim size query failed"); return OCNN_ERR_HIP; }
  if (workspace_bytes < L.total) { set_error("split_children: workspace %lld < %lld", (long long)workspace_bytes, (long long)L.total); return OCNN_ERR_WORKSPACE; }
  hipStream_t st = (hipStream_t)stream;
  char* ws = (char*)workspace;
  int32_t* flag = (int32_t*)(ws + L.flag);
  int32_t* rank = (int32_t*)(ws + L.uid);
  dim3 grid(cdiv(n, 256)), block(256);
  hipLaunchKernelGGL(split_flag_kernel, grid, block, 0, st, split, n, flag);
  size_t tb = (size_t)L.temp_bytes;
  hipError_t e = rocprim::inclusive_scan(ws + L.temp, tb, flag, rank, (size_t)n, rocprim::plus<int32_t>(), st);
  if (e != hipSuccess) { set_error("split_children: scan: %s", hipGetErrorString(e)); return OCNN_ERR_HIP; }
  hipLaunchKernelGGL(split_children_kernel, grid, block, 0, st, flag, rank, n, children, count);
  return check_launch("split_children");
}

extern "C" int ocnn_grow_layer(const int64_t* key_above, const int32_t* nempty_index, int64_t n_nempty,
                               int64_t* keys, int32_t* children, void* stream) {
  OCNN_REQUIRE(n_nempty > 0 && n_nempty < (1ll << 28), "grow_layer: n_nempty=%lld out of range",
               (long long)n_nempty);
  OCNN_REQUIRE_PTRS("grow_layer", key_above, nempty_index, keys, children);
  hipLaunchKernelGGL(grow_layer_kernel, dim3(cdiv(8 * n_nempty, 256)), dim3(256), 0, (hipStream_t)stream,
                     key_above, nempty_index, 8 * n_nempty, keys, children);
  return check_launch("grow_layer");
}

extern "C" int ocnn_leaf_average(const float* src, int channels, const int32_t* perm,
                                 const int32_t* seg_start, int64_t n_leaf, int mode, float* out,
                                 void* stream) {
  OCNN_REQUIRE(channels > 0 && n_leaf > 0, "leaf_average: channels=%d n_leaf=%lld", channels,
               (long long)n_leaf);
  OCNN_REQUIRE_PTRS("leaf_average", src, perm, seg_start, out);
  hipStream_t st = (hipStream_t)stream;
  if (mode == 1) {
    OCNN_REQUIRE(channels == 3, "leaf_average: normalise mode needs 3 channels, got %d", channels);
    hipLaunchKernelGGL(leaf_normal_kernel, dim3(cdiv(n_leaf, 256)), dim3(256), 0, st, src, perm,
                       seg_start, n_leaf, out);
  } else {
    hipLaunchKernelGGL(leaf_mean_kernel, dim3(cdiv(n_leaf * channels, 256)), dim3(256), 0, st, src,
                       channels, perm, seg_start, n_leaf, out);
  }
  return check_launch("leaf_average");
}

extern "C" int ocnn_leaf_points_normals(const float* pts, const float* normals, const int32_t* perm,
                                        const int32_t* seg_start, int64_t n_leaf, float* out_pts, float* out_normals,
                                        void* stream) {
  OCNN_REQUIRE(n_leaf > 0, "leaf_points_normals: n_leaf=%lld", (long long)n_leaf);
  OCNN_REQUIRE_PTRS("leaf_points_normals", pts, normals, perm, seg_start, out_pts, out_normals);
  hipLaunchKernelGGL(leaf_points_normals_kernel, dim3((unsigned)cdiv(n_leaf, 256)), dim3(256), 0, (hipStream_t)stream,
                     pts, normals, perm, seg_start, n_leaf, out_pts, out_normals);
  return check_launch("leaf_points_normals");
}

// ---- fused build ---------------------------------------------------------------------------
static int build_args_ok(int64_t n, int depth, int full_depth, int batch_bits) {
  OCNN_REQUIRE(n > 0 && n < (1ll << 31), "octree_build: n=%lld out of range", (long long)n);
  OCNN_REQUIRE(depth >= 1 && depth <= kBuildMaxDepth && full_depth >= 0 && full_depth <= depth && full_depth <= 8,
               "octree_build: depth=%d full_depth=%d out of range", depth, full_depth);
  OCNN_REQUIRE(batch_bits >= 0 && batch_bits <= 15, "octree_build: batch_bits=%d out of range", batch_bits);
  // (a point counts its node starts in depth - full_depth + 1 layers, sixteen counters at most)
  OCNN_REQUIRE(depth - full_depth + 1 <= 16, "octree_build: %d layers below the full ones, at most 15",
               depth - full_depth);
  return OCNN_OK;
}

extern "C" int64_t ocnn_octree_build_workspace_bytes(int64_t n, int depth, int full_depth, int batch_bits) {
  if (n <= 0 || depth < 1 || depth > kBuildMaxDepth || full_depth < 0 || full_depth > depth ||
      depth - full_depth + 1 > 16)
    return -1;
  const int key_bits = 3 * depth, levels = depth - full_depth;
  BuildLayout L;
#define OCNN_BUILD_BYTES(K, N) (build_layout_t<K, N>(n, &L) == OCNN_OK ? L.total : (int64_t)-1)
  OCNN_BUILD_DISPATCH(OCNN_BUILD_BYTES);
#undef OCNN_BUILD_BYTES
}

extern "C" int ocnn_octree_build_scan(const int64_t* key, int64_t n, int depth, int full_depth, int batch_bits,
                                      void* workspace, int64_t workspace_bytes, int32_t* perm, int64_t* sizes,
                                      void* stream) {
  if (int rc = build_args_ok(n, depth, full_depth, batch_bits)) return rc;
  OCNN_REQUIRE_PTRS("octree_build_scan", key, workspace, perm, sizes);
  const int key_bits = 3 * depth, levels = depth - full_depth;
#define OCNN_BUILD_SCAN(K, N) \
  build_scan_t<K, N>(key, n, key_bits, batch_bits, levels, (char*)workspace, workspace_bytes, perm, sizes, (hipStream_t)stream)
  OCNN_BUILD_DISPATCH(OCNN_BUILD_SCAN);
#undef OCNN_BUILD_SCAN
}

static int build_fill(const void* workspace, int64_t n, int depth, int full_depth, int batch_size, int batch_bits,
                      const int64_t* h_sizes, const int32_t* perm, int64_t* const* h_keys, int32_t* const* h_children,
                      int32_t* const* h_index, const BuildSignal& sig, int64_t* inverse, int32_t* seg_start, void* stream) {
  if (int rc = build_args_ok(n, depth, full_depth, batch_bits)) return rc;
  OCNN_REQUIRE(batch_size >= 1 && batch_size <= (1 << batch_bits) && ((int64_t)batch_size << (3 * full_depth)) < (1ll << 31),
               "octree_build_fill: batch_size=%d does not fit batch_bits=%d / full_depth=%d", batch_size, batch_bits,
               full_depth);
  OCNN_REQUIRE_PTRS("octree_build_fill", workspace, h_sizes, perm, h_keys, h_children, inverse, seg_start);
  const int key_bits = 3 * depth, levels = depth - full_depth;
  BuildTree t;
  t.begin[0] = 0;
  for (int d = 0; d <= depth; ++d) {
    const int64_t nnum = d <= full_depth ? ((int64_t)batch_size << (3 * d)) : 8 * h_sizes[depth - d + 1];
    OCNN_REQUIRE(nnum > 0 && nnum < (1ll << 31) && h_keys[d] && h_children[d],
                 "octree_build_fill: depth %d: %lld nodes or a missing array", d, (long long)nnum);
    t.keys[d] = h_keys[d];
    t.children[d] = h_children[d];
    t.index[d] = h_index ? h_index[d] : nullptr;
    t.begin[d + 1] = t.begin[d] + nnum;
  }
  OCNN_REQUIRE(h_sizes[levels] <= ((int64_t)batch_size << (3 * full_depth)),
               "octree_build_fill: %lld nodes at the deepest full layer of %d octrees", (long long)h_sizes[levels],
               batch_size);
#define OCNN_BUILD_FILL(K, N) \
  build_fill_t<K, N>((const char*)workspace, n, key_bits, depth, full_depth, t, perm, sig, inverse, seg_start, (hipStream_t)stream)
  OCNN_BUILD_DISPATCH(OCNN_BUILD_FILL);
#undef OCNN_BUILD_FILL
}

extern "C" int ocnn_octree_build_fill(const void* workspace, int64_t n, int depth, int full_depth, int batch_size,
                                      int batch_bits, const int64_t* h_sizes, const int32_t* perm,
                                      int64_t* const* h_keys, int32_t* const* h_children, int64_t* inverse,
                                      int32_t* seg_start, void* stream) {
  return build_fill(workspace, n, depth, full_depth, batch_size, batch_bits, h_sizes, perm, h_keys, h_children, nullptr,
                    BuildSignal{}, inverse, seg_start, stream);
}

extern "C" int ocnnx_tree_fill(const void* workspace, int64_t n, int depth, int full_depth, int batch_size, int batch_bits,
                               const int64_t* h_sizes, const int32_t* perm, int64_t* const* h_keys,
                               int32_t* const* h_children, int32_t* const* h_index, int64_t* inverse, int32_t* seg_start,
                               const float* rows, float* out_pts, float* out_normals, void* stream) {
  OCNN_REQUIRE_PTRS("tree_fill", h_index, rows, out_pts);
  return build_fill(workspace, n, depth, full_depth, batch_size, batch_bits, h_sizes, perm, h_keys, h_children, h_index,
                    BuildSignal{(const float4*)rows, out_pts, out_normals}, inverse, seg_start, stream);
}

// ---- keys and sort ----------------------------------------------------------------------------
// The library's radix sort takes 95 us for 20 000 points (five kernels of 15 us, most of it the chains
// of its decoupled look-back, and seven fills), four times what its bytes cost.  Here a
// cloud is a number of spans of kSortSpan points and a pass is counts of the digit by span, then one stable
// scatter.  Digits have up to 11 bits: a depth-6 octree takes two passes, depth 9 with eight clouds three.
// Up to kSortInlineSpans spans every workgroup of the scatter reads the counts of all spans itself; more of
// them are scanned by a launch in between.  Keys to counted nodes, the launches back to back, itself / scanned:
// 24 spans 31 / 33 us at depth 5, 33 / 34 at 6, 44 / 40 at 7, 46 / 48 at 9; 64 spans 38 / 34, 40 / 36, 63 / 41, 57 / 51; 128
// spans 50 / 37, 53 / 39, 95 / 47, 76 / 55.  The line is behind that crossing because a build waits for its sizes, and
// two launches more in front of the wait cost it 10 - 35 us: build and tables of 45 k points at depth 6 126 / 163 us, 60 k at
// depth 7 149 / 168, 131 k at depth 6 135 / 141; 100 k at depth 7 159 / 152, 131 k at depth 8 181 / 176.
constexpr int kSortSpan = 2048;
constexpr int kSortThreads = 256, kSortItems = kSortSpan / kSortThreads;
constexpr int kSortMaxBits = 11;
constexpr int kSortInlineSpans = 64;
constexpr int64_t kSortMaxPoints = 1 << 22;

struct SortPlan {
  int passes, bits;                          // digits of `bits` bits
  int spans;
  int64_t key, pair[2], hist, totals, total;     // workspace offsets: keys, ping-pong (key, point), counts [span][digit]
};

static SortPlan sort_plan(int64_t n, int total_bits) {
  SortPlan s;
  s.passes = std::max(1, (int)cdiv(total_bits, kSortMaxBits));
  s.bits = std::max(1, (int)cdiv(total_bits, s.passes));
  s.spans = (int)cdiv(n, kSortSpan);
  int64_t off = 0;
  s.key = off; off += align_up(n * 4, 256);
  for (int i = 0; i < 2; ++i) { s.pair[i] = off; off += s.passes > 1 + i ? align_up(n * 8, 256) : 0; }
  s.hist = off; off += align_up(((int64_t)s.spans << s.bits) * 4, 256);
  s.totals = off; off += align_up(4ll << s.bits, 256);
  s.total = off;
  return s;
}

// A point's 32 bytes for the scatter: the normalised point and the normal (zeros without one).
static __device__ __forceinline__ void tree_row(float4* __restrict__ rows, int64_t i, float px, float py, float pz,
                                                const float* __restrict__ nrm) {
  const bool with = nrm != nullptr;
  rows[2 * i] = make_float4(px, py, pz, with ? nrm[3 * i] : 0.f);
  rows[2 * i + 1] = make_float4(with ? nrm[3 * i + 1] : 0.f, with ? nrm[3 * i + 2] : 0.f, 0.f, 0.f);
}

__global__ void tree_rows_kernel(const float* __restrict__ pts, const float* __restrict__ nrm, int64_t n, float4* __restrict__ rows) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) tree_row(rows, i, pts[3 * i], pts[3 * i + 1], pts[3 * i + 2], nrm);
}

// Normalised points and normals, sort keys (batch id right above the Morton bits) and the counts of the
// first digit by span.
__global__ __launch_bounds__(kSortThreads) void tree_keys_kernel(
    const float* __restrict__ pts, int64_t n, float bx, float by, float bz, float factor, const void* __restrict__ batch,
    int batch_is_float, int depth, const float* __restrict__ nrm, float4* __restrict__ rows, uint32_t* __restrict__ key, int bits,
    uint32_t* __restrict__ hist) {
  __shared__ uint32_t s_hist[1 << kSortMaxBits];
  const int bins = 1 << bits;
  for (int i = threadIdx.x; i < bins; i += kSortThreads) s_hist[i] = 0u;
  __syncthreads();
#pragma unroll
  for (int it = 0; it < kSortItems; ++it) {
    const int64_t i = (int64_t)blockIdx.x * kSortSpan + it * kSortThreads + threadIdx.x;
    if (i >= n) continue;
    // (p - bbmin) * factor: a subtraction then a multiplication, each rounded
    const float px = (pts[3 * i + 0] - bx) * factor;
    const float py = (pts[3 * i + 1] - by) * factor;
    const float pz = (pts[3 * i + 2] - bz) * factor;
    tree_row(rows, i, px, py, pz, nrm);
    uint64_t k = (uint64_t)encode((int64_t)px, (int64_t)py, (int64_t)pz, depth);      // trunc toward 0
    if (batch) {
      const int64_t b = batch_is_float ? (int64_t)((const float*)batch)[i] : ((const int64_t*)batch)[i];
      k |= ((uint64_t)b & 0xffffull) << (3 * depth);
    }
    key[i] = (uint32_t)k;
    atomicAdd(&s_hist[(uint32_t)k & (uint32_t)(bins - 1)], 1u);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < bins; i += kSortThreads) hist[(int64_t)blockIdx.x * bins + i] = s_hist[i];
}

// The counts of a further digit.  (Counting it with atomics in the scatter before instead: 25.2 / 24.7 us with / without
// for 2 k points at depth 6, 32.7 / 30.8 for 32 k, 42.1 / 40.0 for 131 k.)
__global__ __launch_bounds__(kSortThreads) void tree_digits_kernel(const uint2* __restrict__ pair, int64_t n, int shift,
                                                                   int bits, uint32_t* __restrict__ hist) {
  __shared__ uint32_t s_hist[1 << kSortMaxBits];
  const int bins = 1 << bits;
  for (int i = threadIdx.x; i < bins; i += kSortThreads) s_hist[i] = 0u;
  __syncthreads();
#pragma unroll
  for (int it = 0; it < kSortItems; ++it) {
    const int64_t i = (int64_t)blockIdx.x * kSortSpan + it * kSortThreads + threadIdx.x;
    if (i < n) atomicAdd(&s_hist[(pair[i].x >> shift) & (uint32_t)(bins - 1)], 1u);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < bins; i += kSortThreads) hist[(int64_t)blockIdx.x * bins + i] = s_hist[i];
}

// hist[span][digit] -> points of the digit in the spans before; totals[digit].  A workgroup takes 16
// digits, 64 threads each a run of spans.
__global__ __launch_bounds__(1024) void tree_spans_kernel(uint32_t* __restrict__ hist, int spans, int bins,
                                                          uint32_t* __restrict__ totals) {
  __shared__ uint32_t s_run[64][17];
  const int b = blockIdx.x * 16 + (threadIdx.x & 15), c = threadIdx.x >> 4;
  const int per = (spans + 63) / 64, lo = min(spans, c * per), hi = min(spans, lo + per);
  uint32_t sum = 0u;
  if (b < bins) {
#pragma unroll 8
    for (int sp = lo; sp < hi; ++sp) sum += hist[(int64_t)sp * bins + b];
  }
  s_run[c][threadIdx.x & 15] = sum;
  __syncthreads();
  uint32_t run = 0u;
  for (int i = 0; i < c; ++i) run += s_run[i][threadIdx.x & 15];
  if (b >= bins) return;
  if (c == 63) totals[b] = run + sum;
  for (int sp = lo; sp < hi; ++sp) {
    const uint32_t v = hist[(int64_t)sp * bins + b];
    hist[(int64_t)sp * bins + b] = run;
    run += v;
  }
}

// One stable pass.  A wave takes 128 consecutive points, 64 at a time: the lanes with the same digit
// find each other with one ballot per bit, their rank among the wave's points is kept in registers;
// the counts of the waves and of the spans before turn it into a place.  totals: hist has been scanned.
// (Sixteen waves a span and not four: the ballots of a wave are a serial chain, 23 -> 9 us for 20 000 points.)
// Between passes a point's key and number travel as 8 bytes: its place is a line of its own in memory, touched once and not
// twice (1 M points 27 -> 15.5 us a pass).  FIRST: from the keys; LAST: to keys and numbers.
constexpr int kPassThreads = 1024;
template <bool FIRST, bool LAST>
__global__ __launch_bounds__(kPassThreads) void tree_sort_kernel(
    const uint32_t* __restrict__ key, const uint2* __restrict__ pair, int64_t n, int shift, int bits, int spans,
    const uint32_t* __restrict__ hist, const uint32_t* __restrict__ totals, uint2* __restrict__ pair_out,
    uint32_t* __restrict__ key_out, uint32_t* __restrict__ val_out) {
  constexpr int kWaves = kPassThreads / 64, kMaxBins = 1 << kSortMaxBits, kPer = kMaxBins / kPassThreads;
  constexpr int kItems = kSortSpan / kPassThreads;
  __shared__ uint16_t s_cnt[kWaves][kMaxBins];               // points of a digit: in the wave, then in the waves before
  __shared__ uint32_t s_base[kMaxBins];                      // first place of this span's points of a digit
  __shared__ uint32_t s_wave[kWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int bins = 1 << bits;
  const int64_t first = (int64_t)blockIdx.x * kSortSpan + wave * (kSortSpan / kWaves) + lane;
  uint32_t k[kItems], v[kItems], rank[kItems];
#pragma unroll
  for (int it = 0; it < kItems; ++it) {
    const int64_t i = first + it * 64;
    const uint2 p = FIRST ? make_uint2(i < n ? key[i] : 0u, (uint32_t)i) : (i < n ? pair[i] : make_uint2(0u, 0u));
    k[it] = p.x;
    v[it] = p.y;
  }
  // digit counts of all spans: thread t on the bins 2 t, 2 t + 1
  uint32_t all[kPer], before[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int b = tid * kPer + u;
    all[u] = before[u] = 0u;
    if (b < bins && totals) {
      all[u] = totals[b];
      before[u] = hist[(int64_t)blockIdx.x * bins + b];
    } else if (b < bins) {
#pragma unroll 8
      for (int sp = 0; sp < spans; ++sp) {
        const uint32_t c = hist[(int64_t)sp * bins + b];
        all[u] += c;
        before[u] += sp < (int)blockIdx.x ? c : 0u;
      }
    }
  }
  for (int i = tid; i < bins; i += kPassThreads)
#pragma unroll
    for (int w = 0; w < kWaves; ++w) s_cnt[w][i] = 0;
  uint32_t own = 0u;
#pragma unroll
  for (int u = 0; u < kPer; ++u) own += all[u];
  uint32_t incl = own;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t up = __shfl_up(incl, o);
    if (lane >= o) incl += up;
  }
  if (lane == 63) s_wave[wave] = incl;
  __syncthreads();
  uint32_t at = incl - own;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) at += w < wave ? s_wave[w] : 0u;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int b = tid * kPer + u;
    if (b < bins) s_base[b] = at + before[u];
    at += all[u];
  }
  // ranks within the wave
  volatile uint16_t* cnt = s_cnt[wave];
#pragma unroll
  for (int it = 0; it < kItems; ++it) {
    const bool ok = first + it * 64 < n;
    const uint32_t d = (k[it] >> shift) & (uint32_t)(bins - 1);
    unsigned long long same = __ballot(ok);
    for (int b = 0; b < bits; ++b) {
      const unsigned long long ones = __ballot((d >> b) & 1u);
      same &= (d >> b) & 1u ? ones : ~ones;
    }
    const uint32_t seen = cnt[d], r = lanes_below(same);
    rank[it] = seen + r;
    if (ok && r == 0u) cnt[d] = (uint16_t)(seen + (uint32_t)__popcll(same));
  }
  __syncthreads();
  for (int b = tid; b < bins; b += kPassThreads) {
    uint32_t run = 0u;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const uint32_t c = s_cnt[w][b];
      s_cnt[w][b] = (uint16_t)run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < kItems; ++it) {
    if (first + it * 64 >= n) continue;
    const uint32_t d = (k[it] >> shift) & (uint32_t)(bins - 1);
    const uint32_t to = s_base[d] + s_cnt[wave][d] + rank[it];
    if constexpr (LAST) {
      key_out[to] = k[it];
      val_out[to] = v[it];
    } else {
      pair_out[to] = make_uint2(k[it], v[it]);
    }
  }
}

static int tree_key_bits(int depth, int batch_bits) { return 3 * depth + batch_bits; }
static bool tree_own_sort(int64_t n, int depth, int batch_bits) {
  return n <= kSortMaxPoints && tree_key_bits(depth, batch_bits) <= 32;
}

extern "C" int64_t ocnnx_tree_workspace_bytes(int64_t n, int depth, int full_depth, int batch_bits) {
  const int64_t base = ocnn_octree_build_workspace_bytes(n, depth, full_depth, batch_bits);
  if (base < 0) return base;
  return base + (tree_own_sort(n, depth, batch_bits) ? sort_plan(n, tree_key_bits(depth, batch_bits)).total
                                                   : align_up(n * 8, 256) + align_up(n * 12, 256));
}

extern "C" int ocnnx_tree_scan(const float* pts, int64_t n, const float* h_bbmin, float factor, const void* batch,
                               int batch_is_float, int depth, int full_depth, int batch_bits, const float* normals, float* rows,
                               void* workspace, int64_t workspace_bytes, int32_t* perm, int64_t* sizes, void* stream) {
  if (int rc = build_args_ok(n, depth, full_depth, batch_bits)) return rc;
  OCNN_REQUIRE_PTRS("tree_scan", pts, h_bbmin, rows, workspace, perm, sizes);
  if (workspace_bytes < ocnnx_tree_workspace_bytes(n, depth, full_depth, batch_bits)) {
    set_error("tree_scan: workspace too small");
    return OCNN_ERR_WORKSPACE;
  }
  hipStream_t st = (hipStream_t)stream;
  const int key_bits = 3 * depth, levels = depth - full_depth;
  const int64_t base = ocnn_octree_build_workspace_bytes(n, depth, full_depth, batch_bits);
  char* more = (char*)workspace + base;
  if (!tree_own_sort(n, depth, batch_bits)) {
    int64_t* key = (int64_t*)more;
    float* norm = (float*)(more + align_up(n * 8, 256));
    if (int rc = ocnn_points2key(pts, n, h_bbmin, factor, batch, batch_is_float, depth, norm, key, stream)) return rc;
    hipLaunchKernelGGL(tree_rows_kernel, dim3((unsigned)cdiv(n, 256)), dim3(256), 0, st, norm, normals, n, (float4*)rows);
    return ocnn_octree_build_scan(key, n, depth, full_depth, batch_bits, workspace, base, perm, sizes, stream);
  }
  const SortPlan s = sort_plan(n, tree_key_bits(depth, batch_bits));
  uint32_t* keys = (uint32_t*)(more + s.key);
  uint2* pairs[2] = {(uint2*)(more + s.pair[0]), (uint2*)(more + s.pair[1])};
  uint32_t* hist = (uint32_t*)(more + s.hist);
  uint32_t* totals = s.spans > kSortInlineSpans ? (uint32_t*)(more + s.totals) : nullptr;
  BuildLayout L;
  if (build_layout_t<uint32_t, 8>(n, &L) != OCNN_OK) { set_error("tree_scan: rocprim size query failed"); return OCNN_ERR_HIP; }
  if (levels + 1 > 8 && build_layout_t<uint32_t, 16>(n, &L) != OCNN_OK) { set_error("tree_scan: rocprim size query failed"); return OCNN_ERR_HIP; }
  uint32_t* csorted = (uint32_t*)((char*)workspace + L.csorted);
  uint32_t* sums = (uint32_t*)((char*)workspace + L.sums);
  uint32_t* offs = (uint32_t*)((char*)workspace + L.offs);
  const dim3 grid((unsigned)s.spans), block(kSortThreads);
  hipLaunchKernelGGL(tree_keys_kernel, grid, block, 0, st, pts, n, h_bbmin[0], h_bbmin[1], h_bbmin[2], factor, batch,
                     batch_is_float, depth, normals, (float4*)rows, keys, s.bits, hist);
  for (int p = 0; p < s.passes; ++p) {
    const bool last = p + 1 == s.passes;
    if (p > 0) hipLaunchKernelGGL(tree_digits_kernel, grid, block, 0, st, pairs[(p + 1) & 1], n, p * s.bits, s.bits, hist);
    if (totals)
      hipLaunchKernelGGL(tree_spans_kernel, dim3((unsigned)cdiv(1 << s.bits, 16)), dim3(1024), 0, st, hist, s.spans, 1 << s.bits,
                         totals);
    const auto pass = p == 0 ? (last ? tree_sort_kernel<true, true> : tree_sort_kernel<true, false>)
                             : (last ? tree_sort_kernel<false, true> : tree_sort_kernel<false, false>);
    hipLaunchKernelGGL(pass, grid, dim3(kPassThreads), 0, st, keys, pairs[(p + 1) & 1], n, p * s.bits, s.bits, s.spans, hist, totals,
                       pairs[p & 1], csorted, (uint32_t*)perm);
  }
#define OCNN_TREE_COUNT(N)                                                                          \
  launch_build_count<uint32_t, N>(csorted, n, L.spans, key_bits, levels, sums, st);                  \
  hipLaunchKernelGGL(build_offsets_kernel<N>, dim3(1), dim3(1024), 0, st, sums, L.spans, levels, offs, sizes)
  if (levels + 1 <= 8) { OCNN_TREE_COUNT(8); }
  else { OCNN_TREE_COUNT(16); }
#undef OCNN_TREE_COUNT
  return check_launch("tree_scan");
}

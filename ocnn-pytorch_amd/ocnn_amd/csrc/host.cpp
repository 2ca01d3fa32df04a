// Host path of the layers: what runs between a module's forward() and the launches of the C ABI,
// natively.  A small layer's kernels take a few dozen microseconds; the same calls made from Python
// (argument lists through ctypes, a Python autograd node, the interpreter lock in the backward
// thread) took 100 - 150.
//
// A GatherOp / WgradOp is one pass of a layer with everything that depends on the shapes and the
// table only - which kernel, the plan's arrays and figures, the workspace size - decided when it is
// made (nn/octree_conv.py); run() allocates the result and a workspace and calls the library.  A
// ConvLayer holds the up to three passes of a layer on an octree; conv() is its autograd node.
#include <ATen/ATen.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <memory>
#include <mutex>
#include <optional>
#include <vector>

#include "host_api.hpp"

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

void check(int rc) { TORCH_CHECK(rc == 0, "libocnn_hip: ", ocnn_last_error(), " (code ", rc, ")"); }

void* hip_stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

int code_of(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return OCNN_F32;
    case at::kHalf: return OCNN_F16;
    case at::kBFloat16: return OCNN_BF16;
    default: TORCH_CHECK_TYPE(false, "unsupported feature dtype ", t, "; use float32, float16 or bfloat16");
  }
}

void require_gpu(const Tensor& t) {
  TORCH_CHECK(t.is_cuda(), "ocnn_amd kernels need tensors on a HIP device, got a tensor on ", t.device());
}

const void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
const void* ptr(const OptTensor& t) { return t.has_value() && t->defined() ? t->data_ptr() : nullptr; }
template <typename T> T* typed(const Tensor& t) { return t.defined() ? (T*)t.data_ptr() : nullptr; }

Tensor workspace(int64_t bytes, const Tensor& like) {
  return at::empty({std::max<int64_t>(bytes, 256)}, like.options().dtype(at::kByte));
}

bool capturing() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }

// The rows of the tiles of several plans in the order of ocnnx_plan_order, by their positions.
std::vector<Tensor> tile_orders(const std::vector<Tensor>& locs) {
  std::vector<Tensor> out;
  std::vector<ocnnx_order_item> items;
  int64_t tiles = 0;
  for (const Tensor& loc : locs) {
    require_gpu(loc);
    TORCH_CHECK(loc.scalar_type() == at::kShort && loc.dim() == 3 && loc.size(2) == ocnn_tile_plan_rows() &&
                    loc.is_contiguous() && loc.device() == locs[0].device(),
                "tile_orders: positions of tile plans of one device");
    out.push_back(at::empty({loc.size(0), OCNNX_TILE_ORDER_BYTES}, loc.options().dtype(at::kByte)));
    items.push_back({typed<uint16_t>(loc), typed<uint8_t>(out.back()), loc.size(0), tiles, (int)loc.size(1)});
    tiles += loc.size(0);
  }
  if (!items.empty()) check(ocnnx_plan_order(items.data(), (int)items.size(), hip_stream()));
  return out;
}

// The end of what the current stream has been given so far, for what is made once and read by later work of any stream.
class MadeHere {
 public:
  MadeHere() : stream_(c10::hip::getCurrentHIPStream().stream()) {
    TORCH_CHECK(hipEventCreateWithFlags(&event_, hipEventDisableTiming) == hipSuccess &&
                    hipEventRecord(event_, stream_) == hipSuccess,
                "cannot record an event");
  }
  ~MadeHere() { (void)hipEventDestroy(event_); }
  MadeHere(const MadeHere&) = delete;
  MadeHere& operator=(const MadeHere&) = delete;

  // Makes the current stream wait for it, if need be.  False under a capture that it has not come true before: a graph
  // cannot wait for an event from outside.
  bool before_current() {
    if (done_) return true;
    const bool captures = capturing();
    const hipStream_t st = c10::hip::getCurrentHIPStream().stream();
    if (!captures && st == stream_) return true;
    // (asking is no part of a capture, of this thread or another's)
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    const hipError_t status = hipEventQuery(event_);
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (status == hipSuccess) return done_ = true;
    (void)hipGetLastError();
    if (captures) return false;
    TORCH_CHECK(hipStreamWaitEvent(st, event_, 0) == hipSuccess, "cannot wait for an event");
    return true;
  }

 private:
  hipStream_t stream_;
  hipEvent_t event_ = nullptr;
  std::atomic<bool> done_{false};
};

// The arrays and figures of a tile plan and, where a kernel walks pairs, of its pair plan.
struct PlanArrays {
  Tensor loc, uptr, urows;
  int umax = 0;
  int64_t total = 0;
  double occupancy = 1.0;
  Tensor cptr, ent, lists;                    // pair plan
  int64_t n_blocks = 0;
  int max_blocks = 0, n_lists = 0;
  std::vector<int32_t> lists_host, group_bounds;
  std::vector<int64_t> list_count;

  // The order of the tiles' rows that the passes on this plan share, made by the first that runs without it and waited for
  // on other streams; null under a capture that finds none: what a graph makes holds nothing before its first replay, and a
  // pass is right without.
  const uint8_t* rows_order() {
    std::lock_guard<std::mutex> lock(order_lock);
    if (!order.defined() && !capturing()) {
      at::tracer::impl::NoTracerDispatchMode quiet;
      order = tile_orders({loc})[0];
      order_made = std::make_shared<MadeHere>();
    }
    return order.defined() && order_made->before_current() ? typed<uint8_t>(order) : nullptr;
  }
  std::mutex order_lock;
  Tensor order;
  std::shared_ptr<MadeHere> order_made;
};

// rows_order() of several plans, in one launch
void order_many(const std::vector<std::shared_ptr<PlanArrays>>& plans) {
  std::vector<Tensor> locs;
  for (const auto& p : plans) locs.push_back(p->loc);
  const std::vector<Tensor> orders = tile_orders(locs);
  const auto made = std::make_shared<MadeHere>();
  for (size_t i = 0; i < plans.size(); ++i) {
    std::lock_guard<std::mutex> lock(plans[i]->order_lock);
    if (plans[i]->order.defined()) continue;
    plans[i]->order = orders[i];
    plans[i]->order_made = made;
  }
}

// codes on top of the library's OCNN_GATHER_* / OCNN_WGRAD_*
constexpr int kWgradSparseInverse = 5;        // the pair plan of the inverse table, operands exchanged

struct GatherOp {
  int kernel = OCNN_GATHER_PLAIN, K = 0, cin = 0, cout = 0;
  int64_t rows_in = 0, rows = 0, ws_bytes = 0;
  bool transposed = false, reverse = false;
  std::shared_ptr<PlanArrays> plan;
  bool ordered = false;                       // OCNNX_GATHER_TILE: the kernel takes the plan's rows_order()
  // dense one-slot form: rows read / written through an index of the non-empty nodes
  Tensor in_index, out_index, children;
  int64_t rows_all = 0;                       // rows of the padded result
  // the rows of tiles that are too dense for the plan: table, places in the result, their own pass
  Tensor overflow_table, overflow_rows;
  int bias_repeat = 1, view_cols = 0;         // dense form: bias once per child; result seen with this many columns
  std::shared_ptr<GatherOp> overflow, padded; // padded: this pass with channels in whole multiples (zero-padded)

  // bn: a batch norm with running statistics that follows the layer; in the same pass where the kernel
  // has room for it, in place after it otherwise
  // packed: W as ocnnx_pack_tiles leaves it (the kernel of takes_packed())
  Tensor run(Tensor data, Tensor table, Tensor W, OptTensor bias, const ocnnx_bn* bn = nullptr, const void* packed = nullptr) const {
    require_gpu(data);
    require_gpu(W);
    const int code = code_of(data.scalar_type());
    data = data.contiguous();
    W = W.contiguous();
    TORCH_CHECK(W.scalar_type() == data.scalar_type() && W.numel() == (int64_t)K * cin * cout,
                "weights do not match the table and channels");
    if (bias.has_value()) {
      bias = bias->to(data.scalar_type()).contiguous();
      if (bias_repeat > 1) bias = bias->repeat({bias_repeat});
    }
    if (padded) return followed(run_padded(data, table, W, bias), bn);
    void* st = hip_stream();
    const bool wide_out = kernel == OCNN_GATHER_DENSE_RW && out_index.defined();
    Tensor out = at::empty({wide_out ? rows_all : rows, cout}, data.options());
    Tensor ws = workspace(ws_bytes, data);
    const PlanArrays* p = plan.get();
    switch (kernel) {
      case OCNN_GATHER_DENSE_RW: {
        const int64_t in_rows = data.numel() / cin;
        check(ocnn_conv_dense_rw_indexed(code, ptr(data), in_rows, typed<int32_t>(in_index), rows, ptr(W), cin, cout,
                                         transposed, ptr(bias), out.data_ptr(), out.size(0), typed<int32_t>(out_index),
                                         ws.data_ptr(), ws.numel(), st));
        if (out_index.defined())              // zeros for the empty nodes
          check(ocnn_pad(code, nullptr, typed<int32_t>(children), rows_all, cout, 0.f, out.data_ptr(), st));
        break;
      }
      case OCNN_GATHER_DENSE:
        check(ocnn_conv_dense(code, ptr(data), rows, ptr(W), cin, cout, transposed, ptr(bias), out.data_ptr(),
                              ws.data_ptr(), ws.numel(), st));
        break;
      case OCNNX_GATHER_ROWS:
        TORCH_CHECK(data.numel() == rows * cin, "conv_gather: the rows do not match");
        check(ocnnx_dense_rows(code, ptr(data), rows, ptr(W), cin, cout, transposed, ptr(bias), bn, out.data_ptr(), st));
        bn = nullptr;
        break;
      case OCNN_GATHER_RW:
        check(ocnnx_conv_gather_rw(code, ptr(data), rows_in, typed<uint16_t>(p->loc), typed<int32_t>(p->uptr),
                                   typed<int32_t>(p->urows), p->umax, p->total, rows, K, ptr(W), cin, cout, transposed,
                                   reverse, ptr(bias), overflow ? nullptr : bn, out.data_ptr(), ws.data_ptr(), ws.numel(), st));
        if (!overflow) bn = nullptr;
        break;
      case OCNNX_GATHER_TILE: {
        ocnnx_gather_args args = tile_args(ptr(data), ptr(W), ptr(bias), overflow ? nullptr : bn, out, ws);
        args.packed = packed;
        check(ocnnx_gather_tile_args(code, &args, st));
        if (!overflow) bn = nullptr;
        break;
      }
      case OCNN_GATHER_SPARSE:
        check(ocnn_conv_gather_sparse(code, ptr(data), rows_in, typed<int32_t>(p->uptr), typed<int32_t>(p->urows),
                                      p->umax, p->total, typed<int32_t>(p->cptr), typed<uint32_t>(p->ent), p->n_blocks,
                                      p->max_blocks, typed<int32_t>(p->lists), p->n_lists, p->group_bounds.data(),
                                      rows, K, ptr(W), cin, cout, transposed, reverse, ptr(bias), out.data_ptr(),
                                      ws.data_ptr(), ws.numel(), st));
        break;
      case OCNN_GATHER_PLANNED:               // (tiles of more rows than the other kernels stage)
        check(ocnn_conv_gather_planned(code, ptr(data), rows_in, typed<uint16_t>(p->loc), typed<int32_t>(p->uptr),
                                       typed<int32_t>(p->urows), rows, K, ptr(W), cin, cout, transposed, reverse,
                                       ptr(bias), out.data_ptr(), ws.data_ptr(), ws.numel(), st));
        break;
      default:
        TORCH_CHECK(table.defined(), "this pass needs the neighbour table");
        require_gpu(table);
        TORCH_CHECK(table.scalar_type() == at::kInt && table.is_contiguous() && table.numel() == rows * K,
                    "conv_gather: the table does not match");
        check(ocnnx_conv_gather(code, ptr(data), rows_in, typed<int32_t>(table), rows, K, ptr(W), cin, cout, transposed,
                                reverse, ptr(bias), out.data_ptr(), nullptr, ws.data_ptr(), ws.numel(), st));
    }
    if (overflow) {
      at::tracer::impl::NoTracerDispatchMode quiet;          // (a trace must not own the plan's tensors)
      overflow->run_into(out, overflow_rows, data, overflow_table, W, bias);
    }
    return followed(view_cols ? out.view({-1, view_cols}) : out, bn);
  }

  // the kernel for this shape, of a table with these figures of its plan, and the workspace it takes
  void choose(int code, bool dense, bool has_plan, int umax, int64_t total, double occupancy, double reuse, bool overflows) {
    kernel = ocnnx_gather_choose(code, rows_in, rows, K, cin, cout, dense, has_plan, umax, total, occupancy, reuse, overflows);
    ordered = kernel == OCNNX_GATHER_TILE && ocnnx_gather_tile_ordered(K, occupancy);
    ws_bytes = kernel == OCNN_GATHER_ZERO_PADDED || kernel == OCNNX_GATHER_ROWS ? 0
               : kernel == OCNN_GATHER_SPARSE ? ocnn_conv_gather_sparse_workspace_bytes(cin, cout)
               : kernel == OCNNX_GATHER_TILE  ? ocnnx_gather_tile_workspace_bytes(code, rows, K, cin, cout)
               : kernel == OCNN_GATHER_PLAIN  ? ocnnx_conv_gather_workspace_bytes(code, rows_in, rows, K, cin, cout)
                                              : ocnn_conv_gather_workspace_bytes(code, rows_in, K, cin, cout);
  }

  ocnnx_gather_args tile_args(const void* data, const void* W, const void* bias, const ocnnx_bn* bn, const Tensor& out,
                              const Tensor& ws) const {
    const PlanArrays& p = *plan;
    return {data, rows_in, typed<uint16_t>(p.loc), typed<int32_t>(p.uptr), typed<int32_t>(p.urows), p.umax, p.total,
            p.occupancy, rows, K, W, cin, cout, transposed, reverse, bias, bn, out.data_ptr(), ws.data_ptr(), ws.numel(), 0, 0,
            ordered ? plan->rows_order() : nullptr, nullptr};
  }

  bool takes_packed() const { return kernel == OCNNX_GATHER_TILE && !padded; }

  // this pass with row i of its result written to row index[i] of `out`
  void run_into(Tensor& out, const Tensor& index, const Tensor& data, const Tensor& table, const Tensor& W,
                const OptTensor& bias) const {
    if (kernel != OCNN_GATHER_PLAIN || padded) {
      out.index_copy_(0, index, run(data, table, W, bias));
      return;
    }
    TORCH_CHECK(index.scalar_type() == at::kLong && index.is_contiguous() && index.numel() == rows &&
                    table.scalar_type() == at::kInt && table.is_contiguous() && table.numel() == rows * K,
                "conv_gather: the rows that run apart do not match");
    Tensor ws = workspace(ws_bytes, data);
    check(ocnnx_conv_gather(code_of(data.scalar_type()), ptr(data), rows_in, typed<int32_t>(table), rows, K, ptr(W), cin,
                            cout, transposed, reverse, ptr(bias), out.data_ptr(), typed<int64_t>(index), ws.data_ptr(),
                            ws.numel(), hip_stream()));
  }
 private:
  static Tensor followed(const Tensor& out, const ocnnx_bn* bn) {
    if (bn && out.size(0))
      check(ocnnx_batch_norm_running(code_of(out.scalar_type()), out.data_ptr(), out.size(0), (int)out.size(1), bn->mean,
                                     bn->var, bn->stat_dtype, bn->eps, bn->gamma, bn->beta, bn->param_dtype, bn->relu,
                                     bn->residual, out.data_ptr(), hip_stream()));
    return out;
  }
  Tensor run_padded(const Tensor& data, const Tensor& table, const Tensor& W, const OptTensor& bias) const {
    const int pi = padded->cin - cin, po = padded->cout - cout;
    Tensor Wk = transposed ? W.view({K, cout, cin}) : W.view({K, cin, cout});
    Wk = transposed ? at::constant_pad_nd(Wk, {0, pi, 0, po}) : at::constant_pad_nd(Wk, {0, po, 0, pi});
    OptTensor b;
    if (bias.has_value()) b = at::constant_pad_nd(*bias, {0, po});
    // (the dense form may come as the rows of the children: eight rows of a table row's channels)
    const Tensor rows_in_view = data.view({-1, cin});
    Tensor out = padded->run(pi ? at::constant_pad_nd(rows_in_view, {0, pi}) : rows_in_view, table, Wk, b);
    return po ? out.slice(1, 0, cout).contiguous() : out;
  }
};

struct WgradOp {
  int kernel = OCNN_WGRAD_PLAIN, K = 0, ca = 0, cb = 0;
  int64_t rows_x = 0, rows = 0, ws_bytes = 0;
  bool out_transposed = false;
  std::shared_ptr<PlanArrays> plan;
  Tensor g_index;                             // dense one-slot form: row i of the sum takes row g_index[i] of g
  std::vector<int64_t> shape;                 // shape the result is seen with, if not (K, ca, cb)
  Tensor overflow_table, overflow_rows;
  std::shared_ptr<WgradOp> overflow, padded;

  void choose(int code, bool dense, bool has_plan, int umax, int64_t total, double occupancy) {
    kernel = ocnn_conv_wgrad_choose(code, rows_x, rows, K, ca, cb, dense, has_plan, umax, total, occupancy);
    ws_bytes = kernel == OCNN_WGRAD_ZERO_PADDED ? 0
               : kernel == OCNN_WGRAD_DENSE_RW  ? ocnn_conv_dense_wgrad_rw_workspace_bytes(ca, cb)
               : kernel == OCNN_WGRAD_SPARSE    ? ocnn_conv_wgrad_sparse_workspace_bytes(rows, ca, cb)
               : kernel == OCNN_WGRAD_PLANNED   ? ocnn_conv_wgrad_planned_workspace_bytes_for(code, rows_x, rows, K, ca, cb)
                                                : ocnn_conv_wgrad_workspace_bytes_for(code, rows_x, rows, K, ca, cb);
  }

  Tensor run(Tensor x, Tensor g, Tensor table) const {
    require_gpu(x);
    require_gpu(g);
    const int code = code_of(x.scalar_type());
    TORCH_CHECK(x.scalar_type() == g.scalar_type(), "conv_wgrad: operands of different types");
    x = x.contiguous();
    g = g.contiguous();
    if (padded) {
      x = x.view({-1, ca});
      const int pa = padded->ca - ca, pb = padded->cb - cb;
      Tensor gw = padded->run(pa ? at::constant_pad_nd(x, {0, pa}) : x, pb ? at::constant_pad_nd(g, {0, pb}) : g, table);
      gw = out_transposed ? gw.slice(1, 0, cb).slice(2, 0, ca) : gw.slice(1, 0, ca).slice(2, 0, cb);
      gw = gw.contiguous();
      return shape.empty() ? gw : gw.view(shape);
    }
    void* st = hip_stream();
    Tensor gw = at::empty({K, out_transposed ? cb : ca, out_transposed ? ca : cb}, x.options());
    Tensor ws = workspace(ws_bytes, x);
    const PlanArrays* p = plan.get();
    switch (kernel) {
      case OCNN_WGRAD_DENSE_RW:
        check(ocnn_conv_dense_wgrad_rw_indexed(code, ptr(x), x.numel() / ca, nullptr, ptr(g), g.size(0),
                                               typed<int32_t>(g_index), rows, ca, cb, out_transposed, gw.data_ptr(),
                                               ws.data_ptr(), ws.numel(), st));
        break;
      case OCNN_WGRAD_SPARSE:
        check(ocnn_conv_wgrad_sparse(code, ptr(x), rows_x, ca, ptr(g), rows, cb, typed<int32_t>(p->uptr),
                                     typed<int32_t>(p->urows), p->umax, p->total, typed<int32_t>(p->cptr),
                                     typed<uint32_t>(p->ent), p->n_blocks, p->lists_host.data(), p->list_count.data(),
                                     p->n_lists, K, !out_transposed, gw.data_ptr(), ws.data_ptr(), ws.numel(), st));
        break;
      case kWgradSparseInverse:               // rows: those of x, which are the rows of the inverse table
        check(ocnn_conv_wgrad_sparse(code, ptr(g), rows_x, cb, ptr(x), rows, ca, typed<int32_t>(p->uptr),
                                     typed<int32_t>(p->urows), p->umax, p->total, typed<int32_t>(p->cptr),
                                     typed<uint32_t>(p->ent), p->n_blocks, p->lists_host.data(), p->list_count.data(),
                                     p->n_lists, K, out_transposed, gw.data_ptr(), ws.data_ptr(), ws.numel(), st));
        if (overflow) gw.add_(overflow->run(g, x.index_select(0, overflow_rows), overflow_table));
        return gw;
      case OCNN_WGRAD_PLANNED:
        check(ocnn_conv_wgrad_planned(code, ptr(x), rows_x, ptr(g), typed<uint16_t>(p->loc), typed<int32_t>(p->uptr),
                                      typed<int32_t>(p->urows), p->umax, p->total, rows, K, ca, cb, out_transposed,
                                      gw.data_ptr(), ws.data_ptr(), ws.numel(), st));
        break;
      default:
        TORCH_CHECK(table.defined(), "this pass needs the neighbour table");
        require_gpu(table);
        TORCH_CHECK(table.scalar_type() == at::kInt && table.is_contiguous() && table.numel() == rows * K,
                    "conv_wgrad: the table does not match");
        check(ocnn_conv_wgrad(code, ptr(x), rows_x, ptr(g), typed<int32_t>(table), rows, K, ca, cb, out_transposed,
                              gw.data_ptr(), ws.data_ptr(), ws.numel(), st));
    }
    if (overflow) gw.add_(overflow->run(x, g.index_select(0, overflow_rows), overflow_table));
    return shape.empty() ? gw : gw.view(shape);
  }
};

// Data, weight and (want_bias) bias gradient of a layer in one call, for the pair of kernels whose small launches can
// be merged; false where the passes are others.
bool backward_together(const GatherOp& dgrad, const WgradOp& wgrad, const Tensor& grad, const Tensor& w, const Tensor& x,
                       const Tensor& g, bool want_bias, variable_list& out) {
  if (dgrad.kernel != OCNNX_GATHER_TILE || wgrad.kernel != OCNN_WGRAD_PLANNED || dgrad.padded || wgrad.padded) return false;
  for (const Tensor& t : {grad, w, x, g})
    if (!t.is_cuda() || !t.is_contiguous() || t.scalar_type() != grad.scalar_type()) return false;
  if (w.numel() != (int64_t)dgrad.K * dgrad.cin * dgrad.cout) return false;
  const int code = code_of(grad.scalar_type());
  Tensor gx = at::empty({dgrad.rows, dgrad.cout}, grad.options());
  Tensor gw = at::empty({wgrad.K, wgrad.out_transposed ? wgrad.cb : wgrad.ca, wgrad.out_transposed ? wgrad.ca : wgrad.cb},
                        grad.options());
  Tensor gb = want_bias ? at::empty({grad.size(1)}, grad.options()) : Tensor();
  // (each with a workspace of its own: the passes overlap)
  Tensor ws_d = workspace(dgrad.ws_bytes, grad), ws_w = workspace(wgrad.ws_bytes, grad);
  Tensor ws_b = want_bias ? workspace(ocnn_colsum_workspace_bytes(grad.size(0), (int)grad.size(1)), grad) : Tensor();
  const PlanArrays& q = *wgrad.plan;
  const ocnnx_gather_args da = dgrad.tile_args(ptr(grad), ptr(w), nullptr, nullptr, gx, ws_d);
  const ocnnx_wgrad_args wa{ptr(x), wgrad.rows_x, ptr(g), typed<uint16_t>(q.loc), typed<int32_t>(q.uptr),
                            typed<int32_t>(q.urows), q.umax, q.total, wgrad.rows, wgrad.K, wgrad.ca, wgrad.cb,
                            wgrad.out_transposed, gw.data_ptr(), ws_w.data_ptr(), ws_w.numel()};
  check(ocnnx_conv_backward(code, &da, &wa, ptr(grad), grad.size(0), (int)grad.size(1), gb.defined() ? gb.data_ptr() : nullptr,
                            gb.defined() ? ws_b.data_ptr() : nullptr, gb.defined() ? ws_b.numel() : 0, hip_stream()));
  if (dgrad.overflow) dgrad.overflow->run_into(gx, dgrad.overflow_rows, grad, dgrad.overflow_table, w, std::nullopt);
  if (wgrad.overflow) gw.add_(wgrad.overflow->run(x, g.index_select(0, wgrad.overflow_rows), wgrad.overflow_table));
  out[0] = dgrad.view_cols ? gx.view({-1, dgrad.view_cols}) : gx;
  out[1] = wgrad.shape.empty() ? gw : gw.view(wgrad.shape);
  out[2] = gb;
  return true;
}

Tensor column_sum(Tensor g) {
  require_gpu(g);
  g = g.contiguous();
  Tensor out = at::empty({g.size(1)}, g.options());
  Tensor ws = workspace(ocnn_colsum_workspace_bytes(g.size(0), (int)g.size(1)), g);
  check(ocnn_colsum(code_of(g.scalar_type()), ptr(g), g.size(0), (int)g.size(1), out.data_ptr(), ws.data_ptr(),
                    ws.numel(), hip_stream()));
  return out;
}

// g^T x of fp32 rows (ocnnx_rows_wgrad)
Tensor rows_wgrad(Tensor g, Tensor x) {
  require_gpu(g);
  require_gpu(x);
  TORCH_CHECK(g.dim() == 2 && x.dim() == 2 && g.size(0) == x.size(0) && g.scalar_type() == at::kFloat &&
                  x.scalar_type() == at::kFloat && g.device() == x.device(),
              "rows_wgrad: two fp32 matrices of as many rows");
  g = g.contiguous();
  x = x.contiguous();
  const int ca = (int)g.size(1), cb = (int)x.size(1);
  Tensor out = at::empty({ca, cb}, x.options());
  Tensor ws = workspace(ocnnx_rows_wgrad_workspace_bytes(x.size(0), ca, cb), x);
  check(ocnnx_rows_wgrad(OCNN_F32, ptr(g), ptr(x), x.size(0), ca, cb, 0, out.data_ptr(), ws.data_ptr(), ws.numel(),
                         hip_stream()));
  return out;
}

// The passes of one layer on one octree, in one data type.  fwd: data -> out; dgrad: grad -> data
// gradient; wgrad over (data, grad), for a deconvolution over (grad, data).  The backward passes are
// made when a call first needs them, as a copy with the pass: threads share the object.
struct ConvLayer {
  std::shared_ptr<GatherOp> fwd, dgrad;
  std::shared_ptr<WgradOp> wgrad;
  Tensor fwd_table, dgrad_table, wgrad_table;
  bool wgrad_of_grad = false;                 // deconvolution: x = grad (the fine side), g = data
};

// ---- autograd nodes ---------------------------------------------------------------------------

// The node behind `out` when a gradient can be asked for: its edges lead to `inputs`.
template <typename N> std::shared_ptr<N> make_node(const variable_list& inputs) {
  auto node = std::shared_ptr<N>(new N(), torch::autograd::deleteNode);
  node->set_next_edges(torch::autograd::collect_next_edges(inputs));
  return node;
}

bool any_requires_grad(const variable_list& v) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor& t : v)
    if (t.defined() && t.requires_grad()) return true;
  return false;
}

struct ConvBackward : public Node {
  SavedVariable data, weights;
  std::shared_ptr<ConvLayer> layer;

  variable_list apply(variable_list&& grads) override {
    variable_list out(3);
    if (!grads[0].defined()) return out;
    Tensor grad = grads[0].contiguous(), x = data.unpack(), w = weights.unpack();
    at::AutoDispatchBelowADInplaceOrView below;
    if (task_should_compute_output(0) && task_should_compute_output(1) &&
        backward_together(*layer->dgrad, *layer->wgrad, grad, w, layer->wgrad_of_grad ? grad : x,
                          layer->wgrad_of_grad ? x : grad, task_should_compute_output(2), out))
      return out;
    // The data gradient last: what comes next reads it, and the memory-side cache still holds its end.  First where channels are
    // padded, whose passes are chains of copies: 4 -> 64 and 4 -> 96 on 8 clouds of depth 6, forward + backward, 164.8 and 206 us, last
    // 168.9 and 209.
    const bool wants = task_should_compute_output(0), last = wants && !layer->dgrad->padded;
    if (wants && !last) out[0] = layer->dgrad->run(grad, layer->dgrad_table, w, std::nullopt);
    if (task_should_compute_output(1))
      out[1] = layer->wgrad_of_grad ? layer->wgrad->run(grad, x, layer->wgrad_table)
                                    : layer->wgrad->run(x, grad, layer->wgrad_table);
    if (task_should_compute_output(2)) out[2] = column_sum(grad);
    if (last) out[0] = layer->dgrad->run(grad, layer->dgrad_table, w, std::nullopt);
    return out;
  }
  void release_variables() override {
    data.reset_data();
    weights.reset_data();
  }
  std::string name() const override { return "OctreeConvBackward"; }
};

Tensor conv(const std::shared_ptr<ConvLayer>& layer, const Tensor& data_in, const Tensor& weights, const OptTensor& bias) {
  const variable_list inputs{data_in, weights, bias.has_value() ? *bias : Tensor()};
  const bool track = any_requires_grad(inputs);
  Tensor data, w, out;
  {
    at::AutoDispatchBelowADInplaceOrView below;
    data = data_in.contiguous();
    w = weights.to(data.scalar_type()).contiguous();
    out = layer->fwd->run(data, layer->fwd_table, w, bias);
  }
  if (track) {
    auto node = make_node<ConvBackward>(inputs);
    node->data = SavedVariable(data, false);
    node->weights = SavedVariable(w, false);
    node->layer = layer;
    torch::autograd::set_history(out, node);
  }
  return out;
}

// ---- batch norm (nn/batchnorm.py) -------------------------------------------------------------

// A per-channel parameter as the kernels read it (f32 / f16 / bf16, contiguous).
Tensor as_param(const Tensor& t) {
  if (!t.defined()) return t;
  const auto k = t.scalar_type();
  return (k == at::kFloat || k == at::kHalf || k == at::kBFloat16 ? t : t.to(at::kFloat)).contiguous();
}

int param_code(const Tensor& gamma, const Tensor& beta) {
  const Tensor& t = gamma.defined() ? gamma : beta;
  return t.defined() ? code_of(t.scalar_type()) : OCNN_F32;
}

// What the backward pass reads, and how the forward pass was taken.
struct BatchNormCall {
  Tensor x, mean, invstd, gamma, beta, y;     // (y: only where the ReLU's mask is not a function of x alone)
  bool relu = false, training = false, has_residual = false;
  at::ScalarType wdtype = at::kFloat, bdtype = at::kFloat;
  Tensor mask;                                // the mask itself, a bit a value, in y's place
};

// Gradients of x, weight, bias and residual, those of them that `want` names.
std::array<Tensor, 4> batch_norm_grads(const BatchNormCall& call, const Tensor& dy, std::array<bool, 4> want) {
  const Tensor &xs = call.x, &ga = call.gamma, &be = call.beta;
  const int64_t rows = xs.size(0), c = xs.size(1);
  const auto f32 = xs.options().dtype(at::kFloat);
  Tensor sums = at::empty({2, c}, f32);                     // dgamma, dbeta
  const bool want_res = call.has_residual && want[3];
  Tensor dx, dres, gw, gb;
  if (want[0] || want_res) dx = at::empty_like(xs);
  if (want_res) dres = at::empty_like(xs);
  // the parameter gradients come out in the parameters' dtype where the kernels hold it
  const bool want_w = ga.defined() && want[1], want_b = be.defined() && want[2];
  if (want_w && call.wdtype == ga.scalar_type()) gw = at::empty({c}, ga.options());
  if (want_b && call.bdtype == be.scalar_type() && (!ga.defined() || be.scalar_type() == ga.scalar_type()))
    gb = at::empty({c}, be.options());
  Tensor ws = workspace(ocnn_batch_norm_workspace_bytes((int)c), xs);
  float* s = (float*)sums.data_ptr();
  check(ocnnx_batch_norm_backward(code_of(xs.scalar_type()), ptr(xs), ptr(dy), rows, (int)c, (const float*)ptr(call.mean),
                                 (const float*)ptr(call.invstd), ptr(ga), ptr(be), param_code(ga, be), call.relu,
                                 call.training, ptr(call.y), ptr(call.mask), typed<void>(dx), typed<void>(dres), s, s + c, typed<void>(gw),
                                 typed<void>(gb), ws.data_ptr(), ws.numel(), hip_stream()));
  if (want_w && !gw.defined()) gw = sums[0].to(call.wdtype);
  if (want_b && !gb.defined()) gb = sums[1].to(call.bdtype);
  return {want[0] ? dx : Tensor(), gw, gb, dres};
}

struct BatchNormBackward : public Node {
  SavedVariable x, mean, invstd, gamma, beta, y, mask;
  BatchNormCall call;                         // (its flags; the tensors are the saved ones)
  bool keeps_y = false, keeps_mask = false;

  variable_list apply(variable_list&& grads) override {
    variable_list out(4);
    if (!grads[0].defined()) return out;
    Tensor dy = grads[0].contiguous();
    BatchNormCall now = call;
    now.x = x.unpack();
    now.mean = mean.unpack();
    now.invstd = invstd.unpack();
    now.gamma = gamma.unpack();
    now.beta = beta.unpack();
    if (keeps_y) now.y = y.unpack(shared_from_this());       // (refuses an output that was changed since, also beside the mask)
    if (keeps_mask) now.mask = mask.unpack();
    at::AutoDispatchBelowADInplaceOrView below;
    auto g = batch_norm_grads(now, dy, {task_should_compute_output(0), task_should_compute_output(1),
                                        task_should_compute_output(2), task_should_compute_output(3)});
    for (int i = 0; i < 4; ++i) out[i] = g[i];
    return out;
  }
  void release_variables() override {
    for (SavedVariable* v : {&x, &mean, &invstd, &gamma, &beta, &y, &mask}) v->reset_data();
  }
  std::string name() const override { return "BatchNormReluBackward"; }
};

bool known_type(const Tensor& t) {
  return t.scalar_type() == at::kFloat || t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16;
}

// The result, and in `call` what the backward pass reads.  batch_stats: statistics of this batch (and,
// with track, the running ones moved by `factor`); otherwise the running statistics.  count:
// num_batches_tracked, incremented with the statistics.  backward: a backward pass follows.
Tensor batch_norm_pass(const Tensor& x_in, const Tensor& weight, const Tensor& bias, const Tensor& running_mean,
                       const Tensor& running_var, const Tensor& count, bool batch_stats, bool track, double factor, double eps,
                       bool relu, const Tensor& residual_in, bool backward, BatchNormCall* call, bool masks) {
  at::AutoDispatchBelowADInplaceOrView below;
  const Tensor x = x_in.contiguous();
  const int64_t rows = x.size(0), c = x.size(1);
  const int code = code_of(x.scalar_type());
  void* st = hip_stream();
  Tensor gamma = as_param(weight), beta = as_param(bias), mean, invstd;
  if (gamma.defined() && beta.defined() && beta.scalar_type() != gamma.scalar_type()) beta = beta.to(gamma.scalar_type());
  Tensor y = at::empty_like(x), residual, mask;
  if (residual_in.defined()) {
    residual = residual_in.contiguous();
    TORCH_CHECK(residual.sizes() == x.sizes() && residual.scalar_type() == x.scalar_type(),
                "batch_norm: the residual does not match the input");
  }
  const int pcode = param_code(gamma, beta);
  if (batch_stats) {
    Tensor stats = at::empty({3, c}, x.options().dtype(at::kFloat));
    mean = stats[0];
    invstd = stats[2];
    Tensor var = stats[1], ws = workspace(ocnn_batch_norm_workspace_bytes((int)c), x);
    const bool moves = track && running_mean.defined();
    const bool in_place = moves && known_type(running_mean) && running_mean.scalar_type() == running_var.scalar_type() &&
                          running_mean.is_contiguous() && running_var.is_contiguous();
    if (masks && backward && residual.defined() && relu)
      if (const int64_t bytes = ocnnx_batch_norm_mask_bytes(code, rows, (int)c)) mask = at::empty({bytes}, x.options().dtype(at::kByte));
    check(ocnnx_batch_norm_training(code, ptr(x), rows, (int)c, (float)eps, (float*)mean.data_ptr(), (float*)var.data_ptr(),
                                    (float*)invstd.data_ptr(), in_place ? running_mean.data_ptr() : nullptr,
                                    in_place ? running_var.data_ptr() : nullptr,
                                    in_place ? code_of(running_mean.scalar_type()) : 0, in_place ? (float)factor : 0.f,
                                    typed<int64_t>(count), ptr(gamma), ptr(beta), pcode, relu, ptr(residual), y.data_ptr(),
                                    typed<void>(mask), ws.data_ptr(), ws.numel(), st));
    if (moves && !in_place) {
      Tensor unbiased = var * ((double)rows / (double)std::max<int64_t>(rows - 1, 1));
      running_mean.mul_(1 - factor).add_(mean.to(running_mean.scalar_type()), factor);
      running_var.mul_(1 - factor).add_(unbiased.to(running_var.scalar_type()), factor);
    }
  } else if (!backward && known_type(running_mean) && running_mean.scalar_type() == running_var.scalar_type() &&
             running_mean.is_contiguous() && running_var.is_contiguous()) {
    check(ocnnx_batch_norm_running(code, ptr(x), rows, (int)c, running_mean.data_ptr(), running_var.data_ptr(),
                                   code_of(running_mean.scalar_type()), (float)eps, ptr(gamma), ptr(beta), pcode, relu,
                                   ptr(residual), y.data_ptr(), st));
  } else {                                            // (the backward pass reads mean and invstd)
    mean = running_mean.to(at::kFloat).contiguous();
    invstd = at::rsqrt(running_var.to(at::kFloat) + eps);
    check(ocnn_batch_norm_apply(code, ptr(x), rows, (int)c, (const float*)mean.data_ptr(), (const float*)invstd.data_ptr(),
                                ptr(gamma), ptr(beta), pcode, relu, ptr(residual), y.data_ptr(), st));
  }
  if (backward) {
    *call = {x, mean, invstd, gamma, beta, residual_in.defined() && relu ? y : Tensor(), relu, batch_stats,
             residual_in.defined()};
    call->mask = mask;
    if (weight.defined()) call->wdtype = weight.scalar_type();
    if (bias.defined()) call->bdtype = bias.scalar_type();
  }
  return y;
}

Tensor batch_norm(const Tensor& x, const Tensor& weight, const Tensor& bias, const Tensor& running_mean,
                  const Tensor& running_var, const Tensor& count, bool batch_stats, bool track, double factor, double eps,
                  bool relu, const Tensor& residual) {
  const variable_list inputs{x, weight, bias, residual};
  const bool grad = any_requires_grad(inputs);
  BatchNormCall call;
  Tensor y = batch_norm_pass(x, weight, bias, running_mean, running_var, count, batch_stats, track, factor, eps, relu, residual,
                             grad, &call, true);
  if (grad) {
    auto node = make_node<BatchNormBackward>(inputs);
    node->keeps_y = call.y.defined();
    node->x = SavedVariable(call.x, false);
    node->mean = SavedVariable(call.mean, false);
    node->invstd = SavedVariable(call.invstd, false);
    if (call.gamma.defined()) node->gamma = SavedVariable(call.gamma, false);
    if (call.beta.defined()) node->beta = SavedVariable(call.beta, false);
    node->keeps_mask = call.mask.defined();
    if (node->keeps_mask) node->mask = SavedVariable(call.mask, false);
    call.mask = call.x = call.mean = call.invstd = call.gamma = call.beta = call.y = Tensor();
    node->call = std::move(call);
    torch::autograd::set_history(y, node);
    if (node->keeps_y) node->y = SavedVariable(y, true);
  }
  return y;
}

// A layer and the batch norm (+ residual, + ReLU) behind it, in evaluation and without gradients: the
// normalisation rides on the convolution's own pass over its result where the kernel takes it.
Tensor conv_bn_packed(const std::shared_ptr<ConvLayer>& layer, const Tensor& data_in, const Tensor& weights, const OptTensor& bias,
                      const Tensor& running_mean, const Tensor& running_var, double eps, const OptTensor& gamma_in,
                      const OptTensor& beta_in, bool relu, const OptTensor& residual_in, const void* packed) {
  at::AutoDispatchBelowADInplaceOrView below;
  const Tensor data = data_in.contiguous(), w = weights.to(data.scalar_type()).contiguous();
  const int cols = layer->fwd->view_cols ? layer->fwd->view_cols : layer->fwd->cout;
  TORCH_CHECK(running_mean.numel() == cols && running_var.numel() == cols,
              "running statistics of ", running_mean.numel(), " channels for a layer of ", cols);
  Tensor mean = running_mean, var = running_var;
  if (!known_type(mean) || mean.scalar_type() != var.scalar_type()) {
    mean = mean.to(at::kFloat);
    var = var.to(at::kFloat);
  }
  mean = mean.contiguous();
  var = var.contiguous();
  Tensor gamma = as_param(gamma_in.has_value() ? *gamma_in : Tensor()), beta = as_param(beta_in.has_value() ? *beta_in : Tensor());
  if (gamma.defined() && beta.defined() && beta.scalar_type() != gamma.scalar_type()) beta = beta.to(gamma.scalar_type());
  Tensor residual;
  if (residual_in.has_value()) {
    residual = residual_in->contiguous();
    TORCH_CHECK(residual.scalar_type() == data.scalar_type() && residual.dim() == 2 &&
                    residual.size(0) == layer->fwd->rows && residual.size(1) == running_mean.numel(),
                "conv_bn: the residual does not match the layer");
  }
  const ocnnx_bn bn{mean.data_ptr(), var.data_ptr(), code_of(mean.scalar_type()), (float)eps,
                    ptr(gamma), ptr(beta), param_code(gamma, beta), relu, ptr(residual)};
  return layer->fwd->run(data, layer->fwd_table, w, bias, &bn, packed);
}

Tensor conv_bn(const std::shared_ptr<ConvLayer>& layer, const Tensor& data, const Tensor& weights, const OptTensor& bias,
               const Tensor& running_mean, const Tensor& running_var, double eps, const OptTensor& gamma, const OptTensor& beta,
               bool relu, const OptTensor& residual) {
  return conv_bn_packed(layer, data, weights, bias, running_mean, running_var, eps, gamma, beta, relu, residual, nullptr);
}

// Residual blocks one behind the other, two such layers each, of which the second adds the block's input (the first block
// `shortcut` in its place, if it is given).  Their weights are packed in one launch where the kernels read them packed: the
// segmentation network of 20 blocks on 40 k points takes 1.77 ms so, 1.89 with a call and a packing launch for each layer.
struct BlockLayer {
  std::shared_ptr<ConvLayer> layer;
  Tensor weights, mean, var;
  OptTensor bias, gamma, beta;
  double eps;
  bool relu;
};
Tensor res_blocks(const std::vector<std::shared_ptr<BlockLayer>>& layers, Tensor data, const OptTensor& shortcut) {
  at::AutoDispatchBelowADInplaceOrView below;
  TORCH_CHECK(layers.size() % 2 == 0, "res_blocks: two layers a block");
  require_gpu(data);
  const int code = code_of(data.scalar_type());
  std::vector<Tensor> w(layers.size()), packed(layers.size());
  std::vector<ocnnx_pack_item> items;
  const auto flush = [&]() {
    if (!items.empty()) check(ocnnx_pack_tiles(code, items.data(), (int)items.size(), hip_stream()));
    items.clear();
  };
  for (size_t i = 0; i < layers.size(); ++i) {
    const GatherOp& op = *layers[i]->layer->fwd;
    w[i] = layers[i]->weights.to(data.scalar_type()).contiguous();
    require_gpu(w[i]);
    if (!op.takes_packed() || op.rows == 0 || w[i].numel() != (int64_t)op.K * op.cin * op.cout) continue;
    packed[i] = workspace(ocnnx_gather_tile_packed_bytes(code, op.K, op.cin, op.cout), data);
    items.push_back({ptr(w[i]), packed[i].data_ptr(), op.K, op.cin, op.cout, op.transposed, op.reverse});
    if (items.size() == OCNNX_PACK_MOST) flush();
  }
  flush();
  for (size_t i = 0; i < layers.size(); i += 2) {
    const auto pass = [&](size_t j, const Tensor& x, const OptTensor& residual) {
      const BlockLayer& l = *layers[j];
      const GatherOp& op = *l.layer->fwd;
      TORCH_CHECK(x.dim() == 2 && x.size(0) == op.rows_in && x.size(1) == op.cin, "res_blocks: the layers do not follow each other");
      return conv_bn_packed(l.layer, x, w[j], l.bias, l.mean, l.var, l.eps, l.gamma, l.beta, l.relu, residual,
                            packed[j].defined() ? packed[j].data_ptr() : nullptr);
    };
    const Tensor inner = pass(i, data, std::nullopt);
    data = pass(i + 1, inner, i == 0 && shortcut.has_value() ? shortcut : OptTensor(data));
  }
  return data;
}

// ---- octree (octree/octree.py) ----------------------------------------------------------------

struct Tree {
  std::vector<Tensor> keys, children;
  std::vector<OptTensor> index;               // of the non-empty nodes, from the deepest full layer on
  std::vector<int64_t> nnum, nnum_nempty;
  Tensor idx, points, perm, seg_start;
  OptTensor normals;
  std::vector<int64_t> versions;              // of keys and children, by torch's count of the writes to them

  // Layer d is what the build made: `child` (and `key`, unless null) are its tensors and nobody wrote to
  // them since.  (The writes to a tensor made in inference mode are not counted.)
  bool as_built(size_t d, const Tensor* key, const Tensor& child) const {
    return d < children.size() && !child.is_inference() && child.is_same(children[d]) &&
           child._version() == versions[2 * d + 1] && (!key || (key->is_same(keys[d]) && key->_version() == versions[2 * d]));
  }
};

// Waits for values that a kernel launched on `st` stores into pinned memory, n of them, none negative and all -1 until then.
// They are watched for: a synchronisation comes back several microseconds after the kernel's end, and it would wait for what has
// been launched behind that kernel.  Build and tables of 20 k points at depth 6, one after the other, 110 - 140 -> 92 - 100 us.  One
// that is waited for by itself loses (113 -> 126 - 150; the build alone, 65 k points, 89 -> 98): a synchronisation behind eight
// launches or more, which the one in the middle had kept from adding up, takes 25 us where one behind fewer takes 11.5, and the
// eighth launch 14 us of the host; in a program that goes on (a network has some hundred launches) that is so either way.
// Values that take long (a queue in front of them) are waited for, after a millisecond of watching without the interpreter lock.
void wait_for(const Tensor& values, const c10::hip::HIPStream& st) {
  const volatile int64_t* v = (const volatile int64_t*)values.data_ptr();
  const int64_t n = values.numel();
  const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(1);
  for (int64_t i = 0; i < n;) {
    if (v[i] >= 0) {
      ++i;
    } else if (std::chrono::steady_clock::now() > until) {
      st.synchronize();
      break;
    }
  }
  std::atomic_thread_fence(std::memory_order_acquire);
  for (int64_t i = 0; i < n; ++i) TORCH_CHECK(v[i] >= 0, "a kernel left no sizes");
}

// Memory for a tensor made without elements, on the current device.  The layers of a build get theirs between two kernels, when
// the sizes are known; the tensors around it are made while the sort runs.  Build and tables, us, with tensors made in between /
// so: 20 k points at depth 6 87 / 83, 60 k depth 7 106 / 100, 100 k depth 8 120 / 112, 250 k depth 9 154 / 146.
void room_for(Tensor& made, at::IntArrayRef sizes) {
  at::TensorImpl* impl = made.unsafeGetTensorImpl();
  at::StorageImpl* storage = impl->unsafe_storage().unsafeGetStorageImpl();
  impl->set_sizes_contiguous(sizes);
  const size_t bytes = (size_t)impl->numel() * made.itemsize();
  storage->set_data_ptr_noswap(storage->allocator()->allocate(bytes));
  storage->set_nbytes(bytes);
}

// Build from the points: one sort, one numbering of all layers, one wait for the layers' sizes.
Tree build_octree(Tensor pts, OptTensor normals, OptTensor batch, std::vector<float> bbmin, double factor, int depth,
                  int full_depth, int batch_size) {
  require_gpu(pts);
  for (const OptTensor* t : {&normals, &batch})              // (their pointers go to kernels)
    TORCH_CHECK(!t->has_value() || (*t)->device() == pts.device(), "build_octree: points, normals and batch ids on one device");
  pts = pts.to(at::kFloat).contiguous();
  const int64_t n = pts.size(0);
  TORCH_CHECK(!normals.has_value() || normals->numel() == 3 * n, "build_octree: a normal for every point");
  TORCH_CHECK(batch_size == 1 || (batch.has_value() && batch->numel() == n), "build_octree: a batch id for every point");
  bool batch_is_float = false;
  if (batch.has_value()) {
    batch_is_float = batch->is_floating_point();
    batch = batch->reshape({-1}).to(batch_is_float ? at::kFloat : at::kLong).contiguous();
  }
  const auto i32 = pts.options().dtype(at::kInt), i64 = pts.options().dtype(at::kLong);
  int batch_bits = 0;
  while ((1 << batch_bits) < batch_size) ++batch_bits;
  const int levels = depth - full_depth;
  const int64_t ws_bytes = ocnnx_tree_workspace_bytes(n, depth, full_depth, batch_bits);
  if (normals.has_value()) normals = normals->to(at::kFloat).contiguous();
  Tensor rows = at::empty({n, 8}, pts.options()), ws = workspace(ws_bytes, pts);
  Tree t;
  t.perm = at::empty({n}, i32);
  // (written by the kernel straight into host memory: no copy to wait for on top of the kernel)
  Tensor sizes = at::empty({levels + 1}, at::TensorOptions().dtype(at::kLong).pinned_memory(true));
  std::fill_n((int64_t*)sizes.data_ptr(), levels + 1, -1);
  const auto st = c10::hip::getCurrentHIPStream();
  check(ocnnx_tree_scan((const float*)pts.data_ptr(), n, bbmin.data(), (float)factor, ptr(batch), batch_is_float, depth,
                        full_depth, batch_bits, (const float*)ptr(normals), (float*)rows.data_ptr(), ws.data_ptr(), ws_bytes,
                        (int32_t*)t.perm.data_ptr(), (int64_t*)sizes.data_ptr(), st.stream()));
  // what does not wait for the sizes is allocated while the sort runs
  for (int d = 0; d <= full_depth; ++d) {
    t.nnum.push_back((int64_t)batch_size << (3 * d));
    t.keys.push_back(at::empty({t.nnum[d]}, i64));
    t.children.push_back(at::empty({t.nnum[d]}, i32));
  }
  t.idx = at::empty({n}, i64);
  t.seg_start = at::empty({n + 1}, i32);
  for (int d = 0; d <= depth; ++d) {                         // (room_for)
    if (d > full_depth) {
      t.keys.push_back(at::empty({0}, i64));
      t.children.push_back(at::empty({0}, i32));
    }
    t.index.push_back(d < full_depth ? OptTensor() : at::empty({0}, i32));
  }
  t.points = at::empty({0}, pts.options());
  if (normals.has_value()) t.normals = at::empty({0}, pts.options());
  std::vector<int64_t*> keys(depth + 1);
  std::vector<int32_t*> children(depth + 1), index(depth + 1);
  t.nnum.resize(depth + 1);
  t.nnum_nempty.resize(depth + 1);
  wait_for(sizes, st);
  const std::vector<int64_t> size((int64_t*)sizes.data_ptr(), (int64_t*)sizes.data_ptr() + levels + 1);
  const c10::DeviceGuard device(pts.device());
  for (int d = 0; d <= depth; ++d) {
    if (d > full_depth) {
      t.nnum[d] = 8 * size[depth - d + 1];
      room_for(t.keys[d], {t.nnum[d]});
      room_for(t.children[d], {t.nnum[d]});
    }
    t.nnum_nempty[d] = d < full_depth ? t.nnum[d] : size[depth - d];
    if (d >= full_depth) room_for(*t.index[d], {t.nnum_nempty[d]});
    keys[d] = (int64_t*)t.keys[d].data_ptr();
    children[d] = (int32_t*)t.children[d].data_ptr();
    index[d] = d < full_depth ? nullptr : (int32_t*)t.index[d]->data_ptr();
  }
  room_for(t.points, {size[0], 3});
  if (normals.has_value()) room_for(*t.normals, {size[0], 3});
  check(ocnnx_tree_fill(ws.data_ptr(), n, depth, full_depth, batch_size, batch_bits, size.data(),
                        (const int32_t*)t.perm.data_ptr(), keys.data(), children.data(), index.data(),
                        (int64_t*)t.idx.data_ptr(), (int32_t*)t.seg_start.data_ptr(), (const float*)rows.data_ptr(),
                        (float*)t.points.data_ptr(), t.normals.has_value() ? (float*)t.normals->data_ptr() : nullptr, st.stream()));
  for (int d = 0; d <= depth; ++d)
    for (const Tensor* made : {&t.keys[d], &t.children[d]}) t.versions.push_back(made->is_inference() ? 0 : made->_version());
  return t;
}

// ---- tile plans (octree/octree.py) ----------------------------------------

struct BuiltPlan {
  Tensor loc, uptr, urows, ucount;            // urows undefined: more than `pad` rows in a tile, or given up on
  std::vector<int64_t> stats;
};

// The one-pass plans of several tables, one wait for the sizes of all of them.
// groups[i]: whether table i is one of sibling groups is wanted as well.
std::vector<BuiltPlan> tile_plans(const std::vector<Tensor>& tables, int cap, int pad, const std::vector<bool>& groups) {
  const int n = (int)tables.size();
  std::vector<BuiltPlan> out(n);
  if (n == 0) return out;
  TORCH_CHECK(groups.size() == tables.size(), "tile_plans: one wish a table");
  std::vector<ocnnx_plan_item> items(n);
  const auto i32 = tables[0].options(), i64 = i32.dtype(at::kLong), i16 = i32.dtype(at::kShort);
  const int64_t tile_rows = ocnn_tile_plan_rows();
  int64_t tiles = 0;
  for (int i = 0; i < n; ++i) {
    const Tensor& t = tables[i];
    require_gpu(t);
    TORCH_CHECK(t.scalar_type() == at::kInt && t.dim() == 2 && t.is_contiguous() && t.device() == tables[0].device(),
                "tile_plans: contiguous int32 tables of one device");
    const int64_t own = (t.size(0) + tile_rows - 1) / tile_rows;
    out[i].loc = at::empty({own, t.size(1), tile_rows}, i16);
    out[i].uptr = at::empty({own + 1}, i32);
    items[i] = {typed<int32_t>(t), typed<uint16_t>(out[i].loc), typed<int32_t>(out[i].uptr), nullptr, t.size(0), tiles,
                (int)t.size(1), groups[i]};
    tiles += own;
  }
  Tensor counts = at::empty({2, std::max<int64_t>(tiles, 1)}, i32), lists = at::empty({std::max<int64_t>(tiles, 1) * pad}, i32);
  Tensor stats = at::empty({n, 6}, i64), host = at::empty({n, 6}, at::TensorOptions().dtype(at::kLong).pinned_memory(true));
  std::fill_n(typed<int64_t>(host), 6 * n, -1);
  const auto st = c10::hip::getCurrentHIPStream();
  int32_t* ucount = typed<int32_t>(counts);
  check(ocnnx_plan_build(items.data(), n, cap, pad, ucount, ucount + counts.size(1), typed<int32_t>(lists),
                         typed<int64_t>(stats), typed<int64_t>(host), st.stream()));
  wait_for(host, st);
  bool any = false;
  for (int i = 0; i < n; ++i) {
    const int64_t* v = typed<int64_t>(host) + 6 * i;
    out[i].stats.assign(v, v + 6);
    out[i].ucount = counts[0].slice(0, items[i].tile0, items[i].tile0 + out[i].uptr.size(0) - 1);
    if (v[5] != 0 || v[3] > pad) continue;
    out[i].urows = at::empty({std::max<int64_t>(v[2], 1)}, i32);
    items[i].urows = typed<int32_t>(out[i].urows);
    any = true;
  }
  if (any)
    check(ocnnx_plan_compact(items.data(), n, cap, pad, ucount, typed<int64_t>(stats), typed<int32_t>(lists), st.stream()));
  return out;
}

// The neighbour tables of layers 1 .. depth (entry 0 is left out) of an octree as `tree` was built; none if
// a layer is not, any more: keys, children and counts are public and may be assigned.
std::vector<Tensor> all_neigh(const Tree& tree, const std::vector<OptTensor>& keys_now, const std::vector<Tensor>& children,
                              const std::vector<int64_t>& nnum, const std::vector<int64_t>& nnum_nempty, int full_depth,
                              int batch_size) {
  const int depth = (int)children.size() - 1;
  std::vector<Tensor> out;
  if (children.size() != tree.children.size() || nnum != tree.nnum || nnum_nempty != tree.nnum_nempty) return out;
  for (int d = 0; d <= depth; ++d)
    if (!keys_now[d].has_value() || !tree.as_built(d, &*keys_now[d], children[d])) return out;
  const std::vector<Tensor>& keys = tree.keys;
  const std::vector<OptTensor>& index = tree.index;
  std::vector<const int64_t*> k;
  std::vector<const int32_t*> c, i;
  std::vector<int32_t*> o{nullptr};
  for (int d = 0; d <= depth; ++d) {
    require_gpu(children[d]);
    TORCH_CHECK(keys[d].is_contiguous() && children[d].is_contiguous() && keys[d].numel() == nnum[d] &&
                    children[d].numel() == nnum[d] && keys[d].scalar_type() == at::kLong &&
                    children[d].scalar_type() == at::kInt &&
                    (!index[d].has_value() || (index[d]->numel() == nnum_nempty[d] && index[d]->is_contiguous())),
                "octree layer ", d, " is inconsistent");
    k.push_back((const int64_t*)keys[d].data_ptr());
    c.push_back((const int32_t*)children[d].data_ptr());
    i.push_back((const int32_t*)ptr(index[d]));
    if (d > 0) {
      out.push_back(at::empty({nnum[d], 27}, children[d].options()));
      o.push_back((int32_t*)out.back().data_ptr());
    }
  }
  check(ocnnx_neigh_all(depth, full_depth, batch_size, nnum.data(), nnum_nempty.data(), k.data(), c.data(), i.data(),
                        o.data(), hip_stream()));
  return out;
}

Tensor or_undefined(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }

}  // namespace

PYBIND11_MODULE(ocnn_host, m) {
  namespace py = pybind11;
  // (the constructors take what every plan and pass sets: one call instead of one for each field)
  py::class_<PlanArrays, std::shared_ptr<PlanArrays>>(m, "PlanArrays")
      .def(py::init<>())
      .def(py::init([](Tensor loc, Tensor uptr, Tensor urows, int umax, int64_t total, double occupancy) {
        auto p = std::make_shared<PlanArrays>();
        p->loc = std::move(loc), p->uptr = std::move(uptr), p->urows = std::move(urows);
        p->umax = umax, p->total = total, p->occupancy = occupancy;
        return p;
      }))
#define FIELD(name) .def_readwrite(#name, &PlanArrays::name)
      FIELD(loc) FIELD(uptr) FIELD(urows) FIELD(umax) FIELD(total) FIELD(occupancy) FIELD(cptr) FIELD(ent) FIELD(lists)
          FIELD(n_blocks) FIELD(max_blocks) FIELD(n_lists) FIELD(lists_host) FIELD(group_bounds) FIELD(list_count)
#undef FIELD
      .def_property_readonly("order", [](PlanArrays& p) {
        std::lock_guard<std::mutex> lock(p.order_lock);
        return p.order.defined() ? OptTensor(p.order) : std::nullopt;
      });
  py::class_<GatherOp, std::shared_ptr<GatherOp>>(m, "GatherOp")
      .def(py::init<>())
      .def(py::init([](int64_t rows_in, int64_t rows, int K, int cin, int cout, bool transposed, bool reverse) {
        auto op = std::make_shared<GatherOp>();
        op->rows_in = rows_in, op->rows = rows, op->K = K, op->cin = cin, op->cout = cout;
        op->transposed = transposed, op->reverse = reverse;
        return op;
      }))
#define FIELD(name) .def_readwrite(#name, &GatherOp::name)
      FIELD(kernel) FIELD(K) FIELD(cin) FIELD(cout) FIELD(rows_in) FIELD(rows) FIELD(ws_bytes) FIELD(transposed)
          FIELD(reverse) FIELD(plan) FIELD(ordered) FIELD(in_index) FIELD(out_index) FIELD(children) FIELD(rows_all)
              FIELD(overflow_table) FIELD(overflow_rows) FIELD(overflow) FIELD(padded) FIELD(bias_repeat) FIELD(view_cols)
#undef FIELD
      .def("choose", &GatherOp::choose)
      .def("copy", [](const GatherOp& op) { return std::make_shared<GatherOp>(op); })
      .def("run", [](const GatherOp& op, const Tensor& data, const OptTensor& table, const Tensor& W, const OptTensor& bias) {
        pybind11::gil_scoped_release free;
        at::AutoDispatchBelowADInplaceOrView below;
        return op.run(data, or_undefined(table), W, bias);
      });
  py::class_<WgradOp, std::shared_ptr<WgradOp>>(m, "WgradOp")
      .def(py::init<>())
      .def(py::init([](int64_t rows_x, int64_t rows, int K, int ca, int cb, bool out_transposed) {
        auto op = std::make_shared<WgradOp>();
        op->rows_x = rows_x, op->rows = rows, op->K = K, op->ca = ca, op->cb = cb, op->out_transposed = out_transposed;
        return op;
      }))
#define FIELD(name) .def_readwrite(#name, &WgradOp::name)
      FIELD(kernel) FIELD(K) FIELD(ca) FIELD(cb) FIELD(rows_x) FIELD(rows) FIELD(ws_bytes) FIELD(out_transposed) FIELD(plan)
          FIELD(g_index) FIELD(shape) FIELD(overflow_table) FIELD(overflow_rows) FIELD(overflow) FIELD(padded)
#undef FIELD
      .def("choose", &WgradOp::choose)
      .def("copy", [](const WgradOp& op) { return std::make_shared<WgradOp>(op); })
      .def("seen_as", [](const WgradOp& op, std::vector<int64_t> shape) {
        auto copy = std::make_shared<WgradOp>(op);
        copy->shape = std::move(shape);
        return copy;
      })
      .def("run", [](const WgradOp& op, const Tensor& x, const Tensor& g, const OptTensor& table) {
        pybind11::gil_scoped_release free;
        at::AutoDispatchBelowADInplaceOrView below;
        return op.run(x, g, or_undefined(table));
      });
  py::class_<ConvLayer, std::shared_ptr<ConvLayer>>(m, "ConvLayer")
      .def(py::init([](std::shared_ptr<GatherOp> fwd, const OptTensor& table, bool wgrad_of_grad) {
        auto layer = std::make_shared<ConvLayer>();
        layer->fwd = std::move(fwd);
        layer->fwd_table = or_undefined(table);
        layer->wgrad_of_grad = wgrad_of_grad;
        return layer;
      }))
      .def("with_dgrad", [](const ConvLayer& layer, std::shared_ptr<GatherOp> op, const OptTensor& table) {
        auto copy = std::make_shared<ConvLayer>(layer);
        copy->dgrad = std::move(op);
        copy->dgrad_table = or_undefined(table);
        return copy;
      })
      .def("with_wgrad", [](const ConvLayer& layer, std::shared_ptr<WgradOp> op, const OptTensor& table) {
        auto copy = std::make_shared<ConvLayer>(layer);
        copy->wgrad = std::move(op);
        copy->wgrad_table = or_undefined(table);
        return copy;
      })
#define FIELD(name) .def_readonly(#name, &ConvLayer::name)
      FIELD(fwd) FIELD(dgrad) FIELD(wgrad) FIELD(fwd_table) FIELD(dgrad_table) FIELD(wgrad_table) FIELD(wgrad_of_grad)
#undef FIELD
      .def("with_table", [](const ConvLayer& layer, const Tensor& table, int64_t rows) {      // its first rows
        at::AutoDispatchBelowADInplaceOrView below;
        auto copy = std::make_shared<ConvLayer>(layer);
        copy->fwd_table = copy->dgrad_table = copy->wgrad_table = table.narrow(0, 0, rows);
        return copy;
      });
  py::class_<Tree>(m, "Tree")
#define FIELD(name) .def_readonly(#name, &Tree::name)
      FIELD(keys) FIELD(children) FIELD(index) FIELD(nnum) FIELD(nnum_nempty) FIELD(idx) FIELD(points) FIELD(normals)
          FIELD(perm) FIELD(seg_start)
#undef FIELD
      .def("layers", [](Tree t) {                 // (what an octree keeps of it)
        t.idx = t.points = t.perm = t.seg_start = Tensor();
        t.normals.reset();
        return t;
      })
      .def("as_built", [](const Tree& t, int64_t d, const Tensor& child, int64_t nnum_nempty) {
        return t.as_built(d, nullptr, child) && t.index[d].has_value() && t.index[d]->numel() == nnum_nempty;
      });
#define FIELD(name) .def_readonly(#name, &BuiltPlan::name)
  py::class_<BuiltPlan>(m, "BuiltPlan")
      FIELD(loc) FIELD(uptr) FIELD(urows) FIELD(ucount) FIELD(stats);
#undef FIELD
  m.def("tile_plans", &tile_plans, py::call_guard<py::gil_scoped_release>());
  m.def("order_many", &order_many, py::call_guard<py::gil_scoped_release>());
  m.def("build_octree", &build_octree, py::call_guard<py::gil_scoped_release>());
  m.def("all_neigh", &all_neigh, py::call_guard<py::gil_scoped_release>());
  m.attr("WGRAD_SPARSE_INVERSE") = kWgradSparseInverse;
  m.def("conv", &conv, py::call_guard<py::gil_scoped_release>());
  m.def("conv_bn", &conv_bn, py::call_guard<py::gil_scoped_release>());
  py::class_<BlockLayer, std::shared_ptr<BlockLayer>>(m, "BlockLayer")
      .def(py::init([](std::shared_ptr<ConvLayer> layer, Tensor weights, OptTensor bias, Tensor mean, Tensor var, double eps,
                       OptTensor gamma, OptTensor beta, bool relu) {
        return std::make_shared<BlockLayer>(BlockLayer{std::move(layer), std::move(weights), std::move(mean), std::move(var),
                                                       std::move(bias), std::move(gamma), std::move(beta), eps, relu});
      }));
  m.def("res_blocks", &res_blocks, py::call_guard<py::gil_scoped_release>());
  m.def("column_sum", &column_sum, py::call_guard<py::gil_scoped_release>());
  m.def(
      "rows_wgrad",
      [](const Tensor& g, const Tensor& x) {
        at::AutoDispatchBelowADInplaceOrView below;
        return rows_wgrad(g, x);
      },
      py::call_guard<py::gil_scoped_release>());
  // (the two passes without an autograd node, for an autograd.Function around them)
  m.def(
      "batch_norm_pass",
      [](const Tensor& x, const OptTensor& w, const OptTensor& b, const OptTensor& rm, const OptTensor& rv,
         const OptTensor& count, bool batch_stats, bool track, double factor, double eps, bool relu, const OptTensor& res) {
        BatchNormCall call;
        Tensor y = batch_norm_pass(x, or_undefined(w), or_undefined(b), or_undefined(rm), or_undefined(rv),
                                   or_undefined(count), batch_stats, track, factor, eps, relu, or_undefined(res), true, &call,
                                   false);
        return std::vector<Tensor>{y, call.x, call.mean, call.invstd, call.gamma, call.beta};
      },
      py::call_guard<py::gil_scoped_release>());
  m.def(
      "batch_norm_grads",
      [](const Tensor& dy, const Tensor& x, const Tensor& mean, const Tensor& invstd, const OptTensor& gamma,
         const OptTensor& beta, const OptTensor& y, bool relu, bool training, bool has_residual, at::ScalarType wdtype,
         at::ScalarType bdtype, std::array<bool, 4> want) {
        at::AutoDispatchBelowADInplaceOrView below;
        const auto g = batch_norm_grads({x, mean, invstd, or_undefined(gamma), or_undefined(beta), or_undefined(y), relu,
                                         training, has_residual, wdtype, bdtype}, dy.contiguous(), want);
        return std::vector<Tensor>(g.begin(), g.end());
      },
      py::call_guard<py::gil_scoped_release>());
  m.def(
      "batch_norm",
      [](const Tensor& x, const OptTensor& w, const OptTensor& b, const OptTensor& rm, const OptTensor& rv,
         const OptTensor& count, bool batch_stats, bool track, double factor, double eps, bool relu, const OptTensor& res) {
        return batch_norm(x, or_undefined(w), or_undefined(b), or_undefined(rm), or_undefined(rv), or_undefined(count),
                          batch_stats, track, factor, eps, relu, or_undefined(res));
      },
      py::call_guard<py::gil_scoped_release>());
}

"""OctreeConv / OctreeDeconv with the module and functional API of the
reference (ocnn/nn/octree_conv.py), running on the HIP gather-GEMM and split-K
weight-gradient kernels.

Engine view.  With T the (rows, K) neighbour table of the layer:
  forward_gemm  : out[i]  = sum_k data[T[i,k]] @ W[k]            (gather)
  backward_gemm : gin[j] += sum_{T[i,k]=j} grad[i] @ W[k]^T      (scatter)
  weight_gemm   : gW[k]   = sum_i data[T[i,k]]^T (x) grad[i]
The scatter is run as a gather too: through the mirrored slot K-1-k when the
table is centrally symmetric (stride 1, every kernel but 2x2x2) and through
the inverse table otherwise, so no atomics are involved anywhere.
"""

import threading
from typing import List

import torch
import torch.nn.functional as F
import torch.nn
from torch.autograd import Function

from .. import _lib
from ..octree.contract import tables_of
from ..octree.octree import Octree
from ..utils import list2str, resize_with_last_val, xavier_uniform_
from .octree2col import col2octree, octree2col
from .octree_pad import _depad_raw, _pad_raw, _rows, octree_depad, octree_pad


# (thresholds of the kernel selection live in the library, csrc/select.hip; these are the ones
# the layer level needs: when odd channel counts run zero-padded, and from how many rows on the
# pair-plan kernels pay for loading their weights)
PAD_MIN_ROWS = 16384
_OPS = {}                # passes without a plan, by shape (see _gather_op)
SPARSE_MAX_OCCUPANCY = 0.3
PAIRS_222_MIN_ROWS = 80000   # coarse rows from which _pairs_of_222() may pick them
SPARSE_MIN_ROWS = 32768


# Stride 2 over all nodes, seen from the coarse side.  Row q of such a table is the first child
# of the non-empty coarse node q with its neighbours at the fine offsets delta in {-1, 0, 1}^3
# (ocnn/octree/octree.py:502-506).  The fine node at child c (bits x y z) of the coarse node q'
# is therefore named by the coarse nodes q = q' + e, e in {0, 1}^3 with e <= c per axis, in slot
# delta = c - 2 e: the data gradient of the fine rows, (parents, 8 children x channels) since
# the children of a non-empty node are eight consecutive rows, is a 2x2x2 stride-1 gather over the
# NON-EMPTY COARSE nodes (slots e, the octree's own '222' table) with block weights
# Wb[e][:, c] = W[slot(c - 2 e)]^T, zero where e > c.  That gather issues 8 x 8 blocks of
# matrix work per coarse row, of which 27 are real, where the gather over the inverse table
# (fine rows x all slots of the kernel) issues 8 x 27 for 27.
_BLOCK_MAPS = {}


def _block_map(kernel, device):
  """(index (64,), mask (8, 8, 1, 1)): the kernel's slot for (e, c), e and c as 4 x + 2 y + z."""
  key = (kernel, str(device))
  if key not in _BLOCK_MAPS:
    from ..octree.octree import LUT_KERNEL
    slots = list(range(27)) if kernel == '333' else LUT_KERNEL[kernel]
    m = torch.full((8, 8), -1, dtype=torch.long)
    for e in range(8):
      for c in range(8):
        d = [((c >> a) & 1) - 2 * ((e >> a) & 1) for a in (2, 1, 0)]
        k27 = 9 * (d[0] + 1) + 3 * (d[1] + 1) + (d[2] + 1)
        if min(d) >= -1 and k27 in slots:
          m[e, c] = slots.index(k27)
    m = m.to(device)
    _BLOCK_MAPS[key] = (m.clamp_min(0).view(-1), (m >= 0).view(8, 8, 1, 1))
  return _BLOCK_MAPS[key]



def _plan_args(plan):
  """(has_plan, max distinct rows, entries of the row lists, occupancy, reuse) for the
  selection functions of the library."""
  if plan is None:
    return 0, 0, 0, 1.0, 0.0
  return 1, plan.umax, plan.total, float(plan.occupancy), float(plan.reuse)


def _plan_arrays(plan, pairs):
  """The native view of a tile plan, with its pair plan when `pairs`; kept with the plan."""
  name = '_native_pairs' if pairs else '_native'
  arrays = plan.__dict__.get(name)
  if arrays is None:
    arrays = _lib.native().PlanArrays(plan.loc, plan.uptr, plan.urows, plan.umax, plan.total, float(plan.occupancy))
    if pairs:
      pp = plan.pairs()
      arrays.cptr, arrays.ent, arrays.lists = pp.cptr, pp.ent, pp.lists
      arrays.n_blocks, arrays.max_blocks, arrays.n_lists = pp.n_blocks, pp.max_blocks, pp.n_lists
      arrays.lists_host, arrays.list_count = list(pp.lists_host), list(pp.list_count_host)
      arrays.group_bounds = list(pp.group_bounds_host)
    plan.__dict__[name] = arrays
  return arrays


def _memo(plan):
  """Where the passes made for a plan are kept: with it; those without a plan by shape."""
  memo = _OPS if plan is None else plan.__dict__.setdefault('_ops', {})
  if len(memo) > 256:
    memo.clear()
  return memo


def _gather_op(dtype, rows_in, rows, K, cin, cout, transposed, reverse, plan=None, dense=False):
  """The gather-GEMM of a shape as a native pass (csrc/host.cpp).  The library picks the kernel
  (ocnnx_gather_choose); the choice depends on the shapes and the plan only, so the pass is
  made once per plan.  The few tiles that are too dense for a plan get a pass of their own on the
  plan-free kernel, its rows put in place afterwards."""
  memo, key = _memo(plan), ('g', dtype, rows_in, rows, K, cin, cout, transposed, reverse, dense)
  op = memo.get(key)
  if op is not None:
    return op
  L, code = _lib.lib(), _lib.dtype_code_of(dtype)
  op = _lib.native().GatherOp(rows_in, rows, K, cin, cout, transposed, reverse)
  op.choose(code, dense, *_plan_args(plan), plan is not None and plan.overflow_rows is not None)
  if op.kernel == _lib.GATHER_ZERO_PADDED:
    # (to 32 channels where a kernel on the plan then takes the layer, to 16 for the plan-free one: 64 -> 4 as 64 -> 32
    # on the tile kernel / 64 -> 16 plan-free, us, f16 and fp32: 1.28 M rows 68 % set 210 / 379, 453 / 1380; 1.13 M rows 7 %
    # set 119 / 225, 214 / 728; 41 k rows 17 / 19, 27 / 60)
    wide = -(-cin // 32) * 32, -(-cout // 32) * 32
    on_plan = plan is not None and L.ocnnx_gather_choose(
        code, rows_in, rows, K, *wide, 0, *_plan_args(plan), int(plan.overflow_rows is not None)) in (_lib.GATHER_RW,
                                                                                                  _lib.GATHER_TILE)
    op.padded = _gather_op(dtype, rows_in, rows, K, wide[0], wide[1] if on_plan else -(-cout // 16) * 16, transposed, reverse,
                           plan)
  else:
    if op.kernel in (_lib.GATHER_RW, _lib.GATHER_TILE, _lib.GATHER_SPARSE, _lib.GATHER_PLANNED):
      op.plan = _plan_arrays(plan, op.kernel == _lib.GATHER_SPARSE)
      if op.ordered:
        plan.wish_order()
      if plan.overflow_rows is not None:
        op.overflow_rows, op.overflow_table = plan.overflow_rows, plan.overflow_table
        op.overflow = _gather_op(dtype, rows_in, plan.overflow_table.shape[0], K, cin, cout, transposed, reverse)
  memo[key] = op
  return op


def _indexed_gather_op(dtype, rows, data_rows, cin, cout, transposed, in_index=None, pad_to=None):
  """The dense one-slot pass that reads its rows through `in_index` (int32) and / or writes them
  through the index of the non-empty nodes (pad_to = (octree, depth)).  None when the kernel does
  not take the shape: the indexed form also addresses the tensors over all nodes with 32-bit
  offsets."""
  L = _lib.lib()
  base = _gather_op(dtype, rows, rows, 1, cin, cout, transposed, False, None, True)
  n_out = rows if pad_to is None else int(pad_to[0].nnum[pad_to[1]])
  code = _lib.dtype_code_of(dtype)
  if base.kernel not in (_lib.GATHER_DENSE_RW, _lib.GATHER_ROWS) or \
      not L.ocnn_conv_dense_rw_supported(code, max(data_rows, n_out), cin, cout):
    return None
  op = base.copy()
  op.kernel, op.ws_bytes = _lib.GATHER_DENSE_RW, L.ocnn_conv_gather_workspace_bytes(code, rows, 1, cin, cout)
  if in_index is not None:
    op.in_index = in_index
  if pad_to is not None:
    octree, depth = pad_to
    op.out_index, op.children, op.rows_all = octree._nempty_index32(depth), octree.children[depth], n_out
    assert op.out_index.numel() == rows, 'conv_gather: one result row per non-empty node'
  return op


def conv_gather(data, rows_in, table, W, cout, transposed, reverse, bias=None, plan=None, dense=False,
                in_index=None, pad_to=None):
  """out (rows, cout) = gather-GEMM over `table` (int32, (rows, K)).  With a
  tile plan of the same table (and a supported shape) the staged kernel runs.
  dense: the table is the one-slot identity (row i reads row i).
  in_index (int32, with dense only): row i reads row in_index[i] of `data`, which may then have
  more rows than the table (the compact rows of the non-empty nodes, read from a tensor over
  all nodes without a depad pass).
  pad_to = (octree, depth) (with dense only): the result comes back as octree_pad would make it,
  a row for every node of `depth`, zeros for the empty ones: the kernel writes its rows there."""
  _lib.require_gpu(data, table, W)
  table = table.contiguous()
  rows, K = table.shape
  cin, dtype = data.shape[1], data.dtype
  assert W.dtype == dtype and table.dtype == torch.int32
  assert W.numel() == K * cin * cout, 'weights do not match the table and channels'
  if dense and (in_index is not None or pad_to is not None):
    op = _indexed_gather_op(dtype, rows, data.shape[0], cin, cout, bool(transposed), in_index, pad_to)
    if op is not None:
      return op.run(data, table, W, bias)
  if in_index is not None:                                          # the other kernels take compact rows
    data = data.index_select(0, in_index.long())
  out = _gather_op(dtype, rows_in, rows, K, cin, cout, bool(transposed), bool(reverse), plan,
                   bool(dense)).run(data, table, W, bias)
  return out if pad_to is None else _pad_raw(out, *pad_to)           # .. and write compact rows


def _wgrad_op(dtype, rows_x, rows, K, ca, cb, out_transposed, plan=None, dense=False):
  """The weight gradient of a shape as a native pass; see _gather_op."""
  memo, key = _memo(plan), ('w', dtype, rows_x, rows, K, ca, cb, out_transposed, dense)
  op = memo.get(key)
  if op is not None:
    return op
  op = _lib.native().WgradOp(rows_x, rows, K, ca, cb, out_transposed)
  op.choose(_lib.dtype_code_of(dtype), dense, *_plan_args(plan)[:4])
  if op.kernel == _lib.WGRAD_ZERO_PADDED:
    op.padded = _wgrad_op(dtype, rows_x, rows, K, -(-ca // 32) * 32, -(-cb // 32) * 32, out_transposed, plan)
  if op.kernel in (_lib.WGRAD_SPARSE, _lib.WGRAD_PLANNED):
    op.plan = _plan_arrays(plan, op.kernel == _lib.WGRAD_SPARSE)
    if plan.overflow_rows is not None:                   # (their share of the sums is added)
      op.overflow_rows, op.overflow_table = plan.overflow_rows, plan.overflow_table
      op.overflow = _wgrad_op(dtype, rows_x, plan.overflow_table.shape[0], K, ca, cb, out_transposed)
  memo[key] = op
  return op


def _indexed_wgrad_op(dtype, rows, g_rows, ca, cb, g_index):
  """The dense one-slot sums with row g_index[i] of g for row i, or None (see _indexed_gather_op)."""
  base = _wgrad_op(dtype, rows, rows, 1, ca, cb, False, None, True)
  if base.kernel != _lib.WGRAD_DENSE_RW or \
      not _lib.lib().ocnn_conv_dense_wgrad_rw_supported(_lib.dtype_code_of(dtype), max(rows, g_rows), ca, cb):
    return None
  op = base.copy()
  op.g_index = g_index
  return op


def conv_wgrad(x, g, table, out_transposed=False, plan=None, dense=False, g_index=None):
  """gW (K, ca, cb) [or (K, cb, ca)] = sum_i x[T[i,k]]^T (x) g[i].  With a tile
  plan of the same table (and a supported shape) the staged kernel runs.
  dense: the table is the one-slot identity (row i reads row i).
  g_index (int32, with dense only): row i of the sum takes row g_index[i] of `g`, which may then
  have more rows than the table (see conv_gather)."""
  _lib.require_gpu(x, g, table)
  table = table.contiguous()
  rows, K = table.shape
  ca, cb, dtype = x.shape[1], g.shape[1], x.dtype
  assert dtype == g.dtype and table.dtype == torch.int32
  if g_index is not None:
    op = _indexed_wgrad_op(dtype, rows, g.shape[0], ca, cb, g_index) if dense and not out_transposed else None
    if op is not None:
      return op.run(x, g, table)
    g = g.index_select(0, g_index.long())
  assert g.shape[0] == rows
  return _wgrad_op(dtype, x.shape[0], rows, K, ca, cb, bool(out_transposed), plan, bool(dense)).run(x, g, table)


def _wgrad_inverse_op(dtype, rows_x, rows_g, cx, cg, out_transposed, plan_t):
  """The same sums as conv_wgrad, taken over the INVERSE table (row j, slot k -> the row i
  with table[i][k] == j; plan_t is its tile plan): gW[k] = sum_j x[j]^T (x) g[Tt[j,k]].  For
  tables in which every row is pointed at from one slot only (2x2x2 stride 2: a node has one
  parent) the inverse has 1 / K of its entries set and tiles of few distinct rows, which is
  what the pair-plan kernel is made for.  None when the kernel does not take the shape."""
  L, K, code = _lib.lib(), plan_t.K, _lib.DTYPE_CODE.get(dtype, -1)
  if not (plan_t.rows == rows_x and plan_t.rows >= SPARSE_MIN_ROWS and plan_t.occupancy <= SPARSE_MAX_OCCUPANCY and
          L.ocnn_conv_wgrad_sparse_supported(code, rows_g, rows_x, K, cg, cx, plan_t.umax)):
    return None
  memo, key = _memo(plan_t), ('i', dtype, rows_x, rows_g, cx, cg, out_transposed)
  op = memo.get(key)
  if op is None:
    native = _lib.native()
    op = native.WgradOp()
    op.kernel, op.K, op.ca, op.cb, op.out_transposed = native.WGRAD_SPARSE_INVERSE, K, cx, cg, out_transposed
    op.rows_x, op.rows = rows_g, rows_x                    # rows the inverse table points at; its own rows
    op.ws_bytes = L.ocnn_conv_wgrad_sparse_workspace_bytes(rows_x, cg, cx)
    op.plan = _plan_arrays(plan_t, True)
    if plan_t.overflow_rows is not None:                   # (tiles too dense for the plan)
      op.overflow_rows, op.overflow_table = plan_t.overflow_rows, plan_t.overflow_table
      op.overflow = _wgrad_op(dtype, rows_g, plan_t.overflow_table.shape[0], K, cg, cx, not out_transposed)
    memo[key] = op
  return op


def column_sum(g):
  """g.sum(0) with a fixed reduction order."""
  return _lib.native().column_sum(g)


class OctreeConvBase:
  """Shapes and the three engine passes (ocnn/nn/octree_conv.py:26-202)."""

  def __init__(self, in_channels: int, out_channels: int, kernel_size: List[int] = [3],
               stride: int = 1, nempty: bool = False, max_buffer: int = int(2e8)):
    super().__init__()
    self.in_channels = in_channels
    self.out_channels = out_channels
    self.kernel_size = resize_with_last_val(kernel_size)
    self.kernel = list2str(self.kernel_size)
    self.stride = stride
    self.nempty = nempty
    self.max_buffer = max_buffer      # accepted for compatibility; nothing is buffered
    self.kdim = self.kernel_size[0] * self.kernel_size[1] * self.kernel_size[2]
    self.in_conv = in_channels if self.is_conv_layer() else out_channels
    self.out_conv = out_channels if self.is_conv_layer() else in_channels
    self.weights_shape = (self.kdim, self.in_conv, self.out_conv)

  def is_conv_layer(self):
    raise NotImplementedError

  def setup(self, octree, depth: int):
    """Heights of input/output and the table (ocnn/nn/octree_conv.py:51-100)."""
    # (an octree of another class gets its tables from its public members, octree/contract.py)
    octree = tables_of(octree)
    self.in_depth = self.out_depth = self.neigh_depth = depth
    if self.stride == 2:
      if self.is_conv_layer():
        self.out_depth = depth - 1
      else:
        self.out_depth = depth + 1
        self.neigh_depth = depth + 1
    if self.nempty:
      in_h = octree.nnum_nempty[self.in_depth]
      out_h = octree.nnum_nempty[self.out_depth]
    else:
      in_h = octree.nnum[self.in_depth]
      out_h = octree.nnum[self.out_depth]
      if self.stride == 2:
        if self.is_conv_layer():
          out_h = octree.nnum_nempty[self.out_depth]
        else:
          in_h = octree.nnum_nempty[self.in_depth]
    self.in_h, self.out_h = int(in_h), int(out_h)
    self.in_shape = (self.in_h, self.in_channels)
    self.out_shape = (self.out_h, self.out_channels)
    self.octree = octree
    self.neigh = octree._table(self.neigh_depth, self.kernel, self.stride, self.nempty)
    # rows on the "fine" side of the table (what its entries index)
    self.fine_h = self.in_h if self.is_conv_layer() else self.out_h
    self.symmetric = self.stride == 1 and self.kernel != '222'
    # 2x2x2 stride 2 over all nodes: row p of the table is exactly the 8 children 8p .. 8p+7
    # (children of a non-empty node are numbered consecutively, ocnn/octree/octree.py:235-259),
    # so the layer is a dense GEMM on the (P, 8 * C) view of the fine side: no gather at all
    self.dense_children = (self.kernel == '222' and self.stride == 2 and not self.nempty and
                           self.fine_h == 8 * self.neigh.shape[0])
    # the other kernels at stride 2 over all nodes: the data gradient in block form (_block_map)
    self.coarse_depth = self.out_depth if self.is_conv_layer() else self.in_depth
    self.block_children = (self.kernel != '222' and self.stride == 2 and not self.nempty and
                           self.fine_h == 8 * self.neigh.shape[0])

  def check_and_init(self, data: torch.Tensor):
    check = tuple(data.shape) == self.in_shape
    assert check, ('The shape of input data is wrong: ' +
                   'expected {}, got {}.'.format(self.in_shape, data.shape))

  def _inverse_table(self):
    return self.octree._table_t(self.neigh_depth, self.kernel, self.stride, self.nempty,
                                self.fine_h)

  def _plan(self, dtype, rows, cin, cout, inverse=False):
    """Tile plan of the table (or its inverse), when a kernel on it takes the shape."""
    L, code = _lib.lib(), _lib.DTYPE_CODE.get(dtype, -1)
    if self.neigh.shape[0] >= PAD_MIN_ROWS:               # odd channel counts run zero-padded
      cin, cout = -(-cin // 32) * 32, -(-cout // 32) * 32
    if not (L.ocnnx_gather_tile_supported(code, rows, self.kdim, cin, cout, 0) or
            L.ocnn_conv_gather_rw_supported(code, rows, self.kdim, cin, cout, 0) or
            L.ocnn_conv_gather_planned_supported(code, rows, cin, cout) or
            L.ocnn_conv_gather_sparse_supported(code, rows, self.kdim, cin, cout, 0) or
            L.ocnn_conv_wgrad_planned_supported(code, rows, rows, self.kdim, cin, cout, 0)):
      return None
    return self.octree._plan(self.neigh_depth, self.kernel, self.stride, self.nempty, inverse, self.fine_h)

  def _identity(self, rows, device):
    """(rows, 1) table [0, 1, ..]: the one-slot 'gather' of the dense form."""
    cache = self.octree.__dict__.setdefault('_identity_tables', {})
    key = (rows, str(device))
    if key not in cache:
      cache[key] = torch.arange(rows, dtype=torch.int32, device=device).view(rows, 1)
    return cache[key]

  # The three passes as (native pass, table).  None: not one pass; the *_gemm methods put it together.
  def forward_op(self, dtype, pad_to=None):
    """(fine rows, in_conv) -> (table rows, out_conv); see forward_gemm."""
    if self.dense_children:
      P, cin = self.neigh.shape[0], 8 * self.in_conv
      op = (_gather_op(dtype, P, P, 1, cin, self.out_conv, False, False, None, True) if pad_to is None
            else _indexed_gather_op(dtype, P, P, cin, self.out_conv, False, None, pad_to))
      return op and (op, self._identity(P, self.neigh.device))
    if pad_to is not None:
      return None
    rows, K = self.neigh.shape
    plan = self._plan(dtype, self.fine_h, self.in_conv, self.out_conv)
    return _gather_op(dtype, self.fine_h, rows, K, self.in_conv, self.out_conv, False, False, plan), self.neigh

  def backward_op(self, dtype, coarse_index=None, coarse_rows=0):
    """(table rows, out_conv) -> (fine rows, in_conv); see backward_gemm."""
    rows, K = self.neigh.shape
    if self.dense_children:
      cout = 8 * self.in_conv
      index = None if coarse_index is None else coarse_index
      op = _indexed_gather_op(dtype, rows, max(rows, coarse_rows), self.out_conv, cout, True, index)
      if op is None:
        return None
      op.bias_repeat, op.view_cols = 8, self.in_conv
      return op, self._identity(rows, self.neigh.device)
    if coarse_index is not None or self.block_children:
      return None
    if self.symmetric:
      plan = self._plan(dtype, rows, self.out_conv, self.in_conv)
      return _gather_op(dtype, rows, rows, K, self.out_conv, self.in_conv, True, True, plan), self.neigh
    plan = self._plan(dtype, rows, self.out_conv, self.in_conv, inverse=True)
    return (_gather_op(dtype, rows, self.fine_h, K, self.out_conv, self.in_conv, True, False, plan),
            self._inverse_table())

  def _pairs_of_222(self, dtype):
    """The weight gradient of 2x2x2 stride 2 over the pairs of the inverse table: only where the planned kernel does
    not take the layer, and then with channels that leave the plan-free kernel's 64-channel tiles part empty, on
    many rows (us, f16, pairs / planned: 64 -> 128 on 290 k rows 121 / 70, 947 k 266 / 123, 96 -> 96 138 / 96, 249 / 234;
    pairs / plan-free: 64 -> 128 on 96 k rows 86 / 46, 160 k 113 / 66, 96 -> 96 84 / 111, 131 / 141, on 68 k 78 / 59)."""
    rows, cin, cout = self.neigh.shape[0], self.in_conv, self.out_conv
    plan = self._plan(dtype, self.fine_h, cin, cout)
    if plan is not None and _lib.lib().ocnn_conv_wgrad_planned_supported(
        _lib.DTYPE_CODE.get(dtype, -1), self.fine_h, rows, self.kdim, cin, cout, plan.umax):
      return False
    return rows >= PAIRS_222_MIN_ROWS and min(cin, cout) > 64 and cin % 64 != 0 and cout % 64 != 0

  def weight_op(self, dtype, out_transposed=False, coarse_index=None, coarse_rows=0):
    """data (fine rows), grad (table rows) -> (K, in_conv, out_conv); see weight_gemm."""
    rows, K = self.neigh.shape
    if self.dense_children:
      ca = 8 * self.in_conv
      if out_transposed:
        return None
      op = _indexed_wgrad_op(dtype, rows, max(rows, coarse_rows), ca, self.out_conv, coarse_index) \
          if coarse_index is not None else None
      if op is None:
        return None
      op = op.seen_as([8, self.in_conv, self.out_conv])
      return op, self._identity(rows, self.neigh.device)
    if coarse_index is not None or (self.block_children and self.kernel == '333'):
      return None
    # (3x3x3 over all nodes: 20 of the 27 slots of a table row are set, and the plan-free kernel
    # over the table is faster than the pairs of the inverse)
    if self.stride == 2 and rows >= SPARSE_MIN_ROWS // 8 and \
        ((self.kernel == '333' and self.nempty) or (self.kernel == '222' and self._pairs_of_222(dtype))) and \
        _lib.lib().ocnn_conv_wgrad_sparse_supported(_lib.DTYPE_CODE.get(dtype, -1), rows, self.fine_h, self.kdim,
                                                    self.out_conv, self.in_conv, 0):
      plan_t = self.octree._plan(self.neigh_depth, self.kernel, self.stride, self.nempty, True, self.fine_h)
      op = _wgrad_inverse_op(dtype, self.fine_h, rows, self.in_conv, self.out_conv, out_transposed, plan_t)
      if op is not None:
        return op, self.neigh
    plan = self._plan(dtype, self.fine_h, self.in_conv, self.out_conv)
    return _wgrad_op(dtype, self.fine_h, rows, K, self.in_conv, self.out_conv, out_transposed, plan), self.neigh

  def forward_gemm(self, data, weights, bias=None, pad_to=None):
    """(fine rows, in_conv) -> (table rows, out_conv).  pad_to = (octree, depth): the result
    padded to all nodes of `depth` (octree_pad of the table rows)."""
    made = _lib.unrecorded(self.forward_op, data.dtype, pad_to)
    if made is not None:
      return made[0].run(data, made[1], weights, bias)
    return _pad_raw(self.forward_gemm(data, weights, bias), *pad_to)

  def backward_gemm(self, grad, weights, bias=None, coarse_index=None):
    """(table rows, out_conv) -> (fine rows, in_conv).  coarse_index (int32): `grad` holds the
    table's rows at these rows of a larger tensor (all nodes of the depth, not only the
    non-empty ones the table has rows for)."""
    made = _lib.unrecorded(lambda: self.backward_op(grad.dtype, coarse_index, grad.shape[0]))
    if made is not None:
      return made[0].run(grad, made[1], weights, bias)
    if coarse_index is not None:
      grad = grad.index_select(0, coarse_index.long())
    if self.dense_children:
      # gin.view(P, 8 * in_conv) = grad @ W'^T with W' = weights.view(8 * in_conv, out_conv)
      P = self.neigh.shape[0]
      out = conv_gather(grad, P, self._identity(P, grad.device), weights.view(1, 8 * self.in_conv, self.out_conv),
                        8 * self.in_conv, True, False, None if bias is None else bias.repeat(8), None, dense=True)
      return out.view(8 * P, self.in_conv)
    if self.block_children:
      out = self._backward_blocks(grad, weights, bias)
      if out is not None:
        return out
    plan = self._plan(grad.dtype, grad.shape[0], self.out_conv, self.in_conv, inverse=True)
    return conv_gather(grad, grad.shape[0], self._inverse_table(), weights, self.in_conv, True, False, bias, plan)

  def _backward_blocks(self, grad, weights, bias):
    """backward_gemm of a stride-2 layer over all nodes as a 2x2x2 stride-1 gather over the
    non-empty coarse nodes into the (parents, 8 x in_conv) view of the fine rows (_block_map).
    None where the kernels for wide layers do not take the shape (the caller then goes over
    the inverse table)."""
    L, code = _lib.lib(), _lib.DTYPE_CODE.get(grad.dtype, -1)
    P, wide = self.neigh.shape[0], 8 * self.in_conv
    octree = self.octree
    plan = octree._plan(self.coarse_depth, '222', 1, True)
    if L.ocnn_conv_gather_choose(code, P, P, 8, self.out_conv, wide, 0, *_plan_args(plan)) != _lib.GATHER_WIDE:
      return None
    index, valid = _block_map(self.kernel, grad.device)
    blocks = weights.view(self.kdim, self.in_conv, self.out_conv).index_select(0, index)
    blocks = blocks.view(8, 8, self.in_conv, self.out_conv) * valid.to(weights.dtype)          # e, c, in, out
    blocks = blocks.permute(0, 3, 1, 2).reshape(8, self.out_conv, wide)                        # e, out, (c, in)
    out = conv_gather(grad, P, octree._table(self.coarse_depth, '222', 1, True), blocks, wide, False, False,
                      None if bias is None else bias.repeat(8), plan)
    return out.view(8 * P, self.in_conv)

  def _weight_blocks(self, data, grad, out_transposed):
    """weight_gemm of a stride-2 layer over all nodes on the planned kernel: the fine rows as
    (parents, 8 x in_conv), the table of the eight coarse nodes whose children a row's slots
    reach (offsets {-1, 0}^3: slot delta of coarse node q reads child c = delta mod 2 of the node
    at e = floor(delta / 2)), sums (8, 8 x in_conv, out_conv) of which the kernel's slots are 27
    blocks at most.  None where the planned kernel does not take the shape."""
    L, code = _lib.lib(), _lib.DTYPE_CODE.get(data.dtype, -1)
    P, wide = self.neigh.shape[0], 8 * self.in_conv
    octree = self.octree
    plan = octree._plan(self.coarse_depth, '222m', 1, True)
    if L.ocnn_conv_wgrad_choose(code, P, P, 8, wide, self.out_conv, 0, *_plan_args(plan)[:4]) != _lib.WGRAD_PLANNED:
      return None
    sums = conv_wgrad(data.view(P, wide), grad, octree._table(self.coarse_depth, '222m', 1, True), False, plan)
    key = ('w', self.kernel, str(data.device))
    if key not in _BLOCK_MAPS:
      from ..octree.octree import LUT_KERNEL
      slots = list(range(27)) if self.kernel == '333' else LUT_KERNEL[self.kernel]
      e, c = [], []
      for k27 in slots:
        d = [k27 // 9 - 1, (k27 // 3) % 3 - 1, k27 % 3 - 1]
        e.append(sum((0 if v == -1 else 1) << (2 - a) for a, v in enumerate(d)))      # '222m' slot: offsets -1 -> 0, 0 -> 1
        c.append(sum((v & 1) << (2 - a) for a, v in enumerate(d)))                    # child bit: 1 for delta = +-1
      _BLOCK_MAPS[key] = (torch.tensor(e, device=data.device), torch.tensor(c, device=data.device))
    e, c = _BLOCK_MAPS[key]
    gw = sums.view(8, 8, self.in_conv, self.out_conv)[e, c]                             # (K, in_conv, out_conv)
    return gw.transpose(1, 2).contiguous() if out_transposed else gw

  def weight_gemm(self, data, grad, out_transposed=False, coarse_index=None):
    """data: fine rows; grad: table rows -> (K, in_conv, out_conv).  coarse_index: as in
    backward_gemm."""
    made = _lib.unrecorded(lambda: self.weight_op(data.dtype, out_transposed, coarse_index, grad.shape[0]))
    if made is not None:
      return made[0].run(data, grad, made[1])
    if self.dense_children:
      P = self.neigh.shape[0]
      gw = conv_wgrad(data.view(P, 8 * self.in_conv), grad, self._identity(P, data.device), False,
                      None, dense=True, g_index=coarse_index).view(8, self.in_conv, self.out_conv)
      return gw.transpose(1, 2).contiguous() if out_transposed else gw
    if coarse_index is not None:
      grad = grad.index_select(0, coarse_index.long())
      return self.weight_gemm(data, grad, out_transposed)
    gw = self._weight_blocks(data, grad, out_transposed)  # (8 x 8 blocks issued: a loss for 3 or 9 slots)
    if gw is not None:
      return gw
    plan = self._plan(data.dtype, data.shape[0], self.in_conv, self.out_conv)
    return conv_wgrad(data, grad, self.neigh, out_transposed, plan)


class _OctreeConv(OctreeConvBase):
  def is_conv_layer(self): return True


class _OctreeDeconv(OctreeConvBase):
  def is_conv_layer(self): return False


class OctreeConvFunction(Function):
  """Autograd wiring of the convolution (ocnn/nn/octree_conv.py:219-254).  `bias` (optional)
  is added in the epilogue of the gather-GEMM kernel instead of by a pass of its own; its
  gradient is the fixed-order column sum of the output gradient.  `padded` (stride 2 over all
  nodes): the result comes back padded to all nodes of depth - 1 (what the module's octree_pad
  does, ocnn/nn/octree_conv.py:388-389), and the backward pass reads the rows of the non-empty
  nodes straight from the padded gradient through the octree's index of them: no depad pass."""

  @staticmethod
  def forward(ctx, data, weights, octree, depth: int, in_channels: int, out_channels: int,
              kernel_size: List[int] = [3, 3, 3], stride: int = 1, nempty: bool = False,
              max_buffer: int = int(2e8), bias=None, padded: bool = False):
    eng = _OctreeConv(in_channels, out_channels, kernel_size, stride, nempty, max_buffer)
    _lib.unrecorded(eng.setup, octree, depth)
    octree = eng.octree
    eng.check_and_init(data)
    data = data.contiguous()
    weights = weights.to(data.dtype).contiguous()
    out = eng.forward_gemm(data, weights, bias, pad_to=(octree, depth - 1) if padded else None)
    ctx.save_for_backward(data, weights)
    ctx.eng = eng
    ctx.pad_depth = depth - 1 if padded else None
    return out

  @staticmethod
  def backward(ctx, grad):
    data, weights = ctx.saved_tensors
    eng = ctx.eng
    grad = grad.contiguous()
    index = None
    if ctx.pad_depth is not None:
      if eng.dense_children and not ctx.needs_input_grad[10]:
        index = eng.octree._nempty_index32(ctx.pad_depth)       # the dense kernels read through it
      else:
        grad = _depad_raw(grad, eng.octree, ctx.pad_depth)      # one copy for all three gradients
    grad_out = eng.backward_gemm(grad, weights, coarse_index=index) if ctx.needs_input_grad[0] else None
    grad_w = eng.weight_gemm(data, grad, coarse_index=index) if ctx.needs_input_grad[1] else None
    grad_b = column_sum(grad) if ctx.needs_input_grad[10] else None
    return (grad_out, grad_w) + (None,) * 8 + (grad_b, None)


class OctreeDeconvFunction(Function):
  """Autograd wiring of the deconvolution (ocnn/nn/octree_conv.py:257-292).  `padded` (stride 2
  over all nodes): `data` has a row for every node of `depth` and the rows of the non-empty
  ones are read through the octree's index of them (what the module's octree_depad would copy
  out first, ocnn/nn/octree_conv.py:450-451); the data gradient comes back padded."""

  @staticmethod
  def forward(ctx, data, weights, octree, depth: int, in_channels: int, out_channels: int,
              kernel_size: List[int] = [3, 3, 3], stride: int = 1, nempty: bool = False,
              max_buffer: int = int(2e8), bias=None, padded: bool = False):
    eng = _OctreeDeconv(in_channels, out_channels, kernel_size, stride, nempty, max_buffer)
    _lib.unrecorded(eng.setup, octree, depth)
    octree = eng.octree
    index = None
    data = data.contiguous()
    if padded:
      assert tuple(data.shape) == (_rows(octree, depth)[0], in_channels), 'The shape of input data is wrong'
      if eng.dense_children:
        index = octree._nempty_index32(depth)                   # the dense kernels read through it
      else:
        data = _depad_raw(data, octree, depth)                  # one copy for forward and weight gradient
    else:
      eng.check_and_init(data)
    weights = weights.to(data.dtype).contiguous()
    out = eng.backward_gemm(data, weights, bias, coarse_index=index)
    ctx.save_for_backward(data, weights)
    ctx.eng = eng
    ctx.pad_depth = depth if padded else None
    ctx.indexed = index is not None
    return out

  @staticmethod
  def backward(ctx, grad):
    data, weights = ctx.saved_tensors
    eng = ctx.eng
    grad = grad.contiguous()
    index = eng.octree._nempty_index32(ctx.pad_depth) if ctx.indexed else None
    grad_out = None
    if ctx.needs_input_grad[0]:
      grad_out = eng.forward_gemm(grad, weights,
                                  pad_to=None if ctx.pad_depth is None else (eng.octree, ctx.pad_depth))
    # weights are (K, out_channels, in_channels): x = grad (fine side), g = data
    grad_w = eng.weight_gemm(grad, data, coarse_index=index) if ctx.needs_input_grad[1] else None
    grad_b = column_sum(grad) if ctx.needs_input_grad[10] else None
    return (grad_out, grad_w) + (None,) * 8 + (grad_b, None)


class _NativeLayerFunction(Function):
  """A layer's native passes as an autograd.Function, for calls that something records (_lib.recorded)."""

  @staticmethod
  def forward(ctx, data, weights, bias, native):
    data, weights = data.contiguous(), weights.to(data.dtype).contiguous()
    ctx.save_for_backward(data, weights)
    ctx.native = native
    return native.fwd.run(data, native.fwd_table, weights, bias)

  @staticmethod
  def backward(ctx, grad):
    (data, weights), native, grad = ctx.saved_tensors, ctx.native, grad.contiguous()
    x, g = (grad, data) if native.wgrad_of_grad else (data, grad)
    return (native.dgrad.run(grad, native.dgrad_table, weights, None) if ctx.needs_input_grad[0] else None,
            native.wgrad.run(x, g, native.wgrad_table) if ctx.needs_input_grad[1] else None,
            column_sum(grad) if ctx.needs_input_grad[2] else None, None)


def call_native(native, data, weights, bias):
  """A layer through its native passes (those that the call needs)."""
  if _lib.recorded():
    return _NativeLayerFunction.apply(data, weights, bias, native)
  return _lib.native().conv(native, data, weights, bias)


class _Layer:
  """A layer on an octree in one data type: its native passes and the shape of its input.  (Kept by
  the octree, and therefore without a reference to it.)

  The backward passes are made when a call first needs them.  Threads share the layer, and a call that
  runs holds the native object without the interpreter lock: that object is never changed, one with the
  further pass takes its place."""

  def __init__(self, eng, dtype, padded):
    self.dtype, self.padded = dtype, padded    # padded: stride 2 over all nodes, octree_pad / octree_depad folded in
    self.conv = eng.is_conv_layer()
    self.pad_depth = (eng.out_depth if self.conv else eng.in_depth) if padded else None
    self.shape = eng.in_shape if self.conv or not padded else (int(eng.octree.nnum[eng.in_depth]), eng.in_channels)
    self.dgrad = self.wgrad = None             # None = not made yet, False = not one pass
    self._lock = threading.Lock()
    made = self._pass(eng, True)
    self.ok = made is not None                 # the forward pass is one native pass
    self.native = _lib.native().ConvLayer(*made, not self.conv) if self.ok else None

  def _coarse(self, octree):
    """(index, rows) of the padded side: what the passes read the coarse rows through."""
    if not self.padded:
      return None, 0
    return octree._nempty_index32(self.pad_depth), int(octree.nnum[self.pad_depth])

  def _pass(self, eng, forward):
    if forward == self.conv:
      return eng.forward_op(self.dtype, (eng.octree, self.pad_depth) if self.padded else None)
    return eng.backward_op(self.dtype, *self._coarse(eng.octree))

  def make_dgrad(self, make_engine):
    with self._lock:
      if self.dgrad is None:
        made = self._pass(make_engine(), False)
        if made is not None:
          self.native = self.native.with_dgrad(*made)
        self.dgrad = made is not None

  def make_wgrad(self, make_engine):
    with self._lock:
      if self.wgrad is None:
        eng = make_engine()
        made = eng.weight_op(self.dtype, False, *self._coarse(eng.octree))
        if made is not None:
          self.native = self.native.with_wgrad(*made)
        self.wgrad = made is not None


_WRONG_SHAPE = 'The shape of input data is wrong: expected {}, got {}.'


def _layer_on(engine, dtype, octree, depth, in_channels, out_channels, kernel_size, stride, nempty, max_buffer, padded):
  """The layer's native passes, made at its first call on this octree and kept with it (not `ok` where the forward pass
  is not one native pass), and a function that makes its engine."""
  key = (engine, depth, tuple(kernel_size), stride, nempty, in_channels, out_channels, dtype, padded, SPARSE_MIN_ROWS)
  layer = octree._layers.get(key)

  def made_engine():
    eng = engine(in_channels, out_channels, kernel_size, stride, nempty, max_buffer)
    eng.setup(octree, depth)
    return eng

  if layer is None:
    layer = octree._layers.setdefault(key, _lib.unrecorded(lambda: _Layer(made_engine(), dtype, padded)))
  return layer, made_engine


def _apply(engine, function, data, weights, octree, depth, in_channels, out_channels, kernel_size, stride, nempty,
           max_buffer, bias, padded):
  """The layer through the native node where each of its passes is one, through `function` otherwise."""
  layer = None
  if isinstance(octree, Octree) and data.is_cuda and data.dtype in _lib.DTYPE_CODE:
    layer, made_engine = _layer_on(engine, data.dtype, octree, depth, in_channels, out_channels, kernel_size, stride, nempty,
                                   max_buffer, padded)
  if layer is not None and layer.ok:
    assert data.shape == layer.shape, _WRONG_SHAPE.format(layer.shape, tuple(data.shape))
    ok = True
    if torch.is_grad_enabled():
      # (the rows of a padded gradient are summed over the non-empty nodes only: the other route)
      if padded and layer.conv and bias is not None and bias.requires_grad:
        ok = False
      if ok and data.requires_grad:
        if layer.dgrad is None:
          _lib.unrecorded(layer.make_dgrad, made_engine)
        ok = layer.dgrad
      if ok and weights.requires_grad:
        if layer.wgrad is None:
          _lib.unrecorded(layer.make_wgrad, made_engine)
        ok = layer.wgrad
    if ok:
      return call_native(layer.native, data, weights, bias)
  return function.apply(data, weights, octree, depth, in_channels, out_channels, kernel_size, stride, nempty,
                        max_buffer, bias, padded)


def octree_conv(data, weights, octree, depth: int, in_channels: int, out_channels: int,
                kernel_size: List[int] = [3, 3, 3], stride: int = 1, nempty: bool = False,
                max_buffer: int = int(2e8), bias=None, padded: bool = False):
  """Functional form (ocnn/nn/octree_conv.py:296), with an optional bias that the kernel adds
  and, for stride 2 over all nodes, the octree_pad of the result folded in (`padded`)."""
  return _apply(_OctreeConv, OctreeConvFunction, data, weights, octree, depth, in_channels, out_channels, kernel_size,
                stride, nempty, max_buffer, bias, padded)


def octree_deconv(data, weights, octree, depth: int, in_channels: int, out_channels: int,
                  kernel_size: List[int] = [3, 3, 3], stride: int = 1, nempty: bool = False,
                  max_buffer: int = int(2e8), bias=None, padded: bool = False):
  """Functional form (ocnn/nn/octree_conv.py:297), with an optional bias that the kernel adds
  and, for stride 2 over all nodes, the octree_depad of the input folded in (`padded`)."""
  return _apply(_OctreeDeconv, OctreeDeconvFunction, data, weights, octree, depth, in_channels, out_channels,
                kernel_size, stride, nempty, max_buffer, bias, padded)


class OctreeConv(OctreeConvBase, torch.nn.Module):
  """Octree convolution.  Constructor, parameters (`weights` (kdim, Cin, Cout),
  `bias`) and forward(data, octree, depth) follow ocnn/nn/octree_conv.py:300-431.
  `max_buffer` is accepted and ignored (nothing is buffered).  method='explicit_gemm' takes
  the reference's im2col route (octree2col + torch.mm, ocnn/nn/octree_conv.py:366-376); every
  other method name of the reference ('block_gemm', 'triton') and 'hip' run the HIP engine,
  for every kernel shape, stride and nempty mode."""

  def __init__(self, in_channels: int, out_channels: int, kernel_size: List[int] = [3],
               stride: int = 1, nempty: bool = False, method: str = 'triton',
               use_bias: bool = False, max_buffer: int = int(2e8)):
    super().__init__(in_channels, out_channels, kernel_size, stride, nempty, max_buffer)
    self.use_bias = use_bias
    self.method = self.check_method(method)
    self.weights = torch.nn.Parameter(torch.Tensor(*self.weights_shape))
    self.bias = torch.nn.Parameter(torch.Tensor(out_channels)) if use_bias else None
    self.reset_parameters()

  def check_method(self, method: str):
    if method not in ('explicit_gemm', 'block_gemm', 'triton', 'hip'):
      raise ValueError('Unknown method: {}'.format(method))
    return 'explicit_gemm' if method == 'explicit_gemm' else 'hip'

  def explicit_gemm(self, data: torch.Tensor, octree, depth: int):
    """im2col, then one matrix product (autograd differentiates the torch ops)."""
    col = octree2col(data, tables_of(octree), depth, self.kernel, self.stride, self.nempty)
    return torch.mm(col.flatten(1), self.weights.to(data.dtype).flatten(0, 1))

  def reset_parameters(self):
    xavier_uniform_(self.weights)
    if self.use_bias:
      torch.nn.init.zeros_(self.bias)

  def is_conv_layer(self): return True

  def forward(self, data: torch.Tensor, octree, depth: int):
    pad = self.stride == 2 and not self.nempty
    if self.method == 'explicit_gemm':
      out = self.explicit_gemm(data, octree, depth)
    else:
      # bias: in the kernel's epilogue; the pad: inside the function, whose backward pass then
      # needs no depad
      return octree_conv(data, self.weights, octree, depth, self.in_channels, self.out_channels,
                         self.kernel_size, self.stride, self.nempty, self.max_buffer,
                         self.bias if self.use_bias else None, pad)
    if self.use_bias:
      out = out + self.bias.to(out.dtype)
    if pad:
      out = octree_pad(out, octree, depth - 1)
    return out

  def native_layer(self, data: torch.Tensor, octree, depth: int):
    """The native passes of this layer on `octree`, or None where it takes another route."""
    if self.method != 'hip' or not (isinstance(octree, Octree) and data.is_cuda and data.dtype in _lib.DTYPE_CODE):
      return None
    layer, _ = _layer_on(_OctreeConv if self.is_conv_layer() else _OctreeDeconv, data.dtype, octree, depth,
                         self.in_channels, self.out_channels, self.kernel_size, self.stride, self.nempty,
                         self.max_buffer, self.stride == 2 and not self.nempty)
    if not layer.ok:
      return None
    assert data.shape == layer.shape, _WRONG_SHAPE.format(layer.shape, tuple(data.shape))
    return layer.native

  def native_of_stride_1(self, dtype, shape, octree, depth: int):
    """native_layer for data of this type and shape that is still to be made, of a layer that keeps the rows."""
    if self.method != 'hip' or self.stride != 1 or not self.is_conv_layer():
      return None
    layer, _ = _layer_on(_OctreeConv, dtype, octree, depth, self.in_channels, self.out_channels, self.kernel_size, 1,
                         self.nempty, self.max_buffer, False)
    return layer.native if layer.ok and layer.shape == shape else None

  def extra_repr(self) -> str:
    return ('in_channels={}, out_channels={}, kernel_size={}, stride={}, '
            'nempty={}, bias={}, method={}').format(
                self.in_channels, self.out_channels, self.kernel_size, self.stride,
                self.nempty, self.use_bias, self.method)


class OctreeDeconv(OctreeConv):
  """Octree deconvolution (ocnn/nn/octree_conv.py:433-466); weights are
  (kdim, out_channels, in_channels)."""

  def is_conv_layer(self): return False

  def forward(self, data: torch.Tensor, octree, depth: int):
    depad = self.stride == 2 and not self.nempty
    if self.method != 'explicit_gemm':
      # the depad: inside the function, which reads the rows of the non-empty nodes through an index
      return octree_deconv(data, self.weights, octree, depth, self.in_channels, self.out_channels,
                           self.kernel_size, self.stride, self.nempty, self.max_buffer,
                           self.bias if self.use_bias else None, depad)
    if depad:
      data = octree_depad(data, octree, depth)
    if self.method == 'explicit_gemm':
      # one product for all slots, then the adjoint of im2col (ocnn/nn/octree_conv.py:453-457)
      col = torch.mm(data, self.weights.to(data.dtype).flatten(0, 1).t())
      out = col2octree(col.view(col.shape[0], self.kdim, -1), tables_of(octree), depth + (self.stride == 2), self.kernel,
                       self.stride, self.nempty)
    else:
      out = octree_deconv(data, self.weights, octree, depth, self.in_channels, self.out_channels,
                          self.kernel_size, self.stride, self.nempty, self.max_buffer,
                          self.bias if self.use_bias else None)
    if self.use_bias and self.method == 'explicit_gemm':
      out = out + self.bias.to(out.dtype)
    return out

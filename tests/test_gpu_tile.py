"""The gather-GEMM of csrc/conv_tile.hip at the edges of its ranges: rows around a tile, every
division of the waves, halves of a 64-channel chunk, and the reduction in one and several parts."""

import copy

import numpy as np
import pytest
import torch

from ocnn_amd import _lib
from ocnn_amd.octree.octree import TilePlan
from oracle import conv_ref as C

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 2e-5, torch.float16: 2e-3, torch.bfloat16: 1e-2}


def _gather(x, plan, w, cout, transposed, reverse, b, parts, occupancy):
  L, P, K = _lib.lib(), _lib.ptr, plan.K
  code, cin = _lib.dtype_code(x), x.shape[1]
  assert L.ocnnx_gather_tile_supported(code, x.shape[0], K, cin, cout, plan.umax)
  out = torch.full((plan.rows, cout), float('nan'), dtype=x.dtype, device='cuda')
  size = L.ocnnx_gather_tile_workspace_bytes(code, plan.rows, K, cin, cout)
  if parts != (0, 0):
    size = 8 * K * cin * cout + 1024 + parts[0] * parts[1] * plan.rows * cout * 4
  ws = torch.empty(size, dtype=torch.uint8, device='cuda')
  _lib.check(L.ocnnx_gather_tile(code, P(x), x.shape[0], P(plan.loc), P(plan.uptr), P(plan.urows), plan.umax, plan.total,
                                 occupancy, plan.rows, K, P(w), cin, cout, int(transposed), int(reverse), P(b), None, P(out),
                                 P(ws), size, *parts, _lib.stream()))
  return out


def _ordered_pass(dtype, plan, rows_in, cin, cout, transposed, reverse):
  """A layer's pass on the tile kernel with the plan's row order, whichever kernel the layers of its shape take."""
  from ocnn_amd.nn.octree_conv import _plan_arrays
  code = _lib.DTYPE_CODE[dtype]
  op = _lib.native().GatherOp(rows_in, plan.rows, plan.K, cin, cout, transposed, reverse)
  assert _lib.lib().ocnnx_gather_tile_supported(code, rows_in, plan.K, cin, cout, plan.umax)
  op.kernel, op.ordered, op.plan = _lib.GATHER_TILE, True, _plan_arrays(plan, False)
  op.ws_bytes = _lib.lib().ocnnx_gather_tile_workspace_bytes(code, plan.rows, plan.K, cin, cout)
  return op


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize('cin,cout', [(32, 32), (96, 64), (64, 96), (160, 160), (128, 256)])
def test_tile_kernel(dtype, cin, cout):
  for rows, K in ((1, 27), (127, 9), (129, 27), (2000, 8)):
    print('tile kernel', dtype, cin, cout, 'rows', rows, 'K', K, flush=True)
    g = torch.Generator().manual_seed(rows + cin)
    t = (torch.arange(rows)[:, None] + torch.randint(-40, 41, (rows, K), generator=g)).clamp_(0, rows - 1).int()
    t[torch.rand(rows, K, generator=g) < 0.4] = -1
    plan = TilePlan(t.cuda())
    x = torch.randn(rows, cin, generator=g).to(dtype)
    w = (torch.randn(K, cin, cout, generator=g) / (K * cin) ** 0.5).to(dtype)
    b = torch.randn(cout, generator=g).to(dtype)
    t64, f64 = t.numpy().astype(np.int64), lambda v: v.double().numpy()
    want = C.forward_gemm(f64(x), f64(w), t64) + f64(b)
    wt = w.flip(0).transpose(1, 2).contiguous()          # read transposed and mirrored: the same layer
    for parts in ((0, 0), (1, 1), (2, 1), (3, 4), (64, 27)):
      for occupancy in (1.0, 0.3):                       # without and with the test for empty blocks
        for ww, tr, rev in ((w, False, False), (wt, True, True)):
          got = _gather(x.cuda(), plan, ww.cuda(), cout, tr, rev, b.cuda(), parts, occupancy)
          err = np.abs(got.double().cpu().numpy() - want).max() / np.abs(want).max()
          assert err < TOL[dtype], (parts, occupancy, tr, err)
          again = _gather(x.cuda(), plan, ww.cuda(), cout, tr, rev, b.cuda(), parts, occupancy)
          assert torch.equal(got, again)


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize('cin,cout,rows,K,spread', [
    (64, 256, 257 * 128 + 5, 9, 40),                     # tiles enough for 256 channels a workgroup
    (96, 64, 300, 3, 2),                                 # fewer slots than waves that share them, few distinct rows
    (64, 32, 300, 2, 0), (32, 96, 300, 1, 0), (64, 128, 300, 1, 3),
    (32, 192, 1300, 27, 130)])                           # as many distinct rows as are staged
def test_tile_kernel_wave_shapes(dtype, cin, cout, rows, K, spread):
  """Every division of the waves over channels, rows and slots, against 64-bit sums over the table."""
  print('tile kernel, waves', dtype, cin, cout, 'rows', rows, 'K', K, flush=True)
  g = torch.Generator().manual_seed(rows + cout)
  t = (torch.arange(rows)[:, None] + torch.randint(-spread, spread + 1, (rows, K), generator=g)).clamp_(0, rows - 1).int()
  t[torch.rand(rows, K, generator=g) < 0.5] = -1
  plan = TilePlan(t.cuda())
  x = torch.randn(rows, cin, generator=g).to(dtype).cuda()
  w = (torch.randn(K, cin, cout, generator=g) / (K * cin) ** 0.5).to(dtype).cuda()
  b = torch.randn(cout, generator=g).to(dtype).cuda()
  zero = torch.cat([x.double(), torch.zeros(1, cin, dtype=torch.float64, device='cuda')])
  want = b.double() + sum(zero[t[:, k].long().cuda()] @ w[k].double() for k in range(K))
  for parts in ((0, 0), (1, 1)):
    for occupancy in (1.0, 0.3):
      got = _gather(x, plan, w, cout, False, False, b, parts, occupancy).double()
      assert (got - want).abs().max() / want.abs().max() < TOL[dtype], (parts, occupancy)


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize('cin,rows,K,spread,occupancy', [
    (96, 1152 * 128 + 5, 27, 110, 0.3),                  # the first tile, and the most rows, with three workgroups a CU
    (96, 1152 * 128, 27, 110, 0.3), (32, 1152 * 128 + 5, 27, 120, 0.3),      # a tile less; more rows
    (64, 1153 * 128, 3, 4, 0.45), (128, 1200 * 128 + 1, 1, 0, 0.1),          # slots: an odd number, fewer than waves
    (32, 640 * 128 + 5, 27, 130, 1.0), (32, 640 * 128, 9, 20, 1.0),          # one chunk, nothing left out
    (64, 641 * 128, 2, 3, 0.6)])
def test_tile_kernel_waves_of_64_channels(dtype, cin, rows, K, spread, occupancy):
  """64 output channels on both sides of the lines between their two divisions of the waves, against 64-bit sums; with the
  rows in the plan's order, as the layers run where empty blocks are left out, to the bit as without."""
  print('tile kernel, 64 channels', dtype, cin, 'rows', rows, 'K', K, flush=True)
  g = torch.Generator().manual_seed(rows + cin)
  t = (torch.arange(rows)[:, None] + torch.randint(-spread, spread + 1, (rows, K), generator=g)).clamp_(0, rows - 1).int()
  t[torch.rand(rows, K, generator=g) < 0.6] = -1
  t[(torch.rand(rows // 32 + 1, K, generator=g) < 0.3).repeat_interleave(32, 0)[:rows]] = -1
  plan = TilePlan(t.cuda())
  x = torch.randn(rows, cin, generator=g).to(dtype).cuda()
  w = (torch.randn(K, cin, 64, generator=g) / (K * cin) ** 0.5).to(dtype).cuda()
  b = torch.randn(64, generator=g).to(dtype).cuda()
  zero = torch.cat([x.double(), torch.zeros(1, cin, dtype=torch.float64, device='cuda')])
  want = b.double() + sum(zero[t[:, k].long().cuda()] @ w[k].double() for k in range(K))
  got = _gather(x, plan, w, 64, False, False, b, (0, 0), occupancy)
  assert (got.double() - want).abs().max() / want.abs().max() < TOL[dtype]
  assert torch.equal(got, _gather(x, plan, w, 64, False, False, b, (0, 0), occupancy))
  if _lib.lib().ocnnx_gather_tile_ordered(K, occupancy):
    assert _lib.lib().ocnnx_gather_tile_ordered(K, plan.occupancy)
    assert torch.equal(got, _ordered_pass(dtype, plan, rows, cin, 64, False, False).run(x, None, w, b))


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16])
def test_tile_kernel_weights_off_alignment(dtype):
  """Weights that start one element past a 16-byte boundary give the bits of aligned ones."""
  g = torch.Generator().manual_seed(5)
  rows, K, cin, cout = 300, 27, 96, 64
  t = torch.randint(-1, rows, (rows, K), generator=g).int()
  t[torch.rand(rows, K, generator=g) < 0.9] = -1
  plan = TilePlan(t.cuda())
  x = torch.randn(rows, cin, generator=g).to(dtype).cuda()
  b = torch.zeros(cout, dtype=dtype).cuda()
  for shape, tr in (((K, cin, cout), False), ((K, cout, cin), True)):
    w = torch.randn(shape, generator=g).to(dtype).cuda()
    off = torch.empty(w.numel() + 1, dtype=dtype, device='cuda')[1:].view(shape)
    off.copy_(w)
    assert w.data_ptr() % 16 == 0 and off.data_ptr() % 16 != 0
    assert torch.equal(_gather(x, plan, w, cout, tr, tr, b, (0, 0), 1.0), _gather(x, plan, off, cout, tr, tr, b, (0, 0), 1.0))


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize('ca,cb', [(32, 32), (64, 64), (96, 160), (192, 192), (256, 256), (512, 320)])
def test_planned_weight_gradient_ranges(dtype, ca, cb):
  """The planned weight gradient at the edges of its division into ranges: one tile, fewer tiles than XCDs,
  ranges that do not divide the tiles, more workgroups a range than CUs."""
  L, P = _lib.lib(), _lib.ptr
  code = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}[dtype]
  for rows, K in ((1, 27), (128, 9), (129, 3), (3 * 128, 27), (11 * 128 + 5, 27), (37 * 128 + 127, 8)):
    print('planned weight gradient', dtype, ca, cb, 'rows', rows, 'K', K, flush=True)
    g = torch.Generator().manual_seed(rows + ca)
    t = (torch.arange(rows)[:, None] + torch.randint(-40, 41, (rows, K), generator=g)).clamp_(0, rows - 1).int()
    t[torch.rand(rows, K, generator=g) < 0.4] = -1
    plan = TilePlan(t.cuda())
    x, grad = torch.randn(rows, ca, generator=g).to(dtype), torch.randn(rows, cb, generator=g).to(dtype)
    assert _lib.dtype_code(x) == code and L.ocnn_conv_wgrad_planned_supported(code, rows, rows, K, ca, cb, plan.umax)
    zero = torch.cat([x.double(), torch.zeros(1, ca, dtype=torch.float64)])
    want = torch.stack([zero[t[:, k].long()].T @ grad.double() for k in range(K)])
    size = L.ocnn_conv_wgrad_planned_workspace_bytes_for(code, rows, rows, K, ca, cb)
    ws = torch.empty(size, dtype=torch.uint8, device='cuda')
    xd, gd = x.cuda(), grad.cuda()
    for transposed in (0, 1):
      gw = torch.full((K, cb, ca) if transposed else (K, ca, cb), float('nan'), dtype=dtype, device='cuda')
      _lib.check(L.ocnn_conv_wgrad_planned(code, P(xd), rows, P(gd), P(plan.loc), P(plan.uptr), P(plan.urows), plan.umax,
                                           plan.total, rows, K, ca, cb, transposed, P(gw), P(ws), size, _lib.stream()))
      got = gw.double().cpu()
      if transposed:
        got = got.transpose(1, 2)
      assert (got - want).abs().max() / want.abs().max() < TOL[dtype], (rows, K, transposed)


def _row_order(plan):
  """order() by its definition: in a tile, rows by the set of their slots, the tile's rarest slot first; then of each slot
  which blocks of 32 rows have an entry."""
  loc = plan.loc.cpu().numpy().view(np.uint16)
  out = np.zeros((loc.shape[0], 160), np.uint8)
  for i, tile in enumerate(loc):
    there = tile != 0
    frequent = np.argsort(-there.sum(1), kind='stable')          # (slots as frequent: the lower one first)
    key = np.zeros(128, np.int64)
    for b, k in enumerate(frequent):
      if b >= 2:                                                 # (the two most frequent ones decide nothing)
        key |= there[k].astype(np.int64) << b
    out[i, :128] = np.lexsort((np.arange(128), key))
    blocks = there[:, out[i, :128]].reshape(len(tile), 4, 32).any(2)
    out[i, 128:128 + len(tile)] = (blocks << np.arange(4)).sum(1)
  return out


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize('cin,cout,K', [(96, 96, 27), (32, 64, 27), (160, 128, 9), (64, 256, 27), (128, 128, 3), (32, 32, 27)])
def test_tile_kernel_row_order(dtype, cin, cout, K):
  """The order of a tile's rows, and the pass that takes them in it: one row, a remainder, whole tiles, tiles enough
  for 256 channels a workgroup, rows without an entry, mirrored slots; to the bit as in the table's order."""
  for rows in (1, 129, 2048, 257 * 128 + 5):
    print('tile kernel, order', dtype, cin, cout, 'rows', rows, 'K', K, flush=True)
    g = torch.Generator().manual_seed(rows + cin)
    t = (torch.arange(rows)[:, None] + torch.randint(-30, 31, (rows, K), generator=g)).clamp_(0, rows - 1).int()
    t[torch.rand(rows, K, generator=g) < torch.rand(1, K, generator=g) * 0.4 + 0.6] = -1
    t[torch.rand(rows, generator=g) < 0.1] = -1
    plan = TilePlan(t.cuda())
    assert _lib.lib().ocnnx_gather_tile_ordered(K, plan.occupancy)
    assert np.array_equal(plan.order().cpu().numpy(), _row_order(plan))
    x = torch.randn(rows, cin, generator=g).to(dtype).cuda()
    b = torch.randn(cout, generator=g).to(dtype).cuda()
    zero = torch.cat([x.double(), torch.zeros(1, cin, dtype=torch.float64, device='cuda')])
    for reverse in (False, True):
      w = (torch.randn((K, cout, cin) if reverse else (K, cin, cout), generator=g) / (K * cin) ** 0.5).to(dtype).cuda()
      op = _ordered_pass(dtype, plan, rows, cin, cout, reverse, reverse)
      got = op.run(x, t.cuda(), w, b).double()
      assert torch.equal(got, _gather(x, plan, w, cout, reverse, reverse, b, (0, 0), plan.occupancy).double())
      at = lambda k: w[K - 1 - k].T.double() if reverse else w[k].double()
      want = b.double() + sum(zero[t[:, k].long().cuda()] @ at(k) for k in range(K))
      assert (got - want).abs().max() / want.abs().max() < TOL[dtype], reverse
      assert torch.equal(got, op.run(x, t.cuda(), w, b).double())


def test_orders_of_several_plans():
  """Orders made together are those made alone, with plans without rows and more plans than a launch describes."""
  g = torch.Generator().manual_seed(4)
  plans = []
  for i in range(27):
    rows, K = (0, 1, 130, 1000)[i % 4], (27, 9, 3)[i % 3]
    t = torch.randint(-20, max(rows, 1), (rows, K), generator=g).clamp_(min=-1).int()
    plans.append(TilePlan(t.cuda()))
  alone = [p.order().clone() for p in plans]
  TilePlan.order_many(plans)
  for p, a in zip(plans, alone):
    assert torch.equal(p.order(), a) and np.array_equal(a.cpu().numpy(), _row_order(p))
  others = copy.deepcopy(plans)                            # (copies make theirs again)
  assert all(p._order is None for p in others)
  TilePlan.order_many(others)
  for p, a in zip(others, alone):
    assert torch.equal(p._order, a)


def test_fresh_octree_orders_the_plans_of_its_predecessors():
  """A layer on the tile kernel asks for its plan's order; the next octree of the kind makes it with the plan."""
  from ocnn_amd import synthetic
  from ocnn_amd.nn import OctreeConv
  from ocnn_amd.octree import Octree, Points
  from ocnn_amd.octree.octree import PlanHistory
  history = PlanHistory()
  layer = OctreeConv(96, 96, [3], 1, nempty=True).cuda().half()
  for turn in range(2):
    pts, nrm = synthetic.mixed_cloud(20000, seed=3 + turn)
    octree = Octree(6, 2)
    octree.plan_history = history
    octree.build_octree(Points(pts.cuda(), nrm.cuda()))
    octree.construct_all_neigh()
    octree.prepare()
    key = ((6, '333', 1, True), False)
    assert (key in octree._plans and octree._plans[key]._order is not None) == (turn == 1)
    layer(torch.randn(int(octree.nnum_nempty[6]), 96, device='cuda').half(), octree, 6)
    assert octree._plans[key]._order is not None and history.wished((6, 2), 'order') == {key}
  history.clear()
  assert history.wished((6, 2), 'order') == frozenset()


def test_fresh_octree_finds_the_sibling_groups_its_predecessors_were_asked_for():
  """Whether a table is one of sibling groups: asked of the plan alone, and with the next octree's plan."""
  from ocnn_amd import synthetic
  from ocnn_amd.octree import Octree, Points
  from ocnn_amd.octree.octree import PlanHistory
  history = PlanHistory()
  for turn in range(2):
    pts, nrm = synthetic.mixed_cloud(20000, seed=5 + turn)
    octree = Octree(6, 2)
    octree.plan_history = history
    octree.build_octree(Points(pts.cuda(), nrm.cuda()))
    octree.construct_all_neigh()
    octree.prepare()
    for nempty in (False, True):
      plan = octree._plan(6, '333', 1, nempty)
      assert plan._siblings == (None if turn == 0 else not nempty)
      assert plan.siblings == (not nempty) and TilePlan(octree._table(6, '333', 1, nempty)).siblings == (not nempty)
  broken = octree._table(6, '333', 1, False).clone()
  broken[-1, 13] = -1                                      # one entry of the last group
  assert not TilePlan(broken).siblings and not TilePlan.build_many([broken], groups=[True])[0].siblings
  assert not TilePlan(torch.empty((0, 27), dtype=torch.int32, device='cuda')).siblings


@pytest.mark.parametrize('rows,K,entries', [(500, 8, 512), (500, 8, 700), (300, 8, 100000), (1000, 27, 1000)])
def test_lists_that_no_kernel_reads_are_made_when_read(rows, K, entries):
  """Tiles of more rows than any kernel stages, each used about once: lists and positions are those of the two passes."""
  g = torch.Generator().manual_seed(rows + entries)
  t = torch.stack([torch.randperm(max(entries, K), generator=g)[:K] for _ in range(rows)]).int().cuda()
  plan, other, two = TilePlan(t), TilePlan(t), TilePlan(t, cap=4000)
  assert two.umax == plan.umax
  left = plan.umax > TilePlan.MOST_STAGED and plan.reuse < TilePlan.MULTI_PASS_REUSE
  assert ('loc' not in vars(plan)) == left == (K == 8 and entries > 512)
  other = copy.deepcopy(other)
  for p in (plan, other):
    assert torch.equal(p.loc, two.loc) and torch.equal(p.urows[:p.total], two.urows[:two.total]) and torch.equal(p.uptr, two.uptr)
  with pytest.raises(AttributeError):
    plan.nothing


def test_lists_first_read_under_capture():
  """A capture records the lists and positions it reads and keeps none of them, which hold nothing before the first replay;
  a plan that has made them lets go of its table."""
  g = torch.Generator().manual_seed(8)
  t = torch.stack([torch.randperm(100000, generator=g)[:8] for _ in range(300)]).int().cuda()
  plan, want = TilePlan(t), TilePlan(t, cap=4000)
  assert 'loc' not in vars(plan)
  graph = torch.cuda.CUDAGraph()
  torch.cuda.synchronize()
  with torch.cuda.graph(graph):
    recorded = plan.loc.clone(), plan.urows.clone()
  assert 'loc' not in vars(plan) and 'urows' not in vars(plan)
  assert torch.equal(plan.loc, want.loc) and torch.equal(plan.urows[:plan.total], want.urows[:want.total])
  assert 'loc' in vars(plan) and '_unfilled' not in vars(plan)
  for _ in range(3):
    for r in recorded:
      r.zero_()
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(recorded[0], want.loc) and torch.equal(recorded[1][:want.total], want.urows[:want.total])


def test_layer_first_called_under_capture():
  """A layer whose pass is made while a graph is captured, on a plan that is there already: no order comes out of the capture,
  the first call after it makes one, and all give the same rows to the bit."""
  from ocnn_amd import synthetic
  from ocnn_amd.nn import OctreeConv
  from ocnn_amd.octree import Octree, Points
  from ocnn_amd.octree.octree import PlanHistory
  pts, nrm = synthetic.mixed_cloud(20000, seed=9)
  octree = Octree(6, 2)
  octree.plan_history = PlanHistory()
  octree.build_octree(Points(pts.cuda(), nrm.cuda()))
  octree.construct_all_neigh()
  plan = octree._plan(6, '333', 1, True)
  layer = OctreeConv(96, 96, [3], 1, nempty=True).cuda().half()
  x = torch.randn(int(octree.nnum_nempty[6]), 96, device='cuda').half()
  graph = torch.cuda.CUDAGraph()
  torch.cuda.synchronize()
  with torch.no_grad():
    with torch.cuda.graph(graph):
      recorded = layer(x, octree, 6)
    assert plan._order is None and octree.plan_history.wished((6, 2), 'order')
    eager = layer(x, octree, 6)
    assert np.array_equal(plan._order.cpu().numpy(), _row_order(plan))
    for turn in range(3):
      recorded.zero_()
      graph.replay()
      torch.cuda.synchronize()
      assert torch.equal(recorded, eager) and torch.equal(layer(x, octree, 6), eager), turn
    graph = torch.cuda.CUDAGraph()                         # with an order that another stream has made
    with torch.cuda.graph(graph):
      recorded = layer(x, octree, 6)
    for turn in range(3):
      recorded.zero_()
      graph.replay()
      torch.cuda.synchronize()
      assert torch.equal(recorded, eager) and torch.equal(layer(x, octree, 6), eager), turn


@pytest.mark.parametrize('together', [False, True])
def test_order_made_on_another_stream(together):
  """A pass waits for an order that is still on its way on the stream it is made on, whoever asked for it."""
  from ocnn_amd.nn.octree_conv import _gather_op
  g = torch.Generator().manual_seed(11)
  rows, K = 6000, 27
  t = (torch.arange(rows)[:, None] + torch.randint(-30, 31, (rows, K), generator=g)).clamp_(0, rows - 1).int()
  t[torch.rand(rows, K, generator=g) < 0.8] = -1
  t = t.cuda()
  x, w = torch.randn(rows, 96, generator=g).cuda(), (torch.randn(K, 96, 96, generator=g) / 50).cuda()
  plan, alone = TilePlan(t), TilePlan(t)
  want = _gather_op(torch.float32, rows, rows, K, 96, 96, False, False, alone).run(x, t, w, None)
  busy, side = torch.randn(4096, 4096, device='cuda'), torch.cuda.Stream()
  side.wait_stream(torch.cuda.current_stream())
  torch.cuda.synchronize()
  with torch.cuda.stream(side):
    for _ in range(60):
      product = busy @ busy
    if together:
      TilePlan.order_many([plan])
    else:
      plan.order()
  op = _gather_op(torch.float32, rows, rows, K, 96, 96, False, False, plan)
  assert op.ordered and op.kernel == _lib.GATHER_TILE
  got = op.run(x, t, w, None)
  assert not side.query(), 'the other stream was not busy'
  torch.cuda.synchronize()
  assert torch.equal(got, want) and torch.equal(op.run(x, t, w, None), want)
  assert torch.equal(plan.order(), alone.order())
  del product

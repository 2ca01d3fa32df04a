"""Octree builds at the edges of the sort's ranges: points around a span, one to three digits, counts read
in place or scanned, keys of more than 32 bits; and the tables of octrees whose layers are found by
walking and from their parents."""

import numpy as np
import pytest
import torch

from ocnn_amd.octree import Octree, Points
from oracle import octree_ref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,depth,full_depth,batch', [(1, 3, 1, 1), (2047, 3, 2, 1), (2049, 6, 2, 3), (32768, 7, 2, 1),
                                                      (32769, 6, 3, 5), (131072, 9, 2, 8), (131073, 8, 2, 1), (5000, 11, 2, 2),
                                                      (300001, 8, 2, 4)])
def test_build_and_tables(n, depth, full_depth, batch):
  print('octree', n, depth, full_depth, batch, flush=True)
  g = torch.Generator().manual_seed(n)
  pts = torch.rand(n, 3, generator=g) * 1.98 - 0.99
  pts[:, 2] = 0.3 * pts[:, 0] * pts[:, 1]                 # a surface
  nrm = torch.randn(n, 3, generator=g)
  bid = torch.randint(0, batch, (n, 1), generator=g).float()
  bid[0], bid[-1] = 0, batch - 1
  o = Octree(depth, full_depth, batch_size=batch)
  idx = o.build_octree(Points(pts.cuda(), nrm.cuda(), batch_id=bid.cuda() if batch > 1 else None, batch_size=batch))
  o.construct_all_neigh()
  ref, want_idx = R.build_octree(pts.numpy(), nrm.numpy(), batch_id=bid.numpy() if batch > 1 else None, depth=depth,
                                 full_depth=full_depth, batch_size=batch)
  assert np.array_equal(idx.cpu().numpy(), want_idx)
  for d in range(depth + 1):
    assert np.array_equal(o.keys[d].cpu().numpy(), ref.keys[d]), d
    assert np.array_equal(o.children[d].cpu().numpy(), ref.children[d]), d
    assert int(o.nnum[d]) == ref.keys[d].shape[0]
    if d >= full_depth:
      assert np.array_equal(o._nempty_index32(d).cpu().numpy(), np.nonzero(ref.children[d] >= 0)[0]), d
  assert np.abs(o.points[depth].cpu().numpy() - ref.points[depth]).max() < 1e-4 * 2 ** depth
  again = Octree(depth, full_depth, batch_size=batch)
  again.build_octree(Points(pts.cuda(), nrm.cuda(), batch_id=bid.cuda() if batch > 1 else None, batch_size=batch))
  assert torch.equal(again.points[depth], o.points[depth]) and torch.equal(again.normals[depth], o.normals[depth])
  layer = Octree(depth, full_depth, batch_size=batch)       # the tables layer by layer, from the parents' alone
  layer.build_octree(Points(pts.cuda(), nrm.cuda(), batch_id=bid.cuda() if batch > 1 else None, batch_size=batch))
  for d in range(1, depth + 1):
    layer.construct_neigh(d)
    assert torch.equal(layer.neighs.get32(d), o.neighs.get32(d)), d


@pytest.mark.parametrize('n,depth,batch,same', [(1, 2, 1, False), (255, 2, 1, False), (257, 1, 1, True), (1025, 3, 2, False),
                                                (20011, 4, 1, False), (65536, 3, 1, False), (65537, 3, 1, False), (70000, 2, 1, True),
                                                (9000, 11, 2, False)])
@pytest.mark.parametrize('normals', [True, False])
def test_leaf_averages_across_spans(n, depth, batch, same, normals):
  """Leaves of many points, within a span of the scatter and over several (same: all points in one cell), on both sizes of
  spans and on the library's sort, with and without normals: sums in the order of the points, to the bit of the oracle's."""
  print('leaves', n, depth, batch, same, normals, flush=True)
  g = torch.Generator().manual_seed(n)
  pts = torch.rand(n, 3, generator=g) * (0.01 if same else 1.98) + (0.5 if same else -0.99)
  nrm = torch.randn(n, 3, generator=g) if normals else None
  bid = torch.randint(0, batch, (n, 1), generator=g).float()
  bid[0], bid[-1] = 0, batch - 1
  o = Octree(depth, 1, batch_size=batch)
  idx = o.build_octree(Points(pts.cuda(), None if nrm is None else nrm.cuda(), batch_id=bid.cuda() if batch > 1 else None,
                              batch_size=batch)).cpu().numpy()
  p = ((pts.numpy() - np.float32(-1)) * np.float32(2 ** depth / 2)).astype(np.float32)
  leaves = idx.max() + 1
  sums, count = np.zeros((leaves, 6), np.float32), np.bincount(idx, minlength=leaves).astype(np.float32)
  rows = np.concatenate([p, np.zeros_like(p) if nrm is None else nrm.numpy()], 1)
  for i, leaf in enumerate(idx):
    sums[leaf] += rows[i]
  assert np.array_equal(o.points[depth].cpu().numpy(), sums[:, :3] / count[:, None])
  if normals:
    length = np.maximum(np.sqrt((sums[:, 3:] ** 2).sum(1, keepdims=True)), 1e-12)
    assert np.abs(o.normals[depth].cpu().numpy() - sums[:, 3:] / length).max() < 1e-6
  else:
    assert o.normals[depth] is None


@pytest.mark.parametrize('n', [9001, 262144, 262145])
@pytest.mark.parametrize('long', [255, 256, 257, 511, 512, 513, 1023, 1025, 4096])
def test_leaf_that_leaves_its_span(n, long):
  """One leaf of `long` points among leaves of few, wherever it lies in the spans of 256 and 1024 points: its signals are the
  sums in the order of the points, to the bit, and its neighbours' are untouched."""
  print('long leaf', n, long, flush=True)
  g = torch.Generator().manual_seed(n + long)
  pts = torch.rand(n, 3, generator=g) * 1.98 - 0.99
  at = torch.randperm(n, generator=g)[:long]
  for corner in (-0.9, -0.17, 0.55):                       # (cells at the start, in the middle and towards the end of the order)
    cloud = pts.clone()
    cloud[at] = corner + torch.rand(long, 3, generator=g) * 1e-3
    nrm = torch.randn(n, 3, generator=g)
    o = Octree(5, 2)
    idx = o.build_octree(Points(cloud.cuda(), nrm.cuda())).cpu().numpy()
    p = ((cloud.numpy() - np.float32(-1)) * np.float32(16)).astype(np.float32)
    sums, count = np.zeros((idx.max() + 1, 6), np.float32), np.bincount(idx).astype(np.float32)
    np.add.at(sums, idx, np.concatenate([p, nrm.numpy()], 1))
    assert count.max() >= long
    assert np.array_equal(o.points[5].cpu().numpy(), sums[:, :3] / count[:, None])
    length = np.maximum(np.sqrt((sums[:, 3:] ** 2).sum(1, keepdims=True)), 1e-12)
    assert np.abs(o.normals[5].cpu().numpy() - sums[:, 3:] / length).max() < 1e-6


def test_normals_and_batch_ids_of_another_device_are_refused():
  """Host memory is not handed to the build's kernels."""
  g = torch.Generator().manual_seed(2)
  pts = (torch.rand(500, 3, generator=g) - 0.5).cuda()
  mixed = Points(pts)
  mixed.normals = torch.randn(500, 3, generator=g)
  with pytest.raises(RuntimeError, match='one device'):
    Octree(4, 2).build_octree(mixed)
  ids = (torch.arange(500) % 2).float().view(-1, 1)
  mixed = Points(pts, batch_id=ids.cuda(), batch_size=2)
  mixed.batch_id = ids
  with pytest.raises(RuntimeError, match='one device'):
    Octree(4, 2, batch_size=2).build_octree(mixed)
  mixed = Points(pts)
  mixed.normals = torch.randn(499, 3, generator=g).cuda()
  with pytest.raises(RuntimeError, match='every point'):
    Octree(4, 2).build_octree(mixed)


def test_cloud_in_one_leaf_takes_no_time_a_point():
  """200 000 points of one cell: their sums are one chain of additions, 4.7 ms, but not one of fetches (30 to 51 ms with a
  point fetched at a time; the bound is half of the former)."""
  import time
  g = torch.Generator().manual_seed(1)
  cloud = Points((0.3 + torch.rand(200000, 3, generator=g) * 1e-3).cuda(), torch.randn(200000, 3, generator=g).cuda())
  took = []
  for _ in range(5):
    torch.cuda.synchronize()
    start = time.perf_counter()
    o = Octree(5, 2)
    o.build_octree(cloud)
    torch.cuda.synchronize()
    took.append(time.perf_counter() - start)
  assert int(o.nnum_nempty[5]) == 1 and min(took) < 15e-3, took


@pytest.mark.parametrize('leaves', [0, 1, 255, 257, 70001])
def test_input_feature_kernel(leaves):
  """Every set of letters from one launch against the torch operations one by one (taken for signals that need a gradient);
  the product sums three rounded products, whose order torch chooses: two roundings of a sum of at most 1.5."""
  g = torch.Generator().manual_seed(leaves)
  octree = Octree(5, 2)
  octree.device = torch.device('cuda:0')
  points = (torch.rand(leaves, 3, generator=g) * 34 - 1).cuda()                # (some outside the box: negative fractions)
  normals = torch.nn.functional.normalize(torch.randn(leaves, 3, generator=g)).cuda()
  for bits in range(1, 16):
    letters = ''.join(c for i, c in enumerate('NDLP') if bits >> i & 1)
    octree.points[5], octree.normals[5] = points, normals
    got = octree.get_input_feature(letters, True)
    octree.points[5], octree.normals[5] = points.clone().requires_grad_(), normals.clone().requires_grad_()
    want = octree.get_input_feature(letters, True)
    assert want.requires_grad and got.shape == want.shape and not got.requires_grad
    if leaves:
      assert (got - want).abs().max() <= (4e-7 if 'D' in letters else 0.0), letters

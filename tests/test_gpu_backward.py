"""The backward pass of a layer as one call, with the launches around its kernels merged, against the passes
one by one, which run when only one of the gradients is asked for: the same kernels, so the same bits."""

import pytest
import torch

from ocnn_amd import synthetic
from ocnn_amd.nn import OctreeConv, OctreeDeconv
from ocnn_amd.octree import Octree, Points
from ocnn_amd.octree.octree import TilePlan

pytestmark = pytest.mark.gpu


def _octree(n, depth):
  points, normals = synthetic.sphere_cloud(n)
  octree = Octree(depth, 2, device='cuda')
  octree.build_octree(Points(points, normals).cuda())
  octree.construct_all_neigh()
  return octree


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize('make,cin,cout,depth,nempty,bias', [
    (OctreeConv, 96, 64, 5, True, True), (OctreeConv, 256, 256, 4, True, False), (OctreeConv, 32, 32, 5, False, True),
    (OctreeConv, 64, 160, 3, True, True), (OctreeDeconv, 96, 128, 5, True, True)])
@pytest.mark.parametrize('cap', [None, 203])             # 203: at depth 5 a tile is beyond the limit and runs apart
def test_merged_backward(dtype, make, cin, cout, depth, nempty, bias, cap, monkeypatch):
  print('merged backward', dtype, make.__name__, cin, cout, depth, nempty, bias, cap, flush=True)
  if cap:
    monkeypatch.setattr(TilePlan, 'CAP', cap)
  octree = _octree(3000, depth)
  torch.manual_seed(depth)
  layer = make(cin, cout, [3], 1, nempty=nempty, use_bias=bias).cuda().to(dtype)
  rows = int(octree.nnum_nempty[depth] if nempty else octree.nnum[depth])
  x = torch.randn(rows, cin, device='cuda').to(dtype).requires_grad_(True)
  out = layer(x, octree, depth)
  grad = torch.randn(out.shape[1], out.shape[0], device='cuda').to(dtype).t()   # (of other strides)
  if cap and nempty and depth == 5:
    assert octree._plan(depth, '333', 1, True, False, rows).overflow_rows.numel() == 128
  wanted = [x] + list(layer.parameters())
  together = torch.autograd.grad(out, wanted, grad, retain_graph=True)
  for t, one in zip(wanted, together):
    alone, = torch.autograd.grad(out, [t], grad, retain_graph=True)
    assert one.shape == t.shape and torch.equal(one, alone)

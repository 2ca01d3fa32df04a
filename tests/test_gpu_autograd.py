"""The layers' native nodes under the parts of torch that look on: torch.jit.trace."""

import pytest
import torch

from ocnn_amd import synthetic
from ocnn_amd.modules import Conv1x1BnRelu, OctreeConvBnRelu, OctreeDeconvBnRelu, OctreeResBlock2
from ocnn_amd.octree import Octree, Points

pytestmark = pytest.mark.gpu
DEPTH = 6
EVAL_TOL = {torch.float32: 1e-5, torch.float16: 4e-3}


def _octree(n=20000, depth=DEPTH):
  points, normals = synthetic.sphere_cloud(n)
  octree = Octree(depth, 2, device='cuda')
  octree.build_octree(Points(points, normals).cuda())
  octree.construct_all_neigh()
  return octree


class _Net(torch.nn.Module):
  """Every native node - convolution and deconvolution (padded and not), 1x1 convolution, batch norm with and
  without a residual - and a layer that is none (3x3x3 stride 2 over all nodes)."""

  def __init__(self, octree):
    super().__init__()
    self.octree = octree
    self.down = OctreeConvBnRelu(32, 64, [2], 2)
    self.block = OctreeResBlock2(64, 64)
    self.side = OctreeConvBnRelu(32, 64, [3], 2)
    self.up = OctreeDeconvBnRelu(64, 32, [2], 2)
    self.conv = OctreeConvBnRelu(32, 32)
    self.point = Conv1x1BnRelu(32, 16)

  def forward(self, x):
    x = self.side(x, self.octree, DEPTH) + self.down(x, self.octree, DEPTH)
    x = self.block(x, self.octree, DEPTH - 1)
    return self.point(self.conv(self.up(x, self.octree, DEPTH - 1), self.octree, DEPTH))


def _data(octree, dtype, seed):
  return torch.randn(int(octree.nnum[DEPTH]), 32, generator=torch.Generator().manual_seed(seed)).to('cuda', dtype)


@pytest.mark.parametrize('training', [False, True])
@pytest.mark.parametrize('dtype', [torch.float32, torch.float16])
def test_traced_network(dtype, training):
  """Other data through the traced network: what the network itself gives, its gradients included.  (Training:
  the same kernels, the same bits.  Evaluation: the batch norms ride on the convolutions only where nothing
  records, six roundings of a layer's result; as in test_gpu_layer_bn.py.)"""
  octree = _octree()
  torch.manual_seed(0)
  net = _Net(octree).to('cuda', dtype).train(training)
  with torch.set_grad_enabled(training):
    traced = torch.jit.trace(net, (_data(octree, dtype, 0),), check_trace=False)
    results = []
    for f in (net, traced):
      net.zero_grad()
      x = _data(octree, dtype, 1).requires_grad_(training)
      y = f(x)
      results.append([y.detach()])
      if training:
        y.backward(_data(octree, dtype, 2)[:, :16])
        results[-1] += [x.grad] + [p.grad.clone() for p in net.parameters()]
  for want, got in zip(*results):
    if training:
      assert torch.equal(got, want)
    else:
      assert (got.double() - want.double()).abs().max() < 6 * EVAL_TOL[dtype] * want.double().abs().max()

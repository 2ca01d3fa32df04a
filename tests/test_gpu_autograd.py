"""The layers' native nodes under the parts of torch that look on: torch.jit.trace, forward-mode differentiation
and the transforms of torch.func."""

import pytest
import torch
import torch.autograd.forward_ad as fwAD

from ocnn_amd import synthetic
from ocnn_amd.modules import BatchNormRelu1d, Conv1x1, Conv1x1BnRelu, OctreeConvBnRelu, OctreeDeconvBnRelu, OctreeResBlock2
from ocnn_amd.nn import OctreeConv, OctreeDeconv
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


def _layers(octree):
  """Each kind of native node alone: (module, further arguments)."""
  torch.manual_seed(0)
  return [(OctreeConv(32, 32, use_bias=True), (octree, DEPTH)), (OctreeDeconv(32, 32), (octree, DEPTH)),
          (Conv1x1(32, 16), ()), (BatchNormRelu1d(32, relu=True), ()), (OctreeConvBnRelu(32, 32), (octree, DEPTH))]


@pytest.mark.parametrize('training', [False, True])
def test_forward_mode_is_refused(training):
  """No derivative of the layers in forward mode: a call on a dual tensor is an error, not a value without a
  tangent; a call without one gives what it gives outside."""
  octree = _octree()
  for module, args in _layers(octree):
    module = module.to('cuda', torch.float16).train(training)
    x, tangent = _data(octree, torch.float16, 0), _data(octree, torch.float16, 1)
    with torch.set_grad_enabled(training):
      want = module(x, *args)
      with fwAD.dual_level():
        dual = fwAD.make_dual(x, tangent)
        with pytest.raises(NotImplementedError):
          module(dual, *args)
        got = module(x, *args)
    assert (got - want).abs().max() <= EVAL_TOL[torch.float16] * want.abs().max()


def test_transforms_are_refused():
  octree = _octree()
  for module, args in _layers(octree):
    module = module.to('cuda', torch.float16)
    x = _data(octree, torch.float16, 0)
    f = lambda t: module(t, *args).float().sum()
    with pytest.raises(RuntimeError, match='autograd.Function'):
      torch.func.grad(f)(x)
    with pytest.raises(RuntimeError, match='autograd.Function'):
      torch.func.vmap(lambda t: module(t, *args))(x[None])


@pytest.mark.parametrize('cin,cout,dtype', [(128, 128, torch.float16), (96, 96, torch.float32), (96, 128, torch.bfloat16),
                                            (4, 96, torch.float16), (64, 64, torch.bfloat16)])
@pytest.mark.parametrize('n', [3000, 90000])
def test_gradients_in_either_order(cin, cout, dtype, n):
  """The passes of a backward pass run in an order that hangs on the gradient's type and size (small and large here) and on
  padded channels: the same bits as each pass by itself."""
  octree = _octree(n, 6)
  layer = OctreeConv(cin, cout, nempty=False).to('cuda', dtype)
  x = torch.randn(int(octree.nnum[6]), cin, generator=torch.Generator().manual_seed(n)).to('cuda', dtype).requires_grad_()
  print('gradients in either order', cin, cout, dtype, n, x.shape[0] * cout, flush=True)
  out = layer(x, octree, 6)
  g = torch.randn(out.shape, generator=torch.Generator().manual_seed(n + 1)).to('cuda', dtype)
  both = torch.autograd.grad(out, (x, layer.weights), g, retain_graph=True)
  alone = [torch.autograd.grad(out, t, g, retain_graph=True)[0] for t in (x, layer.weights)]
  assert all(torch.equal(a, b) for a, b in zip(both, alone))

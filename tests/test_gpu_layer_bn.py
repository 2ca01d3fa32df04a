"""A layer and the batch norm behind it as one call in evaluation, against the two calls that run when
gradients are on: every kernel that may take the layer, with and without bias, residual and ReLU."""

import pytest
import torch

from ocnn_amd import _lib, synthetic
from ocnn_amd.modules import Conv1x1, Conv1x1Bn, OctreeConvBnRelu, OctreeDeconvBnRelu, OctreeResBlock2, OctreeResBlocks
from ocnn_amd.nn import OctreeConv
from ocnn_amd.octree import Octree, Points

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 1e-5, torch.float16: 4e-3, torch.bfloat16: 3e-2}


def _octree(n=3000, depth=5):
  points, normals = synthetic.sphere_cloud(n)
  octree = Octree(depth, 2, device='cuda')
  octree.build_octree(Points(points, normals).cuda())
  octree.construct_all_neigh()
  return octree


def _randomise(module, dtype):
  g = torch.Generator().manual_seed(5)
  for m in module.modules():
    if isinstance(m, torch.nn.BatchNorm1d):
      for t, lo in ((m.running_var, 0.5), (m.weight.data, 0.5), (m.running_mean, -0.5), (m.bias.data, -0.5)):
        t.copy_(torch.rand(t.shape, generator=g) + lo)
  return module.to('cuda', dtype).eval()


def _both(module, *args):
  with torch.no_grad():
    one = module(*args)
  with torch.enable_grad():
    two = module(*args).detach()
  assert one.shape == two.shape and one.dtype == two.dtype
  return (one.double() - two.double()).abs().max().item() / two.double().abs().max().item()


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize('nempty', [False, True])
def test_layer_bn(dtype, nempty):
  octree, depth = _octree(), 5
  for cls, cin, cout, kernel, stride, at in ((OctreeConvBnRelu, 32, 32, [3], 1, depth), (OctreeConvBnRelu, 64, 96, [3], 1, 4),
                                             (OctreeConvBnRelu, 4, 32, [3], 1, depth), (OctreeConvBnRelu, 24, 40, [3], 1, depth),
                                             (OctreeConvBnRelu, 32, 64, [2], 2, depth), (OctreeConvBnRelu, 256, 256, [3], 1, 3),
                                             (OctreeDeconvBnRelu, 64, 32, [2], 2, depth - 1)):
    print(cls.__name__, dtype, nempty, cin, cout, kernel, stride, at, flush=True)
    layer = _randomise(cls(cin, cout, kernel, stride, nempty), dtype)
    rows = int((octree.nnum_nempty if nempty else octree.nnum)[at])
    x = torch.randn(rows, cin, generator=torch.Generator().manual_seed(cin)).to('cuda', dtype)
    assert _both(layer, x, octree, at) < TOL[dtype]


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize('cin,cout', [(32, 32), (64, 32), (96, 128)])
def test_residual_block(dtype, cin, cout):
  octree = _octree(20000, 6)
  rows = int(octree.nnum[6])
  print('block', dtype, cin, cout, rows, flush=True)
  x = torch.randn(rows, cin, generator=torch.Generator().manual_seed(cin)).to('cuda', dtype)
  block = _randomise(OctreeResBlock2(cin, cout), dtype)
  assert _both(block, x, octree, 6) < 2 * TOL[dtype]
  shortcut = _randomise(Conv1x1Bn(cin, cout), dtype)
  assert _both(shortcut, x) < TOL[dtype]
  seen = []                                              # hooks of the parts are still called
  handle = block.conv3x3b.conv.register_forward_hook(lambda *a: seen.append(1))
  with torch.no_grad():
    block(x, octree, 6)
  handle.remove()
  assert seen == [1]
  for part in (block.conv3x3b.conv, block.conv3x3b.bn):  # and so is a forward put on the module itself
    own = part.forward
    part.forward = lambda *a, **k: (seen.append(2), own(*a, **k))[1]
    with torch.no_grad():
      block(x, octree, 6)
    del part.forward
  assert seen == [1, 2, 2]


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize('cin,cout,blocks,bottleneck,nempty', [(32, 32, 1, 1, True), (64, 64, 7, 1, True), (64, 32, 7, 1, True), (32, 64, 2, 2, False),
                                                              (24, 40, 2, 1, True), (256, 256, 6, 1, False)])
def test_chain_of_blocks(dtype, cin, cout, blocks, bottleneck, nempty):
  """Blocks in one call give the bits of their layers one by one (which a hook on a part of each asks for): more layers than
  are packed in one launch, a shortcut of the first, channels that run padded, few rows and many."""
  octree = _octree(30000, 7)
  for depth in (3, 7):
    rows = int((octree.nnum_nempty if nempty else octree.nnum)[depth])
    print('chain', dtype, cin, cout, blocks, bottleneck, nempty, depth, rows, flush=True)
    x = torch.randn(rows, cin, generator=torch.Generator().manual_seed(cin)).to('cuda', dtype)
    chain, seen = _randomise(OctreeResBlocks(cin, cout, blocks, bottleneck, nempty), dtype), []
    if depth == 7 and dtype != torch.float32 and bottleneck == 1 and cout in (32, 64):
      last = chain.resblks[-1].conv3x3b.conv.native_of_stride_1(dtype, (rows, cout), octree, depth)
      assert last.fwd.kernel == _lib.GATHER_RW
    for _ in range(2):
      with torch.no_grad():
        one = chain(x, octree, depth)
        hooks = [block.conv3x3a.register_forward_hook(lambda *a: seen.append(1)) for block in chain.resblks]
        assert torch.equal(chain(x, octree, depth), one)
        for hook in hooks:
          hook.remove()
        for m in chain.resblks:
          m.conv3x3b.conv.weights.mul_(0.5)                  # (the weights are read on each call)
    assert len(seen) == 2 * blocks and _both(chain, x, octree, depth) <= 2 * blocks * TOL[dtype]


@pytest.mark.parametrize('part,names', [('conv', ['weights']), ('conv', ['bias']), ('bn', ['weight', 'bias']),
                                        ('bn', ['running_mean', 'running_var'])])
def test_tensors_held_as_plain_attributes(part, names):
  """Parameters and buffers replaced by plain attributes of the module (as libraries that reparametrise
  modules leave them) are the ones that are used: the same values, and then others."""
  octree = _octree()
  block = _randomise(OctreeConvBnRelu(32, 64, nempty=True), torch.float16)
  if names == ['bias']:
    block.conv = OctreeConv(32, 64, nempty=True, use_bias=True).to('cuda', torch.float16).eval()
    torch.nn.init.uniform_(block.conv.bias)
  x = torch.randn(int(octree.nnum_nempty[5]), 32, generator=torch.Generator().manual_seed(1)).to('cuda', torch.float16)
  module = getattr(block, part)
  with torch.no_grad():
    want = block(x, octree, 5)
    held = [getattr(module, n).detach().clone() for n in names]
    for n, t in zip(names, held):
      delattr(module, n)
      setattr(module, n, t)
    # (one pass or two: six roundings of the result apart, as in the tests above)
    assert (block(x, octree, 5).double() - want.double()).abs().max() <= TOL[torch.float16] * want.double().abs().max()
    held[0].mul_(2)
    assert not torch.equal(block(x, octree, 5), want)


# channels of 1x1 layers with a pass over the one-slot table; whether the forward pass is one (else: dense rows)
LINEAR = [(32, 32, False), (192, 96, True), (288, 48, True)]


@pytest.mark.parametrize('cin,cout,forward', LINEAR)
def test_linear_layers_keep_one_table(cin, cout, forward):
  """A 1x1 layer whose row count differs with every call (a new octree every step): what is kept for it on
  the GPU does not grow with the calls."""
  layer = Conv1x1(cin, cout).to('cuda', torch.float16)
  g = torch.Generator(device='cuda').manual_seed(3)

  def step(rows):
    x = torch.randn(rows, cin, device='cuda', generator=g).half().requires_grad_()
    native = layer.native_layer(x)
    assert native.fwd_table.shape[0] == rows and (native.fwd.kernel == _lib.GATHER_PLAIN) == forward
    layer.zero_grad()
    layer(x).backward(torch.ones(rows, cout, device='cuda', dtype=torch.float16))
    want = x.detach().double() @ layer.linear.weight.detach().double().t()
    assert (layer(x).double() - want).abs().max() < TOL[torch.float16] * want.abs().max()

  step(200000)
  torch.cuda.synchronize()
  held = torch.cuda.memory_allocated()
  for i in range(30):
    step(100000 + 3001 * i)
  torch.cuda.synchronize()
  assert torch.cuda.memory_allocated() <= held + 4096


@pytest.mark.parametrize('cin,cout,forward', LINEAR)
def test_linear_layer_in_a_graph(cin, cout, forward):
  """Replays of a captured 1x1 layer while larger ones run beside them: the table that the graph reads is its own."""
  layer = Conv1x1(cin, cout).to('cuda', torch.float16).requires_grad_(False)
  x = torch.randn(5000, cin, device='cuda').half()
  with torch.no_grad():
    assert (layer.native_layer(x).fwd_table is not None) == forward
  want = layer(x).clone()
  graph = torch.cuda.CUDAGraph()
  with torch.cuda.graph(graph):
    out = layer(x)
  for rows in (9000, 70000, 600000):
    out.zero_()
    layer(torch.randn(rows, cin, device='cuda').half())
    torch.full((rows,), -1, dtype=torch.int32, device='cuda')      # (over memory that was given back)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, want)

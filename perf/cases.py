"""The work that programs built on this package have it do, as cases that can be timed: layers on a
resident octree (one layer called many times, as the blocks of a network and the layer benchmarks
do), the construction of an octree from points, and whole steps of the segmentation U-Net that
start from points, as a server or a training loop that gets new clouds with every call does.

  listed()            the cases that stand for the range
  draw(rng)           one more case of the same ranges
  prepare(case, seed) what the user's program holds before the call
  run(state)          one pass through the public entry points
  work(case)          bytes and operations that a pass cannot do without
  tolerance(case)     how far apart two correct implementations' results may be
"""

import functools
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), 'ocnn-pytorch_amd'))

from ocnn_amd import synthetic                                               # noqa: E402
from ocnn_amd.nn import OctreeConv, OctreeDeconv, OctreeDWConv               # noqa: E402
from ocnn_amd.octree import Octree, Points                                   # noqa: E402
from ocnn_amd.octree.octree import PlanHistory                               # noqa: E402
from ocnn_amd.unet import (DECODER_BLOCKS, DECODER_CHANNELS, ENCODER_BLOCKS, ENCODER_CHANNELS, HEAD_CHANNELS,  # noqa: E402
                           UNet)

FULL_DEPTH = 2
CLASSES = 10
LOSS_SCALE, LEARNING_RATE = 1024.0, 0.01
DTYPES = {'fp32': torch.float32, 'fp16': torch.float16, 'bf16': torch.bfloat16}
CLOUDS = {'sphere': synthetic.sphere_cloud, 'mixed': synthetic.mixed_cloud, 'planes': synthetic.planes_cloud,
          'indoor': synthetic.indoor_cloud}


def _conv(name, cloud, batch, points, depth, cin, cout, dtype, nempty, bias, backward=True):
  return {'name': name, 'kind': 'conv', 'cloud': cloud, 'batch': batch, 'points': points, 'depth': depth, 'cin': cin,
          'cout': cout, 'dtype': dtype, 'nempty': nempty, 'bias': bias, 'backward': backward}


def listed():
  return [
      # one object scanned into a shallow octree, single precision, training: the smallest of the
      # single-layer configurations (one 3x3x3 convolution, forward + backward)
      _conv('conv_d6_c32_fp32', 'sphere', 1, 20000, 6, 32, 32, 'fp32', False, False),
      # the bottom level of a network: few nodes, many channels, with bias (the first point of the
      # layer benchmark's sweep is of this size): launches and latency count
      _conv('conv_d5_c256_bf16', 'sphere', 1, 30011, 5, 256, 256, 'bf16', True, True),
      # the headline layer: a batch of eight clouds at depth 8, all nodes
      _conv('conv_d8_c64_bf16', 'mixed', 8, 100000, 8, 64, 64, 'bf16', False, False),
      # the same level in single precision on the non-empty nodes, with bias (the layer benchmark's
      # depth-8 point: about 250 k rows)
      _conv('conv_d8_c64_fp32', 'mixed', 4, 100003, 8, 64, 64, 'fp32', True, True),
      # the finest level of a deep network: the most rows, the fewest channels
      _conv('conv_d9_c32_bf16', 'planes', 4, 250000, 9, 32, 32, 'bf16', False, False),
      # a coarse level with many channels, all nodes: the matrix-bound end
      _conv('conv_d6_c256_bf16', 'planes', 4, 250000, 6, 256, 256, 'bf16', False, False),
      # down by a 2x2x2 stride-2 convolution, a depth-wise convolution there, and up again by the
      # deconvolution, over all nodes
      {'name': 'down_up_d8_bf16', 'kind': 'stage', 'cloud': 'mixed', 'batch': 8, 'points': 100000, 'depth': 8,
       'channels': 64, 'dtype': 'bf16', 'nempty': False},
      # one small cloud to its octree and neighbour tables: what a server or an interactive tool does per request
      {'name': 'octree_d6', 'kind': 'octree', 'cloud': 'sphere', 'batch': 1, 'points': 20011, 'depth': 6},
      # a training batch of a million points to its octree and tables
      {'name': 'octree_d9', 'kind': 'octree', 'cloud': 'planes', 'batch': 4, 'points': 250000, 'depth': 9},
      # segmentation of one cloud, points to logits, by a trained network: the latency of a served request
      {'name': 'unet_infer_d7', 'kind': 'unet', 'cloud': 'indoor', 'batch': 1, 'points': 40009, 'depth': 7,
       'dtype': 'fp16', 'train': False},
      # training steps of the segmentation network on new clouds: octree, forward, loss, backward, update.
      # A small batch in single precision (the network's own default) ...
      {'name': 'unet_train_d7_fp32', 'kind': 'unet', 'cloud': 'mixed', 'batch': 2, 'points': 30011, 'depth': 7,
       'dtype': 'fp32', 'train': True},
      # ... and a large one in half precision, with a scaled loss
      {'name': 'unet_train_d9_fp16', 'kind': 'unet', 'cloud': 'indoor', 'batch': 8, 'points': 150000, 'depth': 9,
       'dtype': 'fp16', 'train': True},
  ]


# points of one cloud, and the channels the levels have, by depth
_POINTS = {5: (3000, 40000), 6: (5000, 80000), 7: (20000, 120000), 8: (50000, 250000), 9: (100000, 250000)}
_CHANNELS = {5: (64, 96, 128, 192, 256), 6: (32, 64, 96, 128, 192, 256), 7: (32, 64, 96, 128, 192), 8: (32, 64, 96, 128),
             9: (32, 64, 96)}
MOST_POINTS = 1200000


def _scene(rng, depths):
  depth = rng.choice(depths)
  lo, hi = _POINTS[depth]
  batch = rng.choice((1, 1, 2, 3, 4, 6, 8))
  points = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
  cloud = rng.choice(('mixed', 'planes', 'indoor') if depth >= 7 else ('sphere', 'mixed', 'indoor'))
  return {'cloud': cloud, 'batch': batch, 'points': min(points, MOST_POINTS // batch), 'depth': depth}


def draw(rng):
  kind = rng.choices(('conv', 'stage', 'octree', 'infer', 'train'), (6, 1, 2, 2, 1))[0]
  if kind == 'conv':
    case = dict(kind='conv', **_scene(rng, (5, 6, 7, 8, 9)))
    channels = _CHANNELS[case['depth']]
    case['cin'], case['cout'] = rng.choice(channels), rng.choice(channels)
    if rng.random() < 0.7:                             # most layers keep their width
      case['cout'] = case['cin']
    elif rng.random() < 0.3:                           # the first layer of a network: normals + displacement
      case['cin'] = 4
    case['dtype'] = rng.choice(('bf16', 'bf16', 'fp16', 'fp32'))
    case['nempty'] = rng.random() < 0.6
    case['bias'] = rng.random() < 0.3
    case['backward'] = rng.random() < 0.75
    if case['dtype'] == 'fp32' and case['depth'] >= 8:
      case['cin'], case['cout'] = min(case['cin'], 64), min(case['cout'], 64)
    return case
  if kind == 'stage':
    case = dict(kind='stage', **_scene(rng, (6, 7, 8)))
    case['channels'] = rng.choice((32, 64))
    case['dtype'] = rng.choice(('bf16', 'fp16'))
    case['nempty'] = rng.random() < 0.4
    return case
  if kind == 'octree':
    return dict(kind='octree', **_scene(rng, (5, 6, 7, 8, 9)))
  case = dict(kind='unet', **_scene(rng, (6, 7, 8) if kind == 'infer' else (6, 7, 8, 9)))
  case['dtype'] = rng.choice(('fp16', 'bf16' if kind == 'infer' else 'fp32'))
  if case['dtype'] == 'fp32' and case['depth'] >= 8:   # large batches are trained in half precision
    case['points'] = min(case['points'], 240000 // case['batch'])
  case['train'] = kind == 'train'
  return case


# ---- what the user's program holds -----------------------------------------------------------------

@functools.lru_cache(maxsize=4)
def _scene_points(cloud, batch, points):
  return [t.cuda() for t in synthetic.batch_clouds(CLOUDS[cloud], batch, 1000, n=points)]


def _points(case, seed):
  """The scene of the case, turned (the axes permuted) and with its points in another order for every
  seed: other keys, rows and neighbours, of the same numbers."""
  pts, nrm, bid = _scene_points(case['cloud'], case['batch'], case['points'])
  gen = torch.Generator(device='cuda').manual_seed(seed)
  order = torch.argsort(torch.rand(pts.shape[0], generator=gen, device='cuda') + bid.view(-1).double())
  axes = ((0, 1, 2), (1, 2, 0), (2, 0, 1), (0, 2, 1), (2, 1, 0), (1, 0, 2))[seed % 6]
  pts, nrm, bid = pts[order][:, axes].contiguous(), nrm[order][:, axes].contiguous(), bid[order]
  return Points(pts, nrm, batch_id=bid if case['batch'] > 1 else None, batch_size=case['batch']), pts, bid


def _octree(case, points, history):
  octree = Octree(case['depth'], FULL_DEPTH, batch_size=case['batch'])
  octree.plan_history = history                        # of this program's octrees, not of every octree in the process
  octree.build_octree(points)
  octree.construct_all_neigh()
  return octree


def _rows(octree, depth, nempty):
  return int(octree.nnum_nempty[depth] if nempty else octree.nnum[depth])


def prepare(case, seed):
  points, pts, bid = _points(case, seed)
  kind, history = case['kind'], PlanHistory()
  state = {'case': case, 'points': points, 'history': history}
  if kind == 'octree':
    return state
  dtype = DTYPES[case['dtype']]
  gen = torch.Generator(device='cuda').manual_seed(seed)
  randn = lambda *shape: torch.randn(*shape, generator=gen, device='cuda').to(dtype)
  torch.manual_seed(seed)                              # the modules' own initialisation
  if kind == 'unet':
    net = UNet(4, CLASSES, 'linear', True).cuda().to(dtype)
    net.train(case['train'])
    with torch.no_grad():
      for name, norm in net.named_modules():           # residual branches that start small, as deep networks' do
        if name.endswith('conv3x3b.bn'):
          norm.weight.fill_(0.25)
    labels = ((pts[:, 2:] + 1) * (CLASSES / 2)).long().clamp_(0, CLASSES - 1)   # what a point is depends on where it is
    params = list(net.parameters())
    state.update(net=net, params=params, optimizer=torch.optim.SGD(params, LEARNING_RATE / LOSS_SCALE),
                 stats=[b for name, b in net.named_buffers() if name.endswith(('running_mean', 'running_var'))],
                 query=torch.cat([pts, bid], 1), dtype=dtype, labels=labels)
    return state
  depth, nempty = case['depth'], case['nempty']
  octree = state['octree'] = _octree(case, points, history)
  rows = _rows(octree, depth, nempty)
  if kind == 'conv':
    layers = [OctreeConv(case['cin'], case['cout'], [3], 1, nempty=nempty, use_bias=case['bias'])]
    cin, cout = case['cin'], case['cout']
  else:
    cin = cout = case['channels']
    layers = [OctreeConv(cin, 2 * cin, [2], 2, nempty=nempty), OctreeDWConv(2 * cin, [3], 1, nempty=nempty),
              OctreeDeconv(2 * cin, cout, [2], 2, nempty=nempty)]
  backward = case.get('backward', True)
  state.update(layers=[m.cuda().to(dtype).requires_grad_(backward) for m in layers], backward=backward,
               x=randn(rows, cin).requires_grad_(backward), grad=randn(rows, cout) if backward else None)
  state['params'] = [p for m in layers for p in m.parameters()]
  return state


# ---- one pass --------------------------------------------------------------------------------------

def _run_octree(state):
  octree = _octree(state['case'], state['points'], state['history'])
  depth = octree.depth
  return {'keys': octree.keys, 'children': octree.children, 'points': octree.points[depth],
          'normals': octree.normals[depth], 'neighs': [octree.neighs.get32(d) for d in range(1, depth + 1)]}


def _run_unet(state):
  case, net = state['case'], state['net']
  octree = _octree(case, state['points'], state['history'])
  feature = octree.get_input_feature('ND', True).to(state['dtype'])
  query = state['query'].clone()                       # (the interpolation rescales its points in place)
  if not case['train']:
    with torch.no_grad():
      return net(feature, octree, case['depth'], query)
  state['optimizer'].zero_grad()
  logits = net(feature, octree, case['depth'], query).float()
  loss = (torch.logsumexp(logits, 1) - logits.gather(1, state['labels']).squeeze(1)).mean()
  (loss * LOSS_SCALE).backward()
  state['optimizer'].step()
  return {'loss': loss.detach(), 'logits': logits.detach(),
          'params': torch.cat([p.detach().view(-1) for p in state['params']]),
          'stats': torch.cat([b.view(-1) for b in state['stats']])}


def _run_layers(state):
  octree, depth = state['octree'], state['case']['depth']
  if not state['backward']:
    return state['layers'][0](state['x'], octree, depth)
  x = state['x']
  x.grad = None
  for p in state['params']:
    p.grad = None
  if len(state['layers']) == 1:
    out = state['layers'][0](x, octree, depth)
  else:
    down, depthwise, up = state['layers']
    out = up(depthwise(down(x, octree, depth), octree, depth - 1), octree, depth - 1)
  out.backward(state['grad'])
  return [out.detach(), x.grad] + [p.grad for p in state['params']]


def run(state):
  kind = state['case']['kind']
  return _run_octree(state) if kind == 'octree' else _run_unet(state) if kind == 'unet' else _run_layers(state)


# ---- what a pass cannot do without -----------------------------------------------------------------

@functools.lru_cache(maxsize=64)
def _counts(cloud, batch, points, depth):
  """{depth: (nodes, non-empty nodes, pairs of neighbouring nodes, of neighbouring non-empty nodes)}
  of the octree, from sorted cell numbers; pairs: entries of a 3x3x3 table that hold a node."""
  pts, _, bid = synthetic.batch_clouds(CLOUDS[cloud], batch, 1000, n=points)
  dev = 'cuda' if torch.cuda.is_available() else 'cpu'
  pts, bid = pts.to(dev).double(), bid.to(dev).long().view(-1)
  out = {}
  for d in range(FULL_DEPTH, depth + 1):
    side = 2 ** d + 2                                  # a rim of one cell: neighbours stay inside the cloud's own range

    def number(xyz, b):
      x, y, z = (xyz + 1).unbind(1)
      return ((b * side + x) * side + y) * side + z

    def pairs(cells):
      n = 0
      for o in range(27):
        near = cells + ((o // 9 - 1) * side + (o // 3) % 3 - 1) * side + o % 3 - 1
        at = torch.searchsorted(cells, near).clamp_max(cells.numel() - 1)
        n += int((cells[at] == near).sum())
      return n

    cell = ((pts + 1) * 2.0 ** (d - 1)).floor().long().clamp(0, 2 ** d - 1)
    leaves = torch.unique(number(cell, bid))
    if d > FULL_DEPTH:
      both = torch.unique(torch.cat([cell // 2, bid.view(-1, 1)], 1), dim=0)
      corner = torch.tensor([[i // 4, (i // 2) % 2, i % 2] for i in range(8)], device=dev)
      xyz = (2 * both[:, None, :3] + corner).view(-1, 3)
      nodes = torch.sort(number(xyz, both[:, 3].repeat_interleave(8)))[0]
      out[d] = (nodes.numel(), leaves.numel(), pairs(nodes), pairs(leaves))
    else:
      n = batch << (3 * d)
      out[d] = (n, leaves.numel(), batch * (3 * 2 ** d - 2) ** 3, pairs(leaves))
  return out


def _octree_bytes(case, counts):
  batch = case['batch']
  nodes = sum(batch << (3 * d) for d in range(FULL_DEPTH)) + sum(c[0] for c in counts.values())
  leaves = counts[case['depth']][1]
  return batch * case['points'] * (12 + 12 + (4 if batch > 1 else 0)) + nodes * (8 + 4 + 27 * 4) + leaves * 24


def _layer(size, fine, coarse, taps, cin, cout, table, backward, groups=1):
  """(bytes, flops) of one layer: features, weights and gradients moved once, 4-byte table entries;
  `fine` rows with cin channels in, `coarse` rows with cout channels out, `taps` pairs of rows."""
  weights = table[1] * cin * cout // groups
  flops = 2.0 * taps * cin * cout / groups
  bytes_ = size * (fine * cin + coarse * cout + weights) + 4 * table[0] * table[1]
  if backward:
    return bytes_ + size * (fine * cin + coarse * cout + weights), 3 * flops
  return bytes_, flops


def _unet_work(case, counts):
  depth, size, train = case['depth'], DTYPES[case['dtype']].itemsize, case['train']
  rows = lambda d: counts[d][1]
  total = [float(_octree_bytes(case, counts)), 0.0]

  def add(layer):
    total[0] += layer[0]
    total[1] += layer[1]

  def conv3(d, cin, cout):
    add(_layer(size, rows(d), rows(d), counts[d][3], cin, cout, (rows(d), 27), train))

  def conv2(d, c_fine, c_coarse):
    add(_layer(size, rows(d), rows(d - 1), rows(d), c_fine, c_coarse, (rows(d - 1), 8), train))

  def rows_linear(n, cin, cout):
    add(_layer(size, n, n, n, cin, cout, (0, 1), train))

  def blocks(d, cin, cout, n):
    for i in range(n):
      conv3(d, cin if i == 0 else cout, cout)
      conv3(d, cout, cout)
    if cin != cout:
      rows_linear(rows(d), cin, cout)

  enc, dec = ENCODER_CHANNELS, DECODER_CHANNELS
  conv3(depth, 4, enc[0])
  for i, n in enumerate(ENCODER_BLOCKS):
    conv2(depth - i, enc[i], enc[i + 1])
    blocks(depth - i - 1, enc[i + 1], enc[i + 1], n)
  d = depth - len(ENCODER_BLOCKS)
  for i, n in enumerate(DECODER_BLOCKS):
    conv2(d + i + 1, dec[i + 1], dec[i])
    blocks(d + i + 1, dec[i + 1] + enc[-i - 2], dec[i + 1], n)
  points = case['batch'] * case['points']
  rows_linear(points, dec[-1], HEAD_CHANNELS)
  rows_linear(points, HEAD_CHANNELS, CLASSES)
  return total


def work(case):
  counts = _counts(case['cloud'], case['batch'], case['points'], case['depth'])
  kind, depth = case['kind'], case['depth']
  if kind == 'octree':
    return {'bytes': _octree_bytes(case, counts), 'flops': 0}
  if kind == 'unet':
    bytes_, flops = _unet_work(case, counts)
    return {'bytes': bytes_, 'flops': flops}
  size, side = DTYPES[case['dtype']].itemsize, 1 if case['nempty'] else 0
  rows, taps = counts[depth][side], counts[depth][2 + side]
  if kind == 'conv':
    bytes_, flops = _layer(size, rows, rows, taps, case['cin'], case['cout'], (rows, 27), case['backward'])
    return {'bytes': bytes_, 'flops': flops}
  c, up_rows, parents = case['channels'], counts[depth - 1][side], counts[depth - 1][1]
  table = (parents, 8) if case['nempty'] else (0, 8)   # (over all nodes the children are consecutive rows)
  parts = [_layer(size, rows, up_rows, rows, c, 2 * c, table, True)] * 2 + [
      _layer(size, up_rows, up_rows, counts[depth - 1][2 + side], 2 * c, 2 * c, (up_rows, 27), True, groups=2 * c)]
  return {'bytes': sum(p[0] for p in parts), 'flops': sum(p[1] for p in parts)}


def tolerance(case):
  if case['kind'] == 'octree':
    return {'rel': 1e-6}                               # whole numbers equal; the leaves' mean points are fp32 sums
  if case['kind'] == 'unet':
    if not case['train']:
      return {'rel': 1e-2 if case['dtype'] == 'bf16' else 2e-3}
    # (rounding grows through some 60 layers with batch statistics)
    return {'rel': 1e-3, 'max': 0.1} if case['dtype'] == 'fp32' else {'rel': 2e-2, 'max': 0.5}
  if case['dtype'] == 'fp32':
    return {'rel': 1e-5}
  return {'rel': 1e-2 if case['dtype'] == 'bf16' else 2e-3}

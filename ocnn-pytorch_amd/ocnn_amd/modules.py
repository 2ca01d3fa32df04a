"""Compositions of the hot-path layers with batch norm / ReLU / Linear under the class and
attribute names of ocnn/modules/modules.py and ocnn/modules/resblocks.py, so that networks
written against the reference (and their state_dicts) work unchanged.  The batch norm is a
BatchNorm1d subclass that runs on fused HIP kernels (statistics, normalise + ReLU in one pass)."""

from typing import List

import torch
import torch.nn
import torch.nn.functional as F

from . import _lib
from .nn import OctreeConv, OctreeDeconv
from .octree import Octree
from .nn.octree_conv import _gather_op, _wgrad_op, call_native, conv_wgrad, column_sum
from .nn.batchnorm import BatchNormRelu1d, kernels_take


class _LayerBn(torch.nn.Module):
  """layer -> BatchNorm1d [-> ReLU]; `name` is the attribute the layer is stored under."""

  def __init__(self, name, layer, channels, relu):
    super().__init__()
    self._name = name
    setattr(self, name, layer)
    self.bn = BatchNormRelu1d(channels, relu=relu)          # BatchNorm1d with the ReLU fused in
    if relu:
      self.relu = torch.nn.ReLU(inplace=True)               # (kept for the module tree; applied by bn)

  def forward(self, data, *args):
    return layer_bn(getattr(self, self._name), self.bn, data, *args)


_nn = torch.nn.modules.module


def _plain(module):
  """A call of the module runs the forward() of its class and nothing else: no hooks, no forward put on the
  module itself (as libraries that place modules on devices do), no compiled call."""
  own = module.__dict__
  return not (own['_forward_hooks'] or own['_forward_pre_hooks'] or 'forward' in own or
              own.get('_compiled_call_impl') is not None)


def layer_bn(layer, bn, data, *args, residual=None, relu=None):
  """bn(layer(data, *args), residual, relu).  In evaluation without gradients, with the layer and the
  batch norm of this package as they are, one native call: the normalisation then rides on the
  convolution's own pass over its result instead of reading and writing it once more."""
  if (not torch.is_grad_enabled() and not _lib.recorded() and type(bn) is BatchNormRelu1d and not bn.training and
      type(layer) in (OctreeConv, OctreeDeconv, Conv1x1) and _plain(layer) and _plain(bn) and
      not (_nn._global_forward_hooks or _nn._global_forward_pre_hooks)):
    # (the tensors out of the modules' own dictionaries: as attributes of a Module each costs a search in Python,
    # a tenth of the host time of a small network; one that is not where the constructor put it: the general route)
    stats, affine = bn._buffers, bn._parameters
    if stats.get('running_mean') is not None and 'running_var' in stats and 'weight' in affine and 'bias' in affine:
      native = layer.native_layer(data, *args)
      if native is not None and kernels_take(data.dtype, bn.num_features):
        own, name = (layer.linear, 'weight') if type(layer) is Conv1x1 else (layer, 'weights')
        held = own._parameters
        return _lib.native().conv_bn(native, data, held[name] if name in held else getattr(own, name),
                                     held['bias'] if 'bias' in held else own.bias, stats['running_mean'],
                                     stats['running_var'], bn.eps, affine['weight'], affine['bias'],
                                     bn.fused_relu if relu is None else relu, residual)
  if residual is None and relu is None:
    return bn(layer(data, *args))
  return bn(layer(data, *args), residual=residual, relu=relu)


def _res_blocks(blocks, data, octree, depth):
  """Residual blocks one behind the other in evaluation without gradients, every layer and batch norm as this package makes
  them: one native call, which packs the weights of all of them in one launch.  None: by the modules themselves."""
  if (torch.is_grad_enabled() or _lib.recorded() or _nn._global_forward_hooks or _nn._global_forward_pre_hooks or
      not (isinstance(octree, Octree) and data.is_cuda and data.dim() == 2 and data.dtype in _lib.DTYPE_CODE)):
    return None
  native, dtype, (rows, width), layers = _lib.native(), data.dtype, data.shape, []
  for block in blocks:
    if type(block) is not OctreeResBlock2 or block.in_channels != width:
      return None
    parts = block._modules
    for name, kind, relu in (('conv3x3a', OctreeConvBnRelu, None), ('conv3x3b', OctreeConvBn, True)):
      part = parts.get(name)
      if type(part) is not kind or not _plain(part):
        return None
      conv, bn = part._modules.get('conv'), part._modules.get('bn')
      if not (type(conv) is OctreeConv and type(bn) is BatchNormRelu1d and not bn.training and _plain(conv) and _plain(bn)):
        return None
      stats, affine, held = bn._buffers, bn._parameters, conv._parameters
      if not (stats.get('running_mean') is not None and 'running_var' in stats and 'weight' in affine and 'bias' in affine and
              'weights' in held):
        return None
      made = conv.native_of_stride_1(dtype, (rows, width), octree, depth)
      if made is None or not kernels_take(dtype, bn.num_features):
        return None
      width = conv.out_channels
      layers.append(native.BlockLayer(made, held['weights'], held['bias'] if 'bias' in held else conv.bias, stats['running_mean'],
                                      stats['running_var'], bn.eps, affine['weight'], affine['bias'],
                                      bn.fused_relu if relu is None else relu))
    if block.in_channels != block.out_channels and block is not blocks[0]:
      return None                                           # (its shortcut is a layer between the blocks)
    if width != block.out_channels:
      return None
  first = blocks[0]
  return native.res_blocks(layers, data, first.conv1x1(data) if first.in_channels != first.out_channels else None)


class OctreeConvBn(_LayerBn):
  """ocnn/modules/modules.py:32-51."""

  def __init__(self, in_channels: int, out_channels: int, kernel_size: List[int] = [3],
               stride: int = 1, nempty: bool = False):
    super().__init__('conv', OctreeConv(in_channels, out_channels, kernel_size, stride, nempty),
                     out_channels, False)


class OctreeConvBnRelu(_LayerBn):
  """ocnn/modules/modules.py:54-75."""

  def __init__(self, in_channels: int, out_channels: int, kernel_size: List[int] = [3],
               stride: int = 1, nempty: bool = False):
    super().__init__('conv', OctreeConv(in_channels, out_channels, kernel_size, stride, nempty),
                     out_channels, True)


class OctreeDeconvBnRelu(_LayerBn):
  """ocnn/modules/modules.py:78-99."""

  def __init__(self, in_channels: int, out_channels: int, kernel_size: List[int] = [3],
               stride: int = 1, nempty: bool = False):
    super().__init__('deconv', OctreeDeconv(in_channels, out_channels, kernel_size, stride, nempty),
                     out_channels, True)


_IDENTITY = {}


def _identity_table(rows, device):
  """(rows or more, 1) table [0, 1, ..]: row i reads row i.  One per device and stream, as long as the
  longest asked for (an eighth longer at most): row counts differ with every octree.  Of each stream its
  own, so that memory given back is not reused before its readers are done; under capture the graph's own."""
  key = (device, _lib.stream())
  table = _IDENTITY.get(key)
  capturing = torch.cuda.is_current_stream_capturing()
  if table is None or table.shape[0] < rows or capturing:
    step = max(1024, 1 << max(rows.bit_length() - 3, 0))
    table = torch.arange(-(-rows // step) * step, dtype=torch.int32, device=device).view(-1, 1)
    if not capturing:
      if len(_IDENTITY) > 16:
        _IDENTITY.clear()
      _IDENTITY[key] = table
  return table


_LINEAR = {}


def _reads_table(op):
  """The pass goes over the one-slot table (the dense kernels do without)."""
  return (op.padded or op).kernel == _lib.GATHER_PLAIN       # (the same number as WGRAD_PLAIN)


def _rows_linear_layer(x, cin, cout):
  """y = x W^T on many rows as the one-slot form of the convolution kernels (weights (out, in) as
  torch.nn.Linear holds them)."""
  rows = x.shape[0]
  key = (rows, cin, cout, x.dtype)
  made = _LINEAR.get(key)
  if made is None:
    if len(_LINEAR) > 64:
      _LINEAR.clear()
    layer = _lib.native().ConvLayer(_gather_op(x.dtype, rows, rows, 1, cin, cout, True, False, None, True), None, False)
    layer = layer.with_dgrad(_gather_op(x.dtype, rows, rows, 1, cout, cin, False, False, None, True), None)
    layer = layer.with_wgrad(_wgrad_op(x.dtype, rows, rows, 1, cin, cout, True, None, True).seen_as([cout, cin]), None)
    # (whole: other threads take it from here.  Without the table, which would outlive the octree)
    forward = _reads_table(layer.fwd)
    made = _LINEAR[key] = (layer, forward, forward or _reads_table(layer.dgrad) or _reads_table(layer.wgrad))
  layer, forward, training = made
  if training if torch.is_grad_enabled() else forward:
    return layer.with_table(_identity_table(rows, x.device), rows)
  return layer


class _RowsLinearNarrow(torch.autograd.Function):
  """y = x W^T + b for few output channels (a classification head: 64 -> 10 on a million
  rows).  Output and input gradient are the library's GEMMs; the weight gradient, a sum over
  all rows into a handful of numbers, is where the library's choice of kernel is slow (0.89 ms
  for 1.2 M x 64 x 10) and runs on this package's split reduction instead (fixed order)."""

  @staticmethod
  def forward(ctx, x, weight, bias):
    x = x.contiguous()
    ctx.save_for_backward(x, weight)
    ctx.has_bias = bias is not None
    return F.linear(x, weight.to(x.dtype), None if bias is None else bias.to(x.dtype))

  @staticmethod
  def backward(ctx, grad):
    x, weight = ctx.saved_tensors
    grad = grad.contiguous()
    rows = x.shape[0]
    gx = gw = gb = None
    if ctx.needs_input_grad[0]:
      gx = grad @ weight.to(grad.dtype)
    if ctx.needs_input_grad[1]:
      gw = conv_wgrad(x, grad, _identity_table(rows, x.device)[:rows], True, None, dense=True)
      gw = gw.view(weight.shape).to(weight.dtype)
    if ctx.has_bias and ctx.needs_input_grad[2]:
      gb = column_sum(grad)
    return gx, gw, gb


class _RowsWgrad(torch.autograd.Function):
  """g^T x of fp32 rows, every product and sum in fp32 (ocnnx_rows_wgrad), and differentiable again."""

  @staticmethod
  def forward(ctx, g, x):
    ctx.save_for_backward(g, x)
    return _lib.native().rows_wgrad(g, x)

  @staticmethod
  def backward(ctx, grad):
    g, x = ctx.saved_tensors
    return (x @ grad.t() if ctx.needs_input_grad[0] else None, g @ grad if ctx.needs_input_grad[1] else None)


def _rows_wgrad(g, x):
  """g^T x on the kernel; the library's product for operands that it cannot read: gradients asked for as a batch
  (is_grads_batched: a tensor without storage), negated views and zeros without memory, subclasses, more than its 4 GB
  (of a trace, which is not asked again), and wherever a tangent, a transform or a trace rides on them."""
  if _lib.recorded() or not all(type(t) is torch.Tensor and torch._C._has_storage(t) and not t.is_neg() and
                                not t._is_zerotensor() for t in (g, x)) or \
      not _lib.lib().ocnnx_rows_wgrad_supported(0, x.shape[0], g.shape[1], x.shape[1]):
    return g.t() @ x
  return _RowsWgrad.apply(g, x) if torch.is_grad_enabled() else _lib.native().rows_wgrad(g, x)


class _RowsLinear32(torch.autograd.Function):
  """torch.nn.functional.linear on many fp32 rows, with the weight gradient on this package's kernel: a sum over all
  rows into a small matrix, for which the library runs a handful of workgroups (us, library / kernel, with a norm of
  the error of 1 - 10e-6 / 0.2 - 1e-6: 31 k rows of 96 -> 64 104 / 16, 192 -> 128 84 / 25, 384 -> 256 112 / 65, 512 -> 512
  180 / 148; 300 k rows 626 / 62, 634 / 171, 752 / 554, 1585 / 1381; 4096 rows 24 - 33 / 10 - 12, 512 -> 512 28 / 30)."""

  @staticmethod
  def forward(ctx, x, weight, bias):
    ctx.save_for_backward(x, weight)
    return F.linear(x, weight, bias)

  @staticmethod
  def backward(ctx, grad):
    x, weight = ctx.saved_tensors
    needs = ctx.needs_input_grad
    return (grad @ weight if needs[0] else None, _rows_wgrad(grad, x) if needs[1] else None,
            grad.sum(0) if needs[2] else None)


def _takes_rows32(data, lin):
  """The fp32 weight gradient of `lin` on `data` can run on this package's kernel: plain tensors of many rows, no hook
  that would miss the Linear, no data type chosen by autocast.  A trace keeps the Linear, which can be saved with it,
  unless what it holds so far cannot be saved anyway: then training gives the bits that it gives outside."""
  weight, bias = lin.weight, lin.bias
  if not (torch.is_grad_enabled() and not torch.compiler.is_compiling() and data.dim() == 2 and data.is_cuda and
          data.dtype == torch.float32 and type(data) is torch.Tensor and weight.requires_grad and
          type(weight) is torch.nn.Parameter and weight.dtype == torch.float32 and weight.device == data.device and
          (bias is None or (bias.dtype == torch.float32 and bias.device == data.device))):
    return False
  if _lib.recorded() and not (lin.training and _lib.only_traced() and _lib.trace_stays_here()):
    return False
  rows, width, cout, cin = _lib.unrecorded(lambda: (*data.shape, *weight.shape))     # (numbers, also in a trace)
  if not (rows >= 4096 and cin == width and cin % 4 == 0 and max(cin, cout) <= 512 and
          _lib.lib().ocnnx_rows_wgrad_supported(0, rows, cout, cin)):
    return False
  return (type(lin) is torch.nn.Linear and _plain(lin) and
          not (lin._backward_hooks or lin._backward_pre_hooks or _nn._global_forward_hooks or
               _nn._global_forward_pre_hooks or _nn._global_backward_hooks or _nn._global_backward_pre_hooks or
               torch.is_autocast_enabled()))


class Conv1x1(torch.nn.Module):
  """ocnn/modules/modules.py:102-117: a 1x1x1 convolution on (N, C) rows is a Linear (same
  parameters as torch.nn.Linear; large 16-bit inputs run on this package's GEMM kernels, and so does the
  weight gradient of large fp32 ones)."""

  def __init__(self, in_channels: int, out_channels: int, use_bias: bool = False):
    super().__init__()
    self.linear = torch.nn.Linear(in_channels, out_channels, use_bias)

  def native_layer(self, data: torch.Tensor):
    """The passes on this package's kernels, or None for the library's."""
    lin = self.linear
    if (data.dim() == 2 and data.is_cuda and data.dtype in (torch.float16, torch.bfloat16) and
        data.shape[0] >= 4096 and lin.in_features % 32 == 0 and lin.out_features % 16 == 0):
      return _lib.unrecorded(_rows_linear_layer, data, lin.in_features, lin.out_features)
    return None

  def forward(self, data: torch.Tensor):
    lin = self.linear
    native = self.native_layer(data)
    if native is not None:
      return call_native(native, data, lin.weight, lin.bias)
    if (data.dim() == 2 and data.is_cuda and data.dtype in (torch.float16, torch.bfloat16) and
        data.shape[0] >= 65536 and lin.in_features % 32 == 0 and lin.out_features < 16):
      return _RowsLinearNarrow.apply(data, lin.weight, lin.bias)
    if _takes_rows32(data, lin):
      return _RowsLinear32.apply(data, lin.weight, lin.bias)
    return lin(data)


class Conv1x1Bn(_LayerBn):
  """ocnn/modules/modules.py:120-134."""

  def __init__(self, in_channels: int, out_channels: int):
    super().__init__('conv', Conv1x1(in_channels, out_channels, use_bias=False), out_channels, False)


class Conv1x1BnRelu(_LayerBn):
  """ocnn/modules/modules.py:137-153."""

  def __init__(self, in_channels: int, out_channels: int):
    super().__init__('conv', Conv1x1(in_channels, out_channels, use_bias=False), out_channels, True)


class OctreeResBlock2(torch.nn.Module):
  """Two 3x3x3 convolutions with a (projected) shortcut, stride 1
  (ocnn/modules/resblocks.py:65-99)."""

  def __init__(self, in_channels, out_channels, stride=1, bottleneck=1, nempty=False):
    super().__init__()
    assert stride == 1, 'OctreeResBlock2: stride 1 only'
    self.in_channels, self.out_channels, self.stride = in_channels, out_channels, stride
    mid = int(out_channels / bottleneck)
    self.conv3x3a = OctreeConvBnRelu(in_channels, mid, nempty=nempty)
    self.conv3x3b = OctreeConvBn(mid, out_channels, nempty=nempty)
    if in_channels != out_channels:
      self.conv1x1 = Conv1x1Bn(in_channels, out_channels)
    self.relu = torch.nn.ReLU(inplace=True)

  def forward(self, data: torch.Tensor, octree, depth: int):
    out = _res_blocks((self,), data, octree, depth)
    if out is not None:
      return out
    out = self.conv3x3a(data, octree, depth)
    if self.in_channels != self.out_channels:
      data = self.conv1x1(data)
    # relu(bn(conv(out)) + data): the sum and the ReLU ride on the batch norm's pass
    last = self.conv3x3b
    return layer_bn(last.conv, last.bn, out, octree, depth, residual=data, relu=True)


class OctreeResBlocks(torch.nn.Module):
  """A chain of residual blocks (ocnn/modules/resblocks.py:134-159)."""

  def __init__(self, in_channels, out_channels, resblk_num, bottleneck=4, nempty=False,
               resblk=OctreeResBlock2, use_checkpoint=False):
    super().__init__()
    self.resblk_num = resblk_num
    self.use_checkpoint = use_checkpoint
    widths = [in_channels] + [out_channels] * resblk_num
    self.resblks = torch.nn.ModuleList(
        [resblk(widths[i], widths[i + 1], 1, bottleneck, nempty) for i in range(resblk_num)])

  def forward(self, data: torch.Tensor, octree, depth: int):
    blocks = tuple(self.resblks)
    if not torch.is_grad_enabled() and not self.use_checkpoint and blocks and all(_plain(blk) for blk in blocks):
      out = _res_blocks(blocks, data, octree, depth)
      if out is not None:
        return out
    for blk in blocks:
      if self.use_checkpoint:
        data = torch.utils.checkpoint.checkpoint(blk, data, octree, depth, use_reentrant=False)
      else:
        data = blk(data, octree, depth)
    return data


class InputFeature(torch.nn.Module):
  """The input signal stored in the octree (ocnn/modules/modules.py:288-305)."""

  def __init__(self, feature: str = 'NDF', nempty: bool = False):
    super().__init__()
    self.nempty = nempty
    self.feature = feature.upper()

  def forward(self, octree):
    return octree.get_input_feature(self.feature, self.nempty)

  def extra_repr(self) -> str:
    return 'feature={}, nempty={}'.format(self.feature, self.nempty)

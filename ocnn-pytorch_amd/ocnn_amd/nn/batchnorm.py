"""torch.nn.BatchNorm1d on (rows, C) feature matrices with an optional fused ReLU, on HIP
kernels (same parameters, buffers and state_dict keys as BatchNorm1d).  What the reference
builds from BatchNorm1d + ReLU(inplace) after every convolution
(ocnn/modules/modules.py:32-99, 120-153)."""

import functools

import torch
import torch.nn

from .. import _lib


@functools.lru_cache(maxsize=256)
def kernels_take(dtype, channels):
  """The kernels take rows of these channels in this type, any number of them but none."""
  code = _lib.DTYPE_CODE.get(dtype, -1)
  return code >= 0 and bool(_lib.lib().ocnn_batch_norm_supported(code, 1, channels))


class _BatchNormFunction(torch.autograd.Function):
  """The module's pass as an autograd.Function, for calls that something records (_lib.recorded)."""

  @staticmethod
  def forward(ctx, x, weight, bias, residual, running_mean, running_var, counter, use_batch_stats, track, factor, eps, relu):
    y, *saved = _lib.native().batch_norm_pass(x, weight, bias, running_mean, running_var, counter, use_batch_stats, track,
                                              factor, eps, relu, residual)
    ctx.save_for_backward(*saved, y if residual is not None and relu else None)
    dtypes = [torch.float32 if p is None else p.dtype for p in (weight, bias)]
    ctx.how = (relu, use_batch_stats, residual is not None, *dtypes)
    return y

  @staticmethod
  def backward(ctx, dy):
    grads = _lib.native().batch_norm_grads(dy, *ctx.saved_tensors, *ctx.how, ctx.needs_input_grad[:4])
    return (*grads,) + (None,) * 8


class BatchNormRelu1d(torch.nn.BatchNorm1d):
  """BatchNorm1d [+ ReLU] in one pass over (rows, C) inputs on the GPU.  Inputs the kernels do
  not take (3-D, channel counts that are not a multiple of 16 bytes, a single row, tensors
  that are not on the GPU) go through torch.nn.BatchNorm1d itself, followed by a ReLU."""

  def __init__(self, num_features: int, relu: bool = False, **kwargs):
    super().__init__(num_features, **kwargs)
    self.fused_relu = relu

  def forward(self, input: torch.Tensor, residual: torch.Tensor = None, relu: bool = None) -> torch.Tensor:
    """residual: added to the normalised values before the ReLU (the tail of a residual
    block), in the same pass.  relu: overrides the module's setting for this call."""
    relu = self.fused_relu if relu is None else relu
    if not (input.dim() == 2 and input.is_cuda and input.shape[0] > 1 and kernels_take(input.dtype, int(input.shape[1]))):
      out = super().forward(input)
      if residual is not None:
        out = out + residual
      return torch.relu(out) if relu else out
    # the bookkeeping of torch.nn.modules.batchnorm._BatchNorm.forward
    factor = 0.0 if self.momentum is None else self.momentum
    counter = None
    if self.training and self.track_running_stats and self.num_batches_tracked is not None:
      nbt = self.num_batches_tracked
      if (self.momentum is not None and nbt.is_cuda and nbt.dtype == torch.long and nbt.device == input.device):
        counter = nbt                        # counted by the statistics kernel: no launch of its own
      else:
        nbt.add_(1)
        factor = 1.0 / float(nbt) if self.momentum is None else self.momentum
    use_batch_stats = self.training or (self.running_mean is None and self.running_var is None)
    track = self.training and self.track_running_stats
    running = not use_batch_stats or track
    stats = (self.running_mean, self.running_var) if running else (None, None)
    how = (counter, use_batch_stats, track, factor if track else 0.0, self.eps, relu)
    if _lib.recorded():
      return _BatchNormFunction.apply(input, self.weight, self.bias, residual, *stats, *how)
    return _lib.native().batch_norm(input, self.weight, self.bias, *stats, *how, residual)

  def extra_repr(self) -> str:
    return super().extra_repr() + ', relu={}'.format(self.fused_relu)

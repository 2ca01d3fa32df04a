"""The passes of a layer on an octree are shared by the threads that use it (no GPU needed: the passes are
made, not run)."""

import threading

import torch

from ocnn_amd import _lib
from ocnn_amd.nn.octree_conv import _Layer


class _Engine:
  """Makes a new pass with every request; the data gradient's waits to be released."""
  in_shape, octree = (8, 32), None

  def __init__(self):
    self.entered, self.release, self.made = threading.Event(), threading.Event(), []

  def is_conv_layer(self): return True

  def forward_op(self, dtype, pad_to):
    return _lib.native().GatherOp(), torch.zeros(8, 27, dtype=torch.int32)

  def backward_op(self, dtype, index, rows):
    self.entered.set()
    assert self.release.wait(10)
    self.made.append(_lib.native().GatherOp())
    return self.made[-1], torch.ones(8, 27, dtype=torch.int32)

  def weight_op(self, dtype, out_transposed, index, rows):
    return _lib.native().WgradOp(), torch.zeros(8, 27, dtype=torch.int32)


def test_passes_made_by_several_threads():
  eng = _Engine()
  layer = _Layer(eng, torch.float16, False)
  held = layer.native                                    # what a running call holds, without the interpreter lock
  assert layer.ok and held.fwd is not None and held.dgrad is None
  threads = [threading.Thread(target=layer.make_dgrad, args=(lambda: eng,)) for _ in range(2)]
  threads += [threading.Thread(target=layer.make_wgrad, args=(lambda: eng,))]
  for t in threads:
    t.start()
  assert eng.entered.wait(10)
  assert layer.dgrad is None                             # not said to be there before it is
  eng.release.set()
  for t in threads:
    t.join(60)
  assert layer.dgrad and layer.wgrad and len(eng.made) == 1
  assert held.dgrad is None and held.wgrad is None       # never changed under a call
  now = layer.native
  assert now.fwd is held.fwd and now.dgrad is eng.made[0] and now.wgrad is not None
  assert int(now.dgrad_table.sum()) == 8 * 27 and not now.wgrad_of_grad

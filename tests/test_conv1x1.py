"""The gradients of modules.Conv1x1 on many fp32 rows for operands that its kernel cannot read: those of
torch.nn.Linear.  (Of the function itself no GPU is needed: none of them may reach the kernel.)"""

import pytest
import torch
import torch.autograd.forward_ad as fwAD

from ocnn_amd.modules import _RowsLinear32


def _layer(f, rows=40, cin=8, cout=6):
  g = torch.Generator().manual_seed(0)
  x, w, b = (torch.randn(*s, generator=g).requires_grad_() for s in ((rows, cin), (cout, cin), (cout,)))
  return f(x, w, b), (x, w, b), g


@pytest.mark.parametrize('kind', ['batch', 'batch_of_second', 'negated', 'zeros', 'dual', 'vmap'])
def test_gradients_the_kernel_cannot_read(kind):
  results = []
  for f in (torch.nn.functional.linear, _RowsLinear32.apply):
    y, params, g = _layer(f)
    many = torch.randn(5, *y.shape, generator=g)
    grads = lambda dy, **k: torch.autograd.grad(y, params, dy, retain_graph=True, **k)
    if kind == 'batch':
      results.append(grads(many, is_grads_batched=True))
    elif kind == 'batch_of_second':                      # (the gradient itself differentiable)
      dy = many.clone().requires_grad_()
      gw = grads(dy, is_grads_batched=True, create_graph=True)[1]
      results.append(torch.autograd.grad((gw * gw).sum(), (dy, params[0])))
    elif kind == 'negated':
      results.append(grads(torch._neg_view(many[0])))
    elif kind == 'zeros':
      results.append(grads(torch._efficientzerotensor(y.shape)))
    elif kind == 'dual':
      with fwAD.dual_level():
        got = grads(fwAD.make_dual(many[0], many[1]))
        results.append([t for p in got for t in fwAD.unpack_dual(p)])
    else:
      results.append(torch.func.vmap(grads)(many))
  for want, got in zip(*results):
    assert got.shape == want.shape and torch.allclose(got, want, rtol=1e-5, atol=1e-5)


@pytest.mark.gpu
def test_module_with_a_batch_of_gradients():
  from ocnn_amd.modules import Conv1x1
  layer = Conv1x1(32, 13, use_bias=True).to('cuda')
  x = torch.randn(4099, 32, device='cuda', generator=torch.Generator('cuda').manual_seed(1)).requires_grad_()
  many = torch.randn(3, 4099, 13, device='cuda', generator=torch.Generator('cuda').manual_seed(2))
  params = [x] + list(layer.parameters())
  y = layer(x)
  assert 'RowsLinear32' in type(y.grad_fn).__name__
  got = torch.autograd.grad(y, params, many, is_grads_batched=True)
  want = torch.autograd.grad(layer.linear(x), params, many, is_grads_batched=True)
  assert torch.equal(got[0], want[0]) and torch.equal(got[2], want[2])
  # (the product over the rows may run in another order: the bound of an fp32 sum against float64, a rounding of
  # 2^-24 of a partial sum in each of sqrt(rows) effective terms, eight of them)
  x64, many64 = x.detach().double(), many.double()
  bound = 8 * 2.0 ** -24 * (many64.abs().transpose(1, 2) @ x64.abs())
  assert ((got[1].double() - many64.transpose(1, 2).contiguous() @ x64).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize('training', [False, True])
def test_traces_keep_the_linear(training, tmp_path):
  """A trace of layers whose other operations can be saved can be saved, in training as in evaluation; no decision on
  the sizes is said to be baked into it."""
  import warnings
  from ocnn_amd.modules import Conv1x1
  net = torch.nn.Sequential(Conv1x1(32, 16), torch.nn.ReLU(), Conv1x1(16, 8, use_bias=True)).to('cuda').train(training)
  x = torch.randn(5000, 32, device='cuda', generator=torch.Generator('cuda').manual_seed(3)).requires_grad_()
  with warnings.catch_warnings():
    warnings.simplefilter('error', torch.jit.TracerWarning)
    traced = torch.jit.trace(net, (x,), check_trace=False)
  traced.save(str(tmp_path / 'net.pt'))
  again = torch.jit.load(str(tmp_path / 'net.pt'))
  assert torch.equal(again(x[:100]), net(x[:100]))
  (got,), (want,) = (torch.autograd.grad(m(x).sum(), x) for m in (again, net))
  assert torch.equal(got, want)

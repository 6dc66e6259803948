"""The recurrence's one-pass kernels (csrc/rg_scan_tiles.hip) at the edges of
their blocks, steps and channel slabs, against float64 loops over time."""

import pytest
import torch

import recurrentgemma_amd as rg
from recurrentgemma_amd import ops
from recurrentgemma_amd import training

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T,W", [
    (1, 1, 8), (2, 3, 64), (1, 4, 72), (2, 8, 64), (1, 255, 136), (2, 256, 64),
    (1, 257, 128), (2, 511, 64), (1, 512, 40), (3, 513, 200), (2, 1025, 64)])
@pytest.mark.parametrize("with_state", [False, True])
def test_plain_recurrence(dtype, B, T, W, with_state):
  g = torch.Generator().manual_seed(T)
  x = torch.randn(B, T, W, generator=g).to(dtype).to(DEV)
  a = (torch.rand(B, T, W, generator=g) * 0.3 + 0.7).to(dtype).to(DEV)
  r = torch.randn(B, T, W, generator=g).to(dtype).to(DEV)
  rh = torch.randn(B, W, generator=g).to(DEV)
  reset = (torch.rand(B, T, generator=g) < 0.04).to(DEV)
  h0 = torch.randn(B, W, generator=g).to(DEV) if with_state else None
  leaves = [t.clone().requires_grad_(True) for t in (x, a)]
  hs = h0.clone().requires_grad_(True) if with_state else None
  with training.differentiable():
    y, h = rg.rnn_scan(*leaves, reset, hs)
  ((y.float() * r.float()).sum() + (h * rh).sum()).backward()

  xd, ad = (t.double().requires_grad_(True) for t in (x, a))
  hd = h0.double().requires_grad_(True) if with_state else None
  s = hd if with_state else torch.zeros(B, W, dtype=torch.float64, device=DEV)
  ys = []
  for t in range(T):
    s = ad[:, t] * (~reset[:, t, None]) * s + xd[:, t]
    ys.append(s)
  yd = torch.stack(ys, 1)
  ((yd * r.double()).sum() + (s * rh.double()).sum()).backward()
  tol = 1e-5 if dtype == torch.float32 else 1e-2

  def near(got, want, what, tol=tol):
    err = (got.double() - want).abs().max().item()
    assert err <= tol * want.abs().max().item() + 1e-30, (what, err)

  near(y.detach(), yd.detach(), "y")
  near(h.detach(), s.detach(), "h_last", 1e-5)
  near(leaves[0].grad, xd.grad, "dx")
  # (da is the product with the rounded y)
  near(leaves[1].grad, ad.grad, "da", tol if dtype == torch.float32 else 2e-2)
  if with_state:
    near(hs.grad, hd.grad, "dh0", 1e-5)
  # run to run the same bits, and the inference call's
  y2, h2 = ops.linear_scan(x, a, reset, h0)
  assert torch.equal(y2, y) and torch.equal(h2, h)


def _gated(x, gate_x, gate_a, a_param):
  """y of the RG-LRU from pre-activations [W], in float64."""
  log_a = -8.0 * torch.sigmoid(gate_a) * torch.nn.functional.softplus(a_param)
  a, m = torch.exp(log_a), torch.sqrt(-torch.expm1(2 * log_a))
  state, ys = torch.zeros_like(x[:, 0]), []
  for t in range(x.shape[1]):
    xn = x[:, t] * torch.sigmoid(gate_x)
    state = a * state + m * xn if t else xn
    ys.append(state)
  return torch.stack(ys, 1)


def _layer(width, heads, gate_x, gate_a, softplus):
  """A float32 layer whose pre-activations are its biases."""
  layer = rg.RGLRU(width=width, num_heads=heads, device=DEV, dtype=torch.float32)
  with torch.no_grad():
    layer.a_param.fill_(softplus).expm1_().log_()
    for gate, bias in ((layer.input_gate, gate_x), (layer.a_gate, gate_a)):
      gate.w.zero_()
      gate.b.copy_(bias.view_as(gate.b))
  return layer


@pytest.mark.parametrize("low,high", [(-1, 1), (-6, -3), (-12, -8), (-25, -15), (3, 12)])
@pytest.mark.parametrize("native", [True, False])
def test_float32_gates_far_from_zero(low, high, native):
  """A sigmoid of float32 is as good where it is small as elsewhere: y and dx within
  2^-23 of their norm.  A term of y is x gate m, two products of 2^-24 each at most,
  and gate and m are off by about one unit in the last place, 2^-24 at most and half
  of that in the mean: together 2^-24 in the mean square.  (a is 0.02 here: nothing
  adds up over time.)"""
  B, T, W, heads = 3, 130, 512, 2
  g = torch.Generator(device=DEV).manual_seed(7)
  uniform = lambda lo, hi: lo + (hi - lo) * torch.rand(W, generator=g, device=DEV)
  gate_x, gate_a = uniform(low, high), uniform(-1, 1)
  layer = _layer(W, heads, gate_x, gate_a, 1.0)
  x = torch.randn(B, T, W, generator=g, device=DEV)
  dy = torch.randn(B, T, W, generator=g, device=DEV)
  pos = torch.arange(T, device=DEV, dtype=torch.int32).repeat(B, 1)
  xd = x.double().requires_grad_()
  want = _gated(xd, gate_x.double(), gate_a.double(), layer.a_param.detach().double())
  if native:
    x.requires_grad_()
    with training.differentiable():
      y, _ = layer(x, pos, return_cache=False)
    pairs = [(y, want)] + list(zip(torch.autograd.grad(y, x, dy),
                                   torch.autograd.grad(want, xd, dy.double())))
  else:  # a prompt pass by several launches
    x, pos, want = (t.repeat(6, 1, 1)[..., :T, :] if t.dim() == 3 else t.repeat(6, 1)
                    for t in (x, pos, want))
    y, _, _ = ops.recurrent_core(
        x, pos, None, None, layer.input_gate.w.detach(), layer.input_gate.b.detach(),
        layer.a_gate.w.detach(), layer.a_gate.b.detach(), layer.a_param.detach())
    pairs = [(y, want)]
  for got, exact in pairs:
    assert (got.double() - exact).norm() <= 2.0**-23 * exact.norm()


def test_float32_gates_beyond_range():
  """Pre-activations that saturate a gate, infinite ones among them, and NaN, which
  stays in its channel."""
  B, T, W = 2, 70, 256
  values = [float("inf"), 1e30, 200.0, 89.0, -89.0, -200.0, -1e30, -float("inf")]
  gate_x = torch.zeros(W, device=DEV)
  gate_x[:8] = torch.tensor(values)
  gate_a = torch.zeros(W, device=DEV)
  gate_a[8:16] = torch.tensor(values)
  gate_x[16], gate_a[17] = float("nan"), float("nan")
  layer = _layer(W, 1, gate_x, gate_a, 1.0)
  x = torch.randn(B, T, W, device=DEV)
  pos = torch.arange(T, device=DEV, dtype=torch.int32).repeat(B, 1)
  with training.differentiable():
    y, _ = layer(x, pos, return_cache=False)
  want = _gated(x.double(), gate_x.double(), gate_a.double(),
                layer.a_param.detach().double())
  assert bool(y[..., 16].isnan().all()) and bool(y[:, 1:, 17].isnan().all())
  keep = [c for c in range(W) if c not in (16, 17)]
  assert bool(torch.isfinite(y[..., keep]).all())
  # (e^-89 is below float32's normal numbers: 2^-126 of x)
  assert float((y.detach()[..., keep].double() - want[..., keep]).abs().max()) <= 1e-6


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T", [5, 257, 514])
def test_kinds_of_document_starts(dtype, T):
  """Positions of 32 and of 64 bits, only whole zeros of which are starts, rows that
  begin at any byte of a mask: the same outputs and gradients."""
  B, W, heads = 3, 256, 1
  g = torch.Generator(device=DEV).manual_seed(T)
  torch.manual_seed(T)
  layer = rg.RGLRU(width=W, num_heads=heads, device=DEV, dtype=dtype)
  x = torch.randn(B, T, W, generator=g, device=DEV).to(dtype).requires_grad_()
  dy = torch.randn(B, T, W, generator=g, device=DEV).to(dtype)
  starts = torch.rand(B, T, generator=g, device=DEV) < 0.1
  got = []
  for far in (7, 2**32, -2**32):
    kind = torch.int32 if far == 7 else torch.int64
    pos = torch.where(starts, 0, far).to(kind)
    with training.differentiable():
      y, _ = layer(x, pos, return_cache=False)
    got.append((y.detach(), *torch.autograd.grad(y, (x, *layer.parameters()), dy)))
  for other in got[1:]:
    assert all(torch.equal(a, b) for a, b in zip(got[0], other))

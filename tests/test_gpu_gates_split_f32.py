"""The float32 gate projections, what they give back to x and their weight
gradients on three bf16 pieces (csrc/rg_gates_split_f32.hip) against float64:
rows around the 128-row tiles, the 32-row steps of the weight gradients and the
edges of their row ranges; gradients down to float32's smallest normal numbers,
inputs up to its largest; infinities."""

import pytest
import torch

import recurrentgemma_amd as rg
from recurrentgemma_amd import training

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _layer(width, heads, seed):
  torch.manual_seed(seed)
  layer = rg.RGLRU(width=width, num_heads=heads, device=DEV,
                   dtype=torch.float32)
  with torch.no_grad():
    for q in (layer.input_gate.b, layer.a_gate.b):
      q.normal_(std=0.2)
  return layer


def _reference(layer, x, pos, dy, dtype):
  p = [q.detach().to(dtype).requires_grad_() for q in
       (layer.a_param, layer.input_gate.w, layer.input_gate.b, layer.a_gate.w,
        layer.a_gate.b)]
  x = x.detach().to(dtype).requires_grad_()
  h, bw, _ = p[1].shape
  xs = x.reshape(*x.shape[:-1], h, bw).transpose(1, 2)
  gates = [torch.sigmoid((xs @ w).transpose(1, 2).reshape(x.shape) +
                         b.reshape(-1)) for w, b in (p[1:3], p[3:5])]
  log_a = -8.0 * gates[1] * torch.nn.functional.softplus(p[0])
  start = (pos == 0)[..., None]
  a = torch.where(start, 0.0, torch.exp(log_a))
  mult = torch.where(start, 1.0, torch.sqrt(-torch.expm1(2 * log_a)))
  xn = x * gates[0] * mult
  state, ys = torch.zeros_like(x[:, 0]), []
  for t in range(x.shape[1]):
    state = a[:, t] * state + xn[:, t]
    ys.append(state)
  y = torch.stack(ys, 1)
  return y, torch.autograd.grad(y, [x] + p, dy.to(dtype))


def _run(layer, x, pos, dy):
  x = x.detach().requires_grad_()
  with training.differentiable():
    y, _ = layer(x, pos, return_cache=False)
    p = (layer.a_param, layer.input_gate.w, layer.input_gate.b, layer.a_gate.w,
         layer.a_gate.b)
    return y, torch.autograd.grad(y, (x,) + p, dy)


@pytest.mark.parametrize("B,T,heads", [
    (1, 1, 1), (1, 15, 2), (1, 16, 1), (1, 33, 3), (1, 127, 1), (1, 128, 2),
    (1, 129, 1), (3, 86, 2), (5, 103, 3), (9, 100, 1), (40, 33, 2)])
@pytest.mark.parametrize("scale", [1.0, 1e-12, 1e-35])
def test_products_against_float64(B, T, heads, scale):
  """Whole RG-LRU step: y and every gradient to 2e-6 of its norm.  A float32 sum
  of 256 products is off by 2e-7 of its norm at worst here (measured 9e-8 for y,
  1.1e-7 for dx, 2.8e-7 for dw at 8192 rows); the recurrence around it multiplies
  that by 1 / (1 - a) <= 10 or so.  Small gradients lose nothing: those of 1e-35 are
  1e-37 and less where the projections take them, float32's smallest 1.2e-38 (and
  their own last digits 1.4e-45)."""
  width = 256 * heads
  layer = _layer(width, heads, seed=B * T)
  x = torch.randn(B, T, width, device=DEV)
  dy = torch.randn(B, T, width, device=DEV) * scale
  pos = torch.arange(T, device=DEV, dtype=torch.int32).expand(B, T).contiguous()
  y, got = _run(layer, x, pos, dy)
  yr, want = _reference(layer, x, pos, dy, torch.float64)
  for g, w in zip((y,) + got, (yr,) + want):
    err = (g.double() - w).norm().item()
    # (one token: the recurrence gate has no gradient at all)
    assert err <= 2e-6 * w.norm().item() + 1e-30 * scale, (err, w.norm().item())


@pytest.mark.parametrize("value", [float("inf"), -float("inf"), 3.4e38, 1e38, 3e31,
                                   1e31])
def test_values_that_pieces_cannot_hold(value):
  """An infinity, and finite values whose nearest bf16 is one or whose products
  overflow: the projections are what float32 gives (gates at 0 or 1, everything
  else finite), in the tile it is in and not beside it."""
  B, T, heads = 1, 200, 2
  layer = _layer(512, heads, seed=5)
  x = torch.randn(B, T, 512, device=DEV)
  x[0, 40, 3] = value
  pos = torch.arange(T, device=DEV).expand(B, T).contiguous()
  dy = torch.randn(B, T, 512, device=DEV)
  y, got = _run(layer, x, pos, dy)
  yr, _ = _reference(layer, x, pos, dy, torch.float64)
  same = [c for c in range(512) if c != 3]
  assert torch.isfinite(y[..., same]).all()
  err = (y[..., same].double() - yr[..., same]).norm() / yr[..., same].norm()
  assert err.item() < 2e-6
  assert torch.equal(y[0, :40], _run(layer, x[:, :40].contiguous(),
                                     pos[:, :40].contiguous(),
                                     dy[:, :40].contiguous())[0][0])
  # the other head's gradients know nothing of it
  x2 = x.clone()
  x2[0, 40, 3] = 0.0
  _, clean = _run(layer, x2, pos, dy)
  assert torch.equal(got[0][..., 256:], clean[0][..., 256:])
  for g, c in zip(got[2:], clean[2:]):
    assert torch.equal(g[1], c[1])


def test_infinite_gradient_stays_in_its_head():
  B, T, heads = 2, 150, 2
  layer = _layer(512, heads, seed=6)
  x = torch.randn(B, T, 512, device=DEV)
  pos = torch.arange(T, device=DEV).expand(B, T).contiguous()
  dy = torch.randn(B, T, 512, device=DEV)
  _, clean = _run(layer, x, pos, dy)
  dy[1, 20, 7] = float("inf")
  _, got = _run(layer, x, pos, dy)
  assert not torch.isfinite(got[0][1, 20, :256]).all()
  assert torch.isfinite(got[0][1, 21:]).all()  # nothing flows forwards
  assert torch.equal(got[0][1, 21:], clean[0][1, 21:])
  assert torch.equal(got[0][0], clean[0][0])
  assert torch.equal(got[0][..., 256:], clean[0][..., 256:])
  for g, c in zip(got[2:], clean[2:]):
    assert torch.equal(g[1], c[1])

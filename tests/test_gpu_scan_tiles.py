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

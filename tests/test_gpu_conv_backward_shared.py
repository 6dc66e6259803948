"""The width-4 conv's backward with a chunk's rows shared by four, two and one waves
(csrc/rg_conv.hip) against float64: rows that end inside, at and behind a wave's
share of a chunk of 32, channels that do not fill the lanes."""

import pytest
import torch

from recurrentgemma_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# workgroups = chunks x blocks of 512 (float32 256) channels: up to 512 take four
# waves, up to 1024 two
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,T,W", [
    (1, 1, 8), (1, 7, 8), (1, 8, 72), (1, 9, 520), (2, 15, 264), (1, 25, 512),
    (3, 11, 1032), (1, 33, 8), (5, 13, 520), (2, 500, 4096), (7, 150, 2560),
    (9, 300, 2560), (3, 1400, 2560)])
def test_against_float64(dtype, B, T, W):
  g = torch.Generator(device=DEV).manual_seed(B * T + W)
  rn = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
  x, dout, w = rn(B, T, W), rn(B, T, W), rn(4, W)
  starts = torch.rand(B, T, generator=g, device=DEV) < 0.1
  starts[:, 0] = True
  at = torch.arange(T, device=DEV).expand(B, T)
  begin = torch.cummax(torch.where(starts, at, torch.zeros_like(at)), 1).values
  pos = (at - begin).to(torch.int32).contiguous()
  dx, dw, db = ops.conv1d_backward(dout, x, pos, w)

  xd, gd, wd = x.double(), dout.double(), w.double()
  want_x = torch.zeros_like(xd)
  want_w, size_w = torch.zeros(4, W, device=DEV).double(), torch.zeros(4, W, device=DEV)
  size_x = torch.zeros_like(xd)
  for tap in range(min(4, T)):  # w[3 - tap] meets x[t - tap]
    n = T - tap
    alive = (pos[:, tap:] >= tap)[..., None]
    gt = gd[:, tap:] * alive
    want_x[:, :n] += wd[3 - tap] * gt
    size_x[:, :n] += (wd[3 - tap] * gt).abs()
    want_w[3 - tap] = (gt * xd[:, :n]).sum((0, 1))
    size_w[3 - tap] = (gt * xd[:, :n]).abs().sum((0, 1))
  # dx: four products and sums in float32, stored in the type; dw and db: at most
  # M / 32 + 32 additions one after the other, each off by 2^-24 of what is there
  eps = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-24
  assert bool(((dx.double() - want_x).abs() <=
               eps * want_x.abs() + 4 * 2.0**-24 * size_x).all())
  steps = (B * T / 32 + 40) * 2.0**-24
  stored = eps if dw.dtype == torch.bfloat16 else 0.0
  assert bool(((dw.double() - want_w).abs() <=
               steps * size_w + stored * want_w.abs() + 1e-30).all())
  want_b = gd.sum((0, 1))
  assert bool(((db.double() - want_b).abs() <= steps * gd.abs().sum((0, 1)) +
               stored * want_b.abs() + 1e-30).all())


# chunks of 64 and 256 rows, whose starts are looked up 48 rows at a time
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,T,W", [(3, 6001, 8), (5, 20003, 8), (70000, 1, 8)])
def test_chunks_of_more_rows(dtype, B, T, W):
  test_against_float64(dtype, B, T, W)

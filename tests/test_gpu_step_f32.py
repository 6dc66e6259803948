"""The float32 decode step in one launch (csrc/rg_step_f32.hip) against the conv
step, gate GEMM and scan step that serve caches updated in place: the same bits."""

import pytest
import torch

from oracle import torch_ref as R
from recurrentgemma_amd import ops
from tests import helpers

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NAMES = ("conv_w", "conv_b", "w_x", "b_x", "w_a", "b_a", "a_param")


# rows at the edges of tiles of 8, 16 and 32 rows and of the rule between them
@pytest.mark.parametrize("B,H", [(1, 1), (7, 10), (8, 2), (9, 10), (16, 3),
                                 (17, 10), (33, 1), (48, 10), (49, 10),
                                 (100, 2), (203, 10)])
@pytest.mark.parametrize("joined", [False, True])
def test_one_launch_equals_three(B, H, joined):
  W = 256 * H
  p = R.make_params(W, H, torch.float32, seed=B + H, gate_bias_std=0.5)
  ws = [p[n].to(DEV) for n in NAMES]
  g = torch.Generator().manual_seed(B)
  x = torch.randn(B, 1, W, generator=g).to(DEV)
  gate = torch.randn(B, 1, W, generator=g).to(DEV) if joined else None
  conv = torch.randn(B, 3, W, generator=g).to(DEV)
  h = torch.randn(B, W, generator=g).to(DEV)
  pos = torch.randint(0, 3, (B, 1), generator=g)  # (a third are starts)
  pos = pos.to(DEV).to(torch.int32 if B % 2 else torch.int64)
  conv_before, h_before = conv.clone(), h.clone()
  y, h1, conv1 = ops.recurrent_step(x, pos, conv, h, *ws, False, gate)
  assert torch.equal(conv, conv_before) and torch.equal(h, h_before)
  want_y, want_h, want_conv = ops.recurrent_step(x, pos, conv, h, *ws, True, gate)
  assert want_h.data_ptr() == h.data_ptr()
  assert torch.equal(y, want_y) and torch.equal(h1, want_h)
  assert torch.equal(conv1, want_conv)


def test_nan_stays_in_its_row():
  B, H = 21, 2
  W = 256 * H
  p = R.make_params(W, H, torch.float32, seed=5, gate_bias_std=0.5)
  ws = [p[n].to(DEV) for n in NAMES]
  g = torch.Generator().manual_seed(6)
  x = torch.randn(B, 1, W, generator=g).to(DEV)
  conv, h = torch.randn(B, 3, W, generator=g).to(DEV), torch.randn(
      B, W, generator=g).to(DEV)
  pos = torch.full((B, 1), 9, device=DEV)
  clean = ops.recurrent_step(x, pos, conv, h, *ws)
  x[4, 0, ::7] = float("nan")
  got = ops.recurrent_step(x, pos, conv, h, *ws)
  others = [b for b in range(B) if b != 4]
  assert not torch.isfinite(got[0][4]).all()
  assert all(torch.equal(a[others], b[others]) for a, b in zip(clean, got))


def test_against_the_oracle():
  B, H = 19, 3
  W = 256 * H
  p = R.make_params(W, H, torch.float32, seed=8, gate_bias_std=0.5)
  g = torch.Generator().manual_seed(9)
  x = torch.randn(B, 6, W, generator=g)
  seg = torch.arange(6).expand(B, 6).clone()
  _, cache = R.recurrent_core(x[:, :5], seg[:, :5], p)
  want, after = R.recurrent_core(x[:, 5:], seg[:, 5:], p, cache)
  y, h, conv = ops.recurrent_step(
      x[:, 5:].contiguous().to(DEV), seg[:, 5:].contiguous().to(DEV),
      cache.conv1d_state.to(DEV), cache.rg_lru_state.to(DEV),
      *[p[n].to(DEV) for n in NAMES])
  assert helpers.max_rel(y, want) < 1e-5
  assert helpers.max_rel(h, after.rg_lru_state) < 1e-5
  assert torch.equal(conv.cpu(), after.conv1d_state)

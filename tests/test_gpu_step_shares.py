"""The decode step's kernel in every way it is dealt out over workgroups (rows
per tile, share of a head) against the one call that deals out differently:
in-place caches keep whole heads, separate outputs share a head among
workgroups.  Same arithmetic, same bits."""

import pytest
import torch

from oracle import torch_ref as R
from recurrentgemma_amd import ops
from tests import helpers

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# rows either side of the lines: a quarter of a head x 8 rows up to 6 tiles of
# 8 at 10 heads, x 16 rows up to 6 tiles of 16, half a head up to 12 tiles of
# 16; whole heads x 8 rows up to 25 tiles of 8, x 16 rows, x 32 rows above
@pytest.mark.parametrize("B", [1, 7, 8, 9, 48, 49, 96, 97, 192, 193, 200, 201,
                               256, 805])
@pytest.mark.parametrize("joined", [False, True])
def test_step_is_the_same_however_it_is_dealt_out(B, joined):
  W, H = 2560, 10
  p = R.make_params(W, H, torch.bfloat16, seed=21, gate_bias_std=0.5)
  P = {k: v.to(DEV) for k, v in p.items()}
  g = torch.Generator().manual_seed(B)
  x = torch.randn(B, 1, W, generator=g).bfloat16()
  gate = torch.randn(B, 1, W, generator=g).bfloat16().to(DEV) if joined else None
  conv = torch.randn(B, 3, W, generator=g).bfloat16()
  h = torch.randn(B, W, generator=g)
  pos = torch.randint(0, 4, (B, 1), generator=g, dtype=torch.int32)
  weights = [P[n] for n in ("conv_w", "conv_b", "w_x", "b_x", "w_a", "b_a",
                            "a_param")]
  xd, posd, cd, hd = (t.to(DEV) for t in (x, pos, conv, h))
  apart = ops.recurrent_step(xd, posd, cd, hd, *weights, gate_branch=gate)
  assert torch.equal(cd.cpu(), conv) and torch.equal(hd.cpu(), h)
  ci, hi = cd.clone(), hd.clone()
  inside = ops.recurrent_step(xd, posd, ci, hi, *weights, in_place=True,
                              gate_branch=gate)
  assert inside[1].data_ptr() == hi.data_ptr()
  for a, b in zip(apart, inside):
    assert torch.equal(a, b)
  if not joined:
    xc, conv_o = R.widened_conv1d_forward(x, pos, p["conv_w"], p["conv_b"],
                                          cache=conv)
    yo, ho = R.widened_rglru_forward(xc, pos, p["a_param"], p["w_x"], p["b_x"],
                                     p["w_a"], p["b_a"], cache=h)
    assert helpers.max_rel(apart[0], yo) < 1e-2  # bf16 outputs
    assert helpers.max_rel(apart[1], ho) < 1e-2
    assert torch.equal(apart[2].cpu(), conv_o)

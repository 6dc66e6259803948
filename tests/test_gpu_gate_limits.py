"""Gate arithmetic of the single-launch prefill kernels at its limits: the
recurrence gate's exponent sigmoid(v) * decay where the decay underflows to
zero or is very large and the gate saturates either way."""

import pytest
import torch

from oracle import torch_ref as R
from recurrentgemma_amd import ops
from tests import helpers

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NAMES = ("conv_w", "conv_b", "w_x", "b_x", "w_a", "b_a", "a_param")


@pytest.mark.parametrize("bias", [-300.0, -60.0, 0.0, 60.0, 300.0])
@pytest.mark.parametrize("B,T,bw,H", [
    (2, 70, 176, 2),     # specialised waves
    (2, 70, 256, 2),     # slices
    (30, 200, 256, 10),  # whole heads
])
def test_decay_and_gate_limits(B, T, bw, H, bias):
  """a_param from -300 (softplus 0: a = 1, the state takes nothing in) to 60,
  but none whose a falls between the two float32 next to 1, where 1 - a^2 is
  noise; each against the widened oracle, all values finite.  y: the conv output
  and y itself are rounded to bf16 and may each land on a neighbour, 2^-7 of the
  value at most."""
  W = bw * H
  p = R.make_params(W, H, torch.bfloat16, seed=51, gate_bias_std=0.4)
  levels = torch.tensor([-300.0, -104.0, -88.0, -8.0, 0.0, 5.0, 60.0])
  p["a_param"] = levels[torch.arange(W) % 7].bfloat16()
  p["b_a"] = torch.full_like(p["b_a"], bias)
  g = torch.Generator().manual_seed(52)
  x = torch.randn(B, T, W, generator=g).bfloat16()
  seg = helpers.document_positions(B, T, 60, seed=53)
  y, h, _ = ops.recurrent_core(x.to(DEV), seg.to(DEV),
                               *[p[n].to(DEV) for n in NAMES])
  assert torch.isfinite(y.float()).all() and torch.isfinite(h).all()
  rows = slice(0, 2)  # (the oracle walks token by token)
  yo, co = R.widened_recurrent_core(x[rows], seg[rows], p, None)
  assert helpers.max_rel(y[rows], yo) < 2 * 2.0 ** -7
  assert helpers.max_rel(h[rows], co.rg_lru_state) < 2e-3

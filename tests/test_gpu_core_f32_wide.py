"""rg_recurrent_core in float32 with 256-wide heads by several launches (conv, gate
projections on bf16 pieces, recurrence): against the oracle around the tiles of
its kernels and on both sides of the lines that pick them."""

import pytest
import torch

from oracle import torch_ref as R
from recurrentgemma_amd import _lib
from recurrentgemma_amd import ops
from tests import helpers

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NAMES = ("conv_w", "conv_b", "w_x", "b_x", "w_a", "b_a", "a_param")


@pytest.mark.parametrize("B,T,H,mean_doc,joined,with_h0,with_conv", [
    # at most 32 pairs: one launch, which asks for no workspace
    (1, 1, 1, 0, True, True, True), (1, 2, 10, 0, False, False, True),
    (2, 31, 10, 7, True, True, True), (3, 64, 10, 20, False, True, False),
    (1, 257, 2, 60, True, False, True), (2, 700, 4, 100, False, True, True),
    # ... and several with the workspace that is brought, where they are ahead
    (1, 641, 1, 70, True, True, True), (2, 1041, 2, 0, False, True, True),
    (3, 401, 7, 100, True, False, True), (20, 513, 1, 60, False, True, False),
    (1, 2047, 10, 300, True, True, True),
    # more pairs: one-pass recurrence, and by the token
    (12, 64, 3, 15, True, True, True), (4, 130, 10, 50, False, False, True),
    (40, 33, 1, 10, True, False, True), (9, 45, 8, 0, False, True, True),
    (64, 9, 8, 4, True, True, False), (33, 300, 1, 80, True, False, True)])
def test_against_the_oracle(B, T, H, mean_doc, joined, with_h0, with_conv):
  """y and the state within 1e-5 of the largest magnitude (the float32 bar), conv
  state exact, every document's first rows included."""
  W = 256 * H
  lib = _lib.lib()
  best = lib.rg_recurrent_core_best_workspace_bytes(B, T, W, H, 0)
  several = (B, T, H) not in [(1, 1, 1), (1, 2, 10), (2, 31, 10), (3, 64, 10),
                              (1, 257, 2), (2, 700, 4)]
  assert best >= 2 * 4 * B * T * W if several else best == 0
  assert lib.rg_recurrent_core_workspace_bytes(B, T, W, H, 0) == (
      0 if B * H <= 32 else best)
  p = R.make_params(W, H, torch.float32, seed=T + H, gate_bias_std=0.3)
  P = {k: v.to(DEV) for k, v in p.items()}
  g = torch.Generator().manual_seed(B + T)
  x = torch.randn(B, T, W, generator=g)
  gate = torch.randn(B, T, W, generator=g) if joined else None
  seg = (helpers.document_positions(B, T, mean_doc, seed=T + 2) if mean_doc
         else torch.arange(T).repeat(B, 1))
  if B > 2:
    seg[1] -= min(5, T)  # left padding
    seg[1].clamp_(min=-1)
  h0 = torch.randn(B, W, generator=g) if with_h0 else None
  cw, cb = (P["conv_w"], P["conv_b"]) if with_conv else (None, None)
  y, h, c = ops.recurrent_core(
      x.to(DEV), seg.to(DEV), cw, cb, P["w_x"], P["b_x"], P["w_a"], P["b_a"],
      P["a_param"], h0=None if h0 is None else h0.to(DEV),
      gate_branch=None if gate is None else gate.to(DEV))
  if with_conv:
    xc, conv_state = R.conv1d_forward(x, seg, p["conv_w"], p["conv_b"])
    assert torch.equal(c.cpu(), conv_state)
  else:
    xc = x
  yo, ho = R.rglru_forward(xc, seg, p["a_param"], p["w_x"], p["b_x"], p["w_a"],
                           p["b_a"], cache=h0)
  if joined:
    yo = yo * torch.nn.functional.gelu(gate, approximate="tanh")
  assert torch.isfinite(y).all()
  assert helpers.max_rel(y, yo) < 1e-5
  assert helpers.max_rel(h, ho) < 1e-5


def test_join_inside_equals_the_pass_apart():
  B, T, W, H = 5, 300, 2048, 8
  p = R.make_params(W, H, torch.float32, seed=3, gate_bias_std=0.3)
  a = [p[n].to(DEV) for n in NAMES]
  x = torch.randn(B, T, W, device=DEV)
  gate = torch.randn(B, T, W, device=DEV)
  seg = torch.arange(T, device=DEV).repeat(B, 1)
  y, h, c = ops.recurrent_core(x, seg, *a)
  yj, hj, cj = ops.recurrent_core(x, seg, *a, gate_branch=gate)
  assert torch.equal(yj, ops.gelu_mul(y, gate))
  assert torch.equal(hj, h) and torch.equal(cj, c)


def test_rows_of_a_batch_stay_apart():
  """A row of NaN and a row with an infinity leave the other rows' bits alone."""
  B, T, W, H = 9, 70, 1024, 4
  p = R.make_params(W, H, torch.float32, seed=4, gate_bias_std=0.3)
  a = [p[n].to(DEV) for n in NAMES]
  x = torch.randn(B, T, W, device=DEV)
  seg = torch.arange(T, device=DEV).repeat(B, 1)
  y, h, _ = ops.recurrent_core(x, seg, *a)
  bad = x.clone()
  bad[3] = float("nan")
  bad[6, 10, 5] = float("inf")
  yb, hb, _ = ops.recurrent_core(bad, seg, *a)
  keep = [0, 1, 2, 4, 5, 7, 8]
  assert torch.equal(yb[keep], y[keep]) and torch.equal(hb[keep], h[keep])
  assert torch.isnan(yb[3]).all()

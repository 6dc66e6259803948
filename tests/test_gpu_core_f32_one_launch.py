"""rg_recurrent_core in float32 in one launch (256-wide heads, at most 32 pairs, no
workspace): around its tiles of 16 tokens, turns of 128 and segments of 512, at the
ends of the range of exponents, and with values that are not finite."""

import pytest
import torch

from oracle import torch_ref as R
from recurrentgemma_amd import _lib
from recurrentgemma_amd import ops
from tests import helpers

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NAMES = ("conv_w", "conv_b", "w_x", "b_x", "w_a", "b_a", "a_param")


def one_launch(x, seg, p, h0=None, gate=None, conv=True):
  lib = _lib.lib()
  B, T, W = x.shape
  H = p["w_x"].shape[0]
  assert lib.rg_recurrent_core_workspace_bytes(B, T, W, H, 0) == 0
  P = {k: p[k].to(DEV) for k in NAMES}
  x, seg = x.to(DEV), seg.to(DEV)
  h0 = None if h0 is None else h0.to(DEV)
  gate = None if gate is None else gate.to(DEV)
  y = torch.empty_like(x)
  h = torch.empty(B, W, device=DEV)
  c = torch.empty(B, 3, W, device=DEV)
  at = lambda t: None if t is None else t.data_ptr()
  _lib.check(lib.rg_recurrent_core(
      at(x), at(gate), at(seg), 1, at(P["conv_w"] if conv else None),
      at(P["conv_b"] if conv else None), at(P["w_x"]), at(P["b_x"]), at(P["w_a"]),
      at(P["b_a"]), None, at(P["a_param"]), at(h0), at(y), at(h),
      at(c if conv else None), None, 0, B, T, W, H, 0,
      torch.cuda.current_stream().cuda_stream))
  return y.cpu(), h.cpu(), c.cpu()


def wanted(x, seg, p, h0=None, gate=None, conv=True):
  state = None
  if conv:
    x, state = R.conv1d_forward(x, seg, p["conv_w"], p["conv_b"])
  y, h = R.rglru_forward(x, seg, p["a_param"], p["w_x"], p["b_x"], p["w_a"], p["b_a"],
                         cache=h0)
  if gate is not None:
    y = y * torch.nn.functional.gelu(gate, approximate="tanh")
  return y, h, state


@pytest.mark.parametrize("B,T,H,mean_doc,joined,with_h0,with_conv", [
    (1, 1, 1, 0, True, True, True), (1, 3, 2, 0, False, False, True),
    (2, 15, 3, 4, True, True, True), (1, 16, 1, 0, False, True, False),
    (3, 17, 2, 5, False, False, True), (1, 127, 10, 30, True, True, True),
    (2, 129, 1, 0, False, True, True), (32, 33, 1, 9, True, False, True),
    (1, 511, 2, 100, False, True, True), (1, 513, 3, 0, True, True, False),
    (2, 1041, 2, 200, True, True, True)])
def test_against_the_oracle(B, T, H, mean_doc, joined, with_h0, with_conv):
  """y and the state within 1e-5 of the largest magnitude (the float32 bar), conv
  state exact."""
  W = 256 * H
  p = R.make_params(W, H, torch.float32, seed=T + H, gate_bias_std=0.3)
  g = torch.Generator().manual_seed(B + T)
  x = torch.randn(B, T, W, generator=g)
  gate = torch.randn(B, T, W, generator=g) if joined else None
  seg = (helpers.document_positions(B, T, mean_doc, seed=T + 2) if mean_doc
         else torch.arange(T).repeat(B, 1))
  h0 = torch.randn(B, W, generator=g) if with_h0 else None
  y, h, c = one_launch(x, seg, p, h0, gate, with_conv)
  yo, ho, co = wanted(x, seg, p, h0, gate, with_conv)
  assert torch.isfinite(y).all()
  assert helpers.max_rel(y, yo) < 1e-5 and helpers.max_rel(h, ho) < 1e-5
  if with_conv:
    assert torch.equal(c, co)


@pytest.mark.parametrize("value", [float("inf"), -float("inf"), 3.3e38])
def test_a_value_whose_pieces_overflow(value):
  """An infinity (or a value whose first piece is one) in one channel: results are
  not finite exactly where the oracle's are not, others are close."""
  B, T, H = 1, 70, 2
  W = 256 * H
  p = R.make_params(W, H, torch.float32, seed=5, gate_bias_std=0.3)
  p["conv_w"][1:3] = 0.0
  g = torch.Generator().manual_seed(6)
  x = torch.randn(B, T, W, generator=g)
  x[0, 20, 300] = value
  # (weights whose products with it stay infinite or large: gates of 0 or 1)
  seg = torch.arange(T).repeat(B, 1)
  y, h, _ = one_launch(x, seg, p)
  yo, ho, _ = wanted(x, seg, p)
  assert torch.equal(torch.isnan(y), torch.isnan(yo))
  both = torch.isfinite(yo) & (yo.abs() < 1e6)
  assert both.any() and helpers.max_rel(y[both], yo[both]) < 1e-5
  assert torch.equal(torch.isinf(y), torch.isinf(yo))


@pytest.mark.parametrize("scale", [1e-30, 1e-34, 1e-36])
def test_small_inputs_keep_their_digits(scale):
  """Inputs whose last digits no bf16 piece can hold: y is as close to 64 bits as at
  ordinary sizes (the float32 bar; pieces put together again are off by 4e-6 at 1e-35
  and 3e-4 at 1e-37, which is where the conv takes 1e-36)."""
  B, T, H = 1, 70, 2
  W = 256 * H
  p = R.make_params(W, H, torch.float32, seed=9, gate_bias_std=0.3)
  p["conv_b"] = torch.zeros_like(p["conv_b"])
  g = torch.Generator().manual_seed(10)
  x = torch.randn(B, T, W, generator=g) * scale
  seg = torch.arange(T).repeat(B, 1)
  y, h, _ = one_launch(x, seg, p)
  yo, ho, _ = wanted(x.double(), seg, {k: v.double() for k, v in p.items()})
  got, want = (y.double() / scale, h.double() / scale), (yo / scale, ho / scale)
  assert all(helpers.max_rel(a, b) < 1e-5 for a, b in zip(got, want))


@pytest.mark.parametrize("B,T,H,several", [
    (1, 500, 10, False), (2, 300, 10, False), (1, 2048, 1, True), (2, 640, 10, True)])
def test_the_form_is_chosen_by_the_time_it_takes(B, T, H, several):
  """With a workspace, on either side of the line between one launch and several: the
  call has the bits of one launch just where it is one."""
  W = 256 * H
  p = R.make_params(W, H, torch.float32, seed=2, gate_bias_std=0.3)
  x = torch.randn(B, T, W, generator=torch.Generator().manual_seed(T))
  seg = torch.arange(T).repeat(B, 1)
  y, h, _ = one_launch(x, seg, p)
  got = ops.recurrent_core(x.to(DEV), seg.to(DEV), *[p[k].to(DEV) for k in NAMES])
  assert torch.equal(got[0].cpu(), y) != several
  assert helpers.max_rel(got[0], y) < 1e-5 and helpers.max_rel(got[1], h) < 1e-5

"""Prefill with the tiles of a row side by side (csrc/rg_prefill_short.hip): 256-wide
heads, at most 32 (row, head) pairs, 129 to 1000 tokens."""

import pytest
import torch

from oracle import torch_ref as R
from recurrentgemma_amd import _lib
from recurrentgemma_amd import ops
from tests import helpers

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NAMES = ("conv_w", "conv_b", "w_x", "b_x", "w_a", "b_a", "a_param")


def unpacked(x, seg, ws, h0, gate):
  """The C call without re-laid-out weights."""
  B, T, W = x.shape
  H = ws[2].shape[0]
  lib = _lib.lib()
  need = lib.rg_recurrent_core_workspace_bytes(B, T, W, H, 1)
  work = torch.empty(max(need, 1), dtype=torch.uint8, device=DEV)
  y, c = torch.empty_like(x), x.new_empty(B, 3, W) if ws[0] is not None else None
  h = torch.empty(B, W, dtype=torch.float32, device=DEV)
  ptr = lambda t: None if t is None else t.data_ptr()
  _lib.check(lib.rg_recurrent_core(
      ptr(x), ptr(gate), ptr(seg), int(seg.dtype == torch.int64),
      *[ptr(t) for t in ws[:6]], None, ptr(ws[6]), ptr(h0), ptr(y), ptr(h), ptr(c),
      ptr(work), need, B, T, W, H, 1, torch.cuda.current_stream().cuda_stream))
  return y, h, c


@pytest.mark.parametrize("B,T,H,mean_doc", [
    # edges of the tiles (16), the turns (128), the chunks of the scan (24), the
    # segments (384) and the range
    (1, 129, 1, 5), (3, 143, 2, 40), (1, 144, 10, 0), (2, 145, 16, -100),
    (1, 255, 3, 30), (1, 256, 1, 0), (5, 257, 2, 9), (1, 383, 2, 100),
    (3, 384, 10, 60), (1, 385, 4, 0), (32, 409, 1, 50), (2, 767, 3, -300),
    (1, 769, 10, 200), (1, 1000, 2, 0)])
@pytest.mark.parametrize("joined", [False, True])
def test_against_the_oracle(B, T, H, mean_doc, joined):
  """Outputs and state as close as the other forms are held, conv state exact; the join
  and weights as the reference lays them out: the same bits."""
  W = 256 * H
  p = R.make_params(W, H, torch.bfloat16, seed=21, gate_bias_std=0.4)
  ws = [p[n].to(DEV) for n in NAMES]
  g = torch.Generator().manual_seed(B + T)
  x = torch.randn(B, T, W, generator=g).bfloat16()
  gate = torch.randn(B, T, W, generator=g).bfloat16().to(DEV) if joined else None
  if mean_doc < 0:
    pads = torch.randint(0, min(T, -mean_doc) + 1, (B, 1), generator=g)
    seg = (torch.arange(T)[None] - pads).clamp(min=-1)
  elif mean_doc:
    seg = helpers.document_positions(B, T, mean_doc, seed=23)
  else:
    seg = torch.arange(T).repeat(B, 1)
  xd, sd = x.to(DEV), seg.to(DEV).to(torch.int32 if T % 2 else torch.int64)
  y, h, c = ops.recurrent_core(xd, sd, *ws)
  yo, co = R.widened_recurrent_core(x, seg, p, None)
  assert helpers.max_rel(y, yo) < 1e-2
  assert helpers.max_rel(h, co.rg_lru_state) < 2e-3
  assert torch.equal(c.cpu(), co.conv1d_state)
  if joined:
    yj, hj, cj = ops.recurrent_core(xd, sd, *ws, gate_branch=gate)
    assert torch.equal(yj, ops.gelu_mul(y, gate))
    assert torch.equal(hj, h) and torch.equal(cj, c)
    y = yj
  for a, b in zip(unpacked(xd, sd, ws, None, gate), (y, h, c)):
    assert torch.equal(a, b)


@pytest.mark.parametrize("B,T,H", [(1, 130, 2), (2, 500, 3), (1, 900, 1)])
def test_without_conv_and_from_a_state(B, T, H):
  """x as the conv output already, rows that go on from h0: the call with the conv
  inside, bit for bit, and its second half from the first half's state."""
  W = 256 * H
  p = R.make_params(W, H, torch.bfloat16, seed=31, gate_bias_std=0.4)
  ws = [p[n].to(DEV) for n in NAMES]
  x = torch.randn(B, T, W, generator=torch.Generator().manual_seed(T)).bfloat16().to(DEV)
  seg = helpers.document_positions(B, T, 60, seed=33).to(DEV)
  y, h, _ = ops.recurrent_core(x, seg, *ws)
  xc, _ = ops.conv1d_prefill(x, seg, ws[0], ws[1])
  bare = [None, None] + ws[2:]
  yc, hc, _ = ops.recurrent_core(xc, seg, *bare)
  assert torch.equal(yc, y) and torch.equal(hc, h)
  cut = T // 3
  _, before, _ = ops.recurrent_core(xc[:, :cut].contiguous(), seg[:, :cut].contiguous(),
                                    *bare)
  tail = xc[:, cut:].clone(), seg[:, cut:].clone()
  yt, ht, _ = ops.recurrent_core(*tail, *bare, h0=before)
  assert helpers.max_rel(yt, y[:, cut:]) < 1e-2 and helpers.max_rel(ht, h) < 2e-3
  assert all(torch.equal(a, b) for a, b in zip(
      unpacked(*tail, bare, before, None)[:2], (yt, ht)))


def test_rows_do_not_see_each_other():
  """A NaN or an infinity in one row leaves the others' bits as they are."""
  B, T, W, H = 3, 333, 2560, 10
  p = R.make_params(W, H, torch.bfloat16, seed=41, gate_bias_std=0.4)
  ws = [p[n].to(DEV) for n in NAMES]
  x = torch.randn(B, T, W, generator=torch.Generator().manual_seed(2)).bfloat16().to(DEV)
  seg = helpers.document_positions(B, T, 60, seed=43).to(DEV)
  clean = ops.recurrent_core(x, seg, *ws)
  for bad, value in enumerate((float("nan"), float("inf"), -float("inf"))):
    xb = x.clone()
    xb[bad, T // 3, ::5] = value
    others = [b for b in range(B) if b != bad]
    for a, b in zip(ops.recurrent_core(xb, seg, *ws), clean):
      assert torch.equal(a[others], b[others])

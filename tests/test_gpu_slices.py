"""Prefill with a head's channels in slices (csrc/rg_prefill_slices.hip): narrow
heads, few (row, head) pairs, rows of a few tokens."""

import pytest
import torch

from oracle import torch_ref as R
from recurrentgemma_amd import _lib
from recurrentgemma_amd import ops
from tests import helpers

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NAMES = ("conv_w", "conv_b", "w_x", "b_x", "w_a", "b_a", "a_param")


@pytest.mark.parametrize("B,T,bw,H,mean_doc", [
    # edges of the 32-token tiles, of a pass (64 or 128 tokens), one row
    (1, 1, 176, 2, 5), (1, 31, 256, 1, 5), (1, 32, 176, 1, 40),
    (1, 33, 256, 2, 7), (1, 64, 176, 2, 9), (1, 65, 176, 2, 30),
    (1, 128, 256, 1, 60), (1, 129, 256, 2, 3), (2, 97, 176, 3, 1000),
    # rows of a few tokens, several of them per workgroup and pass
    (7, 1, 256, 2, 2), (40, 5, 176, 32, 3), (33, 32, 256, 10, 12),
    (50, 33, 176, 32, 20), (48, 16, 256, 10, -5),
    # head widths between the presets': padding in k, in channels, in both
    (2, 70, 136, 2, 20), (2, 70, 168, 3, 20), (3, 150, 184, 2, 50),
    (3, 150, 200, 1, 50), (2, 70, 248, 3, 20),
    # narrow heads, two teams of waves: odd and even numbers of tiles, several rows per
    # workgroup, whole and cut last tiles
    (16, 33, 176, 32, 20), (12, 97, 176, 32, -50), (20, 64, 160, 32, 40),
    (9, 31, 176, 32, 6), (5, 193, 128, 60, 70),
    # long rows, left padding
    (2, 700, 176, 4, -200), (3, 333, 256, 10, 80),
    # 256-wide heads, rows longer than a pass: more than 32 pairs (fewer go to
    # rg_prefill_short.hip)
    (33, 129, 256, 1, 3), (4, 200, 256, 10, 40), (4, 333, 256, 10, -200),
    (17, 300, 256, 2, 1000)])
@pytest.mark.parametrize("joined", [False, True])
def test_prefill_in_slices(B, T, bw, H, mean_doc, joined):
  W = bw * H
  p = R.make_params(W, H, torch.bfloat16, seed=21, gate_bias_std=0.4)
  ws = [p[n].to(DEV) for n in NAMES]
  g = torch.Generator().manual_seed(22)
  x = torch.randn(B, T, W, generator=g).bfloat16()
  gate = torch.randn(B, T, W, generator=g).bfloat16().to(DEV)
  if mean_doc < 0:
    pads = torch.randint(0, min(T, -mean_doc) + 1, (B, 1), generator=g)
    seg = (torch.arange(T)[None] - pads).clamp(min=-1)
  else:
    seg = helpers.document_positions(B, T, mean_doc, seed=23)
  xd, sd = x.to(DEV), seg.to(DEV).to(torch.int32 if B % 2 else torch.int64)
  y, h, c = ops.recurrent_core(xd, sd, *ws)
  yo, co = R.widened_recurrent_core(x, seg, p, None)
  assert helpers.max_rel(y, yo) < 1e-2
  assert helpers.max_rel(h, co.rg_lru_state) < 2e-3
  assert torch.equal(c.cpu(), co.conv1d_state)
  if joined:  # the join inside the kernel: the separate pass, bit for bit
    yj, hj, cj = ops.recurrent_core(xd, sd, *ws, gate_branch=gate)
    assert torch.equal(yj, ops.gelu_mul(y, gate))
    assert torch.equal(hj, h) and torch.equal(cj, c)
  # a carried-in state: the row in two calls
  if T > 1 and mean_doc > 0:
    cut = T // 2
    tail = sd[:, cut:].contiguous()
    gates = ops.recurrent_core(xd[:, :cut].contiguous(),
                               sd[:, :cut].contiguous(), *ws)
    xc, _ = ops.conv1d_prefill(xd, sd, ws[0], ws[1])
    whole = ops.recurrent_core(xc, sd, None, None, *ws[2:])
    part = ops.recurrent_core(xc[:, cut:].contiguous(), tail, None, None,
                              *ws[2:], h0=gates[1])
    assert helpers.max_rel(whole[0], yo) < 1e-2
    assert helpers.max_rel(part[1], h) < 2e-3
    assert helpers.max_rel(part[0], y[:, cut:]) < 1e-2


@pytest.mark.parametrize("B,T,bw,H", [(3, 100, 176, 2), (2, 300, 256, 2),
                                      (5, 40, 200, 3), (4, 200, 256, 10),
                                      (33, 129, 256, 1), (5, 333, 256, 7),
                                      (8, 200, 256, 10)])
@pytest.mark.parametrize("joined", [False, True])
def test_slices_without_packed_weights(B, T, bw, H, joined):
  """w_packed == NULL: the weights fetched from the reference layout, same bits
  (2 rows of 300 tokens in 2 heads of 256: in rg_prefill_short.hip; 80 pairs of 200
  tokens: in slices only joined)."""
  W = bw * H
  p = R.make_params(W, H, torch.bfloat16, seed=31, gate_bias_std=0.4)
  ws = [p[n].to(DEV) for n in NAMES]
  g = torch.Generator().manual_seed(32)
  x = torch.randn(B, T, W, generator=g).bfloat16().to(DEV)
  seg = helpers.document_positions(B, T, 30, seed=33).to(DEV)
  gate = torch.randn(B, T, W, generator=g).bfloat16().to(DEV) if joined else None
  y1, h1, c1 = ops.recurrent_core(x, seg, *ws, gate_branch=gate)
  lib = _lib.lib()
  assert lib.rg_recurrent_core_workspace_bytes(B, T, W, H, 1) == 0
  y2, c2 = torch.empty_like(x), x.new_empty(B, 3, W)
  h2 = torch.empty(B, W, dtype=torch.float32, device=DEV)
  ptr = lambda t: t.data_ptr()
  _lib.check(lib.rg_recurrent_core(
      ptr(x), ptr(gate) if joined else None, ptr(seg), 1,
      *[ptr(t) for t in ws[:6]], None, ptr(ws[6]),
      None, ptr(y2), ptr(h2), ptr(c2), None, 0, B, T, W, H, 1,
      torch.cuda.current_stream().cuda_stream))
  assert torch.equal(y1, y2) and torch.equal(h1, h2) and torch.equal(c1, c2)
  yo, co = R.widened_recurrent_core(x.cpu(), seg.cpu(), p, None)
  if joined:
    yo = (yo.float() * torch.nn.functional.gelu(
        gate.cpu().float(), approximate="tanh").bfloat16().float()).bfloat16()
  assert helpers.max_rel(y2, yo) < 1e-2
  assert helpers.max_rel(h2, co.rg_lru_state) < 2e-3


def _core(x, seg, ws, h0=None, packed=True):
  """recurrent_core, or the same C call without re-laid-out weights."""
  if packed:
    return ops.recurrent_core(x, seg, *ws, h0=h0)
  B, T, W = x.shape
  H = ws[2].shape[0]
  lib = _lib.lib()
  assert lib.rg_recurrent_core_workspace_bytes(B, T, W, H, 1) == 0
  conv = ws[0] is not None
  y, c = torch.empty_like(x), x.new_empty(B, 3, W) if conv else None
  h = torch.empty(B, W, dtype=torch.float32, device=DEV)
  ptr = lambda t: None if t is None else t.data_ptr()
  _lib.check(lib.rg_recurrent_core(
      ptr(x), None, ptr(seg), 1, *[ptr(t) for t in ws[:6]], None, ptr(ws[6]),
      ptr(h0), ptr(y), ptr(h), ptr(c), None, 0, B, T, W, H, 1,
      torch.cuda.current_stream().cuda_stream))
  return y, h, c


@pytest.mark.parametrize("B,T,bw,H", [
    # several rows per workgroup, of one tile, a few and many; whole and cut
    # last tiles; passes that hold several rows, one, and the end of one and
    # the start of the next
    (8, 10, 256, 10), (8, 32, 256, 10), (8, 45, 256, 10), (8, 100, 256, 10),
    (8, 200, 256, 10), (7, 333, 256, 16), (8, 440, 256, 10), (3, 333, 256, 10),
    (9, 10, 176, 32), (9, 32, 176, 32), (8, 50, 176, 32), (7, 100, 176, 32),
    (8, 333, 176, 32), (6, 1000, 176, 32), (8, 70, 200, 12),
    # narrow heads of two teams: a row per tile, rows that end in either team's
    (9, 20, 160, 64), (8, 64, 176, 32), (7, 65, 176, 32), (6, 97, 176, 64)])
@pytest.mark.parametrize("packed", [True, False])
def test_rows_do_not_see_each_other(B, T, bw, H, packed):
  """A NaN or an infinity in one row's x or h0 leaves every other row's outputs
  as they are, bit for bit."""
  W = bw * H
  p = R.make_params(W, H, torch.bfloat16, seed=41, gate_bias_std=0.4)
  ws = [p[n].to(DEV) for n in NAMES]
  g = torch.Generator().manual_seed(42)
  x = torch.randn(B, T, W, generator=g).bfloat16().to(DEV)
  h0 = torch.randn(B, W, generator=g).to(DEV)
  seg = helpers.document_positions(B, T, 60, seed=43).to(DEV)
  seg[:, 0] = 7  # (rows go on from h0, and no start shields the first token)
  bare = [None, None] + ws[2:]
  clean = _core(x, seg, ws, packed=packed)
  carried = _core(x, seg, bare, h0, packed)
  assert all(torch.isfinite(t).all() for t in clean + carried[:2])
  for bad in range(B):
    value = (float("nan"), float("inf"), float("-inf"))[bad % 3]
    others = [b for b in range(B) if b != bad]
    xb, hb = x.clone(), h0.clone()
    xb[bad, T // 3, ::5] = value
    hb[bad, ::3] = value
    got = _core(xb, seg, ws, packed=packed)
    assert not torch.isfinite(got[0][bad]).all()
    for a, b in zip(got, clean):
      assert torch.equal(a[others], b[others]), (bad, value)
    got = _core(x, seg, bare, hb, packed)
    assert not torch.isfinite(got[1][bad]).all()
    for a, b in zip(got[:2], carried[:2]):
      assert torch.equal(a[others], b[others]), (bad, value, "h0")


# several whole rows to a tile: one token each, numbers that leave tokens of the tile
# over, the longest, last tiles with one row and with all, one tile and many
MANY = [(2, 1, 256, 1), (33, 1, 176, 2), (300, 1, 256, 10), (64, 3, 256, 10),
        (11, 5, 200, 3), (65, 9, 176, 32), (23, 11, 256, 2), (2, 16, 256, 2),
        (129, 16, 248, 3), (40, 15, 136, 4)]


@pytest.mark.parametrize("B,T,bw,H", MANY)
@pytest.mark.parametrize("mean_doc", [4, -9])
def test_rows_of_a_few_tokens(B, T, bw, H, mean_doc):
  test_prefill_in_slices(B, T, bw, H, mean_doc, True)


@pytest.mark.parametrize("B,T,bw,H", [(9, 1, 256, 2), (12, 3, 176, 4),
                                      (7, 16, 256, 10), (9, 7, 200, 3)])
def test_rows_of_a_few_tokens_do_not_see_each_other(B, T, bw, H):
  test_rows_do_not_see_each_other(B, T, bw, H, True)


# narrow heads, rows of two tiles: four tiles at once for up to 80 pairs, two teams beyond
@pytest.mark.parametrize("B,T,bw,H", [(1, 33, 136, 1), (1, 64, 176, 32), (5, 50, 176, 8),
                                      (40, 64, 136, 2), (81, 64, 136, 1)])
@pytest.mark.parametrize("joined", [False, True])
def test_rows_of_two_tiles(B, T, bw, H, joined):
  test_prefill_in_slices(B, T, bw, H, 20, joined)


# beyond 512 pairs: where the two calls without a conv (a whole row in one call, and its
# second half with a state) take less than several rows to a tile, and where they do not;
# five heads of three slices, whose pairs are launched in eights
@pytest.mark.parametrize("B,T,bw,H", [(600, 3, 136, 1), (600, 9, 136, 2),
                                      (300, 16, 136, 5), (103, 16, 200, 5)])
@pytest.mark.parametrize("joined", [False, True])
def test_many_rows_of_narrow_heads(B, T, bw, H, joined):
  test_prefill_in_slices(B, T, bw, H, 4, joined)

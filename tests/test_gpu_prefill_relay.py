"""rg_recurrent_core dealt out in blocks of 32 tokens (rg_prefill_relay.hip) against
the same call by whole rows or chunks (rg_recurrent_prefill) and the oracle."""

import pytest
import torch

from oracle import torch_ref as R
from recurrentgemma_amd import _lib
from recurrentgemma_amd import ops
from tests import helpers

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
NAMES = ("conv_w", "conv_b", "w_x", "b_x", "w_a", "b_a", "a_param")


def _case(B, T, H, mean_doc, joined, with_h0, with_conv=True, int64=False):
  W = 256 * H
  # the states between blocks, two words a channel: these shapes go by blocks
  assert (_lib.lib().rg_recurrent_core_best_workspace_bytes(B, T, W, H, 1) >=
          B * 2 * W * 8)
  p = R.make_params(W, H, torch.bfloat16, seed=T + H, gate_bias_std=0.3)
  args = [p[n].to(DEV) for n in NAMES]
  if not with_conv:
    args[0] = args[1] = None
  g = torch.Generator().manual_seed(B + T)
  x = torch.randn(B, T, W, generator=g).bfloat16()
  gate = torch.randn(B, T, W, generator=g).bfloat16() if joined else None
  seg = (helpers.document_positions(B, T, mean_doc, seed=T + 2) if mean_doc
         else torch.arange(T).repeat(B, 1))
  seg[1] = (seg[1] - 37).clamp(min=-1)  # left padding
  seg = seg.to(torch.int64 if int64 else torch.int32)
  h0 = torch.randn(B, W, generator=g) if with_h0 else None
  put = lambda t: None if t is None else t.to(DEV)
  return p, (x.to(DEV), seg.to(DEV), *args), dict(h0=put(h0), gate_branch=put(gate))


def _close(got, want, joined):
  """The state in front of a block is P h + H of the block before instead of that
  block's last token: 32 roundings of float32 in another order, each at most 2^-24 of
  the largest state, on both sides.  y is that rounded to bf16: where it lies on an
  edge one step further, 2^-7 of a value at the lower end of its binade.  The join
  multiplies that step by gelu (none of it is added: it is relative) and rounds once
  more, another step."""
  (y, h, c), (yw, hw, cw) = got, want
  assert (c is None and cw is None) or torch.equal(c, cw)
  top = float(hw.abs().max())
  assert float((h - hw).abs().max()) <= 64 * 2.0**-24 * top
  y, yw = y.float(), yw.float()
  step = (2 if joined else 1) * 2.0**-7
  reach = 8.0 if joined else 1.0  # of the gate branch's gelu
  over = ((y - yw).abs() - step * torch.maximum(y.abs(), yw.abs()) -
          reach * 64 * 2.0**-24 * top)
  assert float(over.max()) <= 0


@pytest.mark.parametrize("B,T,H,mean_doc,joined,with_h0,with_conv,int64", [
    (40, 1000, 1, 90, True, True, True, False),
    (40, 1024, 1, 0, True, False, True, True),
    (7, 1025, 6, 3, True, True, True, False),
    (60, 2000, 1, 300, False, True, True, True),
    (9, 1023, 10, 40, False, False, True, False),
    (96, 1056, 1, 0, False, True, False, False),
    (260, 385, 1, 30, True, False, True, False),
    (87, 447, 3, 0, False, True, True, True),
    (3, 1120, 16, 500, True, True, True, False)])
def test_blocks_against_rows(B, T, H, mean_doc, joined, with_h0, with_conv, int64):
  p, args, kw = _case(B, T, H, mean_doc, joined, with_h0, with_conv, int64)
  got = ops.recurrent_core(*args, **kw, return_conv_cache=with_conv)
  rows = list(args)
  if not with_conv:  # a conv that passes its input on
    rows[2] = torch.zeros(4, 256 * H, device=DEV, dtype=torch.bfloat16)
    rows[2][3] = 1
    rows[3] = torch.zeros(256 * H, device=DEV, dtype=torch.bfloat16)
  want = ops.recurrent_prefill(*rows, **kw, return_conv_cache=with_conv)
  _close(got, want, joined)
  again = ops.recurrent_core(*args, **kw, return_h=False, return_conv_cache=False)
  assert torch.equal(again[0], got[0])


def test_against_the_oracle():
  B, T, H = 40, 1000, 1
  p, args, kw = _case(B, T, H, 60, True, True)
  y, h, _ = ops.recurrent_core(*args, **kw)
  xc, _ = R.conv1d_forward(args[0].cpu(), args[1].cpu(), p["conv_w"], p["conv_b"])
  yo, ho = R.rglru_forward(xc, args[1].cpu(), p["a_param"], p["w_x"], p["b_x"],
                           p["w_a"], p["b_a"], cache=kw["h0"].cpu())
  yo = yo.float() * torch.nn.functional.gelu(kw["gate_branch"].cpu().float(),
                                             approximate="tanh")
  # bf16 gates and outputs: two roundings of 2^-9 and what sqrt(1 - a^2) makes of them
  assert helpers.max_rel(h.cpu(), ho) < 2e-2
  assert helpers.max_rel(y.cpu().float(), yo) < 3e-2


def test_halves_of_a_state_word_vouch_for_themselves():
  """Two lanes fetch a word, four bytes each: each half has to say by itself which
  block it is from.  The words a call leaves in its workspace, and the states in
  them: those that a call ends with whose rows end there."""
  B, T, H = 40, 1056, 1
  W = 256 * H
  _, (x, seg, cw, cb, wx, bx, wa, ba, ap), kw = _case(B, T, H, 90, True, False)
  lib = _lib.lib()
  packed = ops.packed_gate_weights(wx, wa)
  ends = {}
  for n in (T, 1024):
    xn, sn = x[:, :n].contiguous(), seg[:, :n].contiguous()
    gate = kw["gate_branch"][:, :n].contiguous()
    need = lib.rg_recurrent_core_best_workspace_bytes(B, n, W, H, 1)
    assert need >= B * 2 * W * 8
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    y, h = torch.empty_like(xn), torch.empty(B, W, device=DEV)
    ptr = lambda t: None if t is None else t.data_ptr()
    _lib.check(lib.rg_recurrent_core(
        *map(ptr, (xn, gate, sn)), 0, *map(ptr, (
            cw, cb, wx, bx, wa, ba, packed, ap, None, y, h, None, ws)), need, B, n, W,
        H, 1, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    ends[n] = h, ws[:B * 2 * W * 8].cpu().view(torch.int32).view(B, 2, W, 2)
  # 33 blocks: the last word is block 31's, the state behind 1024 tokens; the other
  # one is block 30's
  low, high = (ends[T][1][..., i].to(torch.int64) & 0xffffffff for i in range(2))
  for block in (31, 30):
    assert bool((low[:, block & 1] & 0xffff == block + 1).all())
    assert bool((high[:, block & 1] & 0xffff == block + 1).all())
  bits = (low[:, 1] & 0xffff0000) | high[:, 1] >> 16
  want = ends[1024][0].cpu().view(torch.int32).to(torch.int64) & 0xffffffff
  assert torch.equal(bits, want)


def test_rows_apart():
  """NaN and infinities in one row's input or state stay in that row."""
  _, args, kw = _case(40, 1000, 1, 90, True, True)
  clean = ops.recurrent_core(*args, **kw)
  args[0][3, 500] = float("nan")
  args[0][7, 31] = float("inf")
  kw["h0"][11] = float("nan")
  args[1][11] = torch.arange(1, 1001)  # (goes on from the state)
  y, h, _ = ops.recurrent_core(*args, **kw)
  rest = [b for b in range(40) if b not in (3, 7, 11)]
  assert torch.equal(y[rest], clean[0][rest]) and torch.equal(h[rest], clean[1][rest])
  assert bool(torch.isnan(y[3, 500]).any()) and bool(torch.isnan(h[11]).all())
  assert torch.equal(y[3, :497], clean[0][3, :497])


def test_captured_and_side_by_side():
  """Replays of a captured call and calls on two streams at once give what the
  eager call gives."""
  cases = [_case(40, 1000, 1, 90, True, True), _case(96, 1056, 1, 0, False, False)]
  want = [ops.recurrent_core(*a, **k) for _, a, k in cases]
  torch.cuda.synchronize()
  graph = torch.cuda.CUDAGraph()
  with torch.cuda.graph(graph):
    out = ops.recurrent_core(*cases[0][1], **cases[0][2])
  for _ in range(3):
    for t in out:
      t.zero_()
    graph.replay()
    torch.cuda.synchronize()
    assert all(torch.equal(t, w) for t, w in zip(out, want[0]))
    ops.recurrent_core(*cases[1][1], **cases[1][2])
  streams = [torch.cuda.Stream(), torch.cuda.Stream()]
  torch.cuda.synchronize()
  got = [[], []]
  for _ in range(4):
    for i, s in enumerate(streams):
      with torch.cuda.stream(s):
        got[i].append(ops.recurrent_core(*cases[i][1], **cases[i][2]))
  torch.cuda.synchronize()
  for i in range(2):
    for g in got[i]:
      assert all(torch.equal(t, w) for t, w in zip(g, want[i]))

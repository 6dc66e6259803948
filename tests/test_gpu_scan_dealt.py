"""The recurrence's one-pass kernels with their steps dealt out to the workgroups
(csrc/rg_scan_tiles.hip) against float64 loops over time: rows that end around the
steps of 256 and 512 tokens, slabs of channels that are not full, one slab to more
than there are CUs."""

import pytest
import torch

import recurrentgemma_amd as rg
from recurrentgemma_amd import _lib
from recurrentgemma_amd import ops
from recurrentgemma_amd import training
from tests import test_gpu_core_f32_wide as core_f32
from tests import test_gpu_scan_tiles as one_pass
from tests import test_gpu_training as trained

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF16, F32 = torch.bfloat16, torch.float32


def _dealt(B, T, W, dtype, *modes):
  """Whether the plain forward and backward, the gated ones are dealt out."""
  f = _lib.lib().rg_scan_deal_bytes
  return all(f(B, T, W, int(dtype == BF16), m) > 0 for m in modes)


# (tolerances: those of the undealt kernels, whose sums these are in the same order
# but for the state between two steps, which is P h + H instead of a chain's last)
@pytest.mark.parametrize("dtype,B,T,W", [
    (BF16, 1, 4096, 8), (BF16, 1, 4097, 72), (BF16, 3, 3841, 200),
    (BF16, 2, 4607, 2560), (BF16, 9, 3584, 2304), (F32, 1, 4352, 36),
    (F32, 2, 5119, 200), (F32, 1, 6145, 2560)])
@pytest.mark.parametrize("with_state", [False, True])
def test_plain_recurrence(dtype, B, T, W, with_state):
  assert _dealt(B, T, W, dtype, 0, 1) or W >= 2304 and _dealt(B, T, W, dtype, 1)
  one_pass.test_plain_recurrence(dtype, B, T, W, with_state)


@pytest.mark.parametrize("dtype,B,T,W,H", [
    (BF16, 1, 1537, 256, 1), (BF16, 2, 1791, 512, 2), (BF16, 3, 2048, 256, 1),
    (BF16, 2, 2049, 2560, 10), (F32, 1, 2304, 256, 1), (F32, 2, 2561, 512, 2),
    (F32, 3, 3071, 96, 3)])
def test_gated_recurrence(dtype, B, T, W, H):
  assert _dealt(B, T, W, dtype, 3)
  trained._rglru_against_float64(dtype, B, T, W, H, DEV)


@pytest.mark.parametrize("B,T,H,mean_doc,joined,with_h0,with_conv", [
    (1, 2049, 2, 200, True, True, True), (2, 2303, 1, 0, False, False, True),
    (1, 2560, 3, 60, True, False, False)])
def test_core_of_float32(B, T, H, mean_doc, joined, with_h0, with_conv):
  assert _dealt(B, T, 256 * H, F32, 2)
  core_f32.test_against_the_oracle(B, T, H, mean_doc, joined, with_h0, with_conv)


def _inputs(B, T, W, dtype, seed):
  g = torch.Generator(device=DEV).manual_seed(seed)
  x = torch.randn(B, T, W, generator=g, device=DEV).to(dtype)
  a = torch.sigmoid(torch.randn(B, T, W, generator=g, device=DEV) + 2).to(dtype)
  reset = torch.rand(B, T, generator=g, device=DEV) < 0.002
  return x, a, reset, torch.randn(B, W, generator=g, device=DEV)


def test_rows_apart_and_against_slabs():
  """A row's NaN and infinity stay in it; the others are what more rows, which go by
  the slab, make of them (their order of additions differs between steps: float32
  within 1e-6 of the largest)."""
  B, T, W = 2, 5000, 264
  x, a, reset, h0 = _inputs(B, T, W, F32, 1)
  assert _dealt(B, T, W, F32, 0)
  y, h = ops.linear_scan(x, a, reset, h0)
  many = [t.repeat(60, *[1] * (t.dim() - 1)) for t in (x, a, reset, h0)]
  assert not _dealt(60 * B, T, W, F32, 0)
  ym, hm = ops.linear_scan(*many)
  assert (y - ym[:B]).abs().max() <= 1e-6 * y.abs().max()
  assert (h - hm[:B]).abs().max() <= 1e-6 * h.abs().max()
  x[1, 700], x[1, 3] = float("nan"), float("inf")
  yn, hn = ops.linear_scan(x, a, reset, h0)
  assert torch.equal(yn[0], y[0]) and torch.equal(hn[0], h[0])
  assert torch.equal(yn[1, :3], y[1, :3]) and bool(yn[1, 700].isnan().all())


@pytest.mark.parametrize("dtype,B,T,W", [(BF16, 1, 8000, 512), (F32, 2, 6000, 1024),
                                         (F32, 1, 6145, 2560)])
def test_general_path_is_the_same_call(dtype, B, T, W):
  """Inputs that do not lie densely take the Python path, forward and backward: the
  same form of the call, the same bits."""
  x, a, reset, h0 = _inputs(B, T, W, dtype, 4)
  dy = torch.randn_like(x)
  assert _dealt(B, T, W, dtype, 0, 1)
  leaves = [t.clone().requires_grad_() for t in (x, a, h0)]
  with training.differentiable():
    y, h = rg.rnn_scan(leaves[0], leaves[1], reset, leaves[2])
  grads = torch.autograd.grad(y, leaves, dy)
  wide = torch.empty(B, T, 2 * W, device=DEV, dtype=dtype)[..., :W]
  yg, hg = ops.linear_scan(wide.copy_(x), a, reset, h0)
  assert torch.equal(yg, y) and torch.equal(hg, h)
  got = ops.linear_scan_backward(dy, a, reset, y.detach(), h0)
  assert all(torch.equal(g, w) for g, w in zip(got, grads))


def test_captured_and_side_by_side():
  """Replays of a captured call and calls on two streams at once give the eager
  call's bits."""
  cases = [_inputs(1, 8000, 512, BF16, 2), _inputs(2, 6000, 1024, F32, 3)]
  assert all(_dealt(*c[0].shape, c[0].dtype, 0) for c in cases)
  want = [ops.linear_scan(*c) for c in cases]
  torch.cuda.synchronize()
  graph = torch.cuda.CUDAGraph()
  with torch.cuda.graph(graph):
    out = ops.linear_scan(*cases[0])
  for _ in range(3):
    for t in out:
      t.zero_()
    graph.replay()
    torch.cuda.synchronize()
    assert all(torch.equal(t, w) for t, w in zip(out, want[0]))
    ops.linear_scan(*cases[1])
  streams = [torch.cuda.Stream(), torch.cuda.Stream()]
  torch.cuda.synchronize()
  got = [[], []]
  for _ in range(4):
    for i, s in enumerate(streams):
      with torch.cuda.stream(s):
        got[i].append(ops.linear_scan(*cases[i]))
  torch.cuda.synchronize()
  for i in range(2):
    assert all(torch.equal(t, w) for g in got[i] for t, w in zip(g, want[i]))

"""A recurrent block's decode step in place, its conv state copied beside the linear
layers in front (rg_linear_rows_beside): the bits of the step that returns new caches."""

import pytest
import torch

from recurrentgemma_amd import _lib
from recurrentgemma_amd import modules
from recurrentgemma_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def block_of(width, heads):
  torch.manual_seed(width + heads)
  return modules.RecurrentBlock(width=width, num_heads=heads, lru_width=width,
                                device=DEV, dtype=torch.bfloat16).eval()


@pytest.mark.parametrize("B,width,heads", [
    # shares of a head by the number of rows, one and two tiles a workgroup of the
    # layers (2 x 6400 rows), copies shorter and longer than a turn of the copiers
    (1, 256, 1), (7, 2560, 10), (16, 2560, 10), (17, 2560, 10), (33, 1024, 4),
    (64, 2560, 10), (64, 6400, 25)])
def test_in_place_equals_new_caches(B, width, heads):
  block = block_of(width, heads)
  g = torch.Generator().manual_seed(B)
  xs = torch.randn(4, B, 1, width, generator=g).bfloat16().to(DEV)
  cache = modules.RecurrentBlockCache(
      rg_lru_state=torch.randn(B, width, generator=g).to(DEV),
      conv1d_state=torch.randn(B, 3, width, generator=g).bfloat16().to(DEV))
  own = modules.RecurrentBlockCache(*[t.clone() for t in cache])
  kept = tuple(own)
  seg = torch.full((B, 1), 9, device=DEV)
  seg[::3] = 0  # (a document starts at the second step)
  with torch.no_grad():
    for i, x in enumerate(xs):
      pos = seg if i == 1 else torch.full_like(seg, 9 + i)
      block.decode_in_place = False
      y, cache = block(x, pos, cache)
      block.decode_in_place = True
      # (defer_out: the path of the chained blocks; partial sums or the output)
      out, own = block(x, pos, own, defer_out=True)
      if isinstance(out, ops.PartialSums):
        out = out.sums.sum(0) + (0 if out.bias is None else out.bias.float())
        want = y.reshape(out.shape).float()
        # float32 sums of the same products, one side rounded to bf16
        assert (out - want).abs().max() <= 2.0 ** -8 * want.abs().max()
      else:
        assert torch.equal(out, y)
      assert all(torch.equal(a, b) for a, b in zip(own, cache))
      assert all(a.data_ptr() == b.data_ptr() for a, b in zip(own, kept))


def test_captured_steps():
  """Replays of a captured step on fixed buffers, eager work in between."""
  B, width, heads = 16, 2560, 10
  block = block_of(width, heads)
  block.decode_in_place = True
  cache = block.init_cache(B, width, torch.bfloat16, device=DEV)
  other = modules.RecurrentBlockCache(*[t.clone() for t in cache])
  x = torch.zeros(B, 1, width, dtype=torch.bfloat16, device=DEV)
  seg = torch.full((B, 1), 5, device=DEV)
  with torch.no_grad():
    block(x, seg, modules.RecurrentBlockCache(*[t.clone() for t in cache]),
          defer_out=True)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
      block(x, seg, cache, defer_out=True)
    for i in range(4):
      x.copy_(torch.randn(B, 1, width, generator=torch.Generator().manual_seed(i)))
      graph.replay()
      block.decode_in_place = False
      _, other = block(x, seg, other)
      block.decode_in_place = True
      assert all(torch.equal(a, b) for a, b in zip(cache, other))


def test_refusals():
  lib = _lib.lib()
  x = torch.zeros(4, 256, dtype=torch.bfloat16, device=DEV)
  w = torch.zeros(512 * 256, dtype=torch.bfloat16, device=DEV)
  out = torch.zeros(2, 4, 256, dtype=torch.bfloat16, device=DEV)
  state = torch.zeros(64, dtype=torch.bfloat16, device=DEV)
  to = torch.zeros_like(state)
  s = torch.cuda.current_stream().cuda_stream
  call = lambda M=4, K=256, N=512, frm=state, dst=to, n=128: lib.rg_linear_rows_beside(
      x.data_ptr(), w.data_ptr(), None, out.data_ptr(), M, K, N, 2, frm.data_ptr(),
      dst.data_ptr(), n, s)
  assert call() == 0
  assert call(M=65) != 0 and call(K=100) != 0 and call(n=24) != 0 and call(n=0) != 0
  assert call(K=5120, N=2560) != 0  # (its K is split)
  assert call(frm=state, dst=state) != 0 and call(dst=out) != 0

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


def noted(block, monkeypatch):
  """Per call of the layers with a copy beside them: whether it was made."""
  made, beside = [], block._rows_yx.beside

  def call(x, weights, biases, state):
    done = beside(x, weights, biases, state)
    made.append(done is not None)
    return done

  monkeypatch.setattr(block._rows_yx, "beside", call, raising=False)
  return made


@pytest.mark.parametrize("B,width,heads", [
    # shares of a head by the number of rows, one and two tiles a workgroup of the
    # layers (2 x 6400 rows), copies shorter and longer than a turn of the copiers
    (1, 256, 1), (7, 2560, 10), (16, 2560, 10), (17, 2560, 10), (33, 1024, 4),
    (64, 2560, 10), (64, 6400, 25)])
def test_in_place_equals_new_caches(B, width, heads, monkeypatch):
  block = block_of(width, heads)
  g = torch.Generator().manual_seed(B)
  xs = torch.randn(4, B, 1, width, generator=g).bfloat16().to(DEV)
  cache = modules.RecurrentBlockCache(
      rg_lru_state=torch.randn(B, width, generator=g).to(DEV),
      conv1d_state=torch.randn(B, 3, width, generator=g).bfloat16().to(DEV))
  own = modules.RecurrentBlockCache(*[t.clone() for t in cache])
  kept = tuple(own)
  copies = noted(block, monkeypatch)
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
  # (the layers' weights are packed by the first step, of either kind)
  assert copies == [True] * 4


def test_captured_steps(monkeypatch):
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
    copies = noted(block, monkeypatch)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
      block(x, seg, cache, defer_out=True)
    assert copies == [True]
    for i in range(4):
      x.copy_(torch.randn(B, 1, width, generator=torch.Generator().manual_seed(i)))
      graph.replay()
      block.decode_in_place = False
      _, other = block(x, seg, other)
      block.decode_in_place = True
      assert all(torch.equal(a, b) for a, b in zip(cache, other))


@pytest.mark.parametrize("M", [1, 16, 17, 64])
@pytest.mark.parametrize("N,bias", [(512, True), (12800, False)])
@pytest.mark.parametrize("items", [1, 255, 16 * 512 - 1, 16 * 512, 16 * 512 + 1, 100_000])
def test_copy_and_layers(M, N, bias, items):
  """The copy, 16 bytes an item, is the state, with nothing written behind it, below, at
  and above one turn of the 16 workgroups of 512 threads that make it; the layers' output
  has the bits of the call without a copy."""
  K, lib = 256, _lib.lib()
  g = torch.Generator(device=DEV).manual_seed(items + M)
  normal = lambda *shape: torch.randn(shape, generator=g, device=DEV).bfloat16()
  x, w, b = normal(M, K), normal(N, K), normal(N)
  s = torch.cuda.current_stream().cuda_stream
  packed = torch.empty(lib.rg_linear_packed_bytes(N, K, 0), dtype=torch.uint8, device=DEV)
  _lib.check(lib.rg_linear_pack(w.data_ptr(), 0, 1, 0, packed.data_ptr(), N, K, s))
  state = torch.randint(0, 256, (16 * items,), generator=g, device=DEV, dtype=torch.uint8)
  to = torch.full((16 * items + 4096,), 77, dtype=torch.uint8, device=DEV)
  out, alone = (torch.full((M * N + 4096,), 7.0, dtype=torch.bfloat16, device=DEV)
                for _ in range(2))
  bias = b.data_ptr() if bias else None
  _lib.check(lib.rg_linear_rows_beside(
      x.data_ptr(), packed.data_ptr(), bias, out.data_ptr(), M, K, N, 2,
      state.data_ptr(), to.data_ptr(), 16 * items, s))
  _lib.check(lib.rg_linear_rows(
      x.data_ptr(), packed.data_ptr(), bias, None, alone.data_ptr(), None, 0, M, K, N, 2,
      0, s))
  assert torch.equal(to[:16 * items], state) and (to[16 * items:] == 77).all()
  assert torch.equal(out, alone) and (out[M * N:] == 7.0).all()


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

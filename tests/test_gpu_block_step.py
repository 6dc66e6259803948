"""RecurrentBlock's cached single-token call as one native call (block_step of
csrc/host_ops.cpp) against its separate calls, bit for bit, and what it leaves to
them."""

import pytest
import torch

import recurrentgemma_amd as rg

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _block(width=512, heads=2, lru_width=None, dtype=torch.bfloat16, seed=0):
  torch.manual_seed(seed)
  block = rg.RecurrentBlock(width=width, num_heads=heads, lru_width=lru_width,
                            device=DEV, dtype=dtype)
  with torch.no_grad():
    for name, q in block.named_parameters():
      if name.endswith("bias") or name.endswith(".b"):
        q.normal_(std=0.1)
  return block


def _inputs(B, block, dtype=torch.bfloat16, seed=1):
  g = torch.Generator(device=DEV).manual_seed(seed)
  rn = lambda *s: torch.randn(*s, generator=g, device=DEV)
  W = block.lru_width
  pos = torch.randint(0, 3, (B, 1), generator=g, device=DEV)
  return (rn(B, 1, block.width).to(dtype), pos, rg.RecurrentBlockCache(
      rg_lru_state=rn(B, W), conv1d_state=rn(B, 3, W).to(dtype)))


def _both(block, x, pos, cache, monkeypatch):
  block(x, pos, cache)  # (packs the weights)
  native = block._step_natively(x, pos, cache)
  got = block(x, pos, cache)
  with monkeypatch.context() as m:
    m.setattr(rg.RecurrentBlock, "_step_natively", lambda *a: None)
    want = block(x, pos, cache)
  for a, b in ((got[0], want[0]),
               (got[1].rg_lru_state, want[1].rg_lru_state),
               (got[1].conv1d_state, want[1].conv1d_state)):
    assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b)
  return native is not None


@pytest.mark.parametrize("B", [1, 8, 9, 33, 64])
@pytest.mark.parametrize("lru_width,heads", [(512, 2), (1024, 4)])
@pytest.mark.parametrize("pos_dtype", [torch.int32, torch.int64])
def test_equals_the_separate_calls(B, lru_width, heads, pos_dtype, monkeypatch):
  block = _block(lru_width=lru_width, heads=heads)
  x, pos, cache = _inputs(B, block)
  assert _both(block, x, pos.to(pos_dtype), cache, monkeypatch)


def test_left_to_the_separate_calls(monkeypatch):
  block = _block()
  x, pos, cache = _inputs(65, block)  # too many rows
  assert not _both(block, x, pos, cache, monkeypatch)
  x, pos, cache = _inputs(4, block)
  wide = torch.zeros(4, 1, 1024, device=DEV, dtype=torch.bfloat16)
  wide[..., ::2] = x
  assert not _both(block, wide[..., ::2], pos, cache, monkeypatch)  # strides
  block = _block(width=384, heads=3)  # 128-wide heads
  x, pos, cache = _inputs(4, block)
  assert not _both(block, x, pos, cache, monkeypatch)
  block = _block(dtype=torch.float32)
  x, pos, cache = _inputs(4, block, torch.float32)
  assert not _both(block, x, pos, cache, monkeypatch)


def test_weights_written_to_and_replaced(monkeypatch):
  block = _block()
  x, pos, cache = _inputs(3, block)
  assert _both(block, x, pos, cache, monkeypatch)
  before = block(x, pos, cache)[0]
  with torch.no_grad():
    for layer, name in ((block.linear_x, "weight"), (block.linear_out, "bias"),
                        (block.rg_lru.a_gate, "w"), (block.conv_1d, "w")):
      getattr(layer, name).mul_(1.5)
      # (the first call after a write lays the weights out anew)
      after = block(x, pos, cache)[0]
      assert not torch.equal(before, after)
      before = after
      assert _both(block, x, pos, cache, monkeypatch)
  block.linear_y = torch.nn.Linear(512, 512, device=DEV, dtype=torch.bfloat16)
  assert not torch.equal(before, block(x, pos, cache)[0])
  assert _both(block, x, pos, cache, monkeypatch)


def test_in_place_and_wrong_sizes():
  block = _block()
  x, pos, cache = _inputs(2, block)
  want, new = block(x, pos, cache)
  want, new = block(x, pos, cache)
  block.decode_in_place = True
  got, same = block(x, pos, cache)
  assert torch.equal(got, want)
  assert same.rg_lru_state is cache.rg_lru_state
  assert torch.equal(cache.rg_lru_state, new.rg_lru_state)
  assert torch.equal(cache.conv1d_state, new.conv1d_state)
  block.decode_in_place = False
  with pytest.raises(AssertionError):
    block(x, pos, rg.RecurrentBlockCache(
        rg_lru_state=cache.rg_lru_state[:1], conv1d_state=cache.conv1d_state[:1]))

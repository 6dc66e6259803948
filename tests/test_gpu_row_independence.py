"""Sequences of a batch do not see each other: a NaN or an infinity in one row
leaves every other row's results as they are, bit for bit.  (The prefill forms
that give a workgroup several rows have theirs in test_gpu_slices.py.)"""

import pytest
import torch

import recurrentgemma_amd as rg
from recurrentgemma_amd import ops
from recurrentgemma_amd import training

pytestmark = pytest.mark.gpu
BF16, F32 = torch.bfloat16, torch.float32


def check(call, inputs, rows):
  """call(*inputs) -> tensors with the batch first; every input's row is spoilt."""
  clean = call(*[t.clone() for t in inputs])
  assert all(torch.isfinite(t).all() for t in clean)
  for bad in {0, rows // 2, rows - 1}:
    spoilt = [t.clone() for t in inputs]
    for i, t in enumerate(spoilt):
      t[bad].view(-1)[i::7] = float("nan") if bad % 2 else float("inf")
    got = call(*spoilt)
    others = [b for b in range(rows) if b != bad]
    for a, b in zip(got, clean):
      assert not torch.isfinite(a[bad]).all()
      assert torch.equal(a[others], b[others]), bad


def block_of(width, heads, dtype):
  torch.manual_seed(3)
  return rg.RecurrentBlock(width=width, num_heads=heads, device="cuda",
                           dtype=dtype)


def normal(*shape, dtype=BF16):
  return torch.randn(shape, device="cuda").to(dtype)


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("B", [2, 9, 40])
@pytest.mark.parametrize("in_place", [False, True])
def test_decode_step(B, dtype, in_place):
  block = block_of(512, 2, dtype)
  block.decode_in_place = in_place
  pos = torch.full((B, 1), 9, device="cuda")

  @torch.no_grad()
  def call(x, conv, h):
    y, cache = block(x, pos, rg.RecurrentBlockCache(h, conv))
    return y, cache.rg_lru_state, cache.conv1d_state

  check(call, [normal(B, 1, 512, dtype=dtype), normal(B, 3, 512, dtype=dtype),
               normal(B, 512, dtype=F32)], B)


@pytest.mark.parametrize("rows", [2, 17, 64])
def test_few_row_linear(rows):
  w, b = normal(96, 256), normal(96)
  layer = ops.PackedLinear()
  check(lambda x: (layer(x, (w,), (b,)),), [normal(rows, 256)], rows)


def test_attention_prompt():
  block = rg.LocalAttentionBlock(width=512, num_heads=2, window_size=64,
                                 device="cuda", dtype=BF16)
  pos = torch.arange(150, device="cuda").expand(3, 150).contiguous()

  @torch.no_grad()
  def call(x):
    y, cache = block(x, pos)
    return y, cache.keys, cache.values

  check(call, [normal(3, 150, 512)], 3)


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("B,T", [(3, 70), (3, 300), (40, 9)])
def test_differentiable_rglru(B, T, dtype):
  lru = block_of(512, 2, dtype).rg_lru
  pos = torch.arange(T, device="cuda").expand(B, T).contiguous() + 1

  def call(x, h0, dy):
    x.requires_grad_()
    with training.differentiable():
      y, h = lru(x, pos, h0)
      (dx,) = torch.autograd.grad(y, [x], dy)
    return y.detach(), h.detach(), dx

  check(call, [normal(B, T, 512, dtype=dtype), normal(B, 512, dtype=F32),
               normal(B, T, 512, dtype=dtype)], B)


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("B,T,W", [(3, 70, 64), (3, 700, 200), (40, 9, 512)])
def test_differentiable_scan(B, T, W, dtype):
  reset = torch.zeros(B, T, dtype=torch.bool, device="cuda")

  def call(x, a, h0, dy):
    x.requires_grad_()
    with training.differentiable():
      y, h = rg.rnn_scan(x, torch.sigmoid(a), reset, h0)
      (dx,) = torch.autograd.grad(y, [x], dy)
    return y.detach(), h.detach(), dx

  check(call, [normal(B, T, W, dtype=dtype), normal(B, T, W, dtype=dtype),
               normal(B, W, dtype=F32), normal(B, T, W, dtype=dtype)], B)

"""The native host path (csrc/host_ops.cpp) against the general path in ops.py:
same kernels, same bits; it steps aside for what it does not take and notices
weights that were written to."""

import pytest
import torch

import recurrentgemma_amd as rg
from oracle import torch_ref as R
from recurrentgemma_amd import _lib
from recurrentgemma_amd import ops
from tests import helpers

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _strided(t):
  """The same values, not contiguous: what sends a call to the general path."""
  return torch.stack([t, t], dim=-1)[..., 0]


@pytest.mark.parametrize("dtype,B,T,W,H", [
    (torch.bfloat16, 3, 1, 512, 2), (torch.bfloat16, 2, 70, 512, 2),
    (torch.bfloat16, 2, 1, 384, 3), (torch.float32, 2, 1, 512, 2),
    (torch.float32, 2, 33, 192, 2), (torch.bfloat16, 1, 600, 256, 1)])
@pytest.mark.parametrize("joined", [False, True])
def test_native_calls_equal_the_general_path(dtype, B, T, W, H, joined):
  p = {k: v.to(DEV) for k, v in
       R.make_params(W, H, dtype, seed=3, gate_bias_std=0.3).items()}
  g = torch.Generator().manual_seed(4)
  x = torch.randn(B, T, W, generator=g).to(dtype).to(DEV)
  gate = torch.randn(B, T, W, generator=g).to(dtype).to(DEV) if joined else None
  weights = [p[n] for n in ("conv_w", "conv_b", "w_x", "b_x", "w_a", "b_a",
                            "a_param")]
  if T == 1:
    pos = torch.tensor([[0 if b == 1 else 5] for b in range(B)], device=DEV)
    conv = torch.randn(B, 3, W, generator=g).to(dtype).to(DEV)
    h = torch.randn(B, W, generator=g).to(DEV)

    def call(x, native):
      args = (x, pos, conv, h, *weights, False, gate)
      assert (_lib.host().recurrent_step(*args) is not None) == native
      return ops.recurrent_step(x, pos, conv, h, *weights, gate_branch=gate)
  else:
    pos = helpers.document_positions(B, T, 40, seed=5).to(DEV)

    def call(x, native):
      args = (x, pos, *weights, None, True, True, gate)
      assert (_lib.host().recurrent_core(*args) is not None) == native
      return ops.recurrent_core(x, pos, *weights, gate_branch=gate)

  general = call(_strided(x), False)
  ops.packed_gate_weights(p["w_x"], p["w_a"])  # (a first call packs)
  for got, want in zip(call(x, True), general):
    assert torch.equal(got, want)
  p["w_x"].mul_(2)  # the packed copy is stale now: packed again, not reused
  if dtype == torch.bfloat16 and W == 256 * H:
    fresh = ops.recurrent_step if T == 1 else ops.recurrent_core
    first = ((x, pos, conv, h) if T == 1 else (x, pos))
    again = fresh(*first, *weights, gate_branch=gate)
    want = fresh(_strided(x), *first[1:], *weights, gate_branch=gate)
    assert not torch.equal(again[0], general[0])
    assert all(torch.equal(a, b) for a, b in zip(again, want))


def test_native_linear_rows_follow_their_weights():
  g = torch.Generator().manual_seed(6)
  w = torch.randn(64, 128, generator=g).bfloat16().to(DEV)
  x = torch.randn(5, 128, generator=g).bfloat16().to(DEV)
  b = torch.randn(64, generator=g).bfloat16().to(DEV)
  r = torch.randn(5, 64, generator=g).bfloat16().to(DEV)
  layer = ops.PackedLinear()
  first = layer(x, (w,), (b,), residual=r)       # general path, packs
  assert _lib.host().rows_linear(layer._plan, x, (w,), (b,), r) is not None
  assert torch.equal(layer(x, (w,), (b,), residual=r), first)
  assert _lib.host().rows_linear(layer._plan, x, (w,), None, r) is None
  w.neg_()
  assert _lib.host().rows_linear(layer._plan, x, (w,), (b,), None) is None
  want = (x.double() @ w.double().T + b.double())
  assert helpers.max_rel(layer(x, (w,), (b,)), want) < 1e-2


@pytest.mark.parametrize("B,T,H,window,positions", [
    (1, 65, 10, 2048, torch.int32), (7, 72, 10, 64, torch.int64),
    (3, 43, 2, 2048, torch.int32), (130, 1, 2, 8, torch.int32),
    (1, 700, 16, 500, torch.int32), (2, 1201, 1, 2048, torch.int64)])
def test_attention_prompts_natively(B, T, H, window, positions):
  W = 256 * H
  torch.manual_seed(8)
  block = rg.LocalAttentionBlock(width=W, num_heads=H, window_size=window,
                                 device=DEV, dtype=torch.bfloat16)
  with torch.no_grad():
    block.proj_final.bias.normal_()
  x = torch.randn(B, T, W, device=DEV).bfloat16()
  pos = helpers.document_positions(B, T, 40, seed=9).to(positions).to(DEV)
  with pytest.MonkeyPatch.context() as patch:
    patch.setattr(rg.LocalAttentionBlock, "_prompt_natively",
                  lambda *a: None)
    general = block(x, pos)
  assert block._prompt_natively(_strided(x), pos, True) is None
  assert block._prompt_natively(x, pos, True) is not None
  out, cache = block(x, pos)
  assert torch.equal(out, general[0])
  for got, want in zip(cache, general[1]):
    assert got.dtype == want.dtype and torch.equal(got, want)
  alone, none = block(x, pos, return_cache=False)
  assert none is None and torch.equal(alone, general[0])
  # what is not a plain layer of the block's own takes the general path
  seen = []
  hook = block.proj_k.register_forward_hook(lambda *a: seen.append(1))
  # (other sums in front of four bf16 roundings, 2^-8 of the largest each)
  assert helpers.max_rel(block(x, pos)[0], general[0]) < 4 * 2**-8
  assert seen
  hook.remove()
  block.proj_q.bias = torch.nn.Parameter(torch.ones(W, device=DEV).bfloat16())
  assert block._prompt_natively(x, pos, True) is None

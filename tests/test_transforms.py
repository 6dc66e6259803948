"""Calls that take kernels in place of torch's operators leave tensors that torch.func
or forward-mode differentiation stands behind to the operators (on the CPU: nothing is
launched)."""

import functools

import pytest
import torch
import torch.autograd.forward_ad as fwd

from recurrentgemma_amd import griffin as G
from recurrentgemma_amd import ops


@pytest.fixture
def embedder(monkeypatch):
  """One whose few-row kernel may not be reached."""
  monkeypatch.setattr(ops.PackedLinear, "usable", staticmethod(lambda *a: True))

  def refuse(*a, **k):
    raise AssertionError("the kernel sees no transform")

  monkeypatch.setattr(ops.PackedLinear, "__call__", refuse)
  torch.manual_seed(3)
  e = G.Embedder(32_000, 1024, True, dtype=torch.bfloat16)
  e.requires_grad_(False)
  e.decode = functools.partial(e.decode, step=True)
  return e


def test_logits_under_transforms(embedder):
  table = embedder.input_embedding
  x, dx = torch.randn(2, 3, 1024).bfloat16()
  with pytest.raises(AssertionError):
    embedder.decode(x)
  # (one rounding of float32 sums each, in whatever order)
  close = lambda a, b: torch.testing.assert_close(a, b, rtol=2**-7, atol=1e-5)
  want, tangent = x @ table.T, dx @ table.T
  close(torch.vmap(embedder.decode)(x), want)
  primal, got = torch.func.jvp(embedder.decode, (x,), (dx,))
  close(primal, want)
  close(got, tangent)
  with torch.no_grad(), fwd.dual_level():
    primal, got = fwd.unpack_dual(embedder.decode(fwd.make_dual(x, dx)))
    close(primal, want)
    close(got, tangent)
    with pytest.raises(AssertionError):
      embedder.decode(x)  # (no tangent of its own)


@pytest.mark.parametrize("vocab,width,streamed", [
    (256_000, 2560, True), (256_000, 4096, True), (32_000, 1024, True),
    (128_256, 2560, True), (31_936, 2560, False), (50_304, 2560, False),
    (256_032, 2560, False), (256_000, 512, False), (256_000, 4160, False)])
def test_which_tables_are_streamed(vocab, width, streamed):
  e = G.Embedder(vocab, width, True, device="meta", dtype=torch.bfloat16)
  assert e._steps_stream() == streamed

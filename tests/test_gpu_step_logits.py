"""The copy of the token table that the logits of decode steps are formed from
(Embedder.decode): who makes it, and what it gives."""

import copy
import pickle

import pytest
import torch

from recurrentgemma_amd import griffin as G
from recurrentgemma_amd import sampler as S

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _model():
  torch.manual_seed(6)
  config = G.GriffinConfig(
      vocab_size=32_000, width=1024, mlp_expanded_width=512, lru_width=512,
      num_heads=4, block_types=(G.TemporalBlockType.RECURRENT,
                                G.TemporalBlockType.ATTENTION),
      embeddings_scale_by_sqrt_dim=True, attention_window_size=64,
      logits_soft_cap=30.0)
  return G.Griffin(config, device=DEV, dtype=torch.bfloat16).eval()


def _prompt(rows):
  g = torch.Generator().manual_seed(7)
  tokens = torch.randint(1, 32_000, (rows, 6), generator=g).to(DEV)
  return tokens, torch.arange(6, device=DEV).expand(rows, 6).contiguous()


@pytest.mark.parametrize("rows", [1, 3, 24, 25])
def test_rows_of_a_step(rows):
  e = G.Embedder(32_000, 1024, True, device=DEV, dtype=torch.bfloat16)
  x = torch.randn(rows, 1, 1024, device=DEV).bfloat16()
  with torch.no_grad():
    for _ in range(2):
      got = e.decode(x, step=True)
      assert (e._rows_logits is not None) == (rows <= 24)
      want = x.double() @ e.input_embedding.double().T
      # (half a unit in the last place of bf16, and the float32 sums' order)
      assert ((got.double() - want).abs() <= want.abs() * 2**-8 + 1e-5).all()
      e.input_embedding.neg_()
  assert e.decode(x, step=True).requires_grad


@torch.no_grad()
def test_who_makes_a_copy():
  model = _model()
  tokens, pos = _prompt(3)
  last, after = tokens[:, -1:], pos[:, -1:] + 1
  _, cache = model(tokens, pos)  # a prompt of a few rows, asked once
  model.embedder.decode(torch.randn(2, 1024, device=DEV).bfloat16())
  assert model.embedder._rows_logits is None
  model.embedder.step_copy = False
  model(last, after, cache)
  assert model.embedder._rows_logits is None
  model.embedder.step_copy = True
  model(last, after, cache)
  assert model.embedder._rows_logits._packed is not None
  again = pickle.loads(pickle.dumps(model.embedder))
  assert again._rows_logits._packed is None and copy.deepcopy(model)
  # nothing counts the writes to an inference tensor: a copy would be made anew by
  # every step
  with torch.inference_mode():
    other = _model()
    _, cache = other(tokens, pos)
    other(last, after, cache)
  assert other.embedder._rows_logits is None


@torch.no_grad()
def test_replaced_decode_gets_what_it_takes(monkeypatch):
  model = _model()
  tokens, pos = _prompt(2)
  _, cache = model(tokens, pos)
  flat = lambda x: x.new_zeros(*x.shape[:-1], 5)
  model.embedder.decode = flat
  assert model(tokens[:, -1:], pos[:, -1:] + 1, cache)[0].shape == (2, 1, 5)
  del model.embedder.decode
  monkeypatch.setattr(G.Embedder, "decode", lambda self, x: flat(x))
  assert model(tokens[:, -1:], pos[:, -1:] + 1, cache)[0].shape == (2, 1, 5)


def test_captured_steps_equal_eager_ones():
  model = _model()
  tokens, _ = _prompt(3)
  lens = torch.tensor([6, 1, 4], device=DEV)
  eager, graphed = S.Sampler(model), S.Sampler(model, use_graph=True)
  # (the second generation has its prompts' last tokens, the one that is a row's
  # only one among them, replayed)
  for write in (False, True, False):
    want, want_logits = eager.sample_tokens(tokens, lens, 8, return_logits=True)
    got, logits = graphed.sample_tokens(tokens, lens, 8, return_logits=True)
    torch.cuda.synchronize()
    assert torch.equal(got, want) and torch.equal(logits, want_logits)
    if write:
      with torch.no_grad():
        model.embedder.input_embedding.mul_(0.5)

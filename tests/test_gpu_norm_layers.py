"""A norm and the few-row layers behind it as one launch (csrc/rg_linear.hip,
linear_rows_normed_kernel) against the two calls it stands for, bit for bit."""

import pytest
import torch

from recurrentgemma_amd import griffin as G
from recurrentgemma_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
K = 2560


def _randn(seed, *shape, scale=1.0):
  g = torch.Generator().manual_seed(seed)
  return (torch.randn(*shape, generator=g) * scale).bfloat16().to(DEV)


def _layers(kind):
  """PackedLinear, its weights and biases: two equal layers, three unequal ones
  as one output, the MLP's pair."""
  if kind == "pair":
    return (ops.PackedLinear(layout=1, gelu_pair=True),
            (_randn(1, 2, K, 7680, scale=0.02),), (_randn(2, 2, 1, 1, 7680),))
  rows = (2560, 2560) if kind == "two" else (2560, 256, 256)
  weights = tuple(_randn(3 + i, n, K, scale=0.02) for i, n in enumerate(rows))
  biases = tuple(_randn(7 + i, n) for i, n in enumerate(rows))
  return ops.PackedLinear(), weights, biases if kind == "two" else None


# (more than 32 rows of pairs, and 64 and more of the others, take two launches)
@pytest.mark.parametrize("kind,rows", [
    ("two", 1), ("two", 16), ("two", 17), ("two", 33), ("two", 64),
    ("three", 2), ("three", 32), ("pair", 1), ("pair", 16), ("pair", 31),
    ("pair", 40)])
@pytest.mark.parametrize("patience", [ops.NORM_PATIENCE, 0])
def test_norm_and_layers_equal_their_parts(kind, rows, patience, monkeypatch):
  """patience 0: most workgroups form the norm of all rows themselves."""
  monkeypatch.setattr(ops, "NORM_PATIENCE", patience)
  before, w_before = ops.PackedLinear(), (_randn(20, K, K, scale=0.02),)
  bias, scale = (_randn(21, K),), _randn(22, K, scale=0.2)
  x, skip = _randn(23, rows, 1, K), _randn(24, rows, 1, K)
  state = _randn(25, rows, 3, K)
  layer, weights, biases = _layers(kind)

  def part():
    return before.partial(x, w_before, bias)

  total, normed = ops.add_rms_norm(part(), skip, scale)
  want = layer(normed, weights, biases)  # (and packs the weights)
  fused = not (kind == "pair" and rows > 32)

  def check(pending, got):
    assert torch.equal(pending.total, total)
    assert torch.equal(pending.out, normed)
    wants = want if isinstance(want, tuple) else (want,)
    gots = got if isinstance(got, tuple) else (got,)
    assert len(wants) == len(gots)
    assert all(torch.equal(a, b) for a, b in zip(wants, gots))

  for _ in range(3):  # (the flags are new with every layer in front)
    pending = ops.PendingNorm(part(), skip, scale, 1e-6)
    assert not pending.formed
    called = layer._with_norm(pending, weights, biases)
    assert (called is not None) == fused
    check(pending, called if fused else layer(pending, weights, biases))
  # formed once: its readers from then on take the tensor
  assert pending.formed and pending.tensor() is pending.out
  again = layer(pending, weights, biases)
  check(pending, again)
  if kind == "two":
    pending = ops.PendingNorm(part(), skip, scale, 1e-6)
    *got, copied = layer.beside(pending, weights, biases, state)
    check(pending, tuple(got))
    assert torch.equal(copied, state) and copied.data_ptr() != state.data_ptr()
  # sums that carry the addend, read once: a second norm of them takes no flags
  sums = part()
  sums.addend = skip
  check(*(lambda p: (p, layer(p, weights, biases)))(
      ops.PendingNorm(sums, None, scale, 1e-6)))
  second = ops.PendingNorm(sums, None, scale, 1e-6)
  assert second.flags is None
  check(second, layer(second, weights, biases))


def test_norm_and_layers_in_a_graph():
  """Replays of a captured chain, eager work between them."""
  before, w_before = ops.PackedLinear(), (_randn(20, K, K, scale=0.02),)
  scale, x = _randn(22, K, scale=0.2), _randn(23, 5, 1, K)
  layer, weights, biases = _layers("two")
  out, = (layer(ops.add_rms_norm(before.partial(x, w_before), None, scale)[1],
                weights, biases),)

  def chain():
    sums = before.partial(x, w_before)
    return layer(ops.PendingNorm(sums, None, scale, 1e-6), weights, biases)

  side = torch.cuda.Stream()
  with torch.cuda.stream(side):
    chain()
  torch.cuda.synchronize()
  graph = torch.cuda.CUDAGraph()
  with torch.cuda.graph(graph):
    got = chain()
  for i in range(4):
    x.copy_(_randn(30 + i, 5, 1, K))
    graph.replay()
    want = layer(ops.add_rms_norm(before.partial(x, w_before), None, scale)[1],
                 weights, biases)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want)), i


@pytest.mark.parametrize("width,rows,fused", [
    # (of a step's four norms: in front of two blocks' layers and of two MLPs, but for
    # the first, which reads no sums)
    (2560, 16, 3), (2560, 33, 1), (1024, 16, 0), (4096, 2, 0)])
@torch.no_grad()
def test_norms_wait_only_for_layers_that_form_them(width, rows, fused, monkeypatch):
  torch.manual_seed(9)
  config = G.GriffinConfig(
      vocab_size=64, width=width, mlp_expanded_width=3 * width, lru_width=width,
      num_heads=width // 256, block_types=(G.TemporalBlockType.RECURRENT,
                                           G.TemporalBlockType.ATTENTION),
      embeddings_scale_by_sqrt_dim=True, attention_window_size=64,
      logits_soft_cap=30.0)
  model = G.Griffin(config, device=DEV, dtype=torch.bfloat16).eval()
  tokens = torch.randint(1, 64, (rows, 1), device=DEV)
  pos = torch.ones_like(tokens)

  def step():
    cache = model.init_cache(rows, torch.bfloat16, device=DEV)
    return model(tokens, pos, cache)[0]

  got = step()
  made, formed = [], []
  class Counted(ops.PendingNorm):
    def __init__(self, *a):
      super().__init__(*a)
      made.append(self)
    def tensor(self):
      if not self.formed:
        formed.append(self)
      return super().tensor()
  monkeypatch.setattr(ops, "PendingNorm", Counted)
  assert torch.equal(step(), got)
  assert len(made) == fused and not formed  # (in a launch of its own: none)
  monkeypatch.setattr(G, "_norm_for", lambda reader, norm, *a: norm.add_then_norm(*a))
  assert torch.equal(step(), got)  # the same bits either way

"""Prompt passes that leave padding out (ops.RowRuns, Griffin.prompt_cache):
products and norms of runs of eight rows, and the cache a prompt leaves."""

import pytest
import torch

from recurrentgemma_amd import _lib
from recurrentgemma_amd import griffin as G
from recurrentgemma_amd import ops
from recurrentgemma_amd import sampler as S

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _runs(lengths, tokens):
  runs = ops.RowRuns(lengths, tokens, DEV)
  kept = torch.zeros(runs.rows, dtype=torch.bool)
  for first in runs.first.tolist():
    assert 0 <= first <= runs.rows - 8
    kept[first:first + 8] = True
  for b, n in enumerate(lengths):
    assert kept[(b + 1) * tokens - n:(b + 1) * tokens].all()
  return runs, kept.to(DEV)


def _near(got, want, sums):
  """One bf16 rounding (2^-9 of the value, and as much for a float32 sum next to
  a boundary) of a float32 sum of terms whose magnitudes add up to `sums`."""
  assert ((got.double() - want).abs() <= want.abs() * 2**-8 +
          2**-20 * sums).all()


@pytest.mark.parametrize("lengths,T,K,N", [
    # one run, runs that overlap at the start, a cut tile, every tile size that the
    # cost model picks from, a few hundred rows to several rounds of the chip
    ([8], 8, 64, (64,)), ([3, 9, 1], 9, 64, (128, 8)),
    ([5, 300, 77], 301, 512, (512, 256, 256)),
    ([999, 500, 640, 801, 555], 999, 256, (2560, 2560)),
    ([700, 350, 600, 421, 480], 700, 1024, (320,)),
    ([640] * 9 + [3], 641, 2560, (2560,))])
def test_products_and_norms_of_runs(lengths, T, K, N):
  runs, kept = _runs(lengths, T)
  g = torch.Generator(device=DEV).manual_seed(3)
  normal = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()
  x = normal(runs.rows, K)
  x[~kept] = float("nan")  # (never read)
  ws, bs = [normal(n, K) for n in N], [normal(n) for n in N[:-1]] + [None]
  out = [torch.full((runs.rows, n), 7.0, device=DEV).bfloat16() for n in N]
  ops.linear_many_runs(x, ws, bs, runs, out)
  for o, w, b in zip(out, ws, bs):
    assert (o[~kept] == 7).all()
    want = x[kept].double() @ w.double().T + (0 if b is None else b.double())
    _near(o[kept], want, x[kept].double().abs() @ w.double().abs().T)
  # the pair: what the call for all rows gives for these rows, bit for bit (the same
  # instructions along K, whatever the tile)
  w, b = normal(2, K, 256), normal(2, 1, 1, 256)
  pair = ops.linear_gelu_pair_runs(x, w, b, runs)
  xk = x[kept]
  want = torch.empty(len(xk), 256, device=DEV, dtype=torch.bfloat16)
  _lib.check(_lib.lib().rg_linear_gelu_pair(
      xk.data_ptr(), w.data_ptr(), b.data_ptr(), want.data_ptr(), len(xk), K, 256,
      _lib.RG_DTYPE_BF16, torch.cuda.current_stream().cuda_stream))
  assert torch.equal(pair[kept], want)
  a = normal(runs.rows, K)
  scale = normal(K)
  total, normed = ops.add_rms_norm_runs(x, a, scale, 1e-6, runs)
  want = ops.add_rms_norm(x[kept], a[kept], scale)
  assert torch.equal(total[kept], want[0]) and torch.equal(normed[kept], want[1])


@pytest.mark.parametrize("lengths,T", [
    ([301, 2, 100, 299, 17, 8, 150, 64, 33, 200] * 3, 301),
    ([90, 5, 47] * 30, 97)])
@torch.no_grad()
def test_prompts_without_their_padding(lengths, T):
  torch.manual_seed(11)
  kinds = (G.TemporalBlockType.RECURRENT, G.TemporalBlockType.ATTENTION,
           G.TemporalBlockType.RECURRENT)
  config = G.GriffinConfig(
      vocab_size=640, width=512, mlp_expanded_width=1536, lru_width=512,
      num_heads=2, block_types=kinds, embeddings_scale_by_sqrt_dim=True,
      attention_window_size=64, logits_soft_cap=30.0)
  model = G.Griffin(config, device=DEV, dtype=torch.bfloat16).eval()
  B = len(lengths)
  tokens = torch.randint(1, 640, (B, T), device=DEV)
  lens = torch.tensor(lengths, device=DEV)
  plain, runs = S.Sampler(model), S.Sampler(model)
  plain._prompt_runs = lambda *a: None
  assert runs._prompt_runs(B, T, lens) is not None
  want, want_logits = plain.sample_tokens(tokens, lens, 4, return_logits=True)
  # (whatever a tensor's memory held before: none of it may be looked at)
  junk = [torch.full((1 << 22,), float("nan"), device=DEV) for _ in range(8)]
  del junk
  got, logits = runs.sample_tokens(tokens, lens, 4, return_logits=True)
  assert torch.isfinite(logits).all()
  # other sums in front of the roundings of three blocks, about ten tensors each
  first = (logits[:, 0].float() - want_logits[:, 0].float()).norm()
  assert first <= 30 ** 0.5 * 2**-8 * want_logits[:, 0].float().norm()
  same = (got == want).float().mean()
  assert same > 0.9, same
  # rows of one token, rows that are full beyond their tokens: all rows as before
  lens[1] = 1
  assert runs._prompt_runs(B, T, lens) is None
  handle = model.blocks[0].mlp_block.ffw_down.register_forward_hook(lambda *a: None)
  lens[1] = 2
  assert runs._prompt_runs(B, T, lens) is None
  handle.remove()
  assert runs._prompt_runs(B, T, lens) is not None


@pytest.mark.parametrize("lengths,T,window", [
    ([301, 2, 100, 299, 17, 8, 150, 64, 33, 200], 301, 64),
    ([90, 1, 47, 3], 97, 2048), ([5, 40, 33], 40, 32)])
@torch.no_grad()
def test_cache_without_the_padding(lengths, T, window):
  """Every state that prompt_cache leaves against forward's for the same prompts: h,
  the conv's rows (some of them padding), the rings as far as a step sees them."""
  torch.manual_seed(14)
  kinds = (G.TemporalBlockType.RECURRENT, G.TemporalBlockType.ATTENTION,
           G.TemporalBlockType.RECURRENT)
  model = _small_model(width=512, mlp_expanded_width=1536, lru_width=512,
                       num_heads=2, attention_window_size=window,
                       block_types=kinds)
  B = len(lengths)
  tokens = torch.randint(1, 64, (B, T), device=DEV)
  pos = (torch.arange(T) - T + torch.tensor(lengths)[:, None]).clip(min=-1).to(
      DEV, torch.int32)
  assert model.prompt_runs_serve(B, T)
  _, want = model(tokens, pos, None, return_logits=False)
  junk = [torch.full((1 << 22,), float("nan"), device=DEV) for _ in range(8)]
  del junk
  got = model.prompt_cache(tokens, pos, ops.RowRuns(lengths, T, DEV))

  def near(a, b, tensors):
    """Other sums in front of the roundings of so many tensors."""
    a, b = a.double(), b.double()
    assert torch.isfinite(a).all()
    assert (a - b).norm() <= tensors ** 0.5 * 2**-8 * b.norm()

  assert got.keys() == want.keys()
  for i, kind in enumerate(kinds):
    a, b = got[f"blocks.{i}"], want[f"blocks.{i}"]
    tensors = 4 + 10 * i
    assert [t.dtype for t in a] == [t.dtype for t in b]
    for row, n in enumerate(lengths):
      if kind is G.TemporalBlockType.RECURRENT:
        near(a.rg_lru_state[row], b.rg_lru_state[row], tensors)
        near(a.conv1d_state[row], b.conv1d_state[row], tensors)
        continue
      assert a.num_tokens[row] == b.num_tokens[row] == n
      seen = torch.arange(max(0, n - window), n) % window
      near(a.keys[row, seen], b.keys[row, seen], tensors)
      near(a.values[row, seen], b.values[row, seen], tensors)


def _small_model(**changes):
  config = G.GriffinConfig(
      vocab_size=64, width=256, mlp_expanded_width=256, lru_width=256,
      num_heads=1, block_types=(G.TemporalBlockType.RECURRENT,),
      embeddings_scale_by_sqrt_dim=True, attention_window_size=64,
      logits_soft_cap=30.0)._replace(**changes)
  model = G.Griffin(config, device=DEV, dtype=torch.bfloat16).eval()
  model.prompt_runs_pay = lambda *a: True  # (of such a size it never does)
  return model


@pytest.mark.parametrize("lens", [
    torch.tensor([70]), torch.tensor([70.0]), torch.full((90,), 70.9)])
@torch.no_grad()
def test_lengths_as_positions_take_them(lens):
  """One length for all rows, lengths that are no whole numbers: what the positions
  are made of (broadcast, cut off) is what the padding is."""
  torch.manual_seed(13)
  model = _small_model()
  tokens = torch.randint(1, 64, (90, 100), device=DEV)
  plain, runs = S.Sampler(model), S.Sampler(model)
  plain._prompt_runs = lambda *a: None
  got, _ = runs.sample_tokens(tokens, lens.to(DEV), 2)
  want, _ = plain.sample_tokens(tokens, lens.to(DEV), 2)
  # (other sums in front of the roundings of one block)
  assert (got == want).float().mean() > 0.9


@torch.no_grad()
def test_prompts_beyond_what_the_products_address():
  """Left-padded prompts of more rows than a product of runs takes: all rows, as a
  sampler that knows of no runs."""
  torch.manual_seed(12)
  model = _small_model(mlp_expanded_width=16384)
  plain, runs = S.Sampler(model), S.Sampler(model)
  plain._prompt_runs = lambda *a: None
  lens = torch.full((32,), 900, device=DEV)
  for T, fit in ((2032, True), (2033, False)):  # 64 992 rows, 65 024
    tokens = torch.randint(1, 64, (32, T), device=DEV)
    assert (runs._prompt_runs(32, T, lens) is not None) == fit
    got, _ = runs.sample_tokens(tokens, lens, 2)
    want, _ = plain.sample_tokens(tokens, lens, 2)
    # (one launch or the library's sums in front of the roundings of one block)
    assert torch.equal(got, want) if not fit else (got == want).float().mean() > 0.9


@torch.no_grad()
def test_lengths_are_read_where_they_may_be(monkeypatch):
  """drop_padding=False reads nothing back; prompts without padding do not have the
  model's layers looked at."""
  model = _small_model()
  tokens = torch.randint(1, 64, (90, 100), device=DEV)
  full, half = (torch.full((90,), n, device=DEV) for n in (100, 50))
  declined, runs = S.Sampler(model, drop_padding=False), S.Sampler(model)
  declined.sample_tokens(tokens, half, 3)
  torch.cuda.synchronize()
  torch.cuda.set_sync_debug_mode("error")
  try:
    declined.sample_tokens(tokens, half, 3)
    with pytest.raises(RuntimeError):
      runs._prompt_runs(90, 100, half)
  finally:
    torch.cuda.set_sync_debug_mode("default")
  asked = []
  serve = model.prompt_runs_serve
  monkeypatch.setattr(model, "prompt_runs_serve",
                      lambda *a: asked.append(a) or serve(*a))
  assert runs._prompt_runs(90, 100, full) is None and not asked
  assert runs._prompt_runs(90, 100, half) is not None and asked == [(90, 99)]


class _Around(torch.nn.Module):
  """A caller's own module around the model, with what the sampler asks of one."""

  def __init__(self, model):
    super().__init__()
    self.inner, self.calls = model, 0
    self.config, self.blocks = model.config, model.blocks
    self.init_cache = model.init_cache

  def forward(self, *args, **kwargs):
    self.calls += 1
    return self.inner(*args, **kwargs)


@torch.no_grad()
def test_a_model_of_the_callers_own_is_called():
  model = _Around(_small_model())
  tokens = torch.randint(1, 64, (90, 100), device=DEV)
  lens = torch.full((90,), 50, device=DEV)
  S.Sampler(model).sample_tokens(tokens, lens, 3)
  assert model.calls == 4  # the prompt, its last token, two steps


@torch.no_grad()
def test_prompts_without_their_padding_where_it_pays(monkeypatch):
  """As test_prompts_without_their_padding, at a width where the sampler goes by runs
  of itself; and a narrow model, whose lengths are not even read."""
  model = _small_model(width=2560, mlp_expanded_width=7680, lru_width=2560,
                       num_heads=10, block_types=(
                           G.TemporalBlockType.RECURRENT,
                           G.TemporalBlockType.ATTENTION))
  del model.prompt_runs_pay
  lengths = [301, 2, 100, 299, 17, 8, 150, 64, 33, 200] * 3
  tokens = torch.randint(1, 64, (30, 301), device=DEV)
  lens = torch.tensor(lengths, device=DEV)
  plain, runs = S.Sampler(model, drop_padding=False), S.Sampler(model)
  want, _ = plain.sample_tokens(tokens, lens, 4)
  took = []
  cache = model.prompt_cache
  monkeypatch.setattr(model, "prompt_cache", lambda *a: took.append(a) or cache(*a))
  got, _ = runs.sample_tokens(tokens, lens, 4)
  assert len(took) == 1
  # (other sums in front of the roundings of two blocks)
  assert (got == want).float().mean() > 0.9
  narrow = _small_model()
  del narrow.prompt_runs_pay
  torch.cuda.set_sync_debug_mode("error")
  try:
    assert S.Sampler(narrow)._prompt_runs(30, 301, lens, narrow.prompt_runs_pay) is None
  finally:
    torch.cuda.set_sync_debug_mode("default")

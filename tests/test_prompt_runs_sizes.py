"""Which prompts may leave their padding out (Griffin.prompt_runs_serve), by their
sizes: what the products of runs of rows take, on the CPU (nothing is launched)."""

import ctypes

import pytest
import torch

from recurrentgemma_amd import _lib
from recurrentgemma_amd import griffin as G
from recurrentgemma_amd import ops


def _model(preset, **changes):
  config = G.GriffinConfig.from_preset(preset)._replace(**changes)
  return G.Griffin(config, device="meta", dtype=torch.bfloat16)


# (rows + 512) x the widest layer's features below 2^30: whole batches around it
@pytest.mark.parametrize("preset,batch,most", [
    (G.Preset.RECURRENT_GEMMA_2B_V1, 64, 2176),
    (G.Preset.RECURRENT_GEMMA_2B_V1, 32, 4353),
    (G.Preset.RECURRENT_GEMMA_9B_V1, 64, 1357),
    (G.Preset.RECURRENT_GEMMA_9B_V1, 32, 2714)])
def test_rows_that_the_products_address(preset, batch, most):
  model = _model(preset)
  widest = model.config.mlp_expanded_width
  assert (batch * most + 512) * widest < 2**30 <= (batch * (most + 1) + 512) * widest
  assert model._prompt_runs_sizes_serve(batch, most)
  assert not model._prompt_runs_sizes_serve(batch, most + 1)
  assert not model.prompt_runs_serve(batch, most + 1)


def test_every_layer_is_asked_for():
  # the recurrent branch wider than the MLP, and a row's queries beyond 2 GiB
  wide = _model(G.Preset.RECURRENT_GEMMA_2B_V1, lru_width=10240)
  assert wide._prompt_runs_sizes_serve(32, 3260)  # 104 320 rows
  assert not wide._prompt_runs_sizes_serve(32, 3261)
  long = _model(G.Preset.RECURRENT_GEMMA_2B_V1, width=4096, num_heads=16,
                mlp_expanded_width=64, lru_width=64)
  assert not long._prompt_runs_sizes_serve(1, 262144)
  narrow = _model(G.Preset.RECURRENT_GEMMA_2B_V1, mlp_expanded_width=7720)
  assert not narrow._prompt_runs_sizes_serve(16, 999)


@pytest.mark.parametrize("rows,K,N", [
    (139_299, 2560, 7680), (86_870, 4096, 12288), (7, 2560, 7680),
    (9000, 2560, 7684), (9000, 2568, 7680)])
def test_what_serve_refuses_the_call_refuses(rows, K, N):
  at = [ctypes.c_void_p(4096 * i) for i in range(1, 6)]  # (never dereferenced)
  lib = _lib.lib()
  n = (ctypes.c_int * 1)(N)
  one = ctypes.c_void_p * 1
  assert not ops.linear_gelu_pair_runs_serve(rows, K, N)
  assert lib.rg_linear_gelu_pair_runs(*at[:4], rows, at[4], 1, K, N,
                                      _lib.RG_DTYPE_BF16, None) == -2
  assert not ops.linear_many_runs_serve(rows, K, N)
  assert lib.rg_linear_many_runs(
      at[0], rows, at[4], 1, K, 1, one(at[1]), one(None), one(at[2]), n,
      _lib.RG_DTYPE_BF16, None) == -2
  assert ops.linear_many_runs_serve(8, 2560, 7680, 7680)


@pytest.mark.parametrize("changes,batch,tokens,real,pays", [
    # (measured passes; 3 blocks each)
    (dict(width=512, num_heads=2, lru_width=512, mlp_expanded_width=1536), 16, 512,
     0.5, False),
    (dict(width=512, num_heads=2, lru_width=512, mlp_expanded_width=1536), 60, 500,
     0.75, False),
    (dict(), 16, 1000, 0.75, True), (dict(), 64, 128, 0.85, True),
    (dict(), 16, 1000, 1.0, False),
    (dict(width=4096, num_heads=16, lru_width=4096, mlp_expanded_width=12288), 16, 512,
     0.9, False),
    (dict(width=4096, num_heads=16, lru_width=4096, mlp_expanded_width=12288), 16, 512,
     0.75, True)])
def test_where_leaving_padding_out_pays(changes, batch, tokens, real, pays):
  R, A = G.TemporalBlockType.RECURRENT, G.TemporalBlockType.ATTENTION
  for kinds in ((R, R, A), (R,), (A, A)):
    model = _model(G.Preset.RECURRENT_GEMMA_2B_V1, block_types=kinds, **changes)
    count = int(batch * tokens * real / 8)
    assert model.prompt_runs_pay(batch, tokens, count) == pays
  # beyond what the products address: never
  assert not model.prompt_runs_pay(batch * 1000, tokens, count)

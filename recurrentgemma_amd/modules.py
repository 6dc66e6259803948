"""The caller of the hot path: Griffin's recurrent block, on the fused kernels.

RecurrentBlock / RecurrentBlockCache mirror
recurrentgemma/torch/modules.py:32-37 and :496-680 (same constructor,
parameter names, forward signature and cache tuple).  linear_x / linear_y /
linear_out stay torch.nn.Linear, whose products run on this package's kernels
where those are ahead of hipBLASLt's (linears below, and a few rows); conv_1d -> rg_lru runs as
  prefill: rg_recurrent_core (the single prefill kernel, or rg_gates_gemm with
           the conv on load + rg_lru_scan_fused: the library picks)
  decode : rg_recurrent_step
unless the conv width is not 4, where the stand-alone conv kernel is used.
"""

from __future__ import annotations

import math
from typing import NamedTuple

import torch
from torch import nn

from recurrentgemma_amd import _lib
from recurrentgemma_amd import compiled
from recurrentgemma_amd import layers
from recurrentgemma_amd import ops
from recurrentgemma_amd import training


class RecurrentBlockCache(NamedTuple):
  rg_lru_state: torch.Tensor  # [B, lru_width] float32
  conv1d_state: torch.Tensor  # [B, temporal_width-1, lru_width]


def gelu(x: torch.Tensor) -> torch.Tensor:
  return nn.functional.gelu(x, approximate="tanh")


def _parameters(module, *names):
  """Parameters of a module by name.  nn.Module's attribute lookup costs about
  half a microsecond each, which a decode step with its twenty tensors does
  not have; the dictionary behind it is read instead, and the attribute where
  the name is not in it (a parametrised weight, an object that is no module)."""
  try:
    own = module._parameters
  except AttributeError:
    own = ()
  return [own[n] if n in own else getattr(module, n) for n in names]


def _as_written(module, kind) -> bool:
  """Whether calling the module is nothing but kind.forward on its own
  parameters: no subclass, hook, parametrisation or replaced method."""
  return (type(module) is kind and "forward" not in module.__dict__ and
          not (module._forward_hooks or module._forward_pre_hooks or
               module._backward_hooks or module._backward_pre_hooks))


def _global_hooks() -> bool:
  m = nn.modules.module
  return bool(m._global_forward_hooks or m._global_forward_pre_hooks or
              m._global_backward_hooks or m._global_backward_pre_hooks)


def linears(x, *layers):
  """The outputs of nn.Linear layers that read x.  More rows than a decode
  step's in bf16: one launch (ops.linear_many) where that is ahead of the
  library, as long as calling the layers is nothing but their products (and no
  program is being traced: the kernels are reached through ctypes)."""
  # (what mostly says no comes first: the callers of few rows wait for the host)
  if (x.dtype is torch.bfloat16 and x.dim() > 1 and
      x.numel() > 64 * x.shape[-1] and not compiled.tracing() and
      all(type(layer) is nn.Linear for layer in layers) and
      ops.linear_many_pays(x, *[layer.out_features for layer in layers]) and
      not _global_hooks() and
      all(_as_written(layer, nn.Linear) for layer in layers)):
    parts = [_parameters(layer, "weight", "bias") for layer in layers]
    out = ops.linear_many(x, [w for w, _ in parts], [b for _, b in parts])
    if out is not None:
      return out
  return [layer(x) for layer in layers]


def _core_weights(conv_1d, rg_lru):
  """conv_w, conv_b, w_x, b_x, w_a, b_a, a_param."""
  if compiled.tracing():
    gx, ga = rg_lru.input_gate, rg_lru.a_gate
    return conv_1d.w, conv_1d.b, gx.w, gx.b, ga.w, ga.b, rg_lru.a_param
  try:
    gx, ga = rg_lru._modules["input_gate"], rg_lru._modules["a_gate"]
  except (AttributeError, KeyError):  # no module, or one that passes them through
    gx, ga = rg_lru.input_gate, rg_lru.a_gate
  return (*_parameters(conv_1d, "w", "b"), *_parameters(gx, "w", "b"),
          *_parameters(ga, "w", "b"),
          *_parameters(rg_lru, "a_param"))


def recurrent_core(conv_1d: layers.Conv1D, rg_lru: layers.RGLRU, x,
                   segment_pos, cache: RecurrentBlockCache | None = None,
                   return_cache: bool = True, in_place: bool = False,
                   gate_branch=None):
  """conv_1d -> rg_lru exactly as RecurrentBlock.forward chains them
  (modules.py:632-643), fused.  Returns (y, RecurrentBlockCache | None).
  in_place (decode only): the step overwrites the tensors of `cache` and
  returns them, for callers that replay a captured step on fixed buffers; the
  default returns new tensors like the reference.
  gate_branch: the block's linear_y output; the result is then the join
  y * gelu(gate_branch) of modules.py:627-628, 644 -- inside the prefill
  kernel where that runs, as a pass of its own (ops.gelu_mul) elsewhere."""
  if not torch.is_grad_enabled():
    return _recurrent_core(conv_1d, rg_lru, x, segment_pos, cache, return_cache,
                           in_place, gate_branch)
  with torch.no_grad():
    return _recurrent_core(conv_1d, rg_lru, x, segment_pos, cache, return_cache,
                           in_place, gate_branch)


def _recurrent_core(conv_1d, rg_lru, x, segment_pos, cache, return_cache,
                    in_place, gate_branch, conv_aside=None):
  bs, l, _ = x.shape
  assert segment_pos.shape == (bs, l)
  fused = conv_1d.temporal_width == 4
  if fused:
    weights = _core_weights(conv_1d, rg_lru)
  if cache is not None:
    b, num_tokens, d = x.shape
    assert cache.conv1d_state.shape == (b, conv_1d.temporal_width - 1, d)
    assert num_tokens == 1
    if fused:
      if compiled.tracing() and not in_place:
        # (a traced program holds the step as one operator node)
        y, h, conv_state = torch.ops.recurrentgemma_amd.recurrent_step(
            x, segment_pos, cache.conv1d_state, cache.rg_lru_state, *weights,
            gate_branch)
      else:
        y, h, conv_state = ops.recurrent_step(
            x, segment_pos, cache.conv1d_state, cache.rg_lru_state, *weights,
            in_place, gate_branch, conv_aside)
      if not return_cache:
        return y, None
      return y, RecurrentBlockCache(rg_lru_state=h, conv1d_state=conv_state)
  if not fused or cache is not None:
    if in_place:
      raise ValueError("in-place decode needs the fused step (conv width 4)")
    xc, conv_state = conv_1d(x, segment_pos,
                             None if cache is None else cache.conv1d_state,
                             return_cache)
    y, h = rg_lru(xc, segment_pos,
                  None if cache is None else cache.rg_lru_state, return_cache)
  else:
    # One call; the library picks the kernels (rg_recurrent_core): for bf16
    # and 256-wide heads the single-launch kernel, one workgroup per (row,
    # head), per 32 channels of one (few rows of some hundred tokens), per
    # chunk of one (few long ones) or by blocks of 32 tokens (pairs that
    # do not come out even on the CUs), or several whole rows of up to 16 tokens
    # to a tile; for bf16 heads of 136 to 248 channels slices of heads, alike;
    # 256-wide heads beyond 512 pairs of rows that short or 1024 of up to 32
    # tokens, a few long rows of narrower heads, and every other head width: gate
    # GEMM + scan; float32 with 256-wide heads: one launch
    # for few short rows, else conv, projections and recurrence; and the join with
    # the gate branch inside those kernels (after the two-kernel form it is a pass
    # of its own).
    if compiled.tracing():
      y, h, conv_state = torch.ops.recurrentgemma_amd.recurrent_core(
          x, segment_pos, *weights, None, gate_branch)
    else:
      y, h, conv_state = ops.recurrent_core(
          x, segment_pos, *weights, h0=None, return_h=return_cache,
          return_conv_cache=return_cache, gate_branch=gate_branch)
    gate_branch = None
  if gate_branch is not None:
    y = ops.gelu_mul(y, gate_branch)
  if not return_cache:
    return y, None
  return y, RecurrentBlockCache(rg_lru_state=h, conv1d_state=conv_state)


class RecurrentBlock(nn.Module):
  """Griffin and Hawk's recurrent block."""

  def __init__(self, width, num_heads, lru_width=None, conv1d_temporal_width=4,
               final_w_init_variance_scale=1.0, device=None, dtype=None):
    super().__init__()
    self.width = width
    self.num_heads = num_heads
    self.lru_width = lru_width or width
    self.conv1d_temporal_width = conv1d_temporal_width
    self.final_w_init_variance_scale = final_w_init_variance_scale
    self.linear_y = nn.Linear(self.width, self.lru_width, device=device,
                              dtype=dtype)
    self.linear_x = nn.Linear(self.width, self.lru_width, device=device,
                              dtype=dtype)
    self.linear_out = nn.Linear(self.lru_width, self.width, device=device,
                                dtype=dtype)
    self.conv_1d = layers.Conv1D(width=self.lru_width,
                                 temporal_width=self.conv1d_temporal_width,
                                 device=device, dtype=dtype)
    self.rg_lru = layers.RGLRU(width=self.lru_width, num_heads=self.num_heads,
                               device=device, dtype=dtype)
    # True: a cached single-token call updates the cache tensors it is given
    # instead of returning new ones (set by callers that replay a captured
    # decode step on fixed buffers)
    self.decode_in_place = False
    # the linear layers for at most 64 rows (a decode step): linear_y and
    # linear_x as one pass over both weight matrices, linear_out as another
    self._rows_yx = ops.PackedLinear()
    self._rows_out = ops.PackedLinear()
    self.reset_parameters()

  def reset_parameters(self) -> None:
    self.w_init_(self.linear_x.weight)
    torch.nn.init.zeros_(self.linear_x.bias)
    self.w_init_(self.linear_y.weight)
    torch.nn.init.zeros_(self.linear_y.bias)
    self.out_w_init_(self.linear_out.weight)
    torch.nn.init.zeros_(self.linear_out.bias)
    self.conv_1d.reset_parameters()
    self.rg_lru.reset_parameters()

  def w_init_(self, w: torch.Tensor) -> None:
    torch.nn.init.normal_(w, mean=0.0, std=math.sqrt(1.0 / self.width))

  def out_w_init_(self, w: torch.Tensor) -> None:
    std = math.sqrt(self.final_w_init_variance_scale / self.lru_width)
    torch.nn.init.normal_(w, mean=0.0, std=std)

  def _behind_norm(self):
    """Weight rows of the layers that read a decode step's x in one launch, and
    whether they are the MLP's pair."""
    return 2 * self.lru_width, False

  def forward(self, x, segment_pos, cache=None, return_cache=True,
              defer_out=False):
    """defer_out: the caller adds the result to a residual and normalises it
    next (ops.add_rms_norm) and accepts it as ops.PartialSums, which is what
    it gets where that saves a pass (a few rows, bf16)."""
    if training.is_enabled():
      return self._forward_differentiable(x, segment_pos, cache, return_cache)
    if cache is not None and return_cache and not defer_out:
      done = self._step_natively(x, segment_pos, cache)
      if done is not None:
        y, h, conv_state = done
        return y, RecurrentBlockCache(rg_lru_state=h, conv1d_state=conv_state)
    in_place = self.decode_in_place and cache is not None and return_cache
    aside = None
    with torch.no_grad():
      # (a traced program keeps torch's own linear layers: the few-row
      # kernels are reached through ctypes, which a tracer cannot follow)
      few_rows = (
          not compiled.tracing() and
          ops.PackedLinear.usable(x, self.width, self.lru_width) and
          ops.PackedLinear.usable(x, self.lru_width, self.width))
      if few_rows:
        linear = self._modules
        w_y, b_y = _parameters(linear["linear_y"], "weight", "bias")
        w_x, b_x = _parameters(linear["linear_x"], "weight", "bias")
        w_out, b_out = _parameters(linear["linear_out"], "weight", "bias")
        # (a step in place: the conv state copied beside the layers, so that
        # the step's workgroups may share heads while they overwrite it)
        done = None
        if in_place and self.conv_1d.temporal_width == 4:
          done = self._rows_yx.beside(x, (w_y, w_x), (b_y, b_x),
                                      cache.conv1d_state)
        if done is not None:
          y, x, aside = done
        else:
          y, x = self._rows_yx(x, (w_y, w_x), (b_y, b_x))
      else:
        y, x = linears(ops.formed(x), self.linear_y, self.linear_x)
      # x * gelu(y) (modules.py:627-628, 644) is part of the core call: inside
      # the prefill kernel where that runs, one pass after it elsewhere
      x, new_cache = _recurrent_core(
          self.conv_1d, self.rg_lru, x, segment_pos, cache, return_cache,
          in_place, y, aside)
      if few_rows and defer_out and ops.PackedLinear.partial_slices(
          x, self.lru_width, self.width):
        x = self._rows_out.partial(x, (w_out,), (b_out,))
      elif few_rows:
        x = self._rows_out(x, (w_out,), (b_out,))
      else:
        x, = linears(x, self.linear_out)
    if not return_cache:
      return x, None
    return x, new_cache

  def _step_natively(self, x, segment_pos, cache):
    """A cached single-token call as one native call (csrc/host_ops.cpp), or
    None: before the linear layers are packed, and where the arguments are not
    as that call takes them."""
    yx, out = self._rows_yx._plan, self._rows_out._plan
    if (yx is None or out is None or compiled.tracing() or
        self.conv_1d.temporal_width != 4):
      return None
    return _lib.host().block_step(
        self._modules, yx, out, x, segment_pos, cache.conv1d_state,
        cache.rg_lru_state, self.decode_in_place)

  def _forward_differentiable(self, x, segment_pos, cache, return_cache):
    """The reference's op sequence (modules.py:605-655) under autograd."""
    if cache is not None:
      raise NotImplementedError("the differentiable path is prefill only")
    done = self._differentiable_natively(x, segment_pos, return_cache)
    if done is not None:
      x, h, conv_state = done
      if not return_cache:
        return x, None
      return x, RecurrentBlockCache(rg_lru_state=h, conv1d_state=conv_state)
    y = self.linear_y(x)
    x = self.linear_x(x)
    x, conv_state = self.conv_1d(x, segment_pos, None, return_cache)
    x, h = self.rg_lru(x, segment_pos, None, return_cache)
    x = self.linear_out(training.gelu_mul(x, y))  # x * gelu(y)
    if not return_cache:
      return x, None
    return x, RecurrentBlockCache(rg_lru_state=h, conv1d_state=conv_state)

  def _differentiable_natively(self, x, segment_pos, return_cache):
    """The whole block as one native autograd function (csrc/train_ops.cpp), or
    None: where a layer has been wrapped, hooked or replaced, or the arguments
    are not as that function takes them."""
    own = self._modules
    y, lx, out = own["linear_y"], own["linear_x"], own["linear_out"]
    conv, lru = own["conv_1d"], own["rg_lru"]
    if (compiled.tracing() or _global_hooks() or
        not (_as_written(y, nn.Linear) and _as_written(lx, nn.Linear) and
             _as_written(out, nn.Linear) and _as_written(conv, layers.Conv1D) and
             _as_written(lru, layers.RGLRU))):
      return None
    conv_w, conv_b, w_x, b_x, w_a, b_a, a_param = _core_weights(conv, lru)
    return _lib.host().train_block(
        x, segment_pos, *_parameters(y, "weight", "bias"),
        *_parameters(lx, "weight", "bias"), conv_w, conv_b, a_param, w_x, b_x,
        w_a, b_a, *_parameters(out, "weight", "bias"), bool(return_cache))

  @classmethod
  def init_cache(cls, batch_size, lru_width, dtype, conv1d_temporal_width=4,
                 device=None):
    return RecurrentBlockCache(
        rg_lru_state=layers.RGLRU.init_cache(batch_size=batch_size,
                                             width=lru_width, device=device),
        conv1d_state=layers.Conv1D.init_cache(
            batch_size=batch_size, width=lru_width, dtype=dtype,
            conv1d_temporal_width=conv1d_temporal_width, device=device),
    )

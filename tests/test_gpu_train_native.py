"""The native differentiable path (csrc/train_ops.cpp and the kernels of
csrc/rg_train.hip behind it) against the same block written in float32 tensor
ops under autograd, at the edges of its tiles: rows around multiples of 64 and
32, one token, one head, odd widths (float32), both position types."""

import pytest
import torch
from torch.nn import functional as F

import recurrentgemma_amd as rg
from recurrentgemma_amd import _lib
from recurrentgemma_amd import training

pytestmark = pytest.mark.gpu
BF16, F32 = torch.bfloat16, torch.float32


def close(got, want, dtype, what):
  got, want = got.detach().float(), want.detach().float()
  assert got.shape == want.shape, what
  err = (got - want).norm().item() / max(want.norm().item(), 1e-6)
  assert err < (2e-2 if dtype == BF16 else 2e-5), (what, err)


def reference(block, x, pos, p):
  """modules.py:605-655 of the reference in float32; p: name -> tensor."""
  gate = F.linear(x, p["linear_y.weight"], p["linear_y.bias"])
  h = F.linear(x, p["linear_x.weight"], p["linear_x.bias"])
  h = training.conv1d_tensor_ops(h, pos, p["conv_1d.w"], p["conv_1d.b"])
  h, last = training.rg_lru_tensor_ops(
      h, pos, *(p["rg_lru." + n] for n in (
          "a_param", "input_gate.w", "input_gate.b", "a_gate.w", "a_gate.b")))
  h = h * F.gelu(gate, approximate="tanh")
  return F.linear(h, p["linear_out.weight"], p["linear_out.bias"]), last


def make(B, T, width, heads, dtype, seed=0):
  torch.manual_seed(seed)
  block = rg.RecurrentBlock(width=width, num_heads=heads, device="cuda",
                            dtype=dtype)
  with torch.no_grad():
    for name, q in block.named_parameters():
      if name.endswith("bias") or name.endswith(".b"):
        q.normal_(std=0.1)
      if name.startswith("conv_1d.w"):
        q.normal_(std=0.5)
  x = torch.randn(B, T, width, device="cuda").to(dtype).requires_grad_()
  pos = torch.arange(T, device="cuda").expand(B, T).clone()
  pos[0, T // 2:] -= T // 2  # a second document
  return block, x, pos


SHAPES = [(1, 1, 256, 1, BF16), (1, 63, 256, 1, BF16), (3, 64, 512, 2, BF16),
          (1, 65, 256, 1, BF16), (2, 97, 768, 3, BF16), (5, 333, 512, 2, BF16),
          (1, 1, 48, 2, F32), (2, 130, 48, 2, F32), (3, 65, 512, 2, F32)]


@pytest.mark.parametrize("B,T,width,heads,dtype", SHAPES)
@pytest.mark.parametrize("pos_dtype", [torch.int32, torch.int64])
def test_block_gradients(B, T, width, heads, dtype, pos_dtype, monkeypatch):
  block, x, pos = make(B, T, width, heads, dtype)
  pos = pos.to(pos_dtype)
  # the native function takes the call: the general path is out of reach
  monkeypatch.setattr(training, "gelu_mul", None)
  with training.differentiable():
    y, cache = block(x, pos)
    dy = torch.randn_like(y)
    dh = torch.randn_like(cache.rg_lru_state)
    names = [n for n, _ in block.named_parameters()]
    wanted = [x] + [q for _, q in block.named_parameters()]
    got = torch.autograd.grad((y, cache.rg_lru_state), wanted, (dy, dh))
    p = {n: q.detach().float().requires_grad_() for n, q in
         block.named_parameters()}
    xf = x.detach().float().requires_grad_()
    yr, hr = reference(block, xf, pos, p)
    want = torch.autograd.grad((yr, hr), [xf] + [p[n] for n in names],
                               (dy.float(), dh))
  close(y, yr, dtype, "y")
  close(cache.rg_lru_state, hr, dtype, "h")
  assert cache.conv1d_state.shape == (B, 3, width)
  for name, g, w in zip(["x"] + names, got, want):
    assert g.dtype == dtype
    close(g, w, dtype, name)


@pytest.mark.parametrize("B,T,width,heads,dtype", SHAPES)
def test_rglru_gradients(B, T, width, heads, dtype):
  block, x, pos = make(B, T, width, heads, dtype)
  lru = block.rg_lru
  h0 = torch.randn(B, width, device="cuda").requires_grad_()
  with training.differentiable():
    y, h = lru(x, pos, h0)
    dy = torch.randn_like(y)
    params = list(lru.parameters())
    got = torch.autograd.grad((y,), [x, h0] + params, dy)
    copies = [q.detach().float().requires_grad_() for q in params]
    xf = x.detach().float().requires_grad_()
    hf = h0.detach().clone().requires_grad_()
    by = {n: c for (n, _), c in zip(lru.named_parameters(), copies)}
    yr, hr = training.rg_lru_tensor_ops(
        xf, pos, by["a_param"], by["input_gate.w"], by["input_gate.b"],
        by["a_gate.w"], by["a_gate.b"], hf)
    want = torch.autograd.grad((yr,), [xf, hf] + copies, dy.float())
  close(y, yr, dtype, "y")
  close(h, hr, dtype, "h")
  for i, (g, w) in enumerate(zip(got, want)):
    close(g, w, dtype, i)


# rows around one wave's batch (8), one step of a workgroup (32) and the edges
# of row ranges (128, 512 rows), one to sixteen ranges, the last one short or
# empty
@pytest.mark.parametrize("B,T,heads", [(1, 7, 1), (1, 31, 1), (1, 33, 2),
                                       (1, 129, 1), (3, 171, 1), (1, 2049, 1),
                                       (2, 350, 10), (1, 300, 16), (1, 161, 33)])
def test_float32_gate_weight_gradients(B, T, heads):
  test_rglru_gradients(B, T, 256 * heads, heads, F32)


# bf16, where each direction picks its own kernel: the backward one-pass (rows that
# end just before, at and just behind its steps of 256 tokens), neither (many
# short rows), only the backward (rows the last-level cache does not hold)
@pytest.mark.parametrize("B,T,width", [
    (2, 250, 256), (1, 255, 512), (3, 256, 256), (1, 511, 256), (2, 513, 256),
    (1, 1025, 512), (40, 7, 1024), (36, 100, 1024), (80, 1100, 512)])
def test_directions_on_kernels_of_their_own(B, T, width):
  test_rglru_gradients(B, T, width, width // 256, BF16)


def test_frozen_parts_and_wrapped_layers():
  """Only what needs a gradient gets one, and a hooked layer is called."""
  block, x, pos = make(2, 70, 512, 2, BF16)
  for q in block.parameters():
    q.requires_grad_(False)
  block.linear_y.bias.requires_grad_()
  with training.differentiable():
    y, _ = block(x.detach(), pos, return_cache=False)
    (alone,) = torch.autograd.grad(y.float().square().sum(),
                                   [block.linear_y.bias])
  called = []
  handle = block.linear_x.register_forward_hook(
      lambda *a: called.append(1))
  with training.differentiable():
    y2, _ = block(x.detach(), pos, return_cache=False)
    (hooked,) = torch.autograd.grad(y2.float().square().sum(),
                                    [block.linear_y.bias])
  handle.remove()
  assert called
  close(y, y2, BF16, "y")
  close(alone, hooked, BF16, "bias")
  # a tensor that does not start at 16 bytes takes the general path
  flat = torch.empty(x.numel() + 1, dtype=BF16, device="cuda")
  odd = flat[1:].view(x.shape).copy_(x.detach())
  assert _lib.host().train_block(
      odd, pos, *(getattr(block.linear_y, n) for n in ("weight", "bias")),
      *(getattr(block.linear_x, n) for n in ("weight", "bias")),
      block.conv_1d.w, block.conv_1d.b, block.rg_lru.a_param,
      block.rg_lru.input_gate.w, block.rg_lru.input_gate.b,
      block.rg_lru.a_gate.w, block.rg_lru.a_gate.b, block.linear_out.weight,
      block.linear_out.bias, False) is None


@pytest.mark.parametrize("pos_dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("B,T,width,heads,dtype", [
    (2, 97, 512, 2, BF16), (3, 65, 512, 2, F32), (2, 300, 48, 2, F32),
    (1, 33, 50, 2, F32)])
def test_positions_and_biases_may_be_written_to_before_the_backward(
    B, T, width, heads, dtype, pos_dtype):
  """The RG-LRU's backward reads the positions and gate biases its forward read,
  also where a caller has put the next batch's into the same buffers."""
  block, x, pos = make(B, T, width, heads, dtype)
  lru, pos = block.rg_lru, pos.to(pos_dtype)
  dy = torch.randn_like(x)
  wanted = [x] + list(lru.parameters())

  def gradients(overwrite):
    with training.differentiable():
      y, h = lru(x, pos)
      if overwrite:
        pos.fill_(1)
        with torch.no_grad():
          lru.input_gate.b.add_(1)
          lru.a_gate.b.add_(1)
      return torch.autograd.grad((y, h), wanted, (dy, torch.ones_like(h)))

  want = gradients(False)
  for g, w in zip(gradients(True), want):
    assert torch.equal(g, w)


@pytest.mark.parametrize("dtype", [BF16, F32])
def test_block_biases_may_be_written_to_before_the_backward(dtype):
  block, x, pos = make(2, 97, 512, 2, dtype)
  wanted = [x] + list(block.parameters())
  dy = torch.randn_like(x)

  def gradients(overwrite):
    with training.differentiable():
      y, _ = block(x, pos, return_cache=False)
      if overwrite:
        with torch.no_grad():
          for name, q in block.named_parameters():
            if name.endswith("bias") or name.endswith(".b"):
              q.add_(1)
      return torch.autograd.grad(y, wanted, dy)

  want = gradients(False)
  for g, w in zip(gradients(True), want):
    assert torch.equal(g, w)


def _calls(dtype):
  """One call of each native autograd function: (outputs, wanted) each."""
  block, x, pos = make(2, 97, 512, 2, dtype)
  h0 = torch.randn(2, 512, device="cuda").requires_grad_()
  a = torch.rand_like(x.detach()).requires_grad_()
  reset = pos == 0
  lru = block.rg_lru
  return {
      "scan": (lambda: rg.rnn_scan(x, a, reset, h0), [x, a, h0]),
      "rglru": (lambda: lru(x, pos, h0), [x, h0] + list(lru.parameters())),
      "block": (lambda: block(x, pos, return_cache=False)[:1],
                [x] + list(block.parameters()))}


def _gradients(call, wanted, pack, unpack):
  with training.differentiable():
    with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
      out = call()
    return torch.autograd.grad(out, wanted, [torch.ones_like(o) for o in out])


def _strided(t):
  return torch.stack([t, t], dim=-1)[..., 0]


def _off_by_one(t):
  flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
  return flat[1:].view(t.shape).copy_(t)


@pytest.mark.parametrize("dtype", [BF16, F32])
@pytest.mark.parametrize("name", ["scan", "rglru", "block"])
def test_saved_tensors_come_back_as_they_like(dtype, name):
  """What a hook returns for a saved tensor may lie anyhow; what is another
  tensor is refused before a kernel runs on it."""
  call, wanted = _calls(dtype)[name]
  keep = lambda t: t.detach()
  want = _gradients(call, wanted, keep, keep)
  for unpack in (_strided, _off_by_one, lambda t: t.cpu().cuda()):
    got = _gradients(call, wanted, keep, unpack)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
  for unpack in (lambda t: t[:1], lambda t: t.cpu(), lambda t: t.double(),
                 lambda t: t.flatten()):
    with pytest.raises(RuntimeError, match="came back from its hook"):
      _gradients(call, wanted, keep, unpack)


@pytest.mark.parametrize("name", ["scan", "rglru", "block"])
def test_failures_keep_their_exception(name):
  """A kernel's refusal in a backward pass is the package's exception, a hook's
  own exception stays what it is, in both directions."""
  call, wanted = _calls(BF16)[name]
  keep = lambda t: t.detach()

  def broken(t):
    raise ZeroDivisionError("from a hook")

  with pytest.raises(_lib.KernelError, match="came back from its hook"):
    _gradients(call, wanted, keep, lambda t: t.flatten())
  for hooks in ((broken, keep), (keep, broken)):
    with pytest.raises(ZeroDivisionError, match="from a hook"):
      _gradients(call, wanted, *hooks)

"""What the speed of this package is measured on: the calls its users make.

Six kinds of call, each through the package's public entry points:

  step      one cached token through the recurrent block (the RecurrentBlock
            module with its linear layers, or recurrent_core alone, as a caller
            with linear layers of its own uses it), new cache tensors returned
  prefill   recurrent_core over whole prompts, the state returned for the
            decode that follows
  attention LocalAttentionBlock over whole prompts, ring cache returned
  generate  Sampler.sample_tokens with a random-init model: prompt pass and
            greedy decoding
  train     forward and backward of RecurrentBlock or RGLRU inside
            training.differentiable()
  scan      rnn_scan, forward and backward or forward only

Widths, head counts, windows and vocabulary are those of the presets in
recurrentgemma_amd/griffin.py; batches and lengths those of the benchmark's
workloads and the tests, or generic ones.
"""

from __future__ import annotations

import math

import torch

import recurrentgemma_amd as rg
from recurrentgemma_amd import training

# width of the recurrent path and its heads: 2B and 9B presets (256-wide
# heads), paper presets (176-wide heads)
_SHAPES = ((2560, 10), (4096, 16), (5632, 32))
_DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed():
  return [
      # a chat with one user: the block's decode step, launched from Python
      dict(name="step_one_user", kind="step", via="block", batch=1, width=2560,
           heads=10, dtype="bf16"),
      # a serving batch of 256 sequences at the 9B width
      dict(name="step_256_users", kind="step", via="core", batch=256,
           width=4096, heads=16, dtype="bf16"),
      # three short prompts of different lengths, left-padded as the sampler
      # pads them
      dict(name="prefill_chat_prompts", kind="prefill", batch=3, tokens=333,
           width=2560, heads=10, dtype="bf16", layout="padded", join=True),
      # packed documents at the 2B width
      dict(name="prefill_2b_documents", kind="prefill", batch=8, tokens=4096,
           width=2560, heads=10, dtype="bf16", layout="documents", join=True),
      # the headline: long prompts at the 9B width
      dict(name="prefill_9b", kind="prefill", batch=16, tokens=8192,
           width=4096, heads=16, dtype="bf16", layout="single", join=False),
      # the paper presets' recurrent width, whose heads are 176 wide
      dict(name="prefill_paper", kind="prefill", batch=4, tokens=2048,
           width=5632, heads=32, dtype="bf16", layout="single", join=True),
      # float32, one short prompt: checking results, small-scale research
      dict(name="prefill_f32", kind="prefill", batch=1, tokens=512, width=2560,
           heads=10, dtype="f32", layout="single", join=False),
      # the attention block of the 2B model over prompts that fill its window
      dict(name="attention_prompts", kind="attention", batch=8, tokens=2047,
           width=2560, heads=10, window=2048, layout="padded"),
      # answering a batch of prompts with the 2B model, every token's logits
      # kept for scoring
      dict(name="generate_2b", kind="generate", batch=16, tokens=1000,
           new_tokens=32, blocks=26, width=2560, heads=10, lru_width=2560,
           logits=True),
      # fine-tuning: the block forward and backward on packed documents
      dict(name="train_block", kind="train", via="block", batch=4, tokens=2048,
           width=2560, heads=10, dtype="bf16", layout="documents"),
      # the RG-LRU as a layer in a float32 model, odd sizes
      dict(name="train_rglru_f32", kind="train", via="rglru", batch=3,
           tokens=1001, width=2560, heads=10, dtype="f32",
           layout="documents"),
      # the bare recurrence in a layer of the user's own
      dict(name="scan_train", kind="scan", batch=4, tokens=2048, width=2560,
           dtype="bf16", backward=True),
  ]


def _spread(rng, lo, hi):
  """A whole number from lo to hi, even over its logarithm."""
  return max(lo, min(hi, int(round(math.exp(
      rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
  kind = rng.choice(("step", "step", "prefill", "prefill", "prefill",
                     "attention", "generate", "train", "train", "scan"))
  width, heads = rng.choice(_SHAPES[:2])
  layout = rng.choice(("single", "documents", "padded"))
  if kind == "step":
    via = rng.choice(("block", "core"))
    return dict(kind=kind, via=via, width=width, heads=heads,
                batch=_spread(rng, 1, 64 if via == "block" else 512),
                dtype=rng.choice(("bf16", "bf16", "bf16", "f32")))
  if kind == "prefill":
    width, heads = rng.choice(_SHAPES)
    dtype = "bf16" if heads == 32 else rng.choice(("bf16",) * 3 + ("f32",))
    batch = _spread(rng, 1, 64)
    most = (16384 if dtype == "f32" else 131072) // batch
    return dict(kind=kind, batch=batch, tokens=_spread(rng, 1, min(8192, most)),
                width=width, heads=heads, dtype=dtype, layout=layout,
                join=rng.choice((True, False)))
  if kind == "attention":
    batch = _spread(rng, 1, 32)
    return dict(kind=kind, batch=batch, width=width, heads=heads, window=2048,
                tokens=_spread(rng, 65, min(8192, 65536 // batch)),
                layout=layout)
  if kind == "generate":
    blocks = rng.choice((3, 6, 8, 12))
    return dict(kind=kind, batch=_spread(rng, 1, 64), blocks=blocks,
                tokens=_spread(rng, 8, 512), new_tokens=_spread(rng, 8, 40),
                width=2560, heads=10, lru_width=2560,
                logits=rng.choice((True, False)))
  if kind == "train":
    batch = _spread(rng, 1, 16)
    return dict(kind=kind, via=rng.choice(("block", "rglru")), batch=batch,
                tokens=_spread(rng, 64, 8192 // batch), width=width,
                heads=heads, dtype=rng.choice(("bf16", "bf16", "f32")),
                layout=layout)
  batch = _spread(rng, 1, 16)
  return dict(kind=kind, batch=batch, tokens=_spread(rng, 64, 16384 // batch),
              width=rng.choice((512, 1000, 2048, 2560, 4096)),
              dtype=rng.choice(("bf16", "f32")),
              backward=rng.choice((True, True, False)))


def _positions(case, gen):
  """[B, T] int32 position of every token in its document."""
  batch, tokens = case["batch"], case["tokens"]
  at = torch.arange(tokens, device="cuda", dtype=torch.int32).expand(
      batch, tokens)
  if case["layout"] == "single":
    return at.contiguous()
  if case["layout"] == "padded":
    # left-padded prompts of half to full length, -1 on the padding
    pads = torch.randint(0, tokens // 2 + 1, (batch, 1), generator=gen,
                         device="cuda", dtype=torch.int32)
    pads[0] = 0
    return (at - pads).clamp_(min=-1)
  # packed documents, lengths geometric with a mean of a quarter of the row
  # (at most 1024)
  starts = torch.rand(batch, tokens, generator=gen, device="cuda") < (
      1.0 / max(2, min(1024, tokens // 4)))
  starts[:, 0] = True
  start_at = torch.cummax(torch.where(starts, at, torch.zeros_like(at)),
                          dim=1).values
  return (at - start_at).contiguous()


def _normal(gen, shape, dtype, std=1.0):
  return (torch.randn(shape, generator=gen, device="cuda") * std).to(dtype)


def _recurrent_block(case, gen):
  dtype = _DTYPES[case["dtype"]]
  block = rg.RecurrentBlock(width=case["width"], num_heads=case["heads"],
                            device="cuda", dtype=dtype)
  with torch.no_grad():  # biases as a trained model has them
    for bias in (block.linear_x.bias, block.linear_y.bias,
                 block.linear_out.bias, block.conv_1d.b,
                 block.rg_lru.input_gate.b, block.rg_lru.a_gate.b):
      bias.copy_(_normal(gen, bias.shape, dtype, 0.1))
  return block


def prepare(case, seed):
  """The modules with their parameters, and the inputs of one call."""
  gen = torch.Generator(device="cuda").manual_seed(seed)
  with torch.random.fork_rng(devices=[torch.cuda.current_device()]):
    torch.manual_seed(seed)  # the modules' own initialisation
    return _prepare(case, gen)


def _prepare(case, gen):
  kind = case["kind"]
  batch = case["batch"]
  state = dict(case)
  if kind == "generate":
    cycle = (rg.TemporalBlockType.RECURRENT, rg.TemporalBlockType.RECURRENT,
             rg.TemporalBlockType.ATTENTION)
    config = rg.GriffinConfig.from_preset(
        rg.Preset.RECURRENT_GEMMA_2B_V1)._replace(
            width=case["width"], mlp_expanded_width=3 * case["width"],
            num_heads=case["heads"], lru_width=case["lru_width"],
            block_types=tuple(cycle[i % 3] for i in range(case["blocks"])))
    model = rg.Griffin(config, device="cuda", dtype=torch.bfloat16).eval()
    state["sampler"] = rg.Sampler(model, use_graph=True)
    state["prompts"] = torch.randint(
        1, config.vocab_size, (batch, case["tokens"]), generator=gen,
        device="cuda", dtype=torch.int32)
    lengths = torch.randint((case["tokens"] + 1) // 2, case["tokens"] + 1,
                            (batch,), generator=gen, device="cuda",
                            dtype=torch.int32)
    lengths[0] = case["tokens"]
    state["lengths"] = lengths
    return state

  dtype = _DTYPES[case.get("dtype", "bf16")]
  width, tokens = case["width"], case.get("tokens", 1)
  shape = (batch, tokens, width)
  if kind == "attention":
    state["block"] = rg.LocalAttentionBlock(
        width=width, num_heads=case["heads"], window_size=case["window"],
        device="cuda", dtype=dtype)
    state["x"] = _normal(gen, shape, dtype)
    state["pos"] = _positions(case, gen)
    return state
  if kind == "scan":
    # coefficients as the RG-LRU makes them: mostly in 0.9 .. 1
    a = torch.rand(shape, generator=gen, device="cuda").mul_(0.1).add_(0.9)
    state["a"] = a.to(dtype)
    state["x"] = _normal(gen, shape, dtype, 0.3)
    state["reset"] = torch.rand(batch, tokens, generator=gen,
                                device="cuda") < 1.0 / 512
    state["h0"] = _normal(gen, (batch, width), torch.float32)
    if case["backward"]:
      state["dy"] = _normal(gen, shape, dtype)
      for name in ("x", "a", "h0"):
        state[name].requires_grad_(True)
    return state

  state["block"] = _recurrent_block(case, gen)
  state["x"] = _normal(gen, shape, dtype)
  if kind == "step":
    state["pos"] = torch.randint(1, 4096, (batch, 1), generator=gen,
                                 device="cuda", dtype=torch.int32)
    state["cache"] = rg.RecurrentBlockCache(
        rg_lru_state=_normal(gen, (batch, width), torch.float32),
        conv1d_state=_normal(gen, (batch, 3, width), dtype))
    return state
  state["pos"] = _positions(case, gen)
  if kind == "prefill":
    state["gate"] = _normal(gen, shape, dtype) if case["join"] else None
    return state
  # train
  state["dy"] = _normal(gen, shape, dtype)
  state["x"].requires_grad_(True)
  module = (state["block"] if case["via"] == "block" else
            state["block"].rg_lru)
  state["module"] = module
  state["wanted"] = [state["x"]] + list(module.parameters())
  return state


def run(state):
  kind = state["kind"]
  if kind == "step":
    block = state["block"]
    if state["via"] == "block":
      with torch.no_grad():
        y, cache = block(state["x"], state["pos"], state["cache"])
    else:
      y, cache = rg.recurrent_core(block.conv_1d, block.rg_lru, state["x"],
                                   state["pos"], state["cache"])
    return y, cache
  if kind == "prefill":
    block = state["block"]
    return rg.recurrent_core(block.conv_1d, block.rg_lru, state["x"],
                             state["pos"], gate_branch=state["gate"])
  if kind == "attention":
    with torch.no_grad():
      return state["block"](state["x"], state["pos"])
  if kind == "generate":
    return state["sampler"].sample_tokens(
        state["prompts"], state["lengths"], state["new_tokens"],
        return_logits=state["logits"])
  if kind == "train":
    with training.differentiable():
      y, _ = state["module"](state["x"], state["pos"], return_cache=False)
      grads = torch.autograd.grad(y, state["wanted"], state["dy"])
    return y, grads
  if not state["backward"]:
    return rg.rnn_scan(state["x"], state["a"], state["reset"], state["h0"])
  with training.differentiable():
    y, h_last = rg.rnn_scan(state["x"], state["a"], state["reset"],
                            state["h0"])
    grads = torch.autograd.grad(y, (state["x"], state["a"], state["h0"]),
                                state["dy"])
  return y, h_last, grads


def work(case):
  """One pass: inputs and parameters read once, outputs written once, and the
  multiply-adds of the matrix products (forward 1, backward 2 times)."""
  kind, batch = case["kind"], case["batch"]
  width, heads = case["width"], case.get("heads", 1)
  size = 4 if case.get("dtype") == "f32" else 2
  tokens = case.get("tokens", 1)
  rows = batch * tokens
  n = rows * width
  gates = 2 * width * (width // heads)      # weights of both projections
  states = batch * width * (4 + 3 * size)   # float32 state, 3 conv rows
  if kind == "step":
    nbytes = size * (2 * n + gates) + 2 * states
    flops = 2 * batch * gates
    if case["via"] == "block":
      nbytes += size * 3 * width * width
      flops += 6 * batch * width * width
    return {"bytes": nbytes, "flops": flops}
  if kind == "prefill":
    return {"bytes": size * ((3 if case["join"] else 2) * n + gates) +
                     4 * rows + states,
            "flops": 2 * rows * gates}
  if kind == "attention":
    head = width // heads
    weights = 2 * width * width + 2 * width * head
    window = case["window"]
    short = min(tokens, window)
    pairs = short * (short + 1) // 2 + (tokens - short) * window
    return {"bytes": 2 * (2 * n + weights + 2 * batch * window * head) +
                     4 * rows,
            "flops": 2 * rows * weights + 4 * batch * pairs * width}
  if kind == "generate":
    steps, blocks = case["new_tokens"], case["blocks"]
    head = width // heads
    recurrent = blocks - blocks // 3
    mlp = 9 * width * width
    weights = (recurrent * (3 * width * width + gates) +
               (blocks // 3) * (2 * width * width + 2 * width * head) +
               blocks * mlp)
    table = 256_000 * width
    # the prompt pass reads the weights once, every new token once more (and
    # the token table for its logits), and the rings of the attention blocks
    rings = (blocks // 3) * 2 * batch * head * tokens
    logits = batch * 256_000 if case["logits"] else 0
    return {"bytes": 2 * (weights + steps * (weights + table + rings + logits)),
            "flops": 2 * batch * ((tokens + steps - 1) * weights +
                                  steps * table)}
  if kind == "train":
    weights = gates + (3 * width * width if case["via"] == "block" else 0)
    return {"bytes": size * (4 * n + 2 * weights) + 4 * rows,
            "flops": 6 * rows * weights}
  return {"bytes": size * (6 if case["backward"] else 3) * n + rows +
                   batch * width * (12 if case["backward"] else 8),
          "flops": (6 if case["backward"] else 2) * n}


def tolerance(case):
  if case["kind"] == "generate":
    # token ids (a tie of two logits may go either way), and logits behind up
    # to 26 blocks in bf16, each of which rounds some ten tensors
    return {"rel": 3e-2, "differ": 0.01}
  if case.get("dtype") == "f32":
    return {"rel": 1e-5, "max": 1e-3}
  return {"rel": 1e-2}

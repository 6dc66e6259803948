"""Linear layers of many rows (csrc/rg_matmul.hip) against float64, through the C calls
that the modules make: forward, both directions back, the MLP's pair.  Sizes at the edges
of the tiles (64, 128 and 256 rows, 64 to 320 columns), of the steps (64 of the contraction)
and of the 8 values of a load."""

import ctypes

import pytest
import torch

from recurrentgemma_amd import _lib
from recurrentgemma_amd import ops

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def normal(seed, *shape):
  g = torch.Generator(device="cuda").manual_seed(seed)
  return torch.randn(shape, generator=g, device="cuda").to(BF16)


def pointers(tensors):
  return (ctypes.c_void_p * len(tensors))(
      *[None if t is None else t.data_ptr() for t in tensors])


def ints(values):
  return (ctypes.c_int * len(values))(*values)


def stream():
  return torch.cuda.current_stream().cuda_stream


def guarded(rows, cols):
  """[rows, cols] to be written whole, and the buffer it lies in: 4096 marks behind it."""
  buf = torch.full((rows * cols + 4096,), 7.0, device="cuda", dtype=BF16)
  return buf[:rows * cols].view(rows, cols), buf


def check(got, terms, buf, extra=0.0):
  """got against the float64 sum of terms, products (a, b) of matrices.  bf16 rounds the
  result by at most 2^-9 of it (2^-8 where it is rounded up to a power of two's edge),
  and K float32 sums are off by at most K 2^-24 of the sum of magnitudes."""
  want = sum(a.double() @ b.double() for a, b in terms) + extra
  size = sum(a.double().abs() @ b.double().abs() for a, b in terms)
  depth = sum(a.shape[1] for a, _ in terms)
  bound = want.abs() * 2.0 ** -8 + size * depth * 2.0 ** -24 + 1e-30
  assert ((got.double() - want).abs() <= bound).all()
  assert (buf[got.numel():] == 7.0).all()


# rows, features in, features out
FORWARD = [(1, 64, 8), (63, 64, 72), (65, 448, 136), (127, 128, 264), (129, 192, 256),
           (256, 64, 320), (257, 320, 328), (1000, 2560, 512), (999, 512, 2560),
           # tiles of 128 x 320, 256 x 320, 128 x 256 and 256 x 256
           (4095, 192, 2560), (8191, 192, 2560), (2049, 1024, 2560), (4097, 1024, 2568)]


@pytest.mark.parametrize("M,K,N", FORWARD)
@pytest.mark.parametrize("count", [1, 3])
@pytest.mark.parametrize("bias", [True, False])
def test_forward(M, K, N, count, bias):
  x = normal(1, M, K)
  n = [N, 8, 264][:count]
  w = [normal(2 + i, n[i], K) for i in range(count)]
  b = [normal(7 + i, n[i]) for i in range(count)] if bias else None
  out = [guarded(M, n[i]) for i in range(count)]
  _lib.check(_lib.lib().rg_linear_many(
      x.data_ptr(), M, K, count, pointers(w), pointers(b) if bias else None,
      pointers([o for o, _ in out]), ints(n), _lib.RG_DTYPE_BF16, stream()))
  for i in range(count):
    check(out[i][0], [(x, w[i].t())], out[i][1], b[i].double() if bias else 0.0)


@pytest.mark.parametrize("M,K,N", FORWARD)
@pytest.mark.parametrize("two", [False, True])
def test_back(M, K, N, two):
  dy, w = normal(1, M, K), normal(2, K, N)
  dy2, w2 = (normal(3, M, K), normal(4, K, N)) if two else (None, None)
  dx, buf = guarded(M, N)
  p = lambda t: None if t is None else t.data_ptr()
  _lib.check(_lib.lib().rg_linear_back(
      p(dy), p(w), p(dy2), p(w2), p(dx), M, K, N, _lib.RG_DTYPE_BF16, stream()))
  check(dx, [(dy, w)] + ([(dy2, w2)] if two else []), buf)


# rows; features out, features in
@pytest.mark.parametrize("M", [1, 63, 64, 65, 191, 1003])
@pytest.mark.parametrize("shapes", [[(8, 8)], [(264, 328)], [(256, 320), (8, 264), (512, 256)],
                                    [(2560, 2560)] * 3, [(4096, 4104)]])
def test_weight_gradients(M, shapes):
  dy = [normal(1 + i, M, n) for i, (n, _) in enumerate(shapes)]
  x = [normal(9 + i, M, k) for i, (_, k) in enumerate(shapes)]
  dw = [guarded(n, k) for n, k in shapes]
  _lib.check(_lib.lib().rg_linear_weight_grads(
      pointers(dy), pointers(x), pointers([d for d, _ in dw]),
      ints([n for n, _ in shapes]), ints([k for _, k in shapes]), len(shapes), M,
      _lib.RG_DTYPE_BF16, stream()))
  for i in range(len(shapes)):
    check(dw[i][0], [(dy[i].t(), x[i])], dw[i][1])


@pytest.mark.parametrize("M,K,N", FORWARD)
@pytest.mark.parametrize("bias", [True, False])
def test_gelu_pair(M, K, N, bias):
  x, w = normal(1, M, K), normal(2, 2, K, N) * 0.1
  b = normal(3, 2, N) if bias else None
  out, buf = guarded(M, N)
  _lib.check(_lib.lib().rg_linear_gelu_pair(
      x.data_ptr(), w.data_ptr(), b.data_ptr() if bias else None, out.data_ptr(), M, K, N,
      _lib.RG_DTYPE_BF16, stream()))
  # the two products on their own, each checked, then the join's kernel: the same bits
  parts = [guarded(M, N) for _ in range(2)]
  wt = [w[i].t().contiguous() for i in range(2)]
  for i in range(2):
    _lib.check(_lib.lib().rg_linear_many(
        x.data_ptr(), M, K, 1, pointers([wt[i]]), pointers([b[i].clone()]) if bias else None,
        pointers([parts[i][0]]), ints([N]), _lib.RG_DTYPE_BF16, stream()))
    check(parts[i][0], [(x, wt[i].t())], parts[i][1], b[i].double() if bias else 0.0)
  assert torch.equal(out, ops.gelu_mul(parts[1][0], parts[0][0]))
  assert (buf[out.numel():] == 7.0).all()


def test_infinities_stay_in_their_row_and_column():
  M, K, N = 300, 192, 520
  x, w = normal(1, M, K), normal(2, N, K)
  clean = x @ w.t()
  x[257, 5], w[130, 64] = float("inf"), float("nan")
  out, _ = guarded(M, N)
  _lib.check(_lib.lib().rg_linear_many(
      x.data_ptr(), M, K, 1, pointers([w]), None, pointers([out]), ints([N]),
      _lib.RG_DTYPE_BF16, stream()))
  bad = ~torch.isfinite(out)
  want = torch.zeros_like(bad)
  want[257], want[:, 130] = True, True
  assert torch.equal(bad, want)
  assert (out[~bad].double() - clean[~bad].double()).abs().max() < 0.5


def test_what_does_not_fit_is_refused():
  x, w, out = normal(1, 64, 96), normal(2, 64, 96), normal(3, 64, 64)
  rc = _lib.lib().rg_linear_many(x.data_ptr(), 64, 96, 1, pointers([w]), None,
                                 pointers([out]), ints([64]), _lib.RG_DTYPE_BF16, stream())
  assert rc != _lib.RG_OK  # 96 is no multiple of 64
  assert not _lib.lib().rg_linear_many_pays(64, 96, 1, ints([64]), _lib.RG_DTYPE_BF16)
  assert not _lib.lib().rg_linear_many_pays(8192, 2560, 1, ints([2560]), _lib.RG_DTYPE_F32)


def test_layers_of_the_modules(monkeypatch):
  """Calls that take the launches, and those that must not: a hooked layer, a
  layer under autocast, weights that want gradients, a view."""
  from recurrentgemma_amd import griffin, modules
  layers = [torch.nn.Linear(2560, n, device="cuda", dtype=BF16) for n in (2560, 2560)]
  mlp = griffin.MLPBlock(512, 1536, device="cuda", dtype=BF16)
  x, xm = normal(1, 8, 512, 2560), normal(2, 2, 2048, 512)
  taken = []
  many, pair = ops.linear_many, ops.linear_gelu_pair
  note = lambda f: lambda *a: (taken.append(f(*a) is not None), f(*a))[1]
  monkeypatch.setattr(ops, "linear_many", note(many))
  monkeypatch.setattr(ops, "linear_gelu_pair", note(pair))

  def run(want):
    taken.clear()
    out = modules.linears(x, *layers)
    assert taken == want
    for y, layer in zip(out, layers):
      ref = x.double() @ layer.weight.double().t() + layer.bias.double()
      assert ((y.double() - ref).norm() / ref.norm()).item() < 4e-3  # one rounding
    return out

  with torch.no_grad():
    run([True])
    called = []
    h = layers[1].register_forward_hook(lambda *a: called.append(1))
    run([])
    assert called
    h.remove()
    with torch.autocast("cuda", dtype=BF16):
      run([False])
    x = normal(1, 8, 512, 2568)[..., 8:]
    run([False])
    taken.clear()
    out = mlp(xm)
    assert taken[0]
    gate, up = mlp.ffw_up(xm)
    ref = mlp.ffw_down(ops.gelu_mul(up, gate))
    assert ((out.double() - ref.double()).norm() / ref.double().norm()).item() < 6e-3
  x = normal(1, 8, 512, 2560)
  run([False])
  assert all(y.requires_grad for y in modules.linears(x, *layers))

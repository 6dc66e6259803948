// The differentiable calls (training.differentiable()) as native autograd
// functions: the bare recurrence, the RG-LRU, and the whole recurrent block.
//
// One training step of the block through one Python autograd function per
// operator is 26 to 60 launches and about as many allocations and interpreter
// rounds; float32 RG-LRU at B3 T1001 W2560 spent 640 us of host time on 560 us
// of kernels.  As one function per direction the passes in between can also be
// joined: bias gradients come out of the kernels that write or read the tensor
// anyway, input gradients accumulate where they are, and the reductions left
// share one launch.
//
// As in host_ops.cpp each entry serves the ordinary case and answers None
// otherwise; training.py then takes the general path.
#include "host_call.h"

#include <ATen/autocast_mode.h>
#include <torch/csrc/autograd/custom_function.h>

#include "rg_internal.h"
#include "rg_package_calls.h"

namespace rg_host {
namespace {

using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;
// (an absent last argument is no input edge: the indices before it stay)
using OptTensor = std::optional<Tensor>;

// Raised without the GIL, also on autograd's threads.
void check(int rc) {
  if (rc != RG_OK)
    throw KernelFailure("librg_lru status " + std::to_string(rc) + ": " +
                        rg_last_error());
}
void check_hip(hipError_t e) {
  if (e != hipSuccess)
    throw KernelFailure(std::string("librg_lru launch: ") + hipGetErrorString(e));
}

struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

Tensor empty(at::IntArrayRef shape, at::ScalarType t, const Tensor& like) {
  return at::detail::empty_cuda(shape, t, like.device(), std::nullopt);
}
Tensor empty(at::IntArrayRef shape, const Tensor& like) {
  return empty(shape, like.scalar_type(), like);
}
const void* in(const Tensor& t) {
  return t.defined() ? t.const_data_ptr() : nullptr;
}
void* out(const Tensor& t) { return t.defined() ? t.mutable_data_ptr() : nullptr; }

// A tensor from elsewhere in the graph as the kernels take it.
Tensor dense_tensor(const Tensor& t, at::ScalarType dtype) {
  if (t.scalar_type() == dtype && t.is_contiguous() &&
      !(reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15u))
    return t;
  return t.to(dtype).clone(at::MemoryFormat::Contiguous);
}

// The saved tensors of a backward pass.  Under saved_tensors_hooks they are what
// a hook returned, which may lie otherwise than what was saved (a copy is made)
// or be something else (refused: the kernels count on sizes and types).  One of
// them, [B, T, W], gives the sizes, type and device, the others have to fit.
struct Saved {
  variable_list v;
  Tensor root;
  int64_t B, T, W;
  Saved(AutogradContext* ctx, int at) : v(ctx->get_saved_variables()) {
    const Tensor& r = v[at];
    fits(r.defined() && r.is_cuda() &&
         r.device().index() == c10::hip::current_device() &&
         (r.scalar_type() == at::kBFloat16 || r.scalar_type() == at::kFloat) &&
         r.dim() == 3 && r.numel() > 0);
    for (int i = 0; i < 3; ++i) fits(r.size(i) <= INT32_MAX);
    root = dense_tensor(r, r.scalar_type());
    B = r.size(0);
    T = r.size(1);
    W = r.size(2);
  }
  static void fits(bool ok) {
    if (!ok)
      throw KernelFailure(
          "a tensor saved for the backward pass came back from its hook as "
          "another one");
  }
  Tensor get(int i, at::IntArrayRef shape, at::ScalarType t) const {
    fits(v[i].defined() && v[i].sizes() == shape && v[i].scalar_type() == t &&
         v[i].device() == root.device());
    return dense_tensor(v[i], t);
  }
  Tensor get(int i, at::IntArrayRef shape) const {
    return get(i, shape, root.scalar_type());
  }
  Tensor like_root(int i) const { return get(i, root.sizes()); }
  Tensor state(int i) const {  // [B, W], if there is one
    return v[i].defined() ? get(i, {B, W}, at::kFloat) : Tensor();
  }
  // a weight of the gate projections
  Tensor gate_weight(int i) const {
    fits(v[i].defined() && v[i].dim() == 3);
    const int64_t H = v[i].size(0), bw = v[i].size(1);
    fits(H > 0 && H * bw == W &&
         (root.scalar_type() == at::kFloat || bw == 256));
    return get(i, {H, bw, bw});
  }
};
// ... and the gradient of an output of these sizes, if there is one
Tensor grad_of(const Tensor& grad, at::IntArrayRef shape, at::ScalarType t) {
  if (!grad.defined()) return grad;
  Saved::fits(grad.sizes() == shape);
  return dense_tensor(grad, t);
}

struct Dims {
  int64_t B, T, W;
  int code;
  hipStream_t stream;
  explicit Dims(const Tensor& x)
      : B(x.size(0)),
        T(x.size(1)),
        W(x.size(2)),
        code(dtype_code(x)),
        stream(c10::hip::getCurrentHIPStream(x.device().index()).stream()) {}
  int64_t M() const { return B * T; }
};
int seg_kind(const Tensor& pos) { return pos.scalar_type() == at::kLong ? 1 : 0; }

// What the backward pass of the RG-LRU reads besides the tensors whose values
// it may count on (autograd raises if those were written to in between): a
// caller's positions and biases may hold the next batch's by then.
struct Kept {
  Tensor starts;  // [B, T] bool, where documents start
  Tensor bias;    // [2, W] float32 where the pre-activations are without them
};

// ---------------------------------------------------------- bare recurrence --

void scan_forward(const Tensor& x, const Tensor& a, const Tensor& reset,
                  const Tensor& h0, const Tensor& y, const Tensor& h) {
  const Dims d(x);
  const size_t bytes = rg_linear_scan_best_workspace_bytes(
      (int)d.B, (int)d.T, (int)d.W, d.code, 0);
  Tensor ws;
  if (bytes) ws = empty({(int64_t)bytes}, at::kByte, x);
  check(bytes ? rg_linear_scan_split(in(x), in(a), in(reset), in(h0), out(y),
                                     out(h), out(ws), bytes, (int)d.B, (int)d.T,
                                     (int)d.W, d.code, d.stream)
              : rg_linear_scan(in(x), in(a), in(reset), in(h0), out(y), out(h),
                               (int)d.B, (int)d.T, (int)d.W, d.code, d.stream));
}

struct Scan : Function<Scan> {
  static variable_list forward(AutogradContext* ctx, Tensor x, Tensor a,
                               Tensor reset, OptTensor h0_) {
    const Tensor h0 = h0_.value_or(Tensor());
    ctx->set_materialize_grads(false);
    Tensor y = empty(x.sizes(), x);
    Tensor h = empty({x.size(0), x.size(2)}, at::kFloat, x);
    scan_forward(x, a, reset, h0, y, h);
    ctx->save_for_backward({a, reset, y, h0});
    return {y, h};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    at::AutoGradMode off(false);
    const Saved s(ctx, 2);
    const Tensor a = s.like_root(0), reset = s.get(1, {s.B, s.T}, at::kBool),
                 y = s.root, h0 = s.state(3);
    const Dims d(y);
    Tensor dy = grad_of(grads[0], y.sizes(), y.scalar_type());
    if (!dy.defined()) dy = at::zeros_like(y);
    const Tensor dh = grad_of(grads[1], {d.B, d.W}, at::kFloat);
    Tensor dx = empty(y.sizes(), y), da = empty(y.sizes(), y), dh0;
    if (h0.defined()) dh0 = empty(h0.sizes(), h0);
    const size_t bytes = rg_linear_scan_best_workspace_bytes(
        (int)d.B, (int)d.T, (int)d.W, d.code, 1);
    Tensor ws;
    if (bytes) ws = empty({(int64_t)bytes}, at::kByte, y);
    check(rg_linear_scan_backward_best(in(dy), in(a), in(reset), in(y), in(h0),
                                       in(dh), out(dx), out(da), out(dh0), out(ws),
                                       bytes, (int)d.B, (int)d.T, (int)d.W, d.code,
                                       d.stream));
    return {dx, da, Tensor(), dh0};
  }
};

// ------------------------------------------------------------------ RG-LRU --

struct GateWeights {
  Tensor a_param, w_x, b_x, w_a, b_a;
};

// Which directions of the recurrence run on the one-pass kernels, which take the
// document starts from the positions themselves and, float32, add the gates'
// biases to the pre-activations: both directions or neither there.
struct OnTiles {
  bool forward, backward;
};
OnTiles on_tiles(const Dims& d) {
  auto serve = [&](rg::ScanTileMode mode) {
    return rg::scan_tiles_serve((int)d.B, (int)d.T, (int)d.W, d.code, mode);
  };
  if (d.code == RG_DTYPE_F32) {
    const bool both = serve(rg::kTilesFwdGated) && serve(rg::kTilesPairGated);
    return {both, both};
  }
  const bool dealt = rg_scan_deal_bytes((int)d.B, (int)d.T, (int)d.W, d.code,
                                        rg::kTilesFwdGated) > 0;
  return {dealt || serve(rg::kTilesFwdGated), serve(rg::kTilesBwdGated)};
}

// Workspace of the one-pass kernels' dealt form, where that is the faster one.
Tensor deal_workspace(const Dims& d, rg::ScanTileMode mode, const Tensor& like) {
  const size_t bytes = rg_scan_deal_bytes((int)d.B, (int)d.T, (int)d.W, d.code, mode);
  return bytes ? empty({(int64_t)bytes}, at::kByte, like) : Tensor();
}

// Kept::bias of a backward pass
Tensor kept_bias(const Saved& s, int i) {
  const Dims d(s.root);
  if (d.code != RG_DTYPE_F32 || !on_tiles(d).backward) return Tensor();
  return s.get(i, {2, s.W});
}

// What the block's sums over rows take.
bool block_sums_serve(int64_t B, int64_t T, int64_t W, int64_t D, int code) {
  const int per = code == RG_DTYPE_F32 ? 4 : 8;
  return W % per == 0 && D % per == 0 &&
         (B * T + rg::kColSumRows - 1) / rg::kColSumRows <= 65535 &&
         rg::conv1d_backward_sums_dx((int)B, (int)T, (int)W, 4, code);
}

// [M, W] as a batch of heads [H, M, bw], no copy
Tensor by_head(const Tensor& t, int64_t H) {
  const int64_t bw = t.size(-1) / H;
  return t.view({-1, H, bw}).transpose(0, 1);
}

void gated_forward(const Tensor& x, const Tensor& pos, const GateWeights& g,
                   const Tensor& h0, const Tensor& gx, const Tensor& ga,
                   const Tensor& y, const Tensor& h, Kept& kept) {
  const Dims d(x);
  const int64_t H = g.w_x.size(0);
  const bool tiles = on_tiles(d).forward;
  const bool f32 = d.code == RG_DTYPE_F32;
  if (tiles) {  // (written by the recurrence's kernel)
    kept.starts = empty({d.B, d.T}, at::kBool, x);
    if (f32) kept.bias = empty({2, d.W}, x);
  } else {
    kept.starts = at::eq(pos, 0);
  }
  if (f32) {
    if (rg::gates_f32_serves(d.M(), (int)d.W, (int)H)) {
      check_hip(rg::launch_gates_f32(in(x), in(g.w_x), in(g.w_a), nullptr, nullptr,
                                     out(gx), out(ga), d.M(), (int)d.W, (int)H,
                                     d.stream));
    } else {
      // the library's batched products, on strided views: no permuted copies
      Tensor xs = by_head(x, H), gxs = by_head(gx, H), gas = by_head(ga, H);
      at::bmm_out(gxs, xs, g.w_x);
      at::bmm_out(gas, xs, g.w_a);
    }
    if (!tiles) {
      gx.view({-1, d.W}).add_(g.b_x.view({1, d.W}));
      ga.view({-1, d.W}).add_(g.b_a.view({1, d.W}));
    }
  } else {
    check(rg_gates_gemm(in(x), 0, nullptr, 0, nullptr, nullptr, in(g.w_x),
                        in(g.b_x), in(g.w_a), in(g.b_a), out(gx), out(ga),
                        (int)d.B, (int)d.T, (int)d.W, (int)H, d.code, d.stream));
  }
  if (tiles) {
    rg::ScanTileArgs t{};
    t.in[0] = in(x);
    t.in[1] = in(gx);
    t.in[2] = in(ga);
    t.flags = in(pos);
    t.flag_kind = seg_kind(pos);
    t.a_param = in(g.a_param);
    if (f32) {
      t.bias[0] = in(g.b_x);
      t.bias[1] = in(g.b_a);
      t.bias_out = (float*)out(kept.bias);
    }
    t.starts_out = (uint8_t*)out(kept.starts);
    t.init = (const float*)in(h0);
    t.out[0] = out(y);
    t.last = (float*)out(h);
    t.B = (int)d.B;
    t.T = (int)d.T;
    t.W = (int)d.W;
    const Tensor ws = deal_workspace(d, rg::kTilesFwdGated, x);
    t.deal = out(ws);
    check_hip(rg::launch_scan_tiles(t, rg::kTilesFwdGated, d.code, d.stream));
    return;
  }
  const size_t bytes =
      rg_scan_split_workspace_bytes((int)d.B, (int)d.T, (int)d.W);
  Tensor ws;
  if (bytes) ws = empty({(int64_t)bytes}, at::kByte, x);
  check(bytes
            ? rg_lru_scan_fused_split(
                  in(x), 0, nullptr, nullptr, in(gx), in(ga), in(g.a_param),
                  in(pos), seg_kind(pos), in(h0), out(y), out(h), nullptr, out(ws),
                  bytes, (int)d.B, (int)d.T, (int)d.W, d.code, d.stream)
            : rg_lru_scan_fused(in(x), 0, nullptr, nullptr, in(gx), in(ga),
                                in(g.a_param), in(pos), seg_kind(pos), in(h0),
                                out(y), out(h), nullptr, (int)d.B, (int)d.T,
                                (int)d.W, d.code, d.stream));
}

struct GateNeeds {
  bool w_x, b_x, w_a, b_a;
};

// The reductions over rows that a backward pass ends with, in one launch.
struct Sums {
  rg::SumTask tasks[rg::kMaxSumTasks];
  int count = 0;
  std::vector<Tensor> keep;
  Tensor add(const Tensor& partial, int64_t offset, int64_t rows, int64_t n,
             int64_t ld, at::IntArrayRef shape, const Tensor& like) {
    if (count == rg::kMaxSumTasks) throw KernelFailure("too many row sums");
    Tensor sum = empty(shape, like);
    tasks[count++] = {(const float*)in(partial) + offset, (int)rows, (int)n,
                      (int)ld, out(sum)};
    keep.push_back(partial);
    return sum;
  }
  void launch(const Dims& d) {
    if (count) check_hip(rg::launch_sum_rows(tasks, count, d.code, d.stream));
  }
};

struct GatedGrads {
  Tensor dx, dlam, dw_x, db_x, dw_a, db_a, dh0;
};

GatedGrads gated_backward(const Tensor& dy, const Tensor& dh, const Tensor& x,
                          const Kept& kept, const Tensor& a_param,
                          const Tensor& w_x, const Tensor& w_a, const Tensor& gx,
                          const Tensor& ga, const Tensor& y, const Tensor& h0,
                          const GateNeeds& need_, Sums& sums) {
  const Dims d(x);
  const int64_t H = w_x.size(0), bw = d.W / H;
  const bool f32 = d.code == RG_DTYPE_F32;
  GatedGrads r;
  r.dx = empty(x.sizes(), x);
  Tensor dgx = empty(x.sizes(), x), dga = empty(x.sizes(), x);
  const bool tiles = on_tiles(d).backward;
  Tensor ws_deal, bias_rows;
  if (tiles) ws_deal = deal_workspace(d, rg::kTilesBwdGated, x);
  // (dealt out: a row of sums per step)
  const int64_t rows =
      d.B * (ws_deal.defined() ? rg::scan_tiles_steps((int)d.T, rg::kTilesBwdGated) : 1);
  Tensor lam_rows = empty({rows, d.W}, at::kFloat, x);
  if (h0.defined()) r.dh0 = empty(h0.sizes(), h0);
  if (tiles) {
    rg::ScanTileArgs t{};
    t.deal = out(ws_deal);
    t.in[0] = in(dy);
    t.in[1] = in(x);
    t.in[2] = in(gx);
    t.in[3] = in(ga);
    t.in[4] = in(y);
    t.flags = in(kept.starts);
    t.flag_kind = rg::kSegMaskU8;
    t.a_param = in(a_param);
    if (f32) {
      t.bias[0] = in(kept.bias);
      t.bias[1] = kept.bias.const_data_ptr<float>() + d.W;
      bias_rows = empty({2, rows, d.W}, at::kFloat, x);
      t.dbias = (float*)out(bias_rows);
    }
    t.init = (const float*)in(dh);
    t.h0 = (const float*)in(h0);
    t.out[0] = out(r.dx);
    t.out[1] = out(dgx);
    t.out[2] = out(dga);
    t.last = (float*)out(r.dh0);
    t.dlam = (float*)out(lam_rows);
    t.B = (int)d.B;
    t.T = (int)d.T;
    t.W = (int)d.W;
    check_hip(rg::launch_scan_tiles(t, rg::kTilesBwdGated, d.code, d.stream));
  } else {
    check(rg_rglru_backward(in(dy), in(x), in(gx), in(ga), in(a_param),
                            in(kept.starts), in(y), in(h0), in(dh), out(r.dx), out(dgx),
                            out(dga), (float*)out(lam_rows), out(r.dh0), (int)d.B,
                            (int)d.T, (int)d.W, d.code, d.stream));
  }
  r.dlam = sums.add(lam_rows, 0, rows, d.W, d.W, {d.W}, x);
  if (f32) {
    Tensor xs = by_head(x, H), dxs = by_head(r.dx, H);
    Tensor dgs[2] = {by_head(dgx, H), by_head(dga, H)};
    const Tensor* w[2] = {&w_x, &w_a};
    Tensor* dw[2] = {&r.dw_x, &r.dw_a};
    Tensor* db[2] = {&r.db_x, &r.db_a};
    const bool needs_w[2] = {need_.w_x, need_.w_a};
    const bool needs_b[2] = {need_.b_x, need_.b_a};
    const bool pair = need_.w_x && need_.w_a &&
                      rg::gates_wgrad_f32_serves(d.M(), (int)d.W, (int)H);
    if (pair) {
      r.dw_x = empty({H, bw, bw}, x);
      r.dw_a = empty({H, bw, bw}, x);
      const size_t bytes =
          rg::gates_wgrad_f32_workspace_bytes(d.M(), (int)d.W, (int)H);
      Tensor ws;
      if (bytes) ws = empty({(int64_t)bytes}, at::kByte, x);
      check_hip(rg::launch_gates_wgrad_f32(in(x), in(dgx), in(dga), out(r.dw_x),
                                           out(r.dw_a), out(ws), d.M(), (int)d.W,
                                           (int)H, d.stream));
    }
    const bool data = rg::gates_f32_serves(d.M(), (int)d.W, (int)H);
    if (data)  // added to the recurrence's share where it lies
      check_hip(rg::launch_gates_dgrad_f32(in(dgx), in(dga), in(w_x), in(w_a),
                                           out(r.dx), d.M(), (int)d.W, (int)H,
                                           d.stream));
    for (int i = 0; i < 2; ++i) {
      if (!data)
        at::baddbmm_out(dxs, dxs, dgs[i], w[i]->transpose(1, 2), 1, 1);
      if (needs_w[i] && !pair) *dw[i] = at::bmm(xs.transpose(1, 2), dgs[i]);
      if (!needs_b[i]) continue;
      if (tiles)
        *db[i] = sums.add(bias_rows, i * rows * d.W, rows, d.W, d.W, {H, bw}, x);
      else
        *db[i] = (i ? dga : dgx).view({-1, H, bw}).sum(0);
    }
    return r;
  }
  if (need_.w_x || need_.w_a || need_.b_x || need_.b_a) {
    r.dw_x = empty({H, bw, bw}, x);
    r.dw_a = empty({H, bw, bw}, x);
    if (need_.b_x || need_.b_a) {
      r.db_x = empty({H, bw}, x);
      r.db_a = empty({H, bw}, x);
    }
    const size_t bytes =
        rg_gates_weight_grads_workspace_bytes(d.M(), (int)d.W, (int)H);
    Tensor ws = empty({(int64_t)bytes}, at::kByte, x);
    check(rg_gates_weight_grads(in(x), in(dgx), in(dga), out(r.dw_x), out(r.dw_a),
                                out(r.db_x), out(r.db_a), out(ws), bytes, d.M(),
                                (int)d.W, (int)H, d.code, d.stream));
  }
  check_hip(rg::launch_gates_dgrad(in(dgx), in(dga), in(w_x), in(w_a),
                                   out(r.dx), d.M(), (int)d.W, (int)H, d.stream));
  return r;
}

struct Rglru : Function<Rglru> {
  static variable_list forward(AutogradContext* ctx, Tensor x, Tensor pos,
                               Tensor a_param, Tensor w_x, Tensor b_x, Tensor w_a,
                               Tensor b_a, OptTensor h0_) {
    const Tensor h0 = h0_.value_or(Tensor());
    ctx->set_materialize_grads(false);
    Tensor gx = empty(x.sizes(), x), ga = empty(x.sizes(), x);
    Tensor y = empty(x.sizes(), x);
    Tensor h = empty({x.size(0), x.size(2)}, at::kFloat, x);
    Kept kept;
    gated_forward(x, pos, {a_param, w_x, b_x, w_a, b_a}, h0, gx, ga, y, h, kept);
    ctx->save_for_backward(
        {x, kept.starts, a_param, w_x, w_a, kept.bias, h0, gx, ga, y});
    return {y, h};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    at::AutoGradMode off(false);
    const Saved s(ctx, 0);
    const Tensor x = s.root, y = s.like_root(9);
    const Kept kept{s.get(1, {s.B, s.T}, at::kBool), kept_bias(s, 5)};
    Tensor dy = grad_of(grads[0], y.sizes(), y.scalar_type());
    if (!dy.defined()) dy = at::zeros_like(y);
    const Tensor dh = grad_of(grads[1], {s.B, s.W}, at::kFloat);
    Sums sums;
    GatedGrads r = gated_backward(
        dy, dh, x, kept, s.get(2, {s.W}), s.gate_weight(3),
        s.gate_weight(4), s.like_root(7), s.like_root(8), y, s.state(6),
        {ctx->needs_input_grad(3), ctx->needs_input_grad(4),
         ctx->needs_input_grad(5), ctx->needs_input_grad(6)},
        sums);
    sums.launch(Dims(x));
    return {r.dx, Tensor(), r.dlam, r.dw_x, r.db_x, r.dw_a, r.db_a, r.dh0};
  }
};

// --------------------------------------------------------- recurrent block --

// x [M, K] through layers that share it, each [M, N] of `out` written: one launch where
// that is ahead of the library's products.
void linear_forward(const Tensor& x, std::initializer_list<const Tensor*> w,
                    std::initializer_list<const Tensor*> b,
                    std::initializer_list<const Tensor*> out_, const Dims& d) {
  const void *ws[rg::kMaxMatmuls], *bs[rg::kMaxMatmuls];
  void* outs[rg::kMaxMatmuls];
  int n[rg::kMaxMatmuls];
  const int count = (int)w.size();
  for (int i = 0; i < count; ++i) {
    ws[i] = in(*w.begin()[i]);
    bs[i] = in(*b.begin()[i]);
    outs[i] = out(*out_.begin()[i]);
    n[i] = (int)w.begin()[i]->size(0);
  }
  const int K = (int)x.size(1);
  if (rg_linear_many_pays(x.size(0), K, count, n, d.code)) {
    check(rg_linear_many(in(x), x.size(0), K, count, ws, bs, outs, n, d.code, d.stream));
    return;
  }
  for (int i = 0; i < count; ++i) {
    Tensor y = *out_.begin()[i];
    at::addmm_out(y, *b.begin()[i], x, w.begin()[i]->t());
  }
}

// dy [M, N] back through w [N, K], and dy2 through w2 where there is one (two layers
// that read the same input).
Tensor linear_back(const Tensor& dy, const Tensor& w, const Tensor& dy2, const Tensor& w2,
                   const Dims& d) {
  const int64_t M = dy.size(0);
  const int N = (int)dy.size(1), K = (int)w.size(1);
  Tensor dx = empty({M, K}, dy);
  if (rg_linear_back_pays(M, N, K, dy2.defined(), d.code)) {
    check(rg_linear_back(in(dy), in(w), in(dy2), dy2.defined() ? in(w2) : nullptr,
                         out(dx), M, N, K, d.code, d.stream));
    return dx;
  }
  at::mm_out(dx, dy, w);
  if (dy2.defined()) dx.addmm_(dy2, w2);
  return dx;
}

// The weights' gradients of layers side by side: 100 tiles of a 2560 x 2560 each, whose
// contraction is the rows, leave the chip half idle one by one.
struct LinearWeights {
  std::vector<Tensor> dy, x;
  std::vector<Tensor*> dw;
  void add(const Tensor& dy_, const Tensor& x_, Tensor* to) {
    dy.push_back(dy_);
    x.push_back(x_);
    dw.push_back(to);
  }
  void launch(const Dims& d) {
    const void *dys[rg::kMaxMatmuls], *xs[rg::kMaxMatmuls];
    void* dws[rg::kMaxMatmuls];
    int n[rg::kMaxMatmuls], k[rg::kMaxMatmuls];
    for (size_t i = 0; i < dw.size(); ++i) {
      n[i] = (int)dy[i].size(1);
      k[i] = (int)x[i].size(1);
      *dw[i] = empty({n[i], k[i]}, x[i]);
      dys[i] = in(dy[i]);
      xs[i] = in(x[i]);
      dws[i] = out(*dw[i]);
    }
    if (dw.empty()) return;
    int rc = RG_ERR_UNSUPPORTED;
    if (d.code == RG_DTYPE_BF16)
      rc = rg_linear_weight_grads(dys, xs, dws, n, k, (int)dw.size(), d.M(), d.code,
                                  d.stream);
    if (rc != RG_ERR_UNSUPPORTED) return check(rc);
    for (size_t i = 0; i < dw.size(); ++i) at::mm_out(*dw[i], dy[i].t(), x[i]);
  }
};

// (modules.py:605-655 of the reference, without a cache)
struct Block : Function<Block> {
  static variable_list forward(AutogradContext* ctx, Tensor x, Tensor pos,
                               Tensor w_y, Tensor b_y, Tensor w_lx, Tensor b_lx,
                               Tensor conv_w, Tensor conv_b, Tensor a_param,
                               Tensor w_x, Tensor b_x, Tensor w_a, Tensor b_a,
                               Tensor w_out, Tensor b_out, bool want_cache) {
    ctx->set_materialize_grads(false);
    const int64_t B = x.size(0), T = x.size(1), W = w_y.size(0);
    const int64_t D = x.size(2);
    Tensor x2 = x.view({B * T, D});
    Tensor gate = empty({B * T, W}, x), lx = empty({B * T, W}, x);
    linear_forward(x2, {&w_y, &w_lx}, {&b_y, &b_lx}, {&gate, &lx}, Dims(x));
    gate = gate.view({B, T, W});
    lx = lx.view({B, T, W});
    const Dims d(lx);
    Tensor xc = empty(lx.sizes(), x), conv_state, h;
    if (want_cache) {
      conv_state = empty({B, 3, W}, x);
      h = empty({B, W}, at::kFloat, x);
    }
    check(rg_conv1d_prefill(in(lx), in(pos), seg_kind(pos), in(conv_w), in(conv_b),
                            out(xc), out(conv_state), (int)B, (int)T, (int)W, 4,
                            d.code, d.stream));
    Tensor gx = empty(lx.sizes(), x), ga = empty(lx.sizes(), x);
    Tensor y = empty(lx.sizes(), x);
    Kept kept;
    gated_forward(xc, pos, {a_param, w_x, b_x, w_a, b_a}, Tensor(), gx, ga, y, h,
                  kept);
    Tensor join = empty(lx.sizes(), x);
    check(rg_gelu_mul(in(y), in(gate), out(join), d.M() * W, d.code, d.stream));
    Tensor result = empty({B * T, D}, x);
    linear_forward(join.view({B * T, W}), {&w_out}, {&b_out}, {&result}, d);
    result = result.view({B, T, D});
    ctx->save_for_backward({x, pos, w_y, w_lx, conv_w, a_param, w_x, w_a,
                            kept.bias, w_out, gate, lx, xc, gx, ga, y, join,
                            kept.starts});
    if (!want_cache) return {result};
    ctx->mark_non_differentiable({conv_state});
    return {result, h, conv_state};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    at::AutoGradMode off(false);
    const Saved s(ctx, 11);
    const Tensor lx = s.root, gate = s.like_root(10), xc = s.like_root(12),
                 y = s.like_root(15), join = s.like_root(16);
    const Dims d(lx);
    const int64_t M = d.M(), W = d.W;
    Saved::fits(s.v[0].defined() && s.v[0].dim() == 3 && s.v[1].defined());
    const int64_t D = s.v[0].size(2);
    const Tensor x = s.get(0, {d.B, d.T, D}), w_y = s.get(2, {W, D}),
                 w_lx = s.get(3, {W, D}), conv_w = s.get(4, {4, W}),
                 w_out = s.get(9, {D, W}),
                 pos = s.get(1, {d.B, d.T},
                             s.v[1].scalar_type() == at::kInt ? at::kInt
                                                              : at::kLong);
    Saved::fits(block_sums_serve(d.B, d.T, W, D, d.code));
    const Tensor x2 = x.view({M, D});
    auto needs = [&](int i) { return ctx->needs_input_grad(i); };
    Sums sums;
    variable_list r(16);  // (the flag takes no gradient)
    Tensor dy, dgate2, dout;
    if (grads[0].defined()) {
      dout = grad_of(grads[0], x.sizes(), x.scalar_type()).view({M, D});
      const int64_t parts = (M + rg::kColSumRows - 1) / rg::kColSumRows;
      if (needs(14)) {
        Tensor part = empty({parts, dout.size(1)}, at::kFloat, x);
        check_hip(rg::launch_col_sums(in(dout), (float*)out(part), M,
                                      (int)dout.size(1), d.code, d.stream));
        r[14] = sums.add(part, 0, parts, dout.size(1), dout.size(1),
                         {dout.size(1)}, x);
      }
      const Tensor djoin = linear_back(dout, w_out, Tensor(), Tensor(), d);
      dy = empty(lx.sizes(), x);
      dgate2 = empty({M, W}, x);
      Tensor part = empty({parts, W}, at::kFloat, x);
      check_hip(rg::launch_gelu_mul_backward_sums(
          in(djoin), in(y), in(gate), out(dy), out(dgate2), (float*)out(part), M,
          (int)W, d.code, d.stream));
      if (needs(3)) r[3] = sums.add(part, 0, parts, W, W, {W}, x);
    } else {
      dy = at::zeros_like(y);  // only the final state is differentiated
    }
    Tensor dh;
    if (grads.size() > 1) dh = grad_of(grads[1], {d.B, W}, at::kFloat);
    GatedGrads g = gated_backward(
        dy, dh, xc, {s.get(17, {d.B, d.T}, at::kBool), kept_bias(s, 8)}, s.get(5, {W}),
        s.gate_weight(6), s.gate_weight(7), s.like_root(13), s.like_root(14), y,
        Tensor(), {needs(9), needs(10), needs(11), needs(12)}, sums);
    r[8] = g.dlam;
    r[9] = g.dw_x;
    r[10] = g.db_x;
    r[11] = g.dw_a;
    r[12] = g.db_a;
    rg::ConvBwdArgs c{};
    const int64_t chunks = rg::conv1d_backward_chunks((int)d.B, (int)d.T);
    Tensor part = empty({chunks, 5, W}, at::kFloat, x);
    Tensor dlx_part = empty({chunks, W}, at::kFloat, x);
    Tensor dlx2 = dy.view({M, W});  // (dy has been read)
    c.dout = in(g.dx);
    c.x = in(lx);
    c.segpos = in(pos);
    c.seg_kind = seg_kind(pos);
    c.w = in(conv_w);
    c.dx = out(dlx2);
    c.partial = (float*)out(part);
    c.dx_sums = (float*)out(dlx_part);
    c.B = (int)d.B;
    c.T = (int)d.T;
    c.W = (int)W;
    c.K = 4;
    check_hip(rg::launch_conv1d_backward(c, d.code, d.stream));
    if (needs(6)) r[6] = sums.add(part, 0, chunks, 4 * W, 5 * W, {4, W}, x);
    if (needs(7)) r[7] = sums.add(part, 4 * W, chunks, W, 5 * W, {W}, x);
    if (needs(5)) r[5] = sums.add(dlx_part, 0, chunks, W, W, {W}, x);
    sums.launch(d);
    LinearWeights dw;
    if (dout.defined() && needs(13)) dw.add(dout, join.view({M, W}), &r[13]);
    if (dout.defined() && needs(2)) dw.add(dgate2, x2, &r[2]);
    if (needs(4)) dw.add(dlx2, x2, &r[4]);
    dw.launch(d);
    if (needs(0))
      r[0] = linear_back(dlx2, w_lx, dgate2, w_y, d).view(x.sizes());
    return r;
  }
};

// Shared by the two entries below: the RG-LRU's tensors at v[0..4].
GateWeights gate_weights(const Call& c, PyObject* const* v, int64_t W) {
  GateWeights g{tensor_of(v[0]), tensor_of(v[1]), tensor_of(v[2]), tensor_of(v[3]),
                tensor_of(v[4])};
  need(g.w_x.dim() == 3);
  const int64_t H = g.w_x.size(0);
  need(H > 0 && W % H == 0);
  const int64_t bw = W / H;
  c.shaped(v[0], {W});
  c.shaped(v[1], {H, bw, bw});
  c.shaped(v[2], {H, bw});
  c.shaped(v[3], {H, bw, bw});
  c.shaped(v[4], {H, bw});
  need(c.code == RG_DTYPE_F32 || bw == 256);
  return g;
}

// The calls below: under autograd or not, never under autocast (which would
// have other dtypes in between).
Call plain_call(PyObject* o) {
  need(!at::autocast::is_autocast_enabled(at::kCUDA));
  Call c(o);
  need(c.x.dim() == 3 && c.x.numel() > 0);
  for (int i = 0; i < 3; ++i) need(c.x.size(i) <= INT32_MAX);
  c(o);
  return c;
}

struct ScanCall {
  Call c;
  Tensor a, reset;
  OptTensor h0;
  explicit ScanCall(PyObject* const* v) : c(plain_call(v[0])) {
    const int64_t B = c.x.size(0), T = c.x.size(1), W = c.x.size(2);
    c.shaped(v[1], {B, T, W});
    a = tensor_of(v[1]);
    reset = tensor_of(v[2]);
    need(shape_is(reset, {B, T}));
    dense(reset, at::kBool, c.device);
    if (v[3] != Py_None) {
      c.f32(v[3], {B, W});
      h0 = tensor_of(v[3]);
    }
  }
};

PyObject* pair(const Tensor& a, const Tensor& b) {
  PyObject* t = PyTuple_New(2);
  if (!t) throw Raised{};
  PyTuple_SET_ITEM(t, 0, wrap(a));
  PyTuple_SET_ITEM(t, 1, wrap(b));
  return t;
}

}  // namespace

// (x, a, reset, h0 | None) -> (y, h_last) | None
PyObject* linear_scan(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 4);
    ScanCall s(v);
    Tensor y = empty(s.c.x.sizes(), s.c.x);
    Tensor h = empty({s.c.x.size(0), s.c.x.size(2)}, at::kFloat, s.c.x);
    {
      NoGil nogil;
      scan_forward(s.c.x, s.a, s.reset, s.h0.value_or(Tensor()), y, h);
    }
    return pair(y, h);
  });
}

// (x, a, reset, h0 | None) -> (y, h_last) | None, differentiable
PyObject* train_scan(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 4);
    ScanCall s(v);
    variable_list r;
    {
      NoGil nogil;
      r = Scan::apply(s.c.x, s.a, s.reset, s.h0);
    }
    return pair(r[0], r[1]);
  });
}

// (x, segment_pos, a_param, w_x, b_x, w_a, b_a, h0 | None)
//   -> (y, h_last) | None, differentiable
PyObject* train_rglru(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 8);
    Call c = plain_call(v[0]);
    const int64_t B = c.x.size(0), T = c.x.size(1), W = c.x.size(2);
    int is64;
    c.positions(v[1], B, T, &is64);
    const Tensor pos = tensor_of(v[1]);
    const GateWeights g = gate_weights(c, v + 2, W);
    OptTensor h0;
    if (v[7] != Py_None) {
      c.f32(v[7], {B, W});
      h0 = tensor_of(v[7]);
    }
    variable_list r;
    {
      NoGil nogil;
      r = Rglru::apply(c.x, pos, g.a_param, g.w_x, g.b_x, g.w_a, g.b_a, h0);
    }
    return pair(r[0], r[1]);
  });
}

// (x, segment_pos, w_y, b_y, w_x, b_x, conv_w, conv_b, a_param, gate w_x, b_x,
//  w_a, b_a, w_out, b_out, want_cache)
//   -> (out, h_last | None, conv_state | None) | None, differentiable
PyObject* train_block(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 16);
    Call c = plain_call(v[0]);
    const int64_t B = c.x.size(0), T = c.x.size(1), D = c.x.size(2);
    int is64;
    c.positions(v[1], B, T, &is64);
    Tensor t[14];
    for (int i = 1; i < 15; ++i) t[i - 1] = tensor_of(v[i]);
    need(t[1].dim() == 2);
    const int64_t W = t[1].size(0);
    c.shaped(v[2], {W, D});
    c.shaped(v[3], {W});
    c.shaped(v[4], {W, D});
    c.shaped(v[5], {W});
    c.shaped(v[6], {4, W});
    c.shaped(v[7], {W});
    gate_weights(c, v + 8, W);
    c.shaped(v[13], {D, W});
    c.shaped(v[14], {D});
    need(block_sums_serve(B, T, W, D, c.code));
    const bool want_cache = v[15] == Py_True;
    variable_list r;
    {
      NoGil nogil;
      r = Block::apply(c.x, t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8],
                       t[9], t[10], t[11], t[12], t[13], want_cache);
    }
    return want_cache ? triple(r[0], r[1], r[2]) : triple(r[0], Tensor(), Tensor());
  });
}

}  // namespace rg_host

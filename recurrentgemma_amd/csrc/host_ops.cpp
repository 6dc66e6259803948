// The short host path of the calls that are launched once per token or per
// small prompt: a decode step, a prefill, the linear layers of a few rows.
//
// From Python through ctypes such a call costs 13-23 us of host time (argument
// checks on ~15 tensors, attribute lookups, three allocations, ~20 converted
// arguments) around a kernel of 5-10 us, so the GPU waits for the host.  Here
// the same checks, allocations and the one C-ABI call are native code behind a
// METH_FASTCALL entry.
//
// Each function serves the ordinary case only -- plain dense, 16-byte aligned
// torch tensors of one dtype on the current GPU, shapes as documented -- and
// answers None for anything else; its caller in ops.py then takes the general
// path, which makes copies, converts, or raises the error that belongs to the
// argument.  So there is one place that words the errors, and nothing here
// has to.
//
// Plain C++ on torch's and this library's public interfaces; no device code.
#include <ATen/autocast_mode.h>

#include "host_call.h"
#include "rg_package_calls.h"

namespace {

using namespace rg_host;

// --------------------------------------------------------------- stamps --

// The state of a tensor that something was derived from: same object, same
// storage, not written to since.  Holds a weak reference, so that the
// object's address is not given to another tensor meanwhile.
struct Stamp {
  c10::weak_intrusive_ptr<c10::TensorImpl> ref;
  c10::TensorImpl* impl;
  const void* data;
  int64_t version;
  explicit Stamp(const Tensor& t)
      : ref(t.getIntrusivePtr()),
        impl(t.unsafeGetTensorImpl()),
        data(t.const_data_ptr()),
        version(t.is_inference() ? -1 : t._version()) {}
  bool matches(const Tensor& t) const {
    // (inference tensors keep no version counter: never known to be unchanged)
    return t.unsafeGetTensorImpl() == impl && version >= 0 &&
           !t.is_inference() && t._version() == version &&
           t.const_data_ptr() == data;
  }
};

// Gate weights in operand order, by the pair of tensors they came from.
// ops.packed_gate_weights fills and sweeps it (remember_packed); at most
// kMaxPacked entries are looked up here, the rest take the general path.
struct PackedEntry {
  Stamp x, a;
  Tensor packed;
};
constexpr size_t kMaxPacked = 1024;
std::unordered_map<c10::TensorImpl*, PackedEntry>* g_packed;

// (by value: the caller keeps it alive while it launches without the GIL)
Tensor packed_for(const Tensor& w_x, const Tensor& w_a) {
  auto it = g_packed->find(w_x.unsafeGetTensorImpl());
  need(it != g_packed->end() && it->second.x.matches(w_x) &&
       it->second.a.matches(w_a));
  return it->second.packed;
}

PyObject* remember_packed(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 3);
    const Tensor &w_x = tensor_of(v[0]), &w_a = tensor_of(v[1]);
    const Tensor& packed = tensor_of(v[2]);
    for (auto it = g_packed->begin(); it != g_packed->end();)
      it = it->second.x.ref.expired() || it->second.a.ref.expired()
               ? g_packed->erase(it)
               : std::next(it);
    g_packed->erase(w_x.unsafeGetTensorImpl());
    if (g_packed->size() < kMaxPacked && !w_x.is_inference() &&
        !w_a.is_inference())
      g_packed->emplace(w_x.unsafeGetTensorImpl(),
                        PackedEntry{Stamp(w_x), Stamp(w_a), packed});
    Py_RETURN_NONE;
  });
}

// --------------------------------------------------------- recurrent core --

// (x, segment_pos, conv_state, h, conv_w, conv_b, w_x, b_x, w_a, b_a, a_param,
//  in_place, gate_branch | None, [copy of conv_state | None]) -> (y, h, conv_state) | None
PyObject* recurrent_step(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 13 || n == 14);
    Call c(v[0]);
    need(c.x.dim() == 3 && c.x.size(1) == 1);
    const int64_t B = c.x.size(0), W = c.x.size(2);
    const Tensor &w_x = tensor_of(v[6]), &w_a = tensor_of(v[8]);
    need(B > 0 && w_x.dim() == 3);
    const int64_t H = w_x.size(0);
    need(H > 0 && W % H == 0 && B <= INT32_MAX && W <= INT32_MAX);
    const int64_t bw = W / H;
    void* wx = c.shaped(v[6], {H, bw, bw});
    void* wa = c.shaped(v[8], {H, bw, bw});
    void* x = c(v[0]);
    int is64;
    void* pos = c.positions(v[1], B, 1, &is64);
    void* conv_in = c.shaped(v[2], {B, 3, W});
    void* h_in = c.f32(v[3], {B, W});
    void* conv_w = c.shaped(v[4], {4, W});
    void* conv_b = c.shaped(v[5], {W});
    void* b_x = c.shaped(v[7], {H, bw});
    void* b_a = c.shaped(v[9], {H, bw});
    void* a_param = c.shaped(v[10], {W});
    // one launch on re-laid-out weights, or conv step + gate GEMM + scan step
    // (+ the join) through a workspace
    Tensor packed, ws;
    if (c.code == RG_DTYPE_BF16 && bw == 256) {
      packed = packed_for(w_x, w_a);
      need(packed.device() == c.x.device());
    }
    const bool in_place = v[11] == Py_True;
    void* gate = v[12] == Py_None ? nullptr : c.shaped(v[12], {B, 1, W});
    // (read from the copy, the conv state is written while heads are shared)
    if (n == 14 && v[13] != Py_None) conv_in = c.shaped(v[13], {B, 3, W});
    Tensor y = c.empty(c.x.sizes());
    Tensor h, conv;
    if (in_place) {
      h = THPVariable_Unpack(v[3]);
      conv = THPVariable_Unpack(v[2]);
    } else {
      h = c.empty({B, W}, at::kFloat);
      conv = c.empty({B, 3, W});
    }
    void *yp = y.mutable_data_ptr(), *hp = h.mutable_data_ptr(),
         *cp = conv.mutable_data_ptr();
    void* s = c.stream();
    if (!packed.defined()) {
      const size_t bytes =
          rg_recurrent_step_workspace_bytes((int)B, (int)W, c.code);
      ws = c.empty({(int64_t)bytes}, at::kByte);
      void* wp = ws.mutable_data_ptr();
      launch([&] {
        if (gate)
          return rg_recurrent_step_join(
              x, gate, pos, is64, conv_in, cp, (const float*)h_in, (float*)hp, conv_w,
              conv_b, wx, b_x, wa, b_a, a_param, yp, wp, bytes, (int)B, (int)W, (int)H,
              c.code, s);
        return rg_recurrent_step(
            x, pos, is64, conv_in, cp, (const float*)h_in, (float*)hp, conv_w,
            conv_b, wx, b_x, wa, b_a, a_param, yp, wp, bytes, (int)B, (int)W,
            (int)H, c.code, s);
      });
      return triple(y, h, conv);
    }
    const void* pk = packed.const_data_ptr();
    launch([&] {
      if (gate)
        return rg_recurrent_step_gelu_mul(
            x, gate, pos, is64, conv_in, cp, (const float*)h_in, (float*)hp,
            conv_w, conv_b, pk, b_x, b_a, a_param, yp, (int)B, (int)W, (int)H,
            c.code, s);
      return rg_recurrent_step_packed(
          x, pos, is64, conv_in, cp, (const float*)h_in, (float*)hp, conv_w,
          conv_b, pk, b_x, b_a, a_param, yp, (int)B, (int)W, (int)H, c.code, s);
    });
    return triple(y, h, conv);
  });
}

// (x, segment_pos, conv_w | None, conv_b | None, w_x, b_x, w_a, b_a, a_param,
//  h0 | None, return_h, return_conv_cache, gate_branch | None)
//   -> (y, h | None, conv_cache | None) | None
PyObject* recurrent_core(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 13);
    Call c(v[0]);
    need(c.x.dim() == 3 && c.x.numel() > 0);
    const int64_t B = c.x.size(0), T = c.x.size(1), W = c.x.size(2);
    const Tensor &w_x = tensor_of(v[4]), &w_a = tensor_of(v[6]);
    need(w_x.dim() == 3 && B <= INT32_MAX && T <= INT32_MAX && W <= INT32_MAX);
    const int64_t H = w_x.size(0);
    need(H > 0 && W % H == 0);
    const int64_t bw = W / H;
    void* x = c(v[0]);
    int is64;
    void* pos = c.positions(v[1], B, T, &is64);
    const bool conv = v[2] != Py_None;
    need(conv == (v[3] != Py_None));
    void* conv_w = conv ? c.shaped(v[2], {4, W}) : nullptr;
    void* conv_b = conv ? c.shaped(v[3], {W}) : nullptr;
    void* wx = c.shaped(v[4], {H, bw, bw});
    void* b_x = c.shaped(v[5], {H, bw});
    void* wa = c.shaped(v[6], {H, bw, bw});
    void* b_a = c.shaped(v[7], {H, bw});
    void* a_param = c.shaped(v[8], {W});
    void* h0 = v[9] == Py_None ? nullptr : c.f32(v[9], {B, W});
    void* gate = v[12] == Py_None ? nullptr : c.shaped(v[12], {B, T, W});
    const void* pk = nullptr;
    Tensor packed;
    if (rg_packed_gate_weights_bytes((int)W, (int)H, c.code) > 0) {
      packed = packed_for(w_x, w_a);
      need(packed.device() == c.x.device());
      pk = packed.const_data_ptr();
    }
    Tensor y = c.empty(c.x.sizes()), h, cache, ws;
    if (v[10] == Py_True) h = c.empty({B, W}, at::kFloat);
    if (v[11] == Py_True && conv) cache = c.empty({B, 3, W});
    const size_t bytes = rg_recurrent_core_best_workspace_bytes(
        (int)B, (int)T, (int)W, (int)H, c.code);
    if (bytes) ws = c.empty({(int64_t)bytes}, at::kByte);
    void* yp = y.mutable_data_ptr();
    void* hp = h.defined() ? h.mutable_data_ptr() : nullptr;
    void* cp = cache.defined() ? cache.mutable_data_ptr() : nullptr;
    void* wp = bytes ? ws.mutable_data_ptr() : nullptr;
    void* s = c.stream();
    launch([&] {
      return rg_recurrent_core(x, gate, pos, is64, conv_w, conv_b, wx, b_x, wa,
                               b_a, pk, a_param, h0, yp, hp, cp, wp, bytes,
                               (int)B, (int)T, (int)W, (int)H, c.code, s);
    });
    return triple(y, h, cache);
  });
}

// ------------------------------------------------- linear layers, few rows --

// What ops.PackedLinear prepared from its weights and biases.
struct RowsPlan {
  std::vector<Stamp> sources;
  Tensor packed, bias;
  int N, K, groups;
  bool gelu_pair;
};
const char kPlanName[] = "recurrentgemma_amd.rows_plan";

void free_plan(PyObject* capsule) {
  delete static_cast<RowsPlan*>(PyCapsule_GetPointer(capsule, kPlanName));
}

// (sources tuple, packed, bias | None, N, K, groups, gelu_pair) -> plan
PyObject* rows_plan(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 7 && PyTuple_Check(v[0]));
    auto plan = std::make_unique<RowsPlan>();
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(v[0]); ++i)
      plan->sources.emplace_back(tensor_of(PyTuple_GET_ITEM(v[0], i)));
    plan->packed = tensor_of(v[1]);
    if (v[2] != Py_None) plan->bias = tensor_of(v[2]);
    plan->N = (int)PyLong_AsLong(v[3]);
    plan->K = (int)PyLong_AsLong(v[4]);
    plan->groups = (int)PyLong_AsLong(v[5]);
    plan->gelu_pair = v[6] == Py_True;
    if (PyErr_Occurred()) throw Raised{};
    return PyCapsule_New(plan.release(), kPlanName, free_plan);
  });
}

// The plan of a call, if its weights and biases are what it was made from.
const RowsPlan& plan_of(PyObject* capsule, PyObject* weights, PyObject* biases) {
  need(PyCapsule_IsValid(capsule, kPlanName));
  const auto& p =
      *static_cast<RowsPlan*>(PyCapsule_GetPointer(capsule, kPlanName));
  size_t at = 0;
  for (PyObject* list : {weights, biases}) {
    if (list == Py_None) continue;
    need(PyTuple_Check(list));
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(list); ++i) {
      PyObject* o = PyTuple_GET_ITEM(list, i);
      if (o == Py_None) continue;
      need(at < p.sources.size() && p.sources[at].matches(tensor_of(o)));
      ++at;
    }
  }
  need(at == p.sources.size());
  return p;
}

// leading dimensions of x, and how many rows they make
std::vector<int64_t> lead_of(const Call& c, int K, int64_t* M) {
  need(c.code == RG_DTYPE_BF16 && c.x.dim() >= 1 && c.x.size(-1) == K);
  std::vector<int64_t> lead(c.x.sizes().begin(), c.x.sizes().end() - 1);
  *M = c.x.numel() / K;
  need(*M > 0 && *M <= 64);
  return lead;
}

// (plan, x, weights, biases | None, residual | None[, state]) -> out | tuple | None;
// with a state (layers packed together): (outputs .., a copy of the state made beside them)
PyObject* rows_linear(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 5 || n == 6);
    const RowsPlan& p = plan_of(v[0], v[2], v[3]);
    Call c(v[1]);
    int64_t M;
    std::vector<int64_t> shape = lead_of(c, p.K, &M);
    need(p.packed.device() == c.x.device());
    void* x = c(v[1]);
    const bool grouped = p.groups > 1 && !p.gelu_pair;
    shape.push_back(p.gelu_pair ? p.N / 2 : p.N / p.groups);
    void* residual = nullptr;
    if (v[4] != Py_None) {
      const Tensor& r = tensor_of(v[4]);
      need(!grouped && !p.gelu_pair && r.sizes() == at::IntArrayRef(shape));
      residual = dense(r, c.dtype, c.device);
    }
    // (one allocation per group: the kernel wants [G, M, N / G] in one piece)
    if (grouped) shape.insert(shape.begin(), p.groups);
    Tensor out = c.empty(shape), ws;
    const size_t bytes =
        p.gelu_pair ? 0 : rg_linear_rows_workspace_bytes((int)M, p.K, p.N);
    if (bytes) ws = c.empty({(int64_t)bytes}, at::kByte);
    void* op = out.mutable_data_ptr();
    void* wp = bytes ? ws.mutable_data_ptr() : nullptr;
    const void* pk = p.packed.const_data_ptr();
    const void* bias = p.bias.defined() ? p.bias.const_data_ptr() : nullptr;
    void* s = c.stream();
    Tensor aside;
    if (n == 6) {
      const Tensor& state = tensor_of(v[5]);
      const void* from = dense(state, c.dtype, c.device);
      const int64_t copied = (int64_t)state.nbytes();
      need(grouped && !residual && !bytes && copied > 0 && copied % 16 == 0);
      aside = c.empty(state.sizes());
      void* to = aside.mutable_data_ptr();
      launch([&] {
        return rg_linear_rows_beside(x, pk, bias, op, (int)M, p.K, p.N, p.groups, from,
                                     to, copied, s);
      });
    } else {
      launch([&] {
        return rg_linear_rows(x, pk, bias, residual, op, wp, bytes, (int)M, p.K,
                              p.N, grouped ? p.groups : 1, p.gelu_pair, s);
      });
    }
    if (!grouped) return wrap(out);
    PyObject* t = PyTuple_New(p.groups + (n == 6));
    if (!t) throw Raised{};
    for (int i = 0; i < p.groups; ++i)
      PyTuple_SET_ITEM(t, i, wrap(out.select(0, i)));
    if (n == 6) PyTuple_SET_ITEM(t, p.groups, wrap(aside));
    return t;
  });
}

// (plan, x, weights, biases | None, slices) -> sums [slices, M, N] | None
PyObject* rows_partial(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 5);
    const RowsPlan& p = plan_of(v[0], v[2], v[3]);
    Call c(v[1]);
    int64_t M;
    lead_of(c, p.K, &M);
    need(p.packed.device() == c.x.device() && p.groups == 1 && !p.gelu_pair);
    void* x = c(v[1]);
    const long slices = PyLong_AsLong(v[4]);
    need(slices > 0);
    // (the flags of rg_linear_rows_normed behind the sums)
    const int64_t n = slices * M * p.N;
    Tensor all = c.empty({n + RG_NORM_FLAGS}, at::kFloat);
    void* op = all.mutable_data_ptr();
    Tensor sums = all.narrow(0, 0, n).view({slices, M, (int64_t)p.N});
    const void* pk = p.packed.const_data_ptr();
    void* s = c.stream();
    launch([&] {
      return rg_linear_rows_partial_flags(x, pk, (float*)op, (uint32_t*)((float*)op + n),
                                          (int)M, p.K, p.N, (int)slices, s);
    });
    return wrap(sums);
  });
}

// ------------------------------------------------------ the block's step --

// A parameter of an nn.Module, past the attribute lookup that is written in
// Python; anything but a module that holds it itself takes the general path.
PyObject* parameters(PyObject* module) {
  static PyObject* const key = PyUnicode_InternFromString("_parameters");
  PyObject* own = PyObject_GetAttr(module, key);
  if (!own) {
    PyErr_Clear();
    throw Fallback{};
  }
  Py_DECREF(own);  // (the module keeps it)
  return own;
}
const Tensor& parameter(PyObject* module, PyObject* name) {
  PyObject* own = parameters(module);
  need(PyDict_CheckExact(own));
  PyObject* t = PyDict_GetItemWithError(own, name);
  if (!t) PyErr_Clear();
  need(t != nullptr);
  return tensor_of(t);
}
PyObject* child(PyObject* modules, PyObject* name) {
  need(PyDict_CheckExact(modules));
  PyObject* m = PyDict_GetItemWithError(modules, name);
  if (!m) PyErr_Clear();
  need(m != nullptr);
  return m;
}
PyObject* children(PyObject* module) {
  static PyObject* const key = PyUnicode_InternFromString("_modules");
  PyObject* own = PyObject_GetAttr(module, key);
  if (!own) {
    PyErr_Clear();
    throw Fallback{};
  }
  Py_DECREF(own);
  return own;
}
const RowsPlan& plan_for(PyObject* capsule,
                         std::initializer_list<const Tensor*> sources) {
  need(PyCapsule_IsValid(capsule, kPlanName));
  const auto& p =
      *static_cast<RowsPlan*>(PyCapsule_GetPointer(capsule, kPlanName));
  need(p.sources.size() == sources.size());
  size_t at = 0;
  for (const Tensor* t : sources) need(p.sources[at++].matches(*t));
  return p;
}

// A cached single-token call of RecurrentBlock (at most 64 rows, bf16, 256-wide
// heads): its linear layers on the few-row kernels and the step between them,
// the join written over the gate branch.  As three calls from Python it was 25 us
// of host time around 17 us of kernels.
// (the block's _modules, plan of linear_y and linear_x, plan of linear_out, x,
//  segment_pos, conv_state, h, in_place) -> (out, h, conv_state) | None
PyObject* block_step(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 8);
#define RG_NAME(ID, TEXT) \
  static PyObject* const ID = PyUnicode_InternFromString(TEXT);
    RG_NAME(k_y, "linear_y") RG_NAME(k_x, "linear_x") RG_NAME(k_out, "linear_out")
    RG_NAME(k_conv, "conv_1d") RG_NAME(k_lru, "rg_lru")
    RG_NAME(k_gx, "input_gate") RG_NAME(k_ga, "a_gate") RG_NAME(k_w, "w")
    RG_NAME(k_b, "b") RG_NAME(k_weight, "weight") RG_NAME(k_bias, "bias")
    RG_NAME(k_param, "a_param")
#undef RG_NAME
    PyObject *m_y = child(v[0], k_y), *m_x = child(v[0], k_x),
             *m_out = child(v[0], k_out), *m_conv = child(v[0], k_conv),
             *m_lru = child(v[0], k_lru);
    PyObject* gates = children(m_lru);
    PyObject *m_gx = child(gates, k_gx), *m_ga = child(gates, k_ga);
    const RowsPlan& in_plan =
        plan_for(v[1], {&parameter(m_y, k_weight), &parameter(m_x, k_weight),
                        &parameter(m_y, k_bias), &parameter(m_x, k_bias)});
    const RowsPlan& out_plan = plan_for(
        v[2], {&parameter(m_out, k_weight), &parameter(m_out, k_bias)});
    Call c(v[3]);
    need(c.code == RG_DTYPE_BF16 && c.x.dim() == 3 && c.x.size(1) == 1);
    const int64_t B = c.x.size(0), D = c.x.size(2), W = out_plan.K;
    need(B > 0 && B <= 64 && in_plan.K == D && in_plan.groups == 2 &&
         in_plan.N == 2 * W && !in_plan.gelu_pair && in_plan.bias.defined() &&
         out_plan.groups == 1 && !out_plan.gelu_pair && out_plan.bias.defined() &&
         in_plan.packed.device() == c.x.device() &&
         out_plan.packed.device() == c.x.device());
    auto shaped = [&](const Tensor& t, std::initializer_list<int64_t> want) {
      need(shape_is(t, want));
      return dense(t, c.dtype, c.device);
    };
    const Tensor &w_x = parameter(m_gx, k_w), &w_a = parameter(m_ga, k_w);
    need(w_x.dim() == 3);
    const int64_t H = w_x.size(0), bw = 256;
    need(H > 0 && W == H * bw);
    shaped(w_x, {H, bw, bw});
    shaped(w_a, {H, bw, bw});
    void* x = c(v[3]);
    int is64;
    void* pos = c.positions(v[4], B, 1, &is64);
    void* conv_in = c.shaped(v[5], {B, 3, W});
    void* h_in = c.f32(v[6], {B, W});
    void* conv_w = shaped(parameter(m_conv, k_w), {4, W});
    void* conv_b = shaped(parameter(m_conv, k_b), {W});
    void* b_x = shaped(parameter(m_gx, k_b), {H, bw});
    void* b_a = shaped(parameter(m_ga, k_b), {H, bw});
    void* a_param = shaped(parameter(m_lru, k_param), {W});
    const Tensor packed = packed_for(w_x, w_a);
    need(packed.device() == c.x.device());
    const int N = out_plan.N;
    Tensor yx = c.empty({2, B, W}), out = c.empty({B, 1, N}), ws, h, conv;
    if (v[7] == Py_True) {
      h = THPVariable_Unpack(v[6]);
      conv = THPVariable_Unpack(v[5]);
    } else {
      h = c.empty({B, W}, at::kFloat);
      conv = c.empty({B, 3, W});
    }
    const size_t in_bytes =
        rg_linear_rows_workspace_bytes((int)B, (int)D, (int)(2 * W));
    const size_t out_bytes = rg_linear_rows_workspace_bytes((int)B, (int)W, N);
    const size_t bytes = in_bytes > out_bytes ? in_bytes : out_bytes;
    if (bytes) ws = c.empty({(int64_t)bytes}, at::kByte);
    void* wp = bytes ? ws.mutable_data_ptr() : nullptr;
    char* const y = (char*)yx.mutable_data_ptr();  // the gate branch, then the join
    void* const lx = y + 2 * B * W;
    void *op = out.mutable_data_ptr(), *hp = h.mutable_data_ptr(),
         *cp = conv.mutable_data_ptr();
    const void *in_w = in_plan.packed.const_data_ptr(),
               *in_b = in_plan.bias.const_data_ptr(),
               *out_w = out_plan.packed.const_data_ptr(),
               *out_b = out_plan.bias.const_data_ptr(),
               *gates_w = packed.const_data_ptr();
    // (the plans' tensors, which another thread may replace while this one has
    // let go of the interpreter)
    const Tensor keep[] = {in_plan.packed, in_plan.bias, out_plan.packed,
                           out_plan.bias};
    void* s = c.stream();
    launch([&] {
      int rc = rg_linear_rows(x, in_w, in_b, nullptr, y, wp, bytes, (int)B, (int)D,
                              (int)(2 * W), 2, 0, s);
      if (rc != RG_OK) return rc;
      rc = rg_recurrent_step_gelu_mul(lx, y, pos, is64, conv_in, cp,
                                      (const float*)h_in, (float*)hp, conv_w,
                                      conv_b, gates_w, b_x, b_a, a_param, y,
                                      (int)B, (int)W, (int)H, c.code, s);
      if (rc != RG_OK) return rc;
      return rg_linear_rows(y, out_w, out_b, nullptr, op, wp, bytes, (int)B,
                            (int)W, N, 1, 0, s);
    });
    return triple(out, h, conv);
  });
}

// ------------------------------------------------- a prompt's attention --

struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// LocalAttentionBlock on a prompt without a cache (bf16, 256-wide heads, more rows than
// the few-row kernels take): projections, rotary embedding, attention, ring cache and
// proj_final, each where and as modules.linears and ops.attention_prompt would run it.
// As calls from Python it was 75 to 90 us of host time, which prompts of up to some 900
// tokens in all waited for: us a call, before and after, width 2560, 1 x 135 tokens
// 77 / 42, 7 x 72 88 / 54, 10 x 91 89 / 70, 7 x 739 165 / 164; width 4096, 1 x 300 89 / 69.
// (the block's _modules, x, segment_pos, inv_freq, first_key, heads, window, scale,
//  return_cache) -> (out, ring keys | None, ring values | None, num_tokens | None) | None
PyObject* attention_prompt(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 9);
#define RG_NAME(ID, TEXT) \
  static PyObject* const ID = PyUnicode_InternFromString(TEXT);
    RG_NAME(k_q, "proj_q") RG_NAME(k_k, "proj_k") RG_NAME(k_v, "proj_v")
    RG_NAME(k_final, "proj_final") RG_NAME(k_weight, "weight") RG_NAME(k_bias, "bias")
#undef RG_NAME
    PyObject *m_q = child(v[0], k_q), *m_k = child(v[0], k_k), *m_v = child(v[0], k_v),
             *m_final = child(v[0], k_final);
    for (PyObject* m : {m_q, m_k, m_v}) need(child(parameters(m), k_bias) == Py_None);
    const Tensor &w_q = parameter(m_q, k_weight), &w_k = parameter(m_k, k_weight),
                 &w_v = parameter(m_v, k_weight), &w_o = parameter(m_final, k_weight),
                 &b_o = parameter(m_final, k_bias);
    Call c(v[1]);
    need(c.code == RG_DTYPE_BF16 && c.x.dim() == 3 && c.x.numel() > 0 &&
         !at::autocast::is_autocast_enabled(at::kCUDA));
    const int64_t B = c.x.size(0), T = c.x.size(1), W = c.x.size(2), rows = B * T;
    const long H = PyLong_AsLong(v[5]), window = PyLong_AsLong(v[6]);
    const double scale = PyFloat_AsDouble(v[7]);
    if (PyErr_Occurred()) throw Raised{};
    constexpr int64_t kHead = 256;
    need(H > 0 && window > 0 && W == H * kHead && B <= INT32_MAX && T * H * 512 < INT32_MAX &&
         window <= INT32_MAX);
    need(shape_is(w_q, {W, W}) && shape_is(w_k, {kHead, W}) && shape_is(w_v, {kHead, W}) &&
         shape_is(w_o, {W, W}) && shape_is(b_o, {W}));
    void* x = c(v[1]);
    int is64;
    void* pos = c.positions(v[2], B, T, &is64);
    const float* inv = (const float*)c.f32(v[3], {kHead / 4});
    const Tensor& first = tensor_of(v[4]);
    need(shape_is(first, {B, T}));
    const int32_t* first_key = (const int32_t*)dense(first, at::kInt, c.device);
    for (const Tensor* t : {&w_q, &w_k, &w_v, &w_o, &b_o}) dense(*t, c.dtype, c.device);
    // (another thread may replace a parameter while this one is without the interpreter)
    const Tensor keep[] = {w_q, w_k, w_v, w_o, b_o};
    void* s = c.stream();

    const int n_qkv[3] = {(int)W, (int)kHead, (int)kHead}, n_out[1] = {(int)W};
    const bool qkv_ours = rg_linear_many_pays(rows, (int)W, 3, n_qkv, c.code);
    const bool out_ours = rg_linear_many_pays(rows, (int)W, 1, n_out, c.code);
    Tensor q, k, val, attended = c.empty({B, T, W}), out, ring_k, ring_v, count;
    if (qkv_ours) {
      q = c.empty({B, T, W});
      k = c.empty({B, T, kHead});
      val = c.empty({B, T, kHead});
    } else {
      NoGil free;
      q = at::linear(c.x, keep[0]);
      k = at::linear(c.x, keep[1]);
      val = at::linear(c.x, keep[2]);
    }
    if (v[8] == Py_True) {
      ring_k = c.empty({B, window, 1, kHead});
      ring_v = c.empty({B, window, 1, kHead});
      count = c.empty({B}, at::kInt);
    }
    if (out_ours) out = c.empty({B, T, W});
    Tensor ws = c.empty({(int64_t)rg_attention_prompt_workspace_bytes((int)B, (int)T)},
                        at::kByte);
    auto at_of = [](Tensor& t) { return t.defined() ? t.mutable_data_ptr() : nullptr; };
    void *qp = at_of(q), *kp = at_of(k), *vp = at_of(val), *ap = at_of(attended),
         *op = at_of(out), *rk = at_of(ring_k), *rv = at_of(ring_v), *np = at_of(count),
         *wp = at_of(ws);
    const void* const w3[3] = {keep[0].const_data_ptr(), keep[1].const_data_ptr(),
                               keep[2].const_data_ptr()};
    const void* const w1[1] = {keep[3].const_data_ptr()};
    const void* const b1[1] = {keep[4].const_data_ptr()};
    launch([&] {
      if (qkv_ours) {
        void* const to[3] = {qp, kp, vp};
        const int rc =
            rg_linear_many(x, rows, (int)W, 3, w3, nullptr, to, n_qkv, c.code, s);
        if (rc != RG_OK) return rc;
      }
      const int rc = rg_attention_prompt(
          qp, kp, vp, pos, is64, inv, first_key, ap, rk, rv, (int32_t*)np, wp, (int)B,
          (int)T, (int)H, (int)kHead, (int)window, (float)scale, c.code, s);
      if (rc != RG_OK || !out_ours) return rc;
      void* const to[1] = {op};
      return rg_linear_many(ap, rows, (int)W, 1, w1, b1, to, n_out, c.code, s);
    });
    if (!out_ours) {
      NoGil free;
      out = at::linear(attended, keep[3], keep[4]);
    }
    PyObject* t = PyTuple_New(4);
    if (!t) throw Raised{};
    int i = 0;
    for (const Tensor* each : {&out, &ring_k, &ring_v, &count})
      PyTuple_SET_ITEM(t, i++, wrap(*each));
    return t;
  });
}

PyObject* set_kernel_error(PyObject*, PyObject* type) {
  Py_INCREF(type);
  Py_XDECREF(g_kernel_error);
  g_kernel_error = type;
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"recurrent_step", (PyCFunction)(void*)recurrent_step, METH_FASTCALL, ""},
    {"recurrent_core", (PyCFunction)(void*)recurrent_core, METH_FASTCALL, ""},
    {"block_step", (PyCFunction)(void*)block_step, METH_FASTCALL, ""},
    {"attention_prompt", (PyCFunction)(void*)attention_prompt, METH_FASTCALL, ""},
    {"rows_plan", (PyCFunction)(void*)rows_plan, METH_FASTCALL, ""},
    {"rows_linear", (PyCFunction)(void*)rows_linear, METH_FASTCALL, ""},
    {"rows_partial", (PyCFunction)(void*)rows_partial, METH_FASTCALL, ""},
    {"remember_packed", (PyCFunction)(void*)remember_packed, METH_FASTCALL, ""},
    {"linear_scan", (PyCFunction)(void*)linear_scan, METH_FASTCALL, ""},
    {"train_scan", (PyCFunction)(void*)train_scan, METH_FASTCALL, ""},
    {"train_rglru", (PyCFunction)(void*)train_rglru, METH_FASTCALL, ""},
    {"train_block", (PyCFunction)(void*)train_block, METH_FASTCALL, ""},
    {"set_kernel_error", set_kernel_error, METH_O, ""},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host_ops", nullptr, -1,
                       kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__host_ops(void) {
  g_packed = new std::unordered_map<c10::TensorImpl*, PackedEntry>();
  return PyModule_Create(&kModule);
}

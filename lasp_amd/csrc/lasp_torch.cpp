// The PyTorch side of the library in native code: argument checks, allocations and autograd of the operators' usual
// case, above the C ABI of include/lasp_hip.h.
//
// A call on a short sequence is bound by the host: the kernels of a forward + backward over 256 tokens on 8 heads take
// 23 us, while the Python path around them (ctypes with twenty arguments, a torch.autograd.Function in Python,
// whose backward also has to take the interpreter lock on autograd's thread) took 49-108 us.  Here a forward is one
// C++ call (5.7 us with its launch, against about 22) that leaves one autograd node behind, and a backward never enters
// the interpreter (but for the state exchange of a sequence-parallel chain, which is Python).  Forward + backward, before
// and now: b*h = 8, n = 256: 101 and 53 us, of which some 35 are autograd's own handover to its device thread; b*h = 96,
// n = 512: 108 and 52 us (the kernels); eight chained chunks of 2048 tokens at b*h = 24: 762 and 674 us.
//
// "Usual case": contiguity aside, what the kernels take as it is -- device tensors of one type, fp32 with
// widths that are multiples of 4 or 16 bits with multiples of 8, float32 slopes on the same device.  Everything else (padding, other
// types, errors to report; tensor subclasses, function transforms, tracing and forward-mode differentiation, which a
// node built here would not be seen by) stays with lasp_amd/_abi.py and lasp_amd/_chain.py: the functions below return
// None for it.
#include <ATen/TensorSubclassLikeUtils.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <sstream>
#include <unordered_map>

#include "lasp_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ---- errors ------------------------------------------------------------------------------------------------
PyObject *g_error = nullptr;  // lasp_amd._abi.LaspError

// The Python exception LaspError, from whatever thread autograd runs this on.
[[noreturn]] void raise_lasp(const std::string &msg) {
  pybind11::gil_scoped_acquire gil;
  PyErr_SetString(g_error ? g_error : PyExc_RuntimeError, msg.c_str());
  python_error err;
  err.persist();
  throw err;
}
[[noreturn]] void raise_lasp(int rc, const char *what) {
  raise_lasp(std::string(what) + " failed (code " + std::to_string(rc) + "): " + lasp_last_error());
}

// ---- shapes ------------------------------------------------------------------------------------------------
struct Shape {
  int b, h, d, e, dtype;
  int64_t n;
};

int dtype_code(const Tensor &t) {
  switch (t.scalar_type()) {
    case at::kFloat: return LASP_DTYPE_F32;
    case at::kBFloat16: return LASP_DTYPE_BF16;
    case at::kHalf: return LASP_DTYPE_F16;
    default: return -1;
  }
}

Shape shape_of(const Tensor &q, const Tensor &v) {
  Shape sh;
  sh.b = (int)q.size(0);
  sh.h = (int)q.size(1);
  sh.n = q.size(2);
  sh.d = (int)q.size(3);
  sh.e = (int)v.size(3);
  sh.dtype = dtype_code(q);
  return sh;
}

// A tensor whose operations others follow through the dispatcher or a tangent: only the Python autograd Function is seen
// by them (and refuses what it has no rule for).
bool followed(const Tensor &t) { return at::isTensorSubclassLike(t) || t._fw_grad(0).defined(); }

// What the library takes as a few tokens under their states, of any type and without a workspace.
bool is_step(int64_t n, int64_t d, int64_t e) { return n <= LASP_STEP_TOKENS && d <= 128 && e <= 128 && e % 4 == 0; }

// fp32 rows that the MFMA kernels take under a call of their own
bool is_narrow(const Shape &sh) { return sh.dtype == LASP_DTYPE_F32 && (sh.d != 128 || sh.e != 128); }

// What a narrow row's kernel fetches 16 bytes at a time: memory that starts elsewhere (a view into a larger buffer) is copied, as it
// was when such rows were padded.
Tensor rows(const Tensor &t, const Shape &sh) { return is_narrow(sh) && (uintptr_t)t.data_ptr() % 16 ? t.clone() : t; }

// The usual case, see above; fills `sh`.  `keep`: the segment states are kept for a backward.
bool regular(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &s, Shape &sh, bool keep = true) {
  if (torch::jit::tracer::isTracing() || followed(q) || followed(k) || followed(v) || followed(s)) return false;
  if (!q.is_cuda() || q.dim() != 4 || v.dim() != 4 || k.sizes() != q.sizes() || q.numel() == 0 || v.numel() == 0) return false;
  if (k.device() != q.device() || v.device() != q.device() || s.device() != q.device()) return false;
  if (k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type()) return false;
  for (int i = 0; i < 3; ++i)
    if (v.size(i) != q.size(i)) return false;
  if (q.size(0) > INT32_MAX || q.size(1) > INT32_MAX || s.scalar_type() != at::kFloat || s.numel() != q.size(1) || !s.is_contiguous())
    return false;
  const int dtype = dtype_code(q);
  const int64_t d = q.size(3), e = v.size(3);
  if (keep || dtype < 0 || !is_step(q.size(2), d, e))
    if (dtype == LASP_DTYPE_F32 ? d % 4 || e % 4 || d > 128 || e > 128 : dtype < 0 || d % 8 || e % 8 || d > 1024 || e > 128) return false;
  sh = shape_of(q, v);
  return true;
}

bool state_ok(const Tensor &t, const Shape &sh, const Tensor &q) {
  return !t.defined() || (t.scalar_type() == at::kFloat && t.device() == q.device() && t.is_contiguous() && t.dim() == 4 &&
                          t.size(0) == sh.b && t.size(1) == sh.h && t.size(2) == sh.d && t.size(3) == sh.e);
}

// A state that comes out of the exchange is whatever another chunk of the chain left there: the kernels may read (b, h, d, e)
// floats only where there are as many.
void check_state(const char *name, const Tensor &t, const Shape &sh, const Tensor &q) {
  if (state_ok(t, sh, q)) return;
  std::ostringstream msg;
  msg << name << " must be a contiguous float32 tensor of shape (" << sh.b << ", " << sh.h << ", " << sh.d << ", " << sh.e
      << ") on " << q.device() << ", got " << t.scalar_type() << " " << t.sizes() << " on " << t.device();
  raise_lasp(msg.str());
}

void *data(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }

// ---- the two calls -----------------------------------------------------------------------------------------
struct Plan {
  int seg_len = 0, n_seg = 1;
  size_t bytes = 0;
  bool fused = false;  // one launch, no workspace, no states; seg_len stays 0 so that the backward chooses alike
};
Plan plan_of(const Shape &sh, int seg_len) {
  Plan p;
  if (seg_len == 0) {
    const int path = lasp_kernel_path(sh.b, sh.h, sh.n, sh.d, sh.e, sh.dtype);
    if (path < 0) raise_lasp(path, "lasp_kernel_path");
    if (path == LASP_PATH_MFMA_FUSED) {
      p.fused = true;
      return p;
    }
  }
  const int rc = lasp_plan(sh.b, sh.h, sh.n, sh.d, sh.e, sh.dtype, seg_len, &p.seg_len, &p.n_seg, &p.bytes);
  if (rc) raise_lasp(rc, "lasp_plan");
  return p;
}

// `in`, or a copy where `out` is the same memory and this shape's kernels cannot update a state in place.  States of narrow fp32 rows
// may also lie partly over each other, as they may where rows are padded; the library refuses that.
Tensor private_incoming(const Tensor &in, const Tensor &out, const Shape &sh, int seg_len, bool backward) {
  if (!in.defined() || !out.defined()) return in;
  const uintptr_t a = (uintptr_t)in.data_ptr(), b = (uintptr_t)out.data_ptr();
  if (a != b) return is_narrow(sh) && a < b + out.nbytes() && b < a + in.nbytes() ? in.clone() : in;
  return lasp_inplace_ok(sh.b, sh.h, sh.n, sh.d, sh.e, sh.dtype, seg_len, backward) == 1 ? in : in.clone();
}

Tensor floats(size_t bytes, const Tensor &like) {
  return at::empty({(int64_t)(bytes / sizeof(float))}, like.options().dtype(at::kFloat));
}

struct Forward {
  Tensor o, states;
  int seg_len = 0;
};
// What a forward leaves for a backward: nothing; what `run_backward` below needs to be fast, which is nothing where both run in one launch
// (where the forward leaves a state, it has the segments' too); the segment states, for a caller who may hand them on.
enum Keep { KEEP_NOTHING, KEEP_WHAT_PAYS, KEEP_STATES };
// q, k, v contiguous
Forward run_forward(const Shape &sh, Tensor q, Tensor k, Tensor v, const Tensor &s, Tensor kv_in,
                    const Tensor &kv_out, const Tensor &kv_twin, int seg_len, Keep keep = KEEP_STATES) {
  const auto stream = [&] { return c10::hip::getCurrentHIPStream(q.device().index()).stream(); };
  Forward f;
  f.o = at::empty(v.sizes(), v.options());
  if (keep == KEEP_NOTHING && seg_len == 0 && !kv_twin.defined() && is_step(sh.n, sh.d, sh.e)) {
    const int rc = lasp_step_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), (const float *)s.data_ptr(), (const float *)data(kv_in),
                                 (float *)data(kv_out), f.o.data_ptr(), sh.b, sh.h, sh.n, sh.d, sh.e, sh.dtype, stream());
    if (rc) raise_lasp(rc, "lasp_step_fwd");
    return f;
  }
  if (seg_len == 0 && !kv_in.defined() && !kv_out.defined()) seg_len = lasp_stateless_seg_len(sh.b, sh.h, sh.n, sh.d, sh.e, sh.dtype);
  const Plan p = plan_of(sh, seg_len);
  // (not where a state leaves: the one launch adds all of a chunk up in one accumulator, and without decay KV_out is two to three times
  // as far from 64 bits as sums of segments are: b*h = 24, n = 2048 2.9e-7 and 1.0e-7)
  if (!p.fused && keep != KEEP_STATES && seg_len == 0 && sh.dtype != LASP_DTYPE_F32 && !kv_out.defined() &&
      lasp_whole_ok(sh.b, sh.h, sh.n, sh.d, sh.e, sh.dtype, keep == KEEP_WHAT_PAYS) == 1) {
    const int rc = lasp_whole_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), (const float *)s.data_ptr(), (const float *)data(kv_in),
                                  nullptr, nullptr, f.o.data_ptr(), sh.b, sh.h, sh.n, sh.d, sh.e, sh.dtype, stream());
    if (rc) raise_lasp(rc, "lasp_whole_fwd");
    return f;
  }
  kv_in = private_incoming(kv_in, kv_out, sh, p.seg_len, false);
  q = rows(q, sh), k = rows(k, sh), v = rows(v, sh);
  f.seg_len = p.seg_len;
  if (!p.fused && (p.n_seg > 1 || kv_in.defined() || kv_out.defined())) f.states = floats(p.bytes, q);
  const int rc = (is_narrow(sh) ? lasp_narrow_fwd : lasp_chunk_fwd_twin)(q.data_ptr(), k.data_ptr(), v.data_ptr(), (const float *)s.data_ptr(),
                                     (const float *)data(kv_in), (float *)data(kv_out), (float *)data(kv_twin), f.o.data_ptr(),
                                     (float *)data(f.states), sh.b, sh.h, sh.n, sh.d, sh.e, sh.dtype, p.seg_len, stream());
  if (rc) raise_lasp(rc, "lasp_chunk_fwd");
  return f;
}

struct Backward {
  Tensor dq, dk, dv;
};
// q, k, v, d_o contiguous; `states` undefined: rebuilt
Backward run_backward(const Shape &sh, Tensor q, Tensor k, Tensor v, const Tensor &s, Tensor d_o,
                      const Tensor &kv_in, Tensor dkv_in, const Tensor &dkv_out, const Tensor &dkv_twin, const Tensor &states, int seg_len) {
  const Plan p = plan_of(sh, seg_len);
  dkv_in = private_incoming(dkv_in, dkv_out, sh, p.seg_len, true);
  Backward r;
  r.dq = at::empty(q.sizes(), q.options());
  r.dk = at::empty(q.sizes(), q.options());
  r.dv = at::empty(v.sizes(), v.options());
  const bool need_dkv = !p.fused && (p.n_seg > 1 || dkv_in.defined() || dkv_out.defined());
  const bool need_kv = !p.fused && !states.defined() && (p.n_seg > 1 || kv_in.defined());
  const size_t bytes = p.bytes * ((need_dkv ? 1 : 0) + (need_kv ? 1 : 0));
  Tensor ws;
  if (bytes) ws = floats(bytes, q);
  q = rows(q, sh), k = rows(k, sh), v = rows(v, sh), d_o = rows(d_o, sh);
  const int rc = (is_narrow(sh) ? lasp_narrow_bwd : lasp_chunk_bwd_twin)(q.data_ptr(), k.data_ptr(), v.data_ptr(), (const float *)s.data_ptr(), d_o.data_ptr(),
                                (const float *)data(kv_in), (const float *)data(dkv_in), r.dq.data_ptr(), r.dk.data_ptr(),
                                r.dv.data_ptr(), (float *)data(dkv_out), (float *)data(dkv_twin),
                                p.fused ? nullptr : (const float *)data(states), (float *)data(ws), bytes, sh.b, sh.h, sh.n,
                                sh.d, sh.e, sh.dtype, p.seg_len, c10::hip::getCurrentHIPStream(q.device().index()).stream());
  if (rc) raise_lasp(rc, "lasp_chunk_bwd");
  return r;
}

// ---- autograd ----------------------------------------------------------------------------------------------
// Python side of a chain's backward: before(exchange, DKV) -> (dkv_in, dkv_out, dkv_twin), each may be None, receives the
// state from the next rank; after(exchange, dkv_out, dkv_twin) sends the one that this chunk leaves.
PyObject *g_before = nullptr, *g_after = nullptr;
// sent(exchange, kv_out, kv_twin): sends the state that the forward of a chunk leaves.
PyObject *g_sent = nullptr;

template <class F>
void call_python(F &&f) {
  pybind11::gil_scoped_acquire gil;
  try {
    f();
  } catch (pybind11::error_already_set &e) {
    e.restore();
    python_error err;
    err.persist();
    throw err;
  }
}
pybind11::object borrowed(PyObject *p) { return pybind11::reinterpret_borrow<pybind11::object>(p); }
std::optional<Tensor> or_nothing(const Tensor &t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; }

// A Python object as a tensor: one int64, under which `handles` (guarded by the interpreter lock) holds a reference for as long
// as the tensor's memory lives.  Unlike the object, a tensor may be among the things that an autograd context carries through
// compiled autograd.
std::unordered_map<int64_t, PyObject *> &handles() {
  static auto *table = new std::unordered_map<int64_t, PyObject *>();
  return *table;
}
Tensor handle_of(PyObject *object) {
  static int64_t last = 0;
  pybind11::gil_scoped_acquire gil;
  auto *id = new int64_t(++last);
  Py_INCREF(object);
  handles()[*id] = object;
  const auto drop = [](void *p) {  // on any thread
    auto *id = static_cast<int64_t *>(p);
    if (Py_IsInitialized()) {
      pybind11::gil_scoped_acquire gil;
      const auto held = handles().find(*id);
      PyObject *object = held->second;
      handles().erase(held);
      Py_DECREF(object);
    }
    delete id;
  };
  return at::from_blob(id, {1}, drop, at::TensorOptions().dtype(at::kLong));
}
pybind11::object object_of(const Tensor &handle) {  // under the interpreter lock
  const auto held = handles().find(*handle.data_ptr<int64_t>());
  if (held == handles().end()) raise_lasp("the exchange of this chunk is gone");
  return borrowed(held->second);
}

// What a chunk of a chain brings along beside the inputs that take part in the graph (all empty without a chain).
struct Chain {
  Tensor kv_in, kv_out, kv_twin;
  Tensor dkv_buffer;  // the caller's DKV: later backward calls overwrite it, so it is kept by reference, not as a saved tensor
  PyObject *exchange = nullptr;
};

Forward forward_call(const Shape &sh, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &s, const Chain &chain,
                     Keep keep) {
  Forward f;
  {
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    f = run_forward(sh, q.contiguous(), k.contiguous(), v.contiguous(), s, chain.kv_in, chain.kv_out, chain.kv_twin, 0, keep);
  }
  // Before any tensor is saved: a hook on one may end a recomputed forward there (torch.utils.checkpoint does), and the next
  // rank, which recomputes too, waits for this state.
  if (chain.exchange) call_python([&] { borrowed(g_sent)(borrowed(chain.exchange), or_nothing(chain.kv_out), or_nothing(chain.kv_twin)); });
  return f;
}

// The operator for autograd.  Compiled autograd calls `backward` as it is: it is left at is_traceable = false.
struct LaspChunk : public torch::autograd::Function<LaspChunk> {
  static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &s, const Shape &sh,
                        const Chain &chain) {
    const Forward f = forward_call(sh, q, k, v, s, chain, KEEP_WHAT_PAYS);
    variable_list saved{q, k, v, s};
    if (f.states.defined()) saved.push_back(f.states);
    if (chain.kv_in.defined()) saved.push_back(chain.kv_in);
    ctx->save_for_backward(std::move(saved));
    // (a list, whose numbers compiled autograd takes as constants of the call; a short chunk without a state has none to keep)
    if (f.seg_len != 0 || f.states.defined() || chain.kv_in.defined())
      ctx->saved_data["call"] = c10::List<int64_t>({f.seg_len, f.states.defined(), chain.kv_in.defined()});
    if (chain.exchange) {
      ctx->saved_data["dkv_buffer"] = chain.dkv_buffer;
      ctx->saved_data["exchange"] = handle_of(chain.exchange);
    }
    return f.o;
  }

  // (no gradient for the output arrives as one of zeros: a chunk of a chain still has its neighbours' states to pass on)
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor q = saved[0].contiguous(), k = saved[1].contiguous(), v = saved[2].contiguous(), s = saved[3];
    Tensor states, kv_in;
    int seg_len = 0;
    auto &data = ctx->saved_data;
    const auto call = data.empty() ? data.end() : data.find("call"), in_chain = data.empty() ? data.end() : data.find("exchange");
    if (call != data.end()) {
      const c10::List<int64_t> numbers = call->second.toIntList();
      seg_len = (int)numbers[0];
      if (numbers[1]) states = saved[4];
      if (numbers[2]) kv_in = saved.back();
    }
    const Tensor d_o = grads[0].contiguous();
    const Shape sh = shape_of(q, v);
    c10::OptionalDeviceGuard guard(q.device());
    Tensor dkv_in, dkv_out, dkv_twin, exchange;
    if (in_chain != data.end()) {
      exchange = in_chain->second.toTensor();
      const Tensor dkv_buffer = data.at("dkv_buffer").toTensor();
      call_python([&] {
        auto states = borrowed(g_before)(object_of(exchange), dkv_buffer)
                          .cast<std::tuple<std::optional<Tensor>, std::optional<Tensor>, std::optional<Tensor>>>();
        dkv_in = std::get<0>(states).value_or(Tensor());
        dkv_out = std::get<1>(states).value_or(Tensor());
        dkv_twin = std::get<2>(states).value_or(Tensor());
      });
    }
    check_state("dkv_in", dkv_in, sh, q);
    check_state("dkv_out", dkv_out, sh, q);
    check_state("dkv_twin", dkv_twin, sh, q);
    Backward r;
    {
      at::AutoDispatchBelowADInplaceOrView below_autograd;  // (not around the exchange, whose writes to DKV count as versions)
      r = run_backward(sh, q, k, v, s, d_o, kv_in, dkv_in, dkv_out, dkv_twin, states, seg_len);
    }
    if (exchange.defined()) call_python([&] { borrowed(g_after)(object_of(exchange), or_nothing(dkv_out), or_nothing(dkv_twin)); });
    return {r.dq, r.dk, r.dv, Tensor(), Tensor(), Tensor()};
  }
};

std::optional<Tensor> operator_call(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &s, const Chain &chain) {
  Shape sh;
  if (!regular(q, k, v, s, sh)) return std::nullopt;
  check_state("kv_in", chain.kv_in, sh, q);
  check_state("kv_out", chain.kv_out, sh, q);
  check_state("kv_twin", chain.kv_twin, sh, q);
  const bool grad = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad() || s.requires_grad());
  c10::OptionalDeviceGuard guard(q.device());
  return grad ? LaspChunk::apply(q, k, v, s, sh, chain) : forward_call(sh, q, k, v, s, chain, KEEP_NOTHING).o;
}

Tensor or_none(const std::optional<Tensor> &t) { return t ? *t : Tensor(); }

}  // namespace

PYBIND11_MODULE(_lasp_torch, m) {
  namespace py = pybind11;
  m.def("bind", [](py::object error, py::object before, py::object after, py::object sent) {
    g_error = error.release().ptr();
    g_before = before.release().ptr();
    g_after = after.release().ptr();
    g_sent = sent.release().ptr();
  });
  // The interpreter lock is free while these run, as it is during a ctypes call: an allocation may wait for the driver, and a
  // launch for room in its queue.
  using unlocked = py::call_guard<py::gil_scoped_release>;
  // the stateless operator
  m.def(
      "attention",
      [](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &s) { return operator_call(q, k, v, s, Chain()); },
      unlocked());
  // whether a chain's chunk is a usual case (asked before its incoming state is received); one without a KV or DKV buffer is not
  m.def("takes", [](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &s, const std::optional<Tensor> &KV,
                    const std::optional<Tensor> &DKV) {
    Shape sh;
    return KV && DKV && regular(q, k, v, s, sh) && state_ok(*KV, sh, q) && state_ok(*DKV, sh, q);
  });
  // a chunk of a chain
  m.def(
      "chunk",
      [](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &s, const std::optional<Tensor> &kv_in,
         const std::optional<Tensor> &kv_out, const std::optional<Tensor> &kv_twin, const Tensor &dkv_buffer,
         const py::handle &exchange) {
        return operator_call(q, k, v, s, {or_none(kv_in), or_none(kv_out), or_none(kv_twin), dkv_buffer, exchange.ptr()});
      },
      unlocked());
  // _abi.chunk_fwd / chunk_bwd
  m.def(
      "chunk_fwd",
      [](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &s, const std::optional<Tensor> &kv_in,
         const std::optional<Tensor> &kv_out, int seg_len, bool keep) -> std::optional<std::tuple<Tensor, std::optional<Tensor>, int>> {
        Shape sh;
        const Tensor in = or_none(kv_in), out = or_none(kv_out);
        if (!regular(q, k, v, s, sh, keep) || !state_ok(in, sh, q) || !state_ok(out, sh, q)) return std::nullopt;
        c10::OptionalDeviceGuard guard(q.device());
        at::AutoDispatchBelowADInplaceOrView below_autograd;
        Forward f = run_forward(sh, q.contiguous(), k.contiguous(), v.contiguous(), s, in, out, Tensor(), seg_len, keep ? KEEP_STATES : KEEP_NOTHING);
        return std::make_tuple(f.o, or_nothing(f.states), f.seg_len);
      },
      unlocked());
  m.def(
      "chunk_bwd",
      [](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &s, const Tensor &d_o, const std::optional<Tensor> &kv_in,
         const std::optional<Tensor> &dkv_in, const std::optional<Tensor> &dkv_out, const std::optional<Tensor> &states,
         int seg_len) -> std::optional<std::tuple<Tensor, Tensor, Tensor>> {
        Shape sh;
        const Tensor in = or_none(kv_in), din = or_none(dkv_in), dout = or_none(dkv_out), st = or_none(states);
        if (!regular(q, k, v, s, sh) || !state_ok(in, sh, q) || !state_ok(din, sh, q) || !state_ok(dout, sh, q) ||
            d_o.device() != q.device() || d_o.scalar_type() != q.scalar_type() || d_o.sizes() != v.sizes())
          return std::nullopt;
        if (st.defined()) {  // what chunk_fwd returned for this shape
          const Plan p = plan_of(sh, seg_len);
          if (!p.fused && (st.scalar_type() != at::kFloat || st.device() != q.device() || !st.is_contiguous() ||
                           (size_t)st.numel() * sizeof(float) != p.bytes))
            return std::nullopt;
        }
        c10::OptionalDeviceGuard guard(q.device());
        at::AutoDispatchBelowADInplaceOrView below_autograd;
        Backward r = run_backward(sh, q.contiguous(), k.contiguous(), v.contiguous(), s, d_o.contiguous(), in, din, dout, Tensor(), st, seg_len);
        return std::make_tuple(r.dq, r.dk, r.dv);
      },
      unlocked());
}

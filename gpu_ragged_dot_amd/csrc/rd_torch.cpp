// The torch front end's host path in native code: argument checks, plan, output and workspace allocation, the call across
// the C ABI, and the autograd nodes.  ops.py and moe.py keep the Python signatures and hand their arguments on.
//
// What it is for: a call that keeps the GPU busy for 5-60 us (a decoding step, a toy training step, the routing around a
// small batch) was bound by the interpreter - about 45 us per product forward, and 55 more per gradient through a Python
// autograd node, which also takes the interpreter lock in the engine's thread.  512 x 256 x 512 in 4 groups, forward and
// both gradients: 182 us per pass with Python nodes over ctypes, 69 here (59 since the kernels look their tiles up themselves,
// rd_lookup.h); a decoding step on 13 experts of 512 x 5248: 18.4 -> 8.3 us.  What a call costs the host: 8.6 us a product,
// 4.4 a dispatch, 0.2 of them for giving up the interpreter lock and taking it again.
#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/utils/pybind.h>

#include <limits>
#include <map>
#include <mutex>
#include <optional>
#include <string>
#include <tuple>

#include "../../include/ragged_dot_hip.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

namespace {

constexpr int kOpGmm = 0, kOpGmmTrans = 1, kOpTgmm = 2;

struct StatusError : std::runtime_error {  // becomes _capi.RaggedDotError
  int status;
  StatusError(int s, const char* what) : std::runtime_error(what ? what : ""), status(s) {}
};
struct CheckError : std::runtime_error { using std::runtime_error::runtime_error; };  // AssertionError

void check(int status) {
  if (status != RD_OK) throw StatusError(status, rd_last_error());
}
void expect(bool ok, const char* what) {
  if (!ok) throw CheckError(what);
}

void set_python_error(const StatusError& e) {
  const py::object cls = py::module_::import("gpu_ragged_dot_amd._capi").attr("RaggedDotError");
  PyErr_SetObject(cls.ptr(), cls(e.status, e.what()).ptr());
}
void set_python_error(const CheckError& e) { PyErr_SetString(PyExc_AssertionError, e.what()); }
void set_python_error(const py::builtin_exception& e) { e.set_error(); }

// Only backward gradients are defined.  A tensor that carries a forward-mode tangent is refused, whether or not it asks for
// a gradient as well, as an operand and as a cotangent: the kernels would run on its value alone, and a result without a
// tangent reads as one of zero.
void expect_no_tangent(const Tensor& t) {
  TORCH_CHECK_NOT_IMPLEMENTED(!t.defined() || !t._fw_grad(0).defined(), "forward-mode derivatives are not implemented");
}
void expect_no_tangent(const Tensor& a, const Tensor& b) {
  expect_no_tangent(a);
  expect_no_tangent(b);
}

// The body of an autograd node's backward.  Its errors leave through torch's engine, possibly on a thread of its own, which
// hands on Python errors as they are and makes a RuntimeError of what it does not know: here they become the Python errors
// that the module's entry points raise.
template <class E>
[[noreturn]] void throw_python_error(const E& cause) {
  python_error e;
  {
    const py::gil_scoped_acquire gil;
    set_python_error(cause);
    e.persist();
  }
  throw e;
}
template <class F>
variable_list in_backward(const variable_list& grads, F&& body) {
  for (const Tensor& t : grads) expect_no_tangent(t);
  try {
    return body();
  } catch (const StatusError& e) {
    throw_python_error(e);
  } catch (const CheckError& e) {
    throw_python_error(e);
  } catch (const py::builtin_exception& e) {
    throw_python_error(e);
  }
}

// ---- plans -------------------------------------------------------------------------------------------------------------
// planner.py owns the tuned table and the choice for explicit block sizes; the table is handed over once, at import.  For the
// default block sizes pick_plan() is planner.select_plan() in native code (a host test compares the two).
std::map<std::tuple<int, int64_t, int64_t, int64_t, int64_t>, rd_plan> g_tuned;
std::mutex g_tuned_lock;

bool aligned16(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15) == 0; }

rd_plan pick_plan(int op, int64_t m, int64_t k, int64_t n, int64_t g, int code, bool aligned) {
  rd_plan p{-1, 0, 0, 0, 0};
  if (!aligned) {  // the library chooses among the shapes that take any address, whatever the table says
    check(rd_default_plan_any_address(op, (int)m, (int)k, (int)n, (int)g, code, &p));
    return p;
  }
  if (code == RD_DTYPE_BF16 && k % 8 == 0 && n % 8 == 0) {
    std::lock_guard<std::mutex> hold(g_tuned_lock);
    const auto it = g_tuned.find({op, m, k, n, g});
    if (it != g_tuned.end()) return it->second;
  }
  check(rd_default_plan(op, (int)m, (int)k, (int)n, (int)g, code, &p));
  return p;
}

// The plans of a call that does not leave them to the library: of the product, and of its two gradients where the caller has
// chosen those too (a plan for the product says nothing about the others).
struct Plans {
  size_t given = 0;
  rd_plan p[3];
};
rd_plan plan_from(py::handle h) {
  const auto t = py::cast<std::tuple<int, int, int, int, int>>(h);  // fields in the order of rd_plan
  return rd_plan{std::get<0>(t), std::get<1>(t), std::get<2>(t), std::get<3>(t), std::get<4>(t)};
}
Plans plans_from(const py::object& o) {
  Plans r;
  if (o.is_none()) return r;
  const auto t = py::cast<py::tuple>(o);
  for (; r.given < 3 && r.given < t.size(); ++r.given) r.p[r.given] = plan_from(t[r.given]);
  return r;
}

// ---- the products ------------------------------------------------------------------------------------------------------
void check_devices(const Tensor& a, const Tensor& b) {
  if (!a.is_cuda())
    throw std::runtime_error("ragged_dot runs on a ROCm device only (tensors must be on 'cuda'); there is no CPU path. "
                             "interpret=True of the reference (the Pallas interpreter) has no counterpart here.");
  if (b.device() != a.device()) throw std::runtime_error("all operands must live on the same device");
}

// (also in the gradients: a cotangent need not have its operand's type - float8 products come out as bfloat16)
void same_type(const Tensor& a, const Tensor& b) {
  TORCH_CHECK_TYPE(a.scalar_type() == b.scalar_type(), "the operands are ", a.scalar_type(), " and ", b.scalar_type());
}

// (the C ABI takes 32-bit sizes)
void expect_int(std::initializer_list<int64_t> sizes) {
  for (const int64_t s : sizes)
    if (s > std::numeric_limits<int>::max()) throw StatusError(RD_ERR_INVALID_ARGUMENT, "a size is beyond 2^31 - 1");
}

Tensor sizes_on(const Tensor& gs, const at::Device& dev) {
  Tensor t = gs.scalar_type() == at::kInt ? gs : gs.to(at::kInt);
  if (t.device() != dev) t = t.to(dev);
  return t.contiguous();
}

at::ScalarType out_type(const Tensor& t) { return t.scalar_type() == at::kFloat8_e4m3fn ? at::kBFloat16 : t.scalar_type(); }

// (its own buffer per call: the caching allocator hands it back to the stream that used it)
Tensor scratch(size_t bytes, const at::Device& dev) {
  return at::empty({(int64_t)(bytes < 256 ? 256 : bytes)}, at::TensorOptions().dtype(at::kByte).device(dev));
}

void* stream_of(const at::Device& dev) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).stream(); }

struct Call {
  int code = 0;
  bool trans = false;
  int64_t g_first = -1;  // first group of A / of the result; -1: all groups
  int64_t g_local = -1;  // tgmm: groups of the result; -1: up to the last one
  Plans plans;
};

// gpu_ragged_dot.py:171-228 (_gpu_gmm_fwd)
Tensor gmm_forward(const Tensor& x_, const Tensor& A_, const Tensor& gs_, const Call& c, size_t which, bool trans) {
  expect(A_.dim() == 3 && x_.dim() == 2, "x must be [m, k] and A [g, k, n]");  // :188
  same_type(x_, A_);
  expect(gs_.dim() == 1, "group_sizes must have one dimension");
  const int64_t g_local = A_.size(0), g = gs_.numel(), g_first = c.g_first < 0 ? 0 : c.g_first;
  expect(c.g_first < 0 ? g_local == g : g_first + g_local <= g, "A does not hold the groups that group_sizes describes");  // :189
  const int64_t m = x_.size(0), k = x_.size(1), n = A_.size(trans ? 1 : 2);  // :190
  expect(A_.size(trans ? 2 : 1) == k, "contraction mismatch between x and A");
  expect_int({m, k, n, g});
  check_devices(x_, A_);
  const at::Device dev = x_.device();
  const Tensor x = x_.contiguous(), A = A_.contiguous(), gs = sizes_on(gs_, dev);
  const c10::DeviceGuard guard(dev);
  Tensor y = at::empty({m, n}, x.options().dtype(out_type(x)).requires_grad(false));  // :210
  const bool aligned = aligned16(x) && aligned16(A) && aligned16(y);
  rd_plan p;
  if (which < c.plans.given && (which == 0 || aligned || c.code == RD_DTYPE_F32)) p = c.plans.p[which];
  else p = pick_plan(trans ? kOpGmmTrans : kOpGmm, m, k, n, g, c.code, aligned);
  if (g_first != 0 || g_local != g) p.decode_nb = 0;  // streaming kernels: all groups only
  const Tensor ws = scratch(rd_gmm_workspace_bytes((int)m, (int)g, &p), dev);
  check(rd_gmm_sharded(stream_of(dev), x.const_data_ptr(), A.const_data_ptr(), gs.const_data_ptr<int32_t>(), y.mutable_data_ptr(),
                       (int)m, (int)k, (int)n, (int)g, (int)g_first, (int)g_local, trans, c.code, &p, ws.mutable_data_ptr(), ws.numel()));
  return y;
}

// gpu_ragged_dot.py:287-342 (_gpu_tgmm_fwd)
Tensor tgmm_forward(const Tensor& x_, const Tensor& y_, const Tensor& gs_, const Call& c, size_t which, int64_t g_local) {
  expect(y_.dim() == 2 && x_.dim() == 2 && x_.size(0) == y_.size(0), "x must be [m, k] and y [m, n]");  // :304
  same_type(x_, y_);
  const int64_t m = x_.size(0), k = x_.size(1), n = y_.size(1), g = gs_.numel(), g_first = c.g_first < 0 ? 0 : c.g_first;
  if (g_local < 0) g_local = g - g_first;
  expect(g_local >= 1 && g_first + g_local <= g, "the groups asked for are not within group_sizes");
  expect_int({m, k, n, g});
  check_devices(x_, y_);
  const at::Device dev = x_.device();
  const Tensor x = x_.contiguous(), y = y_.contiguous(), gs = sizes_on(gs_, dev);
  const c10::DeviceGuard guard(dev);
  Tensor out = at::empty({g_local, k, n}, x.options().dtype(out_type(x)).requires_grad(false));  // :324
  const bool aligned = aligned16(x) && aligned16(y) && aligned16(out);
  rd_plan p;
  if (which < c.plans.given && (which == 0 || aligned || c.code == RD_DTYPE_F32)) p = c.plans.p[which];
  else p = pick_plan(kOpTgmm, m, k, n, g, c.code, aligned);
  const Tensor ws = scratch(rd_tgmm_workspace_bytes((int)m, (int)g, &p), dev);
  check(rd_tgmm_sharded(stream_of(dev), x.const_data_ptr(), y.const_data_ptr(), gs.const_data_ptr<int32_t>(), out.mutable_data_ptr(),
                        (int)m, (int)k, (int)n, (int)g, (int)g_first, (int)g_local, c.code, &p, ws.mutable_data_ptr(), ws.numel()));
  return out;
}

struct CallHolder : torch::CustomClassHolder {
  Call c;
  explicit CallHolder(const Call& call) : c(call) {}
};
Call call_of(AutogradContext* ctx) { return static_cast<CallHolder*>(ctx->saved_data["call"].toCapsule().get())->c; }

// The custom VJP of gpu_ragged_dot.py:360-405.
struct GmmNode : torch::autograd::Function<GmmNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& A, const Tensor& gs, const Call& c) {
    const Tensor sizes = sizes_on(gs, x.device());
    ctx->save_for_backward({x, A, sizes});  // residuals, :227
    ctx->saved_data["call"] = c10::IValue::make_capsule(c10::make_intrusive<CallHolder>(c));
    return gmm_forward(x, A, sizes, c, 0, c.trans);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    return in_backward(grads, [&]() -> variable_list {
      const auto saved = ctx->get_saved_variables();
      const Call c = call_of(ctx);
      const Tensor &x = saved[0], &A = saved[1], &gs = saved[2];
      const Tensor dy = grads[0].contiguous();
      Tensor dx, dA;
      if (ctx->needs_input_grad(0)) dx = gmm_forward(dy, A, gs, c, 1, !c.trans);  // :400
      if (ctx->needs_input_grad(1)) dA = c.trans ? tgmm_forward(dy, x, gs, c, 2, A.size(0)) : tgmm_forward(x, dy, gs, c, 2, A.size(0));  // :401
      return {dx, dA, Tensor(), Tensor()};  // group_sizes gets no cotangent, :402
    });
  }
};

// tgmm with the VJP gpu_ragged_dot.py:431-450 intends: dx = gmm(y, do, trans_rhs=True), dy = gmm(x, do).
struct TgmmNode : torch::autograd::Function<TgmmNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& y, const Tensor& gs, const Call& c) {
    const Tensor sizes = sizes_on(gs, x.device());
    ctx->save_for_backward({x, y, sizes});
    ctx->saved_data["call"] = c10::IValue::make_capsule(c10::make_intrusive<CallHolder>(c));
    return tgmm_forward(x, y, sizes, c, 0, c.g_local);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    return in_backward(grads, [&]() -> variable_list {
      const auto saved = ctx->get_saved_variables();
      const Call c = call_of(ctx);
      const Tensor dA = grads[0].contiguous();
      Tensor dx, dy;
      if (ctx->needs_input_grad(0)) dx = gmm_forward(saved[1], dA, saved[2], c, 1, true);
      if (ctx->needs_input_grad(1)) dy = gmm_forward(saved[0], dA, saved[2], c, 2, false);
      return {dx, dy, Tensor(), Tensor()};
    });
  }
};

bool wants_grad(const Tensor& a, const Tensor& b) {
  return at::GradMode::is_enabled() && (a.requires_grad() || b.requires_grad());
}

// Called without the interpreter lock, as everything below that may wait - for memory, for a copy of group_sizes from the
// host, for the driver - so that other Python threads run meanwhile.
Tensor gmm(const Tensor& x, const Tensor& A, const Tensor& gs, bool trans, int code, int64_t g_first, const Plans& plans) {
  expect_no_tangent(x, A);
  if (x.scalar_type() != A.scalar_type()) throw py::type_error("x and A have different element types");
  Call c;
  c.code = code; c.trans = trans; c.g_first = g_first; c.plans = plans;
  if (!wants_grad(x, A)) return gmm_forward(x, A, gs, c, 0, trans);
  check_devices(x, A);
  return GmmNode::apply(x, A, gs, c);
}

Tensor tgmm(const Tensor& x, const Tensor& y, const Tensor& gs, int code, int64_t g_first, int64_t g_local, const Plans& plans) {
  expect_no_tangent(x, y);
  if (x.scalar_type() != y.scalar_type()) throw py::type_error("x and y have different element types");
  Call c;
  // a number of groups without a first one means the first ones (the gradients' A then holds those only)
  c.code = code; c.g_first = g_first < 0 && g_local >= 0 ? 0 : g_first; c.g_local = g_local; c.plans = plans;
  if (!wants_grad(x, y)) return tgmm_forward(x, y, gs, c, 0, g_local);
  check_devices(x, y);
  return TgmmNode::apply(x, y, gs, c);
}

// ---- token routing -----------------------------------------------------------------------------------------------------
struct Routing {
  Tensor row_of_slot, slot_of_row;
  int64_t tokens, top_k;
};

std::tuple<Tensor, Tensor, Tensor> moe_route(const Tensor& ids_, int64_t groups) {
  if (ids_.dim() != 2) throw py::value_error("expert_ids must be [tokens, top_k]");
  expect_int({ids_.size(0), ids_.size(1), groups});
  check_devices(ids_, ids_);
  const at::Device dev = ids_.device();
  const Tensor ids = sizes_on(ids_, dev);
  const c10::DeviceGuard guard(dev);
  const int64_t tokens = ids.size(0), top_k = ids.size(1), slots = tokens * top_k;
  const auto opts = at::TensorOptions().dtype(at::kInt).device(dev);
  Tensor sizes = at::empty({groups}, opts), row_of_slot = at::empty({slots}, opts), slot_of_row = at::empty({slots}, opts);
  const Tensor ws = scratch(rd_moe_route_workspace_bytes((int)tokens, (int)top_k, (int)groups), dev);
  check(rd_moe_route(stream_of(dev), ids.const_data_ptr<int32_t>(), (int)tokens, (int)top_k, (int)groups, sizes.mutable_data_ptr<int32_t>(),
                     row_of_slot.mutable_data_ptr<int32_t>(), slot_of_row.mutable_data_ptr<int32_t>(), ws.mutable_data_ptr(), ws.numel()));
  return {sizes, row_of_slot, slot_of_row};
}

int rows_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return RD_DTYPE_BF16;
    case at::kHalf: return RD_DTYPE_F16;
    case at::kFloat: return RD_DTYPE_F32;
    default: throw py::type_error("unsupported dtype; rows are bfloat16, float16 or float32");
  }
}

// Everything a kernel reads through a pointer is on the rows' device and as long as the kernel takes it to be.
void check_routing(const Tensor& rows, const Routing& r, const Tensor& per_slot) {
  check_devices(rows, r.row_of_slot);
  check_devices(rows, r.slot_of_row);
  if (per_slot.defined()) check_devices(rows, per_slot);
  const int64_t slots = r.tokens * r.top_k;
  if (r.row_of_slot.numel() < slots || r.slot_of_row.numel() < slots || !r.row_of_slot.is_contiguous() || !r.slot_of_row.is_contiguous() ||
      (per_slot.defined() && (per_slot.numel() < slots || !per_slot.is_contiguous())))
    throw py::value_error("a routing of " + std::to_string(slots) + " slots needs that many contiguous entries in each of its arrays");
}

Tensor dispatch_rows(const Tensor& h_, const Routing& r, const Tensor& scale) {
  if (h_.dim() != 2 || h_.size(0) != r.tokens) throw py::value_error("h must be [" + std::to_string(r.tokens) + ", d]");
  expect_int({r.tokens, r.top_k, h_.size(1)});
  check_routing(h_, r, scale);
  const Tensor h = h_.contiguous();
  const int code = rows_code(h);
  const c10::DeviceGuard guard(h.device());
  Tensor x = at::empty({r.tokens * r.top_k, h.size(1)}, h.options().requires_grad(false));
  check(rd_moe_dispatch(stream_of(h.device()), h.const_data_ptr(), r.row_of_slot.const_data_ptr<int32_t>(), r.slot_of_row.const_data_ptr<int32_t>(),
                        scale.defined() ? scale.const_data_ptr<float>() : nullptr, x.mutable_data_ptr(), (int)r.tokens, (int)r.top_k, (int)h.size(1), code));
  return x;
}

Tensor combine_rows(const Tensor& y_, const Routing& r, const Tensor& weights) {
  if (y_.dim() != 2 || y_.size(0) != r.tokens * r.top_k) throw py::value_error("y must be [" + std::to_string(r.tokens * r.top_k) + ", d]");
  expect_int({r.tokens, r.top_k, y_.size(1)});
  check_routing(y_, r, weights);
  const Tensor y = y_.contiguous();
  const int code = rows_code(y);
  const c10::DeviceGuard guard(y.device());
  Tensor out = at::empty({r.tokens, y.size(1)}, y.options().requires_grad(false));
  check(rd_moe_combine(stream_of(y.device()), y.const_data_ptr(), r.row_of_slot.const_data_ptr<int32_t>(),
                       weights.defined() ? weights.const_data_ptr<float>() : nullptr, out.mutable_data_ptr(), (int)r.tokens, (int)r.top_k, (int)y.size(1), code));
  return out;
}

Tensor combine_wgrad(const Tensor& y_, const Tensor& dout_, const Routing& r) {
  check_devices(y_, dout_);
  const Tensor y = y_.contiguous(), dout = dout_.contiguous();
  const c10::DeviceGuard guard(y.device());
  Tensor dw = at::empty({r.tokens * r.top_k}, y.options().dtype(at::kFloat).requires_grad(false));
  check(rd_moe_combine_wgrad(stream_of(y.device()), y.const_data_ptr(), dout.const_data_ptr(), r.row_of_slot.const_data_ptr<int32_t>(),
                             dw.mutable_data_ptr<float>(), (int)r.tokens, (int)r.top_k, (int)y.size(1), rows_code(y)));
  return dw;
}

// A node keeps its routing aside from its saved tensors: a dispatch saves none, so that gradients can be taken through it
// any number of times without retain_graph.
struct RoutingHolder : torch::CustomClassHolder {
  Routing r;
  explicit RoutingHolder(const Routing& routing) : r(routing) {}
};
Routing routing_of(AutogradContext* ctx) { return static_cast<RoutingHolder*>(ctx->saved_data["routing"].toCapsule().get())->r; }
void keep_routing(AutogradContext* ctx, const Routing& r) {
  ctx->saved_data["routing"] = c10::IValue::make_capsule(c10::make_intrusive<RoutingHolder>(r));
}

struct DispatchNode : torch::autograd::Function<DispatchNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& h, const Routing& r) {
    keep_routing(ctx, r);
    return dispatch_rows(h, r, Tensor());
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    return in_backward(grads, [&]() -> variable_list {
      return {combine_rows(grads[0], routing_of(ctx), Tensor()), Tensor()};  // each token collects the gradients of its rows
    });
  }
};

struct CombineNode : torch::autograd::Function<CombineNode> {
  static Tensor forward(AutogradContext* ctx, const Tensor& y, const std::optional<Tensor>& weights, const Routing& r) {
    const Tensor w = weights.value_or(Tensor());
    ctx->save_for_backward({y, w});
    keep_routing(ctx, r);
    return combine_rows(y, r, w);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    return in_backward(grads, [&]() -> variable_list {
      const auto s = ctx->get_saved_variables();
      const Routing r = routing_of(ctx);
      const Tensor &y = s[0], &w = s[1], &dout = grads[0];
      Tensor dy, dw;
      if (ctx->needs_input_grad(0)) dy = dispatch_rows(dout, r, w);  // dy[row] = weight of the row's slot * dout[token]
      if (w.defined() && ctx->needs_input_grad(1)) dw = combine_wgrad(y, dout, r);
      return {dy, dw, Tensor()};
    });
  }
};

Tensor moe_dispatch(const Tensor& h, const Tensor& row_of_slot, const Tensor& slot_of_row, int64_t tokens, int64_t top_k) {
  const Routing r{row_of_slot, slot_of_row, tokens, top_k};
  expect_no_tangent(h, h);
  if (!wants_grad(h, h)) return dispatch_rows(h, r, Tensor());
  return DispatchNode::apply(h, r);
}

Tensor moe_combine(const Tensor& y, const std::optional<Tensor>& weights, const Tensor& row_of_slot, const Tensor& slot_of_row,
                   int64_t tokens, int64_t top_k) {
  const Routing r{row_of_slot, slot_of_row, tokens, top_k};
  expect_no_tangent(y, weights.value_or(y));
  std::optional<Tensor> w;
  if (weights) {
    Tensor t = weights->reshape({-1});
    if (t.scalar_type() != at::kFloat || !t.is_contiguous()) t = t.to(at::kFloat).contiguous();
    if (t.numel() != tokens * top_k) throw py::value_error("weights must have " + std::to_string(tokens * top_k) + " entries");
    w = t;
  }
  if (!wants_grad(y, w ? *w : y)) return combine_rows(y, r, w.value_or(Tensor()));
  return CombineNode::apply(y, w, r);
}

}  // namespace

PYBIND11_MODULE(_rd_torch, mod) {
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const StatusError& e) {
      set_python_error(e);
    } catch (const CheckError& e) {
      set_python_error(e);
    }
  });
  mod.def("set_tuned_plans", [](const py::list& entries) {  // [((op, m, k, n, g), (variant, group_m, group_n, decode_nb, split_k)), ...]
    std::lock_guard<std::mutex> hold(g_tuned_lock);
    g_tuned.clear();
    for (const auto& e : entries) {
      const auto kv = py::cast<py::tuple>(e);
      g_tuned[py::cast<std::tuple<int, int64_t, int64_t, int64_t, int64_t>>(kv[0])] = plan_from(kv[1]);
    }
  });
  mod.def("pick_plan", [](int op, int64_t m, int64_t k, int64_t n, int64_t g, int code, bool aligned) {
    const rd_plan p = pick_plan(op, m, k, n, g, code, aligned);
    return std::make_tuple(p.variant, p.group_m, p.group_n, p.decode_nb, p.split_k);
  });
  typedef py::call_guard<py::gil_scoped_release> unlocked;  // (held again for the result and for errors)
  mod.def("gmm", [](const Tensor& x, const Tensor& A, const Tensor& gs, bool trans, int code, int64_t g_first, const py::object& plans) {
    const Plans p = plans_from(plans);
    const py::gil_scoped_release without_lock;
    return gmm(x, A, gs, trans, code, g_first, p);
  });
  mod.def("tgmm", [](const Tensor& x, const Tensor& y, const Tensor& gs, int code, int64_t g_first, int64_t g_local, const py::object& plans) {
    const Plans p = plans_from(plans);
    const py::gil_scoped_release without_lock;
    return tgmm(x, y, gs, code, g_first, g_local, p);
  });
  mod.def("moe_route", &moe_route, unlocked());
  mod.def("moe_dispatch", &moe_dispatch, unlocked());
  mod.def("moe_dispatch_rows", [](const Tensor& h, const std::optional<Tensor>& scale, const Tensor& row_of_slot, const Tensor& slot_of_row,
                                  int64_t tokens, int64_t top_k) {
    return dispatch_rows(h, Routing{row_of_slot, slot_of_row, tokens, top_k}, scale.value_or(Tensor()));
  }, unlocked());
  mod.def("moe_combine", &moe_combine, unlocked());
}

// A call on a whole sequence from Python: operands, workspace, the library's one call and the autograd node, without
// Python code on the way.  Small calls are host code: the forward of 1024 fp32 tokens, H=4, took 32 us of it as a Python
// autograd function over ctypes for 19 us of kernels, a training call on 2 x 2048 packed tokens 160 for 76; 19 and 91 so.
//
// The library's entry points come in as addresses (init), so that it runs on the build that the package has loaded.  forward and backward
// are the call without its node and conversions.
#include <Python.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/types.h>

#include <atomic>
#include <cmath>
#include <cstring>
#include <vector>

#include "../../include/ring_attention_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

struct Library {
  decltype(&ra_fwd_call) fwd_call;
  decltype(&ra_bwd_call) bwd_call;
  decltype(&ra_bwd_whole_workspace) bwd_workspace;
  decltype(&ra_convert) convert;
  PyObject* check;  // _lib.check: raises what the code says
} g_lib;

// (the error text is the calling thread's, and so is the Python error that check makes of it)
void check(const char* what, int code) {
  if (code == 0) return;
  pybind11::gil_scoped_acquire gil;
  PyObject* r = PyObject_CallFunction(g_lib.check, "si", what, code);
  Py_XDECREF(r);
  TORCH_CHECK(!r, what, " failed with code ", code);
  python_error e;
  e.persist();
  throw e;
}

// (a plan on the host has none: tests of this file)
void* stream(const at::Device& device) { return device.is_cpu() ? nullptr : c10::hip::getCurrentHIPStream().stream(); }

int row_dtype(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return RA_DTYPE_BF16;
    case at::kFloat: return RA_DTYPE_F32;
    case at::kHalf: return RA_DTYPE_F16;
    default: return -1;
  }
}

Tensor empty(at::IntArrayRef shape, at::ScalarType dtype, const at::Device& device) {
  return at::empty(shape, at::TensorOptions().dtype(dtype).device(device));
}

// The ra_rows that converts [b, l, h, *] to contiguous rows of d elements at dst; false for what ra_convert does not take.
bool rows_of(ra_rows& r, const Tensor& t, void* dst, at::ScalarType to, int64_t d) {
  const int src = row_dtype(t.scalar_type()), dt = row_dtype(to);
  const int64_t B = t.size(0), L = t.size(1), H = t.size(2);
  if (src < 0 || dt < 0 || t.stride(3) != 1 || !t.is_cuda() || B >= 65536 || B * L * H <= 0 || L * H >= (int64_t)1 << 27) return false;
  r = ra_rows{t.data_ptr(), dst, src, dt, (int32_t)t.size(3), (int32_t)d, (int32_t)B, (int32_t)L, (int32_t)H,
              t.stride(0), t.stride(1), t.stride(2), L * H * d, H * d, d};
  return true;
}

constexpr int kMostArrays = 4;  // (of one ra_convert)

// [b, l, h, *] tensors as new contiguous [b, l, h, d] ones of the dtypes given, in one launch where ra_convert takes them: cast, and cut or padded with zeros.  What it does
// not take (other dtypes, a head dimension that is not contiguous, more rows than a launch holds) goes through torch.
void convert(Tensor* const* t, const at::ScalarType* to, int n, int64_t d) {
  std::vector<ra_rows> rows;
  std::vector<Tensor> from;  // (alive until the launch)
  const at::Device device = t[0]->device();
  for (int i = 0; i < n; ++i) {
    const Tensor x = *t[i];
    from.push_back(x);
    Tensor o = empty({x.size(0), x.size(1), x.size(2), d}, to[i], device);
    ra_rows r;
    if (x.device() == device && rows_of(r, x, o.data_ptr(), to[i], d)) rows.push_back(r);
    else o.copy_(x.size(3) >= d ? x.narrow(3, 0, d) : at::constant_pad_nd(x, {0, d - x.size(3)}));
    *t[i] = o;
  }
  if (!rows.empty()) check("ra_convert", g_lib.convert(rows.data(), (int)rows.size(), stream(device)));
}

// bf16 [b, l, h, d] as the kernels take it: unit inner stride, aligned rows that do not overlap, within the ABI's row stride.
Tensor ready(const Tensor& t) {
  const bool ok = t.stride(3) == 1 && !((t.stride(0) | t.stride(1) | t.stride(2)) & 7) && !(reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) &&
                  t.size(3) <= t.stride(1) && t.stride(1) <= (int64_t)1 << 27;
  return ok ? t : t.contiguous();
}

bool is_operand(const Tensor& t, int64_t d) { return t.scalar_type() == at::kBFloat16 && t.size(3) == d; }

// Tensors as the kernels of head dim d take them, in place.
void operands(Tensor* const* t, int n, int64_t d) {
  Tensor* todo[kMostArrays];
  const at::ScalarType bf16[kMostArrays] = {at::kBFloat16, at::kBFloat16, at::kBFloat16, at::kBFloat16};
  int m = 0;
  for (int i = 0; i < n; ++i) {
    if (is_operand(*t[i], d)) *t[i] = ready(*t[i]);
    else todo[m++] = t[i];
  }
  if (m) convert(todo, bf16, m, d);
}

ra_tensor view(const Tensor& t) { return ra_tensor{t.data_ptr(), t.stride(0), t.stride(2), t.stride(1)}; }
ra_tensor rows_at(const void* p, int64_t L, int64_t H, int64_t D) { return ra_tensor{p, L * H * D, D, H * D}; }

// What the calls of one plan share.  The arrays are those that the bias points into.
struct Plan : torch::CustomClassHolder {
  int64_t B, H, Lq, Lk, D;
  ra_bias bias;
  int64_t fwd_bytes;
  std::atomic<int64_t> bwd_bytes{-1};  // -1: no backward has asked for it (a call without gradients does not pay for its plan)
  at::Device device = at::kCPU;
  std::vector<Tensor> arrays;
};
struct Call : torch::CustomClassHolder {
  c10::intrusive_ptr<Plan> plan;
  float scale;
  int64_t dim;
  at::ScalarType given[3];
};

// q, k and v of a call: three tensors, or one buffer that holds the three converted ones.
void operand_views(const Plan& p, const variable_list& kept, ra_tensor (&x)[3]) {
  if (kept.size() == 3) {
    for (int i = 0; i < 3; ++i) x[i] = view(kept[i]);
    return;
  }
  const char* at = (const char*)kept[0].data_ptr();
  const int64_t nq = 2 * p.B * p.Lq * p.H * p.D, nk = 2 * p.B * p.Lk * p.H * p.D;
  x[0] = rows_at(at, p.Lq, p.H, p.D);
  x[1] = rows_at(at + nq, p.Lk, p.H, p.D);
  x[2] = rows_at(at + nq + nk, p.Lk, p.H, p.D);
}

Tensor workspace(int64_t bytes, const at::Device& device) { return bytes ? empty({bytes}, at::kByte, device) : Tensor(); }
void* pointer(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// Output and logsumexp [1, b, h, l] of operands as the kernels take them, or as the `rows` before the call make them.
variable_list run_forward(const Plan& p, float scale, const variable_list& kept, const ra_rows* rows, int n_rows, at::ScalarType out_dtype) {
  Tensor out = empty({p.B, p.Lq, p.H, p.D}, out_dtype, p.device), lse = empty({1, p.B, p.H, p.Lq}, at::kFloat, p.device);
  const Tensor ws = workspace(p.fwd_bytes, p.device);
  ra_tensor x[3];
  operand_views(p, kept, x);
  const ra_fwd_step_params a{(int32_t)p.B, (int32_t)p.H, (int32_t)p.Lq, (int32_t)p.Lk, (int32_t)p.D, scale, x[0], x[1], x[2],
                             nullptr, nullptr, nullptr, p.bias};
  check("ra_fwd_call", g_lib.fwd_call(rows, n_rows, &a, out.data_ptr(), row_dtype(out_dtype), p.Lq * p.H * p.D, p.D, p.H * p.D,
                                      (float*)lse.data_ptr(), pointer(ws), p.fwd_bytes, stream(p.device)));
  return {out, lse};
}

// dq, dk and dv, of bf16 precision whatever their dtype.  dout: as the kernels take it, or as `rows` makes it.
variable_list run_backward(Plan& p, float scale, const variable_list& kept, const Tensor& out, const Tensor& lse, const ra_rows* rows, int n_rows,
                           const Tensor& dout, at::ScalarType dtype) {
  Tensor dq, dk, dv;
  if (kept.size() == 3) {
    // laid out as the operands; dk and dv have the same strides, which the library stores them with
    auto like = [&](const Tensor& t, bool preserve) {
      return at::empty_like(t, t.options().dtype(dtype), preserve ? at::MemoryFormat::Preserve : at::MemoryFormat::Contiguous);
    };
    const bool same = kept[1].strides() == kept[2].strides();
    dq = like(kept[0], true);
    dk = like(kept[1], same);
    dv = like(kept[2], same);
  } else {
    dq = empty({p.B, p.Lq, p.H, p.D}, dtype, p.device);
    dk = empty({p.B, p.Lk, p.H, p.D}, dtype, p.device);
    dv = empty({p.B, p.Lk, p.H, p.D}, dtype, p.device);
  }
  ra_tensor x[3];
  operand_views(p, kept, x);
  const float* l = (const float*)lse.data_ptr();
  const ra_bwd_step_params a{(int32_t)p.B, (int32_t)p.H, (int32_t)p.Lq, (int32_t)p.Lk, (int32_t)p.D, scale, x[0], x[1], x[2],
                             view(dout), l, nullptr, nullptr, nullptr, nullptr, p.bias};
  int64_t bytes = p.bwd_bytes.load(std::memory_order_relaxed);
  if (bytes < 0) p.bwd_bytes.store(bytes = g_lib.bwd_workspace(&a), std::memory_order_relaxed);  // (sizes and bias alone decide)
  const Tensor ws = workspace(bytes, p.device);
  const ra_tensor o = view(out), gq = view(dq), gk = view(dk);
  check("ra_bwd_call", g_lib.bwd_call(rows, n_rows, &a, o.ptr, row_dtype(out.scalar_type()), o.stride_b, o.stride_h, o.stride_l,
                                      row_dtype(dtype) | RA_DTYPE_VIA_BF16, dq.data_ptr(), gq.stride_b, gq.stride_h, gq.stride_l,
                                      dk.data_ptr(), dv.data_ptr(), gk.stride_b, gk.stride_h, gk.stride_l, pointer(ws), bytes,
                                      stream(p.device)));
  return {dq, dk, dv};
}

class WholeCall : public torch::autograd::Function<WholeCall> {
 public:
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, c10::intrusive_ptr<Plan> plan,
                               double scale, at::ScalarType out_dtype, at::ScalarType final_dtype, bool any_grad) {
    const Plan& p = *plan;
    auto call = c10::make_intrusive<Call>();
    call->plan = plan;
    call->scale = (float)scale;
    call->dim = q.size(3);
    const at::ScalarType dtype = call->given[0] = q.scalar_type();
    call->given[1] = k.scalar_type();
    call->given[2] = v.scalar_type();
    ra_rows rows[3];
    int n_rows = 0;
    variable_list kept;
    if (dtype == call->given[1] && dtype == call->given[2] && !is_operand(q, p.D)) {
      const int64_t nq = p.B * p.Lq * p.H * p.D, nk = p.B * p.Lk * p.H * p.D;
      Tensor buf = empty({nq + 2 * nk}, at::kBFloat16, q.device());
      char* at = (char*)buf.data_ptr();
      if (rows_of(rows[0], q, at, at::kBFloat16, p.D) && rows_of(rows[1], k, at + 2 * nq, at::kBFloat16, p.D) &&
          rows_of(rows[2], v, at + 2 * (nq + nk), at::kBFloat16, p.D)) {
        n_rows = 3;
        kept = {buf};
      }
    }
    if (!n_rows) {
      kept = {q, k, v};
      Tensor* x[3] = {&kept[0], &kept[1], &kept[2]};
      operands(x, 3, p.D);
    }
    variable_list got = run_forward(p, call->scale, kept, rows, n_rows, out_dtype);
    Tensor out = got[0], lse = got[1];
    kept.push_back(out);
    kept.push_back(lse);
    ctx->save_for_backward(kept);
    ctx->mark_non_differentiable({lse});
    ctx->set_materialize_grads(false);  // no zero fill for the logsumexp's gradient
    ctx->saved_data["call"] = c10::IValue::make_capsule(call);
    if (out_dtype != final_dtype || (call->dim != p.D && any_grad)) {
      Tensor* t = &out;
      convert(&t, &final_dtype, 1, call->dim);
    }
    return {out, lse};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads_in) {
    const auto call = c10::static_intrusive_pointer_cast<Call>(ctx->saved_data["call"].toCapsule());
    Plan& p = *call->plan;
    variable_list kept = ctx->get_saved_variables();
    const Tensor lse = kept.back(), out = kept[kept.size() - 2];
    kept.resize(kept.size() - 2);
    Tensor go = grads_in[0];
    if (!go.defined()) go = at::zeros(out.sizes(), out.options().dtype(at::kBFloat16));  // nothing came back for the output
    // as the caller wants them, where that takes no cut
    const bool direct = call->dim == p.D && row_dtype(call->given[0]) >= 0 && call->given[0] == call->given[1] && call->given[0] == call->given[2];
    const at::ScalarType dtype = direct ? call->given[0] : at::kBFloat16;
    ra_rows rows;
    int n_rows = 0;
    Tensor made = go;
    if (!is_operand(go, p.D) && go.device() == p.device) {
      made = empty({p.B, p.Lq, p.H, p.D}, at::kBFloat16, p.device);
      n_rows = rows_of(rows, go, made.data_ptr(), at::kBFloat16, p.D);
    }
    if (!n_rows) {
      made = go;
      Tensor* t = &made;
      operands(&t, 1, p.D);
    }
    variable_list grads = run_backward(p, call->scale, kept, out, lse, &rows, n_rows, made, dtype);
    Tensor* todo[3];
    at::ScalarType to[3];
    int n = 0;
    for (int i = 0; i < 3; ++i)
      if (ctx->needs_input_grad(i) && (call->dim != p.D || call->given[i] != dtype)) {
        todo[n] = &grads[i];
        to[n++] = call->given[i];
      }
    if (n) convert(todo, to, n, call->dim);
    for (int i = 0; i < 3; ++i)
      if (!ctx->needs_input_grad(i)) grads[i] = Tensor();
    return {grads[0], grads[1], grads[2], Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

constexpr const char* kPlanName = "ring_attention plan";

void drop_plan(PyObject* capsule) {
  delete static_cast<c10::intrusive_ptr<Plan>*>(PyCapsule_GetPointer(capsule, kPlanName));
}

// init(address of ra_fwd_call, of ra_bwd_call, of ra_bwd_whole_workspace, of ra_convert, check)
PyObject* init(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  unsigned long long f, b, w, c;
  PyObject* check_fn;
  if (!PyArg_ParseTuple(args, "KKKKO", &f, &b, &w, &c, &check_fn)) return nullptr;
  g_lib.fwd_call = reinterpret_cast<decltype(g_lib.fwd_call)>(static_cast<uintptr_t>(f));
  g_lib.bwd_call = reinterpret_cast<decltype(g_lib.bwd_call)>(static_cast<uintptr_t>(b));
  g_lib.bwd_workspace = reinterpret_cast<decltype(g_lib.bwd_workspace)>(static_cast<uintptr_t>(w));
  g_lib.convert = reinterpret_cast<decltype(g_lib.convert)>(static_cast<uintptr_t>(c));
  Py_INCREF(check_fn);
  Py_XSETREF(g_lib.check, check_fn);
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// plan(B, H, Lq, Lk, D, ra_bias block, bytes of the forward's workspace, q's device as a tensor, bias arrays)
PyObject* plan(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  long long B, H, Lq, Lk, D, fwd_bytes;
  Py_buffer bias;
  PyObject *like, *arrays;
  if (!PyArg_ParseTuple(args, "LLLLLy*LOO!", &B, &H, &Lq, &Lk, &D, &bias, &fwd_bytes, &like, &PyTuple_Type, &arrays)) return nullptr;
  auto p = c10::make_intrusive<Plan>();
  const bool fits = bias.len == sizeof(ra_bias);
  if (fits) std::memcpy(&p->bias, bias.buf, sizeof(ra_bias));
  PyBuffer_Release(&bias);
  TORCH_CHECK(fits, "the bias block is not an ra_bias");
  p->B = B;
  p->H = H;
  p->Lq = Lq;
  p->Lk = Lk;
  p->D = D;
  p->fwd_bytes = fwd_bytes;
  TORCH_CHECK_TYPE(THPVariable_Check(like), "a tensor is expected");
  p->device = THPVariable_Unpack(like).device();
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(arrays); ++i) {
    TORCH_CHECK_TYPE(THPVariable_Check(PyTuple_GET_ITEM(arrays, i)), "the bias arrays must be tensors");
    p->arrays.push_back(THPVariable_Unpack(PyTuple_GET_ITEM(arrays, i)));
  }
  return PyCapsule_New(new c10::intrusive_ptr<Plan>(std::move(p)), kPlanName, drop_plan);
  END_HANDLE_TH_ERRORS
}

const c10::intrusive_ptr<Plan>& plan_of(PyObject* capsule) {
  auto* p = static_cast<c10::intrusive_ptr<Plan>*>(PyCapsule_GetPointer(capsule, kPlanName));
  if (!p) throw python_error();
  return *p;
}
double scale_of(PyObject* x) {
  const double scale = PyFloat_AsDouble(x);
  if (scale == -1.0 && PyErr_Occurred()) throw python_error();
  return scale;
}
at::ScalarType dtype_of(PyObject* x) {
  TORCH_CHECK_TYPE(THPDtype_Check(x), "a dtype is expected");
  return reinterpret_cast<THPDtype*>(x)->scalar_type;
}
const Tensor& tensor_of(PyObject* x) {
  TORCH_CHECK_TYPE(THPVariable_Check(x), "a tensor is expected");
  return THPVariable_Unpack(x);
}
PyObject* tuple_of(variable_list&& tensors) {
  THPObjectPtr r(PyTuple_New((Py_ssize_t)tensors.size()));
  if (!r) throw python_error();
  for (size_t i = 0; i < tensors.size(); ++i) PyTuple_SET_ITEM(r.get(), (Py_ssize_t)i, THPVariable_Wrap(std::move(tensors[i])));
  return r.release();
}

// Pointers and strides are all that goes on from here.
void check_operands(const Plan& of, const Tensor& q, const Tensor& k, const Tensor& v) {
  const int64_t d = q.dim() == 4 ? q.size(3) : -1;
  TORCH_CHECK(d <= of.D && q.sizes() == at::IntArrayRef({of.B, of.Lq, of.H, d}) && k.sizes() == at::IntArrayRef({of.B, of.Lk, of.H, d}) &&
                  v.sizes() == k.sizes() && q.device() == of.device && k.device() == of.device && v.device() == of.device,
              "q ", q.sizes(), ", k ", k.sizes(), " and v ", v.sizes(), " are not the operands of this plan");
}

// attend(q, k, v, plan, scale, the kernels' output dtype, the caller's) -> output, logsumexp [1, b, h, l]
PyObject* attend(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 7, "attend(q, k, v, plan, scale, dtype, dtype)");
  const Tensor& q = tensor_of(args[0]);
  Tensor k = tensor_of(args[1]), v = tensor_of(args[2]);
  const c10::intrusive_ptr<Plan> p = plan_of(args[3]);
  const double scale = scale_of(args[4]);
  const at::ScalarType dtype = dtype_of(args[5]), final_dtype = dtype_of(args[6]);
  variable_list got;
  {
    pybind11::gil_scoped_release no_gil;  // (allocations may wait for the GPU)
    for (Tensor* t : {&k, &v})
      if (t->device() != q.device()) *t = t->to(q.device());  // (as the bias arrays are)
    check_operands(*p, q, k, v);
    const bool any_grad = q.requires_grad() || k.requires_grad() || v.requires_grad();
    got = WholeCall::apply(q, k, v, p, scale, dtype, final_dtype, any_grad);
  }
  return tuple_of(std::move(got));
  END_HANDLE_TH_ERRORS
}

void check_ready(const Plan& p, const variable_list& kept) {
  check_operands(p, kept[0], kept[1], kept[2]);
  for (const Tensor& t : kept) TORCH_CHECK(is_operand(t, p.D), "operands of bf16 and head dim ", p.D, " are expected, not of ", t.scalar_type(), " and ", t.size(3));
}

// forward(q, k, v, plan, scale, dtype) -> output, logsumexp, of operands as the kernels take them (operands)
PyObject* forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 6, "forward(q, k, v, plan, scale, dtype)");
  const variable_list kept{tensor_of(args[0]), tensor_of(args[1]), tensor_of(args[2])};
  Plan& p = *plan_of(args[3]);
  const double scale = scale_of(args[4]);
  const at::ScalarType dtype = dtype_of(args[5]);
  variable_list got;
  {
    pybind11::gil_scoped_release no_gil;
    check_ready(p, kept);
    got = run_forward(p, (float)scale, kept, nullptr, 0, dtype);
  }
  return tuple_of(std::move(got));
  END_HANDLE_TH_ERRORS
}

// backward(q, k, v, output, logsumexp, dout, plan, scale) -> bf16 dq, dk, dv; dout too as the kernels take it
PyObject* backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 8, "backward(q, k, v, output, logsumexp, dout, plan, scale)");
  const variable_list kept{tensor_of(args[0]), tensor_of(args[1]), tensor_of(args[2])};
  const Tensor out = tensor_of(args[3]), lse = tensor_of(args[4]), dout = tensor_of(args[5]);
  Plan& p = *plan_of(args[6]);
  const double scale = scale_of(args[7]);
  variable_list got;
  {
    pybind11::gil_scoped_release no_gil;
    check_ready(p, kept);
    TORCH_CHECK(out.sizes() == kept[0].sizes() && dout.sizes() == kept[0].sizes() && lse.numel() == p.B * p.H * p.Lq && out.device() == p.device &&
                    dout.device() == p.device && lse.device() == p.device,
                "output ", out.sizes(), ", its gradient ", dout.sizes(), " and logsumexp ", lse.sizes(), " are not those of q ", kept[0].sizes());
    got = run_backward(p, (float)scale, kept, out, lse, nullptr, 0, dout, at::kBFloat16);
  }
  return tuple_of(std::move(got));
  END_HANDLE_TH_ERRORS
}

variable_list tensors_of(PyObject* seq) {
  THPObjectPtr fast(PySequence_Fast(seq, "a sequence of tensors is expected"));
  if (!fast) throw python_error();
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(fast.get());
  TORCH_CHECK(n >= 1 && n <= kMostArrays, "1 to ", kMostArrays, " arrays at a time (got ", n, ")");
  variable_list got;
  for (Py_ssize_t i = 0; i < n; ++i) {
    got.push_back(tensor_of(PySequence_Fast_GET_ITEM(fast.get(), i)));
    TORCH_CHECK(got.back().dim() == 4, "[b, l, h, d] arrays are expected, not ", got.back().sizes());
  }
  return got;
}

// convert(tensors, dtypes, d) -> new contiguous [b, l, h, d] tensors
PyObject* convert_arrays(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 3, "convert(tensors, dtypes, d)");
  variable_list t = tensors_of(args[0]);
  THPObjectPtr dtypes(PySequence_Fast(args[1], "a sequence of dtypes is expected"));
  if (!dtypes) throw python_error();
  TORCH_CHECK(PySequence_Fast_GET_SIZE(dtypes.get()) == (Py_ssize_t)t.size(), "a dtype for each tensor is expected");
  const int64_t d = PyLong_AsLongLong(args[2]);
  if (d == -1 && PyErr_Occurred()) throw python_error();
  Tensor* at[kMostArrays];
  at::ScalarType to[kMostArrays];
  for (size_t i = 0; i < t.size(); ++i) {
    at[i] = &t[i];
    to[i] = dtype_of(PySequence_Fast_GET_ITEM(dtypes.get(), (Py_ssize_t)i));
  }
  {
    pybind11::gil_scoped_release no_gil;
    convert(at, to, (int)t.size(), d);
  }
  return tuple_of(std::move(t));
  END_HANDLE_TH_ERRORS
}

// operands(tensors, d) -> the tensors as the kernels of head dim d take them: themselves where they can be
PyObject* operand_arrays(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 2, "operands(tensors, d)");
  variable_list t = tensors_of(args[0]);
  const int64_t d = PyLong_AsLongLong(args[1]);
  if (d == -1 && PyErr_Occurred()) throw python_error();
  Tensor* at[kMostArrays];
  for (size_t i = 0; i < t.size(); ++i) at[i] = &t[i];
  {
    pybind11::gil_scoped_release no_gil;
    operands(at, (int)t.size(), d);
  }
  return tuple_of(std::move(t));
  END_HANDLE_TH_ERRORS
}

// require_pair(q, k, v, ...): see _require_pair of ring.py
PyObject* require_pair(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n >= 3, "require_pair(q, k, v, ...)");
  const Tensor &q = tensor_of(args[0]), &k = tensor_of(args[1]), &v = tensor_of(args[2]);
  TORCH_CHECK_VALUE(q.dim() == 4 && k.dim() == 4 && v.dim() == 4, "q, k and v must be [b, h, l, d]");
  bool holds = v.size(2) >= k.size(2), exact = v.size(2) == k.size(2);
  for (const Tensor* t : {&k, &v})
    for (int i : {0, 1, 3}) {
      holds &= t->size(i) >= q.size(i);
      exact &= t->size(i) == q.size(i);
    }
  TORCH_CHECK_VALUE(holds, "k ", k.sizes(), " and v ", v.sizes(), " do not hold the batch, heads and head dim of q ", q.sizes(),
                    ", or v not the length of k");
  const at::Device device = q.device();
  for (Py_ssize_t i = 1; i < n; ++i)
    TORCH_CHECK_VALUE(tensor_of(args[i]).device() == device, "all arrays of a block must be on the device of q (", device, ")");
  return PyBool_FromLong(exact);
  END_HANDLE_TH_ERRORS
}

PyMethodDef g_methods[] = {{"init", init, METH_VARARGS, nullptr},
                           {"plan", plan, METH_VARARGS, nullptr},
                           {"attend", (PyCFunction)(void (*)(void))attend, METH_FASTCALL, nullptr},
                           {"require_pair", (PyCFunction)(void (*)(void))require_pair, METH_FASTCALL, nullptr},
                           {"convert", (PyCFunction)(void (*)(void))convert_arrays, METH_FASTCALL, nullptr},
                           {"operands", (PyCFunction)(void (*)(void))operand_arrays, METH_FASTCALL, nullptr},
                           {"forward", (PyCFunction)(void (*)(void))forward, METH_FASTCALL, nullptr},
                           {"backward", (PyCFunction)(void (*)(void))backward, METH_FASTCALL, nullptr},
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_host", "Calls on whole sequences without Python code on the way.", -1, g_methods};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&g_module); }

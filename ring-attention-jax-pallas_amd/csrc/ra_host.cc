// A call on a whole sequence from Python: operands, workspace, the library's one call and the autograd node, without
// Python code on the way.  Small calls are host code: the forward of 1024 fp32 tokens, H=4, took 32 us of it as a Python
// autograd function over ctypes for 19 us of kernels, a training call on 2 x 2048 packed tokens 160 for 76; 19 and 91 so.
//
// Conversions are those of _convert and _kernel_inputs of ring.py, which the launch schemes of several shards keep; the library's entry
// points come in as addresses (init), so that it runs on the build that the package has loaded.
#include <Python.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
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

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

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

// [b, l, h, *] tensors as new contiguous [b, l, h, d] ones of the dtypes given, in one launch where ra_convert takes them.
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
  if (!rows.empty()) check("ra_convert", g_lib.convert(rows.data(), (int)rows.size(), stream()));
}

// bf16 [b, l, h, d] as the kernels take it: unit inner stride, aligned rows that do not overlap, within the ABI's row stride.
Tensor ready(const Tensor& t) {
  const bool ok = t.stride(3) == 1 && !((t.stride(0) | t.stride(1) | t.stride(2)) & 7) && !(reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) &&
                  t.size(3) <= t.stride(1) && t.stride(1) <= (int64_t)1 << 27;
  return ok ? t : t.contiguous();
}

bool is_operand(const Tensor& t, int64_t d) { return t.scalar_type() == at::kBFloat16 && t.size(3) == d; }

void operands(Tensor* const* t, int n, int64_t d) {
  Tensor* todo[3];
  const at::ScalarType bf16[3] = {at::kBFloat16, at::kBFloat16, at::kBFloat16};
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
    Tensor out = empty({p.B, p.Lq, p.H, p.D}, out_dtype, p.device), lse = empty({1, p.B, p.H, p.Lq}, at::kFloat, p.device);
    const Tensor ws = workspace(p.fwd_bytes, p.device);
    ra_tensor x[3];
    operand_views(p, kept, x);
    const ra_fwd_step_params a{(int32_t)p.B, (int32_t)p.H, (int32_t)p.Lq, (int32_t)p.Lk, (int32_t)p.D, call->scale, x[0], x[1], x[2],
                               nullptr, nullptr, nullptr, p.bias};
    check("ra_fwd_call", g_lib.fwd_call(rows, n_rows, &a, out.data_ptr(), row_dtype(out_dtype), p.Lq * p.H * p.D, p.D, p.H * p.D,
                                        (float*)lse.data_ptr(), pointer(ws), p.fwd_bytes, stream()));
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
    ra_tensor x[3];
    operand_views(p, kept, x);
    const float* l = (const float*)lse.data_ptr();
    const ra_bwd_step_params a{(int32_t)p.B, (int32_t)p.H, (int32_t)p.Lq, (int32_t)p.Lk, (int32_t)p.D, call->scale, x[0], x[1], x[2],
                               view(made), l, nullptr, nullptr, nullptr, nullptr, p.bias};
    int64_t bytes = p.bwd_bytes.load(std::memory_order_relaxed);
    if (bytes < 0) p.bwd_bytes.store(bytes = g_lib.bwd_workspace(&a), std::memory_order_relaxed);  // (sizes and bias alone decide)
    const Tensor ws = workspace(bytes, p.device);
    const ra_tensor o = view(out), gq = view(dq), gk = view(dk);
    check("ra_bwd_call", g_lib.bwd_call(&rows, n_rows, &a, o.ptr, row_dtype(out.scalar_type()), o.stride_b, o.stride_h, o.stride_l,
                                        row_dtype(dtype) | RA_DTYPE_VIA_BF16, dq.data_ptr(), gq.stride_b, gq.stride_h, gq.stride_l,
                                        dk.data_ptr(), dv.data_ptr(), gk.stride_b, gk.stride_h, gk.stride_l, pointer(ws), bytes,
                                        stream()));
    Tensor* g[3] = {&dq, &dk, &dv};
    Tensor* todo[3];
    at::ScalarType to[3];
    int n = 0;
    for (int i = 0; i < 3; ++i)
      if (ctx->needs_input_grad(i) && (call->dim != p.D || call->given[i] != dtype)) {
        todo[n] = g[i];
        to[n++] = call->given[i];
      }
    if (n) convert(todo, to, n, call->dim);
    for (int i = 0; i < 3; ++i)
      if (!ctx->needs_input_grad(i)) *g[i] = Tensor();
    return {dq, dk, dv, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
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

// attend(q, k, v, plan, scale, the kernels' output dtype, the caller's) -> output, logsumexp [1, b, h, l]
PyObject* attend(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n == 7 && THPVariable_Check(args[0]) && THPVariable_Check(args[1]) && THPVariable_Check(args[2]) && THPDtype_Check(args[5]) &&
                       THPDtype_Check(args[6]),
                   "attend(q, k, v, plan, scale, dtype, dtype)");
  auto* p = static_cast<c10::intrusive_ptr<Plan>*>(PyCapsule_GetPointer(args[3], kPlanName));
  if (!p) throw python_error();
  const double scale = PyFloat_AsDouble(args[4]);
  if (scale == -1.0 && PyErr_Occurred()) throw python_error();
  const Tensor& q = THPVariable_Unpack(args[0]);
  Tensor k = THPVariable_Unpack(args[1]), v = THPVariable_Unpack(args[2]);
  for (Tensor* t : {&k, &v})
    if (t->device() != q.device()) {  // (the kernels take pointers; the bias arrays went the same way)
      pybind11::gil_scoped_release no_gil;
      *t = t->to(q.device());
    }
  const Plan& of = **p;
  const int64_t d = q.dim() == 4 ? q.size(3) : -1;
  // (pointers and strides are all that goes on from here)
  TORCH_CHECK(d <= of.D && q.sizes() == at::IntArrayRef({of.B, of.Lq, of.H, d}) && k.sizes() == at::IntArrayRef({of.B, of.Lk, of.H, d}) &&
                  v.sizes() == k.sizes() && q.device() == of.device,
              "attend: q ", q.sizes(), " on ", q.device(), ", k ", k.sizes(), " and v ", v.sizes(), " are not the operands of this plan");
  const bool any_grad = q.requires_grad() || k.requires_grad() || v.requires_grad();
  const at::ScalarType dtype = reinterpret_cast<THPDtype*>(args[5])->scalar_type, final_dtype = reinterpret_cast<THPDtype*>(args[6])->scalar_type;
  variable_list got;
  {
    pybind11::gil_scoped_release no_gil;  // (allocations may wait for the GPU)
    got = WholeCall::apply(q, k, v, *p, scale, dtype, final_dtype, any_grad);
  }
  PyObject* r = PyTuple_New(2);
  if (!r) throw python_error();
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(std::move(got[0])));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(std::move(got[1])));
  return r;
  END_HANDLE_TH_ERRORS
}

PyMethodDef g_methods[] = {{"init", init, METH_VARARGS, nullptr},
                           {"plan", plan, METH_VARARGS, nullptr},
                           {"attend", (PyCFunction)(void (*)(void))attend, METH_FASTCALL, nullptr},
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_host", "Calls on whole sequences without Python code on the way.", -1, g_methods};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&g_module); }

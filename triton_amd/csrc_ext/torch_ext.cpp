// PyTorch-ROCm extension over the C ABI of include/mi355_kernels.h: the analogue of the reference's
// generated launcher (third_party/amd/backend/driver.py:326-377), which pulls pointers out of the
// tensor objects (`data_ptr()`, :285-323), takes the stream the caller's framework is on
// (python/triton/runtime/jit.py:588-589 passes torch's current stream) and launches.  Here: tensor
// checks, sizes / strides / dtypes read off the at::Tensor, c10::hip::getCurrentHIPStream(), one C call.
// No device code in this file and no logic beyond checks, allocation and argument marshalling: every status of the C ABI
// becomes the exception the reference raises for the same condition (RuntimeError "Triton Error [HIP]"
// for launch failures, :258-269; ValueError for pointers the device cannot reach, :313-317).
#include <torch/extension.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/mi355_kernels.h"

namespace py = pybind11;

namespace {

int abi_dtype(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kHalf: return MI355_F16;
    case at::kBFloat16: return MI355_BF16;
    case at::kFloat8_e4m3fn: return MI355_F8E4M3;
    case at::kFloat8_e5m2: return MI355_F8E5M2;
    case at::kFloat: return MI355_F32;
    default: throw py::type_error(std::string("unsupported dtype ") + c10::toString(t.scalar_type()));
  }
}

void on_device(const at::Tensor& t, int idx) {
  if (!t.is_cuda())
    throw std::invalid_argument("Pointer argument (at " + std::to_string(idx) + ") cannot be accessed from Triton (cpu tensor?)");
}

void check(int rc, const char* what) {
  if (rc == 0) return;
  const std::string msg = mi355_strerror(rc);
  if (rc > 0)
    throw std::runtime_error("Triton Error [HIP]:  Code: " + std::to_string(rc) + ", Messsage: " + msg + " (" + what + ")");
  throw std::invalid_argument(std::string(what) + ": " + msg + " (code " + std::to_string(rc) + ")");
}

// The C library launches on the CURRENT device: every operator makes its first tensor's device current for the call.
// (the generic guard: it resolves the implementation registered for the tensor's device type, which on ROCm builds of
// torch is the HIP one under the name "cuda")
using DeviceGuard = c10::DeviceGuard;

void* stream_of(const at::Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// Whether nobody stands between a call and the device: no dispatch mode, functorch level or tracer is on.
bool plain_dispatch() {
  return (c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set).empty();
}

// A result or workspace on the device of `like`.  Straight from the device's allocator where plain_dispatch(): the way through the
// dispatcher is host time of its own for every tensor of calls whose kernels run for 4 us.
at::Tensor fresh(at::IntArrayRef sizes, at::ScalarType type, const at::Tensor& like) {
  if (plain_dispatch() && like.layout() == at::kStrided) return at::detail::empty_cuda(sizes, type, like.device(), c10::nullopt);
  return at::empty(sizes, like.options().dtype(type));
}

// (a dimension of one element may have any stride in a contiguous tensor: the backward compares strides, so that these are kept too)
at::Tensor fresh_like(const at::Tensor& t) {
  int64_t dense = 1;
  for (int64_t d = t.dim() - 1; d >= 0; d--) {
    if (t.stride(d) != dense) return at::empty_like(t);
    dense *= t.size(d);
  }
  return fresh(t.sizes(), t.scalar_type(), t);
}

const float* scale_ptr(const c10::optional<at::Tensor>& s) {
  if (!s.has_value()) return nullptr;
  TORCH_CHECK(s->scalar_type() == at::kFloat && s->numel() == 1, "scales are one fp32 value per tensor");
  on_device(*s, -1);
  return s->data_ptr<float>();
}

[[noreturn]] void fail(PyObject* type, const std::string& message) {
  PyErr_SetString(type, message.c_str());
  throw py::error_already_set();
}

// C = softmax_rows?(act((a_scale * b_scale) * A @ B + add)): the checks of the reference's wrapper
// (python/tutorials/03-matrix-multiplication.py:330-348) with its exceptions, the result and the workspace from torch's
// allocator (which orders their reuse on the current stream), one C call.  activation: MI355_ACT_*.
at::Tensor matmul(const at::Tensor& a, const at::Tensor& b_in, int64_t activation, const c10::optional<at::ScalarType>& out_dtype,
                  const c10::optional<at::Tensor>& a_scale, const c10::optional<at::Tensor>& b_scale,
                  const c10::optional<at::Tensor>& add, bool softmax) {
  at::Tensor b = b_in;
  if (a.dim() != 2 || b.dim() != 2 || a.size(1) != b.size(0)) fail(PyExc_AssertionError, "Incompatible dimensions");
  if (!a.is_contiguous()) fail(PyExc_AssertionError, "Matrix A must be contiguous");
  const int in_dt = abi_dtype(a);
  if (a.scalar_type() != b.scalar_type()) fail(PyExc_AssertionError, "Incompatible dtypes");
  on_device(a, 0); on_device(b, 1);
  const DeviceGuard guard(a.device());
  const int64_t M = a.size(0), K = a.size(1), N = b.size(1);
  at::Tensor c = fresh({M, N}, out_dtype.has_value() ? *out_dtype : in_dt == MI355_BF16 ? at::kBFloat16 : at::kHalf, a);
  if (M == 0 || N == 0) return c;
  if (K == 0) return c.zero_();
  // fp32 operands run on the fp32 MFMAs with a K-major B only (the LDS transpose reads stop at 16-bit elements): a
  // row-major B is put K-major first - one transposing copy, 1 / M of the product's work -; small products and a K
  // that is not a multiple of four elements take the any-stride kernel of the C ABI as they are
  if (in_dt == MI355_F32 && b.stride(0) != 1 && K % 4 == 0 && M * N * K >= (1 << 24)) b = b.t().contiguous().t();
  const void* d = nullptr;
  int64_t dsm = 0, dsn = 0;
  int ddt = 0;
  at::Tensor wide;
  if (add.has_value()) {
    on_device(*add, 2);
    ddt = abi_dtype(*add);
    if (ddt != MI355_F16 && ddt != MI355_BF16 && ddt != MI355_F32) fail(PyExc_TypeError, std::string("add must be fp16, bf16 or fp32, got ") + c10::toString(add->scalar_type()));
    wide = add->expand({M, N});   // (zero strides on broadcast axes)
    d = wide.data_ptr(); dsm = wide.stride(0); dsn = wide.stride(1);
  }
  const int64_t need = mi355_gemm_workspace(a.data_ptr(), b.data_ptr(), (int)M, (int)N, (int)K, a.stride(0), a.stride(1), b.stride(0), b.stride(1), in_dt);
  at::Tensor ws;
  if (need > 0) ws = fresh({need}, at::kByte, a);
  const int rc = mi355_gemm_ws(a.data_ptr(), b.data_ptr(), c.data_ptr(), (int)M, (int)N, (int)K, a.stride(0), a.stride(1), b.stride(0), b.stride(1),
                               c.stride(0), c.stride(1), in_dt, abi_dtype(c), scale_ptr(a_scale), scale_ptr(b_scale),
                               d, dsm, dsn, ddt, (int)activation, softmax ? 1 : 0, need > 0 ? ws.data_ptr() : nullptr, (size_t)need, stream_of(a));
  check(rc, "mi355_gemm");
  return c;
}

void mx_gemm(const at::Tensor& a, const at::Tensor& sa, const at::Tensor& b, const at::Tensor& sb, at::Tensor& c, int64_t fmt, int64_t K) {
  on_device(a, 0); on_device(sa, 1); on_device(b, 2); on_device(sb, 3); on_device(c, 4);
  TORCH_CHECK(a.dim() == 2 && b.dim() == 2 && sa.dim() == 2 && sb.dim() == 2 && c.dim() == 2, "MX operands, scales and result are matrices");
  const DeviceGuard guard(a.device());
  const int64_t need = mi355_mx_gemm_workspace((int)a.size(0), (int)b.size(0), (int)K, (int)fmt);
  at::Tensor ws;
  if (need > 0) ws = fresh({need}, at::kByte, c);
  const int rc = mi355_mx_gemm_ws((const uint8_t*)a.data_ptr(), (const uint8_t*)sa.data_ptr(), (const uint8_t*)b.data_ptr(),
                                  (const uint8_t*)sb.data_ptr(), c.data_ptr(), (int)a.size(0), (int)b.size(0), (int)K, (int)fmt,
                                  abi_dtype(c), a.stride(0), b.stride(0), sa.stride(0), sb.stride(0), c.stride(0),
                                  need > 0 ? ws.data_ptr() : nullptr, (size_t)need, stream_of(a));
  check(rc, "mi355_mx_gemm");
}

// [A_i @ B_i for i]: results allocated here, the tables handed over in host memory
std::vector<at::Tensor> group_gemm(const std::vector<at::Tensor>& a, const std::vector<at::Tensor>& b, int64_t num_programs) {
  const size_t n = a.size();
  std::vector<at::Tensor> c;
  if (n == 0) return c;
  const DeviceGuard guard(a[0].device());
  std::vector<const void*> pa(n), pb(n);
  std::vector<void*> pc(n);
  std::vector<int32_t> sizes(3 * n), lds(3 * n);
  c.reserve(n);
  size_t used = 0;
  for (size_t i = 0; i < n; i++) {
    on_device(a[i], 2 * (int)i); on_device(b[i], 2 * (int)i + 1);
    TORCH_CHECK(a[i].dim() == 2 && b[i].dim() == 2, "grouped GEMM takes matrices");
    c.push_back(fresh({a[i].size(0), b[i].size(1)}, a[i].scalar_type(), a[i]));
    if (c[i].numel() == 0) continue;
    if (a[i].size(1) == 0) { c[i].zero_(); continue; }
    pa[used] = a[i].data_ptr(); pb[used] = b[i].data_ptr(); pc[used] = c[i].data_ptr();
    int32_t *s = &sizes[3 * used], *l = &lds[3 * used];
    s[0] = (int32_t)a[i].size(0); s[1] = (int32_t)b[i].size(1); s[2] = (int32_t)a[i].size(1);
    // (a matrix of one row may have any row stride)
    TORCH_CHECK(std::max({a[i].size(0), a[i].stride(0), b[i].size(0), b[i].size(1), b[i].stride(0)}) <= INT32_MAX, "sizes and row strides of a group's matrices are 32-bit");
    l[0] = (int32_t)(s[0] == 1 ? std::max<int64_t>(a[i].stride(0), s[2]) : a[i].stride(0));
    l[1] = (int32_t)(s[2] == 1 ? std::max<int64_t>(b[i].stride(0), s[1]) : b[i].stride(0));
    l[2] = s[1];
    used++;
  }
  check(mi355_grouped_gemm_host(pa.data(), pb.data(), pc.data(), sizes.data(), lds.data(), (int)used, abi_dtype(a[0]), (int)num_programs,
                                stream_of(a[0])), "mi355_grouped_gemm");
  return c;
}

// group_gemm of two lists or tuples of plain tensors that it takes: the checks of `group_gemm_fn` without a Python object for every
// shape and stride (us, four products / thirteen of 18 .. 1306 rows: 11.6 / 27.3 with the checks in Python, 8.5 / 13.0).  None: a call that the
// Python function looks at itself - other types, modes around it, whatever it refuses.
py::object group_gemm_plain(const py::object& group_a, const py::object& group_b, int64_t num_programs) {
  auto sequence = [](const py::object& o) { return PyList_CheckExact(o.ptr()) || PyTuple_CheckExact(o.ptr()); };
  if (!sequence(group_a) || !sequence(group_b) || !plain_dispatch() || at::impl::torch_function_mode_enabled()) return py::none();
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(group_a.ptr());
  if (n == 0 || PySequence_Fast_GET_SIZE(group_b.ptr()) != n) return py::none();
  std::vector<at::Tensor> a, b;
  a.reserve(n);
  b.reserve(n);
  for (Py_ssize_t i = 0; i < n; i++) {
    PyObject *oa = PySequence_Fast_GET_ITEM(group_a.ptr(), i), *ob = PySequence_Fast_GET_ITEM(group_b.ptr(), i);
    if (!THPVariable_CheckExact(oa) || !THPVariable_CheckExact(ob)) return py::none();
    a.push_back(THPVariable_Unpack(oa));
    b.push_back(THPVariable_Unpack(ob));
    const at::Tensor &x = a[i], &y = b[i];
    if (x.layout() != at::kStrided || y.layout() != at::kStrided || !x.is_cuda() || !y.is_cuda() || x.dim() != 2 || y.dim() != 2 ||
        x.scalar_type() != a[0].scalar_type() || y.scalar_type() != a[0].scalar_type() || x.size(1) != y.size(0) || x.stride(1) != 1 || y.stride(1) != 1)
      return py::none();
  }
  if (a[0].scalar_type() != at::kHalf && a[0].scalar_type() != at::kBFloat16) return py::none();
  return py::cast(group_gemm(a, b, num_programs));
}

void strides4(const at::Tensor& t, int64_t (&s)[4]) {
  TORCH_CHECK(t.dim() == 4, "attention tensors are [Z, H, N_CTX, D]");
  for (int i = 0; i < 4; i++) s[i] = t.stride(i);
}

void attn_fwd(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, at::Tensor& o, at::Tensor& M, double sm_scale, bool causal) {
  on_device(q, 0); on_device(k, 1); on_device(v, 2); on_device(o, 3); on_device(M, 4);
  const DeviceGuard guard(q.device());
  int64_t sq[4], sk[4], sv[4], so[4];
  strides4(q, sq); strides4(k, sk); strides4(v, sv); strides4(o, so);
  const int rc = mi355_attn_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), M.data_ptr<float>(), (int)q.size(0),
                                (int)q.size(1), (int)q.size(2), (int)q.size(3), sq, sk, sv, so, (float)sm_scale, causal ? 1 : 0,
                                abi_dtype(q), stream_of(q));
  check(rc, "mi355_attn_fwd");
}

void attn_bwd(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& o, const at::Tensor& d_o,
              const at::Tensor& M, at::Tensor& delta, at::Tensor& dq, at::Tensor& dk, at::Tensor& dv, double sm_scale, bool causal) {
  on_device(q, 0); on_device(k, 1); on_device(v, 2); on_device(o, 3); on_device(d_o, 4); on_device(M, 5);
  on_device(delta, 6); on_device(dq, 7); on_device(dk, 8); on_device(dv, 9);
  const DeviceGuard guard(q.device());
  int64_t s[4];
  strides4(q, s);
  TORCH_CHECK(o.strides() == q.strides() && d_o.strides() == q.strides(), "attention backward: q, o and do must have the same strides");
  const int Z = (int)q.size(0), H = (int)q.size(1), N = (int)q.size(2), D = (int)q.size(3);
  void* stream = stream_of(q);
  const int rc = mi355_attn_bwd_o(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), d_o.data_ptr(), M.data_ptr<float>(),
                                  delta.data_ptr<float>(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), Z, H, N, D, s, (float)sm_scale,
                                  causal ? 1 : 0, abi_dtype(q), stream);
  check(rc, "mi355_attn_bwd");
}

// `attention` with its autograd node in native code: the same saved tensors, launches and checks as `_attention` of ops.py, which
// stays for everything else (tensor subclasses, tracing, functorch, forward-mode differentiation, hooks around launches) and
// for every call that it refuses.  us: forward and backward of [1, 16, 1024, 64] fp16, of which the kernels are 38, 94 through the
// Python function and 66 here, most of it the engine's hand-over to the device's thread and back; a forward alone of [1, 2,
// 256, 64] 14.5 and 7.
[[noreturn]] void assertion(const char* message) {   // (thrown from the engine's own threads too: what PythonEngine expects there)
  py::gil_scoped_acquire gil;
  PyErr_SetString(PyExc_AssertionError, message);
  python_error e;
  e.persist();
  throw e;
}

struct Attention : torch::autograd::Function<Attention> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, double sm_scale, bool causal) {
    at::Tensor o = fresh_like(q), M = fresh({q.size(0), q.size(1), q.size(2)}, at::kFloat, q);
    attn_fwd(q, k, v, o, M, sm_scale, causal);
    ctx->save_for_backward({q, k, v, o, M});
    ctx->saved_data["sm_scale"] = sm_scale;
    ctx->saved_data["causal"] = causal;
    return o;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const at::Tensor &q = saved[0], &k = saved[1], &v = saved[2], &o = saved[3], &M = saved[4], &d_o = grads[0];
    if (!d_o.is_contiguous()) assertion("");
    if (q.strides() != k.strides() || q.strides() != v.strides() || q.strides() != o.strides() || q.strides() != d_o.strides()) assertion("");
    if (q.size(2) % 128 != 0) assertion("");
    at::Tensor dq = fresh_like(q), dk = fresh_like(k), dv = fresh_like(v), delta = fresh_like(M);
    attn_bwd(q, k, v, o, d_o, M, delta, dq, dk, dv, ctx->saved_data["sm_scale"].toDouble(), ctx->saved_data["causal"].toBool());
    return {dq, dk, dv, at::Tensor(), at::Tensor()};
  }
};

c10::optional<at::Tensor> attention(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, double sm_scale, bool causal) {
  const auto type = q.scalar_type();
  const bool is8 = type == at::kFloat8_e4m3fn || type == at::kFloat8_e5m2;
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || k.scalar_type() != type || v.scalar_type() != type || !q.is_cuda() || !k.is_cuda() || !v.is_cuda()) return c10::nullopt;
  const int64_t D = q.size(3);
  if ((type != at::kHalf && type != at::kBFloat16 && !is8) || k.size(3) != D || v.size(3) != D || (D != 16 && D != 32 && D != 64 && D != 128 && D != 256)) return c10::nullopt;
  if (is8 && (v.stride(2) != 1 || q.requires_grad() || k.requires_grad() || v.requires_grad())) return c10::nullopt;
  if (at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad())) return Attention::apply(q, k, v, sm_scale, causal);
  at::Tensor o = fresh_like(q), M = fresh({q.size(0), q.size(1), q.size(2)}, at::kFloat, q);
  attn_fwd(q, k, v, o, M, sm_scale, causal);
  return o;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "PyTorch-ROCm extension over the MI355X kernel library's C ABI";
  m.def("matmul", &matmul);
  m.def("mx_gemm", &mx_gemm);
  m.def("group_gemm", &group_gemm);
  m.def("group_gemm_plain", &group_gemm_plain);
  m.def("attn_fwd", &attn_fwd);
  m.def("attn_bwd", &attn_bwd);
  m.def("attention", &attention);
}

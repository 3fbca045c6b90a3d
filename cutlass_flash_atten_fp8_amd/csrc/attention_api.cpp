// PyTorch binding: module `attention_cutlass_fp8`, function `flash_attention_v2_cutlass`.
//
// Drop-in for the reference extension (reference csrc/attention_api.cpp:6-10, declaration
// include/attention_api.h:10-11, host body csrc/flash_attention.cu:639-668): same module and function
// name, same five leading arguments (q, k, v, is_causal, softmax_scale), returns a one-element list.
// Host C++ only: all GPU work goes through the C ABI of libfa8.so (include/fa8_api.h).
//
// Deliberate differences from the reference host code:
//   * v is [B,H,N,d] like k by default; `v_transposed=True` takes the reference's [B,H,d,N] (test.py:71);
//   * O is fp16 by default; `out_dtype=q.dtype` gives the reference's fp8 O in the input element type (:557, :656);
//   * the kernel runs on torch's current stream and the call does not synchronise the device (:661-665);
//   * bad arguments and HIP errors raise RuntimeError instead of printf + exit (include/attention_api.cuh:20-29).
// Additions the reference declares but never implements (csrc/flash.h:36-45,56): k/v may have fewer heads than q
// (grouped-query attention), `return_lse=True` appends the fp32 log-sum-exp [B,H,Nq] to the returned list, and
// `causal_bottom_right=True` aligns the causal diagonal with the last key when seqlen_q != seqlen_k.  `schedule`
// (FA8_SCHEDULE_*, include/fa8_api.h) picks the kernel's main loop by hand: a performance hint; 0 lets the library choose, and is the only
// value with which it may split the keys of a few query rows and so take the fp32 sums in another order.
//
// The function is a plain CPython one (vectorcall arguments) and takes its outputs straight from torch's CUDA allocator: argument
// matching by pybind11 and the dispatcher's empty() took 0.4 us of a call (4.6 -> 4.2; with return_lse 5.6 -> 4.9), whose kernel takes 4.5 where it is smallest.
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>

#include "fa8_api.h"

namespace {

void check_input(const torch::Tensor& t, const char* name) {
  // same two conditions as the reference CHECK_INPUT (include/attention_api.cuh:12-18)
  TORCH_CHECK(t.is_cuda(), name, " must be a GPU tensor");
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
  TORCH_CHECK(t.dim() == 4, name, " must be 4-dimensional [batch, heads, seqlen, head_dim], got ", t.dim(), " dims");
}

torch::Tensor new_tensor(at::IntArrayRef sizes, at::ScalarType type, const torch::Tensor& like) {
  return torch::Tensor(at::detail::empty_cuda(sizes, type, like.device(), c10::nullopt));
}

struct Outputs {
  torch::Tensor o, lse;  // lse: undefined if it was not asked for
};

Outputs flash_attention_v2_cutlass(const torch::Tensor& q, const torch::Tensor& k, const torch::Tensor& v, bool is_causal,
                                   float softmax_scale, bool v_transposed, c10::optional<at::ScalarType> out_dtype, bool return_lse,
                                   bool causal_bottom_right, int64_t schedule) {
  check_input(q, "q");
  check_input(k, "k");
  check_input(v, "v");
  const auto in_type = q.scalar_type();
  TORCH_CHECK(in_type == at::kFloat8_e4m3fn || in_type == at::kFloat8_e5m2,
              "q must be torch.float8_e4m3fn or torch.float8_e5m2 (OCP fp8), got ", in_type);
  TORCH_CHECK(k.scalar_type() == in_type && v.scalar_type() == in_type, "q, k and v must have the same dtype");
  TORCH_CHECK(k.device() == q.device() && v.device() == q.device(), "q, k and v must be on the same device");
  const int64_t B = q.size(0), H = q.size(1), Nq = q.size(2), D = q.size(3);
  const int64_t Nk = k.size(2), Hk = k.size(1);
  TORCH_CHECK(k.size(0) == B && k.size(3) == D, "k must be [", B, ", heads_k, seqlen_k, ", D, "], got ", k.sizes());
  TORCH_CHECK(Hk >= 1 && H % Hk == 0, "the number of q heads (", H, ") must be a multiple of the number of k/v heads (", Hk, ")");
  if (v_transposed) {
    TORCH_CHECK(v.size(0) == B && v.size(1) == Hk && v.size(2) == D && v.size(3) == Nk, "v (transposed) must be [", B, ", ",
                Hk, ", ", D, ", ", Nk, "], got ", v.sizes());
  } else {
    TORCH_CHECK(v.size(0) == B && v.size(1) == Hk && v.size(2) == Nk && v.size(3) == D, "v must be [", B, ", ", Hk, ", ", Nk,
                ", ", D, "], got ", v.sizes());
  }
  TORCH_CHECK(B >= 1 && H >= 1 && Nq >= 1 && Nk >= 1, "empty tensors are not supported");
  TORCH_CHECK(Nq <= INT32_MAX && Nk <= INT32_MAX && B <= INT32_MAX && H <= INT32_MAX, "tensor too large");
  const at::ScalarType o_type = out_dtype.value_or(at::kHalf);
  TORCH_CHECK(o_type == at::kHalf || o_type == in_type,
              "out_dtype must be torch.float16 or the fp8 type of the inputs (the reference's output type), got ", o_type);

  const torch::Tensor out = new_tensor({B, H, Nq, D}, o_type, q);
  torch::Tensor lse;
  if (return_lse) lse = new_tensor({B, H, Nq}, at::kFloat, q);

  Fa8FwdParams p = {};
  p.q = q.data_ptr();
  p.k = k.data_ptr();
  p.v = v.data_ptr();
  p.o = out.data_ptr();
  p.batch = (int32_t)B;
  p.heads = (int32_t)H;
  p.seqlen_q = (int32_t)Nq;
  p.seqlen_k = (int32_t)Nk;
  p.head_dim = (int32_t)D;
  p.is_causal = is_causal ? 1 : 0;
  p.in_dtype = in_type == at::kFloat8_e5m2 ? FA8_DTYPE_E5M2 : FA8_DTYPE_E4M3;
  p.out_dtype = o_type == at::kHalf ? FA8_OUT_FP16 : (o_type == at::kFloat8_e5m2 ? FA8_OUT_E5M2 : FA8_OUT_E4M3);
  p.v_layout = v_transposed ? FA8_V_TRANSPOSED : FA8_V_ROWS;
  p.softmax_scale = softmax_scale;
  p.q_batch_stride = q.stride(0); p.q_head_stride = q.stride(1); p.q_row_stride = q.stride(2);
  p.k_batch_stride = k.stride(0); p.k_head_stride = k.stride(1); p.k_row_stride = k.stride(2);
  p.v_batch_stride = v.stride(0); p.v_head_stride = v.stride(1); p.v_row_stride = v.stride(2);
  p.o_batch_stride = out.stride(0); p.o_head_stride = out.stride(1); p.o_row_stride = out.stride(2);
  p.heads_k = (int32_t)Hk;
  p.causal_align = causal_bottom_right ? FA8_CAUSAL_BOTTOM_RIGHT : FA8_CAUSAL_TOP_LEFT;
  TORCH_CHECK(schedule >= FA8_SCHEDULE_AUTO && schedule <= FA8_SCHEDULE_DENSE, "schedule must be one of the FA8_SCHEDULE_* codes 0..",
              FA8_SCHEDULE_DENSE, ", got ", schedule);
  p.schedule = (int32_t)schedule;
  if (return_lse) {
    p.lse = lse.data_ptr();
    p.lse_batch_stride = lse.stride(0);
    p.lse_head_stride = lse.stride(1);
  }

  // PyTorch-ROCm presents HIP devices under the "cuda" device type; these are its guard and stream for them.
  const c10::hip::HIPGuardMasqueradingAsCUDA device_guard(q.device());
  const hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(q.device().index()).stream();
  int64_t workspace_bytes = 0;
  torch::Tensor workspace;  // (goes back to torch's allocator on return, for later work of this stream)
  int rc = fa8_fwd_workspace(&p, &workspace_bytes);
  if (rc == FA8_OK) {
    if (workspace_bytes > 0) {
      try {
        workspace = new_tensor({workspace_bytes}, at::kByte, q);
      } catch (const c10::OutOfMemoryError&) {  // the call needs none, it only takes longer
      }
    }
    rc = workspace.defined() ? fa8_fwd_any_order(&p, workspace.data_ptr(), workspace_bytes, (void*)stream)
                             : fa8_fwd_any_order(&p, nullptr, 0, (void*)stream);
  }
  TORCH_CHECK(rc == FA8_OK, "flash_attention_v2_cutlass: ", fa8_error_string(rc), " (code ", rc, ")");
  return {out, lse};
}

// ---- the Python function ----
constexpr int kPositional = 5, kArguments = 10;
const char* const kNames[kArguments] = {"q", "k", "v", "is_causal", "softmax_scale", "v_transposed", "out_dtype", "return_lse",
                                        "causal_bottom_right", "schedule"};
PyObject* interned_names[kArguments];

[[noreturn]] void type_error(const std::string& text) { throw torch::TypeError("flash_attention_v2_cutlass(): " + text); }

const torch::Tensor& tensor_argument(PyObject* v, int i) {
  if (!THPVariable_Check(v)) type_error(std::string("argument '") + kNames[i] + "' must be a torch.Tensor, not " + Py_TYPE(v)->tp_name);
  return THPVariable_Unpack(v);
}

bool bool_argument(PyObject* v, int i) {
  if (v == Py_True) return true;
  if (v == nullptr || v == Py_False || v == Py_None) return false;
  const int x = Py_TYPE(v)->tp_as_number && Py_TYPE(v)->tp_as_number->nb_bool ? PyObject_IsTrue(v) : -1;
  if (x < 0) {
    PyErr_Clear();
    type_error(std::string("argument '") + kNames[i] + "' must be a bool, not " + Py_TYPE(v)->tp_name);
  }
  return x != 0;
}

PyObject* python_flash_attention(PyObject*, PyObject* const* args, Py_ssize_t n_positional, PyObject* keywords) {
  HANDLE_TH_ERRORS
  PyObject* v[kArguments] = {};
  if (n_positional > kPositional)
    type_error("takes " + std::to_string(kPositional) + " positional arguments but " + std::to_string(n_positional) + " were given");
  for (Py_ssize_t i = 0; i < n_positional; ++i) v[i] = args[i];
  const Py_ssize_t n_keywords = keywords ? PyTuple_GET_SIZE(keywords) : 0;
  for (Py_ssize_t x = 0; x < n_keywords; ++x) {
    PyObject* const name = PyTuple_GET_ITEM(keywords, x);
    int i = 0;
    while (i < kArguments && name != interned_names[i]) ++i;  // keywords written in a program are interned
    if (i == kArguments)
      for (i = 0; i < kArguments && PyUnicode_Compare(name, interned_names[i]) != 0;) ++i;
    if (i == kArguments) {  // (a name need not have a UTF-8 form)
      PyErr_Format(PyExc_TypeError, "flash_attention_v2_cutlass(): got an unexpected keyword argument '%U'", name);
      return nullptr;
    }
    if (v[i]) type_error(std::string("got multiple values for argument '") + kNames[i] + "'");
    v[i] = args[n_positional + x];
  }
  for (int i = 0; i < kPositional; ++i)
    if (!v[i]) type_error(std::string("missing required argument '") + kNames[i] + "'");
  const torch::Tensor &q = tensor_argument(v[0], 0), &k = tensor_argument(v[1], 1), &value = tensor_argument(v[2], 2);
  const double scale = PyFloat_AsDouble(v[4]);
  if (scale == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    type_error(std::string("argument 'softmax_scale' must be a float, not ") + Py_TYPE(v[4])->tp_name);
  }
  c10::optional<at::ScalarType> out_dtype;
  if (v[6] && v[6] != Py_None) {
    if (!THPDtype_Check(v[6])) type_error(std::string("argument 'out_dtype' must be a torch.dtype or None, not ") + Py_TYPE(v[6])->tp_name);
    out_dtype = reinterpret_cast<THPDtype*>(v[6])->scalar_type;
  }
  long long schedule = 0;
  if (v[9]) {
    schedule = PyFloat_Check(v[9]) ? -1 : PyLong_AsLongLong(v[9]);
    if (schedule == -1 && !PyFloat_Check(v[9]) && PyErr_Occurred() && PyNumber_Check(v[9])) {  // no __index__: __int__, as pybind11 does
      PyErr_Clear();
      const py::object whole = py::reinterpret_steal<py::object>(PyNumber_Long(v[9]));
      if (whole) schedule = PyLong_AsLongLong(whole.ptr());
    }
    if (PyFloat_Check(v[9]) || (schedule == -1 && PyErr_Occurred())) {
      PyErr_Clear();
      type_error(std::string("argument 'schedule' must be an int, not ") + Py_TYPE(v[9])->tp_name);
    }
  }
  const Outputs out = flash_attention_v2_cutlass(q, k, value, bool_argument(v[3], 3), (float)scale, bool_argument(v[5], 5), out_dtype,
                                                 bool_argument(v[7], 7), bool_argument(v[8], 8), schedule);
  PyObject* const list = PyList_New(out.lse.defined() ? 2 : 1);
  if (!list) throw python_error();
  PyList_SET_ITEM(list, 0, THPVariable_Wrap(out.o));
  if (out.lse.defined()) PyList_SET_ITEM(list, 1, THPVariable_Wrap(out.lse));
  return list;
  END_HANDLE_TH_ERRORS
}

PyMethodDef python_method = {
    "flash_attention_v2_cutlass", (PyCFunction)(void (*)(void))python_flash_attention, METH_FASTCALL | METH_KEYWORDS,
    "flash_attention_v2_cutlass(q, k, v, is_causal, softmax_scale, *, v_transposed=False, out_dtype=None, return_lse=False, "
    "causal_bottom_right=False, schedule=0) -> list of torch.Tensor\n\n"
    "FP8 flash attention forward: fp8 q/k/v [B,H,N,d] -> [O] (fp16 by default), with return_lse=True [O, lse]"};

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "FP8 flash-attention forward for AMD MI355X (gfx950)";
  for (int i = 0; i < kArguments; ++i) interned_names[i] = PyUnicode_InternFromString(kNames[i]);
  m.add_object("flash_attention_v2_cutlass",
               py::reinterpret_steal<py::object>(PyCFunction_NewEx(&python_method, nullptr, m.attr("__name__").ptr())));
  m.def("kv_block", []() { return fa8_query(FA8_QUERY_KV_BLOCK); }, "kv rows per online-softmax step of the kernel");
}

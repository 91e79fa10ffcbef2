// Python extension between the operators (ops.py, comm_quant.py) and libcdit_hip.so: takes
// tensors, allocates results and workspaces, and calls the C entry points on the tensors' device
// and current stream. It decides nothing: shapes, kernels and error texts are the library's.
//
// Why it exists: a Linear with one row of activation is one launch of 7 us of GPU time (K 3072,
// N 9216) whose call took 17.5 us of host time, of which the launch itself was 3.4 and the
// dispatcher 2.5; the rest were attribute reads, three torch.empty calls (1.8 us each) and the
// conversion of the arguments, all in Python. `*_plain` functions look at the arguments and
// run the operator, or give None for anything out of the ordinary (other dtypes, strides, devices,
// empty tensors), which the general Python code then converts or refuses as it always did; the other
// functions launch. linear_w8a8, w8a16_mm, float8_inference_scaled_mm, fp8_rowwise_quant, ln_modulate_quant and
// the comm quantizers are one call each, and the workspaces of a Linear never become Python objects and are
// one allocation: the operator of a one-row Linear 8.0 to 8.4 -> 7.3 us of host time (with one call to look at the
// arguments and allocate, one to launch, and two workspaces, before). linear_w8a8_cat2, the batches and shared
// quantization take their outputs and workspaces from here and launch with further calls.
#define __HIP_PLATFORM_AMD__ 1
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <vector>

#include "cdit_hip.h"

// The torch and Python this is compiled against (_native.host_built_for()); looked for in the file before it is loaded.
extern "C" __attribute__((used, visibility("default"))) const char cdit_host_built_for[] = CDIT_HOST_BUILT_FOR;

namespace {

constexpr int kMaxActs = 4, kMaxGroup = 8;

// ---- the library, bound once (bind()); the same handle as the ctypes binding's
struct Library {
  decltype(&cdit_fp8_linear_w8a8) linear_w8a8;
  decltype(&cdit_fp8_gemm_rowwise) gemm_rowwise;
  decltype(&cdit_fp8_gemm_rowwise_batched) gemm_rowwise_batched;
  decltype(&cdit_w8a16_gemm) w8a16_gemm;
  decltype(&cdit_w8a16_gemm_batched) w8a16_gemm_batched;
  decltype(&cdit_fp8_quant_rowwise) quant_rowwise;
  decltype(&cdit_fp8_quant_rowwise_batched) quant_rowwise_batched;
  decltype(&cdit_fp8_quant_rowwise_cat2) quant_rowwise_cat2;
  decltype(&cdit_fp8_quant_tensorwise) quant_tensorwise;
  decltype(&cdit_fp8_ln_modulate_quant) ln_modulate_quant;
  decltype(&cdit_fp8_comm_per_token_quant) comm_per_token_quant;
  decltype(&cdit_fp8_comm_per_token_dequant) comm_per_token_dequant;
  decltype(&cdit_fp8_comm_qkv_permute_quant) comm_qkv_permute_quant;
  decltype(&cdit_fp8_comm_qkv_permute_dequant) comm_qkv_permute_dequant;
};
Library lib = {};

// ---- arguments
const at::Tensor& tensor(PyObject* o) {
  TORCH_CHECK_TYPE(THPVariable_Check(o), "expected a tensor, got ", Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}
int64_t integer(PyObject* o) {
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw python_error();
  return v;
}
void arity(Py_ssize_t got, Py_ssize_t want) {
  TORCH_CHECK_TYPE(got == want, "expected ", want, " arguments, got ", got);
}
void* bias_ptr(PyObject* o) { return o == Py_None ? nullptr : tensor(o).data_ptr(); }

// The rows of a tensor as the kernels read them: a matrix with any row stride, or a contiguous
// tensor whose leading dimensions are the rows.
struct Rows {
  int64_t M, K, ld;
};
bool rows_of(const at::Tensor& t, Rows* r) {
  const int64_t d = t.dim();
  if (d < 1) return false;
  r->K = t.size(d - 1);
  if (d == 2) {
    r->M = t.size(0);
    r->ld = t.stride(0);
    return r->K > 0 && t.stride(1) == 1;
  }
  if (r->K <= 0 || !t.is_contiguous()) return false;
  r->M = t.numel() / r->K;
  r->ld = r->K;
  return true;
}
// For the launchers: their callers have looked at the last stride.
Rows rows(const at::Tensor& t) {
  Rows r;
  if (t.dim() == 2) return {t.size(0), t.size(1), t.stride(0)};
  TORCH_CHECK_VALUE(rows_of(t, &r), "expected a matrix or a contiguous tensor");
  return r;
}
// Leading dimension of an output [..., N].
int64_t out_ld(const at::Tensor& t) { return t.dim() >= 2 ? t.stride(t.dim() - 2) : t.numel(); }

bool vector_of(const at::Tensor& t, at::ScalarType type, int64_t n) {
  return t.scalar_type() == type && t.numel() == n && t.is_contiguous();
}
bool aligned16(const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

at::Tensor empty(at::IntArrayRef shape, at::ScalarType type, const at::Tensor& like) {
  return at::empty(shape, at::TensorOptions().dtype(type).device(like.device()));
}
at::Tensor empty_like_rows(const at::Tensor& x, int64_t last, at::ScalarType type) {
  c10::SmallVector<int64_t, 6> shape(x.sizes().begin(), x.sizes().end());
  shape.back() = last;
  return empty(shape, type, x);
}
PyObject* wrap(std::initializer_list<at::Tensor> ts) {
  PyObject* t = PyTuple_New((Py_ssize_t)ts.size());
  if (!t) throw python_error();
  Py_ssize_t i = 0;
  for (const at::Tensor& x : ts) {
    PyObject* o = THPVariable_Wrap(x);
    if (!o) {
      Py_DECREF(t);
      throw python_error();
    }
    PyTuple_SET_ITEM(t, i++, o);
  }
  return t;
}

// Calls a library entry point with `t`'s device current, on its current stream (every entry point's
// last argument), without the GIL (a full launch queue blocks); gives the status. The arguments are
// values: tensors are read while the GIL is held, and whoever calls this holds them.
template <class F, class... A>
int status_of(const at::Tensor& t, F f, A... a) {
  TORCH_CHECK(f, "libcdit_hip.so is not bound");
  TORCH_CHECK_VALUE(t.is_cuda(), "expected tensors on the GPU, got a ", t.device(), " tensor");
  const c10::DeviceGuard guard(t.device());
  void* stream = c10::hip::getCurrentHIPStream(t.device().index()).stream();
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = f(a..., stream);
  Py_END_ALLOW_THREADS;
  return rc;
}
template <class F, class... A>
PyObject* launch(const at::Tensor& t, F f, A... a) {
  return PyLong_FromLong(status_of(t, f, a...));
}

constexpr auto kBf16 = at::kBFloat16;
constexpr auto kFp8 = at::kFloat8_e4m3fn;
constexpr auto kF32 = at::kFloat;

// ---- operators on plain arguments (None: the general Python code looks at them). Results are (status, results...):
// the caller raises for a status other than 0. Workspaces are taken from the caching allocator on the current stream
// and given back to it here, behind the launch: what is allocated next on that stream runs behind it.

// (status, results...)
PyObject* with_status(int status, std::initializer_list<at::Tensor> ts) {
  PyObject* t = PyTuple_New((Py_ssize_t)ts.size() + 1);
  if (!t) throw python_error();
  PyObject* o = PyLong_FromLong(status);
  Py_ssize_t i = 0;
  if (o) PyTuple_SET_ITEM(t, i++, o);
  for (const at::Tensor& x : ts) {
    if (o) o = THPVariable_Wrap(x);
    if (!o) break;
    PyTuple_SET_ITEM(t, i++, o);
  }
  if (!o) {
    Py_DECREF(t);
    throw python_error();
  }
  return t;
}

// Scales [M] and behind them codes [M, K] of an activation, in one allocation (an allocation is 0.6 us of host time).
struct Workspace {
  at::Tensor memory;
  float* scales;
  uint8_t* codes;
  Workspace(const at::Tensor& x, int64_t M, int64_t K) {
    const int64_t head = (4 * M + 255) / 256 * 256;
    memory = empty({head + M * K}, at::kByte, x);
    scales = reinterpret_cast<float*>(memory.data_ptr());
    codes = static_cast<uint8_t*>(memory.data_ptr()) + head;
  }
};

// linear_plain(x, weight, weight_scale, bias, scale_mode, epilogue, per_tensor) -> (status, out [..., N])
PyObject* linear_plain(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 7);
  const at::Tensor &x = tensor(a[0]), &w = tensor(a[1]), &ws = tensor(a[2]);
  const int mode = (int)integer(a[4]), epi = (int)integer(a[5]);
  Rows r;
  if (x.scalar_type() != kBf16 || w.scalar_type() != kFp8 || w.dim() != 2 || w.stride(1) != 1 ||
      !rows_of(x, &r) || r.M <= 0 || r.K != w.size(1) || x.device() != w.device() || ws.device() != x.device() ||
      !vector_of(ws, kF32, w.size(0)))
    Py_RETURN_NONE;
  const int64_t N = w.size(0), ldw = w.stride(0);
  void* bias = nullptr;
  if (a[3] != Py_None) {
    const at::Tensor& b = tensor(a[3]);
    if (!vector_of(b, kBf16, N) || b.device() != x.device()) Py_RETURN_NONE;
    bias = b.data_ptr();
  }
  const at::Tensor out = empty_like_rows(x, N, kBf16);
  const int64_t ldo = out_ld(out);
  const float* scale = static_cast<const float*>(ws.data_ptr());
  const Workspace q(x, r.M, r.K);
  if (a[6] != Py_True)
    return with_status(status_of(x, lib.linear_w8a8, x.data_ptr(), w.data_ptr(), scale, bias, out.data_ptr(), q.codes,
                                 q.scales, r.M, N, r.K, r.ld, ldw, ldo, mode, epi, CDIT_DT_BF16), {out});
  const at::Tensor amax = empty({1}, at::kInt, x);
  int rc = status_of(x, lib.quant_tensorwise, x.data_ptr(), r.M, r.K, r.ld, q.codes, r.K, q.scales, amax.data_ptr(), mode);
  if (!rc)
    rc = status_of(x, lib.gemm_rowwise, q.codes, q.scales, w.data_ptr(), scale, bias, out.data_ptr(), r.M, N, r.K, r.K,
                   ldw, ldo, epi, CDIT_DT_BF16);
  return with_status(rc, {out});
  END_HANDLE_TH_ERRORS
}

// w8a16_plain(x, b_data [K, N], b_scale, bias, epilogue) -> (status, out)
PyObject* w8a16_plain(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 5);
  const at::Tensor &x = tensor(a[0]), &b = tensor(a[1]), &bs = tensor(a[2]);
  const int epi = (int)integer(a[4]);
  Rows r;
  if (x.scalar_type() != kBf16 || b.scalar_type() != kFp8 || b.dim() != 2 || b.stride(0) != 1 ||
      !rows_of(x, &r) || r.M <= 0 || r.K != b.size(0) || x.device() != b.device() || bs.device() != x.device() ||
      !vector_of(bs, kF32, b.size(1)))
    Py_RETURN_NONE;
  const int64_t N = b.size(1);
  void* bias = nullptr;
  if (a[3] != Py_None) {
    const at::Tensor& t = tensor(a[3]);
    if (!vector_of(t, kBf16, N) || t.device() != x.device()) Py_RETURN_NONE;
    bias = t.data_ptr();
  }
  const at::Tensor out = empty_like_rows(x, N, kBf16);
  return with_status(status_of(x, lib.w8a16_gemm, x.data_ptr(), b.data_ptr(), static_cast<const float*>(bs.data_ptr()),
                               bias, out.data_ptr(), r.M, N, r.K, r.ld, b.stride(1), out_ld(out), epi, CDIT_DT_BF16), {out});
  END_HANDLE_TH_ERRORS
}

// scaled_mm_plain(a_data, a_scale, b_data [K, N], b_scale, bias, out_dtype_id, epilogue) -> (status, out)
PyObject* scaled_mm_plain(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 7);
  const at::Tensor &x = tensor(a[0]), &xs = tensor(a[1]), &b = tensor(a[2]), &bs = tensor(a[3]);
  const int64_t id = integer(a[5]);
  const int epi = (int)integer(a[6]);
  const at::ScalarType type = id == CDIT_DT_F16 ? at::kHalf : id == CDIT_DT_BF16 ? kBf16 : kF32;
  Rows r;
  if (id < 0 || id > 2 || x.scalar_type() != kFp8 || b.scalar_type() != kFp8 || b.dim() != 2 || b.stride(0) != 1 ||
      !rows_of(x, &r) || r.M <= 0 || r.K != b.size(0) || x.device() != b.device() || xs.device() != x.device() ||
      bs.device() != x.device() || !vector_of(xs, kF32, r.M) || !vector_of(bs, kF32, b.size(1)) || !aligned16(xs) ||
      !aligned16(bs))
    Py_RETURN_NONE;
  const int64_t N = b.size(1);
  void* bias = nullptr;
  if (a[4] != Py_None) {
    const at::Tensor& t = tensor(a[4]);
    if (type == kF32 || !vector_of(t, type, N) || t.device() != x.device() || !aligned16(t)) Py_RETURN_NONE;
    bias = t.data_ptr();
  }
  const at::Tensor out = empty_like_rows(x, N, type);
  return with_status(status_of(x, lib.gemm_rowwise, x.data_ptr(), static_cast<const float*>(xs.data_ptr()), b.data_ptr(),
                               static_cast<const float*>(bs.data_ptr()), bias, out.data_ptr(), r.M, N, r.K, r.ld,
                               b.stride(1), out_ld(out), epi, (int)id), {out});
  END_HANDLE_TH_ERRORS
}

// quant_plain(x, scale_mode) -> (status, codes like x, scales [..., 1])
PyObject* quant_plain(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 2);
  const at::Tensor& x = tensor(a[0]);
  const int mode = (int)integer(a[1]);
  Rows r;
  if (x.scalar_type() != kBf16 || !rows_of(x, &r) || r.M <= 0) Py_RETURN_NONE;
  const at::Tensor q = empty(x.sizes(), kFp8, x), s = empty_like_rows(x, 1, kF32);
  return with_status(status_of(x, lib.quant_rowwise, x.data_ptr(), r.M, r.K, r.ld, q.data_ptr(), r.K,
                               (float*)s.data_ptr(), mode), {q, s});
  END_HANDLE_TH_ERRORS
}

// cat2_plain(x1, x2, weight, weight_scale, bias) -> (out, codes [M, K1 + K2], scales [M])
PyObject* cat2_plain(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 5);
  const at::Tensor &x1 = tensor(a[0]), &x2 = tensor(a[1]), &w = tensor(a[2]), &ws = tensor(a[3]);
  Rows r1, r2;
  if (x1.scalar_type() != kBf16 || x2.scalar_type() != kBf16 || x1.dim() != x2.dim() || !rows_of(x1, &r1) ||
      !rows_of(x2, &r2) || x1.sizes().slice(0, x1.dim() - 1) != x2.sizes().slice(0, x2.dim() - 1) || r1.M <= 16 ||
      r1.K % 8 || r2.K % 8 || r1.K + r2.K > 16384 || r1.ld % 8 || r2.ld % 8 || !aligned16(x1) || !aligned16(x2) ||
      w.scalar_type() != kFp8 || w.dim() != 2 || w.stride(1) != 1 || w.size(1) != r1.K + r2.K ||
      x1.device() != x2.device() || x1.device() != w.device() || ws.device() != x1.device() ||
      !vector_of(ws, kF32, w.size(0)))
    Py_RETURN_NONE;
  if (a[4] != Py_None) {
    const at::Tensor& b = tensor(a[4]);
    if (!vector_of(b, kBf16, w.size(0)) || b.device() != x1.device()) Py_RETURN_NONE;
  }
  return wrap({empty_like_rows(x1, w.size(0), kBf16), empty({r1.M, r1.K + r2.K}, kFp8, x1), empty({r1.M}, kF32, x1)});
  END_HANDLE_TH_ERRORS
}

// outputs(x, [N, ...]) -> [bf16 [..., N], ...]; workspace(x) -> (codes [M, K], scales [M]); x: rows
PyObject* outputs(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 2);
  const at::Tensor& x = tensor(a[0]);
  TORCH_CHECK_TYPE(PyList_Check(a[1]), "expected a list of widths");
  PyObject* list = PyList_New(PyList_GET_SIZE(a[1]));
  if (!list) throw python_error();
  try {
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(a[1]); ++i) {
      PyObject* o = THPVariable_Wrap(empty_like_rows(x, integer(PyList_GET_ITEM(a[1], i)), kBf16));
      if (!o) throw python_error();
      PyList_SET_ITEM(list, i, o);
    }
  } catch (...) {
    Py_DECREF(list);
    throw;
  }
  return list;
  END_HANDLE_TH_ERRORS
}
PyObject* workspace(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 1);
  const at::Tensor& x = tensor(a[0]);
  const Rows r = rows(x);
  return wrap({empty({r.M, r.K}, kFp8, x), empty({r.M}, kF32, x)});
  END_HANDLE_TH_ERRORS
}

// ---- launchers: results are the library's status

// linear_w8a8(x, weight, weight_scale, bias, out, codes, scales, scale_mode, epilogue)
PyObject* linear_w8a8(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 9);
  const at::Tensor &x = tensor(a[0]), &w = tensor(a[1]), &ws = tensor(a[2]), &out = tensor(a[4]), &q = tensor(a[5]),
                   &s = tensor(a[6]);
  void* bias = bias_ptr(a[3]);
  const Rows r = rows(x);
  const int mode = (int)integer(a[7]), epi = (int)integer(a[8]);
  return launch(x, lib.linear_w8a8, x.data_ptr(), w.data_ptr(), (const float*)ws.data_ptr(), bias, out.data_ptr(),
                q.data_ptr(), (float*)s.data_ptr(), r.M, w.size(0), r.K, r.ld, w.stride(0), out_ld(out), mode, epi,
                CDIT_DT_BF16);
  END_HANDLE_TH_ERRORS
}

// gemm_rowwise(a, a_scale, weight, weight_scale, bias, out, epilogue, out_dtype_id)
PyObject* gemm_rowwise(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 8);
  const at::Tensor &x = tensor(a[0]), &xs = tensor(a[1]), &w = tensor(a[2]), &ws = tensor(a[3]), &out = tensor(a[5]);
  void* bias = bias_ptr(a[4]);
  const Rows r = rows(x);
  const int epi = (int)integer(a[6]), id = (int)integer(a[7]);
  return launch(x, lib.gemm_rowwise, x.data_ptr(), (const float*)xs.data_ptr(), w.data_ptr(),
                (const float*)ws.data_ptr(), bias, out.data_ptr(), r.M, w.size(0), r.K, r.ld, w.stride(0),
                out_ld(out), epi, id);
  END_HANDLE_TH_ERRORS
}

// w8a16(x, weight, weight_scale, bias, out, epilogue)
PyObject* w8a16(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 6);
  const at::Tensor &x = tensor(a[0]), &w = tensor(a[1]), &ws = tensor(a[2]), &out = tensor(a[4]);
  void* bias = bias_ptr(a[3]);
  const Rows r = rows(x);
  const int epi = (int)integer(a[5]);
  return launch(x, lib.w8a16_gemm, x.data_ptr(), w.data_ptr(), (const float*)ws.data_ptr(), bias, out.data_ptr(), r.M,
                w.size(0), r.K, r.ld, w.stride(0), out_ld(out), epi, CDIT_DT_BF16);
  END_HANDLE_TH_ERRORS
}

// quant_rowwise(x, codes, scales, scale_mode)
PyObject* quant_rowwise(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 4);
  const at::Tensor &x = tensor(a[0]), &q = tensor(a[1]), &s = tensor(a[2]);
  const Rows r = rows(x);
  const int64_t ldq = rows(q).ld;
  const int mode = (int)integer(a[3]);
  return launch(x, lib.quant_rowwise, x.data_ptr(), r.M, r.K, r.ld, q.data_ptr(), ldq, (float*)s.data_ptr(), mode);
  END_HANDLE_TH_ERRORS
}

// quant_tensorwise(x, codes, scales, amax, scale_mode)
PyObject* quant_tensorwise(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 5);
  const at::Tensor &x = tensor(a[0]), &q = tensor(a[1]), &s = tensor(a[2]), &amax = tensor(a[3]);
  const Rows r = rows(x);
  const int64_t ldq = rows(q).ld;
  const int mode = (int)integer(a[4]);
  return launch(x, lib.quant_tensorwise, x.data_ptr(), r.M, r.K, r.ld, q.data_ptr(), ldq, (float*)s.data_ptr(),
                amax.data_ptr(), mode);
  END_HANDLE_TH_ERRORS
}

// quant_rowwise_cat2(x1, x2, codes, scales, scale_mode)
PyObject* quant_rowwise_cat2(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 5);
  const at::Tensor &x1 = tensor(a[0]), &x2 = tensor(a[1]), &q = tensor(a[2]), &s = tensor(a[3]);
  const Rows r1 = rows(x1), r2 = rows(x2);
  const int64_t ldq = rows(q).ld;
  const int mode = (int)integer(a[4]);
  return launch(x1, lib.quant_rowwise_cat2, x1.data_ptr(), r1.K, r1.ld, x2.data_ptr(), r2.K, r2.ld, r1.M,
                q.data_ptr(), ldq, (float*)s.data_ptr(), mode);
  END_HANDLE_TH_ERRORS
}

// A Python sequence, held for the call.
struct Seq {
  PyObject* fast;
  explicit Seq(PyObject* o) : fast(PySequence_Fast(o, "expected a list")) {
    if (!fast) throw python_error();
  }
  Seq(const Seq&) = delete;
  ~Seq() { Py_DECREF(fast); }
  Py_ssize_t size() const { return PySequence_Fast_GET_SIZE(fast); }
  PyObject* operator[](Py_ssize_t i) const { return PySequence_Fast_GET_ITEM(fast, i); }
};

// quant_rowwise_batched([(x, codes, scales), ...], scale_mode)
PyObject* quant_rowwise_batched(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 2);
  const Seq items(a[0]);
  const int mode = (int)integer(a[1]);
  TORCH_CHECK_VALUE(items.size() >= 1 && items.size() <= kMaxActs, "quant_rowwise_batched_into: 1 to ", kMaxActs,
                    " activations");
  const void* x[kMaxActs];
  void* q[kMaxActs];
  float* s[kMaxActs];
  int64_t m[kMaxActs], ldx[kMaxActs], ldq[kMaxActs], K = 0;
  at::Tensor x0;
  for (Py_ssize_t i = 0; i < items.size(); ++i) {
    const Seq it(items[i]);
    TORCH_CHECK_VALUE(it.size() == 3, "quant_rowwise_batched_into: items are (x, codes, scales)");
    const at::Tensor &xi = tensor(it[0]), &qi = tensor(it[1]);
    const Rows r = rows(xi);
    if (i == 0) x0 = xi, K = r.K;
    TORCH_CHECK_VALUE(r.K == K && xi.device() == x0.device(),
                      "quant_rowwise_batched_into: the activations must share K and the device");
    x[i] = xi.data_ptr();
    q[i] = qi.data_ptr();
    s[i] = (float*)tensor(it[2]).data_ptr();
    m[i] = r.M;
    ldx[i] = r.ld;
    ldq[i] = rows(qi).ld;
  }
  return launch(x0, lib.quant_rowwise_batched, (int)items.size(), x, m, K, ldx, q, ldq, s, mode);
  END_HANDLE_TH_ERRORS
}

// The two batched GEMMs. gemm_batched([(a, a_scale or None, weights, w_scales, biases, outs, epilogues), ...],
// weight_only): one entry per activation.
PyObject* gemm_batched(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 2);
  const Seq acts(args[0]);
  const bool weight_only = args[1] == Py_True;
  const char* name = weight_only ? "w8a16_batched_into" : "gemm_rowwise_batched_into";
  TORCH_CHECK_VALUE(acts.size() >= 1 && acts.size() <= kMaxActs, name, ": 1 to ", kMaxActs, " activations");
  const void *a[kMaxActs], *b[kMaxGroup], *bias[kMaxGroup];
  const float *as[kMaxActs], *bs[kMaxGroup];
  void* out[kMaxGroup];
  int64_t M[kMaxActs], N[kMaxGroup], ldo[kMaxGroup], K = 0, lda = 0, ldb = 0;
  int members[kMaxActs], epi[kMaxGroup], p = 0;
  at::Tensor a0;
  for (Py_ssize_t i = 0; i < acts.size(); ++i) {
    const Seq act(acts[i]);
    TORCH_CHECK_VALUE(act.size() == 7, name, ": entries are (a, a_scale, weights, w_scales, biases, outs, epilogues)");
    const at::Tensor& x = tensor(act[0]);
    const Seq w(act[2]), ws(act[3]), bi(act[4]), o(act[5]), e(act[6]);
    const Rows r = rows(x);
    if (i == 0) {
      a0 = x;
      K = r.K;
      lda = r.ld;
      TORCH_CHECK_VALUE(w.size() >= 1, name, ": an activation without members");
      ldb = tensor(w[0]).stride(0);
    }
    if (weight_only) {
      TORCH_CHECK_VALUE(r.K == K && x.device() == a0.device() && x.scalar_type() == kBf16 && x.stride(-1) == 1, name,
                        ": the activations must be bf16 rows of one K on one device");
    } else {
      TORCH_CHECK_VALUE(r.K == K && r.ld == lda && x.device() == a0.device(), name,
                        ": the activations must share K, the row stride and the device");
    }
    a[i] = x.data_ptr();
    as[i] = act[1] == Py_None ? nullptr : (const float*)tensor(act[1]).data_ptr();
    M[i] = r.M;
    members[i] = (int)w.size();
    TORCH_CHECK_VALUE(ws.size() == w.size() && bi.size() == w.size() && o.size() == w.size() && e.size() == w.size() &&
                          p + w.size() <= kMaxGroup,
                      name, ": at most ", kMaxGroup, " members, each with a scale, a bias, an output and an epilogue");
    for (Py_ssize_t j = 0; j < w.size(); ++j, ++p) {
      const at::Tensor &wj = tensor(w[j]), &oj = tensor(o[j]);
      TORCH_CHECK_VALUE(wj.dim() == 2 && wj.stride(0) == ldb && wj.size(1) == K, name,
                        ": the weights must share K and the row stride");
      b[p] = wj.data_ptr();
      bs[p] = (const float*)tensor(ws[j]).data_ptr();
      bias[p] = bias_ptr(bi[j]);
      out[p] = oj.data_ptr();
      N[p] = wj.size(0);
      ldo[p] = out_ld(oj);
      epi[p] = (int)integer(e[j]);
    }
  }
  const int na = (int)acts.size();
  return weight_only ? launch(a0, lib.w8a16_gemm_batched, na, a, M, K, lda, members, b, bs, bias, out, N, ldb, ldo, epi)
                     : launch(a0, lib.gemm_rowwise_batched, na, a, as, M, K, lda, members, b, bs, bias, out, N, ldb,
                              ldo, epi);
  END_HANDLE_TH_ERRORS
}

// ---- more operators, as above

// ln_modulate_quant(x, shift, scale, eps, scale_mode, write_y) -> (status, y, codes, scales)
PyObject* ln_modulate_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 6);
  const at::Tensor &x = tensor(a[0]), &sh = tensor(a[1]), &sc = tensor(a[2]);
  const double eps = PyFloat_AsDouble(a[3]);
  if (eps == -1.0 && PyErr_Occurred()) throw python_error();
  const int mode = (int)integer(a[4]);
  const bool write_y = a[5] == Py_True;
  Rows r;
  if (x.scalar_type() != kBf16 || sh.scalar_type() != kBf16 || sc.scalar_type() != kBf16 || !rows_of(x, &r) ||
      r.M <= 0 || mode < 0 || mode > 1 || sh.dim() < 1 || sh.sizes() != sc.sizes() || sh.size(-1) != r.K ||
      !sh.is_contiguous() || !sc.is_contiguous() || sh.device() != x.device() || sc.device() != x.device())
    Py_RETURN_NONE;
  const int64_t nb = sh.numel() / r.K;
  if (nb != 1 && !(nb > 0 && x.dim() >= 2 && nb == x.size(0) && r.M % nb == 0)) Py_RETURN_NONE;
  at::Tensor y = empty(x.sizes(), kBf16, x), q = empty(x.sizes(), kFp8, x), s = empty_like_rows(x, 1, kF32);
  return with_status(status_of(x, lib.ln_modulate_quant, x.data_ptr(), r.M, r.K, r.ld, sh.data_ptr(), sc.data_ptr(), r.K,
                            nb == 1 ? r.M : r.M / nb, (float)eps, write_y ? y.data_ptr() : nullptr, r.K, q.data_ptr(),
                            r.K, (float*)s.data_ptr(), mode), {y, q, s});
  END_HANDLE_TH_ERRORS
}

// comm_*(x) -> (status, result)
PyObject* comm_per_token_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 1);
  const at::Tensor& x = tensor(a[0]);
  if (x.scalar_type() != kBf16 || x.dim() < 1 || x.numel() == 0 || !x.is_contiguous()) Py_RETURN_NONE;
  const int64_t H = x.size(-1), M = x.numel() / H;
  at::Tensor y = empty_like_rows(x, H + 2, kFp8);
  return with_status(status_of(x, lib.comm_per_token_quant, x.data_ptr(), M, H, y.data_ptr()), {y});
  END_HANDLE_TH_ERRORS
}
PyObject* comm_per_token_dequant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 1);
  const at::Tensor& x = tensor(a[0]);
  if (x.scalar_type() != kFp8 || x.dim() < 1 || x.numel() == 0 || !x.is_contiguous() || x.size(-1) < 3) Py_RETURN_NONE;
  const int64_t H = x.size(-1) - 2, M = x.numel() / (H + 2);
  at::Tensor y = empty_like_rows(x, H, kBf16);
  return with_status(status_of(x, lib.comm_per_token_dequant, x.data_ptr(), M, H, y.data_ptr()), {y});
  END_HANDLE_TH_ERRORS
}
PyObject* comm_qkv_permute_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 1);
  const at::Tensor& x = tensor(a[0]);
  if (x.scalar_type() != kBf16 || x.dim() != 5 || x.stride(4) != 1 || x.stride(3) != x.size(4)) Py_RETURN_NONE;
  const int64_t B = x.size(0), S = x.size(1), P = x.size(2), N = x.size(3), D = x.size(4);
  at::Tensor y = empty({P, S, B, N, D + 4}, kFp8, x);
  return with_status(status_of(x, lib.comm_qkv_permute_quant, x.data_ptr(), B, S, P, N, D, x.stride(0), x.stride(1),
                            x.stride(2), y.data_ptr()), {y});
  END_HANDLE_TH_ERRORS
}
PyObject* comm_qkv_permute_dequant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 1);
  const at::Tensor& x = tensor(a[0]);
  if (x.scalar_type() != kFp8 || x.dim() != 4 || x.stride(3) != 1 || x.size(3) < 4) Py_RETURN_NONE;
  const int64_t S = x.size(0), B = x.size(1), N = x.size(2), D = x.size(3) - 4;
  at::Tensor y = empty({B, S, N, D}, kBf16, x);
  return with_status(status_of(x, lib.comm_qkv_permute_dequant, x.data_ptr(), S, B, N, D, x.stride(0), x.stride(1),
                            x.stride(2), y.data_ptr()), {y});
  END_HANDLE_TH_ERRORS
}

// bind(path): the library at `path`
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 1);
  const char* path = PyUnicode_AsUTF8(a[0]);
  if (!path) throw python_error();
  void* h = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  TORCH_CHECK(h, "cannot load ", path, ": ", dlerror());
  Library l = {};
  auto find = [&](auto& f, const char* name) {
    f = reinterpret_cast<std::remove_reference_t<decltype(f)>>(dlsym(h, name));
    TORCH_CHECK(f, path, " does not export ", name);
  };
  find(l.linear_w8a8, "cdit_fp8_linear_w8a8");
  find(l.gemm_rowwise, "cdit_fp8_gemm_rowwise");
  find(l.gemm_rowwise_batched, "cdit_fp8_gemm_rowwise_batched");
  find(l.w8a16_gemm, "cdit_w8a16_gemm");
  find(l.w8a16_gemm_batched, "cdit_w8a16_gemm_batched");
  find(l.quant_rowwise, "cdit_fp8_quant_rowwise");
  find(l.quant_rowwise_batched, "cdit_fp8_quant_rowwise_batched");
  find(l.quant_rowwise_cat2, "cdit_fp8_quant_rowwise_cat2");
  find(l.quant_tensorwise, "cdit_fp8_quant_tensorwise");
  find(l.ln_modulate_quant, "cdit_fp8_ln_modulate_quant");
  find(l.comm_per_token_quant, "cdit_fp8_comm_per_token_quant");
  find(l.comm_per_token_dequant, "cdit_fp8_comm_per_token_dequant");
  find(l.comm_qkv_permute_quant, "cdit_fp8_comm_qkv_permute_quant");
  find(l.comm_qkv_permute_dequant, "cdit_fp8_comm_qkv_permute_dequant");
  lib = l;
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

#define CDIT_METHOD(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {CDIT_METHOD(bind),
                         CDIT_METHOD(linear_plain),
                         CDIT_METHOD(w8a16_plain),
                         CDIT_METHOD(scaled_mm_plain),
                         CDIT_METHOD(quant_plain),
                         CDIT_METHOD(cat2_plain),
                         CDIT_METHOD(outputs),
                         CDIT_METHOD(workspace),
                         CDIT_METHOD(linear_w8a8),
                         CDIT_METHOD(gemm_rowwise),
                         CDIT_METHOD(w8a16),
                         CDIT_METHOD(quant_rowwise),
                         CDIT_METHOD(quant_tensorwise),
                         CDIT_METHOD(quant_rowwise_cat2),
                         CDIT_METHOD(quant_rowwise_batched),
                         CDIT_METHOD(gemm_batched),
                         CDIT_METHOD(ln_modulate_quant),
                         CDIT_METHOD(comm_per_token_quant),
                         CDIT_METHOD(comm_per_token_dequant),
                         CDIT_METHOD(comm_qkv_permute_quant),
                         CDIT_METHOD(comm_qkv_permute_dequant),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_cdit_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__cdit_host(void) { return PyModule_Create(&module); }

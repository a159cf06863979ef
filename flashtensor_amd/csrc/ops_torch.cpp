// The operators of flashtensor_amd/ops.py on torch tensors: argument checks, results and workspace from torch's
// allocator, one C ABI call (include/ft_abi.h) on the current stream.  Native because the host side is what a short call
// costs: the same steps as Python over the pybind11 module took 10.3 us of host time per attention call (B1 H8 S200 D64), these
// take 4.5 (three to four of them the launch itself), where the kernel takes 5 to 8.  Bound with the C calling convention of CPython (METH_FASTCALL): ops.py
// passes every argument by position.
#include <torch/csrc/Dtype.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>

#include <cmath>
#include <sstream>
#include <stdexcept>
#include <string>

#include "../../include/ft_abi.h"

namespace {

PyObject* g_raw_stream = nullptr;  // torch._C._cuda_getCurrentRawStream

[[noreturn]] void bad_value(const std::string& m) { throw std::invalid_argument(m); }
[[noreturn]] void bad_call(const std::string& m) { throw std::runtime_error(m); }

std::string str_of(const at::Tensor& t) {
  std::ostringstream s;
  s << "(";
  for (int64_t i = 0; i < t.dim(); ++i) s << (i ? ", " : "") << t.size(i);
  s << (t.dim() == 1 ? ",)" : ")");
  return s.str();
}
std::string str_of(at::IntArrayRef v) {
  std::ostringstream s;
  s << "(";
  for (size_t i = 0; i < v.size(); ++i) s << (i ? ", " : "") << v[i];
  s << (v.size() == 1 ? ",)" : ")");
  return s.str();
}
std::string str_of(at::ScalarType t) {
  PyObject* r = PyObject_Str(reinterpret_cast<PyObject*>(torch::getTHPDtype(t)));
  std::string out = r ? PyUnicode_AsUTF8(r) : "?";
  Py_XDECREF(r);
  return out;
}

// ft_last_error() is thread-local and read before anything else runs on this thread
void check(int rc) {
  if (rc == FT_OK) return;
  const std::string msg = std::string("libflashtensor_hip: ") + ft_last_error() + " (status " + std::to_string(rc) + ")";
  if (rc == FT_EINVAL) bad_value(msg);
  bad_call(msg);
}

// the launches only queue kernels and touch no Python object
template <typename F>
void launch(F&& f) {
  int rc;
  std::string msg;
  Py_BEGIN_ALLOW_THREADS
  rc = f();
  Py_END_ALLOW_THREADS
  check(rc);
}

void* stream_of(const at::Tensor& t) {
  PyObject* dev = PyLong_FromLong(t.get_device());
  PyObject* r = dev ? PyObject_CallOneArg(g_raw_stream, dev) : nullptr;
  Py_XDECREF(dev);
  if (!r) throw python_error();
  void* s = PyLong_AsVoidPtr(r);
  Py_DECREF(r);
  return s;
}

const at::Tensor& tensor_arg(PyObject* o, int i) {
  if (!THPVariable_Check(o)) bad_call("arg " + std::to_string(i) + " need a torch.Tensor but got " + Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}
bool flag_arg(PyObject* o) {
  const int r = PyObject_IsTrue(o);
  if (r < 0) throw python_error();
  return r;
}
double float_arg(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw python_error();
  return v;
}
// Counts and sizes cross the C ABI as int32: what does not fit is refused, here and nowhere else cut.
int32_t int32_arg(PyObject* o, const char* what) {
  int over = 0;
  const long long v = PyLong_AsLongLongAndOverflow(o, &over);
  if (v == -1 && PyErr_Occurred()) throw python_error();
  if (over || v != (int32_t)v) bad_value(std::string(what) + " does not fit 32 bits");
  return (int32_t)v;
}
int32_t size32(const at::Tensor& t, int64_t dim) {
  const int64_t n = t.size(dim);
  if (n != (int32_t)n) bad_value("need sizes that fit 32 bits but got shape " + str_of(t));
  return (int32_t)n;
}

int ft_dtype(at::ScalarType t, bool linear) {
  if (t == at::kHalf) return FT_F16;
  if (t == at::kBFloat16) return FT_BF16;
  return linear && t == at::kFloat ? (int)FT_F32 : -1;
}

void dense_last(const at::Tensor& t) {
  if (t.stride(-1) != 1 && t.size(-1) != 1)
    bad_value("need a contiguous last axis but got strides " + str_of(t.strides()) + " for shape " + str_of(t));
}

FtStrides strides_of(const at::Tensor& t) { return FtStrides{t.stride(0), t.stride(1), t.stride(2)}; }

struct Qkv {
  const at::Tensor &q, &k, &v;
  int32_t B, Sq, H, D, Skv, Hkv;
  int dtype;

  Qkv(PyObject* const* args, bool linear = false) : q(tensor_arg(args[0], 0)), k(tensor_arg(args[1], 1)), v(tensor_arg(args[2], 2)) {
    const at::Tensor* all[3] = {&q, &k, &v};
    for (int i = 0; i < 3; ++i) {
      const at::Tensor& t = *all[i];
      const std::string arg = "arg " + std::to_string(i);
      if (t.dim() != 4) bad_call(arg + " need shape [B, S, H, D] but got " + str_of(t));
      if (!t.is_cuda()) bad_call(arg + " need a GPU tensor but got device " + t.device().str());
      if (t.scalar_type() != q.scalar_type() || t.device() != q.device())
        bad_call(arg + " need dtype " + str_of(q.scalar_type()) + " on " + q.device().str() + " but got " + str_of(t.scalar_type()) + " on " + t.device().str());
    }
    dtype = ft_dtype(q.scalar_type(), linear);
    if (dtype < 0) bad_call(std::string("arg 0 need dtype float16 or bfloat16") + (linear ? " or float32" : "") + " but got " + str_of(q.scalar_type()));
    B = size32(q, 0), Sq = size32(q, 1), H = size32(q, 2), D = size32(q, 3);
    Skv = size32(k, 1), Hkv = size32(k, 2);
    if (k.size(0) != B || k.size(3) != D || Hkv < 1 || H % Hkv != 0)
      bad_call("arg 1 need shape (" + std::to_string(B) + ", " + std::to_string(Skv) + ", 'a divisor of " + std::to_string(H) + "', " + std::to_string(D) +
               ") but got " + str_of(k));
    if (v.sizes() != k.sizes()) bad_call("arg 2 need shape " + str_of(k) + " but got " + str_of(v));
    for (const at::Tensor* t : all) dense_last(*t);
  }
  FtAttnArgs args(const at::Tensor& o, unsigned flags) const {
    return FtAttnArgs{q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), o.data_ptr(), strides_of(q), strides_of(k), strides_of(v), strides_of(o),
                      B, H, Sq, Skv, D, dtype, flags, Hkv};
  }
  at::Tensor out() const { return at::empty({B, Sq, H, D}, q.options()); }
  at::Tensor f32(at::IntArrayRef shape) const { return at::empty(shape, q.options().dtype(at::kFloat)); }
};

unsigned flags_of(PyObject* causal, PyObject* fast) { return (flag_arg(causal) ? FT_CAUSAL : 0u) | (flag_arg(fast) ? FT_FAST_LOGITS : 0u); }

at::Tensor workspace(const at::Tensor& like, size_t bytes) {
  return bytes ? at::empty({(int64_t)bytes}, like.options().dtype(at::kByte)) : at::Tensor();
}
void* ptr(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

PyObject* result(const at::Tensor& t) { return THPVariable_Wrap(t); }
template <typename... Ts>
PyObject* result(const at::Tensor& a, const Ts&... more) {
  PyObject* items[] = {THPVariable_Wrap(a), THPVariable_Wrap(more)...};
  constexpr int n = 1 + sizeof...(more);
  PyObject* tuple = PyTuple_New(n);
  for (int i = 0; i < n; ++i) {
    if (tuple) PyTuple_SET_ITEM(tuple, i, items[i]);
  }
  return tuple;
}

// the attention pass of attn (softcap 0) and gemma2
at::Tensor run_attn(const Qkv& x, unsigned flags, float softcap, const at::Tensor& lse) {
  at::Tensor out = x.out();
  const FtAttnArgs a = x.args(out, flags);
  const size_t bytes = ft_attn_workspace_bytes(&a, softcap);
  const at::Tensor ws = workspace(x.q, bytes);
  void* s = stream_of(x.q);
  launch([&] { return ft_attn_fwd_ws(&a, softcap, static_cast<float*>(ptr(lse)), ptr(ws), bytes, s); });
  return out;
}

// attn(q, k, v, causal, fast_logits, return_lse)
PyObject* attn(PyObject* const* o) {
  const Qkv x(o);
  const unsigned flags = flags_of(o[3], o[4]);
  if (!flag_arg(o[5])) return result(run_attn(x, flags, 0.f, at::Tensor()));
  const at::Tensor lse = x.f32({x.B, x.H, x.Sq});
  return result(run_attn(x, flags, 0.f, lse), lse);
}

// gemma2(q, k, v, softcap, causal, fast_logits)
PyObject* gemma2(PyObject* const* o) {
  const Qkv x(o);
  const float cap = (float)float_arg(o[3]);
  if (!(cap > 0.f) || !std::isfinite(cap)) bad_value("softcap must be positive and finite");
  return result(run_attn(x, flags_of(o[4], o[5]), cap, at::Tensor()));
}

struct Stats {
  at::Tensor out, s1, s2;
};
Stats run_colstats(const Qkv& x, bool want_sq, unsigned flags, void* stream) {
  Stats r{x.out(), x.f32({x.B, x.Hkv, x.Skv}), want_sq ? x.f32({x.B, x.H, x.Skv}) : at::Tensor()};
  const FtAttnArgs a = x.args(r.out, flags);
  const size_t bytes = ft_workspace_bytes_split(FT_OP_COLSTATS, &a);
  const at::Tensor ws = workspace(x.q, bytes);
  launch([&] { return ft_attn_colstats_fwd(&a, static_cast<float*>(ptr(r.s1)), static_cast<float*>(ptr(r.s2)), ptr(ws), bytes, stream); });
  return r;
}

// h2o(q, k, v, causal, fast_logits), roco(...)
PyObject* h2o(PyObject* const* o) {
  const Qkv x(o);
  const Stats r = run_colstats(x, false, flags_of(o[3], o[4]), stream_of(x.q));
  return result(r.out, r.s1);
}
PyObject* roco(PyObject* const* o) {
  const Qkv x(o);
  const Stats r = run_colstats(x, true, flags_of(o[3], o[4]), stream_of(x.q));
  return result(r.out, r.s1, r.s2);
}

// snapkv(q, k, v, kernel_size, causal, fast_logits)
PyObject* snapkv(PyObject* const* o) {
  const Qkv x(o);
  void* s = stream_of(x.q);
  const int32_t kernel = int32_arg(o[3], "kernel_size");
  const at::Tensor out = x.out(), pooled = x.f32({x.B, x.Hkv, x.Skv});
  const FtAttnArgs a = x.args(out, flags_of(o[4], o[5]));
  const size_t bytes = ft_workspace_bytes_split(FT_OP_SNAPKV, &a);
  const at::Tensor ws = workspace(x.q, bytes);
  launch([&] { return ft_snapkv_fwd(&a, kernel, pooled.data_ptr<float>(), ptr(ws), bytes, s); });
  return result(out, pooled);
}

void check_f32(const at::Tensor& t, const at::Tensor& like, at::IntArrayRef shape, const char* arg) {
  if (t.sizes() != shape) bad_call(std::string(arg) + " need shape " + str_of(shape) + " but got " + str_of(t));
  if (t.scalar_type() != at::kFloat || t.device() != like.device())
    bad_call(std::string(arg) + " need dtype torch.float32 on " + like.device().str() + " but got " + str_of(t.scalar_type()) + " on " + t.device().str());
  dense_last(t);
}

// keyformer(q, k, v, exp_rand, tau, seed, causal, fast_logits)
PyObject* keyformer(PyObject* const* o) {
  const Qkv x(o);
  FtNoise noise{nullptr, 0, 0, 0, 0};
  if (o[3] != Py_None) {
    const at::Tensor& e = tensor_arg(o[3], 3);
    check_f32(e, x.q, {x.B, x.H, x.Sq, x.Skv}, "arg 3");
    noise = FtNoise{e.const_data_ptr<float>(), e.stride(0), e.stride(1), e.stride(2), 0};
  } else {
    noise.seed = PyLong_AsUnsignedLongLongMask(o[5]);
    if (PyErr_Occurred()) throw python_error();
  }
  const float tau = (float)float_arg(o[4]);
  const at::Tensor out = x.out(), score = x.f32({x.B, x.H, x.Skv});
  const FtAttnArgs a = x.args(out, flags_of(o[6], o[7]));
  const size_t bytes = ft_workspace_bytes_split(FT_OP_KEYFORMER, &a);
  const at::Tensor ws = workspace(x.q, bytes);
  void* s = stream_of(x.q);
  launch([&] { return ft_keyformer_fwd(&a, &noise, tau, score.data_ptr<float>(), ptr(ws), bytes, s); });
  return result(out, score);
}

// corm(q, k, v, corm_mask, causal, fast_logits, return_margin)
PyObject* corm(PyObject* const* o) {
  const Qkv x(o);
  const float* mask = nullptr;
  int64_t mask_stride = 0;
  if (o[3] != Py_None) {
    const at::Tensor& m = tensor_arg(o[3], 3);
    check_f32(m, x.q, {x.Sq, x.Skv}, "arg 3");
    mask = m.const_data_ptr<float>();
    mask_stride = m.stride(0);
  }
  const at::Tensor out = x.out(), keep = at::empty({x.B, x.H, x.Skv}, x.q.options().dtype(at::kBool));
  const at::Tensor margin = flag_arg(o[6]) ? x.f32({x.B, x.H, x.Skv}) : at::Tensor();
  const FtAttnArgs a = x.args(out, flags_of(o[4], o[5]));
  const size_t bytes = ft_workspace_bytes_split(FT_OP_CORM, &a);
  const at::Tensor ws = workspace(x.q, bytes);
  void* s = stream_of(x.q);
  launch([&] { return ft_corm_fwd(&a, mask, mask_stride, static_cast<uint8_t*>(ptr(keep)), static_cast<float*>(ptr(margin)), ptr(ws), bytes, s); });
  return margin.defined() ? result(out, keep, margin) : result(out, keep);
}

// linattn(q, k, v, kind, normalize_q, out_dtype or None)
PyObject* linattn(PyObject* const* o) {
  const Qkv x(o, true);
  if (x.D == 32) {  // head_dim 32 runs as pairs of adjacent heads: heads must lie 32 elements apart
    const at::Tensor* all[3] = {&x.q, &x.k, &x.v};
    for (int i = 0; i < 3; ++i)
      if (all[i]->stride(2) != 32)
        bad_value("arg " + std::to_string(i) + " with head_dim 32 need heads stored 32 elements apart but got head stride " + std::to_string(all[i]->stride(2)));
  }
  const int kind = int32_arg(o[3], "kind");
  const bool normalize_q = flag_arg(o[4]);
  at::ScalarType out_type = x.q.scalar_type();
  if (o[5] != Py_None) {
    if (!THPDtype_Check(o[5])) bad_call("out_dtype need a torch.dtype");
    out_type = reinterpret_cast<THPDtype*>(o[5])->scalar_type;
    if (out_type != x.q.scalar_type() && out_type != at::kFloat)
      bad_call("out_dtype need " + str_of(x.q.scalar_type()) + " or float32 but got " + str_of(out_type));
  }
  const at::Tensor out = at::empty({x.B, x.Sq, x.H, x.D}, x.q.options().dtype(out_type));
  const FtAttnArgs a = x.args(out, 0);
  const size_t bytes = ft_workspace_bytes(kind, &a);
  const at::Tensor ws = workspace(x.q, bytes);
  void* s = stream_of(x.q);
  launch([&] { return ft_linattn_fwd(&a, kind, normalize_q, ft_dtype(out_type, true), ptr(ws), bytes, s); });
  return result(out);
}

// linattn_block(x, w_qkv, b_qkv, w_out, b_out, head_num, kind, normalize_q)
PyObject* linattn_block(PyObject* const* o) {
  static const char* const names[5] = {"x", "w_qkv", "b_qkv", "w_out", "b_out"};
  const at::Tensor* t[5];
  for (int i = 0; i < 5; ++i) {
    t[i] = nullptr;
    if (o[i] == Py_None && names[i][0] == 'b') continue;
    const std::string arg = "arg " + std::to_string(i) + " (" + names[i] + ")";
    if (!THPVariable_Check(o[i]) || !THPVariable_Unpack(o[i]).is_cuda()) bad_call(arg + " need a GPU tensor");
    t[i] = &THPVariable_Unpack(o[i]);
    if (t[i]->scalar_type() != t[0]->scalar_type()) bad_call(arg + " need " + str_of(t[0]->scalar_type()) + " but got " + str_of(t[i]->scalar_type()));
  }
  const at::Tensor& x = *t[0];
  const int32_t heads = int32_arg(o[5], "head_num");
  if (x.dim() != 3 || heads < 1 || x.size(2) % heads)
    bad_value("x need [B,S,C] with C a multiple of head_num=" + std::to_string(heads) + " but got " + str_of(x));
  const int32_t B = size32(x, 0), S = size32(x, 1);
  const int64_t C = x.size(2);
  if (t[1]->sizes() != at::IntArrayRef{3 * C, C} || t[3]->sizes() != at::IntArrayRef{C, C})
    bad_value("weights need [" + std::to_string(3 * C) + "," + std::to_string(C) + "] and [" + std::to_string(C) + "," + std::to_string(C) + "] but got " +
              str_of(*t[1]) + " and " + str_of(*t[3]));
  if ((t[2] && t[2]->sizes() != at::IntArrayRef{3 * C}) || (t[4] && t[4]->sizes() != at::IntArrayRef{C}))
    bad_value("biases need [" + std::to_string(3 * C) + "] and [" + std::to_string(C) + "]");
  for (int i = 0; i < 5; ++i)
    if (t[i] && !t[i]->is_contiguous())
      bad_value("arg " + std::to_string(i) + " (" + names[i] + ") need a contiguous tensor but got strides " + str_of(t[i]->strides()));
  const int dtype = ft_dtype(x.scalar_type(), true);
  if (dtype < 0) bad_call("arg 0 (x) need float16, bfloat16 or float32 but got " + str_of(x.scalar_type()));
  const int kind = int32_arg(o[6], "kind");
  const bool normalize_q = flag_arg(o[7]);
  const at::Tensor y = at::empty({B, S, C}, x.options());
  auto data = [&](int i) -> const void* { return t[i] ? t[i]->const_data_ptr() : nullptr; };
  const FtLinBlockArgs a{data(0), data(1), data(2), data(3), data(4), y.data_ptr(), B, S, heads, size32(x, 2) / heads, dtype};
  const size_t bytes = ft_linattn_block_workspace_bytes(&a, kind);
  if (bytes == 0) bad_call(std::string("libflashtensor_hip: ") + ft_last_error());
  const at::Tensor ws = workspace(x, bytes);
  void* s = stream_of(x);
  launch([&] { return ft_linattn_block_fwd(&a, kind, normalize_q, ptr(ws), bytes, s); });
  return result(y);
}

// topk(score, k)
PyObject* topk(PyObject* const* o) {
  const at::Tensor& score = tensor_arg(o[0], 0);
  if (score.scalar_type() != at::kFloat || !score.is_cuda())
    bad_call("arg 0 need a float32 GPU tensor but got " + str_of(score.scalar_type()) + " on " + score.device().str());
  if (!score.is_contiguous()) bad_value("arg 0 need a contiguous tensor but got strides " + str_of(score.strides()));
  if (score.dim() < 1 || score.size(-1) < 1) bad_value("arg 0 need a last axis with entries but got " + str_of(score));
  const int32_t S = size32(score, -1), k = int32_arg(o[1], "k");
  const int64_t rows = score.numel() / S;
  std::vector<int64_t> shape = score.sizes().vec();
  shape.back() = k;
  const at::Tensor idx = at::empty(shape, score.options().dtype(at::kLong));
  void* s = stream_of(score);
  launch([&] { return ft_topk(score.const_data_ptr<float>(), rows, S, k, idx.data_ptr<int64_t>(), s); });
  return result(idx);
}

template <PyObject* (*F)(PyObject* const*), int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != N) {
    PyErr_Format(PyExc_TypeError, "%d arguments needed, got %zd", N, n);
    return nullptr;
  }
  try {
    return F(args);
  } catch (const std::invalid_argument& e) {
    PyErr_SetString(PyExc_ValueError, e.what());
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

#define FT_ENTRY(name, n) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<name, n>)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {FT_ENTRY(attn, 6),      FT_ENTRY(gemma2, 6), FT_ENTRY(h2o, 5),     FT_ENTRY(roco, 5),          FT_ENTRY(snapkv, 6),
                           FT_ENTRY(keyformer, 8), FT_ENTRY(corm, 7),   FT_ENTRY(linattn, 6), FT_ENTRY(linattn_block, 8), FT_ENTRY(topk, 2),
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "ft_ops", "flashtensor_amd operators on torch tensors", -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_ft_ops(void) {
  PyObject* c = PyImport_ImportModule("torch._C");
  if (!c) return nullptr;
  g_raw_stream = PyObject_GetAttrString(c, "_cuda_getCurrentRawStream");
  Py_DECREF(c);
  if (!g_raw_stream) return nullptr;
  return PyModule_Create(&g_module);
}

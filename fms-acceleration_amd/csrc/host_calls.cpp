// The tensor-level calls of the operators' hot path as a CPython extension: what fmsa_hip/__init__.py names lora_down,
// gptq_lora_fwd, .. allocates the outputs and partial sums, fills the C-ABI structs and calls libfmsa_hip.so here.  A layer's
// training pass makes 23 of these calls, and in Python (ctypes structs, torch.empty, attribute reads) they cost the host
// 15 to 30 us each, which is more than the GPU spends on them up to a few hundred tokens.  Host code only; arguments are checked
// as the C ABI checks them and a refusal raises the FmsaError that install() was given.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "../../include/fmsa.h"

namespace {

struct PyFailure {};  // a Python error is set

PyObject* g_fmsa_error = nullptr;  // fmsa_hip.FmsaError(fn, code)

void check(const char* fn, int code) {
  if (code == FMSA_OK) return;
  PyObject* err = PyObject_CallFunction(g_fmsa_error, "si", fn, code);
  if (err) {
    PyErr_SetObject(g_fmsa_error, err);
    Py_DECREF(err);
  }
  throw PyFailure();
}

void need(bool ok, const char* what) {
  if (ok) return;
  PyErr_SetString(PyExc_AssertionError, what);
  throw PyFailure();
}

const at::Tensor& tensor(PyObject* o) {
  if (!o || !THPVariable_Check(o)) {
    PyErr_SetString(PyExc_TypeError, "expected a tensor");
    throw PyFailure();
  }
  return THPVariable_Unpack(o);
}

at::Tensor optional(PyObject* o) { return !o || o == Py_None ? at::Tensor() : tensor(o); }

void* ptr(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

int dtype_enum(at::ScalarType t) {
  switch (t) {
    case at::kHalf: return FMSA_F16;
    case at::kBFloat16: return FMSA_BF16;
    case at::kFloat: return FMSA_F32;
    default: PyErr_SetString(PyExc_KeyError, "dtype must be float16, bfloat16 or float32"); throw PyFailure();
  }
}

int act_enum(at::ScalarType t) {
  if (t == at::kHalf) return FMSA_F16;
  if (t == at::kBFloat16) return FMSA_BF16;
  PyErr_Format(PyExc_TypeError, "activations must be float16 or bfloat16, got %s", c10::toString(t));
  throw PyFailure();
}

void* stream(const at::Tensor& t) {
  if (!t.is_cuda()) {
    PyErr_SetString(PyExc_RuntimeError, "libfmsa_hip kernels need tensors on the GPU (there is no CPU implementation)");
    throw PyFailure();
  }
  return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.get_device()).stream();
}

void on_gpu(bool ok) {
  if (ok) return;
  PyErr_SetString(PyExc_RuntimeError, "fmsa_hip needs GPU tensors");
  throw PyFailure();
}

// The call itself without the interpreter lock: a full launch queue blocks it.
template <typename F> int unlocked(F&& f) {
  PyThreadState* s = PyEval_SaveThread();
  const int rc = f();
  PyEval_RestoreThread(s);
  return rc;
}

at::Tensor empty(std::initializer_list<int64_t> sizes, const at::Tensor& like) { return at::empty(sizes, like.options()); }
at::Tensor empty(std::initializer_list<int64_t> sizes, const at::Tensor& like, at::ScalarType t) {
  return at::empty(sizes, like.options().dtype(t));
}
at::Tensor workspace(size_t bytes, const at::Tensor& like) {
  return at::empty({(int64_t)std::max<size_t>(bytes, 16)}, like.options().dtype(at::kByte));
}

// Owned reference released on every way out
struct Ref {
  PyObject* o;
  explicit Ref(PyObject* p) : o(p) {
    if (!p) throw PyFailure();
  }
  ~Ref() { Py_XDECREF(o); }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
  PyObject* release() {
    PyObject* r = o;
    o = nullptr;
    return r;
  }
};

PyObject* wrap(at::Tensor t) { return THPVariable_Wrap(std::move(t)); }

PyObject* wrap_list(const std::vector<at::Tensor>& ts) {
  Ref list(PyList_New((Py_ssize_t)ts.size()));
  for (size_t i = 0; i < ts.size(); ++i) PyList_SET_ITEM(list.o, (Py_ssize_t)i, wrap(ts[i]));
  return list.release();
}

double number(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw PyFailure();
  return v;
}

long integer(PyObject* o) {
  const long v = PyLong_AsLong(o);
  if (v == -1 && PyErr_Occurred()) throw PyFailure();
  return v;
}

bool truth(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw PyFailure();
  return v != 0;
}

at::ScalarType dtype_of(PyObject* o) {
  if (!THPDtype_Check(o)) {
    PyErr_SetString(PyExc_TypeError, "expected a dtype");
    throw PyFailure();
  }
  return reinterpret_cast<THPDtype*>(o)->scalar_type;
}

fmsa_gptq_weight weight(PyObject* o) {  // the ctypes GptqWeight, whose memory is the C struct
  Py_buffer b;
  if (PyObject_GetBuffer(o, &b, PyBUF_SIMPLE) != 0) throw PyFailure();
  const bool ok = b.len == (Py_ssize_t)sizeof(fmsa_gptq_weight);
  fmsa_gptq_weight w{};
  if (ok) w = *static_cast<const fmsa_gptq_weight*>(b.buf);
  PyBuffer_Release(&b);
  need(ok, "w must be a GptqWeight");
  return w;
}

struct Sequence {  // list or tuple
  PyObject* fast;
  explicit Sequence(PyObject* o) : fast(PySequence_Fast(o, "expected a sequence")) {
    if (!fast) throw PyFailure();
  }
  ~Sequence() { Py_DECREF(fast); }
  Sequence(const Sequence&) = delete;
  Sequence& operator=(const Sequence&) = delete;
  Py_ssize_t size() const { return PySequence_Fast_GET_SIZE(fast); }
  PyObject* operator[](Py_ssize_t i) const { return PySequence_Fast_GET_ITEM(fast, i); }
};

PyObject* key(const char* name) { return PyUnicode_InternFromString(name); }

PyObject* item(PyObject* dict, PyObject* k, bool required = true) {  // borrowed; nullptr where absent
  PyObject* v = PyDict_GetItemWithError(dict, k);
  if (!v && (required || PyErr_Occurred())) {
    if (!PyErr_Occurred()) PyErr_SetObject(PyExc_KeyError, k);
    throw PyFailure();
  }
  return v;
}

template <PyObject* (*F)(PyObject* const*, Py_ssize_t), int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != N) {
    PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", N, n);
    return nullptr;
  }
  try {
    return F(args, n);
  } catch (const PyFailure&) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

// ---- rank-r products ----------------------------------------------------------------------------------------------------
at::Tensor down_one(const at::Tensor& x, const at::Tensor& wd, at::Tensor out) {
  need(x.dim() == 2, "lora_down: x2d");
  const int64_t M = x.size(0), C = x.size(1), r = wd.size(0);
  need(wd.size(1) == C && wd.is_contiguous() && wd.scalar_type() == x.scalar_type() && x.stride(1) == 1, "lora_down: x2d, wd");
  if (!out.defined()) out = empty({M, r}, x);
  need(out.dim() == 2 && out.size(0) == M && out.size(1) == r && out.stride(1) == 1 && out.scalar_type() == x.scalar_type(), "lora_down: out");
  const int act = act_enum(x.scalar_type());
  void* st = stream(out);
  const size_t bytes = fmsa_lora_down_split_workspace((int)M, (int)C, (int)r);
  const at::Tensor ws = bytes ? workspace(bytes, x) : at::Tensor();
  check("fmsa_lora_down_split", unlocked([&] {
          return fmsa_lora_down_split(ptr(x), x.stride(0), ptr(wd), (int)M, (int)C, (int)r, act, ptr(out), out.stride(0), ptr(ws),
                                      ws.defined() ? ws.numel() : 0, st);
        }));
  return out;
}

PyObject* lora_down(PyObject* const* a, Py_ssize_t) { return wrap(down_one(tensor(a[0]), tensor(a[1]), optional(a[2]))); }

PyObject* lora_down_batch(PyObject* const* a, Py_ssize_t) {  // jobs, most tokens
  Sequence jobs(a[0]);
  const Py_ssize_t n = jobs.size();
  need(n > 0, "lora_down_batch: no jobs");
  struct Job {
    at::Tensor x, wd, out;
  };
  std::vector<Job> js;
  for (Py_ssize_t i = 0; i < n; ++i) {
    Sequence j(jobs[i]);
    need(j.size() == 3, "lora_down_batch: (x2d, wd, out)");
    js.push_back({tensor(j[0]), tensor(j[1]), optional(j[2])});
  }
  const int64_t M = js[0].x.size(0);
  bool single = n < 2 || M > integer(a[1]);
  for (const Job& j : js)
    single = single || j.x.size(1) % 8 || (j.out.defined() && (reinterpret_cast<uintptr_t>(ptr(j.out)) % 8 || j.out.stride(0) % 4));
  std::vector<at::Tensor> outs;
  if (single) {
    for (const Job& j : js) outs.push_back(down_one(j.x, j.wd, j.out));
    return wrap_list(outs);
  }
  for (const Job& j : js) need(j.x.dim() == 2 && j.wd.dim() == 2, "lora_down_batch: x2d, wd");
  const at::Tensor& x0 = js[0].x;
  const int act = act_enum(x0.scalar_type());
  void* st = stream(x0);
  for (Py_ssize_t i = 0; i < n; i += FMSA_LORA_DOWN_MAX_JOBS) {
    const int m = (int)std::min<Py_ssize_t>(FMSA_LORA_DOWN_MAX_JOBS, n - i);
    fmsa_lora_down_job arr[FMSA_LORA_DOWN_MAX_JOBS] = {};
    for (int q = 0; q < m; ++q) {
      Job& j = js[i + q];
      const int64_t r = j.wd.size(0), C = j.wd.size(1);
      need(j.x.size(0) == M && j.x.size(1) == C && j.wd.is_contiguous() && j.wd.scalar_type() == x0.scalar_type() &&
               j.x.scalar_type() == x0.scalar_type() && j.x.stride(1) == 1, "lora_down_batch: x2d, wd");
      if (!j.out.defined()) j.out = empty({M, r}, j.x);
      need(j.out.dim() == 2 && j.out.size(0) == M && j.out.size(1) == r && j.out.stride(1) == 1 && j.out.scalar_type() == x0.scalar_type(),
           "lora_down_batch: out");
      arr[q].X = ptr(j.x);
      arr[q].Wd = ptr(j.wd);
      arr[q].out = ptr(j.out);
      arr[q].ldx = j.x.stride(0);
      arr[q].ldout = j.out.stride(0);
      arr[q].C = (int)C;
      arr[q].r = (int)r;
      outs.push_back(j.out);
    }
    const at::Tensor ws = workspace(fmsa_lora_down_batch_workspace(arr, m, (int)M), x0);
    check("fmsa_lora_down_batch",
          unlocked([&] { return fmsa_lora_down_batch(arr, m, (int)M, act, ptr(ws), ws.numel(), st); }));
  }
  return wrap_list(outs);
}

PyObject* lora_grad_batch(PyObject* const* a, Py_ssize_t) {  // jobs, most of them a launch
  Sequence jobs(a[0]);
  const Py_ssize_t n = jobs.size();
  const long most = integer(a[1]);
  std::vector<at::Tensor> outs;
  for (Py_ssize_t i = 0; i < n; i += most) {
    const int m = (int)std::min<Py_ssize_t>(most, n - i);
    std::vector<fmsa_lora_grad_job> arr(m);
    at::Tensor r0;
    int64_t M = 0;
    for (int q = 0; q < m; ++q) {
      Sequence j(jobs[i + q]);
      need(j.size() == 5 || j.size() == 7, "lora_grad_batch: (L, R, scale, transpose_out, out_dtype[, Wt, T_out])");
      const at::Tensor &L = tensor(j[0]), &R = tensor(j[1]);
      const at::Tensor Wt = j.size() == 7 ? optional(j[5]) : at::Tensor(), T = j.size() == 7 ? optional(j[6]) : at::Tensor();
      if (q == 0) {
        M = L.size(0);
        r0 = R;
      }
      const int64_t r = L.size(1), C = R.size(1);
      need(L.size(0) == M && R.size(0) == M && L.stride(1) == 1 && R.stride(1) == 1, "lora_grad_batch: L, R");
      need(L.scalar_type() == R.scalar_type() && R.scalar_type() == r0.scalar_type(), "lora_grad_batch: dtypes");
      if (Wt.defined()) {
        need(Wt.dim() == 2 && Wt.size(0) == r && Wt.size(1) == C && Wt.is_contiguous() && Wt.scalar_type() == R.scalar_type(), "lora_grad_batch: Wt");
        need(T.defined() && T.dim() == 2 && T.size(0) == M && T.size(1) == r && T.stride(1) == 1 && T.scalar_type() == R.scalar_type(), "lora_grad_batch: T_out");
      }
      const bool tr = truth(j[3]);
      const at::ScalarType od = dtype_of(j[4]);
      at::Tensor out = tr ? empty({C, r}, R, od) : empty({r, C}, R, od);
      arr[q] = {};
      arr[q].L = ptr(L);
      arr[q].R = ptr(R);
      arr[q].out = ptr(out);
      arr[q].ldl = L.stride(0);
      arr[q].ldr = R.stride(0);
      arr[q].C = (int)C;
      arr[q].r = (int)r;
      arr[q].scale = (float)number(j[2]);
      arr[q].transpose_out = tr;
      arr[q].out_dtype = dtype_enum(od);
      arr[q].Wt = ptr(Wt);
      arr[q].T = ptr(T);
      arr[q].ldt = T.defined() ? T.stride(0) : 0;
      outs.push_back(std::move(out));
    }
    const int act = act_enum(r0.scalar_type());
    void* st = stream(r0);
    const at::Tensor ws = workspace(fmsa_lora_grad_batch_workspace(arr.data(), m, (int)M), r0);
    check("fmsa_lora_grad_batch",
          unlocked([&] { return fmsa_lora_grad_batch(arr.data(), m, (int)M, act, ptr(ws), ws.numel(), st); }));
  }
  return wrap_list(outs);
}

PyObject* lora_pack_batch(PyObject* const* a, Py_ssize_t) {  // adapters, act_dtype, most of them a launch
  Sequence adapters(a[0]);
  const at::ScalarType act = dtype_of(a[1]);
  const int act_e = act_enum(act);
  const long most = integer(a[2]);
  const Py_ssize_t n = adapters.size();
  Ref list(PyList_New(n));
  std::vector<fmsa_lora_pack_job> jobs(n);
  std::vector<at::Tensor> keep;
  void* st = nullptr;
  for (Py_ssize_t i = 0; i < n; ++i) {
    Sequence j(adapters[i]);
    need(j.size() == 3, "lora_pack_batch: (A, B, A16_out)");
    at::Tensor A = tensor(j[0]), B = tensor(j[1]), A16 = optional(j[2]);
    need(A.dim() == 2, "lora_pack_batch: A");
    if (!(A.is_cuda() && B.is_cuda())) {
      PyErr_SetString(PyExc_RuntimeError, "fmsa_hip needs GPU tensors");
      throw PyFailure();
    }
    if (A.scalar_type() != B.scalar_type()) B = B.detach().to(A.scalar_type());
    if (!A.is_contiguous()) A = A.detach().contiguous();
    if (!B.is_contiguous()) B = B.detach().contiguous();
    const int64_t r = A.size(0), K = A.size(1), N = B.size(0);
    if (A16.defined())
      need(A16.dim() == 2 && A16.size(0) == r && A16.size(1) == K && A16.is_contiguous() && A16.scalar_type() == act, "lora_pack_batch: A16_out");
    else
      A16 = empty({r, K}, A, act);
    at::Tensor At = empty({K, r}, A, act), B16 = empty({N, r}, A, act), Bt = empty({r, N}, A, act);
    jobs[i] = {};
    jobs[i].A = ptr(A);
    jobs[i].B = ptr(B);
    jobs[i].A16 = ptr(A16);
    jobs[i].At16 = ptr(At);
    jobs[i].B16 = ptr(B16);
    jobs[i].Bt16 = ptr(Bt);
    jobs[i].r = (int)r;
    jobs[i].K = (int)K;
    jobs[i].N = (int)N;
    jobs[i].param_dtype = dtype_enum(A.scalar_type());
    if (i == 0) st = stream(A);
    keep.push_back(std::move(A));
    keep.push_back(std::move(B));
    Ref quad(PyTuple_New(4));
    PyTuple_SET_ITEM(quad.o, 0, j[2] == Py_None ? wrap(std::move(A16)) : (Py_INCREF(j[2]), j[2]));
    PyTuple_SET_ITEM(quad.o, 1, wrap(std::move(At)));
    PyTuple_SET_ITEM(quad.o, 2, wrap(std::move(B16)));
    PyTuple_SET_ITEM(quad.o, 3, wrap(std::move(Bt)));
    PyList_SET_ITEM(list.o, i, quad.release());
  }
  for (Py_ssize_t i = 0; i < n; i += most)
    check("fmsa_lora_pack_batch", unlocked([&] {
            return fmsa_lora_pack_batch(jobs.data() + i, (int)std::min<Py_ssize_t>(most, n - i), act_e, st);
          }));
  return list.release();
}

// ---- fused GEMMs ----------------------------------------------------------------------------------------------------------
PyObject* gptq_lora_fwd(PyObject* const* a, Py_ssize_t) {  // x2d, projs, mode, split
  const at::Tensor& x = tensor(a[0]);
  Sequence projs(a[1]);
  const int mode = (int)integer(a[2]), n = (int)projs.size();
  const bool split = truth(a[3]);
  static PyObject *kw = key("w"), *kU = key("U"), *kB = key("B"), *kbias = key("bias"), *kr = key("r"), *ks = key("s");
  need(n >= 1 && n <= 3 && x.dim() == 2, "gptq_lora_fwd: one to three projections of x2d [M, K]");
  const int64_t M = x.size(0);
  fmsa_fwd_proj arr[3] = {};
  std::vector<at::Tensor> outs;
  for (int i = 0; i < n; ++i) {
    PyObject* p = projs[i];
    need(PyDict_Check(p), "gptq_lora_fwd: projections are dicts");
    fmsa_fwd_proj& q = arr[i];
    q.w = weight(item(p, kw));
    outs.push_back(empty({M, q.w.N}, x));
    q.Y = ptr(outs[i]);
    q.ldy = outs[i].stride(0);
    q.r = (int)integer(item(p, kr));
    PyObject* s = item(p, ks);
    q.s = s == Py_None ? 0.f : (float)number(s);
    if (q.r) {
      const at::Tensor U = optional(item(p, kU, false)), B = optional(item(p, kB, false));
      if (U.defined()) {
        need(U.stride(1) == 1, "gptq_lora_fwd: U");
        q.U = ptr(U);
        q.ldu = U.stride(0);
      }
      q.B = ptr(B);
    }
    q.bias = ptr(optional(item(p, kbias, false)));
  }
  at::Tensor h;
  if (mode == FMSA_FWD_SWIGLU) h = at::empty_like(outs[0]);
  const int act = act_enum(x.scalar_type());
  void* st = stream(x);
  const int64_t ldh = h.defined() ? h.stride(0) : 0;
  if (split && fmsa_gptq_lora_fwd_is_few(arr, n, (int)M, mode)) {
    check("fmsa_gptq_lora_fwd_few",
          unlocked([&] { return fmsa_gptq_lora_fwd_few(arr, n, ptr(x), x.stride(0), (int)M, mode, ptr(h), ldh, act, st); }));
  } else {
    const size_t bytes = split ? fmsa_gptq_lora_fwd_workspace(arr, n, (int)M, mode) : 0;
    const at::Tensor ws = bytes ? workspace(bytes, x) : at::Tensor();
    check("fmsa_gptq_lora_fwd_ws", unlocked([&] {
            return fmsa_gptq_lora_fwd_ws(arr, n, ptr(x), x.stride(0), (int)M, mode, ptr(h), ldh, act, ptr(ws), bytes, st);
          }));
  }
  if (mode == FMSA_FWD_SWIGLU) {
    Ref t(PyTuple_New(3));
    PyTuple_SET_ITEM(t.o, 0, wrap(outs[0]));
    PyTuple_SET_ITEM(t.o, 1, wrap(outs[1]));
    PyTuple_SET_ITEM(t.o, 2, wrap(h));
    return t.release();
  }
  return wrap_list(outs);
}

PyObject* gptq_lora_bwd_dx(PyObject* const* a, Py_ssize_t) {  // projs, M, K, mode, e, g, split
  Sequence projs(a[0]);
  const int n = (int)projs.size(), M = (int)integer(a[1]), K = (int)integer(a[2]), mode = (int)integer(a[3]);
  const at::Tensor e = optional(a[4]), g = optional(a[5]);
  const bool split = truth(a[6]);
  static PyObject *kw = key("w"), *knsz = key("nsz"), *kdY = key("dY"), *kT = key("T"), *kAt = key("At"), *kms = key("mask_src"), *kr = key("r"),
                  *ks = key("s"), *kqt = key("qweight_t"), *ksf = key("scale_f32"), *knz = key("negzp_f16");
  need(n >= 1 && n <= 3, "gptq_lora_bwd_dx: one to three projections");
  fmsa_bwd_proj arr[3] = {};
  at::Tensor ref;
  for (int i = 0; i < n; ++i) {
    PyObject* p = projs[i];
    need(PyDict_Check(p), "gptq_lora_bwd_dx: projections are dicts");
    fmsa_bwd_proj& q = arr[i];
    const at::Tensor& dy = tensor(item(p, kdY));
    if (i == 0) ref = dy;
    need(dy.dim() == 2 && dy.stride(1) == 1, "gptq_lora_bwd_dx: dY");
    q.w = weight(item(p, kw));
    q.nsz = (const float*)ptr(optional(item(p, knsz)));
    q.dY = ptr(dy);
    q.lddy = dy.stride(0);
    q.r = (int)integer(item(p, kr));
    PyObject* s = item(p, ks);
    q.s = s == Py_None ? 0.f : (float)number(s);
    if (q.r) {
      const at::Tensor T = optional(item(p, kT, false));
      if (T.defined()) {
        need(T.stride(1) == 1, "gptq_lora_bwd_dx: T");
        q.T = ptr(T);
        q.ldt = T.stride(0);
      }
      q.At = ptr(optional(item(p, kAt, false)));
    }
    const at::Tensor ms = optional(item(p, kms, false));
    q.mask_src = ptr(ms);
    q.ldmask = ms.defined() ? ms.stride(0) : 0;
    q.qweight_t = (const int32_t*)ptr(optional(item(p, kqt, false)));
    q.scale_f32 = (const float*)ptr(optional(item(p, ksf, false)));
    q.negzp_f16 = static_cast<decltype(q.negzp_f16)>(ptr(optional(item(p, knz, false))));
  }
  const int act = act_enum(ref.scalar_type());
  void* st = stream(ref);
  const size_t bytes = split ? fmsa_gptq_lora_bwd_dx_workspace(arr, n, M, act) : 0;
  const at::Tensor ws = bytes ? workspace(bytes, ref) : at::Tensor();
  if (mode == FMSA_BWD_SWIGLU) {
    need(e.defined() && g.defined(), "gptq_lora_bwd_dx: e, g");
    at::Tensor h = at::empty_like(e);
    check("fmsa_gptq_lora_bwd_dx_ws", unlocked([&] {
            return fmsa_gptq_lora_bwd_dx_ws(arr, n, M, mode, nullptr, 0, ptr(e), ptr(g), ptr(h), e.stride(0), act, ptr(ws), bytes, st);
          }));
    return wrap(h);
  }
  at::Tensor dx = empty({M, K}, ref);
  check("fmsa_gptq_lora_bwd_dx_ws", unlocked([&] {
          return fmsa_gptq_lora_bwd_dx_ws(arr, n, M, mode, ptr(dx), dx.stride(0), nullptr, nullptr, nullptr, 0, act, ptr(ws), bytes, st);
        }));
  return wrap(dx);
}

PyObject* lora_few(PyObject* const* a, Py_ssize_t) {  // x2d, ((w, A, B, bias, s), ..), mode
  const at::Tensor& x = tensor(a[0]);
  Sequence projs(a[1]);
  const int n = (int)projs.size(), mode = (int)integer(a[2]);
  need(n >= 1 && n <= 3 && x.dim() == 2 && x.stride(1) == 1, "lora_few: one to three projections of x2d [M, K]");
  const int M = (int)x.size(0);
  bool adapters_on_gpu = true;
  fmsa_few_proj arr[3] = {};
  for (int i = 0; i < n; ++i) {
    Sequence p(projs[i]);
    need(p.size() == 5, "lora_few: (w, A, B, bias, s)");
    fmsa_few_proj& q = arr[i];
    q.w = weight(p[0]);
    need(x.size(1) == q.w.K, "lora_few: x2d, w");
    q.ldy = q.w.N;
    const at::Tensor bias = optional(p[3]);
    need(!bias.defined() || (bias.numel() == q.w.N && bias.is_contiguous() && bias.scalar_type() == x.scalar_type()), "lora_few: bias");
    q.bias = ptr(bias);
    const at::Tensor A = optional(p[1]);
    if (A.defined()) {
      const at::Tensor& B = tensor(p[2]);
      need(A.dim() == 2 && B.dim() == 2 && A.size(1) == q.w.K && B.size(0) == q.w.N && B.size(1) == A.size(0) && A.is_contiguous() &&
               B.is_contiguous() && A.scalar_type() == B.scalar_type(),
           "lora_few: A, B");
      adapters_on_gpu = adapters_on_gpu && A.is_cuda() && B.is_cuda();
      q.A = ptr(A);
      q.B = ptr(B);
      q.r = (int)A.size(0);
      q.s = (float)number(p[4]);
      q.param_dtype = dtype_enum(A.scalar_type());
    }
  }
  if (!fmsa_lora_few_is_few(arr, n, M, mode)) Py_RETURN_NONE;
  on_gpu(adapters_on_gpu);
  at::Tensor h;
  std::vector<at::Tensor> outs;
  if (mode == FMSA_FWD_SWIGLU)
    h = empty({M, arr[0].w.N}, x);
  else
    for (int i = 0; i < n; ++i) {
      outs.push_back(empty({M, arr[i].w.N}, x));
      arr[i].Y = ptr(outs[i]);
    }
  const int act = act_enum(x.scalar_type());
  void* st = stream(x);
  const size_t bytes = fmsa_lora_few_workspace(arr, n, M);
  const at::Tensor ws = bytes ? workspace(bytes, x) : at::Tensor();
  check("fmsa_lora_few_fwd", unlocked([&] {
          return fmsa_lora_few_fwd(arr, n, ptr(x), x.stride(0), M, mode, ptr(h), h.defined() ? h.stride(0) : 0, act, ptr(ws), bytes, st);
        }));
  return mode == FMSA_FWD_SWIGLU ? wrap(h) : wrap_list(outs);
}

// ---- adapted projections, read from their modules ---------------------------------------------------------------------------
// What get_lora_parameters, prepare and lora_few_ok of the Python side find, in a third of their time: a pass over a layer without a
// graph asks for seven projections, 50 of its 140 us on the host.  Nothing here raises and nothing is decided that they would decide
// otherwise: whatever is not the ordinary case (`false`, None) is left to them.
struct Obj {  // owned reference or null
  PyObject* o;
  explicit Obj(PyObject* p = nullptr) : o(p) {}
  Obj(Obj&& other) noexcept : o(other.o) { other.o = nullptr; }
  Obj& operator=(Obj&& other) noexcept {
    std::swap(o, other.o);
    return *this;
  }
  ~Obj() { Py_XDECREF(o); }
  Obj(const Obj&) = delete;
  Obj& operator=(const Obj&) = delete;
  explicit operator bool() const { return o != nullptr; }
};

Obj borrowed(PyObject* o) {
  Py_XINCREF(o);
  return Obj(o);
}

PyObject *g_identity = nullptr, *g_module_dict = nullptr, *g_parameter = nullptr;  // torch.nn.Identity, ModuleDict, Parameter

Obj attribute(PyObject* o, PyObject* name) {
  Obj v(PyObject_GetAttr(o, name));
  if (!v) PyErr_Clear();
  return v;
}

Obj item_of(PyObject* container, PyObject* k) {
  Obj v(PyDict_CheckExact(container) ? (Py_XINCREF(PyDict_GetItemWithError(container, k)), PyDict_GetItemWithError(container, k))
                                     : PyObject_GetItem(container, k));
  if (!v) PyErr_Clear();
  return v;
}

// utils.member: the dictionary `kind` of a module first, then getattr
Obj member(PyObject* module, PyObject* kind, PyObject* name) {
  PyObject** own = _PyObject_GetDictPtr(module);
  if (own && *own && PyDict_CheckExact(*own) && !PyDict_GetItemWithError(*own, name)) {
    PyObject* held = PyDict_GetItemWithError(*own, kind);
    if (held && held != Py_None) {
      const int has = PySequence_Contains(held, name);
      if (has > 0) return item_of(held, name);
      if (has < 0) PyErr_Clear();
    }
  }
  PyErr_Clear();
  return attribute(module, name);
}

// getattr(module, name, None) of what modules keep as a buffer, a parameter or an attribute
Obj held(PyObject* module, PyObject* name) {
  static PyObject *buffers = key("_buffers"), *parameters = key("_parameters");
  if (!_PyType_Lookup(Py_TYPE(module), name))
    for (PyObject* kind : {buffers, parameters}) {
      PyObject** own = _PyObject_GetDictPtr(module);
      if (!own || !*own || !PyDict_CheckExact(*own) || PyDict_GetItemWithError(*own, name)) break;
      PyObject* in = PyDict_GetItemWithError(*own, kind);
      if (in && PyDict_CheckExact(in) && PyDict_GetItemWithError(in, name)) return item_of(in, name);
    }
  PyErr_Clear();
  Obj v = attribute(module, name);
  return v ? std::move(v) : borrowed(Py_None);
}

// container[active] of a ModuleDict, or of whatever stands in for one
Obj active_of(PyObject* container, PyObject* active) {
  static PyObject* modules = key("_modules");
  if (reinterpret_cast<PyObject*>(Py_TYPE(container)) == g_module_dict) {
    PyObject** own = _PyObject_GetDictPtr(container);
    PyObject* in = own && *own ? PyDict_GetItemWithError(*own, modules) : nullptr;
    if (in && PyDict_CheckExact(in)) return item_of(in, active);
  }
  return item_of(container, active);
}

// what was set on a tensor (borrowed); none of the names is one of the class
PyObject* mark(PyObject* t, PyObject* name) {
  PyObject** own = _PyObject_GetDictPtr(t);
  PyObject* v = own && *own ? PyDict_GetItemWithError(*own, name) : nullptr;
  PyErr_Clear();
  return v;
}

bool plain(PyObject* o) { return o && THPVariable_CheckExact(o) && !THPVariable_Unpack(o).is_inference(); }

bool equals(PyObject* number, int64_t v) {
  const long long n = PyLong_Check(number) ? PyLong_AsLongLong(number) : -1;
  if (n == -1 && PyErr_Occurred()) PyErr_Clear();
  return PyLong_Check(number) && n == v;
}

// ... or a parameter of a class that stands for its data as torch.nn.Parameter does (bitsandbytes' Params4bit)
bool plain_weight(PyObject* o) {
  static PyObject* function = key("__torch_function__");
  if (plain(o)) return true;
  if (!o || !THPVariable_Check(o) || THPVariable_Unpack(o).is_inference()) return false;
  PyTypeObject* parameter = reinterpret_cast<PyTypeObject*>(g_parameter);
  return PyType_IsSubtype(Py_TYPE(o), parameter) && _PyType_Lookup(Py_TYPE(o), function) == _PyType_Lookup(parameter, function);
}

int64_t address(const at::Tensor& t) { return reinterpret_cast<int64_t>(t.data_ptr()); }

// gptq_prepared.prepare's cached weight where its key still holds (borrowed; null: ask there)
PyObject* prepared_gptq(PyObject* qweight, PyObject* scales, PyObject* qzeros, PyObject* g_idx) {
  static PyObject *kprep = key("_fmsa_prepared"), *koff = key("offset");
  if (!plain(qweight) || !plain(scales) || !plain(qzeros) || !plain(g_idx)) return nullptr;
  PyObject* cached = mark(qweight, kprep);
  if (!cached || !PyTuple_CheckExact(cached) || PyTuple_GET_SIZE(cached) != 2) return nullptr;
  PyObject* k = PyTuple_GET_ITEM(cached, 0);
  if (!PyTuple_CheckExact(k) || PyTuple_GET_SIZE(k) != 9) return nullptr;
  PyObject* off = mark(qzeros, koff);
  const long offset = off && off != Py_None ? (PyLong_CheckExact(off) ? PyLong_AsLong(off) : -1) : 0;
  const at::Tensor &q = THPVariable_Unpack(qweight), &s = THPVariable_Unpack(scales), &z = THPVariable_Unpack(qzeros), &g = THPVariable_Unpack(g_idx);
  const int64_t now[9] = {address(q), address(s), address(z), address(g), (int64_t)g._version(), (int64_t)q._version(), (int64_t)s._version(),
                          (int64_t)z._version(), offset};
  for (int i = 0; i < 9; ++i)
    if (!equals(PyTuple_GET_ITEM(k, i), now[i])) return nullptr;
  return PyTuple_GET_ITEM(cached, 1);
}

// nf4_prepared.prepare's, likewise
PyObject* prepared_nf4(PyObject* W, PyObject* state) {
  static PyObject *kprep = key("_fmsa_prepared"), *kabsmax = key("absmax"), *koff = key("offset"), *kshape = key("shape"), *kblock = key("blocksize");
  if (!plain_weight(W)) return nullptr;
  PyObject* cached = mark(W, kprep);
  if (!cached || !PyTuple_CheckExact(cached) || PyTuple_GET_SIZE(cached) != 2) return nullptr;
  PyObject* k = PyTuple_GET_ITEM(cached, 0);
  if (!PyTuple_CheckExact(k) || PyTuple_GET_SIZE(k) != 7) return nullptr;
  const Obj absmax = attribute(state, kabsmax), off = attribute(state, koff), shape = attribute(state, kshape), block = attribute(state, kblock);
  if (!absmax || !plain(absmax.o) || !off || !plain(off.o) || !shape || !block) return nullptr;
  PyObject* ok = PyTuple_GET_ITEM(k, 4);
  const at::Tensor &w = THPVariable_Unpack(W), &a = THPVariable_Unpack(absmax.o), &o = THPVariable_Unpack(off.o);
  // W.data, whose version counter is its own, for a parameter
  const int64_t version = Py_TYPE(W) == reinterpret_cast<PyTypeObject*>(THPVariableClass) ? (int64_t)w._version() : 0;
  if (!equals(PyTuple_GET_ITEM(k, 0), address(w)) || !equals(PyTuple_GET_ITEM(k, 1), version) || !equals(PyTuple_GET_ITEM(k, 2), address(a)) ||
      !equals(PyTuple_GET_ITEM(k, 3), (int64_t)a._version()) || !PyTuple_CheckExact(ok) || PyTuple_GET_SIZE(ok) != 2 ||
      !equals(PyTuple_GET_ITEM(ok, 0), address(o)) || !equals(PyTuple_GET_ITEM(ok, 1), (int64_t)o._version()) || !PyLong_Check(block.o) ||
      PyObject_RichCompareBool(PyTuple_GET_ITEM(k, 6), block.o, Py_EQ) != 1)
    return nullptr;
  PyObject* kept = PyTuple_GET_ITEM(k, 5);
  const bool same = PyTuple_Check(shape.o) && PyTuple_Check(kept) && PyObject_RichCompareBool(kept, shape.o, Py_EQ) == 1;
  PyErr_Clear();
  return same ? PyTuple_GET_ITEM(cached, 1) : nullptr;
}

struct Adapted {  // an adapted projection whose adapter is active
  Obj parts[5];   // GPTQ: qweight, scales, qzeros, g_idx, bits; NF4: W, quant state
  Obj bias, A, B, scaling, dropout;
};

bool read_adapted(PyObject* proj, bool nf4, Adapted& p) {
  static PyObject *kmod = key("_modules"), *kbuf = key("_buffers"), *kpar = key("_parameters"), *kbase = key("base_layer"),
                  *kdisable = key("disable_adapters"), *kmerged = key("merged"), *kactives = key("active_adapters"), *kactive = key("active_adapter"),
                  *kA = key("lora_A"), *kB = key("lora_B"), *kdrop = key("lora_dropout"), *kweight = key("weight"), *kscaling = key("scaling"),
                  *kbias = key("bias"), *knz = key("_fmsa_nonzero"), *kmodule = key("__module__"), *kbits = key("bits"), *kstate = key("quant_state");
  static PyObject* kq[4] = {key("qweight"), key("scales"), key("qzeros"), key("g_idx")};
  const Obj disabled = attribute(proj, kdisable), merged = attribute(proj, kmerged);
  if (!disabled || !merged || PyObject_IsTrue(disabled.o) != 0 || PyObject_IsTrue(merged.o) != 0) return PyErr_Clear(), false;
  Obj base = member(proj, kmod, kbase);
  if (!base) return false;
  if (nf4) {
    p.parts[0] = member(base.o, kpar, kweight);
    if (!p.parts[0] || !plain_weight(p.parts[0].o)) return false;
    PyObject* state = mark(p.parts[0].o, kstate);
    if (!state || state == Py_None || PyList_Check(state) || PyTuple_Check(state)) return false;
    p.parts[1] = borrowed(state);
    p.bias = held(base.o, kbias);
  } else {
    const Obj where = attribute(base.o, kmodule);
    if (!where || !PyUnicode_Check(where.o)) return false;
    const char* text = PyUnicode_AsUTF8(where.o);
    if (!text || std::strncmp(text, "auto_gptq", 9) == 0) return PyErr_Clear(), false;  // (those get their zero points' offset there)
    Obj inner = member(base.o, kmod, kbase);
    if (inner) base = std::move(inner);
    for (int i = 0; i < 4; ++i)
      if (!(p.parts[i] = member(base.o, kbuf, kq[i]))) return false;
    if (!(p.parts[4] = attribute(base.o, kbits))) return false;
    p.bias = held(base.o, kbias);
    if (p.bias.o != Py_None) {  // dropped where it is all zeros, as found once for its version
      PyObject* known = plain(p.bias.o) ? mark(p.bias.o, knz) : nullptr;
      if (!known || !PyTuple_CheckExact(known) || PyTuple_GET_SIZE(known) != 2 ||
          !equals(PyTuple_GET_ITEM(known, 0), (int64_t)THPVariable_Unpack(p.bias.o)._version()))
        return false;
      if (PyTuple_GET_ITEM(known, 1) != Py_True) p.bias = borrowed(Py_None);
    }
  }
  Obj active = attribute(proj, kactives);
  if (active) {
    active = Obj(PySequence_GetItem(active.o, 0));
    if (!active) return PyErr_Clear(), false;
  } else if (!(active = attribute(proj, kactive))) {
    return false;
  }
  const Obj la = member(proj, kmod, kA), lb = member(proj, kmod, kB), scalings = attribute(proj, kscaling), drops = member(proj, kmod, kdrop);
  if (!la || !lb || !scalings) return false;
  const Obj ma = active_of(la.o, active.o), mb = active_of(lb.o, active.o);
  if (!ma || !mb) return false;
  p.A = member(ma.o, kpar, kweight);
  p.B = member(mb.o, kpar, kweight);
  p.scaling = item_of(scalings.o, active.o);
  p.dropout = !drops || drops.o == Py_None ? borrowed(Py_None) : active_of(drops.o, active.o);
  return p.A && p.B && p.scaling && p.dropout;
}

PyObject* gptq_operands(PyObject* const* a, Py_ssize_t) {  // projection
  Adapted p;
  if (!read_adapted(a[0], false, p)) Py_RETURN_NONE;
  Obj* all[10] = {&p.parts[0], &p.parts[1], &p.parts[2], &p.parts[3], &p.parts[4], &p.bias, &p.A, &p.B, &p.scaling, &p.dropout};
  Ref t(PyTuple_New(10));
  for (int i = 0; i < 10; ++i) {
    PyTuple_SET_ITEM(t.o, i, all[i]->o);
    all[i]->o = nullptr;
  }
  return t.release();
}

PyObject* gptq_prepared(PyObject* const* a, Py_ssize_t) {  // qweight, scales, qzeros, g_idx
  PyObject* w = prepared_gptq(a[0], a[1], a[2], a[3]);
  if (!w) Py_RETURN_NONE;
  Py_INCREF(w);
  return w;
}

// One projection of few tokens: what _few_tokens asks of it, and its operands
bool few_operands(PyObject* proj, bool nf4, const at::Tensor& x, PyObject* dtype, bool& interleaved, Adapted& p, Obj& prepared, fmsa_few_proj& q) {
  static PyObject *kstruct = key("struct"), *kperm = key("perm"), *kok = key("interleaved_ok");
  if (!read_adapted(proj, nf4, p)) return false;
  prepared = borrowed(nf4 ? prepared_nf4(p.parts[0].o, p.parts[1].o) : prepared_gptq(p.parts[0].o, p.parts[1].o, p.parts[2].o, p.parts[3].o));
  if (!prepared) return false;
  const Obj perm = attribute(prepared.o, kperm), view = attribute(prepared.o, kstruct);
  if (!perm || perm.o != Py_None || !view || !plain(p.A.o) || !plain(p.B.o)) return false;
  if (p.dropout.o != Py_None && reinterpret_cast<PyObject*>(Py_TYPE(p.dropout.o)) != g_identity) return false;
  q.w = weight(view.o);
  if (nf4 || x.scalar_type() != at::kHalf) {
    interleaved = false;
  } else if (interleaved) {
    const Obj ok(PyObject_CallMethodObjArgs(prepared.o, kok, dtype, nullptr));
    if (!ok) return PyErr_Clear(), false;
    interleaved = ok.o == Py_True;
  }
  const at::Tensor &A = THPVariable_Unpack(p.A.o), &B = THPVariable_Unpack(p.B.o);
  const at::ScalarType t = A.scalar_type();
  if (q.w.group_size % 64 || x.size(-1) != q.w.K || A.dim() != 2 || B.dim() != 2 || B.scalar_type() != t || (t != at::kFloat && t != x.scalar_type()) ||
      !A.is_cuda() || !B.is_cuda() || !A.is_contiguous() || !B.is_contiguous() || A.size(0) % 8 || A.size(0) <= 0 || A.size(0) > 128 ||
      A.size(1) != q.w.K || B.size(0) != q.w.N || B.size(1) != A.size(0) || (address(A) | address(B)) % 16)
    return false;
  if (p.bias.o != Py_None) {
    if (!plain(p.bias.o)) return false;
    const at::Tensor& b = THPVariable_Unpack(p.bias.o);
    if (b.scalar_type() != x.scalar_type() || b.numel() != q.w.N || !b.is_contiguous() || !b.is_cuda()) return false;
    q.bias = ptr(b);
  }
  if (!PyFloat_Check(p.scaling.o) && !PyLong_Check(p.scaling.o)) return false;
  q.A = ptr(A);
  q.B = ptr(B);
  q.r = (int)A.size(0);
  q.s = (float)number(p.scaling.o);
  q.param_dtype = dtype_enum(t);
  q.ldy = q.w.N;
  return true;
}

struct FewCall {
  Adapted parts[3];
  Obj prepared[3];
  fmsa_few_proj arr[3] = {};
  int n = 0;
  bool read(PyObject* const* projs, int count, bool nf4, const at::Tensor& x, PyObject* dtype) {
    static PyObject* kil = key("struct_interleaved");
    bool interleaved = true;
    n = count;
    for (int i = 0; i < n; ++i)
      if (!few_operands(projs[i], nf4, x, dtype, interleaved, parts[i], prepared[i], arr[i])) return false;
    if (interleaved)
      for (int i = 0; i < n; ++i) {
        const Obj view = attribute(prepared[i].o, kil);
        if (!view) return false;
        arr[i].w = weight(view.o);
      }
    return true;
  }
  // outputs [.., N] (SwiGLU: h is written)
  std::vector<at::Tensor> run(const at::Tensor& x, int M, int mode, const at::Tensor& h = at::Tensor()) {
    auto sizes = x.sizes().vec();
    std::vector<at::Tensor> outs;
    for (int i = 0; i < n && mode != FMSA_FWD_SWIGLU; ++i) {
      sizes.back() = arr[i].w.N;
      outs.push_back(at::empty(sizes, x.options()));
      arr[i].Y = ptr(outs[i]);
    }
    const int act = act_enum(x.scalar_type());
    void* st = stream(x);
    const size_t bytes = fmsa_lora_few_workspace(arr, n, M);
    const at::Tensor ws = bytes ? workspace(bytes, x) : at::Tensor();
    check("fmsa_lora_few_fwd", unlocked([&] {
            return fmsa_lora_few_fwd(arr, n, ptr(x), x.size(-1), M, mode, ptr(h), h.defined() ? arr[0].w.N : 0, act, ptr(ws), bytes, st);
          }));
    return outs;
  }
};

// Tokens of an input that the calls below take as it is, else 0
int few_rows(PyObject* X, long most) {
  if (!plain(X) && !(THPVariable_CheckExact(X) && THPVariable_Unpack(X).is_inference())) return 0;
  const at::Tensor& x = THPVariable_Unpack(X);
  if (x.dim() < 1 || x.numel() == 0 || !x.is_cuda() || !x.is_contiguous() || (x.scalar_type() != at::kHalf && x.scalar_type() != at::kBFloat16)) return 0;
  const int64_t M = x.numel() / x.size(-1);
  return M <= most ? (int)M : 0;
}

// X, projections, whether they are NF4, its dtype, most tokens: their outputs where no graph is built and the kernel for few tokens
// reads everything as it lies; else None
PyObject* few_linear(PyObject* const* a, Py_ssize_t) {
  const int M = few_rows(a[0], integer(a[4]));
  if (!M) Py_RETURN_NONE;
  const at::Tensor& x = THPVariable_Unpack(a[0]);
  Sequence projs(a[1]);
  need(projs.size() >= 1 && projs.size() <= 3, "few_linear: one to three projections");
  PyObject* ps[3];
  for (Py_ssize_t i = 0; i < projs.size(); ++i) ps[i] = projs[i];
  FewCall call;
  if (!call.read(ps, (int)projs.size(), truth(a[2]), x, a[3]) || !fmsa_lora_few_is_few(call.arr, call.n, M, FMSA_FWD_LINEAR)) Py_RETURN_NONE;
  const auto outs = call.run(x, M, FMSA_FWD_LINEAR);
  Ref t(PyTuple_New((Py_ssize_t)outs.size()));
  for (size_t i = 0; i < outs.size(); ++i) PyTuple_SET_ITEM(t.o, (Py_ssize_t)i, wrap(outs[i]));
  return t.release();
}

// X, (gate, up, down), NF4, dtype, most tokens: the output of the SwiGLU MLP, likewise
PyObject* few_mlp(PyObject* const* a, Py_ssize_t) {
  const int M = few_rows(a[0], integer(a[4]));
  if (!M) Py_RETURN_NONE;
  const at::Tensor& x = THPVariable_Unpack(a[0]);
  Sequence projs(a[1]);
  need(projs.size() == 3, "few_mlp: gate, up, down");
  PyObject* const ps[3] = {projs[0], projs[1], projs[2]};
  const bool nf4 = truth(a[2]);
  FewCall first, second;
  if (!first.read(ps, 2, nf4, x, a[3]) || first.arr[0].w.N != first.arr[1].w.N || !fmsa_lora_few_is_few(first.arr, 2, M, FMSA_FWD_SWIGLU)) Py_RETURN_NONE;
  // the second launch is known to follow before the first goes out
  auto sizes = x.sizes().vec();
  sizes.back() = first.arr[0].w.N;
  const at::Tensor h = at::empty(sizes, x.options());
  if (!second.read(ps + 2, 1, nf4, h, a[3]) || !fmsa_lora_few_is_few(second.arr, 1, M, FMSA_FWD_LINEAR)) Py_RETURN_NONE;
  first.run(x, M, FMSA_FWD_SWIGLU, h);
  return wrap(second.run(h, M, FMSA_FWD_LINEAR)[0]);
}

// X, weight, eps, gemma: the normalised X where no graph is built and both lie as the kernel reads them, else None
PyObject* rms_layernorm(PyObject* const* a, Py_ssize_t) {
  if (!THPVariable_CheckExact(a[0]) || !THPVariable_CheckExact(a[1])) Py_RETURN_NONE;
  const at::Tensor &x = THPVariable_Unpack(a[0]), &w = THPVariable_Unpack(a[1]);
  if (x.dim() < 1 || x.numel() == 0 || !x.is_cuda() || !w.is_cuda() || !x.is_contiguous() || !w.is_contiguous() || w.numel() != x.size(-1)) Py_RETURN_NONE;
  for (at::ScalarType t : {x.scalar_type(), w.scalar_type()})
    if (t != at::kHalf && t != at::kBFloat16 && t != at::kFloat) Py_RETURN_NONE;
  const float eps = (float)number(a[2]);
  const int gemma = truth(a[3]), C = (int)x.size(-1), M = (int)(x.numel() / C);
  at::Tensor y = at::empty(x.sizes(), x.options()), r = empty({M}, x, at::kFloat);
  void* st = stream(x);
  check("fmsa_rms_layernorm_fwd", unlocked([&] {
          return fmsa_rms_layernorm_fwd(ptr(x), C, ptr(w), M, C, eps, gemma, dtype_enum(x.scalar_type()), dtype_enum(w.scalar_type()), ptr(y), C,
                                        (float*)ptr(r), st);
        }));
  return wrap(y);
}

PyObject* install_types(PyObject* const* a, Py_ssize_t) {  // torch.nn.Identity, torch.nn.ModuleDict, torch.nn.Parameter
  for (int i = 0; i < 3; ++i) Py_INCREF(a[i]);
  g_identity = a[0];
  g_module_dict = a[1];
  g_parameter = a[2];
  Py_RETURN_NONE;
}

// ---- norm and rotary embedding --------------------------------------------------------------------------------------------
PyObject* rms_layernorm_fwd(PyObject* const* a, Py_ssize_t) {  // x2d, weight, eps, gemma
  const at::Tensor &x = tensor(a[0]), &w = tensor(a[1]);
  on_gpu(x.is_cuda() && w.is_cuda());
  need(x.dim() == 2 && x.stride(1) == 1 && w.is_contiguous() && w.numel() == x.size(1), "rms_layernorm_fwd: x2d, weight");
  const float eps = (float)number(a[2]);
  const int gemma = truth(a[3]), M = (int)x.size(0), C = (int)x.size(1);
  at::Tensor y = empty({M, C}, x), r = empty({M}, x, at::kFloat);
  void* st = stream(x);
  const int xd = dtype_enum(x.scalar_type()), wd = dtype_enum(w.scalar_type());
  check("fmsa_rms_layernorm_fwd", unlocked([&] {
          return fmsa_rms_layernorm_fwd(ptr(x), x.stride(0), ptr(w), M, C, eps, gemma, xd, wd, ptr(y), y.stride(0), (float*)ptr(r), st);
        }));
  Ref t(PyTuple_New(2));
  PyTuple_SET_ITEM(t.o, 0, wrap(y));
  PyTuple_SET_ITEM(t.o, 1, wrap(r));
  return t.release();
}

PyObject* rms_layernorm_bwd(PyObject* const* a, Py_ssize_t) {  // dy2d, x2d, weight, r, gemma
  const at::Tensor &dy = tensor(a[0]), &x = tensor(a[1]), &w = tensor(a[2]), &r = tensor(a[3]);
  need(dy.dim() == 2 && dy.sizes() == x.sizes() && dy.stride(1) == 1 && x.stride(1) == 1 && dy.scalar_type() == x.scalar_type(), "rms_layernorm_bwd: dy2d, x2d");
  const int gemma = truth(a[4]), M = (int)x.size(0), C = (int)x.size(1);
  void* st = stream(x);
  const int xd = dtype_enum(x.scalar_type()), wd = dtype_enum(w.scalar_type());
  check("fmsa_rms_layernorm_bwd", unlocked([&] {
          return fmsa_rms_layernorm_bwd(ptr(dy), dy.stride(0), ptr(x), x.stride(0), ptr(w), (const float*)ptr(r), M, C, gemma, xd, wd, st);
        }));
  Py_INCREF(a[0]);
  return a[0];
}

PyObject* rope_embedding_(PyObject* const* a, Py_ssize_t) {  // q2d, cos2d, sin2d, n_heads, head_dim, backward
  const at::Tensor &q = tensor(a[0]), &c = tensor(a[1]), &s = tensor(a[2]);
  on_gpu(q.is_cuda() && c.is_cuda() && s.is_cuda());
  need(q.stride(1) == 1 && c.stride(1) == 1 && c.strides() == s.strides() && c.scalar_type() == s.scalar_type(), "rope_embedding_: q2d, cos2d, sin2d");
  const int heads = (int)integer(a[3]), hd = (int)integer(a[4]), bwd = truth(a[5]);
  void* st = stream(q);
  const int qd = dtype_enum(q.scalar_type()), cd = dtype_enum(c.scalar_type());
  check("fmsa_rope_embedding", unlocked([&] {
          return fmsa_rope_embedding(ptr(q), q.stride(0), ptr(c), ptr(s), c.stride(0), (int)q.size(0), heads, hd, (int)c.size(0), bwd, qd, cd, st);
        }));
  Py_INCREF(a[0]);
  return a[0];
}

PyObject* rope_embedding_pair_(PyObject* const* a, Py_ssize_t) {  // q2d, k2d, cos2d, sin2d, head_dim
  const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]), &c = tensor(a[2]), &s = tensor(a[3]);
  on_gpu(q.is_cuda() && k.is_cuda() && c.is_cuda() && s.is_cuda());
  const int hd = (int)integer(a[4]);
  need(q.dim() == 2 && k.dim() == 2 && q.size(0) == k.size(0) && q.stride(1) == 1 && k.stride(1) == 1 && q.scalar_type() == k.scalar_type() &&
           q.device() == k.device() && hd > 0 && q.size(1) % hd == 0 && k.size(1) % hd == 0,
       "rope_embedding_pair_: q2d, k2d");
  need(c.stride(1) == 1 && c.strides() == s.strides() && c.scalar_type() == s.scalar_type(), "rope_embedding_pair_: cos2d, sin2d");
  void* st = stream(q);
  const int qd = dtype_enum(q.scalar_type()), cd = dtype_enum(c.scalar_type());
  check("fmsa_rope_embedding_pair", unlocked([&] {
          return fmsa_rope_embedding_pair(ptr(q), q.stride(0), (int)(q.size(1) / hd), ptr(k), k.stride(0), (int)(k.size(1) / hd), ptr(c), ptr(s),
                                          c.stride(0), (int)q.size(0), hd, (int)c.size(0), 0, qd, cd, st);
        }));
  Py_RETURN_NONE;
}

PyObject* rope_embedding_strided(PyObject* const* a, Py_ssize_t) {  // q4d, cos2d, sin2d, backward
  const at::Tensor &q = tensor(a[0]), &c = tensor(a[1]), &s = tensor(a[2]);
  on_gpu(q.is_cuda() && c.is_cuda() && s.is_cuda());
  need(q.dim() == 4 && q.stride(3) == 1 && c.stride(1) == 1 && c.strides() == s.strides() && c.scalar_type() == s.scalar_type(),
       "rope_embedding_strided: q4d, cos2d, sin2d");
  const int bwd = truth(a[3]), b = (int)q.size(0), t = (int)q.size(1), h = (int)q.size(2), d = (int)q.size(3);
  at::Tensor out = empty({(int64_t)b * t, (int64_t)h * d}, q);
  void* st = stream(q);
  const int qd = dtype_enum(q.scalar_type()), cd = dtype_enum(c.scalar_type());
  check("fmsa_rope_embedding_strided", unlocked([&] {
          return fmsa_rope_embedding_strided(ptr(q), q.stride(0), q.stride(1), q.stride(2), ptr(out), ptr(c), ptr(s), c.stride(0), b, t, h, d,
                                             (int)c.size(0), bwd, qd, cd, st);
        }));
  return wrap(out);
}

PyObject* install(PyObject* const* a, Py_ssize_t) {  // FmsaError
  Py_INCREF(a[0]);
  Py_XDECREF(g_fmsa_error);
  g_fmsa_error = a[0];
  return PyLong_FromLong(FMSA_ABI_VERSION);  // of the structs that were compiled in, whatever library is loaded
}

#define ENTRY(name, n) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<name, n>)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {ENTRY(lora_down, 3),           ENTRY(lora_down_batch, 2),   ENTRY(lora_grad_batch, 2),
                           ENTRY(lora_pack_batch, 3),     ENTRY(gptq_lora_fwd, 4),     ENTRY(gptq_lora_bwd_dx, 7),
                           ENTRY(lora_few, 3),            ENTRY(rms_layernorm_fwd, 4), ENTRY(rms_layernorm_bwd, 5),
                           ENTRY(rope_embedding_, 6),     ENTRY(rope_embedding_pair_, 5),
                           ENTRY(rope_embedding_strided, 4), ENTRY(install, 1),
                           ENTRY(install_types, 3),       ENTRY(gptq_operands, 1),     ENTRY(gptq_prepared, 4),
                           ENTRY(few_linear, 5),          ENTRY(few_mlp, 5),           ENTRY(rms_layernorm, 4),
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_fmsa_calls", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fmsa_calls() { return PyModule_Create(&g_module); }

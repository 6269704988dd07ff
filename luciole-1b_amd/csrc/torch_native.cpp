// The launch layer's common case in C++: a Python extension module
// (SSA/_ssa_native.so) that checks the tensors of a call, allocates its outputs
// and workspaces and calls the C ABI, in one step from Python.
//
// A call the kernels can take as it is costs a few microseconds here; the same
// steps through Python attributes and ctypes structures took 25 (forward) to
// 130 us (backward), more than the kernels of a small problem.  Everything else
// returns None and takes the Python path of SSA/ssa_hip_kernel.py, which
// copies, pads, converts or raises: wrong shapes, other dtypes or devices,
// layouts the kernels cannot address, tensor subclasses and functorch wrappers,
// a device other than the current one.  The functions hold no state besides
// the addresses of the C ABI.
//
// A nonzero library status comes back as an int (the Python side raises it).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/core/CachingDeviceAllocator.h>
#include <c10/core/DispatchKeySet.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/headeronly/version.h>

#include <cstring>

#include "../../include/ssa_mi355x.h"

namespace {

struct Abi {
  decltype(&ssa_fwd) fwd;
  decltype(&ssa_bwd) bwd;
  decltype(&ssa_varlen_fwd) varlen_fwd;
  decltype(&ssa_varlen_bwd) varlen_bwd;
  decltype(&ssa_decode) decode;
  decltype(&ssa_bwd_partials_count) partials_count;
  decltype(&ssa_bwd_ds_workspace_bytes) ds_bytes;
  decltype(&ssa_varlen_bwd_ds_workspace_bytes) varlen_ds_bytes;
  decltype(&ssa_decode_workspace_bytes) decode_bytes;
};
Abi abi;

constexpr int64_t kMaxRowStride = int64_t{1} << 24;

// A tensor argument, or nullptr for anything but a plain one: a torch.Tensor or
// Parameter itself, strided, on GPU `dev`, with no wrapper or lazy key.
const at::Tensor* plain(PyObject* o, int dev) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  static const c10::DispatchKeySet odd({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                        c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                        c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                        c10::DispatchKey::ZeroTensor});
  if (!t.defined() || t.layout() != at::kStrided || t.device().type() != c10::DeviceType::CUDA ||
      t.device().index() != dev || t.key_set().has_any(odd))
    return nullptr;
  return &t;
}

int dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return SSA_DTYPE_BF16;
    case at::kHalf: return SSA_DTYPE_FP16;
    case at::kFloat: return SSA_DTYPE_FP32;
    default: return -1;
  }
}

bool has_kernel(int dtype, int64_t D) {
  return D == 32 || D == 64 || D == 128 || D == 256 || (D == 16 && dtype == SSA_DTYPE_FP32);
}

// Layout the kernels address in place ([B, H, S, D] or [T, H, D]; the row
// dimension is `rows`).
bool addressable(const at::Tensor& t, int rows) {
  const int last = static_cast<int>(t.dim()) - 1;
  if (t.stride(last) != 1 || (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) != 0) return false;
  for (int d = 0; d < last; ++d)
    if (t.size(d) > 1 && t.stride(d) % 8 != 0) return false;
  return t.size(rows) <= 1 || t.stride(rows) < kMaxRowStride;
}

int64_t stride1(const at::Tensor& t, int d) { return t.size(d) > 1 ? t.stride(d) : 0; }

ssa_tensor4 view(const at::Tensor& t) {
  if (t.dim() == 3) return {t.data_ptr(), 0, stride1(t, 1), stride1(t, 0)};  // [T, H, D]
  return {t.data_ptr(), stride1(t, 0), stride1(t, 1), stride1(t, 2)};
}

// ssa_n / ssa_b: a one-element contiguous fp32 tensor
const float* scalar(const at::Tensor* t) {
  return t != nullptr && t->numel() == 1 && t->scalar_type() == at::kFloat && t->is_contiguous()
             ? static_cast<const float*>(t->data_ptr())
             : nullptr;
}

at::Tensor floats(at::IntArrayRef size, const at::Tensor& like) {
  return at::empty(size, like.options().dtype(at::kFloat));
}
at::Tensor bytes(int64_t n, const at::Tensor& like) { return at::empty({n}, like.options().dtype(at::kByte)); }

struct Problem {  // sizes of a q / k / v triple, dense (4-D) or packed (3-D)
  int64_t B, Hq, Hkv, N, D;
  int dtype;
  bool ok(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, int dim) {
    if (q.dim() != dim || k.dim() != dim || v.dim() != dim) return false;
    const int rows = dim == 4 ? 2 : 0;
    dtype = dtype_code(q);
    B = dim == 4 ? q.size(0) : 1;
    Hq = q.size(1);
    N = q.size(rows);
    D = q.size(dim - 1);
    Hkv = k.size(1);
    if (dtype < 0 || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type()) return false;
    if (q.numel() == 0 || k.numel() == 0 || Hq % Hkv != 0 || !has_kernel(dtype, D) || k.sizes() != v.sizes())
      return false;
    if ((dim == 4 && k.size(0) != B) || k.size(rows) != N || k.size(dim - 1) != D) return false;
    if (B > INT32_MAX || Hq > INT32_MAX || N > INT32_MAX) return false;
    return addressable(q, rows) && addressable(k, rows) && addressable(v, rows);
  }
};

struct Args {  // positional arguments of a fast call
  PyObject* const* a;
  int dev;
  void* stream;
  bool good = true;
  const at::Tensor* tensor(int i) {
    const at::Tensor* t = plain(a[i], dev);
    if (t == nullptr) good = false;
    return t;
  }
  double number(int i) {
    if (!PyFloat_CheckExact(a[i]) && !PyLong_CheckExact(a[i])) {
      good = false;
      return 0.0;
    }
    const double v = PyFloat_AsDouble(a[i]);
    if (v == -1.0 && PyErr_Occurred()) {  // an int beyond double
      PyErr_Clear();
      good = false;
    }
    return v;
  }
  int64_t integer(int i) {
    if (!PyLong_Check(a[i])) {
      good = false;
      return 0;
    }
    const long long v = PyLong_AsLongLong(a[i]);
    if (v == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      good = false;
    }
    return v;
  }
};

// The trailing two arguments of every call: current device, raw stream.
Args args_of(PyObject* const* a, Py_ssize_t n) {
  Args r{a, 0, nullptr};
  r.dev = static_cast<int>(r.integer(static_cast<int>(n) - 2));
  r.stream = reinterpret_cast<void*>(r.integer(static_cast<int>(n) - 1));
  return r;
}

PyObject* none() { Py_RETURN_NONE; }

PyObject* pack(std::initializer_list<at::Tensor> ts) {
  PyObject* r = PyTuple_New(static_cast<Py_ssize_t>(ts.size()));
  if (r == nullptr) return nullptr;
  Py_ssize_t i = 0;
  for (const at::Tensor& t : ts) {
    PyObject* o = THPVariable_Wrap(t);
    if (o == nullptr) {
      Py_DECREF(r);
      return nullptr;
    }
    PyTuple_SET_ITEM(r, i++, o);
  }
  return r;
}

bool all_set() { return abi.fwd != nullptr; }

// fwd(q, k, v, scale, n, b, causal, dev, stream) -> (out, m) | status | None
// varlen_fwd(q, k, v, cu, max_seqlen, scale, n, b, causal, dev, stream)
template <bool VARLEN>
PyObject* forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  constexpr int X = VARLEN ? 2 : 0;
  if (n != 9 + X || !all_set()) return none();
  Args in = args_of(a, n);
  const at::Tensor *q = in.tensor(0), *k = in.tensor(1), *v = in.tensor(2);
  const at::Tensor* cu = VARLEN ? in.tensor(3) : nullptr;
  const int64_t longest = VARLEN ? in.integer(4) : 0;
  const double scale = in.number(3 + X);
  const float *np = scalar(in.tensor(4 + X)), *bp = scalar(in.tensor(5 + X));
  const int causal = a[6 + X] == Py_True;
  if (!in.good || np == nullptr || bp == nullptr) return none();
  Problem p;
  if (!p.ok(*q, *k, *v, VARLEN ? 3 : 4)) return none();
  if (VARLEN && (cu->dim() != 1 || cu->numel() < 2 || cu->scalar_type() != at::kInt || !cu->is_contiguous() ||
                 longest <= 0 || longest > INT32_MAX || cu->numel() > INT32_MAX))
    return none();
  at::Tensor out, m;
  int32_t status;
  {
    pybind11::gil_scoped_release unlocked;
    out = at::empty_like(*q);
    if (!addressable(out, VARLEN ? 0 : 2)) out = at::empty(q->sizes(), q->options());
    if constexpr (VARLEN)
      m = floats({p.Hq, p.N}, *q);
    else
      m = floats({p.B, p.Hq, p.N}, *q);
    ssa_fwd_args f{view(*q), view(*k), view(*v), view(out), static_cast<float*>(m.data_ptr()), np, bp,
                   static_cast<int32_t>(p.B), static_cast<int32_t>(p.Hq), static_cast<int32_t>(p.Hkv),
                   static_cast<int32_t>(p.N), static_cast<int32_t>(p.D), p.dtype, causal, static_cast<float>(scale)};
    if constexpr (VARLEN) {
      f.batch = static_cast<int32_t>(cu->numel() - 1);
      f.seqlen = static_cast<int32_t>(longest);
      const ssa_varlen_fwd_args vf{f, static_cast<const int32_t*>(cu->data_ptr()), static_cast<int32_t>(p.N)};
      status = abi.varlen_fwd(&vf, in.stream);
    } else {
      status = abi.fwd(&f, in.stream);
    }
  }
  if (status != 0) return PyLong_FromLong(status);
  return pack({out, m});
  END_HANDLE_TH_ERRORS
}

// Bytes that the caching allocator of GPU `dev` holds unused and, with `driver`,
// those that the driver has free besides.  Throws where they are not known.
int64_t free_bytes(int dev, bool driver) {
  c10::DeviceAllocator* a = c10::getDeviceAllocator(c10::DeviceType::CUDA);
  const auto index = static_cast<c10::DeviceIndex>(dev);
  const auto st = a->getDeviceStats(index);
  constexpr auto all = static_cast<size_t>(c10::CachingAllocator::StatType::AGGREGATE);
  const int64_t held = st.reserved_bytes[all].current - st.allocated_bytes[all].current;
  return driver ? held + static_cast<int64_t>(a->getMemoryInfo(index).first) : held;
}

// Whether the dS' workspace stays within half of the headroom.  What the allocator
// holds often answers it without the driver (1 us for 5 to 13, by host): half of it,
// or all of it up to 256 MiB, a thousandth of the card, as a repeated call finds its
// last workspace there.  The same question through torch.cuda takes 90 us and leaves
// some hundred Python objects, enough for a full collection by the interpreter (40
// ms) every hundred steps or so: steps 6 to 25 of a 4 x 16 x 4096 x 128 forward and
// backward took 2.5 ms for 1.4.
constexpr int64_t kSmallWorkspace = int64_t{256} << 20;
bool ds_fits(int64_t nbytes, int dev) {
  try {
    const int64_t held = free_bytes(dev, false);
    return nbytes <= held / 2 || (nbytes <= kSmallWorkspace && nbytes <= held) || nbytes <= free_bytes(dev, true) / 2;
  } catch (const std::exception&) {
    return true;  // unknown: the byte cap alone
  }
}

// headroom(dev) -> bytes | None (unknown)
PyObject* headroom(PyObject*, PyObject* const* a, Py_ssize_t n) {
  Args in{a, 0, nullptr};
  const int64_t dev = n == 1 ? in.integer(0) : -1;
  if (n != 1 || !in.good || dev < 0 || dev > 127) return none();
  int64_t bytes = 0;
  try {
    pybind11::gil_scoped_release unlocked;
    bytes = free_bytes(static_cast<int>(dev), true);
  } catch (const std::exception&) {
    return none();
  }
  return PyLong_FromLongLong(bytes);
}

// bwd(q, k, v, out, dout, m, scale, n, b, causal, ds_max, dev, stream)
// varlen_bwd(q, k, v, out, dout, m, cu, max_seqlen, scale, n, b, causal, ds_max, dev, stream)
//   -> (dq, dk, dv, dn, db) | status | None
// ds_max: the dS' workspace is used up to that many bytes (0: never, -1: any
// size) and half of the device's headroom.  Without one, or where its allocation
// (the call's last) fails, dq recomputes the scores.
template <bool VARLEN>
PyObject* backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  constexpr int X = VARLEN ? 2 : 0;
  if (n != 13 + X || !all_set()) return none();
  Args in = args_of(a, n);
  const at::Tensor *q = in.tensor(0), *k = in.tensor(1), *v = in.tensor(2), *out = in.tensor(3), *dout = in.tensor(4),
                   *m = in.tensor(5);
  const at::Tensor* cu = VARLEN ? in.tensor(6) : nullptr;
  const int64_t longest = VARLEN ? in.integer(7) : 0;
  const double scale = in.number(6 + X);
  const float *np = scalar(in.tensor(7 + X)), *bp = scalar(in.tensor(8 + X));
  const int causal = a[9 + X] == Py_True;
  const int64_t ds_max = in.integer(10 + X);
  if (!in.good || np == nullptr || bp == nullptr) return none();
  constexpr int rows = VARLEN ? 0 : 2;
  Problem p;
  if (!p.ok(*q, *k, *v, VARLEN ? 3 : 4)) return none();
  if (out->sizes() != q->sizes() || dout->sizes() != q->sizes() || out->scalar_type() != q->scalar_type() ||
      dout->scalar_type() != q->scalar_type() || !addressable(*out, rows) || !addressable(*dout, rows))
    return none();
  const int64_t mdim = VARLEN ? 2 : 3;
  if (m->dim() != mdim || m->size(mdim - 1) != p.N || m->size(mdim - 2) != p.Hq || (!VARLEN && m->size(0) != p.B) ||
      m->scalar_type() != at::kFloat || !m->is_contiguous())
    return none();
  if (VARLEN && (cu->dim() != 1 || cu->numel() < 2 || cu->scalar_type() != at::kInt || !cu->is_contiguous() ||
                 longest <= 0 || longest > INT32_MAX || cu->numel() > INT32_MAX))
    return none();
  const int32_t batch = static_cast<int32_t>(VARLEN ? cu->numel() - 1 : p.B);
  const int32_t seqlen = static_cast<int32_t>(VARLEN ? longest : p.N);
  const int32_t Hq = static_cast<int32_t>(p.Hq), Hkv = static_cast<int32_t>(p.Hkv), T = static_cast<int32_t>(p.N);
  const int64_t count = abi.partials_count(batch, Hkv, seqlen);
  int64_t ds_bytes = 0;
  if (p.dtype != SSA_DTYPE_FP32 && p.D <= 128 && ds_max != 0) {  // the fp32-precision kernels use none
    ds_bytes = VARLEN ? abi.varlen_ds_bytes(batch, Hq, seqlen, T, causal) : abi.ds_bytes(batch, Hq, seqlen, causal);
    if (ds_bytes <= 0) return none();
    if (ds_max > 0 && ds_bytes > ds_max) ds_bytes = 0;
  }
  if (count <= 0) return none();
  at::Tensor dq, dk, dv, dn, db;
  int32_t status;
  {
    pybind11::gil_scoped_release unlocked;
    auto grad_of = [&](const at::Tensor& t) {
      at::Tensor g = at::empty_like(t);
      return addressable(g, rows) ? g : at::empty(t.sizes(), t.options());
    };
    dq = grad_of(*q);
    dk = grad_of(*k);
    dv = grad_of(*v);
    dn = floats({}, *q);
    db = floats({}, *q);
    const at::Tensor delta = floats(m->sizes(), *q), partials = floats({count}, *q);
    at::Tensor ds;
    if (ds_bytes > 0) {
      if (ds_max < 0) {
        ds = bytes(ds_bytes, *q);
      } else if (ds_fits(ds_bytes, in.dev)) {
        try {
          ds = bytes(ds_bytes, *q);
        } catch (const c10::OutOfMemoryError&) {
        }
      }
    }
    const ssa_bwd_args f{view(*q), view(*k), view(*v), view(*out), view(*dout), view(dq), view(dk), view(dv),
                         static_cast<const float*>(m->data_ptr()), static_cast<float*>(delta.data_ptr()),
                         static_cast<float*>(partials.data_ptr()), static_cast<float*>(dn.data_ptr()),
                         static_cast<float*>(db.data_ptr()), np, bp, batch, Hq, Hkv, seqlen,
                         static_cast<int32_t>(p.D), p.dtype, causal, static_cast<float>(scale),
                         ds.defined() ? ds.data_ptr() : nullptr};
    if constexpr (VARLEN) {
      const ssa_varlen_bwd_args vf{f, static_cast<const int32_t*>(cu->data_ptr()), T};
      status = abi.varlen_bwd(&vf, in.stream);
    } else {
      status = abi.bwd(&f, in.stream);
    }
  }
  if (status != 0) return PyLong_FromLong(status);
  return pack({dq, dk, dv, dn, db});
  END_HANDLE_TH_ERRORS
}

// The launch layer's key splits for num_splits = 0: about 256 workgroups (one
// per CU), as the library's own choice, but down to 128 keys a split (the library
// stops at 256): a lone short cache is bound by latency, and its splits run side
// by side (us, 256 -> 128 keys: 1 x 16 x 2048 x 128 12.5 -> 9.4, 1 x 32/8 x 2048 x 64
// 9.1 -> 8.0, 1 x 4 x 8192 x 128 12.6 -> 10.6).  Caches up to 256 keys stay whole:
// the merge costs more than they gain (8 x 8 x 150 x 64: 5.2 against 7.4).
int64_t launch_splits(int64_t B, int64_t Hq, int64_t Hkv, int64_t cap) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || cap <= 256) return 1;
  const int64_t units = B * Hkv * ((Hq / Hkv + 31) / 32);
  const int64_t want = (256 + units - 1) / units, most = (cap + 127) / 128;
  return want < most ? want : most;
}

// decode_splits(B, Hq, Hkv, capacity): launch_splits
PyObject* decode_splits(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 4) {
    PyErr_SetString(PyExc_TypeError, "decode_splits: four arguments");
    return nullptr;
  }
  int64_t v[4];
  for (int i = 0; i < 4; ++i) {
    v[i] = PyLong_AsLongLong(a[i]);
    if (v[i] == -1 && PyErr_Occurred()) return nullptr;
    if (v[i] < 0 || v[i] > INT32_MAX) v[i] = 0;  // the library refuses the call
  }
  return PyLong_FromLongLong(launch_splits(v[0], v[1], v[2], v[3]));
}

// decode(q, k_cache, v_cache, lens, scale, n, b, num_splits, dev, stream)
//   -> (out [B, Hq, D],) | status | None
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 10 || !all_set()) return none();
  Args in = args_of(a, n);
  const at::Tensor *q = in.tensor(0), *k = in.tensor(1), *v = in.tensor(2), *lens = in.tensor(3);
  const double scale = in.number(4);
  const float *np = scalar(in.tensor(5)), *bp = scalar(in.tensor(6));
  const int64_t splits = in.integer(7);
  if (!in.good || np == nullptr || bp == nullptr || q->dim() != 3 || k->dim() != 4 || v->dim() != 4) return none();
  const int64_t B = q->size(0), Hq = q->size(1), D = q->size(2), Hkv = k->size(1), cap = k->size(2);
  const int dtype = dtype_code(*q);
  if ((dtype != SSA_DTYPE_BF16 && dtype != SSA_DTYPE_FP16) || (D != 32 && D != 64 && D != 128)) return none();
  if (q->numel() == 0 || k->numel() == 0 || k->sizes() != v->sizes() || k->size(0) != B || k->size(3) != D ||
      Hq % Hkv != 0 || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() ||
      B > INT32_MAX || Hq > INT32_MAX || cap > INT32_MAX || splits < 0 || splits > INT32_MAX)
    return none();
  if (lens->dim() != 1 || lens->size(0) != B || lens->scalar_type() != at::kInt || !lens->is_contiguous())
    return none();
  // q [B, Hq, D] as [B, Hq, 1, D]: its rows are the heads
  if (!addressable(*k, 2) || !addressable(*v, 2) || q->stride(2) != 1 ||
      (reinterpret_cast<uintptr_t>(q->data_ptr()) & 15) != 0 || stride1(*q, 0) % 8 != 0 || stride1(*q, 1) % 8 != 0)
    return none();
  at::Tensor out;
  int32_t status;
  {
    pybind11::gil_scoped_release unlocked;
    const int32_t b32 = static_cast<int32_t>(B), hq = static_cast<int32_t>(Hq), hk = static_cast<int32_t>(Hkv),
                  c32 = static_cast<int32_t>(cap), d32 = static_cast<int32_t>(D),
                  sp = static_cast<int32_t>(splits != 0 ? splits : launch_splits(B, Hq, Hkv, cap));
    out = at::empty({B, Hq, D}, q->options());
    const int64_t ws_bytes = abi.decode_bytes(b32, hq, hk, c32, d32, sp);
    at::Tensor ws;
    if (ws_bytes > 0) ws = bytes(ws_bytes, *q);
    const ssa_decode_args f{{q->data_ptr(), stride1(*q, 0), stride1(*q, 1), 0}, view(*k), view(*v),
                            {out.data_ptr(), stride1(out, 0), stride1(out, 1), 0}, nullptr,
                            static_cast<const int32_t*>(lens->data_ptr()), np, bp, b32, hq, hk, c32, d32, dtype, sp,
                            static_cast<float>(scale), ws.defined() ? ws.data_ptr() : nullptr};
    status = abi.decode(&f, in.stream);
  }
  if (status != 0) return PyLong_FromLong(status);
  return pack({out});
  END_HANDLE_TH_ERRORS
}

// bind(address, ...): the C ABI entry points in the order of Abi
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != static_cast<Py_ssize_t>(sizeof(Abi) / sizeof(void*))) {
    PyErr_SetString(PyExc_TypeError, "bind: wrong number of entry points");
    return nullptr;
  }
  void* p[sizeof(Abi) / sizeof(void*)];
  for (Py_ssize_t i = 0; i < n; ++i) {
    p[i] = PyLong_AsVoidPtr(a[i]);
    if (p[i] == nullptr) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: null entry point");
      return nullptr;
    }
  }
  std::memcpy(&abi, p, sizeof(abi));
  Py_RETURN_NONE;
}

#define SSA_FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(f)), METH_FASTCALL, nullptr
PyMethodDef methods[] = {{"bind", SSA_FAST(&bind)},
                         {"fwd", SSA_FAST(&forward<false>)},
                         {"bwd", SSA_FAST(&backward<false>)},
                         {"varlen_fwd", SSA_FAST(&forward<true>)},
                         {"varlen_bwd", SSA_FAST(&backward<true>)},
                         {"decode", SSA_FAST(&decode)},
                         {"decode_splits", SSA_FAST(&decode_splits)},
                         {"headroom", SSA_FAST(&headroom)},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ssa_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// ABI_VERSION and TORCH_VERSION: what the module was built for, checked by its
// loader (SSA/_lib.py) before bind().
PyMODINIT_FUNC PyInit__ssa_native() {
  PyObject* m = PyModule_Create(&module);
  if (m == nullptr) return nullptr;
  if (PyModule_AddIntConstant(m, "ABI_VERSION", SSA_ABI_VERSION) < 0 ||
      PyModule_AddStringConstant(m, "TORCH_VERSION", TORCH_VERSION) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}

// _hp_calls: what hp_cuda_ops.py does per call, in native code.  Each function takes the argument lists of one
// hp_cuda_* driver (sequences of tensors or raw device addresses, sequences of numbers), checks the tensors, lays
// the lists out as the arrays the C ABI wants and makes the call on the given stream (None: torch's current one)
// with the interpreter lock released.
//
// What bounds it: touching every list element once.  Through ctypes arrays built by list comprehensions an element
// cost 0.3-0.5 us, which for a bucket was several times what the GPU needed (161 tensors, encode + decode:
// 244 us a pass against 50 us of kernels); here a tensor costs about 20 ns and a number 5.
//
// Host C++ only.
#include <torch/extension.h>

#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>

#include <vector>

#include "hpx.h"

namespace {

struct PyError {};  // a Python exception is set

// Any iterable, as a list or tuple of `n` elements.
struct Seq {
  PyObject* fast;
  PyObject** items;
  Py_ssize_t n;
  explicit Seq(PyObject* o) : fast(PySequence_Fast(o, "a sequence is needed")) {
    if (!fast) throw PyError{};
    items = PySequence_Fast_ITEMS(fast);
    n = PySequence_Fast_GET_SIZE(fast);
  }
  Seq(const Seq&) = delete;
  Seq& operator=(const Seq&) = delete;
  ~Seq() { Py_DECREF(fast); }
};

// int(v) modulo 2^64, as a ctypes integer array would store it.
inline uint64_t as_int(PyObject* v) {
  if (PyLong_CheckExact(v)) {
    const uint64_t x = PyLong_AsUnsignedLongLongMask(v);
    if (x == ~0ull && PyErr_Occurred()) throw PyError{};
    return x;
  }
  PyObject* i = PyNumber_Long(v);
  if (!i) throw PyError{};
  const uint64_t x = PyLong_AsUnsignedLongLongMask(i);
  Py_DECREF(i);
  if (x == ~0ull && PyErr_Occurred()) throw PyError{};
  return x;
}

inline double as_float(PyObject* v) {
  if (PyFloat_CheckExact(v)) return PyFloat_AS_DOUBLE(v);
  const double x = PyFloat_AsDouble(v);
  if (x == -1.0 && PyErr_Occurred()) throw PyError{};
  return x;
}

void need(Py_ssize_t have, Py_ssize_t want, const char* what) {
  if (have >= want) return;
  PyErr_Format(PyExc_ValueError, "%s: %zd entries for %zd tensors", what, have, want);
  throw PyError{};
}

template <typename T>
std::vector<T> ints(PyObject* o, Py_ssize_t count, const char* what) {
  Seq s(o);
  need(s.n, count, what);
  std::vector<T> v(static_cast<size_t>(s.n));
  for (Py_ssize_t i = 0; i < s.n; i++) v[size_t(i)] = static_cast<T>(as_int(s.items[i]));
  return v;
}
template <typename T>
std::vector<T> floats(PyObject* o, Py_ssize_t count, const char* what) {
  Seq s(o);
  need(s.n, count, what);
  std::vector<T> v(static_cast<size_t>(s.n));
  for (Py_ssize_t i = 0; i < s.n; i++) v[size_t(i)] = static_cast<T>(as_float(s.items[i]));
  return v;
}

// Device addresses of a list; the tensors among its elements are checked as CHECK_CUDA_INPUT does (hp_cuda.cpp:107-111).
template <typename T>
std::vector<T*> addresses(const Seq& s, Py_ssize_t count, const char* what) {
  std::vector<T*> v(static_cast<size_t>(s.n));
  for (Py_ssize_t i = 0; i < s.n; i++) {
    PyObject* o = s.items[i];
    if (THPVariable_Check(o)) {
      const at::Tensor& t = THPVariable_Unpack(o);
      if (!t.is_cuda()) {
        PyErr_Format(PyExc_RuntimeError, "%s must be a CUDA tensor", what);
        throw PyError{};
      }
      if (!t.is_contiguous()) {
        PyErr_Format(PyExc_RuntimeError, "%s must be contiguous", what);
        throw PyError{};
      }
      v[size_t(i)] = static_cast<T*>(t.data_ptr());
    } else {
      v[size_t(i)] = reinterpret_cast<T*>(static_cast<uintptr_t>(as_int(o)));
    }
  }
  need(s.n, count, what);
  return v;
}
template <typename T>
std::vector<T*> addresses(PyObject* o, Py_ssize_t count, const char* what) {
  return addresses<T>(Seq(o), count, what);
}

const at::Tensor& tensor(PyObject* o, const char* what) {
  if (!THPVariable_Check(o)) {
    PyErr_Format(PyExc_TypeError, "%s must be a tensor", what);
    throw PyError{};
  }
  return THPVariable_Unpack(o);
}

hipStream_t stream_of(PyObject* o) {
  if (o == Py_None) return c10::hip::getCurrentHIPStream().stream();
  return reinterpret_cast<hipStream_t>(static_cast<uintptr_t>(as_int(o)));
}

template <typename F>
PyObject* released(F&& call) {
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = call();
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// The call, then a wait for the stream (hp_cuda_kernel.cu:157, :197).
template <typename F>
PyObject* released_and_waited(hipStream_t st, F&& call) {
  int rc, waited;
  Py_BEGIN_ALLOW_THREADS
  const int begun = hpx_completion_begin();
  rc = call();
  waited = begun == HPX_OK ? hpx_completion_wait(st) : begun;
  Py_END_ALLOW_THREADS
  if (waited != HPX_OK) {
    PyErr_Format(PyExc_RuntimeError, "HIP error: %s", hpx_last_error());
    throw PyError{};
  }
  return PyLong_FromLong(rc);
}

template <typename T>
const T* const* ro(const std::vector<T*>& v) { return const_cast<const T* const*>(v.data()); }

PyObject* terngrad(PyObject* const* a) {  // ins, in_sizes, outs, out_sizes, bitwidths, enable_randoms, stream, seeds
  Seq s(a[0]);
  const Py_ssize_t n = s.n;
  const auto in = addresses<float>(s, n, "tensor");
  const auto out = addresses<uint8_t>(a[2], n, "B");
  const auto in_size = ints<int32_t>(a[1], n, "in sizes"), out_size = ints<int32_t>(a[3], n, "out sizes");
  const auto bits = ints<uint8_t>(a[4], n, "bitwidths");
  const auto rnd = ints<int32_t>(a[5], n, "enable_randoms");
  hipStream_t st = stream_of(a[6]);
  std::vector<uint64_t> seeds;
  if (a[7] != Py_None) seeds = ints<uint64_t>(a[7], n, "seeds");
  const uint64_t* sd = a[7] != Py_None ? seeds.data() : nullptr;
  return released([&] { return hpx_terngrad_encode(int(n), ro(in), in_size.data(), out.data(), out_size.data(), bits.data(), rnd.data(), sd, st); });
}

PyObject* terngradr(PyObject* const* a) {  // outs, out_sizes, ins, in_sizes, is_add_tos, stream
  Seq s(a[0]);
  const Py_ssize_t n = s.n;
  const auto out = addresses<float>(s, n, "tensor");
  const auto in = addresses<uint8_t>(a[2], n, "B");
  const auto out_size = ints<int32_t>(a[1], n, "out sizes"), in_size = ints<int32_t>(a[3], n, "in sizes"), add = ints<int32_t>(a[4], n, "is_add_tos");
  hipStream_t st = stream_of(a[5]);
  return released([&] { return hpx_terngrad_decode(int(n), out.data(), out_size.data(), ro(in), in_size.data(), add.data(), st); });
}

PyObject* tbq(PyObject* const* a) {  // grads, sizes, residuals, outs, thresholds, stream
  Seq s(a[0]);
  const Py_ssize_t n = s.n;
  const auto g = addresses<float>(s, n, "tensor");
  const auto r = addresses<float>(a[2], n, "residual");
  const auto out = addresses<uint8_t>(a[3], n, "B");
  const auto size = ints<int32_t>(a[1], n, "sizes");
  const auto thr = floats<float>(a[4], n, "thresholds");
  hipStream_t st = stream_of(a[5]);
  return released_and_waited(st, [&] { return hpx_tbq_encode(int(n), ro(g), size.data(), r.data(), out.data(), thr.data(), st); });
}

PyObject* tbqr(PyObject* const* a) {  // outs, sizes, ins, thresholds, is_add_tos, stream
  Seq s(a[0]);
  const Py_ssize_t n = s.n;
  const auto out = addresses<float>(s, n, "tensor");
  const auto in = addresses<uint8_t>(a[2], n, "B");
  const auto size = ints<int32_t>(a[1], n, "sizes");
  const auto thr = floats<float>(a[3], n, "thresholds");
  const auto add = ints<int32_t>(a[4], n, "is_add_tos");
  hipStream_t st = stream_of(a[5]);
  return released_and_waited(st, [&] { return hpx_tbq_decode(int(n), out.data(), size.data(), ro(in), thr.data(), add.data(), st); });
}

PyObject* gd(PyObject* const* a) {  // grads, Ns, residuals, outs, sample_rates, drop_ratios, stream, seeds
  Seq s(a[0]);
  const Py_ssize_t n = s.n;
  const auto g = addresses<float>(s, n, "tensor");
  const auto r = addresses<float>(a[2], n, "residual");
  const auto out = addresses<uint8_t>(a[3], n, "B");
  const auto size = ints<int32_t>(a[1], n, "Ns");
  const auto rate = floats<double>(a[4], n, "sample_rates"), drop = floats<double>(a[5], n, "drop_ratios");
  hipStream_t st = stream_of(a[6]);
  std::vector<uint64_t> seeds;
  if (a[7] != Py_None) seeds = ints<uint64_t>(a[7], n, "seeds");
  const uint64_t* sd = a[7] != Py_None ? seeds.data() : nullptr;
  return released([&] { return hpx_gd_encode(int(n), ro(g), size.data(), r.data(), out.data(), rate.data(), drop.data(), sd, st); });
}

PyObject* gdr(PyObject* const* a) {  // ins, in_sizes, outs, out_sizes, is_add_tos, stream
  Seq s(a[0]);
  const Py_ssize_t n = s.n;
  const auto in = addresses<uint8_t>(s, n, "B");
  const auto out = addresses<float>(a[2], n, "tensor");
  const auto in_size = ints<int32_t>(a[1], n, "in sizes"), out_size = ints<int32_t>(a[3], n, "out sizes"), add = ints<int32_t>(a[4], n, "is_add_tos");
  hipStream_t st = stream_of(a[5]);
  return released([&] { return hpx_gd_decode(int(n), ro(in), in_size.data(), out.data(), out_size.data(), add.data(), st); });
}

// Shapes of the matrices M (n x m) and the factors Q (m x r).
struct Dims {
  std::vector<int32_t> n, m, r;
};
Dims dims(const Seq& Ms, const Seq& Qs, Py_ssize_t count) {
  Dims d;
  const Py_ssize_t k = Ms.n < Qs.n ? Ms.n : Qs.n;
  need(k, count, "M and Q");
  for (Py_ssize_t i = 0; i < k; i++) {
    const at::Tensor& M = tensor(Ms.items[i], "M");
    const at::Tensor& Q = tensor(Qs.items[i], "Q");
    if (M.dim() != 2 || Q.dim() != 2 || Q.size(0) != M.size(1)) {
      PyErr_SetString(PyExc_RuntimeError, "M must be n x m and Q m x r");
      throw PyError{};
    }
    d.n.push_back(int32_t(M.size(0)));
    d.m.push_back(int32_t(M.size(1)));
    d.r.push_back(int32_t(Q.size(1)));
  }
  return d;
}
std::vector<int64_t> numels(const Seq& s, const char* what) {
  std::vector<int64_t> v(static_cast<size_t>(s.n));
  for (Py_ssize_t i = 0; i < s.n; i++) v[size_t(i)] = tensor(s.items[i], what).numel();
  return v;
}

PyObject* powersgd_encode1(PyObject* const* a) {  // grads, residuals, Qs, Ms, Ps, stream
  Seq g(a[0]), Q(a[2]), M(a[3]);
  const Py_ssize_t n = g.n;
  const auto gp = addresses<float>(g, n, "tensor");
  const auto rp = addresses<float>(a[1], n, "residual");
  const auto qp = addresses<float>(Q, n, "Q"), mp = addresses<float>(M, n, "M"), pp = addresses<float>(a[4], n, "P");
  const Dims d = dims(M, Q, n);
  const auto numel = numels(g, "tensor");
  hipStream_t st = stream_of(a[5]);
  return released([&] { return hpx_powersgd_encode1(int(n), ro(gp), numel.data(), ro(rp), ro(qp), mp.data(), pp.data(), d.n.data(), d.m.data(), d.r.data(), st); });
}

PyObject* powersgd_encode2(PyObject* const* a) {  // Ps, Ms, Qs, stream
  Seq P(a[0]), M(a[1]), Q(a[2]);
  const Py_ssize_t n = P.n;
  const auto pp = addresses<float>(P, n, "P"), mp = addresses<float>(M, n, "M"), qp = addresses<float>(Q, n, "Q");
  const Dims d = dims(M, Q, n);
  hipStream_t st = stream_of(a[3]);
  return released([&] { return hpx_powersgd_encode2(int(n), pp.data(), ro(mp), qp.data(), d.n.data(), d.m.data(), d.r.data(), st); });
}

PyObject* powersgd_decode(PyObject* const* a) {  // Ps, Qs, Ms, residuals, grads, stream
  Seq Q(a[1]), M(a[2]), g(a[4]);
  const Py_ssize_t n = g.n;
  const auto pp = addresses<float>(a[0], n, "P"), qp = addresses<float>(Q, n, "Q"), mp = addresses<float>(M, n, "M");
  const auto rp = addresses<float>(a[3], n, "residual"), gp = addresses<float>(g, n, "tensor");
  const Dims d = dims(M, Q, n);
  const auto numel = numels(g, "tensor");
  hipStream_t st = stream_of(a[5]);
  return released([&] { return hpx_powersgd_decode(int(n), ro(pp), ro(qp), mp.data(), rp.data(), gp.data(), numel.data(), d.n.data(), d.m.data(), d.r.data(), st); });
}

// A fixed number of positional arguments, and C++ exceptions turned into Python ones.
template <PyObject* (*F)(PyObject* const*), Py_ssize_t ARGS>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != ARGS) return PyErr_Format(PyExc_TypeError, "%zd arguments are needed, %zd were given", ARGS, nargs);
  try {
    return F(args);
  } catch (const PyError&) {
    return nullptr;
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

template <PyObject* (*F)(PyObject* const*), Py_ssize_t ARGS>
PyMethodDef method(const char* name) {
  return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<F, ARGS>)), METH_FASTCALL, nullptr};
}

PyMethodDef g_methods[] = {
    method<terngrad, 8>("terngrad"),
    method<terngradr, 6>("terngradr"),
    method<tbq, 6>("tbq"),
    method<tbqr, 6>("tbqr"),
    method<gd, 8>("gd"),
    method<gdr, 6>("gdr"),
    method<powersgd_encode1, 6>("powersgd_encode1"),
    method<powersgd_encode2, 4>("powersgd_encode2"),
    method<powersgd_decode, 6>("powersgd_decode"),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_hp_calls", "the nine hp_cuda_* drivers' argument lists, laid out natively", -1, g_methods,
                        nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__hp_calls() { return PyModule_Create(&g_module); }

// Native front of the basket queries (vecgeom_amd/queries.py): checks the
// argument tensors, allocates the output and calls the C-ABI entry point, in
// one Python call.  A query on a few hundred points is a 2 us kernel; the same
// checks, allocation and ctypes call in Python took 9 us around it.
//
// run(fn, family, geometry, placed, points, directions, step_max, out, code,
// next) returns (status, output), or None for arguments it does not take
// (wrong type, dtype, device, length or layout, or tensors without storage):
// the Python code then goes through its own checks and raises what it always
// raised.  fn is the address of the entry point, geometry the handle as an
// integer; the work goes on torch's current stream.
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>

#include <cstdint>

namespace {

// Entry points by argument list.
enum Family : long {
  kPoints = 0,      // (g, placed, x, y, z, n, out, stream)
  kRays = 1,        // (g, placed, x, y, z, dx, dy, dz, step_max, n, out, stream)
  kRaysNext = 2,    // the same with next_node before the stream
  kNormal = 3,      // (g, placed, x, y, z, n, nx, ny, nz, valid, stream)
  kRaysNormal = 4,  // (g, placed, x, .. dz, step_max, n, out, nx, ny, nz, valid, convex, stream)
};

using PointsFn = int (*)(const void *, int32_t, const void *, const void *, const void *, size_t, void *, void *);
using RaysFn = int (*)(const void *, int32_t, const void *, const void *, const void *, const void *, const void *,
                       const void *, const void *, size_t, void *, void *);
using RaysNextFn = int (*)(const void *, int32_t, const void *, const void *, const void *, const void *, const void *,
                           const void *, const void *, size_t, void *, void *, void *);
using NormalFn = int (*)(const void *, int32_t, const void *, const void *, const void *, size_t, void *, void *,
                         void *, void *, void *);
using RaysNormalFn = int (*)(const void *, int32_t, const void *, const void *, const void *, const void *,
                             const void *, const void *, const void *, size_t, void *, void *, void *, void *, void *,
                             void *, void *);

constexpr at::ScalarType kCodes[3] = {at::kByte, at::kInt, at::kDouble};

// A contiguous tensor of the type on the device (any index when dev < 0) with
// n entries (any number when n < 0).
bool Fits(PyObject *o, at::ScalarType type, int dev, int64_t n) {
  if (!THPVariable_Check(o)) return false;
  const at::Tensor &t = THPVariable_Unpack(o);
  return t.scalar_type() == type && t.is_cuda() && (dev < 0 || t.get_device() == dev) && (n < 0 || t.numel() == n) &&
         t.is_contiguous();
}

void *Data(PyObject *o) { return THPVariable_Unpack(o).data_ptr(); }

// The three pointers of an SOA triple of doubles; fixes dev and n when open.
bool Triple(PyObject *p, int *dev, int64_t *n, const void *out[3]) {
  if (!(PyTuple_CheckExact(p) || PyList_CheckExact(p)) || PySequence_Fast_GET_SIZE(p) != 3) return false;
  for (int i = 0; i < 3; ++i) {
    PyObject *o = PySequence_Fast_GET_ITEM(p, i);
    if (!Fits(o, at::kDouble, *dev, *n)) return false;
    const at::Tensor &t = THPVariable_Unpack(o);
    if (*dev < 0) {
      *dev = t.get_device();
      *n = t.numel();
    }
    out[i] = t.data_ptr();
  }
  return true;
}

// Calls f without the interpreter lock.
template <class F>
int Unlocked(F f) {
  PyThreadState *state = PyEval_SaveThread();
  const int rc = f();
  PyEval_RestoreThread(state);
  return rc;
}

PyObject *Checked(PyObject *const *a) {
  const auto fn = reinterpret_cast<void *>(PyLong_AsSize_t(a[0]));
  const long family = PyLong_AsLong(a[1]);
  const auto geom = reinterpret_cast<const void *>(PyLong_AsSize_t(a[2]));
  const long placed = PyLong_AsLong(a[3]);
  const long code = PyLong_AsLong(a[8]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  if (!fn || placed != (int32_t)placed || code < 0 || code > 2) Py_RETURN_NONE;
  const int32_t pid = (int32_t)placed;
  int dev = -1;
  int64_t n = -1;
  const void *p[3], *d[3] = {nullptr, nullptr, nullptr};
  if (!Triple(a[4], &dev, &n, p)) Py_RETURN_NONE;
  const bool rays = family == kRays || family == kRaysNext || family == kRaysNormal;
  if (rays && !Triple(a[5], &dev, &n, d)) Py_RETURN_NONE;
  const void *sm = nullptr;
  if (a[6] != Py_None) {
    if (!Fits(a[6], at::kDouble, dev, n)) Py_RETURN_NONE;
    sm = Data(a[6]);
  }
  const at::ScalarType type = kCodes[code];
  if (a[7] != Py_None && !Fits(a[7], type, dev, n)) Py_RETURN_NONE;
  void *next = nullptr;
  if (a[9] != Py_None) {
    if (!Fits(a[9], at::kInt, dev, n)) Py_RETURN_NONE;
    next = Data(a[9]);
  }
  void *const stream = c10::hip::getCurrentHIPStream().stream();
  const auto like = at::TensorOptions().device(THPVariable_Unpack(PySequence_Fast_GET_ITEM(a[4], 0)).device());
  auto fresh = [&](at::ScalarType t) { return at::empty({n}, like.dtype(t)); };
  auto wrap = [](const at::Tensor &t) { return THPVariable_Wrap(t); };
  if (family == kNormal || family == kRaysNormal) {
    const at::Tensor nx = fresh(at::kDouble), ny = fresh(at::kDouble), nz = fresh(at::kDouble),
                     valid = fresh(at::kByte);
    void *const o[4] = {nx.data_ptr(), ny.data_ptr(), nz.data_ptr(), valid.data_ptr()};
    if (family == kNormal) {
      const int rc = Unlocked([&] {
        return reinterpret_cast<NormalFn>(fn)(geom, pid, p[0], p[1], p[2], n, o[0], o[1], o[2], o[3], stream);
      });
      return Py_BuildValue("(i((NNN)N))", rc, wrap(nx), wrap(ny), wrap(nz), wrap(valid));
    }
    const at::Tensor convex = fresh(at::kByte), dist = fresh(at::kDouble);
    void *const t = dist.data_ptr(), *const c = convex.data_ptr();
    const int rc = Unlocked([&] {
      return reinterpret_cast<RaysNormalFn>(fn)(geom, pid, p[0], p[1], p[2], d[0], d[1], d[2], sm, n, t, o[0], o[1],
                                                o[2], o[3], c, stream);
    });
    return Py_BuildValue("(i(N(NNN)NN))", rc, wrap(dist), wrap(nx), wrap(ny), wrap(nz), wrap(valid), wrap(convex));
  }
  const at::Tensor out = a[7] == Py_None ? fresh(type) : THPVariable_Unpack(a[7]);
  void *const o = out.data_ptr();
  const int rc = Unlocked([&] {
    if (family == kPoints) return reinterpret_cast<PointsFn>(fn)(geom, pid, p[0], p[1], p[2], n, o, stream);
    if (family == kRays)
      return reinterpret_cast<RaysFn>(fn)(geom, pid, p[0], p[1], p[2], d[0], d[1], d[2], sm, n, o, stream);
    return reinterpret_cast<RaysNextFn>(fn)(geom, pid, p[0], p[1], p[2], d[0], d[1], d[2], sm, n, o, next, stream);
  });
  if (a[7] == Py_None) return Py_BuildValue("(iN)", rc, wrap(out));
  return Py_BuildValue("(iO)", rc, a[7]);
}

PyObject *Run(PyObject *, PyObject *const *a, Py_ssize_t na) {
  if (na != 10) {
    PyErr_SetString(PyExc_TypeError, "run takes 10 arguments");
    return nullptr;
  }
  // No C++ exception leaves the module: a tensor without storage (a wrapper
  // of a transform) or a failed allocation is left to the Python code.
  try {
    return Checked(a);
  } catch (...) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}

PyMethodDef kMethods[] = {
    {"run", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(Run)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_vgq", nullptr, -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__vgq(void) { return PyModule_Create(&kModule); }

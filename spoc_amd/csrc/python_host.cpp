// CPython extension spoc_amd._host: the launch calls of spoc_amd/sarek.py with their argument lists turned into the C
// structures here.  A launch takes the HIP runtime 2.8 us; building the same structures with ctypes took 2.3 us more for
// one kernel and 5.3 us for a pipeline of two.  The entry points are those of the library the ctypes front end has loaded
// (bind() gets their addresses), so there is one library per process whichever build it is, and their statuses come back
// to the caller, who turns them into exceptions as for every other entry point.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstring>
#include <vector>

#include "sarek_hip.h"

namespace {

decltype(&sarek_hip_execute_run_vectors) g_run_vectors;
decltype(&sarek_hip_execute_run_source) g_run_source;
decltype(&sarek_hip_execute_run_pipeline) g_run_pipeline;
decltype(&sarek_hip_last_run_path) g_last_run_path;
decltype(&sarek_hip_fold_partials_f64) g_fold_partials;

PyObject *s_h, *s_value;   // "_h", "value"

bool bound() {
  if (g_run_vectors) return true;
  PyErr_SetString(PyExc_RuntimeError, "spoc_amd._host: bind() has not been called");
  return false;
}

// What a ctypes integer field takes: an integer (or what __index__ makes one), cut to the field's width.
bool as_bits(PyObject *o, unsigned long long *out) {
  if (PyFloat_Check(o)) {
    PyErr_SetString(PyExc_TypeError, "int expected instead of float instance");
    return false;
  }
  *out = PyLong_AsUnsignedLongLongMask(o);
  return !(*out == static_cast<unsigned long long>(-1) && PyErr_Occurred());
}
bool as_int(PyObject *o, int *out) {
  unsigned long long v;
  if (!as_bits(o, &v)) return false;
  *out = static_cast<int>(v);
  return true;
}

// Sequences are read as tuples: a conversion below may run the caller's code (__index__), which may change a list.

// block or grid: up to three integers, missing ones zero
bool as_dims(PyObject *o, int out[3]) {
  PyObject *seq = PySequence_Tuple(o);
  if (!seq) return false;
  const Py_ssize_t n = PyTuple_GET_SIZE(seq);
  bool ok = n <= 3;
  if (!ok) PyErr_SetString(PyExc_IndexError, "invalid index");
  for (Py_ssize_t i = 0; i < 3 && ok; ++i) {
    out[i] = 0;
    if (i < n) ok = as_int(PyTuple_GET_ITEM(seq, i), out + i);
  }
  Py_DECREF(seq);
  return ok;
}

// A vector's handle: its _h is a ctypes pointer, or None once it is destroyed (the library reports that one)
bool as_handle(PyObject *vector, sarek_hip_vector *out) {
  PyObject *h = PyObject_GetAttr(vector, s_h);
  if (!h) return false;
  bool ok = true;
  *out = nullptr;
  if (h != Py_None) {
    PyObject *value = PyObject_GetAttr(h, s_value);
    ok = value != nullptr;
    if (ok && value != Py_None) {
      *out = static_cast<sarek_hip_vector>(PyLong_AsVoidPtr(value));
      ok = !PyErr_Occurred();
    }
    Py_XDECREF(value);
  }
  Py_DECREF(h);
  return ok;
}

// [(kind, value), ...] as Execute.Vec, .Int, ... make them
bool as_args(PyObject *o, std::vector<sarek_hip_varg> &out) {
  PyObject *seq = PySequence_Tuple(o);
  if (!seq) return false;
  const Py_ssize_t n = PyTuple_GET_SIZE(seq);
  out.resize(static_cast<size_t>(n));
  bool ok = true;
  for (Py_ssize_t i = 0; i < n && ok; ++i) {
    PyObject *item = PySequence_Tuple(PyTuple_GET_ITEM(seq, i));
    if (!item) {
      ok = false;
      break;
    }
    if (PyTuple_GET_SIZE(item) != 2) {
      PyErr_SetString(PyExc_ValueError, "an argument is a pair of kind and value");
      Py_DECREF(item);
      ok = false;
      break;
    }
    PyObject *kind = PyTuple_GET_ITEM(item, 0), *value = PyTuple_GET_ITEM(item, 1);
    sarek_hip_varg &a = out[static_cast<size_t>(i)];
    std::memset(&a, 0, sizeof(a));
    const char *k = PyUnicode_Check(kind) ? PyUnicode_AsUTF8(kind) : "";
    unsigned long long bits = 0;
    if (!k) {
      ok = false;
    } else if (!std::strcmp(k, "vec")) {
      a.kind = SAREK_HIP_VARG_VEC;
      ok = as_handle(value, &a.vec);
    } else if (!std::strcmp(k, "i32")) {
      a.kind = SAREK_HIP_VARG_INT32;
      ok = as_bits(value, &bits);
      a.i32 = static_cast<int32_t>(bits);
    } else if (!std::strcmp(k, "i64")) {
      a.kind = SAREK_HIP_VARG_INT64;
      ok = as_bits(value, &bits);
      a.i64 = static_cast<int64_t>(bits);
    } else if (!std::strcmp(k, "f32")) {
      a.kind = SAREK_HIP_VARG_FLOAT32;
      const double v = PyFloat_AsDouble(value);
      ok = !(v == -1.0 && PyErr_Occurred());
      a.f32 = static_cast<float>(v);
    } else if (!std::strcmp(k, "f64")) {
      a.kind = SAREK_HIP_VARG_FLOAT64;
      a.f64 = PyFloat_AsDouble(value);
      ok = !(a.f64 == -1.0 && PyErr_Occurred());
    } else {
      PyErr_Format(PyExc_ValueError, "unknown vector_arg %R", kind);
      ok = false;
    }
    Py_DECREF(item);
  }
  Py_DECREF(seq);
  return ok;
}

// The status where a call failed, otherwise what `done` makes
template <typename Call, typename Done>
PyObject *finish(Call call, Done done) {
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = call();
  Py_END_ALLOW_THREADS
  return status != SAREK_HIP_OK ? PyLong_FromLong(status) : done();
}
PyObject *path() { return PyUnicode_FromString(g_last_run_path()); }

bool arity(Py_ssize_t given, Py_ssize_t wanted, const char *what) {
  if (given == wanted) return true;
  PyErr_Format(PyExc_TypeError, "%s takes %zd arguments (%zd given)", what, wanted, given);
  return false;
}

// run_vectors(ir, args, block, grid, shared_mem) -> path | status
PyObject *run_vectors(PyObject *, PyObject *const *a, Py_ssize_t n) {
  std::vector<sarek_hip_varg> args;
  int block[3], grid[3], shared;
  if (!bound() || !arity(n, 5, "run_vectors")) return nullptr;
  const char *ir = PyUnicode_AsUTF8(a[0]);
  if (!ir || !as_args(a[1], args) || !as_dims(a[2], block) || !as_dims(a[3], grid) || !as_int(a[4], &shared)) return nullptr;
  return finish([&] { return g_run_vectors(ir, block, grid, shared, args.data(), static_cast<int>(args.size())); }, path);
}

// run_source(source, lang, kernel_name, block, grid, shared_mem, inject_lengths, args) -> path | status
PyObject *run_source(PyObject *, PyObject *const *a, Py_ssize_t n) {
  std::vector<sarek_hip_varg> args;
  int lang, block[3], grid[3], shared, inject;
  if (!bound() || !arity(n, 8, "run_source")) return nullptr;
  const char *source = PyUnicode_AsUTF8(a[0]), *name = source ? PyUnicode_AsUTF8(a[2]) : nullptr;
  if (!name || !as_int(a[1], &lang) || !as_dims(a[3], block) || !as_dims(a[4], grid) || !as_int(a[5], &shared) ||
      !as_int(a[6], &inject) || !as_args(a[7], args))
    return nullptr;
  return finish(
      [&] {
        return g_run_source(source, lang, name, block, grid, shared, inject, args.data(), static_cast<int>(args.size()));
      },
      path);
}

// run_pipeline([(ir, args, block, grid[, shared_mem]), ...]) -> (path, launches) | status
PyObject *run_pipeline(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (!bound() || !arity(n, 1, "run_pipeline")) return nullptr;
  PyObject *seq = PySequence_Tuple(a[0]);
  if (!seq) return nullptr;
  const size_t count = static_cast<size_t>(PyTuple_GET_SIZE(seq));
  std::vector<sarek_hip_pipeline_stage> stages(count);
  std::vector<std::vector<sarek_hip_varg>> args(count);
  // The stages as tuples of their own: they keep the IR texts, which the library reads while other threads run and may
  // change a stage that is a list.
  std::vector<PyObject *> held;
  bool ok = true;
  for (size_t i = 0; i < count && ok; ++i) {
    PyObject *stage = PySequence_Tuple(PyTuple_GET_ITEM(seq, static_cast<Py_ssize_t>(i)));
    if (!stage) {
      ok = false;
      break;
    }
    held.push_back(stage);
    const Py_ssize_t parts = PyTuple_GET_SIZE(stage);
    if (parts < 4) {
      PyErr_Format(PyExc_ValueError, "not enough values to unpack (expected 4, got %zd)", parts);
      ok = false;
      break;
    }
    sarek_hip_pipeline_stage &s = stages[i];
    s.ir_text = PyUnicode_AsUTF8(PyTuple_GET_ITEM(stage, 0));
    s.shared_mem_bytes = 0;
    ok = s.ir_text && as_args(PyTuple_GET_ITEM(stage, 1), args[i]) && as_dims(PyTuple_GET_ITEM(stage, 2), s.block) &&
         as_dims(PyTuple_GET_ITEM(stage, 3), s.grid) && (parts == 4 || as_int(PyTuple_GET_ITEM(stage, 4), &s.shared_mem_bytes));
    s.args = args[i].data();
    s.n_args = static_cast<int>(args[i].size());
  }
  PyObject *result = nullptr;
  int launches = 0;
  if (ok)
    result = finish([&] { return g_run_pipeline(stages.data(), static_cast<int>(count), &launches); },
                    [&] { return Py_BuildValue("(si)", g_last_run_path(), launches); });
  for (PyObject *o : held) Py_DECREF(o);
  Py_DECREF(seq);
  return result;
}

// fold_partials(partials, count, sum, stream) -> status; the pointers and the stream as integers
PyObject *fold_partials(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (!bound() || !arity(n, 4, "fold_partials")) return nullptr;
  void *partials = PyLong_AsVoidPtr(a[0]), *sum = PyLong_AsVoidPtr(a[2]), *stream = PyLong_AsVoidPtr(a[3]);
  const long long count = PyLong_AsLongLong(a[1]);
  if (PyErr_Occurred()) return nullptr;
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = g_fold_partials(static_cast<const float *>(partials), count, static_cast<double *>(sum), stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(status);
}

// bind(addresses of the five entry points above, in the order of their declaration)
PyObject *bind(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (!arity(n, 5, "bind")) return nullptr;
  void *p[5];
  for (int i = 0; i < 5; ++i) p[i] = PyLong_AsVoidPtr(a[i]);
  if (PyErr_Occurred()) return nullptr;
  g_run_source = reinterpret_cast<decltype(g_run_source)>(p[1]);
  g_run_pipeline = reinterpret_cast<decltype(g_run_pipeline)>(p[2]);
  g_last_run_path = reinterpret_cast<decltype(g_last_run_path)>(p[3]);
  g_fold_partials = reinterpret_cast<decltype(g_fold_partials)>(p[4]);
  g_run_vectors = reinterpret_cast<decltype(g_run_vectors)>(p[0]);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", reinterpret_cast<PyCFunction>(bind), METH_FASTCALL, "Addresses of the library's entry points."},
    {"run_vectors", reinterpret_cast<PyCFunction>(run_vectors), METH_FASTCALL, "sarek_hip_execute_run_vectors"},
    {"run_source", reinterpret_cast<PyCFunction>(run_source), METH_FASTCALL, "sarek_hip_execute_run_source"},
    {"run_pipeline", reinterpret_cast<PyCFunction>(run_pipeline), METH_FASTCALL, "sarek_hip_execute_run_pipeline"},
    {"fold_partials", reinterpret_cast<PyCFunction>(fold_partials), METH_FASTCALL, "sarek_hip_fold_partials_f64"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Argument lists of launches, built natively.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
  s_h = PyUnicode_InternFromString("_h");
  s_value = PyUnicode_InternFromString("value");
  return s_h && s_value ? PyModule_Create(&module) : nullptr;
}

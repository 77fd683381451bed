// The two calls of a decode step as Python makes them, in C++: ri_append_kv, and ri_decode_step or ri_host_step by a prepared
// call; and the operators that assembled execution buffers are attended with.  Made by Python a short context's step takes the
// host longer than the GPU (15.3 us against 13.8 captured, 8 groups of 8192 tokens; here 8.7), and beside the launches that is an
// attribute, a method call and a comparison for each of the buffers whose address a prepared call holds, an output tensor, a call
// through ctypes.  Everything is looked at in every call; what is not the usual case (tensors that are not plain ones on one
// device, rows of another shape or type, a buffer that has moved or is too short) is answered with None, and the caller goes its
// general way.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <vector>

#include "../../include/retro_mi355.h"

namespace {

// the tensor behind a Python object, null unless it is a plain one with memory of its own
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.has_storage() ? &t : nullptr;
}

// hipStream_t of the current device's current stream
ri_stream_t current_stream() {
  return (ri_stream_t)c10::hip::getCurrentHIPStream(c10::hip::current_device()).stream();
}

bool shape_is(const at::Tensor& t, PyObject* shape) {
  if (!PyTuple_Check(shape) || PyTuple_GET_SIZE(shape) != t.dim()) return false;
  for (int64_t i = 0; i < t.dim(); ++i) {
    const long long n = PyLong_AsLongLong(PyTuple_GET_ITEM(shape, i));
    if (n == -1 && PyErr_Occurred()) throw python_error();
    if (n != t.size(i)) return false;
  }
  return true;
}

// append(key_row, value_row, steady_k, steady_v, pos, pos_dev or None, row_shape): status, or None where it has to be the general way
PyObject* append(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7) {
    PyErr_SetString(PyExc_TypeError, "append: seven arguments");
    return nullptr;
  }
  const at::Tensor* t[4];
  for (int i = 0; i < 4; ++i)
    if (!(t[i] = plain(args[i]))) Py_RETURN_NONE;
  const at::Tensor &k = *t[2], &v = *t[3];
  const int device = k.get_device();
  const long long pos = PyLong_AsLongLong(args[4]);
  if (pos == -1 && PyErr_Occurred()) return nullptr;
  if (device < 0 || !k.is_cuda() || v.get_device() != device || k.dim() != 4 || v.sizes() != k.sizes() || k.size(3) != 128 ||
      !k.is_contiguous() || !v.is_contiguous() || pos >= k.size(2))
    Py_RETURN_NONE;
  for (int i = 0; i < 2; ++i) {
    const at::Tensor &row = *t[i], &zone = *t[i + 2];
    if (row.get_device() != device || row.scalar_type() != zone.scalar_type() || !row.is_contiguous() ||
        !shape_is(row, args[6]) || row.numel() != k.size(0) * k.size(1) * 128 || (uintptr_t)row.data_ptr() % 16 != 0)
      Py_RETURN_NONE;
  }
  const int64_t* pos_dev = nullptr;
  if (args[5] != Py_None) {
    const at::Tensor* p = plain(args[5]);
    if (!p || p->get_device() != device || p->scalar_type() != at::kLong) Py_RETURN_NONE;
    pos_dev = (const int64_t*)p->data_ptr();
  }
  const void *kr = t[0]->data_ptr(), *vr = t[1]->data_ptr();
  void *kz = k.data_ptr(), *vz = v.data_ptr();
  const int64_t stride = k.size(2);
  const int groups = (int)(k.size(0) * k.size(1));
  const ri_stream_t stream = current_stream();
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = ri_append_kv(kr, vr, kz, vz, stride, pos, pos_dev, groups, stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(status);
  END_HANDLE_TH_ERRORS
}

// A prepared call: the struct's address, the addresses it was made of and the numbers beside them.  The owner keeps the struct
// and the tensors alive.
struct Step {
  PyObject_HEAD
  const ri_decode_step_t* step;
  const ri_lru_t* lru;
  std::vector<const void*>* held;
  std::vector<long long>* numbers;
  at::ScalarType dtype;
  int device;
  int64_t queries;
};

bool addresses(PyObject* tensors, std::vector<const void*>& out) {
  const Py_ssize_t n = PyTuple_GET_SIZE(tensors);
  out.resize(n);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* o = PyTuple_GET_ITEM(tensors, i);
    const at::Tensor* t = o == Py_None ? nullptr : plain(o);
    if (o != Py_None && !t) return false;
    out[i] = t ? t->data_ptr() : nullptr;
  }
  return true;
}

// Step(step address, lru address or 0, centroids, tensors, numbers); tensors and numbers as `run` is given them
PyObject* step_new(PyTypeObject* type, PyObject* args, PyObject*) {
  HANDLE_TH_ERRORS
  unsigned long long step, lru;
  PyObject *centroids, *tensors, *numbers;
  if (!PyArg_ParseTuple(args, "KKOO!O!", &step, &lru, &centroids, &PyTuple_Type, &tensors, &PyTuple_Type, &numbers)) return nullptr;
  const at::Tensor* c = plain(centroids);
  if (!c) {
    PyErr_SetString(PyExc_TypeError, "Step: centroids are not a plain tensor");
    return nullptr;
  }
  std::vector<const void*> held;
  if (!addresses(tensors, held)) {
    PyErr_SetString(PyExc_TypeError, "Step: a buffer is not a plain tensor");
    return nullptr;
  }
  std::vector<long long> values;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(numbers); ++i) {
    values.push_back(PyLong_AsLongLong(PyTuple_GET_ITEM(numbers, i)));
    if (PyErr_Occurred()) return nullptr;
  }
  Step* self = (Step*)type->tp_alloc(type, 0);
  if (!self) return nullptr;
  self->step = (const ri_decode_step_t*)(uintptr_t)step;
  self->lru = (const ri_lru_t*)(uintptr_t)lru;
  self->held = new std::vector<const void*>(std::move(held));
  self->numbers = new std::vector<long long>(std::move(values));
  self->dtype = c->scalar_type();
  self->device = c->get_device();
  self->queries = (int64_t)self->step->BG * self->step->gs * 128;
  return (PyObject*)self;
  END_HANDLE_TH_ERRORS
}

void step_dealloc(PyObject* o) {
  Step* self = (Step*)o;
  delete self->held;
  delete self->numbers;
  PyTypeObject* type = Py_TYPE(o);
  type->tp_free(o);
  Py_DECREF(type);
}

// run(queries, static_len, out_shape, tensors, numbers): the output, None where the call is not this one's, or the status
PyObject* step_run(PyObject* o, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Step* self = (const Step*)o;
  if (n != 5 || !PyTuple_Check(args[2]) || !PyTuple_Check(args[3]) || !PyTuple_Check(args[4])) {
    PyErr_SetString(PyExc_TypeError, "run: queries, static_len, out_shape, tensors, numbers");
    return nullptr;
  }
  const at::Tensor* q = plain(args[0]);
  if (!q || at::impl::torch_function_mode_enabled() || q->get_device() != self->device || q->scalar_type() != self->dtype ||
      !q->is_contiguous() || q->numel() != self->queries)
    Py_RETURN_NONE;
  if ((size_t)PyTuple_GET_SIZE(args[3]) != self->held->size() || (size_t)PyTuple_GET_SIZE(args[4]) != self->numbers->size())
    Py_RETURN_NONE;
  for (size_t i = 0; i < self->held->size(); ++i) {
    PyObject* x = PyTuple_GET_ITEM(args[3], i);
    const at::Tensor* t = x == Py_None ? nullptr : plain(x);
    if ((x != Py_None && !t) || (t ? t->data_ptr() : nullptr) != (*self->held)[i]) Py_RETURN_NONE;
  }
  for (size_t i = 0; i < self->numbers->size(); ++i) {
    const long long x = PyLong_AsLongLong(PyTuple_GET_ITEM(args[4], i));
    if (x == -1 && PyErr_Occurred()) return nullptr;
    if (x != (*self->numbers)[i]) Py_RETURN_NONE;
  }
  const long static_len = PyLong_AsLong(args[1]);
  if (static_len == -1 && PyErr_Occurred()) return nullptr;
  int64_t shape[4], elements = 1;
  if (PyTuple_GET_SIZE(args[2]) != 4) Py_RETURN_NONE;
  for (int i = 0; i < 4; ++i) {
    shape[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(args[2], i));
    elements *= shape[i];
  }
  if (PyErr_Occurred()) return nullptr;
  if (elements != self->queries) Py_RETURN_NONE;
  at::Tensor out = at::empty(at::IntArrayRef(shape, 4), q->options().requires_grad(false));
  const void* qp = q->data_ptr();
  void* op = out.data_ptr();
  const ri_stream_t stream = current_stream();
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = self->lru ? ri_host_step(self->step, self->lru, qp, (int)static_len, op, stream)
                     : ri_decode_step(self->step, qp, (int)static_len, op, stream);
  Py_END_ALLOW_THREADS
  if (status) return PyLong_FromLong(status);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// plain contiguous device tensors of one type (null: not given); null where one is not
bool device_tensors(PyObject* const* args, int n, at::ScalarType dtype, const at::Tensor** out, bool optional = false) {
  for (int i = 0; i < n; ++i) {
    out[i] = nullptr;
    if (optional && args[i] == Py_None) continue;
    const at::Tensor* t = plain(args[i]);
    if (!t || !t->is_cuda() || t->scalar_type() != dtype || !t->is_contiguous()) return false;
    out[i] = t;
  }
  return true;
}
void* address(const at::Tensor* t) { return t ? t->data_ptr() : nullptr; }

bool integers(PyObject* const* args, int n, int64_t* out) {
  for (int i = 0; i < n; ++i) {
    if (!PyLong_Check(args[i])) return false;
    int over;
    out[i] = PyLong_AsLongLongAndOverflow(args[i], &over);
    if (over || out[i] < 0 || out[i] > INT32_MAX) return false;
  }
  return true;
}
// at least a b c elements (each within 32 bits)
bool holds(const at::Tensor* t, int64_t a, int64_t b, int64_t c) { return (__int128)t->numel() >= (__int128)a * b * c; }
bool half_type(const at::Tensor* t, at::ScalarType& dtype) {
  dtype = t ? t->scalar_type() : at::kFloat;
  return dtype == at::kHalf || dtype == at::kBFloat16;
}

// gemm_softmax(A, B, D, Softmax, Norm, Sum, batch_count, m, n, k, alpha, beta): status, or None where the wrapper has to look
PyObject* gemm_softmax(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const at::Tensor* t[6];
  at::ScalarType dtype;
  int64_t x[4];
  if (n != 12 || !half_type(plain(args[0]), dtype) || !device_tensors(args, 4, dtype, t) ||
      !device_tensors(args + 4, 2, at::kFloat, t + 4) || !integers(args + 6, 4, x))
    Py_RETURN_NONE;
  const int64_t bc = x[0], m = x[1], cols = x[2], k = x[3], tiles = (cols + 255) / 256;
  if (!holds(t[0], bc, m, k) || !holds(t[1], bc, cols, k) || !holds(t[2], bc, m, cols) || !holds(t[3], bc, m, cols) ||
      !holds(t[4], bc, tiles, m) || !holds(t[5], bc, tiles, m))
    Py_RETURN_NONE;
  const double alpha = PyFloat_AsDouble(args[10]), beta = PyFloat_AsDouble(args[11]);
  if (PyErr_Occurred()) {   // (float() takes more)
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  void* p[6];
  for (int i = 0; i < 6; ++i) p[i] = address(t[i]);
  const ri_stream_t stream = current_stream();
  auto* call = dtype == at::kHalf ? ri_batch_gemm_softmax_f16 : ri_batch_gemm_softmax;
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = call(p[0], p[1], p[2], (float*)p[4], (float*)p[5], p[3], (int)bc, (int)m, (int)cols, (int)k, (float)alpha, (float)beta,
                stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(status);
  END_HANDLE_TH_ERRORS
}

// gather_vectors(key_data, key_buffer, value_data, value_buffer, src_metadata, dst_metadata, data_offsets, groups, data_length,
// buffer_length, index_size, copy_start, copy_num): as above
PyObject* gather_vectors(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const at::Tensor* t[7];
  at::ScalarType dtype;
  int64_t x[6];
  if (n != 13 || !half_type(plain(args[0]), dtype) || !device_tensors(args, 6, dtype, t) ||
      !device_tensors(args + 6, 1, at::kLong, t + 6) || !integers(args + 7, 6, x))
    Py_RETURN_NONE;
  const int64_t groups = x[0], data = x[1], buffer = x[2];
  if (!holds(t[0], groups, data, 128) || !holds(t[1], groups, buffer, 128) || !holds(t[2], groups, data, 128) ||
      !holds(t[3], groups, buffer, 128) || !holds(t[4], groups, data, 1) || !holds(t[5], groups, buffer, 1) ||
      !holds(t[6], groups, x[3], 1))
    Py_RETURN_NONE;
  void* p[7];
  for (int i = 0; i < 7; ++i) p[i] = address(t[i]);
  const ri_stream_t stream = current_stream();
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = ri_gather_copy_vectors(p[0], p[1], p[2], p[3], p[4], p[5], (const int64_t*)p[6], (int)groups, (int)data, (int)buffer,
                                  (int)x[3], (int)x[4], (int)x[5], stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(status);
  END_HANDLE_TH_ERRORS
}

// flash(q, k, v, weight, previous_out, previous_lse, cache_seqlens, workspace, scale, return_lse): the output, or (output, lse);
// a status that is not zero; None as above.  q [BG, 1, gs, 128], k [BG, S, 1, 128]; the others by their elements.
PyObject* flash(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const at::Tensor *t[7], *ws;
  at::ScalarType dtype;
  if (n != 10 || at::impl::torch_function_mode_enabled() || !half_type(plain(args[0]), dtype) ||
      !device_tensors(args, 3, dtype, t) || !device_tensors(args + 3, 2, dtype, t + 3, true) ||
      !device_tensors(args + 5, 1, at::kFloat, t + 5, true) || !device_tensors(args + 6, 1, at::kInt, t + 6, true) ||
      !device_tensors(args + 7, 1, at::kByte, &ws) || (t[4] && !t[5]))
    Py_RETURN_NONE;
  const at::Tensor &q = *t[0], &k = *t[1];
  if (q.dim() != 4 || k.dim() != 4 || q.size(1) != 1 || q.size(3) != 128 || k.size(2) != 1) Py_RETURN_NONE;
  const int64_t BG = q.size(0), gs = q.size(2), S = k.size(1);
  if (!holds(t[1], BG, S, 128) || !holds(t[2], BG, S, 128) || (t[3] && !holds(t[3], BG, S, 1)) ||
      (t[4] && (!holds(t[4], BG, gs, 128) || !holds(t[5], BG, gs, 1))) || (t[6] && !holds(t[6], BG, 1, 1)))
    Py_RETURN_NONE;
  const double scale = PyFloat_AsDouble(args[8]);
  const int with_lse = PyObject_IsTrue(args[9]);
  if (PyErr_Occurred()) return nullptr;
  at::Tensor out = at::empty_like(q), lse;
  if (with_lse) lse = at::empty({BG, gs}, q.options().dtype(at::kFloat).requires_grad(false));
  void* p[7];
  for (int i = 0; i < 7; ++i) p[i] = address(t[i]);
  void *op = out.data_ptr(), *lp = with_lse ? lse.data_ptr() : nullptr, *wp = ws->data_ptr();
  const size_t bytes = (size_t)ws->numel();
  const ri_stream_t stream = current_stream();
  auto* call = dtype == at::kHalf ? ri_weighted_flash_decoding_f16 : ri_weighted_flash_decoding;
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = call(p[0], p[1], p[2], p[3], (const int32_t*)p[6], p[4], (const float*)p[5], op, (float*)lp, (int)BG, (int)gs, (int)S,
                (int)S, (float)scale, wp, bytes, stream);
  Py_END_ALLOW_THREADS
  if (status) return PyLong_FromLong(status);
  if (!with_lse) return THPVariable_Wrap(std::move(out));
  PyObject *a = THPVariable_Wrap(std::move(out)), *b = THPVariable_Wrap(std::move(lse));
  PyObject* both = a && b ? PyTuple_Pack(2, a, b) : nullptr;
  Py_XDECREF(a);
  Py_XDECREF(b);
  return both;
  END_HANDLE_TH_ERRORS
}

PyMethodDef step_methods[] = {{"run", (PyCFunction)(void (*)(void))step_run, METH_FASTCALL, nullptr},
                              {nullptr, nullptr, 0, nullptr}};
PyType_Slot step_slots[] = {{Py_tp_new, (void*)step_new},
                            {Py_tp_dealloc, (void*)step_dealloc},
                            {Py_tp_methods, (void*)step_methods},
                            {0, nullptr}};
PyType_Spec step_spec = {"_step_calls.Step", sizeof(Step), 0, Py_TPFLAGS_DEFAULT, step_slots};

PyMethodDef methods[] = {{"append", (PyCFunction)(void (*)(void))append, METH_FASTCALL, nullptr},
                         {"gemm_softmax", (PyCFunction)(void (*)(void))gemm_softmax, METH_FASTCALL, nullptr},
                         {"gather_vectors", (PyCFunction)(void (*)(void))gather_vectors, METH_FASTCALL, nullptr},
                         {"flash", (PyCFunction)(void (*)(void))flash, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_step_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__step_calls() {
  PyObject* m = PyModule_Create(&module);
  PyObject* type = m ? PyType_FromSpec(&step_spec) : nullptr;
  if (!type || PyModule_AddObject(m, "Step", type) < 0) return nullptr;
  return m;
}

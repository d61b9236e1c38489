// The Python mirror's call path in native code: ruy_amd.api.mul hands its
// objects over here, where their fields are gathered into the plain structs of
// c_api.h and ruyamd_mul is called. Filling four ctypes structures field by
// field and calling through ctypes took 2.4 us of a call whose launch takes
// 2.4 and whose kernel, for the smallest products, takes no more than both.
//
// Fields are read from the instances' dictionaries, where the classes of
// api.py keep them; an instance that does not have them there (a subclass with
// properties, say) is left to the Python code (kNotHandled).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <cstring>
#include <initializer_list>

#include "ruy_amd/c_api.h"

namespace {

using MulFunction = int (*)(ruyamd_ctx*, const ruyamd_mat*, const ruyamd_mat*, const ruyamd_mul_params*,
                            const ruyamd_mat*);
MulFunction mul_function = nullptr;
PyTypeObject* matrix_type = nullptr;
PyTypeObject* layout_type = nullptr;
PyTypeObject* params_type = nullptr;

#define RUYAMD_NAMES(X)                                                                                        \
  X(dtype) X(data) X(layout) X(zero_point) X(cache_policy) X(rows) X(cols) X(stride) X(order) X(data_ptr)      \
  X(ctypes) X(bias) X(_perchannel) X(_mf) X(_me) X(_mf_pc) X(_me_pc) X(clamp_min) X(clamp_max) X(accum_dtype) \
  X(dst_dtype) X(channel_dimension) X(_rounding_log2)
#define RUYAMD_DECLARE(name) PyObject* name_##name;
RUYAMD_NAMES(RUYAMD_DECLARE)

// What a step of the conversion came to.
enum Outcome { kDone, kNotHandled, kError };

// A reference of our own. Asking a buffer for its address or a value for its
// float may run any code, also code that takes that object out of the instance
// it was found in, or the instance's dictionary away.
class Ref {
 public:
  explicit Ref(PyObject* borrowed) : p_(borrowed) { Py_XINCREF(p_); }
  ~Ref() { Py_XDECREF(p_); }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
  operator PyObject*() const { return p_; }

 private:
  PyObject* p_;
};

// A field of an instance; null if it is not in the dictionary (or there is none).
Ref Field(PyObject* dict, PyObject* name) { return Ref(dict ? PyDict_GetItemWithError(dict, name) : nullptr); }

Ref DictOf(PyObject* object) {
  PyObject** p = _PyObject_GetDictPtr(object);
  return Ref(p ? *p : nullptr);
}

// Only Python integers are taken here (as ctypes does, bits beyond the field's
// are dropped); anything else is left to the Python code.
bool Integer(PyObject* dict, PyObject* name, uint64_t* out) {
  const Ref v = Field(dict, name);
  if (!v || !PyLong_Check(v)) return false;
  *out = PyLong_AsUnsignedLongLongMask(v);
  return true;
}

// api._address: None, an integer, a tensor or an array.
Outcome Address(PyObject* buffer, void** out) {
  if (buffer == Py_None) {
    *out = nullptr;
    return kDone;
  }
  if (PyLong_Check(buffer)) {
    *out = reinterpret_cast<void*>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLongMask(buffer)));
    return kDone;
  }
  PyObject* value = PyObject_CallMethodNoArgs(buffer, name_data_ptr);
  if (!value) {
    if (!PyErr_ExceptionMatches(PyExc_AttributeError)) return kError;
    PyErr_Clear();
    PyObject* ctypes = PyObject_GetAttr(buffer, name_ctypes);
    if (!ctypes) {
      PyErr_Clear();
      return kNotHandled;  // (the Python code raises)
    }
    value = PyObject_GetAttr(ctypes, name_data);
    Py_DECREF(ctypes);
    if (!value) return kError;
  }
  if (!PyLong_Check(value)) {
    Py_DECREF(value);
    return kNotHandled;
  }
  *out = reinterpret_cast<void*>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLongMask(value)));
  Py_DECREF(value);
  return kDone;
}

Outcome Matrix(PyObject* object, ruyamd_mat* m) {
  if (Py_TYPE(object) != matrix_type) return kNotHandled;
  const Ref dict = DictOf(object);
  const Ref layout = Field(dict, name_layout);
  const Ref data = Field(dict, name_data);
  if (!layout || !data || Py_TYPE(layout) != layout_type) return kNotHandled;
  const Ref shape = DictOf(layout);
  uint64_t rows, cols, stride, order, zero_point, dtype, policy;
  if (!Integer(shape, name_rows, &rows) || !Integer(shape, name_cols, &cols) ||
      !Integer(shape, name_stride, &stride) || !Integer(shape, name_order, &order) ||
      !Integer(dict, name_zero_point, &zero_point) || !Integer(dict, name_dtype, &dtype) ||
      !Integer(dict, name_cache_policy, &policy))
    return kNotHandled;
  m->rows = static_cast<int32_t>(rows);
  m->cols = static_cast<int32_t>(cols);
  m->stride = static_cast<int32_t>(stride);
  m->zero_point = static_cast<int32_t>(zero_point);
  m->order = static_cast<uint8_t>(order);
  m->dtype = static_cast<uint8_t>(dtype);
  m->cache_policy = static_cast<uint8_t>(policy);
  m->reserved = 0;
  return Address(data, &m->data);
}

Outcome Params(PyObject* object, ruyamd_mul_params* p, uint64_t* dst_dtype) {
  if (Py_TYPE(object) != params_type) return kNotHandled;
  const Ref dict = DictOf(object);
  const Ref perchannel = Field(dict, name__perchannel);
  uint64_t accum, channel, rounding;
  if (!perchannel || !PyBool_Check(perchannel) || !Integer(dict, name_accum_dtype, &accum) ||
      !Integer(dict, name_dst_dtype, dst_dtype) || !Integer(dict, name_channel_dimension, &channel) ||
      !Integer(dict, name__rounding_log2, &rounding))
    return kNotHandled;
  std::memset(p, 0, sizeof(*p));
  p->accum_dtype = static_cast<uint8_t>(accum);
  p->channel_dimension = static_cast<uint8_t>(channel);
  p->perchannel_buffers_capacity_rounding_log2 = static_cast<uint8_t>(rounding);
  const Ref clamp_min = Field(dict, name_clamp_min);
  const Ref clamp_max = Field(dict, name_clamp_max);
  if (!clamp_min || !clamp_max) return kNotHandled;
  p->clamp_min = PyFloat_AsDouble(clamp_min);
  p->clamp_max = PyFloat_AsDouble(clamp_max);
  if (PyErr_Occurred()) return kError;
  const Ref bias = Field(dict, name_bias);
  if (!bias) return kNotHandled;
  void* address = nullptr;
  if (Outcome o = Address(bias, &address)) return o;
  p->bias = address;
  if (perchannel == Py_True) {
    const Ref mf = Field(dict, name__mf_pc);
    const Ref me = Field(dict, name__me_pc);
    if (!mf || !me) return kNotHandled;
    if (Outcome o = Address(mf, &address)) return o;
    p->multiplier_fixedpoint_perchannel = static_cast<const int32_t*>(address);
    if (Outcome o = Address(me, &address)) return o;
    p->multiplier_exponent_perchannel = static_cast<const int32_t*>(address);
  } else {
    uint64_t mf, me;
    if (!Integer(dict, name__mf, &mf) || !Integer(dict, name__me, &me)) return kNotHandled;
    p->multiplier_fixedpoint = static_cast<int32_t>(mf);
    p->multiplier_exponent = static_cast<int32_t>(me);
  }
  return kDone;
}

// mul(lhs, rhs, mul_params, context address, dst): the return code, or None if
// the objects are not handled here.
PyObject* Mul(PyObject*, PyObject* const* args, Py_ssize_t count) {
  if (count != 5 || !mul_function) {
    PyErr_SetString(PyExc_TypeError, "mul(lhs, rhs, mul_params, context address, dst)");
    return nullptr;
  }
  ruyamd_mat lhs, rhs, dst;
  ruyamd_mul_params params;
  uint64_t dst_dtype = 0;
  Outcome o = Params(args[2], &params, &dst_dtype);
  if (o == kDone) o = Matrix(args[0], &lhs);
  if (o == kDone) o = Matrix(args[1], &rhs);
  if (o == kDone) o = Matrix(args[4], &dst);
  if (o == kError) return nullptr;
  if (o == kNotHandled || dst_dtype != dst.dtype || !PyLong_Check(args[3])) {
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
  }
  ruyamd_ctx* ctx = reinterpret_cast<ruyamd_ctx*>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLongMask(args[3])));
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = mul_function(ctx, &lhs, &rhs, &params, &dst);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// bind(address of ruyamd_mul, Matrix, Layout, MulParams)
PyObject* Bind(PyObject*, PyObject* args) {
  unsigned long long address = 0;
  PyObject *matrix, *layout, *params;
  if (!PyArg_ParseTuple(args, "KO!O!O!", &address, &PyType_Type, &matrix, &PyType_Type, &layout, &PyType_Type, &params))
    return nullptr;
  mul_function = reinterpret_cast<MulFunction>(static_cast<uintptr_t>(address));
  for (PyObject* t : {matrix, layout, params}) Py_INCREF(t);
  matrix_type = reinterpret_cast<PyTypeObject*>(matrix);
  layout_type = reinterpret_cast<PyTypeObject*>(layout);
  params_type = reinterpret_cast<PyTypeObject*>(params);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"mul", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(Mul)), METH_FASTCALL, nullptr},
    {"bind", Bind, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() {
#define RUYAMD_INTERN(name) \
  if (!(name_##name = PyUnicode_InternFromString(#name))) return nullptr;
  RUYAMD_NAMES(RUYAMD_INTERN)
  return PyModule_Create(&module);
}

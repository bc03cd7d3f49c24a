// The host path of mograd_amd in native code: the graph's vertices (Layout, Node), the pool buffers,
// the calls into libmograd_hip, the rewriting pass and the evaluation of a graph.
//
// A small model's step is as long as its host work: a lazily built graph is some 260 nodes per
// four transformer layers, each created, ordered, matched, rewritten and evaluated once, and each
// kernel costs 2.3 us of the HIP runtime before anything of ours.  In Python the same path took
// 3.1 ms for such a step on the box (of which 0.3 ms are the launches); see the figures at the
// functions below.  What is not common (strided operands, ops a training step does not
// contain) stays with the Python exec functions, which evaluate() calls where its own
// forms do not apply.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

#include <dlfcn.h>

#include <cstdint>
#include <cstring>
#include <new>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

#include "mograd_hip.h"

namespace {

// ------------------------------------------------------------------------------------------
// References
// ------------------------------------------------------------------------------------------

struct Ref {  // owned reference
  PyObject* p = nullptr;
  Ref() = default;
  explicit Ref(PyObject* o) : p(o) {}
  Ref(Ref&& o) noexcept : p(o.p) { o.p = nullptr; }
  Ref& operator=(Ref&& o) noexcept {
    std::swap(p, o.p);
    return *this;
  }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
  ~Ref() { Py_XDECREF(p); }
  static Ref to(PyObject* o) {  // a further reference to `o`
    Py_XINCREF(o);
    return Ref(o);
  }
  PyObject* release() {
    PyObject* o = p;
    p = nullptr;
    return o;
  }
  explicit operator bool() const { return p != nullptr; }
};

PyObject* str_(const char* s) { return PyUnicode_InternFromString(s); }

// Names used as attribute and dictionary keys.
struct Names {
  PyObject *index, *eps, *has_bias, *accumulate, *relu_mask, *scale, *is_causal, *stream, *pending, *func, *pat, *op_type,
      *srcs, *subst, *uses, *origin, *consumers, *rules;
} N;

PyObject* g_mograd_error = nullptr;   // MogradError(status, message)
PyObject* g_void_p = nullptr;         // ctypes.c_void_p
PyTypeObject* g_buffer_type = nullptr;  // AnyBuffer
PyTypeObject* g_layout_type = nullptr;  // runtime.Layout
PyObject* g_fallbacks = nullptr;      // name -> ctypes wrapper

// ------------------------------------------------------------------------------------------
// libmograd_hip
// ------------------------------------------------------------------------------------------

#define MG_FUNCTIONS(X)                                                                                                 \
  X(mg_pool_free) X(mg_fill) X(mg_copy_device) X(mg_layer_norm_fwd) X(mg_layer_norm_fwd_stats) X(mg_layer_norm_bwd)       \
  X(mg_layer_norm_bwd_stats) X(mg_layer_norm_bwd_stats_add) X(mg_cross_entropy) X(mg_cross_entropy_grad)                  \
  X(mg_cross_entropy_ids) X(mg_cross_entropy_grad_ids) X(mg_cross_entropy_fused_ids) X(mg_cross_entropy_fused_ids_noalloc) \
  X(mg_cross_entropy_fused) X(mg_matmul) X(mg_matmul_bt) X(mg_matmul_bias_bt) X(mg_linear_bwd) X(mg_matmul_bt_add)        \
  X(mg_matmul_bias_relu_bt) X(mg_linear_bwd_fused) X(mg_sum_axis) X(mg_relu_grad) X(mg_softmax) X(mg_softmax_grad)        \
  X(mg_argmax_axis) X(mg_adam_step) X(mg_sgd_step) X(mg_add) X(mg_relu) X(mg_cast) X(mg_gather) X(mg_scatter_add)         \
  X(mg_finish_deferred) X(mg_linear_bwd_deferred) X(mg_layer_norm_bwd_stats_deferred) X(mg_linear_bwd_layer_norm_bwd)     \
  X(mg_scatter_add_deferred) X(mg_flash_attn_fwd) X(mg_flash_attn_bwd) X(mg_flash_attn_fwd_bshd)                          \
  X(mg_flash_attn_bwd_bshd) X(mg_flash_attn_fwd_packed) X(mg_flash_attn_bwd_packed)

struct Lib {
#define X(f) decltype(&::f) f = nullptr;
  MG_FUNCTIONS(X)
#undef X
  decltype(&::mg_pool_alloc) pool_alloc = nullptr;
  decltype(&::mg_last_error) last_error = nullptr;
} L;

// Sets MogradError(status, the library's message).
void raise_status(int status) {
  Ref e(PyObject_CallFunction(g_mograd_error, "is", status, L.last_error ? L.last_error() : ""));
  if (e) PyErr_SetObject(g_mograd_error, e.p);
}
void raise_invalid(const char* message) {
  Ref e(PyObject_CallFunction(g_mograd_error, "is", 1, message));
  if (e) PyErr_SetObject(g_mograd_error, e.p);
}

// A call without the interpreter lock, as ctypes makes it.
template <class F>
int unlocked(F&& f) {
  int rc;
  Py_BEGIN_ALLOW_THREADS rc = f();
  Py_END_ALLOW_THREADS return rc;
}

bool pointer_of(PyObject* o, void** out) {
  if (o == Py_None) {
    *out = nullptr;
    return true;
  }
  if (PyLong_Check(o)) {
    *out = PyLong_AsVoidPtr(o);
    if (*out == nullptr && PyErr_Occurred()) return PyErr_Clear(), false;
    return true;
  }
  if (reinterpret_cast<PyObject*>(Py_TYPE(o)) != g_void_p) return false;
  Py_buffer view;
  if (PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) != 0) return PyErr_Clear(), false;
  std::memcpy(out, view.buf, sizeof(void*));
  PyBuffer_Release(&view);
  return true;
}

template <class T>
bool convert(PyObject* o, T* out) {
  if constexpr (std::is_floating_point_v<T>) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) return PyErr_Clear(), false;
    *out = static_cast<T>(v);
    return true;
  } else if constexpr (std::is_pointer_v<T>) {
    void* p = nullptr;
    if (!pointer_of(o, &p)) return false;
    *out = static_cast<T>(p);
    return true;
  } else {
    if (!PyLong_Check(o)) return false;
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) return PyErr_Clear(), false;
    *out = static_cast<T>(v);
    return static_cast<long long>(*out) == v;
  }
}

template <class... A, size_t... I>
bool convert_all(PyObject* const* args, std::tuple<A...>& t, std::index_sequence<I...>) {
  return (convert(args[I], &std::get<I>(t)) && ...);
}

// lib.mg_xxx(...) from Python: anything the conversion above does not take goes to ctypes.
template <class... A>
PyObject* call_entry(const char* name, int (*fn)(A...), PyObject* const* args, Py_ssize_t n) {
  std::tuple<A...> t;
  if (fn && n == static_cast<Py_ssize_t>(sizeof...(A)) && convert_all(args, t, std::index_sequence_for<A...>{})) {
    const int rc = unlocked([&] { return std::apply(fn, t); });
    if (rc != 0) return raise_status(rc), nullptr;
    return PyLong_FromLong(0);
  }
  PyObject* fallback = PyDict_GetItemString(g_fallbacks, name);
  if (!fallback) return PyErr_Format(PyExc_RuntimeError, "%s is not available", name), nullptr;
  return PyObject_Vectorcall(fallback, args, static_cast<size_t>(n), nullptr);
}

#define X(f)                                                                                        \
  PyObject* py_##f(PyObject*, PyObject* const* args, Py_ssize_t n) { return call_entry(#f, L.f, args, n); }
MG_FUNCTIONS(X)
#undef X

// ------------------------------------------------------------------------------------------
// Layout: dims, strides (elements) and base offset; immutable
// ------------------------------------------------------------------------------------------

struct LayoutObj {
  PyObject_HEAD PyObject* dims;  // tuples of int
  PyObject* strides;
  long long base_offset, numel;
  bool contiguous;
};
PyTypeObject LayoutType = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyObject* int_tuple(PyObject* seq) {  // a new tuple of ints from a tuple or list
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
  PyObject* t = PyTuple_New(n);
  if (!t) return nullptr;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* o = PySequence_Fast_GET_ITEM(seq, i);
    PyObject* v = PyLong_CheckExact(o) ? (Py_INCREF(o), o) : PyNumber_Long(o);
    if (!v) return Py_DECREF(t), nullptr;
    PyTuple_SET_ITEM(t, i, v);
  }
  return t;
}

PyObject* row_major(PyObject* dims, long long* numel) {
  const Py_ssize_t n = PyTuple_GET_SIZE(dims);
  PyObject* t = PyTuple_New(n);
  if (!t) return nullptr;
  long long s = 1;
  for (Py_ssize_t i = n - 1; i >= 0; --i) {
    PyObject* v = PyLong_FromLongLong(s);
    if (!v) return Py_DECREF(t), nullptr;
    PyTuple_SET_ITEM(t, i, v);
    s *= PyLong_AsLongLong(PyTuple_GET_ITEM(dims, i));
  }
  *numel = s;
  if (PyErr_Occurred()) return Py_DECREF(t), nullptr;
  return t;
}

// Takes over `dims`; `strides` null: row-major, else taken over.
PyObject* layout_make(PyTypeObject* type, PyObject* dims, PyObject* strides, long long base) {
  long long numel = 0;
  Ref d(dims), s(strides), rm(dims ? row_major(dims, &numel) : nullptr);
  if (!rm) return nullptr;
  LayoutObj* o = reinterpret_cast<LayoutObj*>(type->tp_alloc(type, 0));
  if (!o) return nullptr;
  o->contiguous = !s || PyObject_RichCompareBool(s.p, rm.p, Py_EQ) == 1;
  o->dims = d.release();
  o->strides = s ? s.release() : rm.release();
  o->base_offset = base;
  o->numel = numel;
  return reinterpret_cast<PyObject*>(o);
}

PyObject* layout_new(PyTypeObject* type, PyObject* args, PyObject* kw) {
  PyObject* strides = nullptr;
  PyObject* base = nullptr;
  if (kw) {
    PyObject *k, *v;
    Py_ssize_t pos = 0;
    while (PyDict_Next(kw, &pos, &k, &v)) {
      if (PyUnicode_CompareWithASCIIString(k, "strides") == 0) strides = v;
      else if (PyUnicode_CompareWithASCIIString(k, "base_offset") == 0) base = v;
      else return PyErr_Format(PyExc_TypeError, "Layout() got an unexpected keyword argument '%U'", k), nullptr;
    }
  }
  PyObject* shape = args;
  if (PyTuple_GET_SIZE(args) == 1) {
    PyObject* only = PyTuple_GET_ITEM(args, 0);
    if (PyTuple_Check(only) || PyList_Check(only)) shape = only;
  }
  Ref dims(int_tuple(shape));
  if (!dims) return nullptr;
  Ref st;
  if (strides && strides != Py_None) {
    Ref fast(PySequence_Fast(strides, "strides must be a sequence"));
    if (!fast) return nullptr;
    st = Ref(int_tuple(fast.p));
    if (!st) return nullptr;
    if (PyTuple_GET_SIZE(st.p) != PyTuple_GET_SIZE(dims.p)) {
      PyErr_SetString(PyExc_ValueError, "strides rank differs from shape rank");
      return nullptr;
    }
  }
  long long b = 0;
  if (base) {
    Ref as_int(PyNumber_Long(base));
    if (!as_int) return nullptr;
    b = PyLong_AsLongLong(as_int.p);
    if (b == -1 && PyErr_Occurred()) return nullptr;
  }
  return layout_make(type, dims.release(), st.release(), b);
}

void layout_dealloc(PyObject* self) {
  LayoutObj* o = reinterpret_cast<LayoutObj*>(self);
  Py_XDECREF(o->dims);
  Py_XDECREF(o->strides);
  Py_TYPE(self)->tp_free(self);  // (a Python subclass's own deallocator releases its type)
}

LayoutObj* as_layout(PyObject* o) { return reinterpret_cast<LayoutObj*>(o); }
bool is_layout(PyObject* o) { return PyObject_TypeCheck(o, &LayoutType); }
Py_ssize_t rank_of(const LayoutObj* l) { return PyTuple_GET_SIZE(l->dims); }
long long dim_of(const LayoutObj* l, Py_ssize_t i) { return PyLong_AsLongLong(PyTuple_GET_ITEM(l->dims, i < 0 ? i + rank_of(l) : i)); }
long long last_dim(const LayoutObj* l) { return rank_of(l) ? dim_of(l, -1) : 0; }
long long stride_of(const LayoutObj* l, Py_ssize_t i) {
  return PyLong_AsLongLong(PyTuple_GET_ITEM(l->strides, i < 0 ? i + rank_of(l) : i));
}

PyObject* tuple_item(PyObject* tuple, PyObject* const* args, Py_ssize_t n, PyObject* kwnames, const char* who) {
  PyObject* idx = nullptr;
  if (n == 1 && !kwnames) idx = args[0];
  else if (n == 0 && kwnames && PyTuple_GET_SIZE(kwnames) == 1 &&
           PyUnicode_CompareWithASCIIString(PyTuple_GET_ITEM(kwnames, 0), "idx") == 0)
    idx = args[0];
  else if (n > 0 || kwnames) return PyErr_Format(PyExc_TypeError, "%s() takes one argument, idx", who), nullptr;
  if (!idx || idx == Py_None) return Py_INCREF(tuple), tuple;
  return PyObject_GetItem(tuple, idx);
}
PyObject* layout_shape(PyObject* self, PyObject* const* args, Py_ssize_t n, PyObject* kw) {
  return tuple_item(as_layout(self)->dims, args, n, kw, "shape");
}
PyObject* layout_stride(PyObject* self, PyObject* const* args, Py_ssize_t n, PyObject* kw) {
  return tuple_item(as_layout(self)->strides, args, n, kw, "stride");
}
PyObject* layout_rank(PyObject* self, PyObject*) { return PyLong_FromSsize_t(rank_of(as_layout(self))); }
PyObject* layout_numel(PyObject* self, PyObject*) { return PyLong_FromLongLong(as_layout(self)->numel); }
PyObject* layout_is_contiguous(PyObject* self, PyObject*) { return PyBool_FromLong(as_layout(self)->contiguous); }
PyObject* layout_as_contiguous(PyObject* self, PyObject*) {
  LayoutObj* l = as_layout(self);
  if (l->contiguous && l->base_offset == 0) return Py_INCREF(self), self;  // immutable
  Py_INCREF(l->dims);
  return layout_make(Py_TYPE(self), l->dims, nullptr, 0);
}
PyObject* layout_richcompare(PyObject* a, PyObject* b, int op) {
  if ((op != Py_EQ && op != Py_NE) || !is_layout(a) || !is_layout(b)) Py_RETURN_NOTIMPLEMENTED;
  LayoutObj *x = as_layout(a), *y = as_layout(b);
  bool same = a == b || (x->base_offset == y->base_offset && PyObject_RichCompareBool(x->dims, y->dims, Py_EQ) == 1 &&
                         PyObject_RichCompareBool(x->strides, y->strides, Py_EQ) == 1);
  return PyBool_FromLong(same == (op == Py_EQ));
}
Py_hash_t layout_hash(PyObject* self) {
  LayoutObj* l = as_layout(self);
  Ref t(Py_BuildValue("(OOL)", l->dims, l->strides, l->base_offset));
  return t ? PyObject_Hash(t.p) : -1;
}
PyObject* layout_repr(PyObject* self) {
  LayoutObj* l = as_layout(self);
  return PyUnicode_FromFormat("Layout(dims=%R, strides=%R, base_offset=%lld)", l->dims, l->strides, l->base_offset);
}
PyMemberDef layout_members[] = {{"dims", T_OBJECT, offsetof(LayoutObj, dims), READONLY, nullptr},
                                {"strides", T_OBJECT, offsetof(LayoutObj, strides), READONLY, nullptr},
                                {"base_offset", T_LONGLONG, offsetof(LayoutObj, base_offset), READONLY, nullptr},
                                {nullptr, 0, 0, 0, nullptr}};
#define FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f))
PyMethodDef layout_methods[] = {
    {"rank", layout_rank, METH_NOARGS, nullptr},
    {"shape", FAST(layout_shape), METH_FASTCALL | METH_KEYWORDS, nullptr},
    {"stride", FAST(layout_stride), METH_FASTCALL | METH_KEYWORDS, nullptr},
    {"numel", layout_numel, METH_NOARGS, nullptr},
    {"is_contiguous", layout_is_contiguous, METH_NOARGS, nullptr},
    {"as_contiguous", layout_as_contiguous, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};

// ------------------------------------------------------------------------------------------
// Node: a graph vertex; compared and hashed by identity
// ------------------------------------------------------------------------------------------

struct NodeObj {
  PyObject_HEAD PyObject* op_type;
  PyObject* node_layout;
  PyObject* node_dtype;
  PyObject* srcs;        // a list or tuple, as a rule
  PyObject* node_attrs;  // a dict, as a rule
  PyObject* bufs;        // None, or a sequence of buffers
  PyObject* dict;        // attributes that a program adds
  PyObject* weakrefs;
  uint64_t mark;         // the last walk that saw this node
  uint32_t position;     // its place in that walk (between steps that keep the interpreter lock)
};
PyTypeObject NodeType = {PyVarObject_HEAD_INIT(nullptr, 0)};
uint64_t g_epoch = 0;

NodeObj* as_node(PyObject* o) { return reinterpret_cast<NodeObj*>(o); }
bool is_node(PyObject* o) { return PyObject_TypeCheck(o, &NodeType); }

PyObject* new_ref(PyObject* o) { return Py_INCREF(o), o; }

PyObject* node_new(PyTypeObject* type, PyObject*, PyObject*) {
  NodeObj* n = reinterpret_cast<NodeObj*>(type->tp_alloc(type, 0));
  if (!n) return nullptr;
  for (PyObject** field : {&n->op_type, &n->node_layout, &n->node_dtype, &n->srcs, &n->node_attrs, &n->bufs}) *field = new_ref(Py_None);
  n->dict = n->weakrefs = nullptr;
  n->mark = 0, n->position = 0;
  return reinterpret_cast<PyObject*>(n);
}
// Sources as they are kept: a list or tuple itself, any other sequence as a list.
PyObject* sources_of(PyObject* o) {
  if (PyList_Check(o) || PyTuple_Check(o)) return new_ref(o);
  PyObject* list = PySequence_List(o);
  return list ? list : (PyErr_Clear(), new_ref(o));
}
// Takes over srcs and attrs (null: an empty list, an empty dict).
bool node_fill(PyObject* self, PyObject* op, PyObject* layout, PyObject* dtype, PyObject* srcs, PyObject* attrs, PyObject* bufs) {
  Ref s(srcs ? srcs : PyList_New(0)), a(attrs ? attrs : PyDict_New());
  if (!s || !a) return false;
  NodeObj* n = as_node(self);
  Py_SETREF(n->op_type, new_ref(op));
  Py_SETREF(n->node_layout, new_ref(layout));
  Py_SETREF(n->node_dtype, new_ref(dtype));
  Py_SETREF(n->srcs, s.release());
  Py_SETREF(n->node_attrs, a.release());
  Py_SETREF(n->bufs, new_ref(bufs));
  return true;
}
PyObject* node_make(PyObject* op, PyObject* layout, PyObject* dtype, PyObject* srcs, PyObject* attrs, PyObject* bufs) {
  Ref n(node_new(&NodeType, nullptr, nullptr));
  if (!n) return Py_XDECREF(srcs), Py_XDECREF(attrs), nullptr;
  return node_fill(n.p, op, layout, dtype, srcs, attrs, bufs) ? n.release() : nullptr;
}
int node_init(PyObject* self, PyObject* args, PyObject* kw) {
  static const char* names[] = {"op_type", "node_layout", "node_dtype", "srcs", "node_attrs", "bufs", nullptr};
  PyObject *op, *layout, *dtype, *srcs = nullptr, *attrs = nullptr, *bufs = Py_None;
  if (!kw && PyTuple_GET_SIZE(args) >= 3 && PyTuple_GET_SIZE(args) <= 6) {
    const Py_ssize_t n = PyTuple_GET_SIZE(args);
    op = PyTuple_GET_ITEM(args, 0), layout = PyTuple_GET_ITEM(args, 1), dtype = PyTuple_GET_ITEM(args, 2);
    if (n > 3) srcs = PyTuple_GET_ITEM(args, 3);
    if (n > 4) attrs = PyTuple_GET_ITEM(args, 4);
    if (n > 5) bufs = PyTuple_GET_ITEM(args, 5);
  } else if (!PyArg_ParseTupleAndKeywords(args, kw, "OOO|OOO:Node", const_cast<char**>(names), &op, &layout, &dtype, &srcs,
                                          &attrs, &bufs)) {
    return -1;
  }
  Py_XINCREF(attrs);
  return node_fill(self, op, layout, dtype, srcs ? sources_of(srcs) : nullptr, attrs, bufs) ? 0 : -1;
}
int node_traverse(PyObject* self, visitproc visit, void* arg) {
  NodeObj* n = as_node(self);
  for (PyObject* o : {n->op_type, n->node_layout, n->node_dtype, n->srcs, n->node_attrs, n->bufs, n->dict}) Py_VISIT(o);
  return 0;
}
int node_clear(PyObject* self) {  // (what a cycle can run through; the other fields go with the node)
  NodeObj* n = as_node(self);
  for (PyObject** field : {&n->srcs, &n->node_attrs, &n->bufs}) Py_SETREF(*field, new_ref(Py_None));
  Py_CLEAR(n->dict);
  return 0;
}
void node_dealloc(PyObject* self) {
  PyObject_GC_UnTrack(self);
  Py_TRASHCAN_BEGIN(self, node_dealloc)  // a deep graph is freed without deep recursion
  NodeObj* n = as_node(self);
  if (n->weakrefs) PyObject_ClearWeakRefs(self);
  for (PyObject** field : {&n->op_type, &n->node_layout, &n->node_dtype, &n->srcs, &n->node_attrs, &n->bufs, &n->dict})
    Py_CLEAR(*field);
  Py_TYPE(self)->tp_free(self);
  Py_TRASHCAN_END
}
// copy, deepcopy, pickle: (fields, attributes) handed to a new node of the same type.
PyObject* node_reduce(PyObject* self, PyObject*) {
  NodeObj* n = as_node(self);
  Ref copyreg(PyImport_ImportModule("copyreg")), make(copyreg ? PyObject_GetAttrString(copyreg.p, "__newobj__") : nullptr);
  if (!make) return nullptr;
  return Py_BuildValue("(O(O)((OOOOOO)O))", make.p, reinterpret_cast<PyObject*>(Py_TYPE(self)), n->op_type, n->node_layout,
                       n->node_dtype, n->srcs, n->node_attrs, n->bufs, n->dict ? n->dict : Py_None);
}
PyObject* node_setstate(PyObject* self, PyObject* state) {
  PyObject *op, *layout, *dtype, *srcs, *attrs, *bufs, *extra;
  if (!PyArg_ParseTuple(state, "(OOOOOO)O:__setstate__", &op, &layout, &dtype, &srcs, &attrs, &bufs, &extra)) return nullptr;
  if (!node_fill(self, op, layout, dtype, sources_of(srcs), new_ref(attrs), bufs)) return nullptr;
  if (extra != Py_None) {
    Ref dict(PyObject_GetAttrString(self, "__dict__"));
    if (!dict || PyDict_Update(dict.p, extra) != 0) return nullptr;
  }
  Py_RETURN_NONE;
}
PyObject* node_get(PyObject* self, void* offset) {
  return new_ref(*reinterpret_cast<PyObject**>(reinterpret_cast<char*>(self) + reinterpret_cast<uintptr_t>(offset)));
}
int node_set(PyObject* self, PyObject* value, void* offset) {
  if (!value) return PyErr_SetString(PyExc_AttributeError, "a Node's own fields cannot be deleted"), -1;
  PyObject** field = reinterpret_cast<PyObject**>(reinterpret_cast<char*>(self) + reinterpret_cast<uintptr_t>(offset));
  PyObject* old = *field;
  *field = field == &as_node(self)->srcs ? sources_of(value) : new_ref(value);
  Py_DECREF(old);
  return 0;
}
PyObject* node_layout(PyObject* self, PyObject*) {
  PyObject* o = as_node(self)->node_layout;
  return Py_INCREF(o), o;
}
PyObject* node_dtype(PyObject* self, PyObject*) {
  PyObject* o = as_node(self)->node_dtype;
  return Py_INCREF(o), o;
}
PyObject* node_attrs(PyObject* self, PyObject*) {
  PyObject* o = as_node(self)->node_attrs;
  return Py_INCREF(o), o;
}
PyObject* node_numel(PyObject* self, PyObject*) { return PyObject_CallMethod(as_node(self)->node_layout, "numel", nullptr); }
PyObject* node_src(PyObject* self, PyObject* i) { return PyObject_GetItem(as_node(self)->srcs, i); }
PyObject* node_shape(PyObject* self, PyObject* i) { return PyObject_CallMethod(as_node(self)->node_layout, "shape", "O", i); }
PyObject* node_leaf(PyObject*, PyObject* args, PyObject* kw) {
  static const char* names[] = {"layout", "dtype", "buf", nullptr};
  PyObject *layout, *dtype = nullptr, *buf = Py_None;
  if (!PyArg_ParseTupleAndKeywords(args, kw, "O|OO:leaf", const_cast<char**>(names), &layout, &dtype, &buf)) return nullptr;
  static PyObject* kBuffer = str_("BUFFER");
  static PyObject* kF32 = PyLong_FromLong(MG_F32);
  Ref list;
  if (buf != Py_None) {
    list = Ref(PyList_New(1));
    if (!list) return nullptr;
    Py_INCREF(buf);
    PyList_SET_ITEM(list.p, 0, buf);
  }
  return node_make(kBuffer, layout, dtype ? dtype : kF32, PyList_New(0), nullptr, list ? list.p : Py_None);
}
PyObject* node_repr(PyObject* self) {
  NodeObj* n = as_node(self);
  return PyUnicode_FromFormat("Node(op_type=%R, node_layout=%R, node_dtype=%R, %zd srcs, node_attrs=%R)", n->op_type,
                              n->node_layout, n->node_dtype, PySequence_Size(n->srcs), n->node_attrs);
}
#define FIELD(f) {#f, node_get, node_set, nullptr, reinterpret_cast<void*>(offsetof(NodeObj, f))}
PyGetSetDef node_fields[] = {FIELD(op_type), FIELD(node_layout), FIELD(node_dtype), FIELD(srcs), FIELD(node_attrs), FIELD(bufs),
                             {"__dict__", PyObject_GenericGetDict, PyObject_GenericSetDict, nullptr, nullptr},
                             {nullptr, nullptr, nullptr, nullptr, nullptr}};
#undef FIELD
PyMethodDef node_methods[] = {{"layout", node_layout, METH_NOARGS, nullptr},
                              {"dtype", node_dtype, METH_NOARGS, nullptr},
                              {"attrs", node_attrs, METH_NOARGS, nullptr},
                              {"numel", node_numel, METH_NOARGS, nullptr},
                              {"src", node_src, METH_O, nullptr},
                              {"shape", node_shape, METH_O, nullptr},
                              {"leaf", FAST(node_leaf), METH_VARARGS | METH_KEYWORDS | METH_STATIC, nullptr},
                              {"__reduce__", node_reduce, METH_NOARGS, nullptr},
                              {"__setstate__", node_setstate, METH_O, nullptr},
                              {nullptr, nullptr, 0, nullptr}};

Py_ssize_t src_count(const NodeObj* n) { return PySequence_Fast_GET_SIZE(n->srcs); }
PyObject* src_of(const NodeObj* n, Py_ssize_t i) { return PySequence_Fast_GET_ITEM(n->srcs, i); }

bool node_ok(PyObject* o) {
  if (is_node(o) && (PyList_Check(as_node(o)->srcs) || PyTuple_Check(as_node(o)->srcs))) return true;
  PyErr_SetString(PyExc_TypeError, "a graph vertex is a Node with a sequence of Node sources");
  return false;
}

// Sources before consumers, each node once, in the order of a depth-first walk over srcs.
bool toposort(PyObject* const* roots, Py_ssize_t n_roots, std::vector<Ref>& order) {
  const uint64_t epoch = ++g_epoch;
  std::vector<std::pair<NodeObj*, Py_ssize_t>> stack;
  for (Py_ssize_t r = 0; r < n_roots; ++r) {
    if (!node_ok(roots[r])) return false;
    if (as_node(roots[r])->mark == epoch) continue;
    as_node(roots[r])->mark = epoch;
    stack.emplace_back(as_node(roots[r]), 0);
    while (!stack.empty()) {
      NodeObj* n = stack.back().first;
      const Py_ssize_t i = stack.back().second;
      if (i < src_count(n)) {
        stack.back().second = i + 1;
        PyObject* c = src_of(n, i);
        if (!node_ok(c)) return false;
        if (as_node(c)->mark != epoch) {
          as_node(c)->mark = epoch;
          stack.emplace_back(as_node(c), 0);
        }
      } else {
        order.push_back(Ref::to(reinterpret_cast<PyObject*>(n)));
        stack.pop_back();
      }
    }
  }
  return true;
}

PyObject* py_toposort(PyObject*, PyObject* root) {
  std::vector<Ref> order;
  if (!toposort(&root, 1, order)) return nullptr;
  PyObject* list = PyList_New(static_cast<Py_ssize_t>(order.size()));
  if (!list) return nullptr;
  for (size_t i = 0; i < order.size(); ++i) PyList_SET_ITEM(list, static_cast<Py_ssize_t>(i), order[i].release());
  return list;
}

// depends_on(node, target): whether `target` is `node` or feeds it.
PyObject* py_depends_on(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 2 || !node_ok(args[0])) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "depends_on(node, target)");
    return nullptr;
  }
  const uint64_t epoch = ++g_epoch;
  std::vector<NodeObj*> stack{as_node(args[0])};
  as_node(args[0])->mark = epoch;
  while (!stack.empty()) {
    NodeObj* v = stack.back();
    stack.pop_back();
    if (reinterpret_cast<PyObject*>(v) == args[1]) Py_RETURN_TRUE;
    for (Py_ssize_t i = 0; i < src_count(v); ++i) {
      PyObject* c = src_of(v, i);
      if (!node_ok(c)) return nullptr;
      if (as_node(c)->mark != epoch) {
        as_node(c)->mark = epoch;
        stack.push_back(as_node(c));
      }
    }
  }
  Py_RETURN_FALSE;
}

// ------------------------------------------------------------------------------------------
// Storage and Buffer
// ------------------------------------------------------------------------------------------

struct StorageObj {  // one pooled allocation, returned to the pool with the last view of it
  PyObject_HEAD PyObject* device;
  unsigned long long ptr;
  long long nbytes;
};
PyTypeObject StorageType = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyObject* storage_make(PyObject* device, long long nbytes) {
  void* p = nullptr;
  const int rc = unlocked([&] { return L.pool_alloc(&p, nbytes); });
  if (rc != 0) return raise_status(rc), nullptr;
  StorageObj* s = PyObject_GC_New(StorageObj, &StorageType);
  if (!s) return (void)L.mg_pool_free(p), nullptr;
  Py_INCREF(device);
  s->device = device;
  s->ptr = reinterpret_cast<uintptr_t>(p);
  s->nbytes = nbytes;
  PyObject_GC_Track(s);
  return reinterpret_cast<PyObject*>(s);
}
PyObject* storage_new(PyTypeObject*, PyObject* args, PyObject* kw) {
  static const char* names[] = {"device", "nbytes", nullptr};
  PyObject* device;
  long long nbytes;
  if (!PyArg_ParseTupleAndKeywords(args, kw, "OL:Storage", const_cast<char**>(names), &device, &nbytes)) return nullptr;
  return storage_make(device, nbytes);
}
void storage_dealloc(PyObject* self) {
  StorageObj* s = reinterpret_cast<StorageObj*>(self);
  PyObject_GC_UnTrack(self);
  if (s->ptr) (void)L.mg_pool_free(reinterpret_cast<void*>(static_cast<uintptr_t>(s->ptr)));
  Py_XDECREF(s->device);
  PyObject_GC_Del(self);
}
// (No tp_clear here and for buffers: both are immutable in what a cycle can run through, the device is not.)
int storage_traverse(PyObject* self, visitproc visit, void* arg) {
  Py_VISIT(reinterpret_cast<StorageObj*>(self)->device);
  return 0;
}
PyMemberDef storage_members[] = {{"device", T_OBJECT, offsetof(StorageObj, device), READONLY, nullptr},
                                 {"ptr", T_ULONGLONG, offsetof(StorageObj, ptr), READONLY, nullptr},
                                 {"nbytes", T_LONGLONG, offsetof(StorageObj, nbytes), READONLY, nullptr},
                                 {nullptr, 0, 0, 0, nullptr}};

struct BufferObj {  // a typed view of a storage
  PyObject_HEAD PyObject* storage;
  int dtype;
  long long numel, offset_elems;
};
PyTypeObject BufferType = {PyVarObject_HEAD_INIT(nullptr, 0)};

int dtype_size(int dtype) {
  switch (dtype) {
    case MG_F32: case MG_I32: return 4;
    case MG_F16: case MG_BF16: return 2;
    case MG_I64: return 8;
    default: return 0;
  }
}
bool is_float(int dtype) { return dtype == MG_F32 || dtype == MG_F16 || dtype == MG_BF16; }
BufferObj* as_buffer(PyObject* o) { return reinterpret_cast<BufferObj*>(o); }
void* address(const BufferObj* b) {
  return reinterpret_cast<void*>(static_cast<uintptr_t>(reinterpret_cast<StorageObj*>(b->storage)->ptr) +
                                 static_cast<uintptr_t>(b->offset_elems * dtype_size(b->dtype)));
}
// Takes over `storage`.
PyObject* buffer_make(PyTypeObject* type, PyObject* storage, int dtype, long long numel, long long offset) {
  if (!storage) return nullptr;
  BufferObj* b = reinterpret_cast<BufferObj*>(type->tp_alloc(type, 0));
  if (!b) return Py_DECREF(storage), nullptr;
  b->storage = storage;
  b->dtype = dtype;
  b->numel = numel;
  b->offset_elems = offset;
  return reinterpret_cast<PyObject*>(b);
}
PyObject* buffer_new(PyTypeObject* type, PyObject* args, PyObject* kw) {
  static const char* names[] = {"storage", "dtype", "numel", "offset_elems", nullptr};
  PyObject* storage;
  int dtype;
  long long numel, offset = 0;
  if (!PyArg_ParseTupleAndKeywords(args, kw, "O!iL|L:AnyBuffer", const_cast<char**>(names), &StorageType, &storage, &dtype,
                                   &numel, &offset))
    return nullptr;
  Py_INCREF(storage);
  return buffer_make(type, storage, dtype, numel, offset);
}
int buffer_traverse(PyObject* self, visitproc visit, void* arg) {
  Py_VISIT(as_buffer(self)->storage);
  return 0;
}
void buffer_dealloc(PyObject* self) {
  PyObject_GC_UnTrack(self);
  Py_XDECREF(as_buffer(self)->storage);
  Py_TYPE(self)->tp_free(self);  // (a Python subclass's own deallocator releases its type)
}
PyObject* buffer_data_ptr(PyObject* self, PyObject* const* args, Py_ssize_t n, PyObject* kw) {
  bool with_offset = true;
  if (n + (kw ? PyTuple_GET_SIZE(kw) : 0) > 0) {
    const int t = PyObject_IsTrue(args[0]);
    if (t < 0) return nullptr;
    with_offset = t != 0;
  }
  BufferObj* b = as_buffer(self);
  const unsigned long long at = with_offset ? reinterpret_cast<uintptr_t>(address(b))
                                            : reinterpret_cast<StorageObj*>(b->storage)->ptr;
  Ref v(PyLong_FromUnsignedLongLong(at));
  return v ? PyObject_CallOneArg(g_void_p, v.p) : nullptr;
}
PyObject* buffer_view(PyObject* self, PyObject* layout) {
  if (!is_layout(layout)) return PyErr_SetString(PyExc_TypeError, "view() takes a Layout"), nullptr;
  BufferObj* b = as_buffer(self);
  Py_INCREF(b->storage);
  return buffer_make(Py_TYPE(self), b->storage, b->dtype, as_layout(layout)->numel, as_layout(layout)->base_offset);
}
PyObject* buffer_size_bytes(PyObject* self, PyObject*) {
  return PyLong_FromLongLong(as_buffer(self)->numel * dtype_size(as_buffer(self)->dtype));
}
PyObject* buffer_get_storage(PyObject* self, void*) { return new_ref(as_buffer(self)->storage); }
int buffer_set_storage(PyObject* self, PyObject* value, void*) {
  if (!value || Py_TYPE(value) != &StorageType) return PyErr_SetString(PyExc_TypeError, "a buffer's storage is a Storage"), -1;
  Py_SETREF(as_buffer(self)->storage, new_ref(value));
  return 0;
}
PyGetSetDef buffer_fields[] = {{"storage", buffer_get_storage, buffer_set_storage, nullptr, nullptr},
                               {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyMemberDef buffer_members[] = {{"dtype", T_INT, offsetof(BufferObj, dtype), 0, nullptr},
                                {"numel", T_LONGLONG, offsetof(BufferObj, numel), 0, nullptr},
                                {"offset_elems", T_LONGLONG, offsetof(BufferObj, offset_elems), 0, nullptr},
                                {nullptr, 0, 0, 0, nullptr}};
PyMethodDef buffer_methods[] = {{"data_ptr", FAST(buffer_data_ptr), METH_FASTCALL | METH_KEYWORDS, nullptr},
                                {"view", buffer_view, METH_O, nullptr},
                                {"size_bytes", buffer_size_bytes, METH_NOARGS, nullptr},
                                {nullptr, nullptr, 0, nullptr}};

// ------------------------------------------------------------------------------------------
// Evaluation
// ------------------------------------------------------------------------------------------

// 1, 0, or -1 with an error (a name that is no string may compare as it likes).
int op_names_equal(PyObject* a, PyObject* b) {
  if (a == b) return 1;
  if (!PyUnicode_CheckExact(a) || !PyUnicode_CheckExact(b)) return PyObject_RichCompareBool(a, b, Py_EQ);
  if (PyUnicode_CHECK_INTERNED(a) && PyUnicode_CHECK_INTERNED(b)) return 0;  // as names written in a program are
  return PyUnicode_Compare(a, b) == 0;
}

int dtype_of(const NodeObj* n) {  // -1: none of ours
  int over = 0;
  const long v = PyLong_Check(n->node_dtype) ? PyLong_AsLongAndOverflow(n->node_dtype, &over) : -1;
  return over == 0 && v >= 0 && v <= MG_I64 ? static_cast<int>(v) : -1;
}
bool plain_layout(PyObject* o) { return Py_TYPE(o) == g_layout_type || Py_TYPE(o) == &LayoutType; }

// One node's execution: its operands, and what the library needs of the device.  The library is called
// without the interpreter lock, and another thread may evaluate the same nodes meanwhile and
// replace their buffers: the operands are held here, and their addresses taken, before the call.
struct Exec {
  static constexpr int kMost = 12;  // operands
  struct Operand {
    Ref buffer, layout;
    void* p = nullptr;
    int dtype = 0;
  };
  Ref attrs, layout;  // the node's own
  PyObject* device = nullptr;
  void* stream = nullptr;
  void* pending = nullptr;  // the deferred list in use, or null
  int dtype = 0;
  uint32_t want = ~0u;  // bit i: result i is to be made (a form may make more)
  Operand in[kMost];
  LayoutObj* lay[kMost];  // of the sources
  int count = 0;

  // Whether the next operand, a result of `s`, is one of the package's own buffers under one of its layouts
  // (and taken).  Types derived from these, whose methods may say something else, are the Python forms'.
  bool add(Ref buffer, const NodeObj* s) {
    if (Py_TYPE(s) != &NodeType || Py_TYPE(buffer.p) != g_buffer_type || !plain_layout(s->node_layout)) return false;
    Operand& o = in[count];
    o.p = address(as_buffer(buffer.p));
    o.dtype = dtype_of(s);
    o.buffer = std::move(buffer);
    o.layout = Ref::to(s->node_layout);
    lay[count++] = as_layout(s->node_layout);
    return true;
  }
  const LayoutObj* out() const { return as_layout(layout.p); }
  void* p(int i) const { return in[i].p; }
  // The first k operands are contiguous and start on the 16-byte boundary the flat kernels read from.
  bool flat(int k) const {
    if (count < k) return false;
    for (int i = 0; i < k; ++i)
      if (!lay[i]->contiguous || reinterpret_cast<uintptr_t>(p(i)) % 16 != 0) return false;
    return true;
  }
  bool contiguous(int k) const {
    if (count < k) return false;
    for (int i = 0; i < k; ++i)
      if (!lay[i]->contiguous) return false;
    return true;
  }
  // Attributes.  False where one is missing (without `fallback`) or no plain value: left to the Python form,
  // which converts it or says what is wrong.
  bool truth(PyObject* key, bool* out) const {
    PyObject* v = PyDict_GetItem(attrs.p, key);
    if (!v || !(PyBool_Check(v) || PyLong_CheckExact(v))) return false;
    return *out = PyObject_IsTrue(v) == 1, true;
  }
  bool truth(PyObject* key, bool fallback, bool* out) const {
    return PyDict_GetItem(attrs.p, key) ? truth(key, out) : (*out = fallback, true);
  }
  bool number(PyObject* key, float* out) const {
    PyObject* v = PyDict_GetItem(attrs.p, key);
    if (!v || !(PyFloat_CheckExact(v) || PyLong_CheckExact(v))) return false;
    const double d = PyFloat_AsDouble(v);
    if (d == -1.0 && PyErr_Occurred()) return PyErr_Clear(), false;
    return *out = static_cast<float>(d), true;
  }
  PyObject* buffer(int dt, long long numel) const {
    return buffer_make(g_buffer_type, storage_make(device, numel * dtype_size(dt)), dt, numel, 0);
  }
};

// New buffers for a node's results; release() hands them over as a list.
struct Results {
  Ref list;
  std::vector<void*> at;
  const Exec& x;
  bool ok = true;
  explicit Results(const Exec& e) : list(PyList_New(0)), x(e) {}
  void add(int dt, long long numel) {
    if (!ok || !list) return;
    Ref o(x.buffer(dt, numel));
    ok = o && PyList_Append(list.p, o.p) == 0;
    if (ok) at.push_back(address(as_buffer(o.p)));
  }
  void add_none() { ok = ok && list && PyList_Append(list.p, Py_None) == 0, at.push_back(nullptr); }
  void* p(int i) const { return at[i]; }
};

struct GemmDims {
  long long batch, M, N, K, lda0, lda1, ldb0, ldb1, bsa, bsb;
};
// A (.., M, K) by B (.., N, K); false: batch dimensions that do not collapse, left to the Python form.
bool gemm_dims(const Exec& x, GemmDims* g) {
  const LayoutObj *la = x.lay[0], *lb = x.lay[1], *lo = x.out();
  for (const LayoutObj* l : {la, lb})
    for (Py_ssize_t i = rank_of(l) - 4; i >= 0; --i)
      if (stride_of(l, i) != dim_of(l, i + 1) * stride_of(l, i + 1)) return false;
  if (rank_of(la) < 2 || rank_of(lb) < 2 || rank_of(lo) < 1) return false;
  g->N = dim_of(lo, -1);
  g->M = dim_of(la, -2), g->K = dim_of(la, -1);
  if (g->M == 0 || g->K == 0) return false;
  g->lda0 = stride_of(la, -2), g->lda1 = stride_of(la, -1);
  g->ldb0 = stride_of(lb, -2), g->ldb1 = stride_of(lb, -1);
  g->batch = la->numel / (g->M * g->K);
  g->bsa = rank_of(la) >= 3 ? stride_of(la, -3) : g->M * g->K;
  g->bsb = rank_of(lb) >= 3 ? stride_of(lb, -3) : g->N * g->K;
  return true;
}

// The result of an exec form: 1 done (`out` holds the list), 0 not its case, -1 an error is set.
using Form = int (*)(const Exec&, PyObject** out);

int finish(Results& r, int rc, PyObject** out) {
  if (rc != 0) return raise_status(rc), -1;
  *out = r.list.release();
  return 1;
}
#define MG_RUN(call) finish(r, unlocked([&] { return call; }), out)

long long out_numel(const Exec& x) { return x.out()->numel; }

int run_matmul_bt(const Exec& x, PyObject** out) {
  GemmDims g;
  if (x.count < 2 || !gemm_dims(x, &g)) return 0;
  Results r(x);
  r.add(x.dtype, out_numel(x));
  if (!r.ok) return -1;
  return MG_RUN(L.mg_matmul_bt(x.p(0), x.p(1), r.p(0), g.batch, g.M, g.N, g.K, g.lda0, g.lda1, g.ldb0, g.ldb1, g.bsa,
                               g.bsb, x.dtype, x.stream));
}
template <auto Lib::*FN, bool FLAT2>
int run_matmul3(const Exec& x, PyObject** out) {
  GemmDims g;
  if (x.count < 3 || !gemm_dims(x, &g) || (FLAT2 && !x.lay[2]->contiguous)) return 0;
  Results r(x);
  r.add(x.dtype, out_numel(x));
  if (!r.ok) return -1;
  return MG_RUN((L.*FN)(x.p(0), x.p(1), x.p(2), r.p(0), g.batch, g.M, g.N, g.K, g.lda0, g.lda1, g.ldb0, g.ldb1, g.bsa,
                        g.bsb, x.dtype, x.stream));
}

int run_linear_grad(const Exec& x, PyObject** out) {
  bool accumulate, relu, has_bias;
  if (!x.truth(N.accumulate, false, &accumulate) || !x.truth(N.relu_mask, false, &relu) || !x.truth(N.has_bias, true, &has_bias))
    return 0;
  if (!x.contiguous(accumulate ? 4 : 3) || !is_float(x.dtype) || rank_of(x.lay[2]) != 2) return 0;
  const long long n = dim_of(x.lay[2], 0), k = dim_of(x.lay[2], 1);
  if (k == 0 || x.lay[0]->numel != x.lay[1]->numel / k * n) return 0;
  const long long m = x.lay[1]->numel / k;
  Results r(x);
  const long long size[3] = {m * k, n * k, n};
  for (int i = 0; i < (has_bias ? 3 : 2); ++i) {
    if (x.want >> i & 1u) r.add(x.dtype, size[i]);
    else r.add_none();
  }
  if (!r.ok) return -1;
  void *dx = r.p(0), *dw = r.p(1), *db = has_bias ? r.p(2) : nullptr;
  return MG_RUN([&]() -> int {
    if (accumulate && dx)
      if (int rc = L.mg_copy_device(dx, x.p(3), m * k * dtype_size(x.dtype), x.stream)) return rc;
    if (x.pending && dw)
      return L.mg_linear_bwd_deferred(x.p(0), x.p(1), x.p(2), dx, dw, db, m, n, k, accumulate, relu, x.dtype, x.dtype,
                                      x.pending, x.stream);
    return L.mg_linear_bwd_fused(x.p(0), x.p(1), x.p(2), dx, dw, db, m, n, k, accumulate, relu, x.dtype, x.stream);
  }());
}

int run_linear_ln_grad(const Exec& x, PyObject** out) {
  bool accumulate, has_bias;
  if (!x.truth(N.accumulate, false, &accumulate) || !x.truth(N.has_bias, true, &has_bias)) return 0;
  if (!x.contiguous(accumulate ? 8 : 7) || !is_float(x.dtype) || rank_of(x.lay[2]) != 2) return 0;
  const long long n = dim_of(x.lay[2], 0), k = dim_of(x.lay[2], 1);
  if (k == 0) return 0;
  const long long m = x.lay[1]->numel / k;
  if (x.lay[0]->numel != m * n || x.lay[3]->numel != m * k) return 0;
  Results r(x);
  r.add(x.dtype, m * k);
  r.add(x.dtype, k);
  r.add(x.dtype, k);
  r.add(x.dtype, n * k);
  if (has_bias) r.add(x.dtype, n);
  if (!r.ok) return -1;
  return MG_RUN([&]() -> int {
    if (accumulate)
      if (int rc = L.mg_copy_device(r.p(0), x.p(7), m * k * dtype_size(x.dtype), x.stream)) return rc;
    return L.mg_linear_bwd_layer_norm_bwd(x.p(0), x.p(1), x.p(2), x.p(3), x.p(4), static_cast<float*>(x.p(5)),
                                          static_cast<float*>(x.p(6)), r.p(0), r.p(3), has_bias ? r.p(4) : nullptr, r.p(1),
                                          r.p(2), m, n, k, accumulate, x.dtype, x.dtype, x.pending, x.stream);
  }());
}

int run_layer_norm_stats(const Exec& x, PyObject** out) {
  float eps;
  if (!x.contiguous(3) || !is_float(x.dtype) || !x.number(N.eps, &eps)) return 0;
  const long long cols = last_dim(x.lay[0]);
  if (cols == 0) return 0;
  const long long rows = x.lay[0]->numel / cols;
  Results r(x);
  r.add(x.dtype, out_numel(x));
  r.add(MG_F32, rows);
  r.add(MG_F32, rows);
  if (!r.ok) return -1;
  return MG_RUN(L.mg_layer_norm_fwd_stats(x.p(0), x.p(1), x.p(2), r.p(0), static_cast<float*>(r.p(1)),
                                          static_cast<float*>(r.p(2)), rows, cols, eps, x.dtype, x.stream));
}

template <bool RESIDUAL>
int run_layer_norm_stats_grad(const Exec& x, PyObject** out) {
  if (!x.contiguous(RESIDUAL ? 6 : 5) || !is_float(x.dtype)) return 0;
  const long long cols = last_dim(x.lay[1]);
  if (cols == 0) return 0;
  const long long rows = x.lay[1]->numel / cols;
  Results r(x);
  r.add(x.dtype, rows * cols);
  r.add(x.dtype, x.lay[2]->numel);
  r.add(x.dtype, x.lay[2]->numel);
  if (!r.ok) return -1;
  const float *mean = static_cast<float*>(x.p(3)), *rstd = static_cast<float*>(x.p(4));
  void* res = RESIDUAL ? x.p(5) : nullptr;
  return MG_RUN([&]() -> int {
    if (x.pending)
      return L.mg_layer_norm_bwd_stats_deferred(x.p(0), x.p(1), x.p(2), mean, rstd, res, r.p(0), r.p(1), r.p(2), rows, cols,
                                                x.dtype, x.dtype, x.pending, x.stream);
    if (RESIDUAL)
      return L.mg_layer_norm_bwd_stats_add(x.p(0), x.p(1), x.p(2), mean, rstd, res, r.p(0), r.p(1), r.p(2), rows, cols,
                                           x.dtype, x.stream);
    return L.mg_layer_norm_bwd_stats(x.p(0), x.p(1), x.p(2), mean, rstd, r.p(0), r.p(1), r.p(2), rows, cols, x.dtype,
                                     x.stream);
  }());
}

int run_add(const Exec& x, PyObject** out) {
  if (!x.flat(2)) return 0;
  Results r(x);
  r.add(x.dtype, out_numel(x));
  if (!r.ok) return -1;
  return MG_RUN(L.mg_add(x.p(0), x.p(1), r.p(0), out_numel(x), x.dtype, x.stream));
}
int run_relu(const Exec& x, PyObject** out) {
  if (!x.flat(1)) return 0;
  Results r(x);
  r.add(x.dtype, out_numel(x));
  if (!r.ok) return -1;
  return MG_RUN(L.mg_relu(x.p(0), r.p(0), out_numel(x), x.dtype, x.stream));
}
int run_relu_grad(const Exec& x, PyObject** out) {
  if (!x.flat(2)) return 0;
  Results r(x);
  r.add(x.dtype, out_numel(x));
  if (!r.ok) return -1;
  return MG_RUN(L.mg_relu_grad(x.p(0), x.p(1), r.p(0), out_numel(x), x.dtype, x.stream));
}
int run_gather(const Exec& x, PyObject** out) {
  if (x.count < 2 || rank_of(x.lay[0]) != 2 || !x.lay[1]->contiguous) return 0;
  Results r(x);
  r.add(x.dtype, out_numel(x));
  if (!r.ok) return -1;
  return MG_RUN(L.mg_gather(x.p(0), x.p(1), r.p(0), x.lay[1]->numel, dim_of(x.lay[0], 0), dim_of(x.lay[0], 1),
                            stride_of(x.lay[0], 0), stride_of(x.lay[0], 1), x.in[1].dtype, x.dtype, x.stream));
}
int run_scatter_add(const Exec& x, PyObject** out) {
  const LayoutObj* lo = x.out();
  if (!x.contiguous(2) || rank_of(x.lay[1]) != rank_of(x.lay[0]) + 1 || rank_of(lo) < 1) return 0;
  Results r(x);
  r.add(x.dtype, lo->numel);
  if (!r.ok) return -1;
  const long long n_idx = x.lay[0]->numel, rows = dim_of(lo, 0), row_size = dim_of(x.lay[1], -1);
  return MG_RUN(x.pending ? L.mg_scatter_add_deferred(x.p(0), x.p(1), r.p(0), n_idx, rows, row_size, x.in[0].dtype, x.dtype,
                                                      x.dtype, x.pending, x.stream)
                          : L.mg_scatter_add(x.p(0), x.p(1), r.p(0), n_idx, rows, row_size, x.in[0].dtype, x.dtype, x.stream));
}
int run_attn_packed(const Exec& x, PyObject** out) {
  const LayoutObj* q = x.lay[0];
  if (x.count < 1 || !is_float(x.dtype) || rank_of(q) != 5 || dim_of(q, 2) != 3) return 0;
  const long long B = dim_of(q, 0), S = dim_of(q, 1), H = dim_of(q, 3), D = dim_of(q, 4);
  float scale;
  bool causal, bias;
  if (!x.number(N.scale, &scale) || !x.truth(N.is_causal, &causal) || !x.truth(N.has_bias, true, &bias)) return 0;
  Results r(x);
  r.add(x.dtype, out_numel(x));
  r.add(MG_F32, B * H * S);
  if (!r.ok) return -1;
  return MG_RUN(L.mg_flash_attn_fwd_packed(x.p(0), x.count > 1 ? x.p(1) : nullptr, r.p(0), static_cast<float*>(r.p(1)), B, S,
                                           H, D, scale, causal, bias, x.dtype, x.stream));
}
int run_attn_packed_grad(const Exec& x, PyObject** out) {
  if (x.count < 4 || !is_float(x.dtype) || !x.lay[0]->contiguous || rank_of(x.lay[2]) != 5) return 0;
  const LayoutObj* q = x.lay[2];
  const long long B = dim_of(q, 0), S = dim_of(q, 1), H = dim_of(q, 3), D = dim_of(q, 4);
  float scale;
  bool causal, bias;
  if (!x.number(N.scale, &scale) || !x.truth(N.is_causal, &causal) || !x.truth(N.has_bias, !causal, &bias)) return 0;
  Results r(x);
  r.add(x.dtype, out_numel(x));
  if (!r.ok) return -1;
  return MG_RUN(L.mg_flash_attn_bwd_packed(x.p(0), x.p(1), x.p(2), x.count > 4 ? x.p(4) : nullptr,
                                           static_cast<float*>(x.p(3)), r.p(0), B, S, H, D, scale, causal, bias, x.dtype,
                                           x.stream));
}
int run_ce_ids(const Exec& x, PyObject** out) {
  if (!x.contiguous(2) || !is_float(x.dtype)) return 0;
  const long long c = last_dim(x.lay[0]);
  if (c == 0) return 0;
  Results r(x);
  r.add(x.dtype, out_numel(x));
  if (!r.ok) return -1;
  return MG_RUN(L.mg_cross_entropy_ids(x.p(0), x.p(1), r.p(0), x.lay[0]->numel / c, c, x.dtype, x.in[1].dtype, x.stream));
}
int run_ce_grad_ids(const Exec& x, PyObject** out) {
  if (!x.contiguous(2) || x.count < 3 || !is_float(x.dtype)) return 0;
  const long long c = last_dim(x.lay[0]);
  if (c == 0) return 0;
  Results r(x);
  r.add(x.dtype, out_numel(x));
  if (!r.ok) return -1;
  return MG_RUN(L.mg_cross_entropy_grad_ids(x.p(0), x.p(1), x.p(2), r.p(0), x.lay[0]->numel / c, c, x.dtype, x.in[1].dtype,
                                            x.stream));
}
int run_reshape(const Exec& x, PyObject** out) {
  if (!x.contiguous(1)) return 0;
  Ref list(PyList_New(1));
  if (!list) return -1;
  const BufferObj* b = as_buffer(x.in[0].buffer.p);
  Py_INCREF(b->storage);
  PyObject* v = buffer_make(g_buffer_type, b->storage, b->dtype, out_numel(x), b->offset_elems);
  if (!v) return -1;
  PyList_SET_ITEM(list.p, 0, v);
  *out = list.release();
  return 1;
}

PyObject* g_forms = nullptr;  // op type -> index into kForms
const std::pair<const char*, Form> kForms[] = {
    {"MATMUL_BT", run_matmul_bt},
    {"MATMUL_BIAS_BT", run_matmul3<&Lib::mg_matmul_bias_bt, false>},
    {"MATMUL_BIAS_RELU_BT", run_matmul3<&Lib::mg_matmul_bias_relu_bt, false>},
    {"MATMUL_BT_ADD", run_matmul3<&Lib::mg_matmul_bt_add, true>},
    {"LINEAR_GRAD", run_linear_grad},
    {"LINEAR_LAYER_NORM_GRAD", run_linear_ln_grad},
    {"LAYER_NORM_STATS", run_layer_norm_stats},
    {"LAYER_NORM_STATS_GRAD", run_layer_norm_stats_grad<false>},
    {"LAYER_NORM_STATS_GRAD_ADD", run_layer_norm_stats_grad<true>},
    {"ADD", run_add},
    {"RELU", run_relu},
    {"RELU_GRAD", run_relu_grad},
    {"GATHER", run_gather},
    {"SCATTER_ADD", run_scatter_add},
    {"FLASH_ATTN_PACKED", run_attn_packed},
    {"FLASH_ATTN_PACKED_GRAD", run_attn_packed_grad},
    {"CROSS_ENTROPY_IDS", run_ce_ids},
    {"CROSS_ENTROPY_IDS_GRAD", run_ce_grad_ids},
    {"RESHAPE", run_reshape},
};
constexpr size_t kFormCount = sizeof(kForms) / sizeof(kForms[0]);

// The package's own exec functions, and the run() that looks them up: a form stands in for its op's function
// only while the rule table holds that one.
PyObject* g_own_run = nullptr;
PyObject* g_own_rules[kFormCount];

// One evaluate() call: the nodes in order, and what the walk knows of each.  Nothing of a walk is kept on
// the nodes, which other walks (other threads, or an exec function of this one) may visit meanwhile.
struct Evaluation {
  struct Vertex {
    Ref node;
    uint32_t first = 0, count = 0;  // its sources: positions in the walk, sources[first ...]
    uint32_t used = 0;              // which results of a multi-output node are read
  };
  std::vector<Vertex> walk;
  std::vector<uint32_t> sources;
  std::vector<uint32_t> ce_grads;  // CROSS_ENTROPY_IDS_GRAD nodes

  PyObject* device;
  PyObject* run;    // runtime.run(node, inputs, device): the Python exec function of a node
  PyObject* rules;  // the table it looks in
  void* stream = nullptr;
  void* pending = nullptr;
  bool native = true;  // whether the forms of this file may be used at all
  PyObject *kBuffer, *kGetTuple, *kCeIds, *kCeIdsGrad, *kLinearGrad;

  NodeObj* node(uint32_t at) const { return as_node(walk[at].node.p); }
  uint32_t source(uint32_t at, uint32_t i) const { return sources[walk[at].first + i]; }
  static bool op_is(const NodeObj* n, PyObject* name) {
    return n->op_type == name || (PyUnicode_Check(n->op_type) && PyUnicode_Compare(n->op_type, name) == 0);
  }
  bool have(uint32_t at) const { return node(at)->bufs != Py_None; }
  // GETTUPLE's `index`, read like attrs()["index"].
  static bool index_of(const NodeObj* n, Py_ssize_t* out) {
    Ref v(PyObject_GetItem(n->node_attrs, N.index)), as_int(v ? PyNumber_Long(v.p) : nullptr);
    if (!as_int) return false;
    *out = PyLong_AsSsize_t(as_int.p);
    return *out != -1 || !PyErr_Occurred();
  }

  bool build(PyObject* const* roots, Py_ssize_t n_roots) {
    std::vector<Ref> order;
    if (!toposort(roots, n_roots, order)) return false;
    walk.resize(order.size());
    for (uint32_t i = 0; i < walk.size(); ++i) {
      walk[i].node = std::move(order[i]);
      node(i)->position = i;
    }
    std::vector<Py_ssize_t> readers(walk.size(), 0);
    std::vector<uint32_t> at_root;
    for (uint32_t i = 0; i < walk.size(); ++i) {  // (no Python code since toposort: the positions are ours)
      walk[i].first = static_cast<uint32_t>(sources.size());
      walk[i].count = static_cast<uint32_t>(src_count(node(i)));
      for (uint32_t k = 0; k < walk[i].count; ++k) {
        const uint32_t at = as_node(src_of(node(i), k))->position;
        if (at >= i) return raise_invalid("evaluate: the graph has a cycle"), false;
        sources.push_back(at);
        ++readers[at];
      }
    }
    for (Py_ssize_t i = 0; i < n_roots; ++i) at_root.push_back(as_node(roots[i])->position);
    // (Looking up an attribute may run Python code, after which the positions may be another walk's.)
    for (uint32_t i = 0; i < walk.size(); ++i) {
      if (op_is(node(i), kCeIdsGrad)) ce_grads.push_back(i);
      uint32_t bit = 1u;  // a node read directly gives its first result
      if (op_is(node(i), kGetTuple)) {
        PyObject* index = PyDict_Check(node(i)->node_attrs) ? PyDict_GetItem(node(i)->node_attrs, N.index) : nullptr;
        int over = 0;
        const long at = index && PyLong_Check(index) ? PyLong_AsLongAndOverflow(index, &over) : -1;
        bit = at >= 0 && at < 31 ? 1u << at : ~0u;
      }
      for (uint32_t k = 0; k < walk[i].count; ++k) walk[source(i, k)].used |= bit;
    }
    for (const uint32_t i : at_root) walk[i].used = ~0u;
    // A layer's dX that nobody reads (the first layer's input is data) is not computed, unless something
    // outside the walk holds the node too (a selector of dX that is kept for later): its result is
    // that of the operands as they are now.
    for (uint32_t i = 0; i < walk.size(); ++i)
      if (!op_is(node(i), kLinearGrad) || Py_REFCNT(node(i)) > readers[i] + 1) walk[i].used |= 1u;
    return true;
  }

  // Whether an evaluated node's dX was left out.
  bool lacks_dx(uint32_t at) const {
    PyObject* list = node(at)->bufs;
    return PyList_Check(list) && PyList_GET_SIZE(list) > 0 && PyList_GET_ITEM(list, 0) == Py_None && op_is(node(at), kLinearGrad);
  }
  // Makes it after all; the other results stay the ones they are.
  Ref complete(uint32_t at) {
    Ref old = Ref::to(node(at)->bufs), made = make(at, 1u), list;
    if (!made) return Ref();
    if (!PyList_Check(made.p) || PyList_GET_SIZE(made.p) != PyList_GET_SIZE(old.p)) list = std::move(made);
    else list = Ref(PyList_GetSlice(old.p, 0, PyList_GET_SIZE(old.p)));
    if (list && made) {
      Ref dx = Ref::to(PyList_GET_ITEM(made.p, 0));
      PyList_SetItem(list.p, 0, dx.release());
    }
    if (list) set(node(at), Ref::to(list.p));
    return list;
  }
  // Result i of an evaluated node.
  Ref result(uint32_t at, Py_ssize_t i) {
    const bool first = i == 0 || (i < 0 && PyList_Check(node(at)->bufs) && i == -PyList_GET_SIZE(node(at)->bufs));
    Ref list = first && lacks_dx(at) ? complete(at) : Ref::to(node(at)->bufs);
    if (!list) return Ref();
    if (!PyList_Check(list.p) && !PyTuple_Check(list.p)) {
      Ref index(PyLong_FromSsize_t(i));
      return index ? Ref(PyObject_GetItem(list.p, index.p)) : Ref();
    }
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(list.p);
    if (i < -n || i >= n) return PyErr_SetString(PyExc_IndexError, "evaluate: a source has no such result"), Ref();
    return Ref::to(PySequence_Fast_GET_ITEM(list.p, i < 0 ? i + n : i));
  }
  static bool set(NodeObj* n, Ref list) {
    if (!list) return false;
    Py_SETREF(n->bufs, list.release());
    return true;
  }

  // The index of the form for an op, or -1: there is none, or a program has put its own function in its place.
  long form_of(PyObject* op) const {
    PyObject* idx = native ? PyDict_GetItem(g_forms, op) : nullptr;
    const long i = idx ? PyLong_AsLong(idx) : -1;
    return i >= 0 && PyDict_GetItem(rules, op) == g_own_rules[i] ? i : -1;
  }
  // The results of a node whose sources have theirs; without those that are neither wanted nor made anyway.
  Ref make(uint32_t at, uint32_t want) {
    NodeObj* n = node(at);
    const uint32_t count = walk[at].count;
    const long form = form_of(n->op_type);
    const int dtype = dtype_of(n);
    if (form >= 0 && count <= Exec::kMost && Py_TYPE(n) == &NodeType && plain_layout(n->node_layout) &&
        PyDict_CheckExact(n->node_attrs) && dtype >= 0) {
      Exec x;
      x.attrs = Ref::to(n->node_attrs), x.layout = Ref::to(n->node_layout);
      x.device = device, x.stream = stream, x.pending = pending, x.want = want;
      x.dtype = dtype;
      bool plain = true;
      for (uint32_t i = 0; i < count && plain; ++i) {
        Ref b = result(source(at, i), 0);
        if (!b) return Ref();
        plain = x.add(std::move(b), node(source(at, i)));
      }
      if (plain) {
        PyObject* out = nullptr;
        const int rc = kForms[form].second(x, &out);
        if (rc < 0) return Ref();
        if (rc > 0) return Ref(out);
      }
    }
    Ref inputs(PyList_New(count));
    if (!inputs) return Ref();
    for (uint32_t i = 0; i < count; ++i) {
      Ref b = result(source(at, i), 0);
      if (!b) return Ref();
      PyList_SET_ITEM(inputs.p, i, b.release());
    }
    return Ref(PyObject_CallFunctionObjArgs(run, n, inputs.p, device, nullptr));
  }

  // CROSS_ENTROPY_IDS[logits, ids] and the CROSS_ENTROPY_IDS_GRAD of the same operands in this walk: loss
  // and dlogits in one pass over the logits, when the gradient's upstream is already there (it is the
  // graph's root).  1 done, 0 not such a pair, -1 error.
  int cross_entropy_pair(uint32_t at) {
    if (walk[at].count != 2) return 0;
    uint32_t pair = at;
    for (uint32_t c : ce_grads)
      if (!have(c) && walk[c].count == 3 && source(c, 0) == source(at, 0) && source(c, 1) == source(at, 1) &&
          have(source(c, 2)))
        pair = c;
    NodeObj *n = node(at), *g = node(pair);
    if (pair == at || Py_TYPE(n) != &NodeType || Py_TYPE(g) != &NodeType || !plain_layout(n->node_layout) ||
        !plain_layout(g->node_layout))
      return 0;
    Exec x;
    x.layout = Ref::to(n->node_layout);
    Ref grad_layout = Ref::to(g->node_layout);
    x.device = device, x.dtype = dtype_of(n);
    if (form_of(kCeIds) < 0 || form_of(kCeIdsGrad) < 0 || dtype_of(g) != x.dtype || !is_float(x.dtype)) return 0;
    for (uint32_t i = 0; i < 3; ++i) {
      Ref b = result(source(pair, i), 0);
      if (!b) return -1;
      if (!x.add(std::move(b), node(source(pair, i)))) return 0;
    }
    if (!x.contiguous(3)) return 0;
    const long long c = last_dim(x.lay[0]);
    if (c == 0) return 0;
    Results loss(x), grad(x);
    loss.add(x.dtype, out_numel(x));
    grad.add(x.dtype, as_layout(grad_layout.p)->numel);
    if (!loss.ok || !grad.ok) return -1;
    const int rc = unlocked([&] {
      return L.mg_cross_entropy_fused_ids(x.p(0), x.p(1), x.p(2), loss.p(0), grad.p(0), x.lay[0]->numel / c, c, x.dtype,
                                          x.in[1].dtype, stream);
    });
    if (rc != 0) return raise_status(rc), -1;
    return set(n, std::move(loss.list)) && set(g, std::move(grad.list)) ? 1 : -1;
  }

  bool evaluate(uint32_t at) {
    if (have(at)) return walk[at].used != ~0u || !lacks_dx(at) || complete(at);
    NodeObj* n = node(at);
    if (!ce_grads.empty() && op_is(n, kCeIds)) {
      const int rc = cross_entropy_pair(at);
      if (rc != 0) return rc > 0;
    }
    if (op_is(n, kBuffer)) return raise_invalid("evaluate: a leaf node without a buffer"), false;
    if (!op_is(n, kGetTuple)) return set(n, make(at, walk[at].used | ~1u));
    if (walk[at].count == 0) return PyErr_SetString(PyExc_IndexError, "GETTUPLE without a source"), false;
    Py_ssize_t i;
    if (!index_of(n, &i)) return false;
    Ref b = result(source(at, 0), i);
    Ref list(b ? PyList_New(1) : nullptr);
    if (!list) return false;
    PyList_SET_ITEM(list.p, 0, b.release());
    return set(n, std::move(list));
  }
};

// evaluate(nodes, device, run, rules): gives every node of `nodes` and of their sources its buffers.
PyObject* py_evaluate(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 4) return PyErr_SetString(PyExc_TypeError, "evaluate(nodes, device, run, rules)"), nullptr;
  Ref nodes(PySequence_Tuple(args[0]));
  if (!nodes) return nullptr;
  Evaluation e;
  e.device = args[1], e.run = args[2], e.rules = args[3];
  static PyObject *kBuffer = str_("BUFFER"), *kGetTuple = str_("GETTUPLE");
  e.kBuffer = kBuffer, e.kGetTuple = kGetTuple;
  static PyObject *kCeIds = str_("CROSS_ENTROPY_IDS"), *kCeIdsGrad = str_("CROSS_ENTROPY_IDS_GRAD");
  e.kCeIds = kCeIds, e.kCeIdsGrad = kCeIdsGrad;
  static PyObject* kLinearGrad = str_("LINEAR_GRAD");
  e.kLinearGrad = kLinearGrad;
  Ref stream(PyObject_GetAttr(e.device, N.stream)), pending(PyObject_GetAttr(e.device, N.pending));
  if (!stream || !pending) return nullptr;
  e.native = e.run == g_own_run && PyDict_CheckExact(e.rules) && pointer_of(stream.p, &e.stream) && pointer_of(pending.p, &e.pending);
  if (!e.build(PySequence_Fast_ITEMS(nodes.p), PySequence_Fast_GET_SIZE(nodes.p))) return nullptr;
  for (uint32_t i = 0; i < e.walk.size(); ++i)
    if (!e.evaluate(i)) return nullptr;
  Py_RETURN_NONE;
}

// ------------------------------------------------------------------------------------------
// The rewriting pass (mograd_amd/rewrites.py says what it does; this is its loop)
// ------------------------------------------------------------------------------------------

// Pat.matches
int pat_matches(PyObject* pat, NodeObj* n) {
  Ref op(PyObject_GetAttr(pat, N.op_type)), srcs(PyObject_GetAttr(pat, N.srcs));
  if (!op || !srcs) return -1;
  const int same = op.p == Py_None ? 1 : op_names_equal(op.p, n->op_type);
  if (same <= 0) return same;
  Ref fast(PySequence_Fast(srcs.p, "Pat.srcs"));
  if (!fast) return -1;
  const Py_ssize_t k = PySequence_Fast_GET_SIZE(fast.p);
  if (k > src_count(n)) return 0;
  for (Py_ssize_t i = 0; i < k; ++i) {
    Ref s = i < src_count(n) ? Ref::to(src_of(n, i)) : Ref();  // (a pattern's op may compare by Python code)
    if (!s || !node_ok(s.p)) return PyErr_Occurred() ? -1 : 0;
    const int rc = pat_matches(PySequence_Fast_GET_ITEM(fast.p, i), as_node(s.p));
    if (rc <= 0) return rc;
  }
  return 1;
}

struct Pass {
  PyObject* sim;
  PyObject *subst, *uses, *origin, *consumers;  // the Simplifier's dictionaries (borrowed: it holds them)

  // The node that `n` has become (borrowed).
  PyObject* resolve(PyObject* n) const {
    int seen = 0;
    while (PyObject* to = PyDict_GetItem(subst, n)) {
      n = to;
      if (++seen > 64) return raise_invalid("Simplifier: substitutions cycled without converging"), nullptr;
    }
    return n;
  }
  int count(PyObject* n) const {
    PyObject* c = PyDict_GetItem(uses, n);
    return c ? static_cast<int>(PyLong_AsLong(c)) : 0;
  }
  bool set_count(PyObject* n, int c) const {
    Ref v(PyLong_FromLong(c));
    return v && PyDict_SetItem(uses, n, v.p) == 0;
  }
  bool set_origin(PyObject* made, PyObject* from) const {
    PyObject* o = PyDict_GetItem(origin, from);
    return PyDict_SetItem(origin, made, o ? o : from) == 0;
  }
  // A node like `n` over other sources (takes over `srcs`).
  static PyObject* rebuilt(NodeObj* n, PyObject* srcs) {
    PyObject* attrs = PyDict_CheckExact(n->node_attrs) ? PyDict_Copy(n->node_attrs)
                                                       : PyObject_CallOneArg(reinterpret_cast<PyObject*>(&PyDict_Type), n->node_attrs);
    if (!attrs) return Py_DECREF(srcs), nullptr;
    return node_make(n->op_type, n->node_layout, n->node_dtype, srcs, attrs, n->bufs);
  }
  // `node` with every source replaced by what it has become; a new reference.
  PyObject* with_subst(PyObject* node) const {
    NodeObj* n = as_node(node);
    Ref fresh;
    for (Py_ssize_t i = 0; i < src_count(n); ++i) {
      PyObject* s = src_of(n, i);
      PyObject* to = resolve(s);
      if (!to) return nullptr;
      if (to != s && !fresh) {
        fresh = Ref(PySequence_List(n->srcs));
        if (!fresh) return nullptr;
      }
      if (to != s) {
        Py_INCREF(to);
        PyList_SetItem(fresh.p, i, to);
      }
    }
    if (!fresh) return Py_INCREF(node), node;
    Ref out(rebuilt(n, fresh.release()));
    if (!out || !set_count(out.p, count(node)) || !set_origin(out.p, node)) return nullptr;
    return out.release();
  }

  // Every edge of the result follows the final substitution table.
  PyObject* redirect(PyObject* roots) const {
    Ref done(PyDict_New());
    if (!done) return nullptr;
    std::vector<std::pair<PyObject*, Py_ssize_t>> stack;
    const Py_ssize_t n_roots = PySequence_Fast_GET_SIZE(roots);
    for (Py_ssize_t i = n_roots - 1; i >= 0; --i) stack.emplace_back(PySequence_Fast_GET_ITEM(roots, i), 0);
    while (!stack.empty()) {
      PyObject* n = stack.back().first;
      const Py_ssize_t i = stack.back().second;
      PyObject* r = resolve(n);
      if (!r) return nullptr;
      if (PyObject* d = PyDict_GetItem(done.p, r)) {
        stack.pop_back();
        if (n != r && PyDict_SetItem(done.p, n, d) != 0) return nullptr;
        continue;
      }
      NodeObj* v = as_node(r);
      if (!node_ok(r)) return nullptr;
      if (i < src_count(v)) {
        stack.back().second = i + 1;
        PyObject* c = src_of(v, i);
        if (!PyDict_GetItem(done.p, c)) stack.emplace_back(c, 0);
        continue;
      }
      stack.pop_back();
      Ref fresh;
      for (Py_ssize_t k = 0; k < src_count(v); ++k) {
        PyObject* s = src_of(v, k);
        PyObject* to = PyDict_GetItem(done.p, s);
        if (to == s) continue;
        if (!fresh) {
          fresh = Ref(PySequence_List(v->srcs));
          if (!fresh) return nullptr;
        }
        Py_INCREF(to);
        PyList_SetItem(fresh.p, k, to);
      }
      Ref out(fresh ? rebuilt(v, fresh.release()) : (Py_INCREF(r), r));
      if (!out || PyDict_SetItem(done.p, r, out.p) != 0) return nullptr;
      if (n != r && PyDict_SetItem(done.p, n, out.p) != 0) return nullptr;
    }
    PyObject* list = PyList_New(n_roots);
    for (Py_ssize_t i = 0; list && i < n_roots; ++i) {
      PyObject* d = PyDict_GetItem(done.p, PySequence_Fast_GET_ITEM(roots, i));
      Py_INCREF(d);
      PyList_SET_ITEM(list, i, d);
    }
    return list;
  }
};

// ------------------------------------------------------------------------------------------
// The package's own gradient and rewrite rules (runtime.py and rewrites.py define them: what is here is what they do for
// plain nodes, and a node, layout or attribute that is not plain goes to the Python function itself).  With the rules in
// Python a lazily built step of four layers took 861 us and a small classifier's pass 51.4; with these 789 and 47.5.
// ------------------------------------------------------------------------------------------

enum Outcome { kError = -1, kNotMine = 0, kDone = 1 };

struct OpNames {
  PyObject *linear_grad, *gettuple, *layer_norm_stats_grad, *layer_norm_stats_grad_add, *packed_grad, *ce_grad, *ce_ids, *ce_ids_grad,
      *relu_grad, *scatter_add, *reshape, *add, *matmul_bt, *matmul_bias_bt, *matmul_bt_add, *matmul_bias_relu_bt, *linear_ln_grad;
} O;
PyObject* g_small[5];  // 0 .. 4

// A node of the type itself, with nothing of a program's own on it, over nodes, with a layout and dtype of ours and
// attributes whose names and values are looked up and tested without running Python code.
bool plain_node(PyObject* o) {
  if (Py_TYPE(o) != &NodeType) return false;
  const NodeObj* n = as_node(o);
  if ((n->dict && PyDict_GET_SIZE(n->dict) != 0) || !(PyList_CheckExact(n->srcs) || PyTuple_CheckExact(n->srcs)) ||
      !PyDict_CheckExact(n->node_attrs) || !plain_layout(n->node_layout) || !PyUnicode_CheckExact(n->op_type) ||
      !PyLong_CheckExact(n->node_dtype))
    return false;
  PyObject *k, *v;
  Py_ssize_t at = 0;
  while (PyDict_Next(n->node_attrs, &at, &k, &v))
    if (!PyUnicode_CheckExact(k) ||
        !(PyBool_Check(v) || PyLong_CheckExact(v) || PyFloat_CheckExact(v) || PyUnicode_CheckExact(v) || v == Py_None))
      return false;
  return true;
}
// Source i where it is such a node, or null.
NodeObj* plain_src(const NodeObj* n, Py_ssize_t i) {
  if (i >= src_count(n)) return nullptr;
  PyObject* s = src_of(n, i);
  return plain_node(s) ? as_node(s) : nullptr;
}
PyObject* obj(NodeObj* n) { return reinterpret_cast<PyObject*>(n); }
bool op_is_name(const NodeObj* n, PyObject* name) { return op_names_equal(n->op_type, name) == 1; }  // (both are str)
bool same_dtype(const NodeObj* a, const NodeObj* b) { return PyObject_RichCompareBool(a->node_dtype, b->node_dtype, Py_EQ) == 1; }
bool same_dims(const NodeObj* a, const NodeObj* b) {
  return PyObject_RichCompareBool(as_layout(a->node_layout)->dims, as_layout(b->node_layout)->dims, Py_EQ) == 1;
}
Ref contiguous_of(const NodeObj* n) { return Ref(layout_as_contiguous(n->node_layout, nullptr)); }
Ref list_of(std::initializer_list<PyObject*> items) {
  Ref list(PyList_New(static_cast<Py_ssize_t>(items.size())));
  Py_ssize_t i = 0;
  for (PyObject* o : items)
    if (list) PyList_SET_ITEM(list.p, i++, new_ref(o));
  return list;
}
Ref dict_with(PyObject* key, PyObject* value) {
  Ref d(PyDict_New());
  if (d && PyDict_SetItem(d.p, key, value) != 0) return Ref();
  return d;
}
// Node(op, layout, dtype, srcs, attrs)
Ref new_node(PyObject* op, const Ref& layout, PyObject* dtype, Ref srcs, Ref attrs) {
  if (!layout || !srcs || !attrs) return Ref();
  return Ref(node_make(op, layout.p, dtype, srcs.release(), attrs.release(), Py_None));
}
Ref selector(PyObject* src, int index, const Ref& layout, PyObject* dtype) {
  return new_node(O.gettuple, layout, dtype, list_of({src}), dict_with(N.index, g_small[index]));
}
Ref layout_of(std::initializer_list<long long> dims) {
  Ref t(PyTuple_New(static_cast<Py_ssize_t>(dims.size())));
  Py_ssize_t i = 0;
  for (long long d : dims) {
    PyObject* v = t ? PyLong_FromLongLong(d) : nullptr;
    if (!v) return Ref();
    PyTuple_SET_ITEM(t.p, i++, v);
  }
  return Ref(t ? layout_make(g_layout_type, t.release(), nullptr, 0) : nullptr);
}
long long dim_of(const NodeObj* n, Py_ssize_t i) { return PyLong_AsLongLong(PyTuple_GET_ITEM(as_layout(n->node_layout)->dims, i)); }

using Grads = std::vector<Ref>;
bool filled(const Grads& g) {
  for (const Ref& r : g)
    if (!r) return false;
  return true;
}

// Gradient rules: `node` is plain.  `up` may be any node.
Outcome grad_linear(NodeObj* node, PyObject* up, Grads& out) {
  const bool has_bias = op_is_name(node, O.matmul_bias_bt);
  NodeObj *x = plain_src(node, 0), *w = plain_src(node, 1), *b = has_bias ? plain_src(node, 2) : nullptr;
  if (!x || !w || (has_bias && !b)) return kNotMine;
  Ref xl = contiguous_of(x), wl = contiguous_of(w);
  Ref bwd = new_node(O.linear_grad, xl, x->node_dtype, list_of({up, obj(x), obj(w)}), dict_with(N.has_bias, has_bias ? Py_True : Py_False));
  if (!bwd) return kError;
  out.push_back(selector(bwd.p, 0, xl, x->node_dtype));
  out.push_back(selector(bwd.p, 1, wl, w->node_dtype));
  if (has_bias) out.push_back(selector(bwd.p, 2, contiguous_of(b), b->node_dtype));
  return filled(out) ? kDone : kError;
}
Outcome grad_layer_norm_stats(NodeObj* node, PyObject* up, Grads& out) {
  NodeObj *x = plain_src(node, 0), *gamma = plain_src(node, 1);
  const Py_ssize_t rank = x ? rank_of(as_layout(x->node_layout)) : 0;
  const long long cols = rank > 0 ? dim_of(x, rank - 1) : 0;
  if (!gamma || cols <= 0) return kNotMine;
  Ref rows = layout_of({as_layout(x->node_layout)->numel / cols});
  Ref mean = selector(obj(node), 1, rows, g_small[MG_F32]), rstd = selector(obj(node), 2, rows, g_small[MG_F32]);
  if (!mean || !rstd) return kError;
  Ref xl = contiguous_of(x), gl = contiguous_of(gamma);
  Ref bwd = new_node(O.layer_norm_stats_grad, xl, x->node_dtype, list_of({up, obj(x), obj(gamma), mean.p, rstd.p}), Ref(PyDict_New()));
  if (!bwd) return kError;
  out.push_back(selector(bwd.p, 0, xl, x->node_dtype));
  out.push_back(selector(bwd.p, 1, gl, gamma->node_dtype));
  out.push_back(selector(bwd.p, 2, gl, gamma->node_dtype));
  return filled(out) ? kDone : kError;
}
Outcome grad_packed_attention(NodeObj* node, PyObject* up, Grads& out) {
  NodeObj* qkv = plain_src(node, 0);
  if (!qkv || rank_of(as_layout(qkv->node_layout)) != 5 || !PyList_CheckExact(node->srcs) || !plain_node(up) ||
      !as_layout(as_node(up)->node_layout)->contiguous)
    return kNotMine;
  Ref own = Ref::to(node->node_layout);
  Ref o = selector(obj(node), 0, own, node->node_dtype);
  Ref lse = selector(obj(node), 1, layout_of({dim_of(qkv, 0), dim_of(qkv, 3), dim_of(qkv, 1)}), g_small[MG_F32]);
  if (!o || !lse) return kError;
  Ref srcs = list_of({up, o.p, obj(qkv), lse.p});
  for (Py_ssize_t i = 1; srcs && i < src_count(node); ++i)
    if (PyList_Append(srcs.p, src_of(node, i)) != 0) return kError;
  out.push_back(new_node(O.packed_grad, contiguous_of(qkv), qkv->node_dtype, std::move(srcs), Ref(PyDict_Copy(node->node_attrs))));
  for (Py_ssize_t i = 1; i < src_count(node); ++i) out.push_back(Ref::to(Py_None));
  return filled(out) ? kDone : kError;
}
Outcome grad_cross_entropy(NodeObj* node, PyObject* up, Grads& out) {
  NodeObj *logits = plain_src(node, 0), *labels = plain_src(node, 1);
  if (!logits || !labels) return kNotMine;
  out.push_back(new_node(op_is_name(node, O.ce_ids) ? O.ce_ids_grad : O.ce_grad, contiguous_of(logits), logits->node_dtype,
                         list_of({obj(logits), obj(labels), up}), Ref(PyDict_New())));
  out.push_back(Ref::to(Py_None));
  return filled(out) ? kDone : kError;
}
Outcome grad_relu(NodeObj* node, PyObject* up, Grads& out) {
  out.push_back(new_node(O.relu_grad, contiguous_of(node), node->node_dtype, list_of({obj(node), up}), Ref(PyDict_New())));
  return filled(out) ? kDone : kError;
}
Outcome grad_gettuple(NodeObj*, PyObject* up, Grads& out) {
  out.push_back(Ref::to(up));
  return kDone;
}
Outcome grad_add(NodeObj* node, PyObject* up, Grads& out) {
  for (Py_ssize_t i = 0; i < src_count(node); ++i) {
    NodeObj* s = plain_src(node, i);
    if (!s || !same_dims(s, node)) return kNotMine;
  }
  out.push_back(Ref::to(up));
  out.push_back(Ref::to(up));
  return kDone;
}
Outcome grad_gather(NodeObj* node, PyObject* up, Grads& out) {
  NodeObj *table = plain_src(node, 0), *indices = plain_src(node, 1);
  if (!table || !indices) return kNotMine;
  out.push_back(new_node(O.scatter_add, contiguous_of(table), table->node_dtype, list_of({obj(indices), up}), Ref(PyDict_New())));
  out.push_back(Ref::to(Py_None));
  return filled(out) ? kDone : kError;
}
Outcome grad_reshape(NodeObj* node, PyObject* up, Grads& out) {
  NodeObj* src = plain_src(node, 0);
  if (!src || !plain_node(up)) return kNotMine;
  out.push_back(new_node(O.reshape, contiguous_of(src), as_node(up)->node_dtype, list_of({up}), Ref(PyDict_New())));
  return filled(out) ? kDone : kError;
}
using GradForm = Outcome (*)(NodeObj*, PyObject*, Grads&);
const std::pair<const char*, GradForm> kGradForms[] = {
    {"MATMUL_BT", grad_linear},      {"MATMUL_BIAS_BT", grad_linear}, {"LAYER_NORM_STATS", grad_layer_norm_stats},
    {"FLASH_ATTN_PACKED", grad_packed_attention}, {"CROSS_ENTROPY", grad_cross_entropy}, {"CROSS_ENTROPY_IDS", grad_cross_entropy},
    {"RELU", grad_relu},             {"GETTUPLE", grad_gettuple},     {"ADD", grad_add},
    {"GATHER", grad_gather},         {"RESHAPE", grad_reshape},
};
PyObject* g_own_grads = nullptr;  // the package's own function -> index into kGradForms

// gradient(root, initial_grad, targets, rules): runtime.gradient.
PyObject* py_gradient(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  if (n_args != 4) return PyErr_SetString(PyExc_TypeError, "gradient(root, initial_grad, targets, rules)"), nullptr;
  PyObject* rules = args[3];
  std::vector<Ref> topo;
  if (!toposort(args, 1, topo)) return nullptr;
  Ref map(PyDict_New());
  if (!map || PyDict_SetItem(map.p, args[0], args[1]) != 0) return nullptr;
  for (size_t at = topo.size(); at-- > 0;) {
    PyObject* node = topo[at].p;
    Ref up = Ref::to(PyDict_GetItemWithError(map.p, node));
    if (!up && PyErr_Occurred()) return nullptr;
    if (!up || up.p == Py_None) continue;
    const bool plain = plain_node(node);
    Ref dtype(plain ? new_ref(as_node(node)->node_dtype) : PyObject_CallMethod(node, "dtype", nullptr));
    if (!dtype) return nullptr;
    int is_float = 0;
    for (int d : {MG_F32, MG_F16, MG_BF16}) {
      if (is_float == 0) is_float = PyObject_RichCompareBool(dtype.p, g_small[d], Py_EQ);
      if (is_float < 0) return nullptr;
    }
    if (!is_float) continue;
    PyObject* op = as_node(node)->op_type;
    Ref rule;
    if (PyDict_CheckExact(rules)) {
      rule = Ref::to(PyDict_GetItemWithError(rules, op));
      if (!rule && PyErr_Occurred()) return nullptr;
    } else {
      rule = Ref(PyObject_CallMethod(rules, "get", "O", op));
      if (!rule) return nullptr;
    }
    if (!rule || rule.p == Py_None) {
      const int has = PyObject_IsTrue(as_node(node)->srcs);
      if (has < 0) return nullptr;
      if (has) {
        Ref text(PyUnicode_FromFormat("no gradient rule for op: %S", op));
        Ref e(text ? PyObject_CallFunction(g_mograd_error, "iO", 2, text.p) : nullptr);
        if (e) PyErr_SetObject(g_mograd_error, e.p);
        return nullptr;
      }
      continue;
    }
    Grads grads;
    Outcome done = kNotMine;
    if (plain && PyFunction_Check(rule.p)) {
      PyObject* own = PyDict_GetItemWithError(g_own_grads, rule.p);
      if (!own && PyErr_Occurred()) return nullptr;
      if (own) done = kGradForms[PyLong_AsLong(own)].second(as_node(node), up.p, grads);
      if (done == kError) return nullptr;
    }
    Ref sources = Ref::to(as_node(node)->srcs);
    if (done == kNotMine) {
      grads.clear();
      Ref made(PyObject_CallFunctionObjArgs(rule.p, node, up.p, nullptr));
      Ref list(made ? PySequence_List(made.p) : nullptr);
      if (!list) return nullptr;
      for (Py_ssize_t i = 0; i < PyList_GET_SIZE(list.p); ++i) grads.push_back(Ref::to(PyList_GET_ITEM(list.p, i)));
      sources = Ref(PySequence_List(as_node(node)->srcs));
      if (!sources) return nullptr;
    }
    for (size_t i = 0; i < grads.size() && static_cast<Py_ssize_t>(i) < PySequence_Fast_GET_SIZE(sources.p); ++i) {
      PyObject* g = grads[i].p;
      if (g == Py_None) continue;
      PyObject* src = PySequence_Fast_GET_ITEM(sources.p, static_cast<Py_ssize_t>(i));
      Ref prev = Ref::to(PyDict_GetItemWithError(map.p, src));
      if (!prev && PyErr_Occurred()) return nullptr;
      Ref sum;
      if (prev && prev.p != Py_None) {
        Ref layout(is_node(g) && Py_TYPE(g) == &NodeType ? new_ref(as_node(g)->node_layout) : PyObject_CallMethod(g, "layout", nullptr));
        Ref type(layout ? (Py_TYPE(g) == &NodeType ? new_ref(as_node(g)->node_dtype) : PyObject_CallMethod(g, "dtype", nullptr)) : nullptr);
        if (!type) return nullptr;
        sum = new_node(O.add, layout, type.p, list_of({prev.p, g}), Ref(PyDict_New()));
        if (!sum) return nullptr;
        g = sum.p;
      }
      if (PyDict_SetItem(map.p, src, g) != 0) return nullptr;
    }
  }
  Ref targets(PySequence_List(args[2]));
  if (!targets) return nullptr;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(targets.p); ++i) {
    PyObject* g = PyDict_GetItemWithError(map.p, PyList_GET_ITEM(targets.p, i));
    if (!g && PyErr_Occurred()) return nullptr;
    PyList_SetItem(targets.p, i, new_ref(g ? g : Py_None));
  }
  return targets.release();
}

// Rewrite rules: kDone with `made` the new node, or None for a rule that does not apply.
struct Rewriting {
  const Pass& pass;
  bool single_use(PyObject* n) const { return pass.count(n) <= 1; }
  bool replace(PyObject* old, PyObject* made) const {
    if (PyDict_SetItem(pass.subst, old, made) != 0) return false;
    PyObject* o = PyDict_GetItem(pass.origin, old);
    return PyDict_SetItem(pass.origin, made, o ? o : old) == 0;
  }
};
bool attr_true(const NodeObj* n, PyObject* key) {
  PyObject* v = PyDict_GetItem(n->node_attrs, key);
  return v && PyObject_IsTrue(v) == 1;
}
// int(attrs.get("index", -1)); -2: not an int
long index_of(const NodeObj* n) {
  PyObject* v = PyDict_GetItem(n->node_attrs, N.index);
  if (!v) return -1;
  if (!PyLong_CheckExact(v)) return -2;
  int over = 0;
  const long i = PyLong_AsLongAndOverflow(v, &over);
  return over || i < 0 ? -1 : i;
}
bool reaches(PyObject* from, PyObject* target, int& error) {  // depends_on
  PyObject* const args[] = {from, target};
  Ref r(py_depends_on(nullptr, args, 2));
  error = !r;
  return r && r.p == Py_True;
}
Ref none() { return Ref::to(Py_None); }
// {**attrs, key: True}
Ref attrs_with(const NodeObj* n, PyObject* key) {
  Ref d(PyDict_Copy(n->node_attrs));
  if (d && PyDict_SetItem(d.p, key, Py_True) != 0) return Ref();
  return d;
}
Ref sources_and(const NodeObj* n, PyObject* more) {
  Ref list(PySequence_List(n->srcs));
  if (list && more && PyList_Append(list.p, more) != 0) return Ref();
  return list;
}

Outcome rewrite_matmul_add(NodeObj* node, const Rewriting& w, Ref& made) {
  NodeObj *a = plain_src(node, 0), *b = plain_src(node, 1);
  if (!a || !b) return kNotMine;
  for (auto [mm, other] : {std::pair(a, b), std::pair(b, a)}) {
    if (!op_is_name(mm, O.matmul_bt) || !w.single_use(obj(mm)) || !same_dims(mm, other) || !same_dtype(mm, other)) continue;
    if (src_count(mm) < 2) return kNotMine;
    made = new_node(O.matmul_bt_add, Ref::to(mm->node_layout), node->node_dtype, list_of({src_of(mm, 0), src_of(mm, 1), obj(other)}),
                    Ref(PyDict_New()));
    return made ? kDone : kError;
  }
  return made = none(), kDone;
}
Outcome rewrite_matmul_bias_relu(NodeObj* node, const Rewriting& w, Ref& made) {
  NodeObj* mm = plain_src(node, 0);
  if (!mm) return kNotMine;
  if (!w.single_use(obj(mm))) return made = none(), kDone;
  made = new_node(O.matmul_bias_relu_bt, Ref::to(mm->node_layout), node->node_dtype, sources_and(mm, nullptr), Ref(PyDict_New()));
  return made ? kDone : kError;
}
Outcome rewrite_relu_grad(NodeObj* node, const Rewriting& w, Ref& made) {
  NodeObj *sel = plain_src(node, 1), *lin = sel ? plain_src(sel, 0) : nullptr;
  if (!plain_src(node, 0) || !lin || src_count(lin) < 2) return kNotMine;
  const long index = index_of(sel);
  if (index == -2) return kNotMine;
  if (index != 0 || src_of(lin, 1) != src_of(node, 0) || !w.single_use(obj(sel)) || attr_true(lin, N.relu_mask) ||
      attr_true(lin, N.accumulate))
    return made = none(), kDone;
  Ref fused = new_node(O.linear_grad, Ref::to(lin->node_layout), lin->node_dtype, sources_and(lin, nullptr), attrs_with(lin, N.relu_mask));
  if (!fused || !w.replace(obj(lin), fused.p)) return kError;
  made = selector(fused.p, 0, Ref::to(sel->node_layout), sel->node_dtype);
  return made ? kDone : kError;
}
// ADD(other, GETTUPLE0(producer)) -> GETTUPLE0(producer{op, accumulate}(.., other))
template <bool ACCUMULATE>
Outcome rewrite_add_into(NodeObj* node, const Rewriting& w, Ref& made, PyObject* producer, PyObject* op) {
  NodeObj *a = plain_src(node, 0), *b = plain_src(node, 1);
  if (!a || !b) return kNotMine;
  for (auto [sel, other] : {std::pair(a, b), std::pair(b, a)}) {
    if (!op_is_name(sel, O.gettuple)) continue;
    NodeObj* from = plain_src(sel, 0);
    if (!from) return kNotMine;
    if (!op_is_name(from, producer)) continue;
    const long index = index_of(sel);
    if (index == -2) return kNotMine;
    if (index != 0 || (ACCUMULATE && attr_true(from, N.accumulate)) || !w.single_use(obj(sel)) || !same_dims(sel, other) ||
        !same_dtype(other, sel))
      continue;
    int error = 0;
    const bool cycle = reaches(obj(other), obj(from), error);
    if (error) return kError;
    if (cycle) continue;
    Ref fused = new_node(op, Ref::to(from->node_layout), from->node_dtype, sources_and(from, obj(other)),
                         ACCUMULATE ? attrs_with(from, N.accumulate) : Ref(PyDict_Copy(from->node_attrs)));
    if (!fused || !w.replace(obj(from), fused.p)) return kError;
    made = selector(fused.p, 0, Ref::to(sel->node_layout), sel->node_dtype);
    return made ? kDone : kError;
  }
  return made = none(), kDone;
}
Outcome rewrite_add_into_linear(NodeObj* n, const Rewriting& w, Ref& made) {
  return rewrite_add_into<true>(n, w, made, O.linear_grad, O.linear_grad);
}
Outcome rewrite_add_into_layer_norm(NodeObj* n, const Rewriting& w, Ref& made) {
  return rewrite_add_into<false>(n, w, made, O.layer_norm_stats_grad, O.layer_norm_stats_grad_add);
}
Outcome rewrite_add_into_linear_layer_norm(NodeObj* n, const Rewriting& w, Ref& made) {
  return rewrite_add_into<true>(n, w, made, O.linear_ln_grad, O.linear_ln_grad);
}
Outcome rewrite_linear_into_layer_norm(NodeObj* node, const Rewriting& w, Ref& made) {
  NodeObj* sel = plain_src(node, 0);
  if (!sel) return kNotMine;
  if (!op_is_name(sel, O.gettuple)) return made = none(), kDone;
  const long index = index_of(sel);
  NodeObj* lin = plain_src(sel, 0);
  if (index == -2 || !lin) return kNotMine;
  if (index != 0 || !op_is_name(lin, O.linear_grad) || attr_true(lin, N.relu_mask) || attr_true(lin, N.accumulate) ||
      !w.single_use(obj(sel)))
    return made = none(), kDone;
  NodeObj* h = plain_src(node, 1);
  const bool add = op_is_name(node, O.layer_norm_stats_grad_add);
  if (!h || src_count(lin) < 3 || src_count(node) < (add ? 6 : 5)) return kNotMine;
  if (as_layout(h->node_layout)->numel != as_layout(sel->node_layout)->numel || !same_dtype(node, lin)) return made = none(), kDone;
  // the readers of the product, which may be any nodes
  const Pass& p = w.pass;
  PyObject* origin = PyDict_GetItem(p.origin, obj(lin));
  PyObject* readers = PyDict_GetItem(p.consumers, origin ? origin : obj(lin));
  if (readers && !PyList_CheckExact(readers)) return kNotMine;
  for (Py_ssize_t i = 0; readers && i < PyList_GET_SIZE(readers); ++i) {
    PyObject* c = PyList_GET_ITEM(readers, i);
    if (!plain_node(c) || index_of(as_node(c)) == -2) return kNotMine;
  }
  PyObject* bias = PyDict_GetItem(lin->node_attrs, N.has_bias);
  const int has_bias = bias ? PyObject_IsTrue(bias) : 1;
  if (has_bias < 0) return kError;
  Ref attrs = dict_with(N.has_bias, has_bias ? Py_True : Py_False);
  if (attrs && add && PyDict_SetItem(attrs.p, N.accumulate, Py_True) != 0) return kError;
  Ref srcs = list_of({src_of(lin, 0), src_of(lin, 1), src_of(lin, 2), src_of(node, 1), src_of(node, 2), src_of(node, 3), src_of(node, 4)});
  if (srcs && add && PyList_Append(srcs.p, src_of(node, 5)) != 0) return kError;
  Ref fused = new_node(O.linear_ln_grad, Ref::to(node->node_layout), node->node_dtype, std::move(srcs), std::move(attrs));
  if (!fused) return kError;
  for (Py_ssize_t i = 0; readers && i < PyList_GET_SIZE(readers); ++i) {  // dW and db of the product now come from the new node
    NodeObj* c = as_node(PyList_GET_ITEM(readers, i));
    const long at = op_is_name(c, O.gettuple) ? index_of(c) : -1;
    if (at != 1 && at != 2) continue;
    Ref moved = selector(fused.p, static_cast<int>(at) + 2, Ref::to(c->node_layout), c->node_dtype);
    PyObject* now = p.resolve(obj(c));
    if (!moved || !now || !w.replace(now, moved.p)) return kError;
  }
  made = std::move(fused);
  return kDone;
}
using RewriteForm = Outcome (*)(NodeObj*, const Rewriting&, Ref&);
const std::pair<const char*, RewriteForm> kRewriteForms[] = {
    {"fuse_matmul_add", rewrite_matmul_add},
    {"fuse_matmul_bias_relu", rewrite_matmul_bias_relu},
    {"fuse_relu_grad_into_linear_grad", rewrite_relu_grad},
    {"fuse_add_into_linear_grad", rewrite_add_into_linear},
    {"fuse_add_into_layer_norm_grad", rewrite_add_into_layer_norm},
    {"fuse_linear_grad_into_layer_norm_grad", rewrite_linear_into_layer_norm},
    {"fuse_add_into_linear_layer_norm_grad", rewrite_add_into_linear_layer_norm},
};
PyObject* g_own_rewrites = nullptr;       // the package's own function -> index into kRewriteForms
PyObject* g_simplifier_type = nullptr;    // rewrites.Simplifier
// The methods that the rules in Python call, as the package has them: a program may put others in their place on the class.
struct SimplifierMethod {
  const char* text;
  PyObject *name = nullptr, *own = nullptr;
} g_simplifier_methods[] = {{"single_use"}, {"replace"}, {"consumers_of"}, {"resolve"}};
bool simplifier_methods_own() {
  PyObject* const dict = reinterpret_cast<PyTypeObject*>(g_simplifier_type)->tp_dict;
  for (const SimplifierMethod& m : g_simplifier_methods)
    if (PyDict_GetItem(dict, m.name) != m.own) return false;
  return true;
}

// name -> function of `given`, for every name of `forms`, as function -> place.
template <class Table>
PyObject* own_functions(const Table& forms, PyObject* given) {
  Ref own(PyDict_New());
  size_t i = 0;
  for (const auto& form : forms) {
    PyObject* f = PyDict_GetItemString(given, form.first);
    if (!f) return PyErr_Format(PyExc_KeyError, "%s", form.first), nullptr;
    Ref at(PyLong_FromSize_t(i++));
    if (!own || !at || PyDict_SetItem(own.p, f, at.p) != 0) return nullptr;
  }
  return own.release();
}
// set_gradients(rules, MogradError), set_rewrites(Simplifier, functions by name): the package's own.  (Graphs are
// differentiated and rewritten without the library too, which is what bind() comes with.)
PyObject* py_set_gradients(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 2 || !PyDict_Check(args[0])) return PyErr_SetString(PyExc_TypeError, "set_gradients(rules, MogradError)"), nullptr;
  PyObject* own = own_functions(kGradForms, args[0]);
  if (!own) return nullptr;
  Py_XSETREF(g_own_grads, own);
  Py_XSETREF(g_mograd_error, new_ref(args[1]));
  Py_RETURN_NONE;
}
PyObject* py_set_rewrites(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 2 || !PyType_Check(args[0]) || !PyDict_Check(args[1]))
    return PyErr_SetString(PyExc_TypeError, "set_rewrites(Simplifier, functions)"), nullptr;
  PyObject* own = own_functions(kRewriteForms, args[1]);
  if (!own) return nullptr;
  PyObject* const dict = reinterpret_cast<PyTypeObject*>(args[0])->tp_dict;
  for (SimplifierMethod& m : g_simplifier_methods) {
    if (!m.name) m.name = str_(m.text);
    PyObject* const f = m.name ? PyDict_GetItem(dict, m.name) : nullptr;
    if (!f) return Py_DECREF(own), PyErr_Format(PyExc_AttributeError, "Simplifier.%s", m.text), nullptr;
    Py_XSETREF(m.own, new_ref(f));
  }
  Py_XSETREF(g_own_rewrites, own);
  Py_XSETREF(g_simplifier_type, new_ref(args[0]));
  Py_RETURN_NONE;
}

// A Rule or Pat like `o`, its own object down to the last pattern (a new reference).
PyObject* rule_copy(PyObject* o) {
  PyObject** from = _PyObject_GetDictPtr(o);
  Ref made(Py_TYPE(o)->tp_alloc(Py_TYPE(o), 0));
  PyObject** to = made ? _PyObject_GetDictPtr(made.p) : nullptr;
  if (!from || !*from || !to || !(*to = PyDict_Copy(*from))) return nullptr;
  if (PyObject* pat = PyDict_GetItem(*to, N.pat)) {
    Ref fresh(rule_copy(pat));
    if (!fresh || PyDict_SetItem(*to, N.pat, fresh.p) != 0) return nullptr;
  }
  PyObject* srcs = PyDict_GetItem(*to, N.srcs);
  if (srcs && PyList_Check(srcs)) {
    Ref list(PyList_GetSlice(srcs, 0, PyList_GET_SIZE(srcs)));
    if (!list) return nullptr;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(list.p); ++i) {
      PyObject* fresh = rule_copy(PyList_GET_ITEM(list.p, i));
      if (!fresh) return nullptr;
      PyList_SetItem(list.p, i, fresh);
    }
    if (PyDict_SetItem(*to, N.srcs, list.p) != 0) return nullptr;
  }
  return made.release();
}
// copy_rules(rules): a list of new Rule objects over new patterns.
PyObject* py_copy_rules(PyObject*, PyObject* rules) {
  Ref list(PySequence_List(rules));
  if (!list) return nullptr;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(list.p); ++i) {
    PyObject* fresh = rule_copy(PyList_GET_ITEM(list.p, i));
    if (!fresh) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "copy_rules: not a Rule");
      return nullptr;
    }
    PyList_SetItem(list.p, i, fresh);
  }
  return list.release();
}

// simplify(sim, roots): Simplifier.run_many.
PyObject* py_simplify(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  if (n_args != 2) return PyErr_SetString(PyExc_TypeError, "simplify(sim, roots)"), nullptr;
  PyObject* sim = args[0];
  Ref roots(PySequence_Tuple(args[1]));
  if (!roots) return nullptr;
  std::vector<Ref> topo;
  if (!toposort(PySequence_Fast_ITEMS(roots.p), PySequence_Fast_GET_SIZE(roots.p), topo)) return nullptr;
  Ref subst(PyDict_New()), uses(PyDict_New()), origin(PyDict_New()), consumers(PyDict_New());
  if (!subst || !uses || !origin || !consumers || PyObject_SetAttr(sim, N.subst, subst.p) != 0 ||
      PyObject_SetAttr(sim, N.uses, uses.p) != 0 || PyObject_SetAttr(sim, N.origin, origin.p) != 0 ||
      PyObject_SetAttr(sim, N.consumers, consumers.p) != 0)
    return nullptr;
  Pass pass{sim, subst.p, uses.p, origin.p, consumers.p};
  for (const Ref& v : topo)
    for (Py_ssize_t i = 0; i < src_count(as_node(v.p)); ++i) {
      PyObject* s = src_of(as_node(v.p), i);
      PyObject* list = PyDict_GetItem(consumers.p, s);
      if (!list) {
        Ref fresh(PyList_New(0));
        if (!fresh || PyDict_SetItem(consumers.p, s, fresh.p) != 0) return nullptr;
        list = PyDict_GetItem(consumers.p, s);
      }
      if (PyList_Append(list, v.p) != 0) return nullptr;
    }
  {
    PyObject *k, *v;
    Py_ssize_t pos = 0;
    while (PyDict_Next(consumers.p, &pos, &k, &v))
      if (!pass.set_count(k, static_cast<int>(PyList_GET_SIZE(v)))) return nullptr;
  }
  for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(roots.p); ++i) {  // a root is read by the caller
    PyObject* r = PySequence_Fast_GET_ITEM(roots.p, i);
    if (!pass.set_count(r, pass.count(r) + 1)) return nullptr;
  }
  Ref rules_attr(PyObject_GetAttr(sim, N.rules));
  if (!rules_attr) return nullptr;
  Ref rules(PySequence_Fast(rules_attr.p, "Simplifier.rules"));
  if (!rules) return nullptr;
  // The package's own rules where the pass is its own Simplifier, with no method of a program's own on it or on its class.
  PyObject** sim_dict = Py_TYPE(sim) == reinterpret_cast<PyTypeObject*>(g_simplifier_type) ? _PyObject_GetDictPtr(sim) : nullptr;
  const bool own_pass = sim_dict && *sim_dict && PyDict_GET_SIZE(*sim_dict) == 5 && simplifier_methods_own();
  const Rewriting rewriting{pass};
  struct Compiled {
    Ref pat, func, op;
    RewriteForm form = nullptr;
  };
  std::vector<Compiled> compiled;
  for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(rules.p); ++i) {
    PyObject* r = PySequence_Fast_GET_ITEM(rules.p, i);
    Compiled c;
    c.pat = Ref(PyObject_GetAttr(r, N.pat));
    c.func = Ref(PyObject_GetAttr(r, N.func));
    if (!c.pat || !c.func) return nullptr;
    c.op = Ref(PyObject_GetAttr(c.pat.p, N.op_type));
    if (!c.op) return nullptr;
    if (own_pass && PyFunction_Check(c.func.p)) {
      PyObject* own = PyDict_GetItemWithError(g_own_rewrites, c.func.p);
      if (!own && PyErr_Occurred()) return nullptr;
      if (own) c.form = kRewriteForms[PyLong_AsLong(own)].second;
    }
    compiled.push_back(std::move(c));
  }
  for (const Ref& v : topo) {
    PyObject* node = v.p;
    if (PyDict_GetItem(subst.p, node)) continue;  // a rule that ran on another node has already replaced this one
    Ref now(pass.with_subst(node));
    if (!now) return nullptr;
    int round = 0;
    for (; round < 64; ++round) {
      bool progressed = false;
      for (Compiled& c : compiled) {
        int m = c.op.p == Py_None ? 1 : op_names_equal(c.op.p, as_node(now.p)->op_type);
        if (m > 0) m = pat_matches(c.pat.p, as_node(now.p));
        if (m < 0) return nullptr;
        if (m == 0) continue;
        Ref made;
        Outcome done = c.form && plain_node(now.p) ? c.form(as_node(now.p), rewriting, made) : kNotMine;
        if (done == kError) return PyErr_Occurred() ? nullptr : PyErr_NoMemory();
        if (done == kNotMine) made = Ref(PyObject_CallFunctionObjArgs(c.func.p, now.p, sim, nullptr));
        if (!made) return nullptr;
        if (made.p == Py_None) continue;
        if (!node_ok(made.p) || !pass.set_count(made.p, pass.count(now.p))) return nullptr;
        if (!PyDict_GetItem(origin.p, made.p) && !pass.set_origin(made.p, now.p)) return nullptr;
        now = Ref(pass.with_subst(made.p));
        if (!now) return nullptr;
        progressed = true;
        break;
      }
      if (!progressed) break;
    }
    if (round == 64) return raise_invalid("Simplifier: rewrite rules cycled without converging"), nullptr;
    if (now.p != node && PyDict_SetItem(subst.p, node, now.p) != 0) return nullptr;
  }
  return pass.redirect(roots.p);
}

// ------------------------------------------------------------------------------------------
// Module
// ------------------------------------------------------------------------------------------

// bind(handle, MogradError, c_void_p, fallbacks): the library's functions, from its dlopen handle.
PyObject* py_bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 4) return PyErr_SetString(PyExc_TypeError, "bind(handle, MogradError, c_void_p, fallbacks)"), nullptr;
  void* handle = PyLong_AsVoidPtr(args[0]);
  if (!handle && PyErr_Occurred()) return nullptr;
#define X(f) L.f = reinterpret_cast<decltype(L.f)>(dlsym(handle, #f));
  MG_FUNCTIONS(X)
#undef X
  L.pool_alloc = reinterpret_cast<decltype(L.pool_alloc)>(dlsym(handle, "mg_pool_alloc"));
  L.last_error = reinterpret_cast<decltype(L.last_error)>(dlsym(handle, "mg_last_error"));
  for (int i = 1; i < 4; ++i) Py_INCREF(args[i]);
  Py_XSETREF(g_mograd_error, args[1]);
  Py_XSETREF(g_void_p, args[2]);
  Py_XSETREF(g_fallbacks, args[3]);
  Py_RETURN_NONE;
}
// set_types(AnyBuffer, Layout): the package's own buffers and layouts.
PyObject* py_set_types(PyObject*, PyObject* const* args, Py_ssize_t n) {
  auto derived = [&](int i, PyTypeObject* base) {
    return PyType_Check(args[i]) && PyType_IsSubtype(reinterpret_cast<PyTypeObject*>(args[i]), base);
  };
  if (n != 2 || !derived(0, &BufferType) || !derived(1, &LayoutType))
    return PyErr_SetString(PyExc_TypeError, "set_types(AnyBuffer, Layout)"), nullptr;
  Py_XSETREF(g_buffer_type, reinterpret_cast<PyTypeObject*>(new_ref(args[0])));
  Py_XSETREF(g_layout_type, reinterpret_cast<PyTypeObject*>(new_ref(args[1])));
  Py_RETURN_NONE;
}

// set_rules(run, rules): the package's own exec functions.
PyObject* py_set_rules(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 2 || !PyDict_Check(args[1])) return PyErr_SetString(PyExc_TypeError, "set_rules(run, rules)"), nullptr;
  Py_XSETREF(g_own_run, new_ref(args[0]));
  for (size_t i = 0; i < kFormCount; ++i) {
    PyObject* own = PyDict_GetItemString(args[1], kForms[i].first);
    if (!own) return PyErr_Format(PyExc_KeyError, "%s", kForms[i].first), nullptr;
    Py_XSETREF(g_own_rules[i], new_ref(own));
  }
  Py_RETURN_NONE;
}

// An entry whose containers may fail to grow: a MemoryError instead of an exception through the interpreter.
template <auto F, class... A>
PyObject* guarded(PyObject* self, A... args) {
  try {
    return F(self, args...);
  } catch (const std::bad_alloc&) {
    return PyErr_NoMemory();
  }
}
using FastArgs = PyObject* const*;

PyMethodDef module_methods[] = {
    {"toposort", guarded<py_toposort, PyObject*>, METH_O, "Sources before consumers, each node once."},
    {"depends_on", FAST((guarded<py_depends_on, FastArgs, Py_ssize_t>)), METH_FASTCALL, "depends_on(node, target): whether target is node or feeds it."},
    {"evaluate", FAST((guarded<py_evaluate, FastArgs, Py_ssize_t>)), METH_FASTCALL, "evaluate(nodes, device, run, rules)"},
    {"set_rules", FAST(py_set_rules), METH_FASTCALL, "set_rules(run, rules): the package's own."},
    {"simplify", FAST((guarded<py_simplify, FastArgs, Py_ssize_t>)), METH_FASTCALL, "simplify(sim, roots)"},
    {"gradient", FAST((guarded<py_gradient, FastArgs, Py_ssize_t>)), METH_FASTCALL, "gradient(root, initial_grad, targets, rules)"},
    {"set_gradients", FAST(py_set_gradients), METH_FASTCALL, "set_gradients(rules, MogradError): the package's own."},
    {"set_rewrites", FAST(py_set_rewrites), METH_FASTCALL, "set_rewrites(Simplifier, functions): the package's own."},
    {"copy_rules", py_copy_rules, METH_O, "copy_rules(rules): new Rule objects over new patterns"},
    {"bind", FAST(py_bind), METH_FASTCALL, "bind(handle, MogradError, c_void_p, fallbacks)"},
    {"set_types", FAST(py_set_types), METH_FASTCALL, "set_types(AnyBuffer, Layout)"},
    {nullptr, nullptr, 0, nullptr}};
PyMethodDef library_methods[] = {
#define X(f) {#f, FAST(py_##f), METH_FASTCALL, nullptr},
    MG_FUNCTIONS(X)
#undef X
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_graph", "Native host path of mograd_amd.", -1, module_methods, nullptr,
                          nullptr, nullptr, nullptr};

bool add_type(PyObject* m, PyTypeObject* t, const char* name) {
  if (PyType_Ready(t) != 0) return false;
  Py_INCREF(t);
  return PyModule_AddObject(m, name, reinterpret_cast<PyObject*>(t)) == 0;
}

}  // namespace

PyMODINIT_FUNC PyInit__graph() {
  LayoutType.tp_name = "mograd_amd._graph.Layout";
  LayoutType.tp_basicsize = sizeof(LayoutObj);
  LayoutType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE;
  LayoutType.tp_new = layout_new;
  LayoutType.tp_dealloc = layout_dealloc;
  LayoutType.tp_members = layout_members;
  LayoutType.tp_methods = layout_methods;
  LayoutType.tp_richcompare = layout_richcompare;
  LayoutType.tp_hash = layout_hash;
  LayoutType.tp_repr = layout_repr;

  NodeType.tp_name = "mograd_amd._graph.Node";
  NodeType.tp_basicsize = sizeof(NodeObj);
  NodeType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC | Py_TPFLAGS_BASETYPE;
  NodeType.tp_dictoffset = offsetof(NodeObj, dict);
  NodeType.tp_weaklistoffset = offsetof(NodeObj, weakrefs);
  NodeType.tp_doc =
      "Just enough of an op node for the exec functions: its own layout and dtype, the layouts of its\n"
      "sources, and its attributes (mograd/op.mojo:124-185).  `bufs` is what the reference keeps in op().buf\n"
      "(mograd/scheduler.mojo:74-78): a leaf's buffer, or the results of an evaluated node.";
  NodeType.tp_new = node_new;
  NodeType.tp_init = node_init;
  NodeType.tp_dealloc = node_dealloc;
  NodeType.tp_traverse = node_traverse;
  NodeType.tp_clear = node_clear;
  NodeType.tp_getset = node_fields;
  NodeType.tp_methods = node_methods;
  NodeType.tp_repr = node_repr;

  StorageType.tp_name = "mograd_amd._graph.Storage";
  StorageType.tp_basicsize = sizeof(StorageObj);
  StorageType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC;
  StorageType.tp_traverse = storage_traverse;
  StorageType.tp_new = storage_new;
  StorageType.tp_dealloc = storage_dealloc;
  StorageType.tp_members = storage_members;

  BufferType.tp_name = "mograd_amd._graph.Buffer";
  BufferType.tp_basicsize = sizeof(BufferObj);
  BufferType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC;
  BufferType.tp_traverse = buffer_traverse;
  BufferType.tp_getset = buffer_fields;
  BufferType.tp_new = buffer_new;
  BufferType.tp_dealloc = buffer_dealloc;
  BufferType.tp_members = buffer_members;
  BufferType.tp_methods = buffer_methods;

  N = {str_("index"), str_("eps"), str_("has_bias"), str_("accumulate"), str_("relu_mask"), str_("scale"), str_("is_causal"),
       str_("stream"), str_("pending"), str_("func"), str_("pat"), str_("op_type"), str_("srcs"), str_("subst"), str_("uses"),
       str_("origin"), str_("consumers"), str_("rules")};
  O = {str_("LINEAR_GRAD"), str_("GETTUPLE"), str_("LAYER_NORM_STATS_GRAD"), str_("LAYER_NORM_STATS_GRAD_ADD"),
       str_("FLASH_ATTN_PACKED_GRAD"), str_("CROSS_ENTROPY_GRAD"), str_("CROSS_ENTROPY_IDS"), str_("CROSS_ENTROPY_IDS_GRAD"),
       str_("RELU_GRAD"), str_("SCATTER_ADD"), str_("RESHAPE"), str_("ADD"), str_("MATMUL_BT"), str_("MATMUL_BIAS_BT"),
       str_("MATMUL_BT_ADD"), str_("MATMUL_BIAS_RELU_BT"), str_("LINEAR_LAYER_NORM_GRAD")};
  for (int i = 0; i < 5; ++i) g_small[i] = PyLong_FromLong(i);
  PyObject* m = PyModule_Create(&module_def);
  if (!m) return nullptr;
  if (!add_type(m, &LayoutType, "Layout") || !add_type(m, &NodeType, "Node") || !add_type(m, &StorageType, "Storage") ||
      !add_type(m, &BufferType, "Buffer"))
    return nullptr;
  g_forms = PyDict_New();
  for (size_t i = 0; i < kFormCount; ++i) {
    Ref v(PyLong_FromSize_t(i)), k(str_(kForms[i].first));
    if (!v || PyDict_SetItem(g_forms, k.p, v.p) != 0) return nullptr;
  }
  PyObject* lib = PyDict_New();
  for (PyMethodDef* d = library_methods; lib && d->ml_name; ++d) {
    Ref f(PyCFunction_New(d, nullptr));
    if (!f || PyDict_SetItemString(lib, d->ml_name, f.p) != 0) return nullptr;
  }
  if (!lib || PyModule_AddObject(m, "library", lib) != 0) return nullptr;
  return m;
}

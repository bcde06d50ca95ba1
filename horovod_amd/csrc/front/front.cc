// front.cc -- what the torch front end does for every tensor and every rank, as a CPython extension module.  A step
// hands over hundreds of tensors, and a simulated world of R ranks asks a callback for R - 1 more of each: checking them
// and taking their addresses in Python cost 2.2 us per tensor and 0.35 us per peer, several times what the kernels
// behind them take (161 gradients of ResNet-50 from eight ranks: 960 us a step, 150 of it kernels).
//
// Nothing is decided here that engine.py and mpi_ops.py do not decide as well: a call that is not the plain case
// (a tensor of a subclass or under a transform, a name already in flight, an unknown op ...) is handed back, and the
// Python code behind it does the work or raises the error.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Dtype.h>

#include <c10/core/impl/VirtualGuardImpl.h>
#include <structmember.h>

#include <cstdint>
#include <unordered_set>
#include <vector>

// What this was built for, as _lib.front_for() says it; read before the module is imported.
extern "C" {
extern const char hvd_front_built_for[];
const char hvd_front_built_for[] = HVD_FRONT_FOR;
}

namespace {

// Owned reference.
class Ref {
 public:
  Ref() = default;
  explicit Ref(PyObject* p) : p_(p) {}
  Ref(Ref&& o) noexcept : p_(o.release()) {}
  Ref(const Ref&) = delete;
  Ref& operator=(Ref&& o) noexcept {
    Py_XSETREF(p_, o.release());
    return *this;
  }
  ~Ref() { Py_XDECREF(p_); }
  PyObject* get() const { return p_; }
  PyObject* release() {
    PyObject* p = p_;
    p_ = nullptr;
    return p;
  }
  explicit operator bool() const { return p_ != nullptr; }

 private:
  PyObject* p_ = nullptr;
};
PyObject* borrowed(PyObject* p) {
  Py_XINCREF(p);
  return p;
}

// ---- the records of a request (the fields are those that engine.py describes) --------------------

template <typename T>
int traverse(PyObject* self, visitproc visit, void* arg) {
  for (PyObject* o : reinterpret_cast<T*>(self)->objects) Py_VISIT(o);
  return 0;
}
template <typename T>
int clear(PyObject* self) {
  for (PyObject*& o : reinterpret_cast<T*>(self)->objects) Py_CLEAR(o);
  return 0;
}
template <typename T>
void dealloc(PyObject* self) {
  PyObject_GC_UnTrack(self);
  clear<T>(self);
  Py_TYPE(self)->tp_free(self);
}
template <typename T>
T* make(PyTypeObject* type) {  // tp_alloc clears the memory and starts the tracking
  return reinterpret_cast<T*>(type->tp_alloc(type, 0));
}
template <typename T>
PyTypeObject type_of(const char* name, PyMemberDef* members, newfunc make_new) {
  PyTypeObject t = {PyVarObject_HEAD_INIT(nullptr, 0)};
  t.tp_name = name;
  t.tp_basicsize = sizeof(T);
  t.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC;
  t.tp_traverse = traverse<T>;
  t.tp_clear = clear<T>;
  t.tp_dealloc = dealloc<T>;
  t.tp_members = members;
  t.tp_new = make_new;
  return t;
}
#define OBJECT_AT(T, field) (Py_ssize_t)(offsetof(T, objects) + T::field * sizeof(PyObject*))

struct Entry {
  enum { name, tensor, output, parts, kObjects };
  PyObject_HEAD
  PyObject* objects[kObjects];
  long long count;
};
PyMemberDef entry_members[] = {
    {"name", T_OBJECT, OBJECT_AT(Entry, name), READONLY, nullptr},
    {"tensor", T_OBJECT, OBJECT_AT(Entry, tensor), READONLY, nullptr},
    {"output", T_OBJECT, OBJECT_AT(Entry, output), READONLY, nullptr},
    {"parts", T_OBJECT, OBJECT_AT(Entry, parts), 0, "allgather: what every rank contributes, rank 0 first"},
    {"count", T_LONGLONG, offsetof(Entry, count), READONLY, nullptr},
    {nullptr, 0, 0, 0, nullptr}};
PyObject* entry_new(PyTypeObject* type, PyObject* args, PyObject*) {
  PyObject *name, *tensor, *output;
  if (!PyArg_ParseTuple(args, "OOO", &name, &tensor, &output)) return nullptr;
  Ref count(PyObject_CallMethod(tensor, "numel", nullptr));
  if (!count) return nullptr;
  const long long n = PyLong_AsLongLong(count.get());
  if (n == -1 && PyErr_Occurred()) return nullptr;
  Entry* e = make<Entry>(type);
  if (!e) return nullptr;
  e->objects[Entry::name] = borrowed(name);
  e->objects[Entry::tensor] = borrowed(tensor);
  e->objects[Entry::output] = borrowed(output);
  e->count = n;
  return reinterpret_cast<PyObject*>(e);
}
PyTypeObject entry_type = type_of<Entry>("horovod_amd.torch._front.Entry", entry_members, entry_new);

struct Request {
  enum { kind, entries, device, producer, markers, error, kObjects };
  PyObject_HEAD
  PyObject* objects[kObjects];
  int op, tensor_dtype, wire_dtype;
  double prescale, postscale;
  Py_ssize_t left;  // entries whose response has not been executed
  char submitted, grouped;
};
PyMemberDef request_members[] = {
    {"kind", T_OBJECT, OBJECT_AT(Request, kind), READONLY, nullptr},
    {"entries", T_OBJECT, OBJECT_AT(Request, entries), READONLY, nullptr},
    {"device", T_OBJECT, OBJECT_AT(Request, device), READONLY, nullptr},
    {"producer", T_OBJECT, OBJECT_AT(Request, producer), 0, "the framework stream that was current at enqueue"},
    {"markers", T_OBJECT, OBJECT_AT(Request, markers), 0, "one Marker per fused response with one of the entries"},
    {"error", T_OBJECT, OBJECT_AT(Request, error), 0, nullptr},
    {"op", T_INT, offsetof(Request, op), 0, nullptr},
    {"tensor_dtype", T_INT, offsetof(Request, tensor_dtype), 0, nullptr},
    {"wire_dtype", T_INT, offsetof(Request, wire_dtype), 0, nullptr},
    {"prescale", T_DOUBLE, offsetof(Request, prescale), 0, nullptr},
    {"postscale", T_DOUBLE, offsetof(Request, postscale), 0, nullptr},
    {"submitted", T_BOOL, offsetof(Request, submitted), 0, nullptr},
    {"grouped", T_BOOL, offsetof(Request, grouped), 0, nullptr},
    {nullptr, 0, 0, 0, nullptr}};
PyObject* g_allreduce;  // the kinds, interned
PyObject* g_allgather;
Request* new_request(PyTypeObject* type, PyObject* entries, PyObject* device, PyObject* kind) {
  Ref markers(PyList_New(0));
  if (!markers) return nullptr;
  Request* r = make<Request>(type);
  if (!r) return nullptr;
  r->objects[Request::kind] = borrowed(kind);
  r->objects[Request::entries] = borrowed(entries);
  r->objects[Request::device] = borrowed(device);
  r->objects[Request::markers] = markers.release();
  r->left = PyList_GET_SIZE(entries);
  return r;
}
PyObject* request_new(PyTypeObject* type, PyObject* args, PyObject* kwargs) {
  static const char* names[] = {"entries", "op", "prescale", "postscale", "tensor_dtype", "wire_dtype",
                                "device", "kind", "grouped", nullptr};
  PyObject *entries, *pre, *post, *device, *kind = g_allreduce;
  int op, tensor_dtype, wire_dtype, grouped = 0;
  if (!PyArg_ParseTupleAndKeywords(args, kwargs, "O!iOOiiO|Up", const_cast<char**>(names), &PyList_Type, &entries, &op, &pre,
                                   &post, &tensor_dtype, &wire_dtype, &device, &kind, &grouped))
    return nullptr;
  Ref prescale(PyNumber_Float(pre)), postscale(prescale ? PyNumber_Float(post) : nullptr);  // what float() takes, text too
  if (!postscale) return nullptr;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(entries); ++i)
    if (Py_TYPE(PyList_GET_ITEM(entries, i)) != &entry_type) {
      PyErr_SetString(PyExc_TypeError, "a request holds entries");
      return nullptr;
    }
  Request* r = new_request(type, entries, device, kind);
  if (!r) return nullptr;
  r->op = op;
  r->tensor_dtype = tensor_dtype;
  r->wire_dtype = wire_dtype;
  r->prescale = PyFloat_AS_DOUBLE(prescale.get());
  r->postscale = PyFloat_AS_DOUBLE(postscale.get());
  r->grouped = (char)grouped;
  return reinterpret_cast<PyObject*>(r);
}
PyTypeObject request_type = type_of<Request>("horovod_amd.torch._front.Request", request_members, request_new);

struct Marker {
  enum { stream, event, keepalive, kObjects };
  PyObject_HEAD
  PyObject* objects[kObjects];
  long refs;
  char done;
};
PyMemberDef marker_members[] = {
    {"stream", T_OBJECT, OBJECT_AT(Marker, stream), 0, nullptr},
    {"event", T_OBJECT, OBJECT_AT(Marker, event), 0, nullptr},
    {"keepalive", T_OBJECT, OBJECT_AT(Marker, keepalive), 0, "the other ranks' tensors, until the response has completed"},
    {"refs", T_LONG, offsetof(Marker, refs), 0, nullptr},
    {"done", T_BOOL, offsetof(Marker, done), 0, nullptr},
    {nullptr, 0, 0, 0, nullptr}};
PyObject* marker_new(PyTypeObject* type, PyObject* args, PyObject*) {
  PyObject *stream, *event, *keepalive;
  long refs;
  if (!PyArg_ParseTuple(args, "OOlO", &stream, &event, &refs, &keepalive)) return nullptr;
  Marker* m = make<Marker>(type);
  if (!m) return nullptr;
  m->objects[Marker::stream] = borrowed(stream);
  m->objects[Marker::event] = borrowed(event);
  m->objects[Marker::keepalive] = borrowed(keepalive);
  m->refs = refs;
  return reinterpret_cast<PyObject*>(m);
}
PyTypeObject marker_type = type_of<Marker>("horovod_amd.torch._front.Marker", marker_members, marker_new);

Entry* as_entry(PyObject* o) { return reinterpret_cast<Entry*>(o); }
Request* as_request(PyObject* o) { return reinterpret_cast<Request*>(o); }

// ---- tensors -------------------------------------------------------------------------------------

// A tensor (or parameter) whose memory is its own: no subclass, no wrapper of a transform.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckTypeExact(Py_TYPE(o))) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  constexpr c10::DispatchKeySet kWrapped({c10::DispatchKey::Python, c10::DispatchKey::Functionalize,
                                          c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                          c10::DispatchKey::BatchedNestedTensor, c10::DispatchKey::NestedTensor});
  if (!t.defined() || t.layout() != c10::kStrided || !t.has_storage() || t.key_set().has_any(kWrapped)) return nullptr;
  return &t;
}

// The wire code of an element type (horovod's DataType), or -1.
int code_of(c10::ScalarType t) {
  switch (t) {
  case c10::ScalarType::Byte: return 0;
  case c10::ScalarType::Char: return 1;
  case c10::ScalarType::Short: return 3;
  case c10::ScalarType::Int: return 4;
  case c10::ScalarType::Long: return 5;
  case c10::ScalarType::Half: return 6;
  case c10::ScalarType::Float: return 7;
  case c10::ScalarType::Double: return 8;
  case c10::ScalarType::Bool: return 9;
  default: return -1;
  }
}
constexpr int kHalf = 6, kDouble = 8;
constexpr int64_t kSizes[] = {1, 1, 2, 2, 4, 8, 2, 4, 8, 1};

uint64_t address(const at::Tensor& t) { return (uint64_t)reinterpret_cast<uintptr_t>(t.data_ptr()); }

// The address that Python's data_ptr() gives; false with an error set.
bool address_of(PyObject* o, uint64_t* out) {
  if (const at::Tensor* t = plain(o)) {
    *out = address(*t);
    return true;
  }
  Ref r(PyObject_CallMethod(o, "data_ptr", nullptr));
  if (!r) return false;
  *out = PyLong_AsUnsignedLongLong(r.get());
  return !PyErr_Occurred();
}

// C++ exceptions stop here.
template <typename F>
PyObject* guarded(F&& f) {
  try {
    return f();
  } catch (const std::bad_alloc&) {
    return PyErr_NoMemory();
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

// ---- submission and completion -------------------------------------------------------------------

PyObject* g_pending;  // what State.finish returns for a handle that is not finished here

struct State {
  enum { inflight, queue, handles, next_handle, noname, release, producer, kObjects };
  PyObject_HEAD
  PyObject* objects[kObjects];
  long size, local_size;
  int64_t producer_id;  // of the tuple in objects[producer]
  int producer_device, producer_type;
};

// (stream_id, device_index, device_type) of the current stream, as torch._C._cuda_getCurrentStream() gives it.
PyObject* current_producer(State* s) {
  const c10::impl::VirtualGuardImpl impl(c10::DeviceType::CUDA);
  const c10::Stream now = impl.getStream(impl.getDevice());
  const int64_t id = now.id();
  const int device = now.device_index(), type = (int)now.device_type();
  PyObject*& known = s->objects[State::producer];
  if (!known || id != s->producer_id || device != s->producer_device || type != s->producer_type) {
    PyObject* t = Py_BuildValue("(Lii)", (long long)id, device, type);
    if (!t) return nullptr;
    Py_XSETREF(known, t);
    s->producer_id = id;
    s->producer_device = device;
    s->producer_type = type;
  }
  return borrowed(known);
}

// What the counter in a list of one comes to next; counted() moves it there.  False with an error set.
bool next_of(PyObject* counter, long long* value) {
  *value = PyLong_AsLongLong(PyList_GET_ITEM(counter, 0)) + 1;
  return !PyErr_Occurred();
}
bool counted(PyObject* counter, long long value) {
  PyObject* next = PyLong_FromLongLong(value);
  return next && PyList_SetItem(counter, 0, next) == 0;
}

bool number(PyObject* o, double* out) {
  if (PyFloat_CheckExact(o)) {
    *out = PyFloat_AS_DOUBLE(o);
    return true;
  }
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
  if (overflow || v > (1ll << 53) || v < -(1ll << 53)) return false;
  *out = (double)v;
  return true;
}

bool power_of_two(long n) { return n > 0 && (n & (n - 1)) == 0; }

struct Call {
  int dtype, on_wire, reduction;
  double pre, post;
};

// What an allreduce of tensors like `t` is, from the arguments that follow the name; false for one that Python has to
// look at.
bool call_of(const State* s, const at::Tensor& t, PyObject* op, PyObject* pre, PyObject* post, PyObject* wire, Call* c) {
  if (!t.is_cuda() || !PyLong_CheckExact(op) || !number(pre, &c->pre) || !number(post, &c->post)) return false;
  c->dtype = c->on_wire = code_of(t.scalar_type());
  if (wire != Py_None) {
    if (!THPDtype_Check(wire)) return false;
    c->on_wire = code_of(reinterpret_cast<THPDtype*>(wire)->scalar_type);
  }
  if (c->dtype < 0 || c->on_wire < 0) return false;
  c->reduction = 1;
  switch (PyLong_AsLong(op)) {
  case 0: c->post /= (double)s->size; return true;  // Average
  case 1: return true;                              // Sum
  case 2:                                           // Adasum
    c->post /= (double)s->local_size;
    c->reduction = 2;
    return c->on_wire >= kHalf && c->on_wire <= kDouble && power_of_two(s->size / s->local_size);
  default:
    PyErr_Clear();  // of a number beyond a long
    return false;
  }
}

// Whether a tensor and its output can go with tensors like `first`.
bool fits(const at::Tensor& first, const at::Tensor* t, const at::Tensor* o) {
  if (!t || !o || !t->is_contiguous() || t->scalar_type() != first.scalar_type() || t->device() != first.device())
    return false;
  return o == t || (o->sizes() == t->sizes() && o->scalar_type() == t->scalar_type() && o->device() == t->device() &&
                    o->is_contiguous());
}

PyObject* new_entry(PyObject* name, PyObject* tensor, PyObject* output, const at::Tensor& t) {
  Entry* e = make<Entry>(&entry_type);
  if (!e) return nullptr;
  e->objects[Entry::name] = borrowed(name);
  e->objects[Entry::tensor] = borrowed(tensor);
  e->objects[Entry::output] = borrowed(output);
  e->count = t.numel();
  return reinterpret_cast<PyObject*>(e);
}

// Queues a request of the entries, none of whose names is in flight; returns its handle.
PyObject* enqueue(State* s, PyObject* entries, const at::Tensor& first, const Call& c, bool grouped) {
  Ref device(PyLong_FromLong(first.device().index()));
  if (!device) return nullptr;
  Ref request(reinterpret_cast<PyObject*>(new_request(&request_type, entries, device.get(), g_allreduce)));
  if (!request) return nullptr;
  Request* r = as_request(request.get());
  r->op = c.reduction;
  r->tensor_dtype = c.dtype;
  r->wire_dtype = c.on_wire;
  r->prescale = c.pre;
  r->postscale = c.post;
  r->grouped = grouped;
  r->objects[Request::producer] = current_producer(s);
  if (!r->objects[Request::producer]) return nullptr;
  long long handle;
  if (!next_of(s->objects[State::next_handle], &handle) || !counted(s->objects[State::next_handle], handle)) return nullptr;
  Ref h(PyLong_FromLongLong(handle));
  if (!h) return nullptr;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(entries); ++i) {
    PyObject* name = as_entry(PyList_GET_ITEM(entries, i))->objects[Entry::name];
    if (PyDict_SetItem(s->objects[State::inflight], name, request.get())) return nullptr;
  }
  if (PyDict_SetItem(s->objects[State::handles], h.get(), request.get()) ||
      PyList_Append(s->objects[State::queue], request.get()))
    return nullptr;
  return h.release();
}

// submit(tensor, output, name, op, prescale, postscale, wire dtype): the handle of an allreduce of one tensor, or None for
// a call that Python has to look at (nothing has happened then).
PyObject* state_submit(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    if (nargs != 7) {
      PyErr_SetString(PyExc_TypeError, "submit takes 7 arguments");
      return nullptr;
    }
    State* s = reinterpret_cast<State*>(self);
    PyObject* name = args[2];
    const at::Tensor *t = plain(args[0]), *o = args[1] == args[0] ? t : plain(args[1]);
    Call c;
    if (!t || !fits(*t, t, o) || !call_of(s, *t, args[3], args[4], args[5], args[6], &c)) Py_RETURN_NONE;
    Ref full;
    long long unnamed = 0;
    if (name != Py_None) {
      if (!PyUnicode_CheckExact(name)) Py_RETURN_NONE;
      full = Ref(PyUnicode_FromFormat("allreduce.%U", name));
    } else {
      if (!next_of(s->objects[State::noname], &unnamed)) return nullptr;
      full = Ref(PyUnicode_FromFormat("allreduce.noname.%lld", unnamed));
    }
    if (!full) return nullptr;
    const int there = PyDict_Contains(s->objects[State::inflight], full.get());
    if (there < 0) return nullptr;
    if (there) Py_RETURN_NONE;  // before the name is counted, which Python does
    if (unnamed && !counted(s->objects[State::noname], unnamed)) return nullptr;
    Ref entries(PyList_New(1));
    if (!entries) return nullptr;
    PyObject* entry = new_entry(full.get(), args[0], args[1], *t);
    if (!entry) return nullptr;
    PyList_SET_ITEM(entries.get(), 0, entry);
    return enqueue(s, entries.get(), *t, c, false);
  });
}

// submit_group(tensors, outputs, name, op, prescale, postscale, wire dtype): the same for the tensors of a group, under
// the names that horovod/torch/mpi_ops_v2.cc:207 gives them.
PyObject* state_submit_group(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
  return guarded([&]() -> PyObject* {
    if (nargs != 7 || !PyList_CheckExact(args[0]) || !PyList_CheckExact(args[1]) || !PyUnicode_CheckExact(args[2])) {
      PyErr_SetString(PyExc_TypeError, "submit_group takes two lists, a name and 4 arguments more");
      return nullptr;
    }
    State* s = reinterpret_cast<State*>(self);
    const Py_ssize_t n = PyList_GET_SIZE(args[0]);
    if (n == 0 || PyList_GET_SIZE(args[1]) != n) Py_RETURN_NONE;
    const at::Tensor* first = plain(PyList_GET_ITEM(args[0], 0));
    Call c;
    if (!first || !call_of(s, *first, args[3], args[4], args[5], args[6], &c)) Py_RETURN_NONE;
    Ref entries(PyList_New(n));
    if (!entries) return nullptr;
    for (Py_ssize_t i = 0; i < n; ++i) {
      PyObject *tensor = PyList_GET_ITEM(args[0], i), *output = PyList_GET_ITEM(args[1], i);
      const at::Tensor *t = plain(tensor), *o = output == tensor ? t : plain(output);
      if (!fits(*first, t, o)) Py_RETURN_NONE;
      Ref name(PyUnicode_FromFormat("%U_%zdof%zd", args[2], i + 1, n));
      if (!name) return nullptr;
      const int there = PyDict_Contains(s->objects[State::inflight], name.get());
      if (there < 0) return nullptr;
      if (there) Py_RETURN_NONE;
      PyObject* entry = new_entry(name.get(), tensor, output, *t);
      if (!entry) return nullptr;
      PyList_SET_ITEM(entries.get(), i, entry);
    }
    return enqueue(s, entries.get(), *first, c, true);
  });
}

// finish(handle): the output (or outputs) of a request whose responses have all been waited for, or the pending object.
PyObject* state_finish(PyObject* self, PyObject* handle) {
  State* s = reinterpret_cast<State*>(self);
  PyObject* o = PyDict_GetItemWithError(s->objects[State::handles], handle);
  if (!o) return PyErr_Occurred() ? nullptr : borrowed(g_pending);
  if (Py_TYPE(o) != &request_type) return borrowed(g_pending);
  Request* r = as_request(o);
  PyObject *markers = r->objects[Request::markers], *error = r->objects[Request::error];
  if (!r->submitted || (error && error != Py_None) || !markers || !PyList_CheckExact(markers)) return borrowed(g_pending);
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(markers); ++i) {
    PyObject* m = PyList_GET_ITEM(markers, i);
    if (Py_TYPE(m) != &marker_type || !reinterpret_cast<Marker*>(m)->done) return borrowed(g_pending);
  }
  Ref hold(borrowed(o)), list(borrowed(markers));
  if (PyDict_DelItem(s->objects[State::handles], handle)) return nullptr;
  Ref none(PyList_New(0));
  if (!none) return nullptr;
  Py_SETREF(r->objects[Request::markers], none.release());
  PyObject* entries = r->objects[Request::entries];
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(entries); ++i) {
    PyObject* name = as_entry(PyList_GET_ITEM(entries, i))->objects[Entry::name];
    if (PyDict_DelItem(s->objects[State::inflight], name)) PyErr_Clear();  // it may be gone already
  }
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(list.get()); ++i) {
    PyObject* m = PyList_GET_ITEM(list.get(), i);
    if (--reinterpret_cast<Marker*>(m)->refs == 0) {  // the last request of the response hands the event back
      Ref done(PyObject_CallFunctionObjArgs(s->objects[State::release], m, nullptr));
      if (!done) return nullptr;
    }
  }
  if (!r->grouped && PyList_GET_SIZE(entries) >= 1)
    return borrowed(as_entry(PyList_GET_ITEM(entries, 0))->objects[Entry::output]);
  Ref outputs(PyList_New(PyList_GET_SIZE(entries)));
  if (!outputs) return nullptr;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(entries); ++i)
    PyList_SET_ITEM(outputs.get(), i, borrowed(as_entry(PyList_GET_ITEM(entries, i))->objects[Entry::output]));
  return outputs.release();
}

PyObject* state_producer(PyObject* self, PyObject*) {
  return guarded([&] { return current_producer(reinterpret_cast<State*>(self)); });
}

PyObject* state_new(PyTypeObject* type, PyObject* args, PyObject*) {
  long size, local_size;
  PyObject *inflight, *queue, *handles, *next_handle, *noname, *release;
  if (!PyArg_ParseTuple(args, "llO!O!O!O!O!O", &size, &local_size, &PyDict_Type, &inflight, &PyList_Type, &queue,
                        &PyDict_Type, &handles, &PyList_Type, &next_handle, &PyList_Type, &noname, &release))
    return nullptr;
  if (size < 1 || local_size < 1 || PyList_GET_SIZE(next_handle) != 1 || PyList_GET_SIZE(noname) != 1) {
    PyErr_SetString(PyExc_ValueError, "bad sizes or counters");
    return nullptr;
  }
  State* s = make<State>(type);
  if (!s) return nullptr;
  PyObject* held[] = {inflight, queue, handles, next_handle, noname, release};
  for (int i = 0; i < State::producer; ++i) s->objects[i] = borrowed(held[i]);
  s->size = size;
  s->local_size = local_size;
  return reinterpret_cast<PyObject*>(s);
}
PyMethodDef state_methods[] = {
    {"submit", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(state_submit)), METH_FASTCALL, nullptr},
    {"submit_group", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(state_submit_group)), METH_FASTCALL, nullptr},
    {"finish", state_finish, METH_O, nullptr},
    {"producer", state_producer, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyTypeObject state_type = type_of<State>("horovod_amd.torch._front.State", nullptr, state_new);

// ---- a cycle -------------------------------------------------------------------------------------

// take(queue): a list of what the queue holds, which is empty then.  One step for the threads that append to it: nothing
// between the two copies allocates an object or runs Python code, so the interpreter changes no threads there.
PyObject* take(PyObject*, PyObject* queue) {
  if (!PyList_CheckExact(queue)) {
    PyErr_SetString(PyExc_TypeError, "the queue is a list");
    return nullptr;
  }
  Ref taken(PyList_New(0));
  if (!taken || PyList_SetSlice(taken.get(), 0, 0, queue) || PyList_SetSlice(queue, 0, PyList_GET_SIZE(queue), nullptr))
    return nullptr;
  return taken.release();
}

typedef int (*Fuse)(const int64_t* sizes, const int* keys, int n, int64_t threshold, int unpadded, int* group_of);

// plan(requests, padded, threshold, address of hvd_adapter_fuse_keyed): the fused responses, each a list of (request,
// entry).
PyObject* plan(PyObject*, PyObject* args) {
  PyObject* requests;
  int padded;
  long long threshold;
  unsigned long long fuse;
  if (!PyArg_ParseTuple(args, "O!pLK", &PyList_Type, &requests, &padded, &threshold, &fuse)) return nullptr;
  return guarded([&]() -> PyObject* {
    struct Class {
      const Request* r;
      bool gathers;
      long device;
    };
    std::vector<Class> classes;
    std::vector<std::pair<PyObject*, PyObject*>> flat;
    std::vector<int64_t> sizes;
    std::vector<int> keys;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(requests); ++i) {
      PyObject* o = PyList_GET_ITEM(requests, i);
      if (Py_TYPE(o) != &request_type) {
        PyErr_SetString(PyExc_TypeError, "plan takes requests");
        return nullptr;
      }
      const Request* r = as_request(o);
      const bool gathers = PyUnicode_Compare(r->objects[Request::kind], g_allgather) == 0;
      long device = -1;
      if (r->objects[Request::device] && r->objects[Request::device] != Py_None) {
        device = PyLong_AsLong(r->objects[Request::device]);
        if (device == -1 && PyErr_Occurred()) return nullptr;
      }
      size_t key = 0;
      for (; key < classes.size(); ++key) {
        const Class& c = classes[key];
        if (c.gathers == gathers && c.device == device && c.r->op == r->op && c.r->tensor_dtype == r->tensor_dtype &&
            c.r->wire_dtype == r->wire_dtype && c.r->prescale == r->prescale && c.r->postscale == r->postscale)
          break;
      }
      if (key == classes.size()) classes.push_back(Class{r, gathers, device});
      const int code = gathers ? r->tensor_dtype : r->wire_dtype;
      if (code < 0 || code > 9) {
        PyErr_Format(PyExc_ValueError, "unknown dtype %d", code);
        return nullptr;
      }
      PyObject* entries = r->objects[Request::entries];
      for (Py_ssize_t k = 0; k < PyList_GET_SIZE(entries); ++k) {
        PyObject* e = PyList_GET_ITEM(entries, k);
        int64_t n = as_entry(e)->count;
        if (gathers) {
          PyObject* output = as_entry(e)->objects[Entry::output];
          if (const at::Tensor* t = plain(output)) {
            n = t->numel();
          } else {
            Ref numel(PyObject_CallMethod(output, "numel", nullptr));
            if (!numel) return nullptr;
            n = PyLong_AsLongLong(numel.get());
            if (n == -1 && PyErr_Occurred()) return nullptr;
          }
        }
        int64_t bytes = n * kSizes[code];
        if (padded && !gathers) bytes = (bytes + 15) / 16 * 16;  // no padding on the allgather path
        flat.emplace_back(o, e);
        sizes.push_back(bytes);
        keys.push_back((int)key);
      }
    }
    std::vector<int> group_of(flat.size());
    const int groups = reinterpret_cast<Fuse>((uintptr_t)fuse)(sizes.data(), keys.data(), (int)flat.size(), threshold, 0,
                                                               group_of.data());
    Ref result(PyList_New(groups));
    if (!result) return nullptr;
    for (int g = 0; g < groups; ++g) {
      PyObject* list = PyList_New(0);
      if (!list) return nullptr;
      PyList_SET_ITEM(result.get(), g, list);
    }
    for (size_t i = 0; i < flat.size(); ++i) {
      Ref pair(PyTuple_Pack(2, flat[i].first, flat[i].second));
      if (!pair || PyList_Append(PyList_GET_ITEM(result.get(), group_of[i]), pair.get())) return nullptr;
    }
    return result.release();
  });
}

PyObject* g_array;  // array.array

// An array.array of 64-bit values.
PyObject* array_of(const char* type, const void* data, size_t n) {
  Ref bytes(PyBytes_FromStringAndSize(static_cast<const char*>(data), (Py_ssize_t)(8 * n)));
  if (!bytes) return nullptr;
  return PyObject_CallFunction(g_array, "sO", type, bytes.get());
}

bool is_group(PyObject* group) {
  if (!PyList_CheckExact(group) || PyList_GET_SIZE(group) == 0) return false;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(group); ++i) {
    PyObject* p = PyList_GET_ITEM(group, i);
    if (!PyTuple_CheckExact(p) || PyTuple_GET_SIZE(p) != 2 || Py_TYPE(PyTuple_GET_ITEM(p, 0)) != &request_type ||
        Py_TYPE(PyTuple_GET_ITEM(p, 1)) != &entry_type)
      return false;
  }
  return true;
}
Entry* entry_at(PyObject* group, Py_ssize_t i) { return as_entry(PyTuple_GET_ITEM(PyList_GET_ITEM(group, i), 1)); }

// addresses(group, size, source, odd): (inputs rank by rank, outputs, counts, the peers' tensors).  source(rank, name,
// tensor) gives what another rank passes; None stands for rank 0's own.  odd(tensor, entry) gives the address of a peer
// that is not the plain case, or raises.
PyObject* addresses(PyObject*, PyObject* args) {
  PyObject *group, *source, *odd;
  long size;
  if (!PyArg_ParseTuple(args, "OlOO", &group, &size, &source, &odd)) return nullptr;
  if (!is_group(group)) {
    PyErr_SetString(PyExc_TypeError, "a group is a list of (request, entry)");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    const Py_ssize_t n = PyList_GET_SIZE(group);
    std::vector<uint64_t> inputs((size_t)n), outputs((size_t)n);
    std::vector<int64_t> counts((size_t)n);
    const at::Tensor* first = plain(entry_at(group, 0)->objects[Entry::tensor]);
    for (Py_ssize_t i = 0; i < n; ++i) {
      Entry* e = entry_at(group, i);
      if (!address_of(e->objects[Entry::tensor], &inputs[(size_t)i])) return nullptr;
      if (!address_of(e->objects[Entry::output], &outputs[(size_t)i])) return nullptr;
      counts[(size_t)i] = e->count;
    }
    Ref peers(PyList_New(0));
    if (!peers) return nullptr;
    inputs.reserve((size_t)(n * size));
    for (long rank = 1; rank < size; ++rank) {
      if (source == Py_None) {
        for (Py_ssize_t i = 0; i < n; ++i) inputs.push_back(inputs[(size_t)i]);
        continue;
      }
      Ref r(PyLong_FromLong(rank));
      if (!r) return nullptr;
      for (Py_ssize_t i = 0; i < n; ++i) {
        Ref entry(borrowed(reinterpret_cast<PyObject*>(entry_at(group, i))));
        Entry* e = as_entry(entry.get());
        PyObject* call[] = {nullptr, r.get(), e->objects[Entry::name], e->objects[Entry::tensor]};
        Ref t(PyObject_Vectorcall(source, call + 1, 3 | PY_VECTORCALL_ARGUMENTS_OFFSET, nullptr));
        if (!t) return nullptr;
        const at::Tensor* peer = first ? plain(t.get()) : nullptr;
        uint64_t at;
        if (peer && peer->is_cuda() && peer->scalar_type() == first->scalar_type() && peer->numel() == e->count &&
            peer->is_contiguous()) {
          at = address(*peer);
        } else {
          Ref v(PyObject_CallFunctionObjArgs(odd, t.get(), entry.get(), nullptr));
          if (!v) return nullptr;
          at = PyLong_AsUnsignedLongLong(v.get());
          if (PyErr_Occurred()) return nullptr;
        }
        if (PyList_Append(peers.get(), t.get())) return nullptr;
        inputs.push_back(at);
      }
    }
    Ref in(array_of("Q", inputs.data(), inputs.size())), out(array_of("Q", outputs.data(), outputs.size()));
    Ref sizes(array_of("q", counts.data(), counts.size()));
    if (!in || !out || !sizes) return nullptr;
    return PyTuple_Pack(4, in.get(), out.get(), sizes.get(), peers.get());
  });
}

// requests(group): (its requests, each once and in order; the streams that they were enqueued on, each once).
PyObject* requests(PyObject*, PyObject* group) {
  if (!is_group(group)) {
    PyErr_SetString(PyExc_TypeError, "a group is a list of (request, entry)");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    Ref list(PyList_New(0)), producers(PyList_New(0));
    if (!list || !producers) return nullptr;
    std::unordered_set<PyObject*> seen;
    PyObject* last = nullptr;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(group); ++i) {
      PyObject* r = PyTuple_GET_ITEM(PyList_GET_ITEM(group, i), 0);
      if (!seen.insert(r).second) continue;
      if (PyList_Append(list.get(), r)) return nullptr;
      PyObject* p = as_request(r)->objects[Request::producer];
      if (!p || p == last) continue;
      last = p;
      const int there = PySequence_Contains(producers.get(), p);
      if (there < 0 || (!there && PyList_Append(producers.get(), p))) return nullptr;
    }
    return PyTuple_Pack(2, list.get(), producers.get());
  });
}

// executed(group): the response has been queued, or has failed; a request is submitted with the last of its responses.
PyObject* executed(PyObject*, PyObject* group) {
  if (!is_group(group)) {
    PyErr_SetString(PyExc_TypeError, "a group is a list of (request, entry)");
    return nullptr;
  }
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(group); ++i) {
    Request* r = as_request(PyTuple_GET_ITEM(PyList_GET_ITEM(group, i), 0));
    if (--r->left == 0) r->submitted = 1;
  }
  Py_RETURN_NONE;
}

// attach(requests, marker): the marker of the response that carries an entry of each.
PyObject* attach(PyObject*, PyObject* args) {
  PyObject *list, *marker;
  if (!PyArg_ParseTuple(args, "O!O!", &PyList_Type, &list, &marker_type, &marker)) return nullptr;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(list); ++i) {
    PyObject* r = PyList_GET_ITEM(list, i);
    if (Py_TYPE(r) != &request_type || PyList_Append(as_request(r)->objects[Request::markers], marker)) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "attach takes requests");
      return nullptr;
    }
  }
  Py_RETURN_NONE;
}

// ---- allgather -----------------------------------------------------------------------------------

// parts(entry, size, source, odd): (every rank's tensor, rows in all), or None where one differs from rank 0's in more than
// its first dimension.  odd(tensor, entry) says whether one that is not the plain case fits.
PyObject* parts(PyObject*, PyObject* args) {
  PyObject *entry, *source, *odd;
  long size;
  if (!PyArg_ParseTuple(args, "O!lOO", &entry_type, &entry, &size, &source, &odd)) return nullptr;
  return guarded([&]() -> PyObject* {
    Entry* e = as_entry(entry);
    PyObject* own = e->objects[Entry::tensor];
    const at::Tensor* mine = plain(own);
    Ref list(PyList_New(0));
    if (!list) return nullptr;
    int64_t rows = 0;
    for (long rank = 0; rank < size; ++rank) {
      Ref r(PyLong_FromLong(rank));
      if (!r) return nullptr;
      PyObject* call[] = {nullptr, r.get(), e->objects[Entry::name], own};
      Ref t(rank == 0 || source == Py_None
                ? borrowed(own)
                : PyObject_Vectorcall(source, call + 1, 3 | PY_VECTORCALL_ARGUMENTS_OFFSET, nullptr));
      if (!t) return nullptr;
      const at::Tensor* part = mine ? plain(t.get()) : nullptr;
      if (part && part->is_cuda() && part->scalar_type() == mine->scalar_type() && part->dim() == mine->dim() &&
          part->dim() > 0 && part->sizes().slice(1) == mine->sizes().slice(1) && part->is_contiguous()) {
        rows += part->size(0);
      } else {
        if (rank > 0) {
          Ref v(PyObject_CallFunctionObjArgs(odd, t.get(), entry, nullptr));
          if (!v) return nullptr;
          const int fits = PyObject_IsTrue(v.get());
          if (fits < 0) return nullptr;
          if (!fits) Py_RETURN_NONE;
        }
        Ref shape(PyObject_GetAttrString(t.get(), "shape"));
        Ref first(shape ? PySequence_GetItem(shape.get(), 0) : nullptr);
        if (!first) return nullptr;
        rows += PyLong_AsLongLong(first.get());
        if (PyErr_Occurred()) return nullptr;
      }
      if (PyList_Append(list.get(), t.get())) return nullptr;
    }
    return Py_BuildValue("(OL)", list.get(), (long long)rows);
  });
}

// places(group, element size): (where every rank's rows go, where they come from, their elements), one after the other for
// each entry's output; parts without elements are left out.
PyObject* places(PyObject*, PyObject* args) {
  PyObject* group;
  long long es;
  if (!PyArg_ParseTuple(args, "OL", &group, &es)) return nullptr;
  if (!is_group(group)) {
    PyErr_SetString(PyExc_TypeError, "a group is a list of (request, entry)");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    std::vector<uint64_t> to, from;
    std::vector<int64_t> counts;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(group); ++i) {
      Entry* e = entry_at(group, i);
      uint64_t at;
      if (!address_of(e->objects[Entry::output], &at)) return nullptr;
      PyObject* list = e->objects[Entry::parts];
      if (!list || !PyList_CheckExact(list)) {
        PyErr_SetString(PyExc_TypeError, "an allgather's entry has a list of parts");
        return nullptr;
      }
      for (Py_ssize_t k = 0; k < PyList_GET_SIZE(list); ++k) {
        PyObject* part = PyList_GET_ITEM(list, k);
        int64_t n;
        uint64_t source;
        if (const at::Tensor* t = plain(part)) {
          n = t->numel();
        } else {
          Ref numel(PyObject_CallMethod(part, "numel", nullptr));
          if (!numel) return nullptr;
          n = PyLong_AsLongLong(numel.get());
          if (n == -1 && PyErr_Occurred()) return nullptr;
        }
        if (n == 0) continue;
        if (!address_of(part, &source)) return nullptr;
        to.push_back(at);
        from.push_back(source);
        counts.push_back(n);
        at += (uint64_t)(n * es);
      }
    }
    Ref a(array_of("Q", to.data(), to.size())), b(array_of("Q", from.data(), from.size()));
    Ref c(array_of("q", counts.data(), counts.size()));
    if (!a || !b || !c) return nullptr;
    return PyTuple_Pack(3, a.get(), b.get(), c.get());
  });
}

PyMethodDef methods[] = {{"take", take, METH_O, nullptr},
                         {"plan", plan, METH_VARARGS, nullptr},
                         {"addresses", addresses, METH_VARARGS, nullptr},
                         {"requests", requests, METH_O, nullptr},
                         {"executed", executed, METH_O, nullptr},
                         {"attach", attach, METH_VARARGS, nullptr},
                         {"parts", parts, METH_VARARGS, nullptr},
                         {"places", places, METH_VARARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_front", "The per-tensor part of horovod_amd.torch.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__front(void) {
  state_type.tp_methods = state_methods;
  Ref m(PyModule_Create(&module));
  if (!m) return nullptr;
  const struct {
    const char* name;
    PyTypeObject* type;
  } types[] = {{"Entry", &entry_type}, {"Request", &request_type}, {"Marker", &marker_type}, {"State", &state_type}};
  for (const auto& t : types) {
    if (PyType_Ready(t.type)) return nullptr;
    Py_INCREF(t.type);
    if (PyModule_AddObject(m.get(), t.name, reinterpret_cast<PyObject*>(t.type))) return nullptr;
  }
  g_allreduce = PyUnicode_InternFromString("allreduce");
  g_allgather = PyUnicode_InternFromString("allgather");
  g_pending = PyObject_CallObject(reinterpret_cast<PyObject*>(&PyBaseObject_Type), nullptr);
  Ref arrays(PyImport_ImportModule("array"));
  g_array = arrays ? PyObject_GetAttrString(arrays.get(), "array") : nullptr;
  if (!g_allreduce || !g_allgather || !g_pending || !g_array) return nullptr;
  Py_INCREF(g_pending);
  if (PyModule_AddObject(m.get(), "PENDING", g_pending)) return nullptr;
  return m.release();
}

// Host side of the one-call forward for Python callers: a CPython extension (kernel_amd._host).
//
// A call of the smallest tables takes the GPU four microseconds, and a launch costs the host two and a
// half; checking the tensors, allocating the result and filling in the argument block from Python took
// seven more (9.5 us per call of custom_kernel at 7 tokens).  Here the same steps read the tensors'
// own C++ records.
//
//   Ring   the two alternating buffer sets of one token count: which set is next, when they were used last and,
//          from a set's first forward on (`bind`), its argument block and the tensors a call hands out.
//   Rings  those of one host object.  `forward` takes the caller's tensors, or returns None without side
//          effects when no ring is of their shape, its next set is not bound yet, or anything about them is not
//          as the argument block was built for (the caller then goes the long way, which raises the right
//          error or binds the set).
//          Calls whose token counts change from one to the next find their ring here too.
//   Memo   the configurations of recent custom_kernel calls and the host objects they belong to (one process
//          may run every rank of a world in turn).
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>

#include "moe_a2a.h"

namespace {

// interned attribute names
PyObject *s_stub_kind, *s_combine_mode, *s_fuse_route, *s_fuse_stub, *s_last, *s_rings, *s_num_experts,
    *s_experts_per_token, *s_hidden_dim, *s_max_num_tokens, *s_in_dtype, *s_out_dtype, *s_x, *s_indices, *s_weights,
    *s_num_tokens, *s_always;

struct Ref {  // owned reference
  PyObject* p;
  explicit Ref(PyObject* p_ = nullptr) : p(p_) {}
  ~Ref() { Py_XDECREF(p); }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
  explicit operator bool() const { return p != nullptr; }
};

enum Outcome { kDone, kNotThisWay, kError };

// After a failed lookup or conversion: an attribute that is not there, or of another kind than expected, is for the long
// way to judge (its error is cleared); whatever else was raised, an interrupt or no memory among them, is the caller's.
Outcome failed() {
  if (!PyErr_ExceptionMatches(PyExc_AttributeError) && !PyErr_ExceptionMatches(PyExc_TypeError) &&
      !PyErr_ExceptionMatches(PyExc_OverflowError))
    return kError;
  PyErr_Clear();
  return kNotThisWay;
}
Outcome get_attr(PyObject* o, PyObject* name, Ref& v) {
  v.p = PyObject_GetAttr(o, name);
  return v ? kDone : failed();
}
Outcome int_attr(PyObject* o, PyObject* name, long& v) {
  Ref a;
  if (const Outcome got = get_attr(o, name, a)) return got;
  v = PyLong_AsLong(a.p);
  return v == -1 && PyErr_Occurred() ? failed() : kDone;
}
// what a Python caller gets for it: None, or the exception
PyObject* outcome(Outcome o) {
  if (o == kError) return nullptr;
  Py_RETURN_NONE;
}

struct Ring {
  PyObject_HEAD
  long T, K, H, W;
  long long used;  // the clock of its Rings at the last use: the one with the lowest goes first
  int device, cur;
  int bound;  // bit i: set i
  at::ScalarType in_type, out_type;
  moe_a2a_forward_args args[2];
  PyObject* outs[2];
  PyObject* records[2];
  PyObject* keep[2];  // what the argument blocks point into
};

PyObject* ring_new(PyTypeObject* type, PyObject* args, PyObject*) {
  long T, K, H, W;
  int device;
  PyObject *in_type, *out_type;
  if (!PyArg_ParseTuple(args, "lllliO!O!", &T, &K, &H, &W, &device, &THPDtypeType, &in_type, &THPDtypeType, &out_type))
    return nullptr;
  Ring* r = (Ring*)type->tp_alloc(type, 0);  // zeroed
  if (!r) return nullptr;
  r->T = T, r->K = K, r->H = H, r->W = W, r->device = device;
  r->in_type = ((THPDtype*)in_type)->scalar_type;
  r->out_type = ((THPDtype*)out_type)->scalar_type;
  return (PyObject*)r;
}

// bind(set, block, out, record, an object that keeps what the block points into)
PyObject* ring_bind(Ring* r, PyObject* args) {
  int set;
  PyObject *out, *record, *keep;
  const char* block;
  Py_ssize_t len;
  if (!PyArg_ParseTuple(args, "iy#OOO", &set, &block, &len, &out, &record, &keep)) return nullptr;
  if (set != 0 && set != 1) {
    PyErr_SetString(PyExc_ValueError, "the sets are 0 and 1");
    return nullptr;
  }
  if (len != (Py_ssize_t)sizeof(moe_a2a_forward_args)) {
    PyErr_SetString(PyExc_ValueError, "the argument block is not a moe_a2a_forward_args");
    return nullptr;
  }
  if (r->bound >> set & 1) Py_RETURN_NONE;  // by another thread, since the caller looked
  std::memcpy(&r->args[set], block, sizeof(moe_a2a_forward_args));
  Py_INCREF(out);
  Py_INCREF(record);
  Py_INCREF(keep);
  r->outs[set] = out;
  r->records[set] = record;
  r->keep[set] = keep;
  r->bound |= 1 << set;
  Py_RETURN_NONE;
}

int ring_clear(Ring* r) {
  r->bound = 0;
  for (int i = 0; i < 2; ++i) {
    Py_CLEAR(r->outs[i]);
    Py_CLEAR(r->records[i]);
    Py_CLEAR(r->keep[i]);
  }
  return 0;
}
int ring_traverse(Ring* r, visitproc visit, void* arg) {
  for (int i = 0; i < 2; ++i) {
    Py_VISIT(r->outs[i]);
    Py_VISIT(r->records[i]);
    Py_VISIT(r->keep[i]);
  }
  return 0;
}
void ring_dealloc(Ring* r) {
  PyObject_GC_UnTrack(r);
  ring_clear(r);
  Py_TYPE(r)->tp_free((PyObject*)r);
}

bool plain_matrix(const at::Tensor& t, at::ScalarType type, long rows, long cols, int device) {
  return t.dim() == 2 && t.size(0) == rows && t.size(1) == cols && t.scalar_type() == type && t.is_contiguous() &&
         t.is_cuda() && t.get_device() == device;
}

// One call on the next set; out: where the result goes (already checked).  Sets a Python error on kError.
Outcome ring_forward(Ring* r, PyObject* owner, const at::Tensor& x, const at::Tensor& indices,
                     const at::Tensor& weights, const at::Tensor* rank_start, void* out, int& set) {
  if (!plain_matrix(x, r->in_type, r->T, r->H, r->device) ||
      !plain_matrix(indices, at::kInt, r->T, r->K, r->device) ||
      !plain_matrix(weights, at::kFloat, r->T, r->K, r->device))
    return kNotThisWay;
  if (rank_start && !(rank_start->scalar_type() == at::kInt && rank_start->numel() == r->W + 1 &&
                      rank_start->is_contiguous() && rank_start->is_cuda() && rank_start->get_device() == r->device))
    return kNotThisWay;
  if (c10::hip::current_device() != r->device) return kNotThisWay;
  // switches of the host object that may change between two calls
  long stub_kind, combine_mode, fuse_route = 2;
  Ref route, stub;
  Outcome got;
  if ((got = int_attr(owner, s_stub_kind, stub_kind)) || (got = int_attr(owner, s_combine_mode, combine_mode)) ||
      (got = get_attr(owner, s_fuse_route, route)) || (got = get_attr(owner, s_fuse_stub, stub)))
    return got;
  if (PyLong_Check(route.p))  // (a truth value is one)
    fuse_route = PyObject_IsTrue(route.p);
  else if (!PyUnicode_Check(route.p) || PyUnicode_Compare(route.p, s_always) != 0)
    return kNotThisWay;
  if (!PyLong_Check(stub.p)) return kNotThisWay;
  if (!(r->bound >> (r->cur ^ 1) & 1)) return kNotThisWay;  // (the lookups above may have run Python code)
  set = r->cur ^= 1;
  moe_a2a_forward_args a = r->args[set];  // a copy: the launch runs without the interpreter's lock
  a.x = x.const_data_ptr();
  a.indices = (const int32_t*)indices.const_data_ptr();
  a.weights = (const float*)weights.const_data_ptr();
  a.rank_start = rank_start ? (const int32_t*)rank_start->const_data_ptr() : nullptr;
  if (out) a.out = out;
  a.stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)r->device).stream();
  a.stub_kind = (int)stub_kind;
  a.combine_mode = (int)combine_mode;
  a.fuse_route = (int)fuse_route;
  a.fuse_stub = PyObject_IsTrue(stub.p);
  PyObject* record = r->records[set];
  Py_INCREF(record);
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = moe_a2a_forward_packed(&a);
  Py_END_ALLOW_THREADS;
  if (rc != 0) {
    Py_DECREF(record);
    Ref lib(PyImport_ImportModule("kernel_amd._lib"));  // raises MoeA2AError
    Ref raised(lib ? PyObject_CallMethod(lib.p, "check", "is", rc, "moe_a2a_forward") : nullptr);
    return kError;
  }
  const int bad = PyObject_SetAttr(owner, s_last, record);
  Py_DECREF(record);
  return bad ? kError : kDone;
}

PyMethodDef ring_methods[] = {{"bind", (PyCFunction)ring_bind, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyMemberDef ring_members[] = {{"cur", T_INT, offsetof(Ring, cur), 0, nullptr},
                              {"used", T_LONGLONG, offsetof(Ring, used), READONLY, nullptr},
                              {"bound", T_INT, offsetof(Ring, bound), READONLY, nullptr},
                              {nullptr, 0, 0, 0, nullptr}};
PyTypeObject RingType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---------------------------------------------------------------------------------------
struct Rings {
  PyObject_HEAD
  long long clock;
  PyObject* all;  // list of Ring
};

// the ring of these rows, if its next set is bound (a new reference, marked as used), or null
Ring* rings_find(Rings* rs, const at::Tensor& x) {
  if (x.dim() != 2 || !x.is_cuda()) return nullptr;
  const long T = (long)x.size(0);
  const int device = x.get_device();
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(rs->all); ++i) {
    Ring* r = (Ring*)PyList_GET_ITEM(rs->all, i);
    if (r->T == T && r->device == device && (r->bound >> (r->cur ^ 1) & 1)) {
      r->used = ++rs->clock;
      Py_INCREF(r);
      return r;
    }
  }
  return nullptr;
}

// forward(owner, x, indices, weights, rank_start or None, out or None) -> y, or None: not this way
PyObject* rings_forward(Rings* rs, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6) {
    PyErr_SetString(PyExc_TypeError, "forward takes owner, x, indices, weights, rank_start, out");
    return nullptr;
  }
  for (int i = 1; i < 6; ++i)
    if (!THPVariable_Check(args[i]) && !(i >= 4 && args[i] == Py_None)) Py_RETURN_NONE;
  const at::Tensor& x = THPVariable_Unpack(args[1]);
  Ref ring((PyObject*)rings_find(rs, x));
  if (!ring) Py_RETURN_NONE;
  Ring* r = (Ring*)ring.p;
  const at::Tensor* rank_start = args[4] == Py_None ? nullptr : &THPVariable_Unpack(args[4]);
  void* out = nullptr;
  if (args[5] != Py_None) {
    const at::Tensor& o = THPVariable_Unpack(args[5]);
    if (o.dim() != 2 || o.size(0) < r->T || !plain_matrix(o, r->out_type, o.size(0), r->H, r->device)) Py_RETURN_NONE;
    out = o.data_ptr();
  }
  int set = 0;
  if (const Outcome got = ring_forward(r, args[0], x, THPVariable_Unpack(args[2]), THPVariable_Unpack(args[3]), rank_start,
                                       out, set))
    return outcome(got);
  PyObject* y = out ? args[5] : r->outs[set];
  Py_INCREF(y);
  return y;
  END_HANDLE_TH_ERRORS
}

PyObject* rings_new(PyTypeObject* type, PyObject*, PyObject*) {
  Rings* rs = (Rings*)type->tp_alloc(type, 0);
  if (rs && !(rs->all = PyList_New(0))) Py_CLEAR(rs);
  return (PyObject*)rs;
}
// add(ring)
PyObject* rings_add(Rings* rs, PyObject* ring) {
  if (Py_TYPE(ring) != &RingType) {
    PyErr_SetString(PyExc_TypeError, "add takes a Ring");
    return nullptr;
  }
  if (PyList_Append(rs->all, ring) < 0) return nullptr;
  Py_RETURN_NONE;
}
// touch(ring): used now
PyObject* rings_touch(Rings* rs, PyObject* ring) {
  if (Py_TYPE(ring) != &RingType) {
    PyErr_SetString(PyExc_TypeError, "touch takes a Ring");
    return nullptr;
  }
  ((Ring*)ring)->used = ++rs->clock;
  Py_RETURN_NONE;
}
PyObject* rings_drop(Rings* rs, PyObject* ring) {
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(rs->all); ++i)
    if (PyList_GET_ITEM(rs->all, i) == ring) {
      if (PyList_SetSlice(rs->all, i, i + 1, nullptr) < 0) return nullptr;
      break;
    }
  Py_RETURN_NONE;
}
PyObject* rings_clear_py(Rings* rs, PyObject*) {
  if (PyList_SetSlice(rs->all, 0, PyList_GET_SIZE(rs->all), nullptr) < 0) return nullptr;
  Py_RETURN_NONE;
}
int rings_traverse(Rings* rs, visitproc visit, void* arg) {
  Py_VISIT(rs->all);
  return 0;
}
// (an object in a cycle that is being taken apart may still be asked for: an empty list serves)
int rings_clear(Rings* rs) {
  return rs->all ? PyList_SetSlice(rs->all, 0, PyList_GET_SIZE(rs->all), nullptr) : 0;
}
void rings_dealloc(Rings* rs) {
  PyObject_GC_UnTrack(rs);
  Py_CLEAR(rs->all);
  Py_TYPE(rs)->tp_free((PyObject*)rs);
}
PyMethodDef rings_methods[] = {{"forward", (PyCFunction)(void (*)(void))rings_forward, METH_FASTCALL, nullptr},
                               {"add", (PyCFunction)rings_add, METH_O, nullptr},
                               {"touch", (PyCFunction)rings_touch, METH_O, nullptr},
                               {"drop", (PyCFunction)rings_drop, METH_O, nullptr},
                               {"clear", (PyCFunction)rings_clear_py, METH_NOARGS, nullptr},
                               {nullptr, nullptr, 0, nullptr}};
PyTypeObject RingsType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---------------------------------------------------------------------------------------
constexpr int kMemoEntries = 16;
struct MemoEntry {
  long config[4], call[5];  // call: rank, world_size, stub_kind, combine_mode, device of the inputs
  PyObject *in_dtype, *out_dtype, *owner;
};
struct Memo {
  PyObject_HEAD
  int used;
  MemoEntry entry[kMemoEntries];  // most recently used first
};
void entry_drop(MemoEntry& e) {
  Py_CLEAR(e.in_dtype);
  Py_CLEAR(e.out_dtype);
  Py_CLEAR(e.owner);
}
// entry i becomes the first
void entry_front(Memo* m, int i) {
  if (i == 0) return;
  const MemoEntry e = m->entry[i];
  std::memmove(&m->entry[1], &m->entry[0], i * sizeof(MemoEntry));
  m->entry[0] = e;
}

// what custom_kernel's instance depends on, read from the config record at every call
Outcome memo_read(PyObject* cfg, long (&v)[4], Ref& in_dtype, Ref& out_dtype) {
  Outcome got;
  if ((got = int_attr(cfg, s_num_experts, v[0])) || (got = int_attr(cfg, s_experts_per_token, v[1])) ||
      (got = int_attr(cfg, s_hidden_dim, v[2])) || (got = int_attr(cfg, s_max_num_tokens, v[3])) ||
      (got = get_attr(cfg, s_in_dtype, in_dtype)) || (got = get_attr(cfg, s_out_dtype, out_dtype)))
    return got;
  return kDone;
}

// the entry of these values, or -1
int memo_find(const Memo* m, const long (&config)[4], const long (&call)[5], const PyObject* in_dtype,
              const PyObject* out_dtype) {
  for (int i = 0; i < m->used; ++i) {
    const MemoEntry& e = m->entry[i];
    if (std::memcmp(e.call, call, sizeof(call)) == 0 && std::memcmp(e.config, config, sizeof(config)) == 0 &&
        e.in_dtype == in_dtype && e.out_dtype == out_dtype)
      return i;
  }
  return -1;
}

// remember(cfg, rank, world_size, stub_kind, combine_mode, device index, owner)
PyObject* memo_remember(Memo* m, PyObject* const* args, Py_ssize_t n) {
  if (n != 7) {
    PyErr_SetString(PyExc_TypeError, "remember takes cfg, rank, world_size, stub_kind, combine_mode, device, owner");
    return nullptr;
  }
  MemoEntry fresh;
  for (int i = 0; i < 5; ++i) {
    fresh.call[i] = PyLong_AsLong(args[1 + i]);
    if (fresh.call[i] == -1 && PyErr_Occurred()) return outcome(failed());
  }
  Ref in_dtype, out_dtype;
  if (const Outcome got = memo_read(args[0], fresh.config, in_dtype, out_dtype)) return outcome(got);
  const int at = memo_find(m, fresh.config, fresh.call, in_dtype.p, out_dtype.p);
  Py_INCREF(args[6]);
  if (at >= 0) {
    PyObject* before = m->entry[at].owner;
    m->entry[at].owner = args[6];
    entry_front(m, at);
    Py_DECREF(before);
    Py_RETURN_NONE;
  }
  fresh.in_dtype = in_dtype.p;
  fresh.out_dtype = out_dtype.p;
  fresh.owner = args[6];
  in_dtype.p = out_dtype.p = nullptr;
  const bool full = m->used == kMemoEntries;
  MemoEntry longest_unused = m->entry[kMemoEntries - 1];
  if (!full) ++m->used;
  m->entry[m->used - 1] = fresh;
  entry_front(m, m->used - 1);
  if (full) entry_drop(longest_unused);  // last: this may run Python code, which finds a whole table
  Py_RETURN_NONE;
}

// run(data, stub_kind, combine_mode) -> y, or None: not this way
PyObject* memo_run(Memo* m, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3) {
    PyErr_SetString(PyExc_TypeError, "run takes data, stub_kind, combine_mode");
    return nullptr;
  }
  if (!PyTuple_CheckExact(args[0]) || PyTuple_GET_SIZE(args[0]) != 4) Py_RETURN_NONE;
  long call[5];
  PyObject* given[4] = {PyTuple_GET_ITEM(args[0], 2), PyTuple_GET_ITEM(args[0], 3), args[1], args[2]};
  for (int i = 0; i < 4; ++i) {
    call[i] = PyLong_CheckExact(given[i]) ? PyLong_AsLong(given[i]) : -1;
    if (call[i] == -1 && PyErr_Occurred()) return outcome(failed());
    if (call[i] < 0) Py_RETURN_NONE;
  }
  PyObject* rank_data = PyTuple_GET_ITEM(args[0], 1);
  long num_tokens;
  Ref x, indices, weights;
  Outcome got;
  if ((got = get_attr(rank_data, s_x, x)) || (got = get_attr(rank_data, s_indices, indices)) ||
      (got = get_attr(rank_data, s_weights, weights)) || (got = int_attr(rank_data, s_num_tokens, num_tokens)))
    return outcome(got);
  if (!THPVariable_Check(x.p) || !THPVariable_Check(indices.p) || !THPVariable_Check(weights.p)) Py_RETURN_NONE;
  const at::Tensor& xt = THPVariable_Unpack(x.p);
  call[4] = xt.get_device();
  long config[4];
  Ref in_dtype, out_dtype;
  if ((got = memo_read(PyTuple_GET_ITEM(args[0], 0), config, in_dtype, out_dtype))) return outcome(got);
  const int at = memo_find(m, config, call, in_dtype.p, out_dtype.p);
  if (at < 0) Py_RETURN_NONE;
  entry_front(m, at);
  Ref owner(m->entry[0].owner), rings, ring;  // taken here: the lookups below may run Python code, and other threads
  Py_INCREF(owner.p);
  if ((got = get_attr(owner.p, s_rings, rings))) return outcome(got);
  if (Py_TYPE(rings.p) != &RingsType) Py_RETURN_NONE;
  ring.p = (PyObject*)rings_find((Rings*)rings.p, xt);
  if (!ring) Py_RETURN_NONE;
  Ring* r = (Ring*)ring.p;
  if (num_tokens < 0 || num_tokens > r->T || !plain_matrix(xt, r->in_type, r->T, r->H, r->device)) Py_RETURN_NONE;
  // the caller owns its result: the combine writes straight into a fresh tensor
  at::Tensor y = at::empty({r->T, r->H}, xt.options().dtype(r->out_type));
  int set = 0;
  if ((got = ring_forward(r, owner.p, xt, THPVariable_Unpack(indices.p), THPVariable_Unpack(weights.p), nullptr, y.data_ptr(),
                          set)))
    return outcome(got);
  return THPVariable_Wrap(num_tokens == r->T ? y : y.narrow(0, 0, num_tokens));
  END_HANDLE_TH_ERRORS
}

PyObject* memo_new(PyTypeObject* type, PyObject*, PyObject*) { return type->tp_alloc(type, 0); }
int memo_clear(Memo* m) {
  while (m->used > 0) {  // an entry is off the table before what it held goes, which may run Python code
    MemoEntry e = m->entry[--m->used];
    entry_drop(e);
  }
  return 0;
}
int memo_traverse(Memo* m, visitproc visit, void* arg) {
  for (int i = 0; i < m->used; ++i) Py_VISIT(m->entry[i].owner);
  return 0;
}
void memo_dealloc(Memo* m) {
  PyObject_GC_UnTrack(m);
  memo_clear(m);
  Py_TYPE(m)->tp_free((PyObject*)m);
}
PyObject* memo_clear_py(Memo* m, PyObject*) {
  memo_clear(m);
  Py_RETURN_NONE;
}
PyMethodDef memo_methods[] = {{"clear", (PyCFunction)memo_clear_py, METH_NOARGS, nullptr},
                              {"remember", (PyCFunction)(void (*)(void))memo_remember, METH_FASTCALL, nullptr},
                              {"run", (PyCFunction)(void (*)(void))memo_run, METH_FASTCALL, nullptr},
                              {nullptr, nullptr, 0, nullptr}};
PyTypeObject MemoType = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, nullptr, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
  struct {
    PyObject*& var;
    const char* text;
  } names[] = {{s_stub_kind, "stub_kind"},     {s_combine_mode, "combine_mode"},
               {s_fuse_route, "fuse_route"},   {s_fuse_stub, "fuse_stub"},
               {s_last, "last"},               {s_rings, "_rings"},
               {s_num_experts, "num_experts"}, {s_experts_per_token, "experts_per_token"},
               {s_hidden_dim, "hidden_dim"},   {s_max_num_tokens, "max_num_tokens"},
               {s_in_dtype, "in_dtype"},       {s_out_dtype, "out_dtype"},
               {s_x, "x"},                     {s_indices, "indices"},
               {s_weights, "weights"},         {s_num_tokens, "num_tokens"},
               {s_always, "always"}};
  for (auto& name : names)
    if (!(name.var = PyUnicode_InternFromString(name.text))) return nullptr;
  RingType.tp_name = "kernel_amd._host.Ring";
  RingType.tp_basicsize = sizeof(Ring);
  RingType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC;
  RingType.tp_new = ring_new;
  RingType.tp_dealloc = (destructor)ring_dealloc;
  RingType.tp_traverse = (traverseproc)ring_traverse;
  RingType.tp_clear = (inquiry)ring_clear;
  RingType.tp_methods = ring_methods;
  RingType.tp_members = ring_members;
  RingsType.tp_name = "kernel_amd._host.Rings";
  RingsType.tp_basicsize = sizeof(Rings);
  RingsType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC;
  RingsType.tp_new = rings_new;
  RingsType.tp_dealloc = (destructor)rings_dealloc;
  RingsType.tp_traverse = (traverseproc)rings_traverse;
  RingsType.tp_clear = (inquiry)rings_clear;
  RingsType.tp_methods = rings_methods;
  MemoType.tp_name = "kernel_amd._host.Memo";
  MemoType.tp_basicsize = sizeof(Memo);
  MemoType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC;
  MemoType.tp_new = memo_new;
  MemoType.tp_dealloc = (destructor)memo_dealloc;
  MemoType.tp_traverse = (traverseproc)memo_traverse;
  MemoType.tp_clear = (inquiry)memo_clear;
  MemoType.tp_methods = memo_methods;
  if (PyType_Ready(&RingType) < 0 || PyType_Ready(&RingsType) < 0 || PyType_Ready(&MemoType) < 0) return nullptr;
  PyObject* m = PyModule_Create(&module);
  if (!m) return nullptr;
  Py_INCREF(&RingType);
  Py_INCREF(&RingsType);
  Py_INCREF(&MemoType);
  if (PyModule_AddObject(m, "Ring", (PyObject*)&RingType) < 0 ||
      PyModule_AddObject(m, "Rings", (PyObject*)&RingsType) < 0 || PyModule_AddObject(m, "Memo", (PyObject*)&MemoType) < 0)
    return nullptr;
  return m;
}

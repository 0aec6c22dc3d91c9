// sparsetir_amd._host: what a call of a Python operator does between the interpreter and the C ABI.
//
// A small launch runs for a few microseconds; checking its arguments, finding its plan and reading
// the current stream took 10.5 us in Python for five arrays and 16 us for the 32 arrays of a hyb
// operator, so the interpreter and not the GPU set the pace.  A Launcher does the same in native
// code: 3.3 us for the five arrays, 5 us for the 32, the launch itself included.
//
// The Launcher takes a call only when nothing is out of the ordinary: every argument a strided
// tensor of the expected type and length on the current device and, for operators with plans, the
// arrays those of a plan it was told of (same addresses, same torch version counters).  Anything else
// is left to the Python code, which words the errors, makes the plans and keeps them.
//
// column_part_hyb() is the decomposition of one column partition for tensors on the current device: its
// launches, its one wait and the tensors it returns (40 of them with ten buckets and values, 3 us each
// when sliced and reshaped from Python).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <sched.h>

#include <algorithm>
#include <new>
#include <vector>

#include "../../../include/sparsetir_amd.h"
#include "../format_one.h"

namespace {

enum Kind { kCsr, kSddmmPreproc, kSddmm, kSddmmScaled, kBsr, kDbsr, kTc, kRgms, kRgmsF32, kRgmsCsf, kHyb, kKinds };
enum { kKeyAddress = 1, kKeyVersion = 2 };
enum { kLaunched = 0, kFailed = -1, kNotTaken = 1 };

struct Operand {
  c10::ScalarType dtype;
  int64_t length;
  int key;  // which of the tensor's properties a plan depends on
};

// A plan of the operator, the properties of the arrays it was made from, and the operator's name for it
struct Plan {
  void* plan;
  int device;
  std::vector<int64_t> key;
  PyObject* name;
};

// What a call needs of its stream's workspace: counters, which are zero between launches, and the rest.
struct Need {
  size_t counters, rest;
};

// Counters at the front, zeroed once; then left to the calls on one stream, which run one after the other
struct Workspace {
  c10::hip::HIPStream stream;
  Need has;
  at::Tensor memory;
};
constexpr size_t kWorkspaces = 4;  // streams an operator keeps one for

struct Launcher {
  PyObject_HEAD
  Kind kind;
  std::vector<int64_t>* sizes;
  std::vector<Operand>* operands;
  std::vector<Plan>* plans;     // as many as the operator keeps, the one used last in front
  std::vector<int64_t>* key;    // of the call in hand, for as long as it holds the GIL
  std::vector<void*>* in_use;   // a plan per launch that is under way without the GIL
  Need csr;                     // of a CSR product
  std::vector<Workspace>* workspaces;  // one per stream the operator runs on, the one used last in front
};

// The tensor behind `o` when it is what the operand wants, else null.
const at::Tensor* take(PyObject* o, const Operand& want, int device) {
  if (!THPVariable_Check(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.scalar_type() != want.dtype || t.layout() != c10::kStrided || t.dim() != 1 ||
      t.size(0) != want.length || !t.is_contiguous() || t.get_device() != device ||
      ((want.key & kKeyVersion) && t.is_inference()))  // an inference tensor counts no versions
    return nullptr;
  return &t;
}

int64_t version_of(const at::Tensor& t) { return (int64_t)t.unsafeGetTensorImpl()->version_counter().current_version(); }

Need need_of(const Launcher* l, const void* plan) {
  if (l->kind == kCsr) return l->csr;
  if (l->kind != kTc) return {0, 0};
  const stir_tc_plan* q = static_cast<const stir_tc_plan*>(plan);
  const int32_t tile = (int32_t)(*l->sizes)[2], feat = (int32_t)(*l->sizes)[4];
  return {stir_tc_plan_counter_bytes(q, feat), stir_tc_plan_partial_bytes(q, tile, feat)};
}

Workspace new_workspace(const c10::hip::HIPStream& st, const Need& need) {
  const at::TensorOptions on = at::TensorOptions(c10::ScalarType::Byte).device(c10::DeviceType::CUDA, st.device_index());
  Workspace w{st, need, at::empty({(int64_t)(need.counters + need.rest)}, on)};
  w.memory.narrow(0, 0, (int64_t)need.counters).zero_();
  return w;
}

// Where the two parts of a call's workspace are.
struct Scratch {
  char *counters = nullptr, *rest = nullptr;
};
Scratch scratch_of(const Workspace& w) {
  char* p = static_cast<char*>(w.memory.data_ptr());
  return {p, p + w.has.counters};
}

// The workspace of a call on `st`.  A call that is being captured gets one of its own, its counters cleared by
// the graph itself: the graph may be replayed on any stream.  `held` keeps the memory until the call is recorded or
// in its queue: while it has let go of the GIL another thread may take the workspace off the list, and what the
// allocator gave out then would be used before the kernel that is yet to come.
Scratch workspace(Launcher* l, const c10::hip::HIPStream& st, const Need& need, at::Tensor* held) {
  std::vector<Workspace>& all = *l->workspaces;
  if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) {
    const Workspace w = new_workspace(st, need);
    *held = w.memory;
    return scratch_of(w);
  }
  size_t at = 0;
  while (at < all.size() && all[at].stream != st) ++at;
  if (at == all.size()) {
    if (at == kWorkspaces) all.pop_back(), --at;  // back to the allocator of its stream
    all.push_back(new_workspace(st, need));
  } else if (all[at].has.counters < need.counters || all[at].has.rest < need.rest) {  // another plan's call
    all[at] = new_workspace(st, {std::max(all[at].has.counters, need.counters), std::max(all[at].has.rest, need.rest)});
  }
  if (at > 0) std::rotate(all.begin(), all.begin() + at, all.begin() + at + 1);
  *held = all.front().memory;
  return scratch_of(all.front());
}

int call(const Launcher* l, void* const* p, void* plan, const Scratch& ws, void* st) {
  const std::vector<int64_t>& n = *l->sizes;
  auto i = [&](int k) { return (int32_t)n[k]; };
  auto f = [&](int k) { return static_cast<float*>(p[k]); };
  auto x = [&](int k) { return static_cast<int32_t*>(p[k]); };
  switch (l->kind) {
    case kCsr: return stir_csr_spmm_f32_workspace(i(0), i(1), i(2), n[3], f(0), f(1), f(2), x(3), x(4), ws.counters, st);
    case kSddmmPreproc: return stir_sddmm_preproc(i(0), n[3], x(3), x(5), st);
    case kSddmm: return stir_sddmm_f32(i(0), i(1), i(2), n[3], f(0), f(1), f(2), x(3), x(4), x(5), st);
    case kSddmmScaled:
      return stir_sddmm_scaled_f32(i(0), i(1), i(2), n[3], f(0), f(1), f(2), x(3), x(4), x(5), f(6), st);
    case kBsr: return stir_bsr_spmm(i(0), i(1), i(2), i(3), i(4), i(5), n[6], p[0], p[1], p[2], x(3), x(4), st);
    case kDbsr:
      return stir_dbsr_spmm(i(0), i(1), i(2), i(3), i(4), i(5), n[6], p[0], p[1], p[2], x(4), x(5), x(6), st);
    case kTc:
      return stir_tc_spmm_f16_workspace(static_cast<const stir_tc_plan*>(plan), i(0), i(1), i(2), i(3), i(4), n[5], p[0],
                                        p[1], p[2], x(3), x(4), ws.counters, ws.rest, st);
    case kRgms: {
      stir_rgms_plan* q = static_cast<stir_rgms_plan*>(plan);
      if (n[5] == 2) return stir_rgms_bf16(q, i(0), i(1), i(2), i(3), i(4), p[0], p[1], f(2), st);
      if (n[5] == 1) return stir_rgms_f16_out_f16(q, i(0), i(1), i(2), i(3), i(4), p[0], p[1], p[2], st);
      return stir_rgms_f16(q, i(0), i(1), i(2), i(3), i(4), p[0], p[1], f(2), st);
    }
    case kRgmsF32:
      return stir_rgms_f32(static_cast<stir_rgms_f32_plan*>(plan), i(0), i(1), i(2), i(3), i(4), f(0), f(1), f(2), st);
    case kRgmsCsf:
      return stir_rgms_csf_f32_planned(static_cast<stir_rgms_csf_f32_plan*>(plan), i(0), i(1), i(2), i(3), i(4), f(1),
                                       f(2), f(3), st);
    case kHyb: return stir_hyb_spmm_f32(static_cast<const stir_hyb_plan*>(plan), i(0), f(0), f(1), st);
    default: return -1;
  }
}

bool planned(Kind k) { return k >= kTc; }

// call() without the GIL (a launch waits when the queue is full).  Other threads may use the launcher meanwhile, so
// nothing of it is read here but its kind and sizes, and nobody destroys `plan` before the call is done with it.
int call_unlocked(Launcher* l, void* const* p, void* plan, const Scratch& ws, void* st) {
  int rc;
  if (plan) l->in_use->push_back(plan);
  Py_BEGIN_ALLOW_THREADS
  rc = call(l, p, plan, ws, st);
  Py_END_ALLOW_THREADS
  if (plan) l->in_use->erase(std::find(l->in_use->begin(), l->in_use->end(), plan));
  return rc;
}

// Lets go of the GIL until no launch uses `plan`, which is in the launcher's list no more.
void wait_until_unused(Launcher* l, void* plan) {
  while (std::find(l->in_use->begin(), l->in_use->end(), plan) != l->in_use->end()) {
    Py_BEGIN_ALLOW_THREADS
    sched_yield();
    Py_END_ALLOW_THREADS
  }
}

constexpr size_t kPassed = 8;  // a C entry point takes at most this many of the leading arguments

// Looks at the whole argument tuple and fills p with the addresses of the leading arguments.
// visit(property) is called for every property a plan depends on, in order, and ends the walk by
// returning false.
template <class F>
bool walk(const Launcher* l, PyObject* args, int device, void* (&p)[kPassed], F visit) {
  const size_t count = l->operands->size();
  if (!PyTuple_CheckExact(args) || (size_t)PyTuple_GET_SIZE(args) != count || count == 0) return false;
  for (size_t k = 0; k < count; ++k) {
    const Operand& want = (*l->operands)[k];
    const at::Tensor* t = take(PyTuple_GET_ITEM(args, k), want, device);
    if (!t) return false;
    void* address = want.length ? t->data_ptr() : nullptr;
    if (k < kPassed) p[k] = address;
    if ((want.key & kKeyAddress) && !visit(reinterpret_cast<int64_t>(address))) return false;
    if ((want.key & kKeyVersion) && !visit(version_of(*t))) return false;
  }
  return true;
}

// launch(args) -> 0: launched; -1: the C ABI refused (stir_last_error says why); 1: not taken; or the
// name of the plan, launched as well, that was not the one used last
PyObject* launch(PyObject* self, PyObject* args) {
  Launcher* l = reinterpret_cast<Launcher*>(self);
  int rc = kNotTaken;
  PyObject* moved = nullptr;
  try {
    const int device = (int)c10::hip::current_device();
    void* plan = nullptr;
    void* p[kPassed];
    if (planned(l->kind)) {
      std::vector<int64_t>& key = *l->key;
      key.clear();
      if (l->plans->empty() || !walk(l, args, device, p, [&](int64_t v) { return key.push_back(v), true; }))
        return PyLong_FromLong(kNotTaken);
      size_t at = 0;
      while (at < l->plans->size() && ((*l->plans)[at].device != device || (*l->plans)[at].key != key)) ++at;
      if (at == l->plans->size()) return PyLong_FromLong(kNotTaken);
      if (at > 0) {
        std::rotate(l->plans->begin(), l->plans->begin() + at, l->plans->begin() + at + 1);
        moved = l->plans->front().name;
        Py_INCREF(moved);
      }
      plan = l->plans->front().plan;
    } else if (!walk(l, args, device, p, [](int64_t) { return true; })) {
      return PyLong_FromLong(kNotTaken);
    }
    const c10::hip::HIPStream stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)device);
    at::Tensor held;
    const Need need = need_of(l, plan);
    const Scratch ws = need.counters ? workspace(l, stream, need, &held) : Scratch();
    rc = call_unlocked(l, p, plan, ws, stream.stream());
  } catch (...) {  // a tensor without storage: the Python code says what is wrong with it
    rc = kNotTaken;
  }
  if (rc == kLaunched && moved) return moved;
  Py_XDECREF(moved);
  return PyLong_FromLong(rc);
}

// Takes the plan of that name (null: every plan) off the list; the caller may destroy it then.
void drop(Launcher* l, PyObject* name) {
  std::vector<Plan> gone;
  for (size_t k = l->plans->size(); k-- > 0;) {
    const int same = name ? PyObject_RichCompareBool((*l->plans)[k].name, name, Py_EQ) : 1;
    if (same < 0) PyErr_Clear();
    if (same == 0) continue;
    gone.push_back(std::move((*l->plans)[k]));
    l->plans->erase(l->plans->begin() + k);
  }
  for (Plan& g : gone) {
    wait_until_unused(l, g.plan);
    Py_DECREF(g.name);
  }
}

// remember(args, plan, name): `plan` was made from these arguments, checked by the caller, and used last
PyObject* remember(PyObject* self, PyObject* args) {
  Launcher* l = reinterpret_cast<Launcher*>(self);
  PyObject *tensors, *name;
  unsigned long long plan;
  if (!PyArg_ParseTuple(args, "O!KO", &PyTuple_Type, &tensors, &plan, &name)) return nullptr;
  drop(l, name);
  try {
    void* p[kPassed];
    Plan q{reinterpret_cast<void*>(plan), (int)c10::hip::current_device(), {}, name};
    if (walk(l, tensors, q.device, p, [&](int64_t v) { return q.key.push_back(v), true; })) {
      l->plans->insert(l->plans->begin(), std::move(q));
      Py_INCREF(name);
    }
  } catch (...) {  // not taken by launch() either
  }
  Py_RETURN_NONE;
}

// forget(name), forget(None): the plan of that name, or all of them, is no more
PyObject* forget(PyObject* self, PyObject* name) {
  drop(reinterpret_cast<Launcher*>(self), name == Py_None ? nullptr : name);
  Py_RETURN_NONE;
}

// launch_new_hyb(args) -> (name, plan) of a new plan for arguments launch() did not know, remembered and
// launched; 0 when another thread made the plan meanwhile (launched with it); None when they are not the ordinary
// ones, -1 when the C ABI refused.  The name is the properties the plan depends on.  Other threads run while the
// plan is made: everything about this call is its own until the plan is put into the list, whole.
PyObject* launch_new_hyb(PyObject* self, PyObject* args) {
  Launcher* l = reinterpret_cast<Launcher*>(self);
  stir_hyb_plan* plan = nullptr;
  PyObject* out = nullptr;
  Plan made{nullptr, 0, {}, nullptr};
  try {
    if (l->kind != kHyb) Py_RETURN_NONE;
    const int64_t device = c10::hip::current_device();
    void* p[kPassed];
    std::vector<int64_t> key(1, device);
    if (!walk(l, args, (int)device, p, [&](int64_t v) { return key.push_back(v), true; })) Py_RETURN_NONE;
    // key: device, then per bucket the address of A, address and version of rows, of cols
    const size_t nk = (l->operands->size() - 2) / 3;
    const std::vector<int64_t>& n = *l->sizes;  // feat, m, n, parts, widths ...
    const size_t nb = n.size() - 4;
    std::vector<int32_t> widths(n.begin() + 4, n.end());
    std::vector<int64_t> nrows(nk + 1);
    std::vector<const float*> A(nk + 1);
    std::vector<const int32_t*> rows(nk + 1), cols(nk + 1);
    for (size_t k = 0; k < nk; ++k) {
      const int64_t* q = key.data() + 1 + 5 * k;
      A[k] = reinterpret_cast<const float*>(q[0]);
      rows[k] = reinterpret_cast<const int32_t*>(q[1]);
      cols[k] = reinterpret_cast<const int32_t*>(q[3]);
      nrows[k] = (*l->operands)[2 + 3 * k + 1].length;
    }
    if (nb == 0 || nk != nb * (size_t)n[3]) Py_RETURN_NONE;
    void* st = c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream();
    made.device = (int)device;
    made.key.assign(key.begin() + 1, key.end());
    for (const Plan& q : *l->plans)
      if (q.device == made.device && q.key == made.key) return PyLong_FromLong(call_unlocked(l, p, q.plan, Scratch(), st));
    made.name = PyBytes_FromStringAndSize(reinterpret_cast<const char*>(key.data()),
                                          (Py_ssize_t)(key.size() * sizeof(int64_t)));
    if (!made.name) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = stir_hyb_plan_create(&plan, (int32_t)n[1], (int32_t)n[2], (int32_t)n[3], (int32_t)nb, widths.data(),
                              nrows.data(), A.data(), rows.data(), cols.data());
    if (rc == 0) rc = call(l, p, plan, Scratch(), st);
    Py_END_ALLOW_THREADS
    made.plan = plan;
    out = rc == 0 ? Py_BuildValue("(OK)", made.name, reinterpret_cast<unsigned long long>(plan)) : PyLong_FromLong(kFailed);
    if (rc == 0 && out) {
      l->plans->insert(l->plans->begin(), std::move(made));
      return out;
    }
  } catch (...) {  // out of memory: the Python code makes the plan, or says so
    Py_CLEAR(out);
    Py_INCREF(Py_None);
    out = Py_None;
  }
  Py_XDECREF(made.name);  // nobody would own the plan
  if (plan) stir_hyb_plan_destroy(plan);
  return out;
}

bool scalar_type(long code, c10::ScalarType* out) {
  switch (code) {
    case 0: *out = c10::ScalarType::Half; return true;
    case 1: *out = c10::ScalarType::BFloat16; return true;
    case 2: *out = c10::ScalarType::Float; return true;
    case 3: *out = c10::ScalarType::Int; return true;
    case -1: *out = c10::ScalarType::Undefined; return true;  // no tensor's type: nothing is taken
    default: return false;
  }
}

PyTypeObject launcher_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

Launcher* make(Kind kind) {
  Launcher* l = reinterpret_cast<Launcher*>(launcher_type.tp_alloc(&launcher_type, 0));
  if (!l) return nullptr;
  l->kind = kind;
  l->sizes = new (std::nothrow) std::vector<int64_t>();
  l->operands = new (std::nothrow) std::vector<Operand>();
  l->plans = new (std::nothrow) std::vector<Plan>();
  l->key = new (std::nothrow) std::vector<int64_t>();
  l->in_use = new (std::nothrow) std::vector<void*>();
  l->workspaces = new (std::nothrow) std::vector<Workspace>();
  if (l->sizes && l->operands && l->plans && l->key && l->in_use && l->workspaces) return l;
  Py_DECREF(l);
  PyErr_NoMemory();
  return nullptr;
}

// The entries of a sequence of ints; false with an exception set when it is none.
bool ints_of(PyObject* o, std::vector<int64_t>* out) {
  PyObject* fast = PySequence_Fast(o, "a sequence of ints is expected");
  if (!fast) return false;
  for (Py_ssize_t k = 0; k < PySequence_Fast_GET_SIZE(fast) && !PyErr_Occurred(); ++k)
    out->push_back(PyLong_AsLongLong(PySequence_Fast_GET_ITEM(fast, k)));
  Py_DECREF(fast);
  return !PyErr_Occurred();
}

// Launcher.hyb(n, m, feat, parts, buckets, nrows): the operands of the hyb operator, B and C followed by
// (A_k, rows_k, cols_k) of every bucket of every partition
PyObject* launcher_hyb(PyObject*, PyObject* args) {
  long long n, m, feat, parts;
  PyObject *buckets, *nrows;
  if (!PyArg_ParseTuple(args, "LLLLOO", &n, &m, &feat, &parts, &buckets, &nrows)) return nullptr;
  std::vector<int64_t> w, r;
  if (!ints_of(buckets, &w) || !ints_of(nrows, &r)) return nullptr;
  if (w.empty() && !r.empty()) {
    PyErr_SetString(PyExc_ValueError, "rows without buckets");
    return nullptr;
  }
  Launcher* l = make(kHyb);
  if (!l) return nullptr;
  *l->sizes = {feat, m, n, parts};
  l->sizes->insert(l->sizes->end(), w.begin(), w.end());
  l->operands->push_back({c10::ScalarType::Float, n * feat, 0});
  l->operands->push_back({c10::ScalarType::Float, m * feat, 0});
  for (size_t k = 0; k < r.size(); ++k) {
    const int64_t slots = r[k] * w[k % w.size()];
    l->operands->push_back({c10::ScalarType::Float, slots, kKeyAddress});
    l->operands->push_back({c10::ScalarType::Int, r[k], kKeyAddress | kKeyVersion});
    l->operands->push_back({c10::ScalarType::Int, slots, kKeyAddress | kKeyVersion});
  }
  return reinterpret_cast<PyObject*>(l);
}

// Launcher(kind, sizes, operands): sizes a sequence of ints, operands a sequence of
// (type code, length, key bits), type codes STIR_F16, STIR_BF16, STIR_F32 and 3 for int32
PyObject* launcher_new(PyTypeObject*, PyObject* args, PyObject*) {
  int kind;
  PyObject *sizes, *operands;
  if (!PyArg_ParseTuple(args, "iOO", &kind, &sizes, &operands)) return nullptr;
  if (kind < 0 || kind >= kKinds) {
    PyErr_SetString(PyExc_ValueError, "unknown kind of launcher");
    return nullptr;
  }
  Launcher* l = make((Kind)kind);
  if (!l) return nullptr;
  PyObject* fo = PySequence_Fast(operands, "operands must be a sequence");
  bool ok = fo && ints_of(sizes, l->sizes);
  for (Py_ssize_t k = 0; ok && k < PySequence_Fast_GET_SIZE(fo); ++k) {
    int code, key;
    long long length;
    Operand o;
    ok = PyArg_ParseTuple(PySequence_Fast_GET_ITEM(fo, k), "iLi", &code, &length, &key) && scalar_type(code, &o.dtype);
    o.length = length;
    o.key = key;
    l->operands->push_back(o);
  }
  Py_XDECREF(fo);
  if (!ok) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bad launcher description");
    Py_DECREF(l);
    return nullptr;
  }
  if (l->kind == kCsr && l->sizes->size() == 4) {
    const std::vector<int64_t>& n = *l->sizes;
    l->csr.counters = stir_csr_spmm_workspace_clear_bytes((int32_t)n[0], (int32_t)n[1], (int32_t)n[2], n[3]);
    l->csr.rest = stir_csr_spmm_workspace_bytes((int32_t)n[0], (int32_t)n[1], (int32_t)n[2], n[3]) - l->csr.counters;
  }
  return reinterpret_cast<PyObject*>(l);
}

void launcher_dealloc(PyObject* self) {
  Launcher* l = reinterpret_cast<Launcher*>(self);
  delete l->sizes;
  delete l->operands;
  if (l->plans) drop(l, nullptr);
  delete l->plans;
  delete l->key;
  delete l->in_use;
  delete l->workspaces;
  Py_TYPE(self)->tp_free(self);
}

PyMethodDef launcher_methods[] = {
    {"launch", launch, METH_O, "launch(args) -> 0: launched, -1: refused, 1: not taken, or the name of the plan"},
    {"remember", remember, METH_VARARGS, "remember(args, plan, name): a plan made from these arguments"},
    {"launch_new_hyb", launch_new_hyb, METH_O, "launch_new_hyb(args) -> (name, plan), 0: launched, None: not taken, -1: refused"},
    {"forget", forget, METH_O, "forget(name): the plan is no more; None: all of them"},
    {"hyb", launcher_hyb, METH_VARARGS | METH_STATIC, "hyb(n, m, feat, parts, buckets, nrows): launcher of the hyb operator"},
    {nullptr, nullptr, 0, nullptr}};

// ---- decomposition

// A tensor over `sizes` elements of the pool from `offset` on.
PyObject* piece(const at::Tensor& pool, int64_t offset, c10::IntArrayRef sizes) {
  at::Tensor t = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(pool.storage()), pool.key_set(), pool.dtype());
  t.unsafeGetTensorImpl()->set_sizes_contiguous(sizes);
  t.unsafeGetTensorImpl()->set_storage_offset(offset);
  return THPVariable_Wrap(std::move(t));
}

// Appends the buckets' pieces of a pool to `list` (256-byte aligned pieces, as their addresses say).
bool append_pieces(PyObject* list, const at::Tensor& pool, const std::vector<int64_t>& offsets,
                   const std::vector<int64_t>& nrows, const std::vector<int64_t>* widths) {
  for (size_t k = 0; k < nrows.size(); ++k) {
    const int64_t both[2] = {nrows[k], widths ? (*widths)[k] : 0};
    PyObject* t = piece(pool, offsets[k], c10::IntArrayRef(both, widths ? 2 : 1));
    if (!t || PyList_Append(list, t) < 0) {
      Py_XDECREF(t);
      return false;
    }
    Py_DECREF(t);
  }
  return true;
}

// column_part_hyb(num_rows, num_cols, indptr, indices, buckets, values or None) for one column partition
// -> (rows, cols, mask, values) lists over the buckets, values None without; None: not taken; -1: refused
PyObject* column_part_hyb(PyObject*, PyObject* args) {
  int m, n;
  PyObject *o_ptr, *o_idx, *o_buckets, *o_values;
  if (!PyArg_ParseTuple(args, "iiOOOO", &m, &n, &o_ptr, &o_idx, &o_buckets, &o_values)) return nullptr;
  std::vector<int64_t> widths;
  if (!ints_of(o_buckets, &widths)) return nullptr;
  PyObject* lists[4] = {nullptr, nullptr, nullptr, nullptr};
  bool ok = true;
  try {
    const int device = (int)c10::hip::current_device();
    const size_t nb = widths.size();
    if (m < 0 || nb == 0 || nb > 32 || !THPVariable_Check(o_idx)) Py_RETURN_NONE;
    const int64_t nnz = THPVariable_Unpack(o_idx).numel();
    const at::Tensor* ptr = take(o_ptr, {c10::ScalarType::Int, (int64_t)m + 1, kKeyVersion}, device);
    const at::Tensor* idx = take(o_idx, {c10::ScalarType::Int, nnz, kKeyVersion}, device);
    const bool with_values = o_values != Py_None;
    const at::Tensor* val = with_values ? take(o_values, {c10::ScalarType::Float, nnz, kKeyVersion}, device) : nullptr;
    if (!ptr || !idx || (with_values && !val)) Py_RETURN_NONE;
    void* st = c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream();
    const int32_t* d_ptr = static_cast<const int32_t*>(ptr->data_ptr());
    const int32_t* d_idx = static_cast<const int32_t*>(idx->data_ptr());
    const float* d_val = val ? static_cast<const float*>(val->data_ptr()) : nullptr;
    std::vector<int32_t> w32(widths.begin(), widths.end());
    std::vector<int64_t> nrows(nb), row_at(nb), slot_at(nb);
    const at::TensorOptions on = ptr->options();
    const int64_t ws_bytes = (int64_t)stir_column_part_hyb_device_workspace_bytes(m, 1, (int32_t)nb, nnz);
    // freed to the allocator of this stream when the call returns: what uses it next runs after the
    // kernels below
    const at::Tensor ws = at::empty({std::max<int64_t>(ws_bytes, 256)}, on.dtype(c10::ScalarType::Byte));
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = stir::column_part_hyb_one_sizes(m, n, d_ptr, d_idx, nnz, w32.data(), (int32_t)nb, ws.data_ptr(), nrows.data(), st);
    Py_END_ALLOW_THREADS
    if (rc != 0) return PyLong_FromLong(kFailed);
    int64_t rows = 0, slots = 0;
    for (size_t k = 0; k < nb; ++k) {
      row_at[k] = rows, slot_at[k] = slots;
      rows += (nrows[k] + 63) / 64 * 64;
      slots += (nrows[k] * widths[k] + 63) / 64 * 64;
    }
    const at::Tensor pool_rows = at::empty({std::max<int64_t>(rows, 1)}, on);
    const at::Tensor pool_cols = at::empty({std::max<int64_t>(slots, 1)}, on);
    const at::Tensor pool_mask = at::empty({std::max<int64_t>(slots, 1)}, on);
    const at::Tensor pool_vals =
        val ? at::empty({std::max<int64_t>(slots, 1)}, on.dtype(c10::ScalarType::Float)) : at::Tensor();
    std::vector<int32_t*> r(nb), c(nb), k01(nb);
    std::vector<float*> a(nb);
    for (size_t k = 0; k < nb; ++k) {
      r[k] = static_cast<int32_t*>(pool_rows.data_ptr()) + row_at[k];
      c[k] = static_cast<int32_t*>(pool_cols.data_ptr()) + slot_at[k];
      k01[k] = static_cast<int32_t*>(pool_mask.data_ptr()) + slot_at[k];
      if (val) a[k] = static_cast<float*>(pool_vals.data_ptr()) + slot_at[k];
    }
    rc = stir_column_part_hyb_one_fill(m, n, d_ptr, d_idx, nnz, d_val, (int32_t)nb, ws.data_ptr(), r.data(), c.data(),
                                       k01.data(), val ? a.data() : nullptr, st);
    if (rc != 0) return PyLong_FromLong(kFailed);
    for (PyObject*& list : lists) ok = (list = PyList_New(0)) != nullptr && ok;
    ok = ok && append_pieces(lists[0], pool_rows, row_at, nrows, nullptr) &&
         append_pieces(lists[1], pool_cols, slot_at, nrows, &widths) &&
         append_pieces(lists[2], pool_mask, slot_at, nrows, &widths) &&
         (!val || append_pieces(lists[3], pool_vals, slot_at, nrows, &widths));
    if (ok && !val) {
      Py_INCREF(Py_None);
      Py_SETREF(lists[3], Py_None);
    }
  } catch (const std::exception& e) {  // out of memory, in torch's words
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
    ok = false;
  }
  PyObject* out = ok ? PyTuple_Pack(4, lists[0], lists[1], lists[2], lists[3]) : nullptr;
  for (PyObject* list : lists) Py_XDECREF(list);
  return out;
}

PyMethodDef module_methods[] = {
    {"column_part_hyb", column_part_hyb, METH_VARARGS,
     "column_part_hyb(num_rows, num_cols, indptr, indices, buckets, values) -> (rows, cols, mask, values)"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "host path of the operators", -1, module_methods};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
  launcher_type.tp_name = "sparsetir_amd._host.Launcher";
  launcher_type.tp_basicsize = sizeof(Launcher);
  launcher_type.tp_flags = Py_TPFLAGS_DEFAULT;
  launcher_type.tp_doc = "Launcher(kind, sizes, operands)";
  launcher_type.tp_new = launcher_new;
  launcher_type.tp_dealloc = launcher_dealloc;
  launcher_type.tp_methods = launcher_methods;
  if (PyType_Ready(&launcher_type) < 0) return nullptr;
  PyObject* m = PyModule_Create(&module);
  if (!m) return nullptr;
  const char* names[kKinds] = {"CSR", "SDDMM_PREPROC", "SDDMM", "SDDMM_SCALED", "BSR", "DBSR",
                               "TC", "RGMS", "RGMS_F32", "RGMS_CSF", "HYB"};
  for (int k = 0; k < kKinds; ++k) PyModule_AddIntConstant(m, names[k], k);
  Py_INCREF(&launcher_type);
  PyModule_AddObject(m, "Launcher", reinterpret_cast<PyObject*>(&launcher_type));
  return m;
}

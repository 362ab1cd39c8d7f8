// wir_plans.cpp -- launch plans: the native half of warpir_amd.plans.
//
// A public call (api.gemm, api.attention_forward, api.attention_backward)
// validates its tensors, picks kernels, allocates outputs and packs one
// argument struct per launch.  All of that follows from the tensors' shapes,
// strides, dtypes and device, and in Python it took 5-14 us a call, more
// than the small kernels themselves.  Python does it once per such signature
// and leaves a plan here: the tensors to allocate, and per launch the
// function, grid and argument bytes with the places of the tensor pointers.
// A later call with the same signature allocates, fills the pointers in and
// launches.  Nothing is kept by a tensor's address or identity, and a table
// holds at most MAX_PLANS plans (a new one then takes the place of another,
// drawn at random: a program that goes round more signatures than that still
// finds part of them, where dropping the oldest or all would find none).
//
// run() returns False for every call that it does not know and None for those
// it must not take (tensor subclasses, functorch or Python-dispatch wrappers,
// active torch function / dispatch modes, empty or not 16-byte aligned
// tensors); the Python path then does, with its own checks and errors, and
// leaves a plan after False only.  The interpreter
// lock guards the tables; it is released around the launches only.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <memory>
#include <string>
#include <unordered_map>
#include <vector>

namespace {

typedef int (*launch_fn)(void* function, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by, unsigned bz,
                         unsigned dyn_lds, void* stream, const void* kernarg, size_t kernarg_size);

launch_fn g_launch = nullptr;          // wir_launch of libwarpir_rt.so
PyObject* g_current_stream = nullptr;  // torch._C._cuda_getCurrentRawStream

constexpr size_t MAX_PLANS = 256;
constexpr int MAX_SLOTS = 16;
constexpr size_t MAX_ARGS = 1024;      // bytes of one launch's arguments

struct Pointer {
  unsigned offset;    // of the pointer in the argument bytes
  int slot;           // inputs first, then the plan's allocations
  long long addend;   // bytes past the tensor's data
};

struct Launch {
  void* function;
  unsigned grid[3], block[3], dyn_lds;
  std::string args;
  std::vector<Pointer> pointers;
};

struct Alloc {
  std::vector<int64_t> sizes, strides;
  at::ScalarType dtype;
};

struct Plan {
  std::vector<Alloc> allocs;
  std::vector<Launch> launches;
  std::vector<int> results;   // slots
};

struct Table {
  std::unordered_map<std::string, std::shared_ptr<Plan>> plans;
  std::vector<const std::string*> keys;   // of every plan (a map's keys stay where they are)
  uint32_t draw = 0x9e3779b9u;            // xorshift state

  void keep(const std::string& key, std::shared_ptr<Plan> plan) {
    auto found = plans.find(key);
    if (found != plans.end()) {
      found->second = std::move(plan);
      return;
    }
    auto it = plans.emplace(key, std::move(plan)).first;
    if (keys.size() < MAX_PLANS) {
      keys.push_back(&it->first);
      return;
    }
    draw ^= draw << 13, draw ^= draw >> 17, draw ^= draw << 5;
    const std::string*& slot = keys[draw % MAX_PLANS];
    const std::string old = *slot;
    slot = &it->first;
    plans.erase(old);
  }
};

const char* kTableName = "warpir_amd.plans.Table";

Table* table_of(PyObject* capsule) { return static_cast<Table*>(PyCapsule_GetPointer(capsule, kTableName)); }

void free_table(PyObject* capsule) { delete table_of(capsule); }

// A dense, strided, non-empty GPU tensor with nothing wrapped around it.
bool plain(const at::Tensor& t) {
  static const c10::DispatchKeySet allowed =
      c10::DispatchKeySet(c10::DispatchKey::CUDA) | c10::DispatchKeySet(c10::DispatchKey::AutogradCUDA) |
      c10::DispatchKeySet(c10::DispatchKey::AutocastCUDA) | c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView);
  const c10::TensorImpl* impl = t.unsafeGetTensorImpl();
  return (impl->key_set().raw_repr() & ~allowed.raw_repr()) == 0 && t.is_cuda() && !impl->has_symbolic_sizes_strides() && t.numel() > 0 &&
         t.dim() <= 8;
}

// The signature of `flags` and the tensors (None allowed) args[0..n), whose
// tensors go to `slots`; false when the call is not one for a plan.
bool signature(long long flags, PyObject* const* args, Py_ssize_t n, std::string& key, const at::Tensor** slots,
               int* device) {
  if (n > MAX_SLOTS || c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled())
    return false;
  long long buf[2 + MAX_SLOTS * 18];
  int w = 0;
  buf[w++] = flags;
  *device = -1;
  for (Py_ssize_t i = 0; i < n; ++i) {
    slots[i] = nullptr;
    if (args[i] == Py_None) {
      buf[w++] = -1;
      continue;
    }
    if (!THPVariable_CheckExact(args[i])) return false;
    const at::Tensor& t = THPVariable_Unpack(args[i]);
    if (!t.defined() || !plain(t)) return false;
    if (((uintptr_t)t.data_ptr() & 15) != 0) return false;
    slots[i] = &t;
    if (*device < 0) *device = t.get_device();
    buf[w++] = ((long long)t.get_device() << 32) | ((long long)t.scalar_type() << 8) | t.dim();
    for (int64_t d = 0; d < t.dim(); ++d) {
      buf[w++] = t.sizes()[d];
      buf[w++] = t.strides()[d];
    }
  }
  if (*device < 0) return false;
  key.assign(reinterpret_cast<const char*>(buf), w * sizeof(buf[0]));
  return true;
}

bool flags_of(PyObject* o, long long* flags) {
  *flags = PyLong_AsLongLong(o);
  if (!PyErr_Occurred()) return true;
  PyErr_Clear();
  return false;
}

// Whether no tensor is given twice: the launches of a call that gives one
// twice do not tell which argument a pointer came from.
bool distinct(PyObject* const* args, Py_ssize_t n) {
  for (Py_ssize_t i = 0; i < n; ++i)
    for (Py_ssize_t j = i + 1; j < n; ++j)
      if (args[i] == args[j] && args[i] != Py_None) return false;
  return true;
}

// run(table, flags, *tensors) -> the plan's result tensors (one, or a tuple),
// an int error code of a failed launch, False where the call has no plan yet
// and can leave one, or None where it can not.
PyObject* run(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs < 3 || !g_launch) Py_RETURN_NONE;
  Table* table = table_of(args[0]);
  if (!table) return nullptr;
  const Py_ssize_t n = nargs - 2;
  const at::Tensor* slots[MAX_SLOTS];
  std::string key;
  int device = -1;
  long long flags;
  if (!flags_of(args[1], &flags) || !signature(flags, args + 2, n, key, slots, &device)) Py_RETURN_NONE;
  auto it = table->plans.find(key);
  if (it == table->plans.end()) {
    if (distinct(args + 2, n)) Py_RETURN_FALSE;
    Py_RETURN_NONE;
  }
  const std::shared_ptr<Plan> plan = it->second;   // stays alive if another thread drops it from the table

  std::vector<at::Tensor> made;
  made.reserve(plan->allocs.size());
  for (const Alloc& a : plan->allocs) {
    made.push_back(at::empty_strided(
        a.sizes, a.strides, at::TensorOptions().dtype(a.dtype).device(c10::Device(c10::DeviceType::CUDA, device))));
    if (!plain(made.back())) Py_RETURN_NONE;
  }
  char* data[MAX_SLOTS];
  for (Py_ssize_t i = 0; i < n; ++i) data[i] = slots[i] ? (char*)slots[i]->data_ptr() : nullptr;
  for (size_t i = 0; i < made.size(); ++i) data[n + i] = (char*)made[i].data_ptr();

  PyObject* index = PyLong_FromLong(device);
  PyObject* raw = index ? PyObject_CallFunctionObjArgs(g_current_stream, index, nullptr) : nullptr;
  Py_XDECREF(index);
  if (!raw) return nullptr;
  void* stream = PyLong_AsVoidPtr(raw);
  Py_DECREF(raw);
  if (PyErr_Occurred()) return nullptr;

  int code = 0;
  Py_BEGIN_ALLOW_THREADS
  alignas(16) char buf[MAX_ARGS];
  for (const Launch& l : plan->launches) {
    std::memcpy(buf, l.args.data(), l.args.size());
    for (const Pointer& p : l.pointers) {
      char* x = data[p.slot] + p.addend;
      std::memcpy(buf + p.offset, &x, sizeof(x));
    }
    code = g_launch(l.function, l.grid[0], l.grid[1], l.grid[2], l.block[0], l.block[1], l.block[2], l.dyn_lds, stream,
                    buf, l.args.size());
    if (code) break;
  }
  Py_END_ALLOW_THREADS
  if (code) return PyLong_FromLong(code);

  auto result = [&](int slot) -> PyObject* {
    if (slot >= n) return THPVariable_Wrap(made[slot - n]);
    Py_INCREF(args[2 + slot]);
    return args[2 + slot];
  };
  if (plan->results.size() == 1) return result(plan->results[0]);
  PyObject* out = PyTuple_New((Py_ssize_t)plan->results.size());
  if (!out) return nullptr;
  for (size_t i = 0; i < plan->results.size(); ++i) {
    PyObject* x = result(plan->results[i]);
    if (!x) {
      Py_DECREF(out);
      return nullptr;
    }
    PyTuple_SET_ITEM(out, (Py_ssize_t)i, x);
  }
  return out;
  END_HANDLE_TH_ERRORS
}

// add(table, flags, inputs, allocs, launches, results): the plan of a call.
//   inputs   tuple of tensors or None
//   allocs   list of tensors the call allocated (shape, strides, dtype)
//   launches list of (function, (gx, gy, gz), (bx, by, bz), dyn_lds, args bytes,
//            [(offset, slot, addend), ...])
//   results  list of slots
// Returns whether the plan was kept.
PyObject* add(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *capsule, *flags, *inputs, *allocs, *launches, *results;
  if (!PyArg_ParseTuple(args, "OOO!O!O!O!", &capsule, &flags, &PyTuple_Type, &inputs, &PyList_Type, &allocs,
                        &PyList_Type, &launches, &PyList_Type, &results))
    return nullptr;
  Table* table = table_of(capsule);
  if (!table) return nullptr;
  const Py_ssize_t n = PyTuple_GET_SIZE(inputs), made = PyList_GET_SIZE(allocs);
  const at::Tensor* slots[MAX_SLOTS];
  std::string key;
  int device = -1;
  if (n + made > MAX_SLOTS || n < 1) Py_RETURN_FALSE;
  long long bits;
  PyObject* const* given = &PyTuple_GET_ITEM(inputs, 0);
  if (!flags_of(flags, &bits) || !distinct(given, n) || !signature(bits, given, n, key, slots, &device))
    Py_RETURN_FALSE;
  auto plan = std::make_shared<Plan>();
  for (Py_ssize_t i = 0; i < made; ++i) {
    PyObject* o = PyList_GET_ITEM(allocs, i);
    if (!THPVariable_CheckExact(o)) Py_RETURN_FALSE;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!plain(t) || t.get_device() != device) Py_RETURN_FALSE;
    plan->allocs.push_back({t.sizes().vec(), t.strides().vec(), t.scalar_type()});
  }
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(launches); ++i) {
    Launch l;
    unsigned long long fn;
    const char* bytes;
    Py_ssize_t size;
    PyObject* pointers;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(launches, i), "K(III)(III)Iy#O!", &fn, &l.grid[0], &l.grid[1], &l.grid[2],
                          &l.block[0], &l.block[1], &l.block[2], &l.dyn_lds, &bytes, &size, &PyList_Type, &pointers))
      return nullptr;
    if (!fn || (size_t)size > MAX_ARGS) Py_RETURN_FALSE;
    l.function = (void*)fn;
    l.args.assign(bytes, size);
    for (Py_ssize_t j = 0; j < PyList_GET_SIZE(pointers); ++j) {
      Pointer p;
      if (!PyArg_ParseTuple(PyList_GET_ITEM(pointers, j), "IiL", &p.offset, &p.slot, &p.addend)) return nullptr;
      if (p.offset + sizeof(void*) > (size_t)size || p.slot < 0 || p.slot >= n + made ||
          (p.slot < n && !slots[p.slot]))
        Py_RETURN_FALSE;
      l.pointers.push_back(p);
    }
    plan->launches.push_back(std::move(l));
  }
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(results); ++i) {
    const long s = PyLong_AsLong(PyList_GET_ITEM(results, i));
    if (s == -1 && PyErr_Occurred()) return nullptr;
    if (s < 0 || s >= n + made || (s < n && !slots[s])) Py_RETURN_FALSE;
    plan->results.push_back((int)s);
  }
  if (plan->results.empty()) Py_RETURN_FALSE;
  table->keep(key, std::move(plan));
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// size(table): the number of plans held.
PyObject* size(PyObject*, PyObject* capsule) {
  Table* table = table_of(capsule);
  return table ? PyLong_FromSize_t(table->plans.size()) : nullptr;
}

PyObject* new_table(PyObject*, PyObject*) { return PyCapsule_New(new Table, kTableName, free_table); }

// init(address of wir_launch, torch._C._cuda_getCurrentRawStream)
PyObject* init(PyObject*, PyObject* args) {
  unsigned long long fn;
  PyObject* stream;
  if (!PyArg_ParseTuple(args, "KO", &fn, &stream)) return nullptr;
  Py_INCREF(stream);
  Py_XDECREF(g_current_stream);
  g_current_stream = stream;
  g_launch = (launch_fn)fn;
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"run", (PyCFunction)(void (*)(void))run, METH_FASTCALL, nullptr},
                         {"add", add, METH_VARARGS, nullptr},
                         {"size", size, METH_O, nullptr},
                         {"table", new_table, METH_NOARGS, nullptr},
                         {"init", init, METH_VARARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_wir_plans", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__wir_plans() { return PyModule_Create(&module); }

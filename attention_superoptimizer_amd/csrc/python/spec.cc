// _spec: builds a graph spec (workloads.py: a list of dicts) through the C facade of the host API.
// A search builds a graph per candidate and drops it after one verification; through ctypes that was
// a call, its argument conversions and a tensor query per operator: 18 us a graph, two thirds of a
// candidate's cost.  Here the dicts are read where they are: 3.0 us (4.0 while the tensors' __init__ was called
// and plans were copied into their operators).
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

#include <cstring>
#include <vector>

#include "mirage/c_plan.h"

extern "C" {
void *mirage_graph_new_input(void *g, int const *dims, int nd, int dtype, int layout);
void *mirage_graph_matmul(void *g, void *a, void *b);
void *mirage_graph_unary(void *g, int op, void *a);
void *mirage_graph_binary(void *g, int op, void *a, void *b);
void *mirage_graph_reduction(void *g, void *a, int dim, int size);
int mirage_graph_customized(void *g, void *const *inputs, int num_inputs, mirage_c_plan const *p, void **outputs,
                            int max_outputs);
int mirage_tensor_info(void *t, int *num_dims, int *dims, int *dtype, int *layout, long long *guid);
}

namespace {

constexpr int kMaxOutputs = 4;

struct Names {
  PyObject *op, *dims, *layout, *in, *dim, *size, *plan;
  PyObject *grid_dim, *block_dim, *output_map, *forloop_range, *reduction_dimx, *input_map, *forloop_dim,
      *input_smem_layouts, *ops, *h, *data_type, *guid, *init, *keeping_init;
} names;

struct Tables {  // of graph.py: name -> code
  PyObject *dmem_layout, *smem_layout, *kn_op, *tb_op, *infeasible;
};

struct Built {
  void *out[kMaxOutputs];
  int n;
};

bool to_int(PyObject *o, int *v) {
  long const x = o == nullptr ? -1 : PyLong_AsLong(o);
  if (o == nullptr || (x == -1 && PyErr_Occurred())) {
    if (!PyErr_Occurred()) {
      PyErr_SetString(PyExc_TypeError, "a number is missing");
    }
    return false;
  }
  *v = (int)x;
  return true;
}

// dict[key], borrowed; KeyError when it is missing
PyObject *item(PyObject *dict, PyObject *key) {
  PyObject *v = PyDict_GetItemWithError(dict, key);
  if (v == nullptr && !PyErr_Occurred()) {
    PyErr_SetObject(PyExc_KeyError, key);
  }
  return v;
}

// `n` numbers of a list or tuple
bool ints(PyObject *seq, int n, int *out) {
  if (seq == nullptr) {
    return false;
  }
  PyObject *fast = PySequence_Fast(seq, "a sequence of numbers is expected");
  if (fast == nullptr) {
    return false;
  }
  bool ok = PySequence_Fast_GET_SIZE(fast) >= n;
  if (!ok) {
    PyErr_SetString(PyExc_IndexError, "list index out of range");
  }
  for (int i = 0; ok && i < n; i++) {
    ok = to_int(PySequence_Fast_GET_ITEM(fast, i), out + i);
  }
  Py_DECREF(fast);
  return ok;
}

// a list or tuple of exactly two, as unpacking it wants
bool is_pair(PyObject *o) {
  Py_ssize_t const n = PySequence_Size(o);
  if (n >= 0 && n != 2) {
    PyErr_SetString(PyExc_ValueError, "two values are expected");
  }
  return n == 2;
}

// a code given by name, or as a number where `number_too`
bool code(PyObject *table, PyObject *o, bool number_too, int *v) {
  if (number_too && !PyUnicode_Check(o)) {
    return to_int(o, v);
  }
  PyObject *c = item(table, o);
  return c != nullptr && to_int(c, v);
}

bool read_plan(PyObject *plan, Tables const &t, mirage_c_plan *p) {
  std::memset(p, 0, sizeof(*p));
  PyObject *input_map = item(plan, names.input_map), *ops = input_map == nullptr ? nullptr : item(plan, names.ops);
  if (ops == nullptr) {
    return false;
  }
  Py_ssize_t const n_in = PySequence_Size(input_map), n_ops = PySequence_Size(ops);
  if (n_in < 0 || n_ops < 0) {
    return false;
  }
  if (n_in > 4 || n_ops > 16) {
    PyErr_SetString(PyExc_AssertionError, "at most 4 inputs and 16 operators");
    return false;
  }
  PyObject *block = PyDict_GetItemWithError(plan, names.block_dim);
  if (block == nullptr) {
    p->block_dim[0] = 128;
    p->block_dim[1] = p->block_dim[2] = 1;
  } else if (!ints(block, 3, p->block_dim)) {
    return false;
  }
  if (PyErr_Occurred() || !ints(item(plan, names.grid_dim), 3, p->grid_dim) ||
      !ints(item(plan, names.output_map), 3, p->output_map) || !to_int(item(plan, names.forloop_range), &p->forloop_range)) {
    return false;
  }
  PyObject *dimx = PyDict_GetItemWithError(plan, names.reduction_dimx);
  p->reduction_dimx = 64;
  if (PyErr_Occurred() || (dimx != nullptr && !to_int(dimx, &p->reduction_dimx))) {
    return false;
  }
  p->num_inputs = (int)n_in;
  p->num_ops = (int)n_ops;
  if (!ints(item(plan, names.forloop_dim), (int)n_in, p->forloop_dim)) {
    return false;
  }
  PyObject *smem = PyDict_GetItemWithError(plan, names.input_smem_layouts);
  int const truth = smem == nullptr ? 0 : PyObject_IsTrue(smem);
  if (PyErr_Occurred() || truth < 0) {
    return false;
  }
  for (int i = 0; i < (int)n_in; i++) {
    PyObject *map = PySequence_GetItem(input_map, i);
    bool ok = map != nullptr && ints(map, 3, p->input_map[i]);
    Py_XDECREF(map);
    p->input_smem_layout[i] = 200;  // SmemRowMajor
    if (ok && truth) {
      PyObject *lay = PySequence_GetItem(smem, i);
      ok = lay != nullptr && code(t.smem_layout, lay, true, &p->input_smem_layout[i]);
      Py_XDECREF(lay);
    }
    if (!ok) {
      return false;
    }
  }
  for (int i = 0; i < (int)n_ops; i++) {
    PyObject *op = PySequence_GetItem(ops, i);
    PyObject *name = op == nullptr || !is_pair(op) ? nullptr : PySequence_GetItem(op, 0);
    PyObject *operands = name == nullptr ? nullptr : PySequence_GetItem(op, 1);
    bool ok = operands != nullptr && code(t.tb_op, name, true, &p->op_type[i]);
    Py_ssize_t const n = ok ? PySequence_Size(operands) : -1;
    ok = ok && n >= 0;
    if (ok && n > 2) {
      PyErr_SetString(PyExc_AssertionError, "at most 2 operands");
      ok = false;
    }
    p->op_num_operands[i] = (int)n;
    for (int j = 0; ok && j < (int)n; j++) {
      PyObject *pair = PySequence_GetItem(operands, j);
      ok = pair != nullptr && is_pair(pair) && ints(pair, 2, p->op_operands[i][j]);
      Py_XDECREF(pair);
    }
    Py_XDECREF(operands);
    Py_XDECREF(name);
    Py_XDECREF(op);
    if (!ok) {
      return false;
    }
  }
  return true;
}

// the tensor [operator, output] that element `i` of an operator's "in" names
bool operand(PyObject *in, Py_ssize_t i, Built const *built, int count, void **h) {
  PyObject *ref = PySequence_GetItem(in, i);
  int at[2];
  bool ok = ref != nullptr && ints(ref, 2, at);
  Py_XDECREF(ref);
  if (!ok) {
    return false;
  }
  if (at[0] < 0) {
    at[0] += count;
  }
  if (at[0] < 0 || at[0] >= count || (at[1] < 0 ? at[1] += built[at[0]].n : at[1]) < 0 || at[1] >= built[at[0]].n) {
    PyErr_SetString(PyExc_IndexError, "list index out of range");
    return false;
  }
  *h = built[at[0]].out[at[1]];
  return true;
}

// One operator of a spec.
bool build_op(void *g, PyObject *op, Tables const &t, Built *built, int count) {
  PyObject *kind = item(op, names.op);
  char const *k = kind == nullptr ? nullptr : PyUnicode_AsUTF8(kind);
  if (k == nullptr) {
    return false;
  }
  Built &b = built[count];
  b.n = 1;
  b.out[0] = nullptr;
  if (std::strcmp(k, "input") == 0) {
    PyObject *dims = item(op, names.dims);
    Py_ssize_t const nd = dims == nullptr ? -1 : PySequence_Size(dims);
    int d[8], layout = 100;  // DmemRowMajor
    if (nd < 0 || nd > 8) {
      if (nd > 8) {
        PyErr_SetString(PyExc_ValueError, "too many dimensions");
      }
      return false;
    }
    PyObject *lay = PyDict_GetItemWithError(op, names.layout);
    if (PyErr_Occurred() || !ints(dims, (int)nd, d) || (lay != nullptr && !code(t.dmem_layout, lay, false, &layout))) {
      return false;
    }
    b.out[0] = mirage_graph_new_input(g, d, (int)nd, 921 /* DT_FLOAT16 */, layout);
    k = "new_input";
  } else {
    bool const known = std::strcmp(k, "matmul") == 0 || std::strcmp(k, "reduction") == 0 || std::strcmp(k, "customized") == 0;
    int op_code = 0;
    if (!known) {
      PyObject *c = PyDict_GetItemWithError(t.kn_op, kind);
      if (c == nullptr) {
        if (!PyErr_Occurred()) {
          PyErr_SetObject(PyExc_ValueError, kind);
        }
        return false;
      }
      if (!to_int(c, &op_code)) {
        return false;
      }
    }
    PyObject *in = item(op, names.in);
    Py_ssize_t const n = in == nullptr ? -1 : PySequence_Size(in);
    void *h[8];
    if (n < 0) {
      return false;
    }
    if (n > 8) {
      PyErr_SetString(PyExc_ValueError, "too many operands");
      return false;
    }
    bool const binary = std::strcmp(k, "matmul") == 0 || std::strcmp(k, "add") == 0 || std::strcmp(k, "mul") == 0 ||
                        std::strcmp(k, "div") == 0;
    bool const customized = std::strcmp(k, "customized") == 0;
    Py_ssize_t const wanted = customized ? n : binary ? 2 : 1;
    for (Py_ssize_t i = 0; i < wanted; i++) {
      if (!operand(in, i, built, count, h + i)) {
        return false;
      }
    }
    if (customized) {
      mirage_c_plan p;
      PyObject *plan = item(op, names.plan);
      if (plan == nullptr || !read_plan(plan, t, &p)) {
        return false;
      }
      b.n = mirage_graph_customized(g, h, (int)n, &p, b.out, kMaxOutputs);
      if (b.n < 0) {
        b.n = 1;
        b.out[0] = nullptr;
      }
    } else if (std::strcmp(k, "matmul") == 0) {
      b.out[0] = mirage_graph_matmul(g, h[0], h[1]);
    } else if (std::strcmp(k, "reduction") == 0) {
      int dim, size = 1;
      PyObject *s = PyDict_GetItemWithError(op, names.size);
      if (PyErr_Occurred() || !to_int(item(op, names.dim), &dim) || (s != nullptr && !to_int(s, &size))) {
        return false;
      }
      b.out[0] = mirage_graph_reduction(g, h[0], dim, size);
    } else if (binary) {
      b.out[0] = mirage_graph_binary(g, op_code, h[0], h[1]);
    } else {
      b.out[0] = mirage_graph_unary(g, op_code, h[0]);
    }
  }
  if (b.n > 0 && b.out[0] == nullptr) {
    PyErr_SetString(t.infeasible, k);
    return false;
  }
  return true;
}

// The slots of a tensor type that says its __init__ only keeps its arguments in them: where they lie.
struct TensorSlots {
  Py_ssize_t at[4];  // _h, dims, data_type, guid
  bool plain;
};
TensorSlots tensor_slots(PyObject *type) {
  TensorSlots s = {{0, 0, 0, 0}, PyType_Check(type) != 0};
  PyObject *const all[4] = {names.h, names.dims, names.data_type, names.guid};
  PyTypeObject *const t = reinterpret_cast<PyTypeObject *>(type);
  // (no other slots to fill, no __new__, and the __init__ it says so of is the one it has: any other type is called)
  s.plain = s.plain && t->tp_base == &PyBaseObject_Type && t->tp_new == PyBaseObject_Type.tp_new &&
            t->tp_basicsize == (Py_ssize_t)(sizeof(PyObject) + (4 + (t->tp_weaklistoffset != 0)) * sizeof(PyObject *));
  if (s.plain) {
    PyObject *const init = PyDict_GetItem(t->tp_dict, names.init);
    s.plain = init != nullptr && init == PyDict_GetItem(t->tp_dict, names.keeping_init);
  }
  for (int i = 0; s.plain && i < 4; i++) {
    PyObject *const d = PyDict_GetItem(t->tp_dict, all[i]);
    s.plain = d != nullptr && Py_IS_TYPE(d, &PyMemberDescr_Type);
    if (s.plain) {
      PyMemberDef const *const m = reinterpret_cast<PyMemberDescrObject *>(d)->d_member;
      s.plain = m->type == T_OBJECT_EX;
      s.at[i] = m->offset;
    }
  }
  return s;
}

PyObject *make_tensor(PyObject *type, TensorSlots const &slots, void *handle) {
  int nd = 0, dims[4], dtype = 0, layout = 0;
  long long guid = 0;
  mirage_tensor_info(handle, &nd, dims, &dtype, &layout, &guid);
  PyObject *shape = PyTuple_New(nd);
  for (int d = 0; shape != nullptr && d < nd; d++) {
    PyTuple_SET_ITEM(shape, d, PyLong_FromLong(dims[d]));
  }
  PyObject *args[4] = {PyLong_FromVoidPtr(handle), shape, PyLong_FromLong(dtype), PyLong_FromLongLong(guid)};
  PyObject *x = nullptr;
  bool const whole = args[0] != nullptr && args[1] != nullptr && args[2] != nullptr && args[3] != nullptr;
  if (whole && slots.plain) {  // what its __init__ does, 0.2 us of interpreter a tensor
    auto *const t = reinterpret_cast<PyTypeObject *>(type);
    x = t->tp_alloc(t, 0);
    for (int i = 0; x != nullptr && i < 4; i++) {
      *reinterpret_cast<PyObject **>(reinterpret_cast<char *>(x) + slots.at[i]) = args[i];
      args[i] = nullptr;
    }
  } else if (whole) {
    x = PyObject_Vectorcall(type, args, 4, nullptr);
  }
  for (PyObject *a : args) {
    Py_XDECREF(a);
  }
  return x;
}

// build(graph handle, spec, tensor type, four tables, exception) -> list per operator of its output tensors
PyObject *build(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  if (nargs != 8 || !PyList_Check(args[1])) {
    PyErr_SetString(PyExc_TypeError, "a graph handle, a list, a type, four dicts and an exception are expected");
    return nullptr;
  }
  unsigned long long const graph = PyLong_AsUnsignedLongLong(args[0]);
  if (graph == (unsigned long long)-1 && PyErr_Occurred()) {
    return nullptr;
  }
  PyObject *const spec = args[1], *const tensor = args[2];
  Tables t;
  PyObject **const tables[4] = {&t.dmem_layout, &t.smem_layout, &t.kn_op, &t.tb_op};
  for (int i = 0; i < 4; i++) {
    *tables[i] = args[3 + i];
    if (!PyDict_Check(*tables[i])) {
      PyErr_SetString(PyExc_TypeError, "a table is a dict");
      return nullptr;
    }
  }
  t.infeasible = args[7];
  Py_ssize_t const n = PyList_GET_SIZE(spec);
  TensorSlots const slots = tensor_slots(tensor);
  std::vector<Built> built((size_t)n);
  PyObject *all = PyList_New(n);
  if (all == nullptr) {
    return nullptr;
  }
  for (Py_ssize_t i = 0; i < n; i++) {
    PyObject *op = PyList_GET_ITEM(spec, i);
    if (!PyDict_Check(op)) {
      PyErr_SetString(PyExc_TypeError, "an operator is a dict");
      Py_DECREF(all);
      return nullptr;
    }
    if (!build_op(reinterpret_cast<void *>((uintptr_t)graph), op, t, built.data(), (int)i)) {
      Py_DECREF(all);
      return nullptr;
    }
    PyObject *outs = PyList_New(built[i].n);
    if (outs == nullptr) {
      Py_DECREF(all);
      return nullptr;
    }
    PyList_SET_ITEM(all, i, outs);
    for (int j = 0; j < built[i].n; j++) {
      PyObject *x = make_tensor(tensor, slots, built[i].out[j]);
      if (x == nullptr) {
        Py_DECREF(all);
        return nullptr;
      }
      PyList_SET_ITEM(outs, j, x);
    }
  }
  return all;
}

PyMethodDef methods[] = {{"build", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(build)), METH_FASTCALL,
                          "Builds a graph spec; one list of output tensors per operator."},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_spec", "Graph specs read in native code.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__spec(void) {
  struct {
    PyObject **slot;
    char const *text;
  } const all[] = {{&names.op, "op"}, {&names.dims, "dims"}, {&names.layout, "layout"}, {&names.in, "in"}, {&names.dim, "dim"},
                   {&names.size, "size"}, {&names.plan, "plan"}, {&names.grid_dim, "grid_dim"}, {&names.block_dim, "block_dim"},
                   {&names.output_map, "output_map"}, {&names.forloop_range, "forloop_range"},
                   {&names.reduction_dimx, "reduction_dimx"}, {&names.input_map, "input_map"}, {&names.forloop_dim, "forloop_dim"},
                   {&names.input_smem_layouts, "input_smem_layouts"}, {&names.ops, "ops"}, {&names.h, "_h"}, {&names.data_type, "data_type"}, {&names.guid, "guid"},
                   {&names.init, "__init__"}, {&names.keeping_init, "_keeping_init"}};
  for (auto const &n : all) {
    *n.slot = PyUnicode_InternFromString(n.text);
    if (*n.slot == nullptr) {
      return nullptr;
    }
  }
  return PyModule_Create(&module);
}

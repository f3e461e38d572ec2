// tam_host.cpp -- the per-parameter host work of a steady TurboAdam step, in
// C++ (a torch extension module, _tam_host).
//
// A steady step (turboadam_amd/optimizer.py, _FastStep) reuses the descriptor
// table of the previous step and rewrites only what changes: each row's
// gradient pointer and step number.  Before it may, it checks that the step is
// in fact steady: the same parameters have gradients, each parameter still
// has the storage, size and dtype its row was built for, each gradient is a
// dense, contiguous tensor of its parameter's dtype and size on the step's
// device, and each row's state tensors are the objects the row was built from,
// at the same addresses.  Doing this per row in Python costs about a microsecond
// per parameter; here it is a few dictionary lookups and comparisons.
//
// steady_rows() returns False, with nothing written, when any check fails
// (the optimizer then takes its full path, which validates and raises where
// something is wrong); steady_groups() writes the fields the parameter groups
// set (numpy column writes took 20 us a step); advance_steps() adds 1 to each
// state's step counter once the step has been launched.  state_addresses() checks
// the state arrays of a table that is being built.
#include <torch/extension.h>

#include <array>
#include <cmath>
#include <cstdint>
#include <cstring>

#include "../../include/turboadam_amd.h"

namespace py = pybind11;

namespace {

// Borrowed item of a dict by an interned key, or nullptr (no exception set).
PyObject* item(PyObject* d, PyObject* key) {
  if (!PyDict_Check(d)) return nullptr;
  return PyDict_GetItemWithError(d, key);
}

struct Keys {
  PyObject *grad, *compressed_v, *indices, *scales, *exp_avg_sq, *exp_avg, *compress_m, *m_mgr, *encoded,
      *sign_packed, *labels, *block_norms, *alpha, *ef_residual, *step, *lr, *betas, *eps, *weight_decay, *bc1, *bc2;
  Keys() {
    grad = PyUnicode_InternFromString("grad");
    compressed_v = PyUnicode_InternFromString("compressed_v");
    indices = PyUnicode_InternFromString("indices");
    scales = PyUnicode_InternFromString("scales");
    exp_avg_sq = PyUnicode_InternFromString("exp_avg_sq");
    exp_avg = PyUnicode_InternFromString("exp_avg");
    compress_m = PyUnicode_InternFromString("_compress_m");
    m_mgr = PyUnicode_InternFromString("m_mgr");
    encoded = PyUnicode_InternFromString("_encoded");
    sign_packed = PyUnicode_InternFromString("sign_packed");
    labels = PyUnicode_InternFromString("labels");
    block_norms = PyUnicode_InternFromString("block_norms");
    alpha = PyUnicode_InternFromString("_alpha");
    ef_residual = PyUnicode_InternFromString("_ef_residual");
    step = PyUnicode_InternFromString("step");
    lr = PyUnicode_InternFromString("lr");
    betas = PyUnicode_InternFromString("betas");
    eps = PyUnicode_InternFromString("eps");
    weight_decay = PyUnicode_InternFromString("weight_decay");
    bc1 = PyUnicode_InternFromString("bc1");
    bc2 = PyUnicode_InternFromString("bc2");
  }
};

const Keys& keys() {
  static const Keys k;
  return k;
}

// Where a tensor's elements were: its implementation, storage, the storage's
// memory and the offset in it.  None: all zero.
struct Place {  // 32 bytes (optimizer._FastStep)
  const at::TensorImpl* impl;
  c10::StorageImpl* storage;
  const void* data;
  int64_t offset;
};
static_assert(sizeof(Place) == 32, "the array's size in _FastStep");
Place place_of(PyObject* o) {
  if (o == Py_None) return Place{nullptr, nullptr, nullptr, 0};
  const at::TensorImpl* t = THPVariable_Unpack(o).unsafeGetTensorImpl();
  c10::StorageImpl* s = t->has_storage() ? t->unsafe_storage().unsafeGetStorageImpl() : nullptr;
  return Place{t, s, s ? s->mutable_data() : nullptr, s ? t->storage_offset() : 0};
}
// Whether the tensor is still there.  A kept pointer is followed only once the
// object above it has been seen to hold it still (nothing keeps them alive).
bool in_place(PyObject* o, const Place& at) {
  if (o == Py_None) return !at.impl;
  const at::TensorImpl* t = THPVariable_Unpack(o).unsafeGetTensorImpl();
  if (t != at.impl || !t->has_storage() || t->unsafe_storage().unsafeGetStorageImpl() != at.storage) return false;
  return at.storage->mutable_data() == at.data && t->storage_offset() == at.offset;
}

// Whether the state tensors of one row are, in order, the kept objects at
// kept[*pos ...] (the order of optimizer._row_tensors), in their places at[*pos
// ...]; advances *pos.
bool row_tensors_kept(PyObject* st, bool compress_v, PyObject* kept, const Place* at, Py_ssize_t n_kept,
                      Py_ssize_t* pos) {
  const Keys& K = keys();
  PyObject* got[8];
  int n = 0;
  if (compress_v) {
    PyObject* cv = item(st, K.compressed_v);
    if (!cv) return false;
    got[n++] = item(cv, K.indices);
    got[n++] = item(cv, K.scales);
  } else {
    got[n++] = item(st, K.exp_avg_sq);
  }
  PyObject* cm = item(st, K.compress_m);
  if (!cm) return false;
  const int costate = PyObject_IsTrue(cm);
  if (costate < 0) return false;
  if (costate) {
    PyObject* mgr = item(st, K.m_mgr);
    if (!mgr) return false;
    // the manager's attributes from its instance dict (an attribute held
    // elsewhere is not found: the step is then not taken as steady)
    PyObject* md = PyObject_GenericGetDict(mgr, nullptr);  // new reference
    if (!md) return false;
    PyObject* enc = item(md, K.encoded);
    PyObject* a = item(md, K.alpha);
    PyObject* r = item(md, K.ef_residual);
    Py_DECREF(md);  // the manager keeps its dict and the objects alive
    if (!enc || !a || !r) return false;
    got[n++] = item(enc, K.sign_packed);
    got[n++] = item(enc, K.labels);
    got[n++] = item(enc, K.block_norms);
    got[n++] = item(enc, K.scales);
    got[n++] = a;
    got[n++] = r;
  } else {
    got[n++] = item(st, K.exp_avg);
  }
  for (int i = 0; i < n; ++i) {
    if (!got[i] || *pos >= n_kept) return false;
    // None in the kept list stands for a missing error-feedback residual
    if (PyList_GET_ITEM(kept, *pos) != got[i] || !in_place(got[i], at[*pos])) return false;
    ++*pos;
  }
  return true;
}

// The address of a tensor's elements for writing (a copy-on-write tensor gets its
// own memory first), 0 for None.
uint64_t address_of(PyObject* o) {
  return o == Py_None ? 0u : (uint64_t)(uintptr_t)THPVariable_Unpack(o).data_ptr();
}

// Whether every row's state tensors are the kept objects (lists: the rows'
// state dicts, their compress_v flags, the kept tensors flattened) at their kept
// places (one per kept tensor): a tensor whose .data was replaced is the same
// object elsewhere.  What the places' comparison reads is fetched while the
// dictionaries are walked: in training the caches hold little of it, and tensor by
// tensor its loads wait on one another (5000 tensors of 1000 parameters, caches
// cleared: 220 us without the comparison, 540 with it unfetched, 450 so; caches
// warm: 70, 185 and 165).
bool all_rows_kept(PyObject* S, PyObject* CV, PyObject* T, const Place* at) {
  if (!PyList_Check(S) || !PyList_Check(CV) || !PyList_Check(T) || PyList_GET_SIZE(S) != PyList_GET_SIZE(CV))
    return false;
  Py_ssize_t pos = 0, ahead = 0;
  const Py_ssize_t n_kept = PyList_GET_SIZE(T), n_rows = PyList_GET_SIZE(S);
  for (Py_ssize_t j = 0; j < n_rows; ++j) {
    for (; ahead < n_kept && ahead < pos + 32; ++ahead) {
      __builtin_prefetch(PyList_GET_ITEM(T, ahead));
      __builtin_prefetch(at[ahead].impl);
      __builtin_prefetch((const char*)at[ahead].impl + 128);  // the storage offset's line
      __builtin_prefetch(at[ahead].storage);
    }
    if (j + 8 < n_rows) __builtin_prefetch(PyList_GET_ITEM(S, j + 8));
    if (j + 4 < n_rows && PyDict_Check(PyList_GET_ITEM(S, j + 4)))
      __builtin_prefetch(((PyDictObject*)PyList_GET_ITEM(S, j + 4))->ma_keys);
    if (!row_tensors_kept(PyList_GET_ITEM(S, j), PyList_GET_ITEM(CV, j) == Py_True, T, at, n_kept, &pos)) {
      PyErr_Clear();
      return false;
    }
  }
  return pos == n_kept;
}

// What a steady step reads of the kept _FastStep (its tuple `native`): one
// attribute lookup for all of it.
struct Native {
  PyObject *params;   // list: every parameter
  PyObject *absent;   // list of bools: it had no gradient
  PyObject *grads;    // list: the rows' gradients, kept until the next step
  PyObject *states;   // list: the rows' state dicts
  PyObject *row_cv;   // list of bools: the rows' compress_v
  PyObject *tensors;  // list: the rows' state tensors, flattened
  const Place* tensor_at;     // their places
  const int64_t* rows;        // the rows' positions in params (after the places in memory)
  int64_t dev_index;
};
bool native_of(py::handle f, py::object* hold, Native* n) {
  *hold = f.attr("native");
  PyObject* t = hold->ptr();
  if (!PyTuple_Check(t) || PyTuple_GET_SIZE(t) != 8) return false;
  PyObject** lists[6] = {&n->params, &n->absent, &n->grads, &n->states, &n->row_cv, &n->tensors};
  for (int i = 0; i < 6; ++i) {
    *lists[i] = PyTuple_GET_ITEM(t, i);
    if (!PyList_Check(*lists[i])) return false;
  }
  n->tensor_at = (const Place*)(uintptr_t)PyLong_AsUnsignedLongLong(PyTuple_GET_ITEM(t, 6));
  n->rows = (const int64_t*)(n->tensor_at + PyList_GET_SIZE(n->tensors));
  n->dev_index = PyLong_AsLongLong(PyTuple_GET_ITEM(t, 7));
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

}  // namespace

// Whether the rows' state tensors of the kept _FastStep f are still the
// objects its descriptor rows were built from, at the same addresses.
bool states_kept(py::handle f) {
  py::object hold;
  Native n;
  return native_of(f, &hold, &n) && all_rows_kept(n.states, n.row_cv, n.tensors, n.tensor_at);
}

// An array's memory of at least `bytes` (without the format string, which takes
// numpy longer than the checks below for a table of descriptors).
void* writable(py::handle array, size_t bytes) {
  Py_buffer view;
  if (PyObject_GetBuffer(array.ptr(), &view, PyBUF_WRITABLE) != 0) throw py::error_already_set();
  void* at = view.buf;
  const bool fits = (size_t)view.len >= bytes;
  PyBuffer_Release(&view);
  if (!fits) throw py::value_error("the array is too short");
  return at;
}

// The places of a list of tensors and, after them, the integers of a list, written
// to an array; its address.
uint64_t tensor_places(py::list tensors, py::list rows, py::handle out) {
  const Py_ssize_t n = PyList_GET_SIZE(tensors.ptr()), m = PyList_GET_SIZE(rows.ptr());
  Place* at = (Place*)writable(out, sizeof(Place) * (size_t)n + sizeof(int64_t) * (size_t)m);
  int64_t* r = (int64_t*)(at + n);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* o = PyList_GET_ITEM(tensors.ptr(), i);
    if (o != Py_None && !THPVariable_Check(o)) throw py::type_error("tensor_places: not a tensor");
    at[i] = place_of(o);
  }
  for (Py_ssize_t i = 0; i < m; ++i) r[i] = py::handle(PyList_GET_ITEM(rows.ptr(), i)).cast<int64_t>();
  return (uint64_t)(uintptr_t)at;
}

// The addresses of the shared bias-correction tensors (map[key]["bc1"] and "bc2"
// for each key), written to out_addr in order, for kernels that store one float
// to each.  False, with nothing written, unless every one of them is a
// one-element fp32 tensor on the HIP device dev_index (the full path's fill_
// takes any tensor).
bool bias_addresses(py::handle map, py::handle keys_, int64_t dev_index, uint64_t out_addr) {
  const Keys& K = keys();
  PyObject *M = map.ptr(), *L = keys_.ptr();
  if (!PyDict_Check(M) || !PyList_Check(L)) return false;
  std::vector<void*> at;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(L); ++i) {
    PyObject* pair = PyDict_GetItemWithError(M, PyList_GET_ITEM(L, i));
    for (PyObject* name : {K.bc1, K.bc2}) {
      PyObject* o = pair ? item(pair, name) : nullptr;
      if (!o || !THPVariable_Check(o)) {
        PyErr_Clear();
        return false;
      }
      const at::Tensor& t = THPVariable_Unpack(o);
      if (!t.is_cuda() || t.get_device() != dev_index || t.layout() != at::kStrided ||
          t.scalar_type() != at::kFloat || t.numel() != 1)
        return false;
      at.push_back(t.data_ptr());
    }
  }
  for (size_t i = 0; i < at.size(); ++i) ((void**)(uintptr_t)out_addr)[i] = at[i];
  return true;
}

// The addresses of the state arrays of descriptor rows, ten to a row in the order
// of optimizer._STATE_SLOTS (None: the row has no such array, address 0), written
// to the rows of the table.  Each array must be a contiguous tensor of its slot's
// dtype on the row's parameter's device, with at least the elements the kernels
// touch.  Returns -1, or the position in `tensors` of the first that is not.
// (One call for a table: eight checks per tensor in Python took 2 ms of the
// first step of 1000 tensors.)
int64_t state_addresses(py::list params, py::list tensors, py::handle table) {
  static const at::ScalarType dtypes[10] = {at::kByte, at::kHalf,  at::kFloat, at::kFloat, at::kByte,
                                            at::kByte, at::kFloat, at::kHalf,  at::kFloat, at::kFloat};
  const Py_ssize_t rows = PyList_GET_SIZE(params.ptr());
  if (PyList_GET_SIZE(tensors.ptr()) != 10 * rows) throw py::value_error("state_addresses: ten arrays to a row");
  TamTensor* T = (TamTensor*)writable(table, (size_t)rows * sizeof(TamTensor));
  for (Py_ssize_t j = 0; j < rows; ++j) {
    PyObject* po = PyList_GET_ITEM(params.ptr(), j);
    if (!THPVariable_Check(po)) throw py::type_error("state_addresses: not a parameter");
    const at::Tensor& p = THPVariable_Unpack(po);
    const int64_t n = p.numel(), nb = (n + TAM_BLOCK_SIZE - 1) / TAM_BLOCK_SIZE;
    const int64_t need[10] = {nb * TAM_BLOCK_SIZE, 2 * nb, n, n, (n + 7) / 8, nb, nb, nb, 1, n};
    uint64_t at[10];
    for (int k = 0; k < 10; ++k) {
      PyObject* o = PyList_GET_ITEM(tensors.ptr(), 10 * j + k);
      if (o != Py_None) {
        if (!THPVariable_Check(o)) return 10 * j + k;
        const at::Tensor& t = THPVariable_Unpack(o);
        if (t.layout() != at::kStrided || t.scalar_type() != dtypes[k] || t.device() != p.device() ||
            t.numel() < need[k] || !t.is_contiguous())
          return 10 * j + k;
      }
      at[k] = address_of(o);
    }
    TamTensor& t = T[j];
    t.v_idx = (uint8_t*)at[0];
    t.v_scales = (uint16_t*)at[1];
    t.exp_avg_sq = (float*)at[2];
    t.exp_avg = (float*)at[3];
    t.signs = (uint8_t*)at[4];
    t.labels = (uint8_t*)at[5];
    t.norms = (float*)at[6];
    t.amp = (uint16_t*)at[7];
    t.alpha = (float*)at[8];
    t.ef_residual = (float*)at[9];
  }
  return -1;
}

// The addresses of a list of tensors (0 for None).
py::list tensor_addresses(py::list tensors) {
  const Py_ssize_t n = PyList_GET_SIZE(tensors.ptr());
  py::list out(n);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* o = PyList_GET_ITEM(tensors.ptr(), i);
    if (o != Py_None && !THPVariable_Check(o)) throw py::type_error("tensor_addresses: not a tensor");
    PyList_SET_ITEM(out.ptr(), i, PyLong_FromUnsignedLongLong(address_of(o)));
  }
  return out;
}

// The fields that parameter groups set in the rows of a descriptor table: for each
// row j those of group_rows[gsel[j]] (tuples in the order of
// TurboAdam._group_fields), and the weight-decay flag (wd, a list of bools).
// (Column by column in numpy this took 70 us of a 12-tensor set's first step.)
void set_group_fields(py::handle table, py::handle gsel, py::list group_rows, py::list wd) {
  const size_t groups = group_rows.size();
  std::vector<std::array<double, 12>> v(groups);
  for (size_t g = 0; g < groups; ++g) {
    const py::tuple t = group_rows[g].cast<py::tuple>();
    if (t.size() != 12) throw py::value_error("set_group_fields: twelve fields to a group");
    for (size_t k = 0; k < 12; ++k) v[g][k] = t[k].cast<double>();
  }
  const Py_ssize_t rows = PyObject_Length(gsel.ptr());
  if (rows < 0 || wd.size() != groups) throw py::value_error("set_group_fields: lists of different length");
  TamTensor* T = (TamTensor*)writable(table, (size_t)rows * sizeof(TamTensor));
  const intptr_t* sel = (const intptr_t*)writable(gsel, (size_t)rows * sizeof(intptr_t));
  for (Py_ssize_t j = 0; j < rows; ++j) {
    if (sel[j] < 0 || (size_t)sel[j] >= groups) throw py::value_error("set_group_fields: no such group");
    const std::array<double, 12>& f = v[(size_t)sel[j]];
    TamTensor& t = T[j];
    t.c_wd = (float)f[0];
    t.beta1 = (float)f[1];
    t.one_minus_beta1 = (float)f[2];
    t.beta2 = (float)f[3];
    t.one_minus_beta2 = (float)f[4];
    t.bias_correction1 = (float)f[5];
    t.bias_correction2 = (float)f[6];
    t.inv_bc2 = f[7];
    t.inv_bc2_f32 = (float)f[8];
    t.eps = (float)f[9];
    t.neg_lr = (float)f[10];
    t.sqrt_block = (float)f[11];
    t.flags = (t.flags & ~TAM_FLAG_WD) | (wd[(size_t)sel[j]].cast<bool>() ? TAM_FLAG_WD : 0u);
  }
}

// The per-row part of a steady step (optimizer.TurboAdam._fast_step), given
// the kept _FastStep f and the descriptor table's memory: the state tensors,
// each row's parameter against its descriptor (address, dtype, size, layout),
// its gradient's checks (those of TurboAdam._grad_ptr, also for an object seen
// before: its data may have been replaced), and the shared bias-correction
// tensors (bias_addresses).  On success the gradient pointers and step numbers
// of every row are written and f.grads holds this step's gradients.
bool steady_rows(py::handle f, uint64_t table_addr, py::handle bias_map, py::handle bias_keys, uint64_t bias_out) {
  if (PyErr_Occurred()) return false;
  const Keys& K = keys();
  py::object hold;
  Native N;
  if (!native_of(f, &hold, &N)) return false;
  const Py_ssize_t np_ = PyList_GET_SIZE(N.params), nr = PyList_GET_SIZE(N.states);
  if (PyList_GET_SIZE(N.absent) != np_ || PyList_GET_SIZE(N.grads) != nr) return false;
  if (!all_rows_kept(N.states, N.row_cv, N.tensors, N.tensor_at)) return false;
  // the same parameters have gradients
  std::vector<at::Tensor> gs((size_t)np_);
  for (Py_ssize_t i = 0; i < np_; ++i) {
    PyObject* p = PyList_GET_ITEM(N.params, i);
    if (THPVariable_CheckExact(p)) {  // a tensor or parameter: its grad as the attribute gives it
      gs[(size_t)i] = THPVariable_Unpack(p).grad();
    } else {
      py::object g = py::reinterpret_steal<py::object>(PyObject_GetAttr(p, K.grad));
      if (!g || !(g.is_none() || THPVariable_Check(g.ptr()))) {
        PyErr_Clear();
        return false;
      }
      if (!g.is_none()) gs[(size_t)i] = THPVariable_Unpack(g.ptr());
    }
    if (gs[(size_t)i].defined() == (PyList_GET_ITEM(N.absent, i) == Py_True)) return false;
  }
  TamTensor* T = (TamTensor*)(uintptr_t)table_addr;
  for (Py_ssize_t j = 0; j < nr; ++j) {
    const int64_t i = N.rows[j];
    if (i < 0 || i >= np_ || !THPVariable_Check(PyList_GET_ITEM(N.params, i))) return false;
    const at::Tensor &p = THPVariable_Unpack(PyList_GET_ITEM(N.params, i)), &g = gs[(size_t)i];
    const uint32_t dt = T[j].dtype;
    const at::ScalarType want =
        dt == TAM_DTYPE_F32 ? at::kFloat : dt == TAM_DTYPE_BF16 ? at::kBFloat16 : at::kHalf;
    if (p.scalar_type() != want || !p.is_contiguous() || (uint64_t)p.numel() != T[j].n ||
        p.data_ptr() != T[j].param)
      return false;
    if (!g.defined() || g.scalar_type() != want || g.layout() != at::kStrided || !g.is_cuda() ||
        g.get_device() != N.dev_index || !g.is_contiguous() || g.numel() != p.numel())
      return false;
    PyObject* stp = item(PyList_GET_ITEM(N.states, j), K.step);
    if (!stp || !PyLong_Check(stp) || PyLong_AsLongLong(stp) < 0) {
      PyErr_Clear();
      return false;
    }
  }
  if (!bias_addresses(bias_map, bias_keys, N.dev_index, bias_out)) return false;
  // steady: write the rows' gradient pointers and step numbers
  for (Py_ssize_t j = 0; j < nr; ++j) {
    const at::Tensor& g = gs[(size_t)N.rows[j]];
    T[j].grad = g.const_data_ptr();
    T[j].step = (uint32_t)(PyLong_AsLongLong(item(PyList_GET_ITEM(N.states, j), K.step)) + 1);
    PyObject* o = THPVariable_Wrap(g);
    if (!o) {
      PyErr_Clear();
      return false;
    }
    PyList_SetItem(N.grads, j, o);  // steals the new reference
  }
  return true;
}

// Whether the dict holds exactly the kept values, in order, by identity.
bool values_kept(py::handle map, py::handle kept) {
  PyObject *D = map.ptr(), *L = kept.ptr(), *key = nullptr, *value = nullptr;
  if (!PyDict_Check(D) || !PyList_Check(L) || PyDict_Size(D) != PyList_GET_SIZE(L)) return false;
  Py_ssize_t pos = 0;
  for (Py_ssize_t i = 0; PyDict_Next(D, &pos, &key, &value); ++i)
    if (i >= PyList_GET_SIZE(L) || PyList_GET_ITEM(L, i) != value) return false;
  return true;
}

namespace {

// A Python float or int as a double; false for anything else.
bool number(PyObject* o, double* out) {
  if (!o || !(PyFloat_Check(o) || PyLong_Check(o))) return false;
  *out = PyFloat_AsDouble(o);
  if (*out == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

// betas of a parameter group.
bool betas_of(PyObject* group, double* b1, double* b2) {
  PyObject* t = item(group, keys().betas);
  if (!t || !(PyTuple_Check(t) || PyList_Check(t)) || PySequence_Fast_GET_SIZE(t) != 2) return false;
  return number(PySequence_Fast_GET_ITEM(t, 0), b1) && number(PySequence_Fast_GET_ITEM(t, 1), b2);
}

}  // namespace

// The fields that parameter groups set in the descriptor rows of a steady step
// (optimizer.TurboAdam._group_fields, set_group_fields: each scalar a double
// rounded to fp32 once) and the rows' flags, given the kept _FastStep f: its
// `bc` list of (group, state dict whose step sets the group's bias corrections),
// `groups` list of (group, index into bc or -1) and the addresses of the table,
// of the rows' group numbers (intp) and static flags (uint32), and of 2 floats
// per bc entry that receive the bias corrections.  False, with nothing written,
// for a hyperparameter that is no plain number or gives no finite correction.
bool steady_groups(py::handle f, uint64_t table_addr, int64_t rows, uint64_t gsel_addr, uint64_t flags_addr,
                   uint64_t bc_addr) {
  const Keys& K = keys();
  py::object groups = f.attr("groups"), bc = f.attr("bc");
  PyObject *G = groups.ptr(), *B = bc.ptr();
  if (!PyList_Check(G) || !PyList_Check(B)) return false;
  std::vector<double> corr;  // (1 - beta1^t, 1 - beta2^t) of each bc entry (reference optimizer.py:172-188)
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(B); ++i) {
    PyObject* e = PyList_GET_ITEM(B, i);
    double b1, b2;
    PyObject* step = item(PyTuple_GET_ITEM(e, 1), K.step);
    if (!step || !PyLong_Check(step) || !betas_of(PyTuple_GET_ITEM(e, 0), &b1, &b2)) return false;
    const long long s = PyLong_AsLongLong(step);
    if (s < 0) {
      PyErr_Clear();
      return false;
    }
    const double t = (double)(s + 1), c1 = 1.0 - std::pow(b1, t), c2 = 1.0 - std::pow(b2, t);
    if (!std::isfinite(c1) || !std::isfinite(c2)) return false;
    corr.push_back(c1);
    corr.push_back(c2);
  }
  std::vector<TamTensor> vals;  // the group fields of each group
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(G); ++i) {
    PyObject* e = PyList_GET_ITEM(G, i);
    PyObject* g = PyTuple_GET_ITEM(e, 0);
    const Py_ssize_t k = PyLong_AsSsize_t(PyTuple_GET_ITEM(e, 1));
    double lr, b1, b2, eps, wd;
    if (!number(item(g, K.lr), &lr) || !number(item(g, K.eps), &eps) || !number(item(g, K.weight_decay), &wd) ||
        !betas_of(g, &b1, &b2) || (size_t)(2 * (k + 1)) > corr.size()) {
      PyErr_Clear();
      return false;
    }
    TamTensor v;
    std::memset(&v, 0, sizeof(v));
    v.c_wd = (float)(1.0 - lr * wd);
    v.beta1 = (float)b1;
    v.one_minus_beta1 = (float)(1.0 - b1);
    v.beta2 = (float)b2;
    v.one_minus_beta2 = (float)(1.0 - b2);
    v.bias_correction1 = (float)(k < 0 ? 1.0 : corr[2 * k]);
    v.bias_correction2 = (float)(k < 0 ? 1.0 : corr[2 * k + 1]);
    if (v.bias_correction2 == 0.0f) return false;
    v.inv_bc2 = 1.0 / (double)v.bias_correction2;
    v.inv_bc2_f32 = (float)v.inv_bc2;
    v.eps = (float)eps;
    v.neg_lr = (float)-lr;
    v.flags = wd != 0.0 ? TAM_FLAG_WD : 0u;
    vals.push_back(v);
  }
  TamTensor* T = (TamTensor*)(uintptr_t)table_addr;
  const intptr_t* gsel = (const intptr_t*)(uintptr_t)gsel_addr;
  const uint32_t* flags = (const uint32_t*)(uintptr_t)flags_addr;
  for (int64_t j = 0; j < rows; ++j)
    if (gsel[j] < 0 || (size_t)gsel[j] >= vals.size()) return false;
  for (int64_t j = 0; j < rows; ++j) {
    const TamTensor& v = vals[(size_t)gsel[j]];
    TamTensor& t = T[j];
    t.c_wd = v.c_wd;
    t.beta1 = v.beta1;
    t.one_minus_beta1 = v.one_minus_beta1;
    t.beta2 = v.beta2;
    t.one_minus_beta2 = v.one_minus_beta2;
    t.bias_correction1 = v.bias_correction1;
    t.bias_correction2 = v.bias_correction2;
    t.inv_bc2 = v.inv_bc2;
    t.inv_bc2_f32 = v.inv_bc2_f32;
    t.eps = v.eps;
    t.neg_lr = v.neg_lr;
    t.flags = flags[j] | v.flags;  // a steady step has every encoding and residual (_keep_fast)
    if (flags[j] & TAM_FLAG_COSTATE) t.flags |= TAM_FLAG_HAS_STATE;
    if (flags[j] & TAM_FLAG_EF) t.flags |= TAM_FLAG_HAS_EF;
  }
  float* out = (float*)(uintptr_t)bc_addr;
  for (size_t i = 0; i < corr.size(); ++i) out[i] = (float)corr[i];
  return true;
}

// state["step"] += 1 for each state dict (once the step has been launched).
void advance_steps(py::list states) {
  const Keys& K = keys();
  for (py::handle st : states) {
    PyObject* s = item(st.ptr(), K.step);
    if (!s) throw py::key_error("step");
    PyObject* one = PyLong_FromLong(1);
    PyObject* s1 = PyNumber_Add(s, one);
    Py_DECREF(one);
    if (!s1 || PyDict_SetItem(st.ptr(), K.step, s1) != 0) {
      Py_XDECREF(s1);
      throw py::error_already_set();
    }
    Py_DECREF(s1);
  }
}

PYBIND11_MODULE(_tam_host, m) {
  m.doc() = "Host side of a steady TurboAdam step (turboadam_amd.optimizer)";
  m.def("tensor_addresses", &tensor_addresses, py::arg("tensors"));
  m.def("set_group_fields", &set_group_fields, py::arg("table"), py::arg("gsel"), py::arg("group_rows"),
        py::arg("wd"));
  m.def("state_addresses", &state_addresses, py::arg("params"), py::arg("tensors"), py::arg("table"));
  m.def("steady_rows", &steady_rows, py::arg("f"), py::arg("table_addr"), py::arg("bias_map"), py::arg("bias_keys"),
        py::arg("bias_out"));
  m.def("advance_steps", &advance_steps, py::arg("states"));
  m.def("values_kept", &values_kept, py::arg("map"), py::arg("kept"));
  m.def("steady_groups", &steady_groups, py::arg("f"), py::arg("table_addr"), py::arg("rows"), py::arg("gsel_addr"),
        py::arg("flags_addr"), py::arg("bc_addr"));
  m.def("bias_addresses", &bias_addresses, py::arg("map"), py::arg("keys"), py::arg("dev_index"),
        py::arg("out_addr"));
  m.def("tensor_places", &tensor_places, py::arg("tensors"), py::arg("rows"), py::arg("out"));
  m.def("states_kept", &states_kept, py::arg("f"));
}

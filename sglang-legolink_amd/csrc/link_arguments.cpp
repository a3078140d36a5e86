// The argument blocks of a link and of a repaired-row write-back, filled from
// their tensors.
//
// A link of a 28-layer model names 56 layer buffers.  Checking each of them
// (type, device, shape, dtype, density) and writing its address into the
// pointer tables takes Python 0.6 us a buffer, which for a short request is
// more than the GPU's time; here it takes 30 ns.
//
// Each function returns True when every check of the Python operator holds
// (kv_link._eligibility, PreparedKVScatter) and the block is filled, and False
// otherwise, with nothing to rely on in it: the caller then runs the Python
// checks, which name the reason.  Only plain tensors are taken here.
//
// The module names the torch version and the block sizes that it was built
// for: the caller uses it only where they are its own.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <cstdint>
#include <cstring>

#include "legolink_kv.h"

namespace {

// The tensor of a plain torch.Tensor (or Parameter), else nullptr.
const at::Tensor *plain(PyObject *object) {
  return object != nullptr && THPVariable_CheckExact(object) ? &THPVariable_Unpack(object) : nullptr;
}

int64_t float16_code(at::ScalarType type) {
  return type == at::kHalf ? LL_DTYPE_FLOAT16 : type == at::kBFloat16 ? LL_DTYPE_BFLOAT16 : -1;
}

int64_t index_code(at::ScalarType type) {
  return type == at::kInt ? LL_DTYPE_INT32 : type == at::kLong ? LL_DTYPE_INT64 : -1;
}

// Dense [rows, heads, dim] layers of one device, shape and dtype, their
// addresses in `table`.
struct Layers {
  at::Device device{at::kCPU};
  at::ScalarType type = at::kFloat;
  int64_t count = 0, rows = 0, heads = 0, dim = 0;
};

bool read_layers(PyObject *list, void **table, Layers &out) {
  if (!PyList_CheckExact(list)) return false;
  out.count = PyList_GET_SIZE(list);
  for (int64_t i = 0; i < out.count; ++i) {
    const at::Tensor *t = plain(PyList_GET_ITEM(list, i));
    if (t == nullptr || !t->is_cuda() || t->layout() != at::kStrided || t->dim() != 3 || !t->is_contiguous())
      return false;
    if (i == 0) {
      out.device = t->device();
      out.type = t->scalar_type();
      out.rows = t->size(0);
      out.heads = t->size(1);
      out.dim = t->size(2);
    } else if (t->device() != out.device || t->scalar_type() != out.type || t->size(0) != out.rows ||
               t->size(1) != out.heads || t->size(2) != out.dim) {
      return false;
    }
    table[i] = t->data_ptr();
  }
  return true;
}

// K and V layers of one pool.
bool read_pool(PyObject *keys, PyObject *values, void **tables, Layers &k, Layers &v) {
  if (!PyList_CheckExact(keys) || !PyList_CheckExact(values) || PyList_GET_SIZE(keys) != PyList_GET_SIZE(values) ||
      PyList_GET_SIZE(keys) == 0)
    return false;
  return read_layers(keys, tables, k) && read_layers(values, tables + k.count, v) && k.device == v.device &&
         k.type == v.type && k.rows == v.rows && k.heads == v.heads && float16_code(k.type) >= 0;
}

bool read_index(PyObject *object, at::Device device, int64_t count, const void **address, int64_t *dtype) {
  const at::Tensor *t = plain(object);
  if (t == nullptr || t->device() != device || t->layout() != at::kStrided || t->numel() != count ||
      !t->is_contiguous())
    return false;
  *dtype = index_code(t->scalar_type());
  *address = t->data_ptr();
  return *dtype >= 0;
}

bool fill_link(PyObject *const *a, Py_ssize_t n) {
  if (n != 13) return false;
  auto *args = static_cast<ll_kv_link_args *>(PyLong_AsVoidPtr(a[0]));
  auto **tables = static_cast<void **>(PyLong_AsVoidPtr(a[1]));
  const int64_t rotary = PyLong_AsLongLong(a[12]);
  if (PyErr_Occurred() || args == nullptr || tables == nullptr) return false;
  Layers k, v;
  if (!read_pool(a[2], a[3], tables, k, v)) return false;
  if (k.dim < 1 || k.dim > 256 || v.dim < 1 || v.dim > 256) return false;
  if (!PyList_CheckExact(a[4]) || !PyList_CheckExact(a[5])) return false;
  const int64_t sources = PyList_GET_SIZE(a[4]);
  if (PyList_GET_SIZE(a[5]) != sources || (sources != 0 && sources != k.count)) return false;
  Layers sk, sv;
  if (sources != 0) {
    if (!read_pool(a[4], a[5], tables + 2 * k.count, sk, sv)) return false;
    if (sk.device != k.device || sk.type != k.type || sk.heads != k.heads || sk.dim != k.dim || sv.dim != v.dim)
      return false;
  }
  const at::Tensor *source_slots = plain(a[6]);
  if (source_slots == nullptr) return false;
  const int64_t tokens = source_slots->numel();
  if (tokens == 0) return false;
  if (!read_index(a[6], k.device, tokens, &args->source_slots, &args->source_slots_dtype) ||
      !read_index(a[7], k.device, tokens, &args->destination_slots, &args->destination_slots_dtype) ||
      !read_index(a[8], k.device, tokens, &args->local_positions, &args->local_positions_dtype) ||
      !read_index(a[9], k.device, tokens, &args->global_positions, &args->global_positions_dtype))
    return false;
  const at::Tensor *cache = plain(a[10]);
  if (rotary <= 0 || rotary % 2 != 0 || rotary > k.dim) return false;
  if (cache == nullptr || cache->device() != k.device || cache->layout() != at::kStrided || cache->dim() != 2 ||
      cache->size(1) < rotary)
    return false;
  const int64_t cache_type = cache->scalar_type() == at::kFloat ? LL_DTYPE_FLOAT32 : float16_code(cache->scalar_type());
  if (cache_type < 0) return false;
  args->repair_mask = nullptr;
  if (a[11] != Py_None) {
    const at::Tensor *mask = plain(a[11]);
    if (mask == nullptr || mask->device() != k.device || mask->layout() != at::kStrided || mask->numel() != tokens ||
        !mask->is_contiguous() || (mask->scalar_type() != at::kBool && mask->scalar_type() != at::kByte))
      return false;
    args->repair_mask = static_cast<const uint8_t *>(mask->data_ptr());
  }
  args->repair_mask_dtype = LL_DTYPE_UINT8;
  args->num_layers = k.count;
  args->key_layers = tables;
  args->value_layers = tables + k.count;
  if (sources != 0) {
    args->source_key_layers = tables + 2 * k.count;
    args->source_value_layers = tables + 3 * k.count;
    args->source_num_slots = sk.rows;
  }
  args->num_slots = k.rows;
  args->num_heads = k.heads;
  args->key_head_dim = k.dim;
  args->value_head_dim = v.dim;
  args->kv_dtype = float16_code(k.type);
  args->num_tokens = tokens;
  args->cos_sin_cache = cache->data_ptr();
  args->cos_sin_dtype = cache_type;
  args->cos_sin_rows = cache->size(0);
  args->cos_sin_cols = cache->size(1);
  args->cos_sin_stride_row = cache->stride(0);
  args->cos_sin_stride_col = cache->stride(1);
  args->rotary_dim = rotary;
  return true;
}

// Repaired rows [layers, rows, heads, dim] with dense layers.
bool read_repaired(PyObject *object, const Layers &layers, int64_t rows, const void **address, int64_t *stride) {
  const at::Tensor *t = plain(object);
  if (t == nullptr || t->device() != layers.device || t->layout() != at::kStrided ||
      t->scalar_type() != layers.type || t->dim() != 4 || t->size(0) != layers.count || t->size(1) != rows ||
      t->size(2) != layers.heads || t->size(3) != layers.dim)
    return false;
  if (rows == 0 || t->stride(3) != 1 || t->stride(2) != layers.dim || t->stride(1) != layers.heads * layers.dim)
    return false;  // (sizes of one may have any stride: the Python check decides)
  *address = t->data_ptr();
  *stride = layers.count > 1 ? t->stride(0) : 0;
  return true;
}

bool fill_scatter(PyObject *const *a, Py_ssize_t n) {
  if (n != 7) return false;
  auto *args = static_cast<ll_kv_scatter_args *>(PyLong_AsVoidPtr(a[0]));
  auto **tables = static_cast<void **>(PyLong_AsVoidPtr(a[1]));
  if (PyErr_Occurred() || args == nullptr || tables == nullptr) return false;
  Layers k, v;
  if (!read_pool(a[2], a[3], tables, k, v)) return false;
  const at::Tensor *slots = plain(a[4]);
  if (slots == nullptr) return false;
  const int64_t rows = slots->numel();
  if (!read_index(a[4], k.device, rows, &args->destination_slots, &args->destination_slots_dtype) ||
      !read_repaired(a[5], k, rows, &args->repaired_key, &args->repaired_key_layer_stride) ||
      !read_repaired(a[6], v, rows, &args->repaired_value, &args->repaired_value_layer_stride))
    return false;
  args->num_layers = k.count;
  args->key_layers = tables;
  args->value_layers = tables + k.count;
  args->num_slots = k.rows;
  args->num_heads = k.heads;
  args->key_head_dim = k.dim;
  args->value_head_dim = v.dim;
  args->kv_dtype = float16_code(k.type);
  args->num_rows = rows;
  return true;
}

// No C++ exception and no Python error leaves a call.
template <bool (*kFill)(PyObject *const *, Py_ssize_t)>
PyObject *guarded(PyObject *, PyObject *const *arguments, Py_ssize_t count) {
  bool filled = false;
  try {
    filled = kFill(arguments, count);
  } catch (...) {
    filled = false;
  }
  if (PyErr_Occurred()) {
    PyErr_Clear();
    filled = false;
  }
  return PyBool_FromLong(filled);
}

template <bool (*kFill)(PyObject *const *, Py_ssize_t)>
PyCFunction entry() {
  return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&guarded<kFill>));
}

PyMethodDef methods[] = {
    {"fill_link", entry<fill_link>(), METH_FASTCALL,
     "fill_link(args_address, tables_address, keys, values, source_keys, source_values, source_slots, "
     "destination_slots, local_positions, global_positions, cos_sin_cache, repair_mask, rotary_dim) -> bool"},
    {"fill_scatter", entry<fill_scatter>(), METH_FASTCALL,
     "fill_scatter(args_address, tables_address, keys, values, destination_slots, repaired_keys, repaired_values) "
     "-> bool"},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_link_arguments", "Link argument blocks from tensors.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__link_arguments(void) {
  PyObject *created = PyModule_Create(&module);
  if (created == nullptr) return nullptr;
  if (PyModule_AddStringConstant(created, "TORCH_VERSION", TORCH_VERSION) != 0 ||
      PyModule_AddIntConstant(created, "LINK_ARGS_SIZE", sizeof(ll_kv_link_args)) != 0 ||
      PyModule_AddIntConstant(created, "SCATTER_ARGS_SIZE", sizeof(ll_kv_scatter_args)) != 0) {
    Py_DECREF(created);
    return nullptr;
  }
  return created;
}

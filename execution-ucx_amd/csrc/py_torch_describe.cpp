// Descriptors of a list of torch tensors without one DLPack capsule per tensor: the per-tensor
// loop of the reference's ExtractDlpackTensor + ExtractTensorMetaFromDlm
// (axon/python/src/dlpack_helpers.cpp:136-156, 696-724) for the case where every producer is a
// plain torch.Tensor.  The fields come from torch's own converter (at::toDLPackNonOwning, the
// code Tensor.__dlpack__ ends in, minus the allocation of a managed tensor and a capsule), so
// dtype codes, device types and the strides of size-1 dimensions are what the capsule would
// carry.
//
// describe(sequence, device_id) -> (descs: bytearray, dims: bytearray, owners: list) | None
//   descs   n * sizeof(axr_tensor_t); shape/strides point into `dims`
//   dims    the copied shapes and strides (int64)
//   owners  the tensors themselves (they own the memory the descriptors name)
// None when any element is not exactly a torch.Tensor, requires grad, carries the conjugate or
// negative bit, is not strided, lives on another GPU than `device_id`, or is refused by the
// converter: the caller then takes the capsule route, which gives Tensor.__dlpack__'s answer.
//
// plan_create(sequence, device_id, align, function) -> (plan, owners) | None
// plan_bind(header: bytes, sequence, device_id, function) -> (plan, owners) | None
//   axr_plan_create_from / axr_plan_bind_from, whose address is `function`, for a list or a tuple: the
//   descriptors go to the planner a few at a time and nothing is kept of them.  None where describe()
//   gives None and where the planner refuses: the caller then takes the steps one by one and gets
//   the answer, or the error, that those give.  plan_bind's plan reads `header` in place.
//
// Built against the torch that is installed; importable only after `import torch`.
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/DLConvertor.h>
#include <c10/core/impl/COW.h>

#include <Python.h>

#include <cstdint>
#include <cstring>

#include "axon_rocm.h"
#include "axr_source.h"

static_assert(sizeof(axr_tensor_t) == sizeof(DLTensor), "axr_tensor_t mirrors DLTensor");
static_assert(offsetof(axr_tensor_t, shape) == offsetof(DLTensor, shape), "axr_tensor_t mirrors DLTensor");
static_assert(offsetof(axr_tensor_t, byte_offset) == offsetof(DLTensor, byte_offset), "axr_tensor_t mirrors DLTensor");

namespace {

// The tensor behind an object when the capsule route would export it unchanged, else nullptr.
struct Exportable {
  long device_id;
  uint64_t plain_keys = 0;   // the dispatch keys of a tensor that passed: all but the last two questions ask these

  const at::Tensor* operator()(PyObject* obj) {
    if (!THPVariable_CheckExact(obj)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(obj);
    if (!t.defined()) return nullptr;
    const uint64_t keys = t.key_set().raw_repr();
    if (keys != plain_keys || keys == 0) {
      if (t.layout() != c10::kStrided || t.is_nested() || t.is_quantized() || t.is_conj() || t.is_neg() ||
          t._is_zerotensor()) {
        return nullptr;
      }
      plain_keys = keys;
    }
    if (!t.has_storage() || t.requires_grad()) return nullptr;
    const c10::Device dev = t.device();
    if (dev.is_cuda()) {
      if (dev.index() != device_id) return nullptr;
    } else if (!dev.is_cpu()) {
      return nullptr;
    }
    return &t;
  }
};

// A tensor object is three to five cache lines in two places, the tensor being reached through its
// Python object; sequences of many thousands are fetched this many tensors ahead.
constexpr Py_ssize_t kAheadObject = 24, kAheadTensor = 12;
void prefetch(PyObject* const* items, Py_ssize_t i, Py_ssize_t n) {
  if (i + kAheadObject < n) __builtin_prefetch(items[i + kAheadObject], 1);   // its reference count is written
  if (i + kAheadTensor < n && THPVariable_CheckExact(items[i + kAheadTensor])) {
    const char* impl = reinterpret_cast<const char*>(THPVariable_Unpack(items[i + kAheadTensor]).unsafeGetTensorImpl());
    for (size_t at = 0; at < sizeof(at::TensorImpl); at += 64) __builtin_prefetch(impl + at);
  }
}

// The converter's answers on one GPU's tensors: the device is the same for all of them and the type a
// function of the scalar type, so that it is asked once for each; the other fields are read directly.
// Fresh plan of 4096 GPU tensors 80 us when the converter was asked for each, 65,536 tensors 2640; now
// 60 and 1090, records and header included.
struct Fields {
  bool device_known = false;
  DLDevice device;
  struct Type {
    bool known;
    DLDataType type;
    int64_t bytes;
  } types[64] = {};
  // the storage that the latest tensor lay in; null where its tensors are the converter's business (memory
  // that is shared until it is written)
  const c10::StorageImpl* storage = nullptr;
  const char* base = nullptr;
  bool plain_storage = false;

  void read(const at::Tensor& t, DLTensor* out) {   // may throw what the converter throws
    const at::TensorImpl* impl = t.unsafeGetTensorImpl();
    const auto type = static_cast<size_t>(t.scalar_type());
    const c10::StorageImpl* in = impl->unsafe_storage().unsafeGetStorageImpl();
    if (in != storage) {
      storage = in;
      base = static_cast<const char*>(in->data());
      plain_storage = in->device_type() == c10::kCUDA && !c10::impl::cow::is_cow_data_ptr(in->data_ptr());
    }
    if (!plain_storage || type >= 64 || !types[type].known || !device_known) {
      at::toDLPackNonOwning(t, out);   // shape/strides point at the tensor's own arrays
      if (plain_storage && type < 64) {
        types[type].known = device_known = true;
        types[type].type = out->dtype;
        types[type].bytes = static_cast<int64_t>(t.element_size());
        device = out->device;
      }
      return;
    }
    const auto sizes = impl->sizes();
    out->data = impl->numel() == 0 ? nullptr : const_cast<char*>(base) + impl->storage_offset() * types[type].bytes;
    out->device = device;
    out->ndim = static_cast<int32_t>(sizes.size());
    out->dtype = types[type].type;
    out->shape = const_cast<int64_t*>(sizes.data());
    out->strides = const_cast<int64_t*>(impl->strides().data());
    out->byte_offset = 0;
  }
};

PyObject* describe(PyObject*, PyObject* args) {
  PyObject* arg = nullptr;
  long device_id = -1;
  if (!PyArg_ParseTuple(args, "Ol", &arg, &device_id)) return nullptr;
  PyObject* seq = PySequence_Fast(arg, "describe() needs a sequence of tensors");
  if (!seq) return nullptr;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
  PyObject** items = PySequence_Fast_ITEMS(seq);
  PyObject* descs = nullptr;
  PyObject* dims = nullptr;
  PyObject* owners = nullptr;
  PyObject* result = nullptr;
  bool refused = false;
  Exportable exportable{device_id};

  Py_ssize_t total_dims = 0;
  for (Py_ssize_t i = 0; i < n && !refused; ++i) {
    prefetch(items, i, n);
    const at::Tensor* t = exportable(items[i]);
    if (!t) {
      refused = true;
    } else {
      total_dims += 2 * t->dim();
    }
  }
  if (!refused) {
    descs = PyByteArray_FromStringAndSize(nullptr, n * static_cast<Py_ssize_t>(sizeof(axr_tensor_t)));
    dims = PyByteArray_FromStringAndSize(nullptr, total_dims * static_cast<Py_ssize_t>(sizeof(int64_t)));
    owners = PyList_New(n);
  }
  if (!refused && descs && dims && owners) {
    auto* out = reinterpret_cast<DLTensor*>(PyByteArray_AS_STRING(descs));
    auto* d = reinterpret_cast<int64_t*>(PyByteArray_AS_STRING(dims));
    Fields fields;
    try {
      for (Py_ssize_t i = 0; i < n; ++i) {
        prefetch(items, i, n);
        const at::Tensor& t = THPVariable_Unpack(items[i]);
        fields.read(t, &out[i]);
        const int nd = out[i].ndim;
        if (nd > 0) {
          std::memcpy(d, out[i].shape, sizeof(int64_t) * nd);
          out[i].shape = d;
          d += nd;
          if (out[i].strides) {
            std::memcpy(d, out[i].strides, sizeof(int64_t) * nd);
            out[i].strides = d;
            d += nd;
          }
        } else {
          out[i].shape = nullptr;
          out[i].strides = nullptr;
        }
        Py_INCREF(items[i]);
        PyList_SET_ITEM(owners, i, items[i]);
      }
      result = PyTuple_Pack(3, descs, dims, owners);
    } catch (...) {   // a dtype or device the converter does not export
      refused = true;
    }
  }
  if (!result && !PyErr_Occurred()) {
    result = Py_None;
    Py_INCREF(result);
  }
  Py_XDECREF(descs);
  Py_XDECREF(dims);
  Py_XDECREF(owners);   // a partly filled list releases what it holds
  Py_DECREF(seq);
  return result;
}

// The tensors of a list or tuple as a source for the planner, which keeps a reference to each
// in `owners`.  The interpreter's lock is held from the first tensor to the last.
struct Sequence : axr_tensor_source {
  PyObject** items;
  PyObject* owners;
  Exportable exportable;
  Fields fields;

  static int lot(axr_tensor_source* self, size_t first, size_t n, axr_tensor_t* out) {
    auto* s = static_cast<Sequence*>(self);
    try {
      for (size_t i = first; i < first + n; ++i) {
        prefetch(s->items, static_cast<Py_ssize_t>(i), static_cast<Py_ssize_t>(s->count));
        const at::Tensor* t = s->exportable(s->items[i]);
        if (!t) return 1;
        auto* d = reinterpret_cast<DLTensor*>(&out[i - first]);
        s->fields.read(*t, d);
        if (d->ndim == 0) d->shape = d->strides = nullptr;
        Py_INCREF(s->items[i]);
        PyList_SET_ITEM(s->owners, static_cast<Py_ssize_t>(i), s->items[i]);
      }
    } catch (...) {   // a dtype or device the converter does not export
      return 1;
    }
    return 0;
  }
};

template <typename Make>
PyObject* plan_from(PyObject* seq, long device_id, Make&& make) {
  if (!PyList_CheckExact(seq) && !PyTuple_CheckExact(seq)) Py_RETURN_NONE;
  Sequence source;
  source.count = static_cast<size_t>(PySequence_Fast_GET_SIZE(seq));
  source.describe = Sequence::lot;
  source.items = PySequence_Fast_ITEMS(seq);
  source.exportable.device_id = device_id;
  source.owners = PyList_New(static_cast<Py_ssize_t>(source.count));
  if (!source.owners) return nullptr;
  axr_plan_t* plan = nullptr;
  if (make(&source, &plan) != AXR_OK) {
    Py_DECREF(source.owners);   // a partly filled list releases what it holds
    Py_RETURN_NONE;
  }
  return Py_BuildValue("KN", static_cast<unsigned long long>(reinterpret_cast<uintptr_t>(plan)), source.owners);
}

PyObject* plan_create(PyObject*, PyObject* args) {
  PyObject* seq = nullptr;
  long device_id = -1;
  unsigned int align = 0;
  unsigned long long function = 0;
  if (!PyArg_ParseTuple(args, "OlIK", &seq, &device_id, &align, &function)) return nullptr;
  auto* make = reinterpret_cast<axr_plan_create_from_fn*>(static_cast<uintptr_t>(function));
  return plan_from(seq, device_id,
                   [&](axr_tensor_source* source, axr_plan_t** plan) { return make(source, align, plan); });
}

PyObject* plan_bind(PyObject*, PyObject* args) {
  PyObject *header = nullptr, *seq = nullptr;
  long device_id = -1;
  unsigned long long function = 0;
  if (!PyArg_ParseTuple(args, "SOlK", &header, &seq, &device_id, &function)) return nullptr;
  auto* make = reinterpret_cast<axr_plan_bind_from_fn*>(static_cast<uintptr_t>(function));
  return plan_from(seq, device_id, [&](axr_tensor_source* source, axr_plan_t** plan) {
    return make(PyBytes_AS_STRING(header), static_cast<size_t>(PyBytes_GET_SIZE(header)), source, plan);
  });
}

PyMethodDef methods[] = {
    {"plan_create", plan_create, METH_VARARGS,
     "plan_create(sequence, device_id, align, function) -> (plan, owners list) or None"},
    {"plan_bind", plan_bind, METH_VARARGS,
     "plan_bind(header, sequence, device_id, function) -> (plan, owners list) or None"},
    {"describe", describe, METH_VARARGS,
     "describe(sequence, device_id) -> (descs bytearray, dims bytearray, owners list) or None"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_axr_torch", "Descriptors of torch tensors for tensor bundles.",
                      -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__axr_torch(void) {
  PyObject* m = PyModule_Create(&module);
  if (m) PyModule_AddIntConstant(m, "TENSOR_BYTES", static_cast<long>(sizeof(axr_tensor_t)));
  return m;
}

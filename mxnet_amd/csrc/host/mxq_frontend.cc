// mxnet_amd._frontend: the imperative call path of the Python package in native code.
//
// What an operator call costs a small program is not its kernel but the host work in front of
// it: building the node, inferring shapes and types, allocating outputs and temp space,
// unpacking tensors.  Written in Python over ctypes that was 35 us a call (a 128 x 1024
// quantize kernel runs 3.5 us).  Here one call
//   - finds its node by operator name and attribute text in a table of parsed nodes,
//   - finds what the node's outputs look like for these input shapes and types in the node's
//     own table (the inference functions run once per combination),
//   - allocates the outputs and the temp space through torch's caching allocator,
//   - runs mxq_node_forward on torch's current stream with the interpreter lock released.
// Nothing that depends on a tensor's contents is kept.
//
// Both tables are bounded and guarded by the interpreter lock.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdlib>
#include <cstring>
#include <memory>
#include <string>
#include <unordered_map>
#include <vector>

#include "../../../include/mxq.h"
#include "../../../include/mxq_ops.h"
#include "mxq_plan.h"

namespace {

PyObject* g_op_error = nullptr;   // operator.MXNetError
PyObject* g_lib_error = nullptr;  // _lib.MXQError

constexpr int kMaxInputs = 64;
constexpr int kMaxOutputs = 8;
constexpr size_t kMaxSignatures = 32;  // per node: input shape combinations remembered
constexpr size_t kMaxNodes = 4096;     // nodes of imperative calls remembered

// mshadow::TypeFlag <-> torch dtype; -1: no counterpart
int flag_of(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return 0;
    case at::kDouble: return 1;
    case at::kHalf: return 2;
    case at::kByte: return 3;
    case at::kInt: return 4;
    case at::kChar: return 5;
    case at::kLong: return 6;
    case at::kBool: return 7;
    case at::kBFloat16: return 12;
    default: return -1;
  }
}

bool dtype_of(int flag, at::ScalarType* t) {
  switch (flag) {
    case 0: *t = at::kFloat; return true;
    case 1: *t = at::kDouble; return true;
    case 2: *t = at::kHalf; return true;
    case 3: *t = at::kByte; return true;
    case 4: *t = at::kInt; return true;
    case 5: *t = at::kChar; return true;
    case 6: *t = at::kLong; return true;
    case 7: *t = at::kBool; return true;
    case 12: *t = at::kBFloat16; return true;
    default: return false;
  }
}

void* current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

// Memory from torch's caching allocator of the current device and stream, as a storage of its
// own.  at::empty ends there as well, by way of its dispatcher (0.9 us a tensor; 0.4 us this way);
// the allocator is the one that a tensor of at::empty names.
c10::Storage storage_on(int64_t bytes, const at::Device& dev) {
  static c10::Allocator* const allocator =
      at::empty({1}, at::TensorOptions().dtype(at::kByte).device(dev)).storage().allocator();
  if (dev.has_index() && dev.index() != c10::hip::current_device()) {
    const c10::DeviceGuard guard(dev);
    return c10::Storage(c10::Storage::use_byte_size_t(), bytes, allocator->allocate(bytes),
                        allocator, true);
  }
  return c10::Storage(c10::Storage::use_byte_size_t(), bytes, allocator->allocate(bytes),
                      allocator, true);
}

at::Tensor tensor_on(c10::Storage storage, int64_t offset, at::IntArrayRef shape,
                     at::ScalarType type) {
  at::Tensor t = at::detail::make_tensor<c10::TensorImpl>(
      std::move(storage), c10::DispatchKeySet(c10::DispatchKey::CUDA),
      c10::scalarTypeToTypeMeta(type));
  if (offset != 0) t.unsafeGetTensorImpl()->set_storage_offset(offset);
  t.unsafeGetTensorImpl()->set_sizes_contiguous(shape);
  return t;
}

at::Tensor empty_on(at::IntArrayRef shape, at::ScalarType type, const at::Device& dev) {
  int64_t count = 1;
  for (const int64_t d : shape) count *= d;
  return tensor_on(storage_on(count * static_cast<int64_t>(c10::elementSize(type)), dev), 0, shape,
                   type);
}

// The range scalars come in pairs: two one-element tensors over one 8-byte allocation.
void empty_scalar_pair(const at::Device& dev, at::Tensor* lo, at::Tensor* hi) {
  const int64_t one = 1;
  const at::IntArrayRef shape(&one, 1);
  c10::Storage pair = storage_on(2 * sizeof(float), dev);
  *lo = tensor_on(pair, 0, shape, at::kFloat);
  *hi = tensor_on(std::move(pair), 1, shape, at::kFloat);
}

// ---- nodes -----------------------------------------------------------------------------------

struct OutMeta {
  int ndim;
  int64_t shape[MXQ_MAX_NDIM];
  int flag;
  at::ScalarType type;
};

struct Signature {
  std::vector<int64_t> key;  // per input: type flag, ndim, extents
  std::vector<OutMeta> outs;
  size_t temp_bytes;
};

struct OpNode {
  void* handle = nullptr;
  bool owned = false;
  std::string op;
  int num_inputs = 0;
  std::vector<std::shared_ptr<const Signature>> known;
  size_t next = 0;  // the entry that the next new signature replaces once the table is full
  ~OpNode() {
    if (owned && handle != nullptr) mxq_node_free(handle);
  }
};

bool op_failed(int rc) {
  if (rc == 0) return false;
  PyErr_SetString(g_op_error, mxq_ops_last_error());
  return true;
}

bool fill_node(OpNode* n) { return !op_failed(mxq_node_num_inputs(n->handle, &n->num_inputs)); }

void wrong_count(const OpNode& n, Py_ssize_t given) {
  const char* names = nullptr;
  mxq_node_input_names(n.handle, &names);
  std::string list = "[";
  for (const char* p = names; p != nullptr && *p != 0;) {
    const char* end = std::strchr(p, ',');
    const std::string one = end != nullptr ? std::string(p, end) : std::string(p);
    list += (list.size() > 1 ? ", '" : "'") + one + "'";
    p = end != nullptr ? end + 1 : nullptr;
  }
  list += "]";
  PyErr_Format(g_op_error, "%s expects %d inputs %s, got %zd", n.op.c_str(), n.num_inputs,
               list.c_str(), given);
}

// shapes and types of the outputs for these inputs, from the node's table or inferred
std::shared_ptr<const Signature> signature_of(OpNode* n, const mxq_blob* in, int num_in) {
  int64_t key[kMaxInputs * (MXQ_MAX_NDIM + 2)];
  size_t len = 0;
  for (int i = 0; i < num_in; ++i) {
    key[len++] = in[i].dtype;
    key[len++] = in[i].ndim;
    for (int d = 0; d < in[i].ndim; ++d) key[len++] = in[i].shape[d];
  }
  for (const auto& s : n->known)
    if (s->key.size() == len && std::memcmp(s->key.data(), key, len * sizeof(int64_t)) == 0)
      return s;
  mxq_blob out[kMaxOutputs];
  int count = 0;
  size_t temp = 0;
  if (op_failed(mxq_node_describe(n->handle, num_in, in, kMaxOutputs, out, &count, &temp)))
    return nullptr;
  auto s = std::make_shared<Signature>();
  s->key.assign(key, key + len);
  s->temp_bytes = temp;
  for (int i = 0; i < count; ++i) {
    OutMeta m;
    m.ndim = out[i].ndim;
    m.flag = out[i].dtype;
    if (m.ndim < 0 || !dtype_of(m.flag, &m.type)) {
      PyErr_Format(PyExc_TypeError, "%s: the shape or type of output %d stays unknown",
                   n->op.c_str(), i);
      return nullptr;
    }
    std::memcpy(m.shape, out[i].shape, sizeof(m.shape));
    s->outs.push_back(m);
  }
  if (n->known.size() < kMaxSignatures) {
    n->known.push_back(s);
  } else {
    n->known[n->next] = s;
    n->next = (n->next + 1) % kMaxSignatures;
  }
  return s;
}

bool is_range(const OutMeta& m) { return m.ndim == 1 && m.shape[0] == 1 && m.type == at::kFloat; }

// One forward call; `args` may hold None (left out, as an absent optional input).
PyObject* run_node(OpNode* n, PyObject* const* args, Py_ssize_t nargs) {
  mxq_blob in[kMaxInputs], out[kMaxOutputs];
  const at::Tensor* first = nullptr;
  int num_in = 0;
  for (Py_ssize_t i = 0; i < nargs; ++i) num_in += args[i] != Py_None;
  if (num_in != n->num_inputs || num_in > kMaxInputs) {
    wrong_count(*n, num_in);
    return nullptr;
  }
  num_in = 0;
  for (Py_ssize_t i = 0; i < nargs; ++i) {
    if (args[i] == Py_None) continue;
    if (!THPVariable_Check(args[i])) {
      PyErr_Format(PyExc_AttributeError, "'%s' object has no attribute 'is_cuda'",
                   Py_TYPE(args[i])->tp_name);
      return nullptr;
    }
    const at::Tensor& t = THPVariable_Unpack(args[i]);
    if (!t.is_cuda() || !t.is_contiguous()) {
      PyErr_SetString(g_op_error, "inputs must be contiguous device tensors");
      return nullptr;
    }
    if (first == nullptr) first = &t;
    mxq_blob& b = in[num_in++];
    b.ndim = static_cast<int>(t.dim());
    if (b.ndim > MXQ_MAX_NDIM) {
      PyErr_SetString(PyExc_IndexError, "too many dimensions");
      return nullptr;
    }
    b.dtype = flag_of(t.scalar_type());
    if (b.dtype < 0) {
      PyObject* dtype = PyObject_GetAttrString(args[i], "dtype");
      if (dtype != nullptr) PyErr_SetObject(PyExc_KeyError, dtype);
      Py_XDECREF(dtype);
      return nullptr;
    }
    for (int d = 0; d < b.ndim; ++d) b.shape[d] = t.size(d);
    b.data = t.data_ptr();
  }
  if (first == nullptr) {
    wrong_count(*n, 0);
    return nullptr;
  }
  const auto sig = signature_of(n, in, num_in);
  if (sig == nullptr) return nullptr;
  const at::Device dev = first->device();
  const int num_out = static_cast<int>(sig->outs.size());
  at::Tensor outs[kMaxOutputs], temp;
  for (int i = 0; i < num_out; ++i) {
    const OutMeta& m = sig->outs[i];
    if (!outs[i].defined()) {
      if (is_range(m) && i + 1 < num_out && is_range(sig->outs[i + 1]))
        empty_scalar_pair(dev, &outs[i], &outs[i + 1]);
      else
        outs[i] = empty_on(at::IntArrayRef(m.shape, m.ndim), m.type, dev);
    }
    out[i].data = outs[i].data_ptr();
    out[i].ndim = m.ndim;
    std::memcpy(out[i].shape, m.shape, sizeof(m.shape));
    out[i].dtype = m.flag;
  }
  if (sig->temp_bytes != 0) {
    const int64_t bytes = static_cast<int64_t>(sig->temp_bytes);
    temp = empty_on(at::IntArrayRef(&bytes, 1), at::kByte, dev);
  }
  void* stream = current_stream();
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = mxq_node_forward(n->handle, stream, dev.has_index() ? dev.index() : 0, num_in, in, num_out,
                        out, temp.defined() ? temp.data_ptr() : nullptr, sig->temp_bytes);
  Py_END_ALLOW_THREADS;
  if (op_failed(rc)) return nullptr;
  if (num_out == 1) return THPVariable_Wrap(std::move(outs[0]));
  PyObject* result = PyTuple_New(num_out);
  if (result == nullptr) return nullptr;
  for (int i = 0; i < num_out; ++i) {
    PyObject* o = THPVariable_Wrap(std::move(outs[i]));
    if (o == nullptr) {
      Py_DECREF(result);
      return nullptr;
    }
    PyTuple_SET_ITEM(result, i, o);
  }
  return result;
}

// ---- Python value -> the string MXNet's frontend puts in the node dict -------------------------

bool append_text(PyObject* text, std::string* out) {
  if (text == nullptr) return false;
  Py_ssize_t len = 0;
  const char* s = PyUnicode_AsUTF8AndSize(text, &len);
  if (s != nullptr) out->append(s, len);
  Py_DECREF(text);
  return s != nullptr;
}

bool append_attr(PyObject* v, std::string* out) {
  if (v == Py_None) {
    *out += "None";
    return true;
  }
  if (PyBool_Check(v)) {
    *out += v == Py_True ? "True" : "False";
    return true;
  }
  if (PyTuple_Check(v) || PyList_Check(v)) {
    PyObject* seq = PySequence_Fast(v, "");
    if (seq == nullptr) return false;
    const Py_ssize_t len = PySequence_Fast_GET_SIZE(seq);
    *out += "(";
    for (Py_ssize_t i = 0; i < len; ++i) {
      if (i != 0) *out += ", ";
      PyObject* x = PyNumber_Long(PySequence_Fast_GET_ITEM(seq, i));
      const bool ok = x != nullptr && append_text(PyObject_Str(x), out);
      Py_XDECREF(x);
      if (!ok) {
        Py_DECREF(seq);
        return false;
      }
    }
    *out += len == 1 ? ",)" : ")";
    Py_DECREF(seq);
    return true;
  }
  if (PyUnicode_CheckExact(v)) {
    Py_INCREF(v);
    return append_text(v, out);
  }
  return append_text(PyFloat_Check(v) ? PyObject_Repr(v) : PyObject_Str(v), out);
}

// ---- module functions ----------------------------------------------------------------------------

std::unordered_map<std::string, std::shared_ptr<OpNode>>& node_table() {
  static auto* t = new std::unordered_map<std::string, std::shared_ptr<OpNode>>();
  return *t;
}

// invoke(op, *tensors, **attrs)
PyObject* py_invoke(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
  HANDLE_TH_ERRORS
  if (nargs < 1 || !PyUnicode_Check(args[0])) {
    PyErr_SetString(PyExc_TypeError, "invoke(op, *tensors, **attrs)");
    return nullptr;
  }
  std::string key;
  std::vector<size_t> cut;  // where each attribute's name and value end
  key.reserve(192);
  cut.reserve(16);
  Py_ssize_t len = 0;
  const char* op = PyUnicode_AsUTF8AndSize(args[0], &len);
  if (op == nullptr) return nullptr;
  key.assign(op, len);
  key.push_back('\0');
  const Py_ssize_t nkw = kwnames != nullptr ? PyTuple_GET_SIZE(kwnames) : 0;
  for (Py_ssize_t i = 0; i < nkw; ++i) {
    PyObject* v = args[nargs + i];
    if (v == Py_None) continue;  // an attribute left at its default
    Py_ssize_t klen = 0;
    const char* k = PyUnicode_AsUTF8AndSize(PyTuple_GET_ITEM(kwnames, i), &klen);
    if (k == nullptr) return nullptr;
    key.append(k, klen);
    cut.push_back(key.size());
    key.push_back('\0');
    if (!append_attr(v, &key)) return nullptr;
    cut.push_back(key.size());
    key.push_back('\0');
  }
  auto& table = node_table();
  auto it = table.find(key);
  std::shared_ptr<OpNode> node;
  if (it != table.end()) {
    node = it->second;
  } else {
    std::vector<const char*> keys, values;
    size_t at = static_cast<size_t>(len) + 1;
    for (size_t i = 0; i + 1 < cut.size(); i += 2) {
      keys.push_back(key.data() + at);
      values.push_back(key.data() + cut[i] + 1);
      at = cut[i + 1] + 1;
    }
    node = std::make_shared<OpNode>();
    node->op.assign(op, len);
    node->owned = true;
    if (op_failed(mxq_node_create(node->op.c_str(), "", static_cast<int>(keys.size()),
                                  keys.data(), values.data(), &node->handle)) ||
        !fill_node(node.get()))
      return nullptr;
    if (table.size() >= kMaxNodes) table.clear();  // calls in flight hold their node themselves
    table.emplace(key, node);
  }
  return run_node(node.get(), args + 1, nargs - 1);
  END_HANDLE_TH_ERRORS
}

constexpr const char* kNodeCapsule = "mxnet_amd.node";

void free_node(PyObject* capsule) {
  delete static_cast<OpNode*>(PyCapsule_GetPointer(capsule, kNodeCapsule));
}

// node(handle, op): the call table of a node that the caller owns and keeps alive
PyObject* py_node(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  unsigned long long handle;
  const char* op;
  if (!PyArg_ParseTuple(args, "Ks", &handle, &op)) return nullptr;
  std::unique_ptr<OpNode> n(new OpNode());
  n->handle = reinterpret_cast<void*>(static_cast<uintptr_t>(handle));
  n->op = op;
  if (!fill_node(n.get())) return nullptr;
  PyObject* capsule = PyCapsule_New(n.get(), kNodeCapsule, free_node);
  if (capsule != nullptr) n.release();
  return capsule;
  END_HANDLE_TH_ERRORS
}

// forward(node, *tensors)
PyObject* py_forward(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs < 1) {
    PyErr_SetString(PyExc_TypeError, "forward(node, *tensors)");
    return nullptr;
  }
  OpNode* n = static_cast<OpNode*>(PyCapsule_GetPointer(args[0], kNodeCapsule));
  if (n == nullptr) return nullptr;
  return run_node(n, args + 1, nargs - 1);
  END_HANDLE_TH_ERRORS
}

// ---- the C entry points that capi.py wraps -----------------------------------------------------

bool lib_failed(int rc) {
  if (rc == 0) return false;
  PyErr_SetString(g_lib_error, mxq_last_error());
  return true;
}

// A tensor argument of a C entry point: contiguous, on the device; None where `optional`.
bool tensor_arg(PyObject* o, at::Tensor* t, bool optional = false) {
  if (o == Py_None && optional) return true;
  if (!THPVariable_Check(o)) {
    PyErr_Format(PyExc_TypeError, "expected a tensor, got '%s'", Py_TYPE(o)->tp_name);
    return false;
  }
  *t = THPVariable_Unpack(o);
  if (!t->is_cuda() || !t->is_contiguous()) {
    PyErr_SetString(PyExc_AssertionError, "need a contiguous device tensor");
    return false;
  }
  return true;
}

template <typename T>
T* ptr(const at::Tensor& t) {
  return t.defined() ? static_cast<T*>(t.data_ptr()) : nullptr;
}

bool float_arg(PyObject* o, float* v) {
  PyObject* f = PyNumber_Float(o);
  if (f == nullptr) return false;
  *v = static_cast<float>(PyFloat_AS_DOUBLE(f));
  Py_DECREF(f);
  return true;
}

// calibration range: None or a pair; `given` says which
bool range_arg(PyObject* o, bool* given, float* lo, float* hi) {
  *given = o != Py_None;
  *lo = *hi = 0.0f;
  if (!*given) return true;
  for (int i = 0; i < 2; ++i) {
    PyObject* x = PySequence_GetItem(o, i);
    const bool ok = x != nullptr && float_arg(x, i == 0 ? lo : hi);
    Py_XDECREF(x);
    if (!ok) return false;
  }
  return true;
}

bool dims_are(const at::Tensor& t, int ndim) {
  if (t.dim() == ndim) return true;
  PyErr_Format(PyExc_ValueError, "expected a tensor of %d dimensions, got %d", ndim,
               static_cast<int>(t.dim()));
  return false;
}

bool same_extent(int64_t a, int64_t b) {
  if (a == b) return true;
  PyErr_Format(PyExc_AssertionError, "operand extents differ: %lld and %lld",
               static_cast<long long>(a), static_cast<long long>(b));
  return false;
}

// dict(out32, omin, omax, out8, rmin, rmax), None for what was not asked for
PyObject* result_dict(const at::Tensor& omin, const at::Tensor& omax, const at::Tensor& out32,
                      const at::Tensor& out8, const at::Tensor& rmin, const at::Tensor& rmax) {
  static const char* const names[] = {"omin", "omax", "out32", "out8", "rmin", "rmax"};
  static PyObject* keys[6] = {};
  const at::Tensor* const values[] = {&omin, &omax, &out32, &out8, &rmin, &rmax};
  PyObject* d = PyDict_New();
  if (d == nullptr) return nullptr;
  for (int i = 0; i < 6; ++i) {
    if (keys[i] == nullptr) keys[i] = PyUnicode_InternFromString(names[i]);
    PyObject* v = nullptr;
    if (values[i]->defined()) {
      v = THPVariable_Wrap(*values[i]);
    } else {
      v = Py_None;
      Py_INCREF(v);
    }
    const bool ok = v != nullptr && keys[i] != nullptr && PyDict_SetItem(d, keys[i], v) == 0;
    Py_XDECREF(v);
    if (!ok) {
      Py_DECREF(d);
      return nullptr;
    }
  }
  return d;
}

at::Tensor workspace(size_t bytes, const at::Device& dev) {
  if (bytes == 0) return at::Tensor();
  const int64_t n = static_cast<int64_t>(bytes);
  return empty_on(at::IntArrayRef(&n, 1), at::kByte, dev);
}

// operands shared by the FC and the convolution: data, weight, bias and the six ranges
struct Operands {
  at::Tensor t[9];
  bool parse(PyObject* const* args) {
    for (int i = 0; i < 9; ++i)
      if (!tensor_arg(args[i], &t[i], i == 2 || i >= 7)) return false;
    return true;
  }
  const float* range(int i) const { return ptr<const float>(t[3 + i]); }
};

// quantized_fc(data, weight, bias, six ranges, want_int32, calib, relu)
PyObject* py_quantized_fc(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Operands a;
  bool fused;
  float lo, hi;
  if (nargs != 12) {
    PyErr_SetString(PyExc_TypeError, "quantized_fc takes 12 arguments");
    return nullptr;
  }
  if (!a.parse(args) || !range_arg(args[10], &fused, &lo, &hi)) return nullptr;
  const int want32 = PyObject_IsTrue(args[9]), relu = PyObject_IsTrue(args[11]);
  if (want32 < 0 || relu < 0 || !dims_are(a.t[0], 2) || !dims_are(a.t[1], 2)) return nullptr;
  const int M = a.t[0].size(0), K = a.t[0].size(1), N = a.t[1].size(0);
  if (!same_extent(K, a.t[1].size(1))) return nullptr;
  const at::Device dev = a.t[0].device();
  at::Tensor omin, omax, out32, out8, rmin, rmax;
  const int64_t shape[] = {M, N};
  empty_scalar_pair(dev, &omin, &omax);
  if (want32) out32 = empty_on(at::IntArrayRef(shape, 2), at::kInt, dev);
  if (fused) {
    out8 = empty_on(at::IntArrayRef(shape, 2), at::kChar, dev);
    empty_scalar_pair(dev, &rmin, &rmax);
  }
  const size_t bytes = mxq_quantized_fc_workspace(M, N, K, !want32);
  const at::Tensor ws = workspace(bytes, dev);
  void* stream = current_stream();
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = mxq_quantized_fc(stream, ptr<int8_t>(a.t[0]), ptr<int8_t>(a.t[1]), ptr<int8_t>(a.t[2]), M,
                        N, K, a.range(0), a.range(1), a.range(2), a.range(3), a.range(4),
                        a.range(5), ptr<int32_t>(out32), ptr<float>(omin), ptr<float>(omax),
                        ptr<int8_t>(out8), ptr<float>(rmin), ptr<float>(rmax), relu, lo, hi,
                        ptr<void>(ws), bytes);
  Py_END_ALLOW_THREADS;
  if (lib_failed(rc)) return nullptr;
  return result_dict(omin, omax, out32, out8, rmin, rmax);
  END_HANDLE_TH_ERRORS
}

// quantized_conv_nhwc(data, weight, bias, six ranges, stride, pad, dilate, want_int32, calib, relu)
PyObject* py_quantized_conv_nhwc(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  Operands a;
  bool fused;
  float lo, hi;
  if (nargs != 15) {
    PyErr_SetString(PyExc_TypeError, "quantized_conv_nhwc takes 15 arguments");
    return nullptr;
  }
  if (!a.parse(args) || !range_arg(args[13], &fused, &lo, &hi)) return nullptr;
  int step[6];  // stride, pad, dilate as height, width
  for (int i = 0; i < 6; ++i) {
    PyObject* x = PySequence_GetItem(args[9 + i / 2], i % 2);
    if (x == nullptr) return nullptr;
    step[i] = static_cast<int>(PyLong_AsLong(x));
    Py_DECREF(x);
    if (PyErr_Occurred()) return nullptr;
  }
  const int want32 = PyObject_IsTrue(args[12]), relu = PyObject_IsTrue(args[14]);
  if (want32 < 0 || relu < 0 || !dims_are(a.t[0], 4) || !dims_are(a.t[1], 4)) return nullptr;
  const int N = a.t[0].size(0), H = a.t[0].size(1), W = a.t[0].size(2), C = a.t[0].size(3);
  const int O = a.t[1].size(0), KH = a.t[1].size(1), KW = a.t[1].size(2);
  if (!same_extent(C, a.t[1].size(3))) return nullptr;
  const int sh = step[0], sw = step[1], ph = step[2], pw = step[3], dh = step[4], dw = step[5];
  if (sh == 0 || sw == 0) {
    PyErr_SetString(PyExc_ZeroDivisionError, "integer division or modulo by zero");
    return nullptr;
  }
  auto floor_div = [](int x, int y) { return x / y - ((x % y != 0) && ((x < 0) != (y < 0))); };
  const int OH = floor_div(H + 2 * ph - (dh * (KH - 1) + 1), sh) + 1;
  const int OW = floor_div(W + 2 * pw - (dw * (KW - 1) + 1), sw) + 1;
  const at::Device dev = a.t[0].device();
  at::Tensor omin, omax, out32, out8, rmin, rmax;
  const int64_t shape[] = {N, OH, OW, O};
  empty_scalar_pair(dev, &omin, &omax);
  if (want32) out32 = empty_on(at::IntArrayRef(shape, 4), at::kInt, dev);
  if (fused) {
    out8 = empty_on(at::IntArrayRef(shape, 4), at::kChar, dev);
    empty_scalar_pair(dev, &rmin, &rmax);
  }
  const size_t bytes =
      mxq_quantized_conv_workspace(N, H, W, C, O, KH, KW, sh, sw, ph, pw, dh, dw, !want32);
  const at::Tensor ws = workspace(bytes, dev);
  void* stream = current_stream();
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = mxq_quantized_conv_nhwc(
      stream, ptr<int8_t>(a.t[0]), ptr<int8_t>(a.t[1]), ptr<int8_t>(a.t[2]), N, H, W, C, O, KH,
      KW, sh, sw, ph, pw, dh, dw, a.range(0), a.range(1), a.range(2), a.range(3), a.range(4),
      a.range(5), ptr<int32_t>(out32), ptr<float>(omin), ptr<float>(omax), ptr<int8_t>(out8),
      ptr<float>(rmin), ptr<float>(rmax), relu, lo, hi, ptr<void>(ws), bytes);
  Py_END_ALLOW_THREADS;
  if (lib_failed(rc)) return nullptr;
  return result_dict(omin, omax, out32, out8, rmin, rmax);
  END_HANDLE_TH_ERRORS
}

// ---- plans (mxq_plan.h) ------------------------------------------------------------------------

// describe(node, ((type flag, shape), ...)) -> ([(type flag, shape), ...], temp-space bytes)
PyObject* py_describe(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *capsule, *given;
  if (!PyArg_ParseTuple(args, "OO!", &capsule, &PyTuple_Type, &given)) return nullptr;
  OpNode* n = static_cast<OpNode*>(PyCapsule_GetPointer(capsule, kNodeCapsule));
  if (n == nullptr) return nullptr;
  mxq_blob in[kMaxInputs];
  const Py_ssize_t num_in = PyTuple_GET_SIZE(given);
  if (num_in != n->num_inputs || num_in > kMaxInputs) {
    wrong_count(*n, num_in);
    return nullptr;
  }
  for (Py_ssize_t i = 0; i < num_in; ++i) {
    PyObject* shape;
    if (!PyArg_ParseTuple(PyTuple_GET_ITEM(given, i), "iO!", &in[i].dtype, &PyTuple_Type, &shape))
      return nullptr;
    in[i].ndim = static_cast<int>(PyTuple_GET_SIZE(shape));
    if (in[i].ndim > MXQ_MAX_NDIM) {
      PyErr_SetString(PyExc_IndexError, "too many dimensions");
      return nullptr;
    }
    for (int d = 0; d < in[i].ndim; ++d)
      in[i].shape[d] = PyLong_AsLongLong(PyTuple_GET_ITEM(shape, d));
  }
  if (PyErr_Occurred()) return nullptr;
  const auto sig = signature_of(n, in, static_cast<int>(num_in));
  if (sig == nullptr) return nullptr;
  PyObject* outs = PyList_New(0);
  for (const OutMeta& m : sig->outs) {
    PyObject* shape = PyTuple_New(m.ndim);
    for (int d = 0; d < m.ndim; ++d) PyTuple_SET_ITEM(shape, d, PyLong_FromLongLong(m.shape[d]));
    PyObject* one = Py_BuildValue("(iN)", m.flag, shape);
    if (one == nullptr || PyList_Append(outs, one) != 0) {
      Py_XDECREF(one);
      Py_DECREF(outs);
      return nullptr;
    }
    Py_DECREF(one);
  }
  return Py_BuildValue("(NK)", outs, static_cast<unsigned long long>(sig->temp_bytes));
  END_HANDLE_TH_ERRORS
}

constexpr const char* kPlanCapsule = "mxnet_amd.plan";

void free_plan(PyObject* capsule) {
  delete static_cast<mxq_plan::Plan*>(PyCapsule_GetPointer(capsule, kPlanCapsule));
}

bool int_list(PyObject* tuple, std::vector<int64_t>* out) {
  if (!PyTuple_Check(tuple)) {
    PyErr_SetString(PyExc_TypeError, "expected a tuple");
    return false;
  }
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(tuple); ++i)
    out->push_back(PyLong_AsLongLong(PyTuple_GET_ITEM(tuple, i)));
  return !PyErr_Occurred();
}

// step tuple: (kind, ints, floats, ((base, index, offset), ...)[, node, (num_in, ((flag, shape), ...))])
bool parse_step(PyObject* item, mxq_plan::Step* s) {
  int kind;
  PyObject *ints, *floats, *refs, *node = nullptr, *blobs = nullptr;
  if (!PyArg_ParseTuple(item, "iOO!O!|OO!", &kind, &ints, &PyTuple_Type, &floats, &PyTuple_Type,
                        &refs, &node, &PyTuple_Type, &blobs))
    return false;
  s->kind = static_cast<mxq_plan::Kind>(kind);
  if (!int_list(ints, &s->ints)) return false;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(floats); ++i)
    s->floats.push_back(static_cast<float>(PyFloat_AsDouble(PyTuple_GET_ITEM(floats, i))));
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(refs); ++i) {
    mxq_plan::Ref r;
    long long offset;
    if (!PyArg_ParseTuple(PyTuple_GET_ITEM(refs, i), "iiL", &r.base, &r.index, &offset))
      return false;
    r.offset = offset;
    s->refs.push_back(r);
  }
  if (node != nullptr) {
    const OpNode* n = static_cast<OpNode*>(PyCapsule_GetPointer(node, kNodeCapsule));
    if (n == nullptr) return false;
    s->node = n->handle;
    PyObject* list;
    if (!PyArg_ParseTuple(blobs, "iO!", &s->num_in, &PyTuple_Type, &list)) return false;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(list); ++i) {
      mxq_blob b = {};
      PyObject* shape;
      if (!PyArg_ParseTuple(PyTuple_GET_ITEM(list, i), "iO!", &b.dtype, &PyTuple_Type, &shape))
        return false;
      b.ndim = static_cast<int>(PyTuple_GET_SIZE(shape));
      if (b.ndim > MXQ_MAX_NDIM) {
        PyErr_SetString(PyExc_IndexError, "too many dimensions");
        return false;
      }
      for (int d = 0; d < b.ndim; ++d)
        b.shape[d] = PyLong_AsLongLong(PyTuple_GET_ITEM(shape, d));
      s->blobs.push_back(b);
    }
    if (s->refs.size() != s->blobs.size() + 1) {
      PyErr_SetString(PyExc_ValueError, "a node step has one reference per tensor and a workspace");
      return false;
    }
  }
  return !PyErr_Occurred();
}

// plan(arena bytes, [held tensors], [steps], [(type flag, shape) of the outputs])
PyObject* py_plan(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  long long arena;
  PyObject *held, *steps, *outputs;
  if (!PyArg_ParseTuple(args, "LO!O!O!", &arena, &PyList_Type, &held, &PyList_Type, &steps,
                        &PyList_Type, &outputs))
    return nullptr;
  std::unique_ptr<mxq_plan::Plan> plan(new mxq_plan::Plan());
  plan->arena_bytes = arena;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(held); ++i) {
    at::Tensor t;
    if (!tensor_arg(PyList_GET_ITEM(held, i), &t)) return nullptr;
    plan->held.push_back(t);
  }
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(steps); ++i) {
    mxq_plan::Step s;
    if (!parse_step(PyList_GET_ITEM(steps, i), &s)) return nullptr;
    plan->steps.push_back(std::move(s));
  }
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(outputs); ++i) {
    int flag;
    PyObject* shape;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(outputs, i), "iO!", &flag, &PyTuple_Type, &shape))
      return nullptr;
    mxq_plan::Output o;
    if (!dtype_of(flag, &o.type) || !int_list(shape, &o.shape)) return nullptr;
    plan->outputs.push_back(o);
  }
  PyObject* capsule = PyCapsule_New(plan.get(), kPlanCapsule, free_plan);
  if (capsule != nullptr) plan.release();
  return capsule;
  END_HANDLE_TH_ERRORS
}

// run_plan(plan, *feeds) -> [outputs]
PyObject* py_run_plan(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs < 2) {
    PyErr_SetString(PyExc_TypeError, "run_plan(plan, *feeds)");
    return nullptr;
  }
  const auto* plan = static_cast<mxq_plan::Plan*>(PyCapsule_GetPointer(args[0], kPlanCapsule));
  if (plan == nullptr) return nullptr;
  std::vector<at::Tensor> feeds(nargs - 1), outs;
  for (Py_ssize_t i = 1; i < nargs; ++i)
    if (!tensor_arg(args[i], &feeds[i - 1])) return nullptr;
  const at::Device dev = feeds[0].device();
  for (const auto& o : plan->outputs) outs.push_back(empty_on(o.shape, o.type, dev));
  at::Tensor arena;
  if (plan->arena_bytes != 0) arena = workspace(static_cast<size_t>(plan->arena_bytes), dev);
  void* stream = current_stream();
  std::string error;
  bool ok;
  Py_BEGIN_ALLOW_THREADS;
  ok = plan->run(stream, feeds, outs, arena, &error);
  Py_END_ALLOW_THREADS;
  if (!ok) {
    PyErr_SetString(g_op_error, error.c_str());
    return nullptr;
  }
  PyObject* list = PyList_New(static_cast<Py_ssize_t>(outs.size()));
  for (size_t i = 0; i < outs.size(); ++i) {
    PyObject* o = THPVariable_Wrap(std::move(outs[i]));
    if (o == nullptr) {
      Py_DECREF(list);
      return nullptr;
    }
    PyList_SET_ITEM(list, static_cast<Py_ssize_t>(i), o);
  }
  return list;
  END_HANDLE_TH_ERRORS
}

// same_params(dict, ((name, tensor, version), ...)): the dict still holds these tensors, unwritten
PyObject* py_same_params(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 2 || !PyDict_Check(args[0]) || !PyTuple_Check(args[1])) {
    PyErr_SetString(PyExc_TypeError, "same_params(dict, entries)");
    return nullptr;
  }
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(args[1]); ++i) {
    PyObject* entry = PyTuple_GET_ITEM(args[1], i);
    PyObject* now = PyDict_GetItemWithError(args[0], PyTuple_GET_ITEM(entry, 0));
    PyObject* was = PyTuple_GET_ITEM(entry, 1);
    if (now == nullptr && PyErr_Occurred()) return nullptr;
    if (now != was) Py_RETURN_FALSE;
    const at::Tensor& t = THPVariable_Unpack(was);
    if (static_cast<long>(t._version()) != PyLong_AsLong(PyTuple_GET_ITEM(entry, 2)))
      Py_RETURN_FALSE;
  }
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// float_of(text): an attribute's value as the operators parse it
PyObject* py_float_of(PyObject*, PyObject* text) {
  const char* s = PyUnicode_AsUTF8(text);
  if (s == nullptr) return nullptr;
  char* end = nullptr;
  const float v = std::strtof(s, &end);
  if (end == s) {
    PyErr_SetString(PyExc_ValueError, "not a number");
    return nullptr;
  }
  return PyFloat_FromDouble(v);
}

// init(MXNetError, MXQError)
PyObject* py_init(PyObject*, PyObject* args) {
  PyObject *op_error, *lib_error;
  if (!PyArg_ParseTuple(args, "OO", &op_error, &lib_error)) return nullptr;
  Py_INCREF(op_error);
  Py_INCREF(lib_error);
  Py_XSETREF(g_op_error, op_error);
  Py_XSETREF(g_lib_error, lib_error);
  Py_RETURN_NONE;
}

template <typename F>
PyCFunction as_cfunction(F f) {
  return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f));
}

PyMethodDef methods[] = {
    {"init", py_init, METH_VARARGS, "Registers the package's exception classes."},
    {"invoke", as_cfunction(py_invoke), METH_FASTCALL | METH_KEYWORDS,
     "invoke(op, *tensors, **attrs): one imperative operator call."},
    {"node", py_node, METH_VARARGS, "The call table of an existing node."},
    {"forward", as_cfunction(py_forward), METH_FASTCALL, "One call of an existing node."},
    {"quantized_fc", as_cfunction(py_quantized_fc), METH_FASTCALL, nullptr},
    {"quantized_conv_nhwc", as_cfunction(py_quantized_conv_nhwc), METH_FASTCALL, nullptr},
    {"describe", py_describe, METH_VARARGS, nullptr},
    {"plan", py_plan, METH_VARARGS, nullptr},
    {"run_plan", as_cfunction(py_run_plan), METH_FASTCALL, nullptr},
    {"same_params", as_cfunction(py_same_params), METH_FASTCALL, nullptr},
    {"float_of", py_float_of, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_frontend", nullptr, -1, methods, nullptr, nullptr,
                      nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__frontend(void) { return PyModule_Create(&module); }

// The layer calls of dispatch.py in native code: a CPython module (`_gguf_calls`) whose functions take the tensors of
// one call, check them, pick the path, allocate the result and the workspace and launch through the C ABI, all in one
// step from the interpreter.  What bounds a decode step of a small matrix is the host: through ops.py and ctypes a call
// costs about 11 us, three times what the kernel of a [3072,1024] Q8_0 matrix runs for.
//
// Every function returns None for a call it does not serve (another device than the current one, tensors that are not
// plain dense ones, a malformed shape, an unquantized type, ...) before anything is allocated or launched; dispatch.py
// then takes its Python path, which raises what there is to raise.  Both make the same calls of the C ABI with the same
// arguments, and so have the same results bit for bit.
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/EmptyTensor.h>
#include <ATen/autocast_mode.h>
#include <ATen/ops/matmul.h>
#include <ATen/hip/impl/HIPCachingAllocatorMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <vector>

#include "../dense_api.h"
#include "gguf_hip.h"

namespace {

// ---- what dispatch.py decides (select_mul_mat_path, mmvq_safe, select_moe_path), restated; tests compare the two
enum Path { PATH_OTHER = 0, PATH_MMVQ = 1, PATH_MMQ = 2, PATH_DENSE = 3 };

bool is_matrix_type(int t) { return t == 2 || t == 3 || (t >= 6 && t <= 8) || (t >= 10 && t <= 14); }
bool is_imatrix_type(int t) { return (t >= 16 && t <= 23) || t == 29; }

Path mul_mat_path(int type, int64_t batch, int64_t rows) {
  const bool im = is_imatrix_type(type);
  if (batch <= 0 || !(im || is_matrix_type(type))) return PATH_OTHER;
  const int64_t safe = im ? (rows > 5120 ? 8 : 16) : (rows > 5120 ? 2 : 6);
  if (batch <= safe) return PATH_MMVQ;
  return im ? PATH_DENSE : PATH_MMQ;
}

constexpr int64_t kMoeVecMaxTokens = 64, kMoeGroupedMaxExperts = 256;

// ---- tensors
int dtype_code(at::ScalarType t) {
  return t == at::kHalf ? GGUF_DTYPE_F16 : t == at::kBFloat16 ? GGUF_DTYPE_BF16 : t == at::kFloat ? GGUF_DTYPE_F32 : -1;
}

// A plain dense tensor on GPU `dev` (no subclass with behaviour of its own)
const at::Tensor* plain(PyObject* o, int dev) {
  if (!THPVariable_Check(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.get_device() != dev || t.layout() != at::kStrided) return nullptr;
  if (t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::Functionalize, c10::DispatchKey::Negative,
                                               c10::DispatchKey::Conjugate, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper})))
    return nullptr;
  return &t;
}

// Whether torch would do more in the dense path's `x @ dense.T` (then `add_` of the bias, `copy_` to the result) than
// multiply: record it for a gradient, carry a tangent along, hand it to a tensor subclass, cast its operands.  A kernel
// on raw pointers cannot stand in for that; dispatch.py then takes the two steps.
bool product_is_watched(PyObject* const* objects, std::initializer_list<const at::Tensor*> tensors) {
  for (const at::Tensor* t : tensors) {
    PyObject* const o = *objects++;
    if (!t) continue;
    if (!THPVariable_CheckExact(o) || (at::GradMode::is_enabled() && t->requires_grad()) || t->_fw_grad(0).defined()) return true;
  }
  const at::Tensor& x = **tensors.begin();
  return at::autocast::is_autocast_enabled(at::kCUDA) && at::autocast::get_autocast_dtype(at::kCUDA) != x.scalar_type();
}

// the current GPU, or -1 where a dispatch mode (tracing, fake tensors) watches torch's calls
int current_gpu() {
  int dev = -1;
  if (c10::impl::TorchDispatchModeTLS::any_modes_set() || hipGetDevice(&dev) != hipSuccess) return -1;
  return dev;
}

// torch's caching allocator for tensors of device type "cuda"
c10::Allocator* gpu_allocator() { return c10::hip::HIPCachingAllocatorMasqueradingAsCUDA::get(); }

at::Tensor new_tensor(at::IntArrayRef size, at::ScalarType dtype) {   // on the current GPU, like torch.empty
  static const c10::DispatchKeySet keys(c10::DispatchKey::CUDA);
  return at::Tensor(at::detail::empty_generic(size, gpu_allocator(), keys, dtype, std::nullopt));
}

// stream-ordered scratch from torch's allocator: given back when it goes out of scope, after the launches that use it
c10::DataPtr scratch(int64_t bytes) { return gpu_allocator()->allocate((size_t)std::max<int64_t>(bytes, 16)); }

gguf_stream_t stream_of(int dev) { return (gguf_stream_t)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA((c10::DeviceIndex)dev).stream(); }

struct NoGil {   // other threads run while a call allocates and launches, also when an allocation throws
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

PyObject* fail(int rc, const char* what) {
  PyErr_Format(rc == GGUF_ERR_TYPE ? PyExc_NotImplementedError : PyExc_ValueError, "%s: error %d from libgguf_hip (see gguf_hip.h)", what, rc);
  return nullptr;
}

bool as_int(PyObject* o, int64_t* v) {
  *v = PyLong_AsLongLong(o);
  if (*v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

// ---- one shard of a linear layer
struct Shard {
  Path path;
  int type;
  const void* w;
  int64_t pitch, rows;   // bytes between rows of W, output features
  void* y;
  int64_t ldy;
  const void* bias;
};

// launches one shard on the current GPU; the workspace lives until the launches are queued
int run_shard(const Shard& s, const at::Tensor& x, int xcode, gguf_stream_t stream) {
  const int64_t m = x.size(0), k = x.size(1);
  if (s.path == PATH_DENSE) {
    const int64_t bytes = gguf_dense_linear_workspace_bytes(s.rows, k, m);
    const c10::DataPtr ws = scratch(bytes);
    return gguf_dense_linear(s.w, s.pitch, x.const_data_ptr(), xcode, ws.get(), s.y, s.ldy, s.bias, s.type, s.rows, k, m, bytes, stream);
  }
  // (scratch that no kernel of the call uses: host time of a call of [3072,1024] Q8_0, one row, with / without 4.11 / 3.82 us)
  if (s.path == PATH_MMVQ) {
    int taken;
    const int rc = gguf_mmvq_linear_whole(s.w, s.pitch, x.const_data_ptr(), xcode, s.y, s.ldy, s.bias, s.type, s.rows, k, m, stream, &taken);
    if (taken) return rc;
  }
  const int64_t bytes = s.path == PATH_MMQ ? gguf_mmq_layer_workspace_bytes(s.type, s.rows, k, m, s.pitch) : m * gguf_q8_1_row_bytes(k);
  const c10::DataPtr ws = scratch(bytes);
  if (s.path == PATH_MMVQ)
    return gguf_mmvq_linear(s.w, s.pitch, x.const_data_ptr(), xcode, ws.get(), s.y, s.ldy, s.bias, s.type, s.rows, k, m, stream);
  return gguf_mmq_linear(s.w, s.pitch, x.const_data_ptr(), xcode, ws.get(), s.y, s.ldy, s.bias, s.type, s.rows, k, m, GGUF_MMQ_AUTO,
                         std::max<int64_t>(bytes, 16), stream);
}

// activations the kernels take as they lie
bool rows_ok(const at::Tensor& x) { return x.dim() == 2 && x.size(0) > 0 && x.size(1) > 0 && x.is_contiguous() && dtype_code(x.scalar_type()) >= 0; }
bool packed_ok(const at::Tensor& w) { return w.dim() == 2 && w.scalar_type() == at::kByte && (w.size(1) <= 1 || w.stride(1) == 1); }
// whether a call on this path is served here
bool path_ok(Path p, int type, const at::Tensor& x, const at::Tensor& w, int64_t rows) {
  if (p == PATH_DENSE)
    return gguf_dense_linear_takes(type, dtype_code(x.scalar_type()), rows, x.size(1), x.size(0)) && ((uintptr_t)x.const_data_ptr() & 15) == 0 &&
           ((uintptr_t)w.const_data_ptr() & 1) == 0 && (w.stride(0) & 1) == 0;
  return p != PATH_OTHER;
}
int64_t row_bytes(int type, int64_t k) {   // 0 where K is not whole blocks of the type
  const int qk = gguf_block_elems(type);
  return qk == 0 || k % qk ? 0 : k / qk * gguf_block_bytes(type);
}

// a dense copy of the weights and a library product, the reference's two steps (quantization/linear.py:50-58)
at::Tensor dense_copy_product(const at::Tensor& x, const at::Tensor& w, int type, gguf_stream_t stream) {
  const NoGil nogil;
  const at::Tensor dense = new_tensor({w.size(0), x.size(1)}, x.scalar_type());
  if (gguf_dequantize(w.const_data_ptr(), type, dense.mutable_data_ptr(), dtype_code(x.scalar_type()), dense.numel(), stream) != GGUF_OK) return {};
  return at::matmul(x, dense.t());
}

// linear(x, weight, weight_type, out, bias) -> Tensor | None
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 5) return PyErr_Format(PyExc_TypeError, "linear takes 5 arguments"), nullptr;
  const int dev = current_gpu();
  int64_t type;
  const at::Tensor *x = dev < 0 ? nullptr : plain(a[0], dev), *w = x ? plain(a[1], dev) : nullptr;
  if (!w || !as_int(a[2], &type) || !rows_ok(*x) || !packed_ok(*w)) Py_RETURN_NONE;
  const int64_t m = x->size(0), k = x->size(1), rows = w->size(0), rb = row_bytes((int)type, k);
  const Path path = mul_mat_path((int)type, m, rows);
  if (rb == 0 || w->size(1) < rb || rows == 0) Py_RETURN_NONE;
  if (path == PATH_DENSE && w->size(1) != rb) Py_RETURN_NONE;   // (wider weights do not fit x in the product of a dense copy)
  if (!path_ok(path, (int)type, *x, *w, rows)) {
    if (path != PATH_DENSE || !w->is_contiguous() || a[3] != Py_None || a[4] != Py_None || !THPVariable_CheckExact(a[0])) Py_RETURN_NONE;
    at::Tensor y = dense_copy_product(*x, *w, (int)type, stream_of(dev));
    if (!y.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(y));
  }
  const at::Tensor *out = nullptr, *bias = nullptr;
  if (a[3] != Py_None) {
    out = plain(a[3], dev);
    if (!out || out->dim() != 2 || out->size(0) != m || out->size(1) != rows || out->scalar_type() != x->scalar_type() ||
        (rows > 1 && out->stride(1) != 1))
      Py_RETURN_NONE;
    // (`out.copy_(y)`, which the dense path's store stands in for, refuses rows that overlap and takes memory shared with x)
    if (path == PATH_DENSE && ((m > 1 && out->stride(0) < rows) || out->is_alias_of(*x) || out->is_alias_of(*w))) Py_RETURN_NONE;
  }
  if (a[4] != Py_None) {
    bias = plain(a[4], dev);
    if (!bias || bias->dim() != 1 || bias->size(0) != rows || bias->scalar_type() != x->scalar_type() || !bias->is_contiguous()) Py_RETURN_NONE;
    if (path == PATH_DENSE && out && out->is_alias_of(*bias)) Py_RETURN_NONE;
  }
  if (path == PATH_DENSE) {
    PyObject* const objects[] = {a[0], a[3], a[4]};
    if (product_is_watched(objects, {x, out, bias})) Py_RETURN_NONE;
  }
  at::Tensor y;
  int rc;
  {
    const NoGil nogil;
    if (!out) y = new_tensor({m, rows}, x->scalar_type());
    const at::Tensor& dst = out ? *out : y;
    const Shard s{path, (int)type, w->const_data_ptr(), rows > 1 ? w->stride(0) : rb, rows, dst.mutable_data_ptr(), m > 1 ? dst.stride(0) : rows,
                  bias ? bias->const_data_ptr() : nullptr};
    rc = run_shard(s, *x, dtype_code(x->scalar_type()), stream_of(dev));
  }
  if (rc != GGUF_OK) return fail(rc, path == PATH_MMVQ ? "ggml_mul_mat_vec_a8" : path == PATH_MMQ ? "ggml_mul_mat_a8" : "dense_linear");
  if (out) {
    if (path == PATH_DENSE && !out->is_inference()) out->unsafeGetTensorImpl()->bump_version();   // (as copy_ does)
    return Py_NewRef(a[3]);
  }
  return THPVariable_Wrap(std::move(y));
}

// merged_linear(x, weight, shard_ids, shard_offset_map, types, bias) -> Tensor | None: the shards of a merged layer
// whose types differ, in the order of shard_ids; shard_offset_map[id] = (first row, row behind the last, bytes of a row)
// and types lists their ggml types.  Neighbouring shards of one type whose rows lie next to each other and which take
// the same path are one matrix with more rows and so one call: q and k of a mixed recipe, [4096 + 1024, 4096] Q4_K,
// 9.1 -> 5.6 us of kernel time.  The path is that of the shards, each by its own rows, as in the reference's policy, and past
// 32 rows of X a run keeps to the matrix unit that its largest shard takes by itself, or both are on the walking tiles
// (csrc/tile_walk_core.h), whatever stands behind those: 120 such q and k of 33 to 2037 rows took 1.43 times as long shard
// by shard as they take as one matrix.  Within that, how K is shared depends on the rows of the whole matrix, so a result may differ from
// the single shard's by the order of a 32-bit sum.  (dispatch.py, _shard_runs, does the same.)
PyObject* merged_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 6) return PyErr_Format(PyExc_TypeError, "merged_linear takes 6 arguments"), nullptr;
  const int dev = current_gpu();
  const at::Tensor *x = dev < 0 ? nullptr : plain(a[0], dev), *w = x ? plain(a[1], dev) : nullptr;
  if (!w || !rows_ok(*x) || !packed_ok(*w) || !PyList_Check(a[2]) || !PyDict_Check(a[3]) || !PyList_Check(a[4])) Py_RETURN_NONE;
  const Py_ssize_t count = PyList_GET_SIZE(a[2]);
  if (count == 0 || PyList_GET_SIZE(a[4]) != count) Py_RETURN_NONE;
  const int64_t m = x->size(0), k = x->size(1);
  const size_t esz = x->element_size();
  struct Part { int64_t start, end, type, rb, largest; Path path; };
  const auto same_unit = [&](const Part& p, int64_t rows, int64_t rows2) {
    if (m <= 32) return true;
    const int64_t pitch = w->size(0) > 1 ? w->stride(0) : p.rb;
    const int64_t room = gguf_mmq_layer_workspace_bytes((int)p.type, rows, k, m, pitch), room2 = gguf_mmq_layer_workspace_bytes((int)p.type, rows2, k, m, pitch);
    return gguf_mmq_layer_unit((int)p.type, rows, k, m, pitch, room) == gguf_mmq_layer_unit((int)p.type, rows2, k, m, pitch, room2) ||
           (gguf_linear_walk((int)p.type, rows, k, m, pitch, room) && gguf_linear_walk((int)p.type, rows2, k, m, pitch, room2));
  };
  std::vector<Part> parts;
  int64_t width = 0;
  for (Py_ssize_t i = 0; i < count; ++i) {
    PyObject* at = PyDict_GetItemWithError(a[3], PyList_GET_ITEM(a[2], i));
    if (!at) PyErr_Clear();
    Part p;
    if (!at || !PyTuple_Check(at) || PyTuple_GET_SIZE(at) != 3 || !as_int(PyTuple_GET_ITEM(at, 0), &p.start) || !as_int(PyTuple_GET_ITEM(at, 1), &p.end) ||
        !as_int(PyTuple_GET_ITEM(at, 2), &p.rb) || !as_int(PyList_GET_ITEM(a[4], i), &p.type))
      Py_RETURN_NONE;
    const int64_t rows = p.end - p.start, rb = row_bytes((int)p.type, k);
    p.path = mul_mat_path((int)p.type, m, rows);
    if (rows <= 0 || p.start < 0 || p.end > w->size(0) || rb == 0 || p.rb < rb || p.rb > w->size(1) ||
        (p.path == PATH_DENSE && p.rb != rb))
      Py_RETURN_NONE;
    width += rows;
    p.largest = rows;
    if (!parts.empty()) {
      Part& last = parts.back();
      const int64_t largest = std::max(last.largest, rows);
      if (last.end == p.start && last.type == p.type && last.rb == p.rb && last.path == p.path &&
          (p.path != PATH_MMQ || same_unit(p, largest, p.end - last.start))) {
        last.end = p.end;
        last.largest = largest;
        continue;
      }
    }
    parts.push_back(p);
  }
  for (const Part& p : parts)
    if (!path_ok(p.path, (int)p.type, *x, *w, p.end - p.start)) Py_RETURN_NONE;
  const at::Tensor* bias = nullptr;
  if (a[5] != Py_None) {
    bias = plain(a[5], dev);
    if (!bias || bias->dim() != 1 || bias->size(0) != width || bias->scalar_type() != x->scalar_type() || !bias->is_contiguous()) Py_RETURN_NONE;
  }
  if (std::any_of(parts.begin(), parts.end(), [](const Part& p) { return p.path == PATH_DENSE; })) {
    PyObject* const objects[] = {a[0], a[5]};
    if (product_is_watched(objects, {x, bias})) Py_RETURN_NONE;
  }
  at::Tensor y;
  int rc = GGUF_OK;
  {
    const NoGil nogil;
    y = new_tensor({m, width}, x->scalar_type());
    const gguf_stream_t stream = stream_of(dev);
    char* dst = (char*)y.mutable_data_ptr();
    const char* b = bias ? (const char*)bias->const_data_ptr() : nullptr;
    // two matrices on the GEMV or the kernels of a few rows: x is quantized once, and they run side by side
    const auto pitch_of = [&](const Part& p) { return w->size(0) > 1 ? w->stride(0) : p.rb; };
    const bool two = parts.size() == 2 && m <= 32 && parts[0].path != PATH_DENSE && parts[1].path != PATH_DENSE;
    const int gemv = two ? (parts[0].path == PATH_MMVQ) | (parts[1].path == PATH_MMVQ) << 1 : 0;
    if (two &&
        gguf_linear_two_takes((int)parts[0].type, parts[0].end - parts[0].start, pitch_of(parts[0]), (int)parts[1].type, parts[1].end - parts[1].start, pitch_of(parts[1]), k, m, gemv)) {
      const Part &p = parts[0], &q = parts[1];
      const int64_t rows = p.end - p.start;
      const c10::DataPtr ws = scratch(m * gguf_q8_1_row_bytes(k));
      rc = gguf_linear_two((const char*)w->const_data_ptr() + p.start * pitch_of(p), pitch_of(p), (int)p.type, rows, dst, b,
                           (const char*)w->const_data_ptr() + q.start * pitch_of(q), pitch_of(q), (int)q.type, q.end - q.start, dst + rows * esz, b ? b + rows * esz : nullptr,
                           x->const_data_ptr(), dtype_code(x->scalar_type()), ws.get(), width, k, m, gemv, stream);
      parts.clear();
    }
    for (const Part& p : parts) {
      const int64_t rows = p.end - p.start;
      const int64_t pitch = w->size(0) > 1 ? w->stride(0) : p.rb;
      const Shard s{p.path, (int)p.type, (const char*)w->const_data_ptr() + p.start * pitch, pitch, rows, dst, width, b};
      rc = run_shard(s, *x, dtype_code(x->scalar_type()), stream);
      if (rc != GGUF_OK) break;
      dst += rows * esz;
      if (b) b += rows * esz;
  }
  }
  if (rc != GGUF_OK) return fail(rc, "apply_linear");
  return THPVariable_Wrap(std::move(y));
}

// moe(x, w1, w2, topk_weights, topk_ids, type, type2, activation) -> Tensor | None: the layers that one entry point of
// the C ABI serves whole
PyObject* moe(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 8) return PyErr_Format(PyExc_TypeError, "moe takes 8 arguments"), nullptr;
  const int dev = current_gpu();
  const at::Tensor* t[5];
  for (int i = 0; i < 5; ++i) {
    t[i] = dev < 0 ? nullptr : plain(a[i], dev);
    if (!t[i] || !t[i]->is_contiguous()) Py_RETURN_NONE;
  }
  const at::Tensor &x = *t[0], &w1 = *t[1], &w2 = *t[2], &tw = *t[3], &ids = *t[4];
  int64_t type, type2;
  if (!as_int(a[5], &type) || !as_int(a[6], &type2) || !PyUnicode_Check(a[7]) || !rows_ok(x) || w1.dim() != 3 || w2.dim() != 3 ||
      w1.scalar_type() != at::kByte || w2.scalar_type() != at::kByte || ids.dim() != 2 || ids.scalar_type() != at::kInt ||
      tw.scalar_type() != at::kFloat || tw.numel() != ids.numel())
    Py_RETURN_NONE;
  const int act = PyUnicode_CompareWithASCIIString(a[7], "silu") == 0 ? 1 : PyUnicode_CompareWithASCIIString(a[7], "gelu") == 0 ? 2 : 0;
  const int64_t tokens = ids.size(0), top_k = ids.size(1), hidden = x.size(1), experts = w1.size(0), inner = w1.size(1) / 2, n_out = w2.size(1);
  const bool known = (is_matrix_type((int)type) || is_imatrix_type((int)type)) && (is_matrix_type((int)type2) || is_imatrix_type((int)type2));
  if (!act || !known || tokens != x.size(0) || top_k <= 0 || w2.size(0) != experts || n_out != hidden || w1.size(1) % 2 != 0 ||
      row_bytes((int)type, hidden) == 0 || w1.size(2) != row_bytes((int)type, hidden) || row_bytes((int)type2, inner) == 0 ||
      w2.size(2) != row_bytes((int)type2, inner))
    Py_RETURN_NONE;
  const bool grouped = is_matrix_type((int)type) && is_matrix_type((int)type2) && tokens > kMoeVecMaxTokens && experts <= kMoeGroupedMaxExperts;
  const int xcode = dtype_code(x.scalar_type()), t1 = (int)type, t2 = (int)type2;
  if (!(grouped ? gguf_moe_mmq_layer_takes(t1, t2, hidden, inner, n_out, top_k, tokens, experts)
                : gguf_moe_vec_layer_takes(t1, t2, hidden, inner, n_out, top_k, tokens, experts)))
    Py_RETURN_NONE;
  at::Tensor y;
  int rc;
  {
    const NoGil nogil;
    y = new_tensor({tokens, n_out}, x.scalar_type());
    const int64_t bytes = std::max<int64_t>(16, grouped ? gguf_moe_mmq_layer_workspace_bytes(t1, t2, tokens, top_k, hidden, inner, n_out, experts, xcode)
                                                        : gguf_moe_vec_layer_workspace_bytes(tokens, top_k, hidden, inner, n_out, experts, xcode));
    const c10::DataPtr ws = scratch(bytes);
    rc = (grouped ? gguf_moe_mmq_layer : gguf_moe_vec_layer)(x.const_data_ptr(), xcode, w1.const_data_ptr(), t1, w2.const_data_ptr(), t2,
                                                             ids.const_data_ptr<int32_t>(), tw.const_data_ptr<float>(), ws.get(), bytes, y.mutable_data_ptr(),
                                                             hidden, inner, n_out, top_k, tokens, act, experts, stream_of(dev));
  }
  if (rc != GGUF_OK) return fail(rc, grouped ? "moe_mmq_layer" : "moe_vec_layer");
  return THPVariable_Wrap(std::move(y));
}

// embedding(ids, weight, type, hidden, dtype) -> Tensor | None
PyObject* embedding(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 5) return PyErr_Format(PyExc_TypeError, "embedding takes 5 arguments"), nullptr;
  const int dev = current_gpu();
  int64_t type, hidden;
  const at::Tensor *ids = dev < 0 ? nullptr : plain(a[0], dev), *w = ids ? plain(a[1], dev) : nullptr;
  if (!w || !as_int(a[2], &type) || !as_int(a[3], &hidden) || ids->scalar_type() != at::kLong || !ids->is_contiguous() || ids->numel() == 0 ||
      !packed_ok(*w) || !w->is_contiguous() || hidden <= 0 || !(is_matrix_type((int)type) || is_imatrix_type((int)type)) ||
      row_bytes((int)type, hidden) == 0 || row_bytes((int)type, hidden) != w->size(1))
    Py_RETURN_NONE;
  at::ScalarType dtype = at::kHalf;
  if (a[4] != Py_None) {
    if (!THPDtype_Check(a[4])) Py_RETURN_NONE;
    dtype = reinterpret_cast<THPDtype*>(a[4])->scalar_type;
  }
  const int code = dtype_code(dtype);
  if (code < 0) Py_RETURN_NONE;
  at::Tensor y;
  int rc;
  {
    const NoGil nogil;
    c10::SmallVector<int64_t, 4> shape(ids->sizes().begin(), ids->sizes().end());
    shape.push_back(hidden);
    y = new_tensor(shape, dtype);
    rc = gguf_dequantize_rows(w->const_data_ptr(), (int)type, ids->const_data_ptr<int64_t>(), ids->numel(), w->size(0), hidden, y.mutable_data_ptr(),
                              code, stream_of(dev));
  }
  if (rc != GGUF_OK) return fail(rc, "ggml_dequantize_rows");
  return THPVariable_Wrap(std::move(y));
}

// mul_mat_path(type, batch, rows) -> "mmvq" | "mmq" | None, for the test that compares it with dispatch.py
PyObject* path_name(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t v[3];
  if (n != 3 || !as_int(a[0], v) || !as_int(a[1], v + 1) || !as_int(a[2], v + 2)) return PyErr_Format(PyExc_TypeError, "mul_mat_path takes 3 integers"), nullptr;
  const Path p = mul_mat_path((int)v[0], v[1], v[2]);
  if (p != PATH_MMVQ && p != PATH_MMQ) Py_RETURN_NONE;
  return PyUnicode_FromString(p == PATH_MMVQ ? "mmvq" : "mmq");
}

// a C++ exception of torch (out of memory) becomes the Python exception it stands for
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  return F(self, a, n);
  END_HANDLE_TH_ERRORS
}

#define CALL(name, fn) {name, (PyCFunction)(void (*)(void))&guarded<&fn>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {CALL("linear", linear), CALL("merged_linear", merged_linear), CALL("moe", moe), CALL("embedding", embedding),
                         CALL("mul_mat_path", path_name), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_gguf_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__gguf_calls() { return PyModule_Create(&module); }

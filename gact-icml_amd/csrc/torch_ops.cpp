// The host side of the operators: what Python did for every saved tensor - look at the arguments, allocate the results
// with torch, find the stream, call the library - in one native call.
//
// Every function answers the ordinary call: plain tensors on the GPU, contiguous and aligned as the kernels need (quantize: of
// any strides, in place or through a contiguous copy), no mode or transform of torch's active.  Anything else, an argument that has to be refused included, gets None and nothing is
// launched: the Python operator then takes its general path, which accepts or raises as it always did.
//
// Arguments come through the C API's fast call and tensors through torch's own wrap / unpack (no pybind11).
#include <torch/csrc/python_headers.h>

#include <ATen/Context.h>
#include <ATen/EmptyTensor.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/CachingHostAllocator.h>
#include <ATen/core/Tensor.h>
#include <ATen/detail/CUDAHooksInterface.h>
#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <thread>
#include <vector>

#include "gact_hip.h"

namespace {

constexpr int64_t kGroup = 256;

// torch.empty, called below, would mean something else: a mode that looks at every call, a transform, a trace
bool ordinary_call() {
  static const c10::DispatchKeySet special({c10::DispatchKey::Python, c10::DispatchKey::Functionalize, c10::DispatchKey::Tracer,
                                            c10::DispatchKey::FuncTorchDynamicLayerFrontMode, c10::DispatchKey::FuncTorchVmapMode});
  return !c10::impl::tls_local_dispatch_key_set().included_.has_any(special) && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         !at::impl::torch_function_mode_enabled();
}

// a tensor (or parameter) itself, no subclass and no wrapper, no lazily negated view, dense on the GPU
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  static const c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::Functionalize, c10::DispatchKey::ZeroTensor,
                                            c10::DispatchKey::Negative, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper});
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() || t.key_set().has_any(wrapped)) return nullptr;
  return &t;
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return GACT_F32;
    case at::kHalf: return GACT_F16;
    case at::kBFloat16: return GACT_BF16;
    default: return -1;
  }
}
bool float_or_half(const at::Tensor& t) { return t.scalar_type() == at::kFloat || t.scalar_type() == at::kHalf; }

bool integer(PyObject* o, int64_t* v) {   // an int and nothing else (no bool)
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  *v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}
bool width(PyObject* o, int* bits) {
  int64_t v;
  if (!integer(o, &v) || (v != 1 && v != 2 && v != 4 && v != 8)) return false;
  *bits = (int)v;
  return true;
}
bool seed_of(PyObject* o, uint64_t* seed) {   // the reference's binding takes an int and widens it
  int64_t v;
  if (!integer(o, &v) || v < INT32_MIN || v > INT32_MAX) return false;
  *seed = (uint64_t)v;
  return true;
}
// what the kernels draw without further inputs; a stream's name that is not known arrives as -1
bool noise_mode(PyObject* o, int* mode) {
  int64_t v;
  if (!integer(o, &v) || (v != GACT_NOISE_CONST && v != GACT_NOISE_REF && v != GACT_NOISE_FAST)) return false;
  *mode = (int)v;
  return true;
}
// elements of the packed tensor: the reference allocates one byte more than is ever written
int64_t packed_numel(int bits, int64_t N, int64_t row) {
  const int64_t wpt = 8 / bits;
  return (bits * ((N + wpt - 1) / wpt * wpt) * row + 8) / 8;
}

// torch.empty on the GPU without the dispatcher's way there, half of what an allocation costs: every caller has looked whether anything
// listens to that (ordinary_call).  torch's deterministic mode fills new memory, so it goes through torch.
at::Tensor make(c10::IntArrayRef shape, at::ScalarType dtype, c10::Device device) {
  if (at::globalContext().deterministicAlgorithms() && at::globalContext().deterministicFillUninitializedMemory())
    return at::empty(shape, at::TensorOptions().dtype(dtype).device(device));
  const c10::DeviceGuard guard(device);
  return at::detail::empty_generic(shape, at::detail::getCUDAHooks().getCUDADeviceAllocator(), c10::DispatchKeySet(c10::DispatchKey::CUDA), dtype, std::nullopt);
}
void* stream_on(c10::Device device) { return c10::hip::getCurrentHIPStream(device.index()).stream(); }
const void* in(const at::Tensor& t) { return t.const_data_ptr(); }
void* out(const at::Tensor& t) { return t.mutable_data_ptr(); }

// The GIL is released as long as this lives, and is back before an exception that leaves its scope becomes one of Python's
struct WithoutGil {
  PyThreadState* const state = PyEval_SaveThread();
  WithoutGil() = default;
  WithoutGil(const WithoutGil&) = delete;
  ~WithoutGil() { PyEval_RestoreThread(state); }
};
// The library's call with the GIL released and the data's device current
template <typename F>
int on(c10::Device device, const F& call) {
  const c10::DeviceGuard guard(device);
  void* const stream = stream_on(device);
  const WithoutGil released;
  return call(stream);
}

PyObject* tuple_of(std::initializer_list<at::Tensor> tensors) {
  PyObject* const t = PyTuple_New((Py_ssize_t)tensors.size());
  if (!t) return nullptr;
  Py_ssize_t i = 0;
  for (const at::Tensor& e : tensors) {
    PyObject* const w = THPVariable_Wrap(e);
    if (!w) {
      Py_DECREF(t);
      return nullptr;
    }
    PyTuple_SET_ITEM(t, i++, w);
  }
  return t;
}

bool one_pass(int64_t group, int dtype) { return group == kGroup || ((group == 64 || group == 128 || group == 512) && dtype != GACT_BF16); }

// quantize(x, bits, seed, noise mode, group size) -> (codes, scale, min)
PyObject* quantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int bits, mode;
  uint64_t seed;
  int64_t group;
  const at::Tensor* x;
  if (n != 5 || !(x = plain(args[0])) || !width(args[1], &bits) || !seed_of(args[2], &seed) || !noise_mode(args[3], &mode) ||
      !integer(args[4], &group) || !ordinary_call())
    Py_RETURN_NONE;
  const int dtype = dtype_code(x->scalar_type());
  const int64_t numel = x->numel();
  if (dtype < 0 || numel == 0 || !one_pass(group, dtype) || (group != kGroup && mode == GACT_NOISE_REF)) Py_RETURN_NONE;
  const bool contiguous = x->is_contiguous();
  if (contiguous && (reinterpret_cast<uintptr_t>(in(*x)) & 15u) != 0) Py_RETURN_NONE;
  const int64_t N = (numel + group - 1) / group;
  const c10::Device device = x->device();
  const at::Tensor codes = make({packed_numel(bits, N, group)}, at::kChar, device);
  const at::Tensor scale = make({N, 1, 1}, dtype == GACT_BF16 ? at::kFloat : x->scalar_type(), device);
  const at::Tensor mn = make({N, 1, 1}, x->scalar_type(), device);
  int rc = GACT_ESHAPE;
  if (!contiguous && group == kGroup && mode != GACT_NOISE_REF) {
    rc = on(device, [&](void* stream) {
      return gact_quantize_strided(in(*x), dtype, (int)x->dim(), x->sizes().data(), x->strides().data(), bits, mode, seed, nullptr,
                                   out(codes), out(scale), out(mn), nullptr, stream);
    });
  }
  if (rc == GACT_ESHAPE) {   // contiguous, or a layout that is copied first
    const at::Tensor dense = x->contiguous();
    rc = on(device, [&](void* stream) {
      if (group == kGroup)
        return gact_quantize(in(dense), dtype, numel, bits, mode, seed, nullptr, out(codes), out(scale), out(mn), nullptr, stream);
      return gact_quantize_groups(in(dense), dtype, numel, (int)group, bits, mode, seed, nullptr, nullptr, out(codes), out(scale),
                                  out(mn), nullptr, stream);
    });
  }
  if (rc == GACT_OK) return tuple_of({codes, scale, mn});
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// dequantize(codes, shape, bits, scale, min, group size) -> tensor of that shape
PyObject* dequantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int bits;
  int64_t group;
  const at::Tensor *codes, *scale, *mn;
  if (n != 6 || !(codes = plain(args[0])) || !PyTuple_Check(args[1]) || !width(args[2], &bits) || !(scale = plain(args[3])) ||
      !(mn = plain(args[4])) || !integer(args[5], &group) || !ordinary_call())
    Py_RETURN_NONE;
  const int dtype = dtype_code(mn->scalar_type());
  const c10::Device device = codes->device();
  if (dtype < 0 || !one_pass(group, dtype) || codes->scalar_type() != at::kChar || codes->dim() != 1 || scale->device() != device ||
      mn->device() != device || scale->scalar_type() != (dtype == GACT_BF16 ? at::kFloat : mn->scalar_type()) ||
      !codes->is_contiguous() || !scale->is_contiguous() || !mn->is_contiguous() ||
      (group != kGroup && (scale->dim() != 3 || mn->dim() != 3)))
    Py_RETURN_NONE;
  const Py_ssize_t dims = PyTuple_GET_SIZE(args[1]);
  int64_t numel = 1;
  c10::SmallVector<int64_t, 8> shape;
  for (Py_ssize_t d = 0; d < dims; d++) {
    int64_t size;
    if (!integer(PyTuple_GET_ITEM(args[1], d), &size) || size <= 0 || __builtin_mul_overflow(numel, size, &numel)) Py_RETURN_NONE;
    shape.push_back(size);
  }
  if (numel > INT64_MAX / 2) Py_RETURN_NONE;
  const int64_t N = (numel + group - 1) / group;
  if (codes->numel() < packed_numel(bits, N, group) - 1 || scale->numel() < N || mn->numel() < N) Py_RETURN_NONE;
  const at::Tensor data = make(shape, mn->scalar_type(), device);
  const int rc = on(device, [&](void* stream) {
    if (group == kGroup) return gact_dequantize(in(*codes), bits, in(*scale), in(*mn), dtype, numel, out(data), stream);
    return gact_dequantize_groups(in(*codes), bits, in(*scale), in(*mn), dtype, numel, (int)group, out(data), stream);
  });
  if (rc == GACT_OK) return THPVariable_Wrap(data);
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// minimax(data[N, D]) -> (min[N], max[N])
PyObject* minimax(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const at::Tensor* x;
  if (n != 1 || !(x = plain(args[0])) || !x->is_contiguous() || !float_or_half(*x) || x->dim() != 2 || x->numel() == 0 || !ordinary_call())
    Py_RETURN_NONE;
  const int64_t N = x->size(0), D = x->size(1);
  if (D % 32 != 0 || D <= 32) Py_RETURN_NONE;
  const c10::Device device = x->device();
  const at::Tensor mn = make({N}, x->scalar_type(), device), mx = make({N}, x->scalar_type(), device);
  const int rc = on(device, [&](void* stream) { return gact_minimax(in(*x), dtype_code(x->scalar_type()), N, D, out(mn), out(mx), stream); });
  if (rc == GACT_OK) return tuple_of({mn, mx});
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// pack(data[N, G, D], min, max, bits, seed, noise mode) -> (codes, scale[N, G, 1])
PyObject* pack(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int bits, mode;
  uint64_t seed;
  const at::Tensor *x, *mn, *mx;
  if (n != 6 || !(x = plain(args[0])) || !(mn = plain(args[1])) || !(mx = plain(args[2])) || !width(args[3], &bits) ||
      !seed_of(args[4], &seed) || !noise_mode(args[5], &mode) || !ordinary_call())
    Py_RETURN_NONE;
  const c10::Device device = x->device();
  for (const at::Tensor* t : {x, mn, mx})
    if (!t->is_contiguous() || t->dim() != 3 || t->scalar_type() != x->scalar_type() || t->device() != device) Py_RETURN_NONE;
  const int64_t N = x->size(0), G = x->size(1), D = x->size(2);
  if (!float_or_half(*x) || x->numel() == 0 || mn->numel() != N * G || mx->numel() != N * G) Py_RETURN_NONE;
  const at::Tensor codes = make({packed_numel(bits, N, G * D)}, at::kChar, device), scale = make({N, G, 1}, x->scalar_type(), device);
  const int rc = on(device, [&](void* stream) {
    return gact_pack(in(*x), in(*mn), in(*mx), dtype_code(x->scalar_type()), bits, N, G, D, mode, seed, nullptr, out(codes), out(scale), stream);
  });
  if (rc == GACT_OK) return tuple_of({codes, scale});
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// unpack(codes, bits, scale, min, N, groups, group size) -> tensor[N, groups, group size]
PyObject* unpack(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int bits;
  int64_t N, G, D;
  const at::Tensor *codes, *scale, *mn;
  if (n != 7 || !(codes = plain(args[0])) || !width(args[1], &bits) || !(scale = plain(args[2])) || !(mn = plain(args[3])) ||
      !integer(args[4], &N) || !integer(args[5], &G) || !integer(args[6], &D) || !ordinary_call())
    Py_RETURN_NONE;
  const c10::Device device = codes->device();
  if (!codes->is_contiguous() || codes->dim() != 1 || codes->scalar_type() != at::kChar) Py_RETURN_NONE;
  for (const at::Tensor* t : {scale, mn})
    if (!t->is_contiguous() || t->dim() != 3 || !float_or_half(*t) || t->scalar_type() != scale->scalar_type() || t->device() != device)
      Py_RETURN_NONE;
  int64_t rows, numel;
  if (N <= 0 || G <= 0 || D <= 0 || __builtin_mul_overflow(N, G, &rows) || __builtin_mul_overflow(rows, D, &numel) ||
      numel > INT64_MAX / 16 || codes->numel() < packed_numel(bits, N, G * D) - 1 || scale->numel() < rows || mn->numel() < rows)
    Py_RETURN_NONE;
  const at::Tensor data = make({N, G, D}, scale->scalar_type(), device);
  const int rc = on(device, [&](void* stream) {
    return gact_unpack(in(*codes), bits, in(*scale), in(*mn), dtype_code(scale->scalar_type()), N, G, D, out(data), stream);
  });
  if (rc == GACT_OK) return THPVariable_Wrap(data);
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// mask_pack(0/1 bytes) -> int32[ceil(n/32)]
PyObject* mask_pack(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const at::Tensor* x;
  if (n != 1 || !(x = plain(args[0])) || !x->is_contiguous() || x->scalar_type() != at::kByte || x->numel() == 0 || !ordinary_call())
    Py_RETURN_NONE;
  const c10::Device device = x->device();
  const at::Tensor mask = make({(x->numel() + 31) / 32}, at::kInt, device);
  const int rc = on(device, [&](void* stream) { return gact_mask_pack((const uint8_t*)in(*x), x->numel(), (int32_t*)out(mask), stream); });
  if (rc == GACT_OK) return THPVariable_Wrap(mask);
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// mask_unpack(mask, n) -> uint8[n]
PyObject* mask_unpack(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const at::Tensor* mask;
  int64_t numel;
  if (n != 2 || !(mask = plain(args[0])) || !integer(args[1], &numel) || mask->scalar_type() != at::kInt || !mask->is_contiguous() || numel <= 0 ||
      numel > INT64_MAX / 2 || mask->numel() < (numel + 31) / 32 || !ordinary_call())
    Py_RETURN_NONE;
  const c10::Device device = mask->device();
  const at::Tensor data = make({numel}, at::kByte, device);
  const int rc = on(device, [&](void* stream) { return gact_mask_unpack((const int32_t*)in(*mask), numel, (uint8_t*)out(data), stream); });
  if (rc == GACT_OK) return THPVariable_Wrap(data);
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// batch_table(entries, tensors, seeds) -> the table as bytes on the host, in pinned memory: `entries` (bytes, one
// gact_batch_entry per tensor) with each tensor's address and seed filled in
PyObject* batch_table(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3 || !PyBytes_CheckExact(args[0]) || !PyList_CheckExact(args[1]) || !PyList_CheckExact(args[2]) || !ordinary_call()) Py_RETURN_NONE;
  const Py_ssize_t count = PyList_GET_SIZE(args[1]), bytes = PyBytes_GET_SIZE(args[0]);
  if (count == 0 || PyList_GET_SIZE(args[2]) != count || bytes != count * (Py_ssize_t)sizeof(gact_batch_entry)) Py_RETURN_NONE;
  const at::Tensor table = at::empty({(int64_t)bytes}, at::TensorOptions().dtype(at::kByte).pinned_memory(true));
  gact_batch_entry* const entry = (gact_batch_entry*)out(table);
  std::memcpy(entry, PyBytes_AS_STRING(args[0]), (size_t)bytes);
  for (Py_ssize_t i = 0; i < count; i++) {
    const at::Tensor* const t = plain(PyList_GET_ITEM(args[1], i));
    int64_t seed;
    if (!t || !integer(PyList_GET_ITEM(args[2], i), &seed) || t->numel() != entry[i].numel ||
        dtype_code(t->scalar_type()) != entry[i].dtype || !t->is_contiguous() || (reinterpret_cast<uintptr_t>(in(*t)) & 15u) != 0)
      Py_RETURN_NONE;
    entry[i].x = in(*t);
    entry[i].seed = (uint64_t)seed;
  }
  return THPVariable_Wrap(table);
  END_HANDLE_TH_ERRORS
}

// What both batched calls take first: entries (bytes, one gact_batch_entry per tensor) and the same on the GPU, the tensors, their seeds and
// the widths; false where anything is not as the launch needs it
struct Batch {
  int64_t count;
  const at::Tensor *geometry, *bits;
  c10::SmallVector<const void*, GACT_BATCH_ARGS> x;
  c10::SmallVector<uint64_t, GACT_BATCH_ARGS> seeds;
};
bool batch_of(PyObject* const* args, Batch* b) {
  if (!PyBytes_CheckExact(args[0]) || !(b->geometry = plain(args[1])) || !PyList_CheckExact(args[2]) || !PyList_CheckExact(args[3]) ||
      !(b->bits = plain(args[4])) || !ordinary_call())
    return false;
  const Py_ssize_t count = PyList_GET_SIZE(args[2]), bytes = PyBytes_GET_SIZE(args[0]);
  const c10::Device device = b->geometry->device();
  if (count == 0 || count > GACT_BATCH_ARGS || PyList_GET_SIZE(args[3]) != count || bytes != count * (Py_ssize_t)sizeof(gact_batch_entry) ||
      b->geometry->numel() != bytes || !b->geometry->is_contiguous() || b->bits->scalar_type() != at::kInt || b->bits->numel() != count ||
      !b->bits->is_contiguous() || b->bits->device() != device)
    return false;
  b->count = count;
  for (Py_ssize_t i = 0; i < count; i++) {
    gact_batch_entry entry;   // a bytes object promises no alignment
    std::memcpy(&entry, PyBytes_AS_STRING(args[0]) + i * sizeof entry, sizeof entry);
    const at::Tensor* const t = plain(PyList_GET_ITEM(args[2], i));
    int64_t seed;
    if (!t || !integer(PyList_GET_ITEM(args[3], i), &seed) || t->device() != device || t->numel() != entry.numel ||
        dtype_code(t->scalar_type()) != entry.dtype || !t->is_contiguous() || (reinterpret_cast<uintptr_t>(in(*t)) & 15u) != 0)
      return false;
    b->x.push_back(in(*t));
    b->seeds.push_back((uint64_t)seed);
  }
  return true;
}
// What outlives the call that made it - the geometry, all that a compressed batch holds - may be used on another stream and dropped before
// that stream gets to it: its memory waits for that stream too (the allocator passes over its own stream)
void used_on(const at::Tensor& t, c10::hip::HIPStream stream) { c10::hip::HIPCachingAllocator::recordStream(t.storage().data_ptr(), stream); }
bool capturing(c10::Device device) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing((hipStream_t)stream_on(device), &status) != hipSuccess || status != hipStreamCaptureStatusNone;
}

// What the plan says, two words in pinned memory (bytes the table needs, whether all is well) that its kernel writes through to the
// host: they are there as soon as both have changed from kUnwritten.  An event behind the plan said the same and kept the stream 6 us
// from the next kernel, as does the one that the allocator of pinned memory records where it is told of the stream.  calc_precision, quantize
// and dequantize, us, events / words: 40 bfloat16 tensors of 9 M elements together 42.6 / 35.2, 44 float 10 M 44.3 / 36.6, 69 half 16 M
// 44.5 / 39.3, 139 float 17 M 56.4 / 50.5, 20 bfloat16 83 M 92.6 / 86.3, 45 half 117 M 117.5 / 111.3, 119 float 168 M 260 / 253,
// 120 half 1.83 G 1329 / 1325.
constexpr int64_t kUnwritten = -1;
constexpr const char* kVerdict = "gact verdict";
struct Verdict {
  at::Tensor words;
  c10::Device device;
  hipStream_t stream;         // one of torch's, which live as long as the process
  hipEvent_t event = nullptr; // behind the plan, where the stream is not torch's own and may be gone before the wait
  ~Verdict() {
    if (event) (void)hipEventDestroy(event);
  }
};
int64_t word_of(const at::Tensor& words, int i) { return __atomic_load_n((const int64_t*)words.const_data_ptr() + i, __ATOMIC_ACQUIRE); }
bool written(const at::Tensor& words) { return word_of(words, 0) != kUnwritten && word_of(words, 1) != kUnwritten; }
// Words that a plan has still to write are not handed out again before it has: those of a verdict that is dropped earlier are held here
// until a later verdict comes or goes and finds them written.  As many as there are such plans under way; guarded by the GIL; never
// destroyed, as a plan may outlast the process's own objects.
void hold_unwritten(const at::Tensor* dropped) {
  static std::vector<at::Tensor>* const held = new std::vector<at::Tensor>;
  held->erase(std::remove_if(held->begin(), held->end(), written), held->end());
  if (dropped && !written(*dropped)) held->push_back(*dropped);
}
void drop_verdict(PyObject* capsule) {
  Verdict* const v = (Verdict*)PyCapsule_GetPointer(capsule, kVerdict);
  try {
    hold_unwritten(&v->words);
  } catch (...) {   // no memory to hold them in: they stay allocated
    (void)v->words.unsafeReleaseTensorImpl();
  }
  delete v;
}

// batch_quantize(entries, geometry, tensors, seeds, bits, (blocks, groups, workspace bytes, arena bytes, noise mode, element types)) ->
// ((codes, scale, min, table, widths kept, workspace), the plan's verdict for verdict_wait)
PyObject* batch_quantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Batch b;
  int64_t blocks, groups, ws_bytes, arena, mode, dtypes;
  if (n != 6 || !PyTuple_CheckExact(args[5]) || PyTuple_GET_SIZE(args[5]) != 6 || !integer(PyTuple_GET_ITEM(args[5], 0), &blocks) ||
      !integer(PyTuple_GET_ITEM(args[5], 1), &groups) || !integer(PyTuple_GET_ITEM(args[5], 2), &ws_bytes) ||
      !integer(PyTuple_GET_ITEM(args[5], 3), &arena) || !integer(PyTuple_GET_ITEM(args[5], 4), &mode) ||
      !integer(PyTuple_GET_ITEM(args[5], 5), &dtypes) || blocks <= 0 || arena <= 0 || !batch_of(args, &b))
    Py_RETURN_NONE;
  const c10::Device device = b.geometry->device();
  const c10::DeviceGuard guard(device);
  if (capturing(device)) Py_RETURN_NONE;
  const at::Tensor packed = make({arena}, at::kByte, device), scale = make({groups * 4}, at::kByte, device), mn = make({groups * 4}, at::kByte, device);
  const at::Tensor table = make({b.geometry->numel()}, at::kByte, device), kept = make(b.bits->sizes(), at::kInt, device), ws = make({ws_bytes}, at::kByte, device);
  hold_unwritten(nullptr);
  const at::Tensor words = at::empty({2}, at::TensorOptions().dtype(at::kLong).pinned_memory(true));
  const c10::hip::HIPStream stream = c10::hip::getCurrentHIPStream(device.index());
  used_on(*b.geometry, stream);
  int64_t* const word = (int64_t*)out(words);
  __atomic_store_n(word, kUnwritten, __ATOMIC_RELAXED);
  __atomic_store_n(word + 1, kUnwritten, __ATOMIC_RELEASE);
  Verdict* const verdict = new Verdict{words, device, stream.stream()};
  const THPObjectPtr capsule(PyCapsule_New(verdict, kVerdict, drop_verdict));
  if (!capsule) {
    delete verdict;
    return nullptr;
  }
  // torch's name for a stream that it was given is the stream's own handle
  const bool foreign = stream.stream() != nullptr && (int64_t)(intptr_t)stream.stream() == (int64_t)stream.id();
  int rc = GACT_ELAUNCH;
  {
    const WithoutGil released;
    if (!foreign || hipEventCreateWithFlags(&verdict->event, hipEventDisableTiming) == hipSuccess)
      rc = gact_batch_plan_args((const gact_batch_entry*)in(*b.geometry), b.x.data(), b.seeds.data(), (gact_batch_entry*)out(table),
                                (const int32_t*)in(*b.bits), (int32_t*)out(kept), b.count, blocks, arena, out(ws), word, stream.stream());
    if (rc != GACT_OK)
      word[0] = word[1] = 0;   // nobody will write them
    else if (foreign && hipEventRecord(verdict->event, stream.stream()) != hipSuccess)
      rc = GACT_ELAUNCH;
    else
      rc = gact_quantize_batched((const gact_batch_entry*)out(table), (const int32_t*)out(kept), b.count, blocks, (int)mode, (int)dtypes, out(ws),
                                 out(packed), out(scale), out(mn), stream.stream());
  }
  if (rc != GACT_OK) Py_RETURN_NONE;
  const THPObjectPtr tensors(tuple_of({packed, scale, mn, table, kept, ws}));
  return tensors ? PyTuple_Pack(2, tensors.get(), capsule.get()) : nullptr;
  END_HANDLE_TH_ERRORS
}

// Until the words are written, or cannot be any more.  A plan is a few microseconds behind what the stream has to do before it, so the
// thread keeps looking, as one that waits for an event does; after about a millisecond it lets others run in between (sleeps of
// 20 us came back 40 us late).  From then on it looks at the stream, too, every 50 ms or so, to end with it whatever became of it.
hipError_t wait_written(const Verdict& v) {
  if (v.event) return hipEventSynchronize(v.event);
  for (int64_t looks = 0; !written(v.words); looks++) {
    if (looks < 20000) {
      __builtin_ia32_pause();
      continue;
    }
    std::this_thread::yield();
    if ((looks - 20000) % (1 << 16) != 0) continue;
    const c10::DeviceGuard guard(v.device);
    // "not ready" is an error of its own to the runtime: it must not take the place of one that another call left for its caller
    const bool unread = hipPeekAtLastError() != hipSuccess;
    const hipError_t rc = unread ? hipStreamSynchronize(v.stream) : hipStreamQuery(v.stream);
    if (rc != hipErrorNotReady) return rc;
    if (hipPeekAtLastError() == hipErrorNotReady) (void)hipGetLastError();
  }
  return hipSuccess;
}

// verdict_wait(verdict of batch_quantize) -> (bytes the table needs, 1 where all is well), once the plan has run
PyObject* verdict_wait(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Verdict* const v = n == 1 ? (Verdict*)PyCapsule_GetPointer(args[0], kVerdict) : nullptr;
  if (!v) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "verdict_wait takes one verdict");
    return nullptr;
  }
  hipError_t rc;
  {
    const WithoutGil released;
    rc = wait_written(*v);
  }
  if (!written(v->words)) {
    PyErr_SetString(PyExc_RuntimeError, rc != hipSuccess ? hipGetErrorString(rc) : "gact: the plan of a batch did not run");
    return nullptr;
  }
  return Py_BuildValue("(LL)", (long long)word_of(v->words, 0), (long long)word_of(v->words, 1));
  END_HANDLE_TH_ERRORS
}

// batch_dequantize(entries, geometry, outputs, seeds, widths, codes, scale, min, table, workspace, (blocks, workspace bytes, element types)) -> True
PyObject* batch_dequantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Batch b;
  int64_t blocks, ws_bytes, dtypes;
  const at::Tensor *packed, *scale, *mn, *table, *ws;
  if (n != 11 || !(packed = plain(args[5])) || !(scale = plain(args[6])) || !(mn = plain(args[7])) || !(table = plain(args[8])) ||
      !(ws = plain(args[9])) || !PyTuple_CheckExact(args[10]) || PyTuple_GET_SIZE(args[10]) != 3 ||
      !integer(PyTuple_GET_ITEM(args[10], 0), &blocks) || !integer(PyTuple_GET_ITEM(args[10], 1), &ws_bytes) ||
      !integer(PyTuple_GET_ITEM(args[10], 2), &dtypes) || blocks <= 0 || !batch_of(args, &b))
    Py_RETURN_NONE;
  const c10::Device device = b.geometry->device();
  for (const at::Tensor* t : {packed, scale, mn, table, ws})
    if (t->scalar_type() != at::kByte || !t->is_contiguous() || t->device() != device) Py_RETURN_NONE;
  if (table->numel() != b.geometry->numel() || ws->numel() != ws_bytes || capturing(device)) Py_RETURN_NONE;
  const c10::hip::HIPStream stream = c10::hip::getCurrentHIPStream(device.index());
  for (const at::Tensor* t : {packed, scale, mn, table, ws, b.bits}) used_on(*t, stream);
  void* x[GACT_BATCH_ARGS];
  for (int64_t i = 0; i < b.count; i++) x[i] = const_cast<void*>(b.x[i]);
  const int rc = on(device, [&](void* stream) {
    return gact_dequantize_batched_to((const gact_batch_entry*)in(*table), x, (const int32_t*)in(*b.bits), b.count, blocks, (int)dtypes, in(*ws),
                                      in(*packed), in(*scale), in(*mn), stream);
  });
  if (rc == GACT_OK) Py_RETURN_TRUE;
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// ordinary() -> whether what is made now is what it will be later: no mode, transform or trace around the call
PyObject* ordinary(PyObject*, PyObject* const*, Py_ssize_t) {
  if (ordinary_call()) Py_RETURN_TRUE;
  Py_RETURN_FALSE;
}

#define FASTCALL(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FASTCALL(quantize), FASTCALL(dequantize), FASTCALL(minimax),     FASTCALL(pack),        FASTCALL(unpack),
                         FASTCALL(mask_pack), FASTCALL(mask_unpack), FASTCALL(batch_table),
                         FASTCALL(batch_quantize), FASTCALL(batch_dequantize), FASTCALL(verdict_wait),
                         FASTCALL(ordinary), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "gact_torch", "The operators' host side.", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_gact_torch(void) {
  static const char built_with[] = "torch " GACT_TORCH_VERSION;   // the build looks for it in the library
  PyObject* const m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", built_with + 6) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}

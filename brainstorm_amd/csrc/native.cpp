// Host side of the routing ops and the grouped GEMM: argument checks, output allocation and the call
// into libbrt_hip.so, for tensors handed over by Python (brainstorm_amd/_C/router.py and
// brainstorm_amd/jit are thin wrappers around these functions and document them).
//
// Why native: a routed layer is 4 to 7 launches of 2.7 us of host time each, and the same work in
// Python (a torch.empty is 1.7 us there and 0.4 us here, a foreign call with 17 converted arguments
// 3 us, every check 0.1 us) took longer than most layers take on the device.  Positional arguments
// only, no argument parser.
//
// Nothing is kept between calls: outputs and scratch memory come from torch's caching allocator, which
// knows the stream.  Errors are raised as the exceptions the reference's binding raises
// (src/backend/torch/torch.h:16-21, router.cc:266).
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/CachingHostAllocator.h>
#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/full.h>
#include <ATen/ops/zeros.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <chrono>
#include <stdexcept>
#include <string>
#include <vector>

#include "brt_hip.h"

namespace {

using at::Tensor;

unsigned long long g_calls = 0;  // calls into the library that queued device work (under the GIL)

// An error with the Python type it is raised as.
struct Raised : std::runtime_error {
  PyObject* type;
  Raised(PyObject* t, const std::string& what) : std::runtime_error(what), type(t) {}
};
[[noreturn]] void runtime_error(const std::string& what) { throw Raised(PyExc_RuntimeError, what); }
[[noreturn]] void index_error(const std::string& what) { throw Raised(PyExc_IndexError, what); }
[[noreturn]] void not_implemented(const std::string& what) { throw Raised(PyExc_NotImplementedError, what); }

void check(int code) {
  ++g_calls;
  if (code == BRT_OK) return;
  const std::string msg = brt_hip_last_error();
  if (code == BRT_E_UNSUPPORTED) not_implemented(msg);
  runtime_error("libbrt_hip error " + std::to_string(code) + ": " + msg);
}

// ---- arguments -----------------------------------------------------------------------------------
struct Args {
  PyObject* const* v;
  Py_ssize_t n;

  Tensor tensor(Py_ssize_t i) const {
    PyObject* const o = v[i];
    if (!THPVariable_CheckExact(o)) {
      if (!THPVariable_Check(o)) throw Raised(PyExc_TypeError, "a tensor is expected");
      // a subclass may stand for rows that are not there yet: asking for the address fills them
      PyObject* const address = PyObject_CallMethod(o, "data_ptr", nullptr);
      if (address == nullptr) throw Raised(nullptr, "");
      Py_DECREF(address);
    }
    return THPVariable_Unpack(o);
  }
  bool none(Py_ssize_t i) const { return v[i] == Py_None; }
  Tensor tensor_or_none(Py_ssize_t i) const { return none(i) ? Tensor() : tensor(i); }
  long integer(Py_ssize_t i) const {
    const long r = PyLong_AsLong(v[i]);
    if (r == -1 && PyErr_Occurred()) throw Raised(nullptr, "");
    return r;
  }
  bool flag(Py_ssize_t i) const {
    const int r = PyObject_IsTrue(v[i]);
    if (r < 0) throw Raised(nullptr, "");
    return r != 0;
  }
  bool dtype(Py_ssize_t i, at::ScalarType* out) const {
    if (none(i)) return false;
    if (!THPDtype_Check(v[i])) throw Raised(PyExc_TypeError, "a dtype is expected");
    *out = reinterpret_cast<THPDtype*>(v[i])->scalar_type;
    return true;
  }
};

PyObject* wrap(Tensor t) { return THPVariable_Wrap(std::move(t)); }
PyObject* none() { Py_RETURN_NONE; }
template <typename... T>
PyObject* tuple(T... items) {
  PyObject* const made[] = {items...};
  PyObject* const t = PyTuple_New(sizeof...(items));
  for (size_t i = 0; i < sizeof...(items); ++i) PyTuple_SET_ITEM(t, i, made[i]);
  return t;
}

void on_device(const Tensor& t, const char* name) {
  if (!t.is_cuda()) runtime_error(std::string(name) + " must be a CUDA tensor");
}
void int32(const Tensor& t, const char* name) {
  if (t.scalar_type() != at::kInt)
    runtime_error(std::string(name) + " must be an int32 tensor, got " + c10::toString(t.scalar_type()));
}
int64_t divided(int64_t a, int64_t b) {
  if (b == 0) throw Raised(PyExc_ZeroDivisionError, "no cells or no paths to divide by");
  return a / b;
}
int code_of(at::ScalarType t) {  // BRT_F32 / BRT_F16 / BRT_BF16, -1 for anything else
  return t == at::kFloat ? BRT_F32 : t == at::kHalf ? BRT_F16 : t == at::kBFloat16 ? BRT_BF16 : -1;
}
int data_type(const Tensor& t, const char* what) {
  const int c = code_of(t.scalar_type());
  if (c < 0) not_implemented(std::string(what) + " is not supported");
  return c;
}
Tensor dense(const Tensor& t) { return t.is_contiguous() ? t : t.contiguous(); }
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
int32_t* iptr(const Tensor& t) { return static_cast<int32_t*>(ptr(t)); }
float* fptr(const Tensor& t) { return static_cast<float*>(ptr(t)); }
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

Tensor empty(at::IntArrayRef shape, at::ScalarType type, const Tensor& like) {
  return Tensor(at::detail::empty_cuda(shape, type, like.device(), std::nullopt));
}
Tensor zeros(at::IntArrayRef shape, at::ScalarType type, const Tensor& like) {
  return at::zeros(shape, at::TensorOptions().dtype(type).device(like.device()));
}
Tensor scratch(size_t bytes, const Tensor& like) {
  return empty({static_cast<int64_t>(bytes < 16 ? 16 : bytes)}, at::kByte, like);
}
at::DimVector rows_of(const Tensor& t, int64_t rows) {  // the shape of t with another first dimension
  at::DimVector s(t.sizes().begin(), t.sizes().end());
  s[0] = rows;
  return s;
}

// The menu of capacities of an index generation.
struct Caps {
  Tensor t;
  int n = 0;
  Caps(const Tensor& given, bool padding) {
    if (given.defined()) {
      on_device(given, "supported_capacities");
      int32(given, "supported_capacities");
      t = dense(given);
      n = static_cast<int>(t.size(0));
    }
    if (padding && n < 1) runtime_error("capacity_padding requires at least one supported capacity");  // location.cu:350,365
  }
};

// ---- gate ------------------------------------------------------------------------------------------
Tensor scores(const Tensor& given, long top_k) {
  on_device(given, "score");
  if (given.dim() != 2) runtime_error("score must be [cells, paths]");
  data_type(given, "score data type");
  if (top_k < 0 || top_k > given.size(1)) runtime_error("selected index k out of range");  // the message torch.topk gives
  return dense(given);
}

PyObject* topk_hot_mask(const Args& a) {
  const long k = a.integer(1);
  const Tensor score = scores(a.tensor(0), k);
  const c10::DeviceGuard guard(score.device());
  Tensor mask = empty(score.sizes(), at::kInt, score);
  check(brt_hip_topk_hot_mask(ptr(score), iptr(mask), score.size(0), score.size(1), k, code_of(score.scalar_type()),
                              stream_of(score)));
  return wrap(mask);
}

PyObject* gate_topk(const Args& a) {  // score, k, softmax, hot_mask
  const long k = a.integer(1);
  const Tensor score = scores(a.tensor(0), k);
  const c10::DeviceGuard guard(score.device());
  const int64_t T = score.size(0);
  Tensor ids = empty({T, k}, at::kInt, score), weights = empty({T, k}, at::kFloat, score), mask;
  if (a.flag(3)) mask = empty(score.sizes(), at::kInt, score);
  if (k > 0 || mask.defined())
    check(brt_hip_gate_topk(ptr(score), T, score.size(1), k, code_of(score.scalar_type()), a.flag(2), iptr(ids),
                            fptr(weights), iptr(mask), stream_of(score)));
  return mask.defined() ? tuple(wrap(ids), wrap(weights), wrap(mask)) : tuple(wrap(ids), wrap(weights));
}

// ---- index generation --------------------------------------------------------------------------------
PyObject* throttle_hotmask(const Args& a) {  // hot_mask, prefix (updated in place), threshold
  const Tensor given = a.tensor(0), prefix = a.tensor(1), threshold = a.tensor(2);
  on_device(given, "hot_mask"), on_device(prefix, "prefix"), on_device(threshold, "threshold");
  int32(given, "hot_mask"), int32(prefix, "prefix"), int32(threshold, "threshold");
  if (given.dim() != 2) throw Raised(PyExc_ValueError, "hot_mask must be [cells, paths]");
  if (given.size(1) != prefix.size(0) || given.size(1) != threshold.size(0))
    runtime_error("prefix/threshold must have one entry per path");
  const Tensor mask = dense(given);
  const c10::DeviceGuard guard(mask.device());
  const int T = mask.size(0), E = mask.size(1);
  Tensor out = empty(mask.sizes(), at::kInt, mask);
  if (T > 0) {
    const size_t bytes = brt_hip_scan_workspace_bytes(T, E);
    const Tensor ws = scratch(bytes, mask), thr = dense(threshold);
    check(brt_hip_throttle_hotmask(iptr(mask), iptr(out), iptr(prefix), iptr(thr), T, E, ptr(ws), ws.numel(),
                                   stream_of(mask)));
  }
  return wrap(out);
}

// score, capacity -> (the top-1 hot mask throttled to it, the capacity of every path), or None where the fused
// kernels do not take the shape
PyObject* top1_to_capacity(const Args& a) {
  const Tensor score = scores(a.tensor(0), 1);
  const long capacity = a.integer(1);
  const int64_t T = score.size(0), E = score.size(1);
  if (T == 0 || E > 64 || capacity < 0 || capacity > INT32_MAX) return none();
  const c10::DeviceGuard guard(score.device());
  Tensor mask = empty(score.sizes(), at::kInt, score), out = empty(score.sizes(), at::kInt, score), caps = empty({E}, at::kInt, score);
  const Tensor ws = scratch(brt_hip_scan_workspace_bytes(T, E), score);
  check(brt_hip_top1_to_capacity(ptr(score), code_of(score.scalar_type()), iptr(mask), iptr(out), iptr(caps),
                                 static_cast<int>(capacity), T, E, ptr(ws), ws.numel(), stream_of(score)));
  return tuple(wrap(out), wrap(caps));
}

// ... and the route of the throttled mask: score, capacity, capacity_padding, path_wise_padding -> (mask, capacities, seats,
// loads, counts), or None likewise
PyObject* top1_route_to_capacity(const Args& a) {
  const Tensor score = scores(a.tensor(0), 1);
  const long capacity = a.integer(1);
  const int64_t T = score.size(0), E = score.size(1);
  if (T == 0 || E > 64 || capacity < 0 || capacity > INT32_MAX) return none();
  const c10::DeviceGuard guard(score.device());
  Tensor mask = empty(score.sizes(), at::kInt, score), out = empty(score.sizes(), at::kInt, score), caps = empty({E}, at::kInt, score);
  Tensor seats = empty(score.sizes(), at::kInt, score), loads = empty({E}, at::kInt, score), counts = empty({E}, at::kInt, score);
  const Tensor ws = scratch(brt_hip_scan_workspace_bytes(T, E), score);
  check(brt_hip_top1_route_to_capacity(ptr(score), code_of(score.scalar_type()), iptr(mask), iptr(out), iptr(seats), iptr(loads),
                                       iptr(counts), iptr(caps), static_cast<int>(capacity), a.flag(2), a.flag(3), T, E, ptr(ws),
                                       ws.numel(), stream_of(score)));
  return tuple(wrap(out), wrap(caps), wrap(seats), wrap(loads), wrap(counts));
}

PyObject* generate(const Args& a) {  // hot_mask, capacities, capacity_padding, path_wise_padding, is_tag_index
  const Tensor given = a.tensor(0);
  on_device(given, "hot_mask");
  int32(given, "hot_mask");
  const c10::DeviceGuard guard(given.device());
  const int64_t T = given.size(0), E = given.size(1);
  if (given.numel() == 0) {  // router.cc:59-62
    Tensor both = zeros({2, E}, at::kInt, given);
    return tuple(wrap(zeros({0, E}, at::kInt, given)), wrap(both.select(0, 0)), wrap(both.select(0, 1)));
  }
  const bool cap_pad = a.flag(2), path_pad = a.flag(3), tag = a.flag(4);
  const Caps caps(a.tensor_or_none(1), cap_pad);
  const Tensor mask = dense(given);
  Tensor indices = empty(mask.sizes(), at::kInt, mask);  // the kernel writes every element in both formats
  Tensor loads = empty({E}, at::kInt, mask), counts = empty({E}, at::kInt, mask);
  const Tensor ws = scratch(brt_hip_scan_workspace_bytes(T, E), mask);
  check(brt_hip_generate_indices_and_loads(iptr(mask), iptr(indices), iptr(loads), iptr(counts), T, E, iptr(caps.t),
                                           caps.n, cap_pad, path_pad, tag, ptr(ws), ws.numel(), stream_of(mask)));
  return tuple(wrap(indices), wrap(loads), wrap(counts));
}

// in_data, hot_mask, rows, capacities, capacity_padding, path_wise_padding, row_tags wanted
// -> (indices, loads, counts, out, row_tags), or None where the fused kernel does not take the shape
PyObject* route_and_dispatch(const Args& a) {
  const Tensor cells = a.tensor(0), given = a.tensor(1);
  on_device(cells, "in_data"), on_device(given, "hot_mask");
  int32(given, "hot_mask");
  const int64_t T = given.size(0), E = given.size(1), rows = a.integer(2);
  if (cells.size(0) != T) runtime_error("in_data and hot_mask must have one row per cell");
  const bool cap_pad = a.flag(4), path_pad = a.flag(5), want_tags = a.flag(6);
  const Tensor menu = a.tensor_or_none(3);
  const size_t cell_bytes = T > 0 ? cells.numel() / T * cells.element_size() : 0;
  // (a contiguous view whose storage offset breaks the 16-byte alignment takes the two calls)
  if (T == 0 || code_of(cells.scalar_type()) < 0 || reinterpret_cast<uintptr_t>(cells.data_ptr()) % 16 != 0 ||
      brt_hip_route_and_dispatch_supported(T, E, cell_bytes, menu.defined() ? menu.size(0) : 0, path_pad && cap_pad) != 1)
    return none();
  const c10::DeviceGuard guard(cells.device());
  const Caps caps(menu, cap_pad);
  const Tensor mask = dense(given), in = dense(cells);
  Tensor indices = empty(mask.sizes(), at::kInt, mask);
  Tensor loads = empty({E}, at::kInt, mask), counts = empty({E}, at::kInt, mask);
  Tensor out = empty(rows_of(in, rows), in.scalar_type(), in), tags;
  if (want_tags) tags = empty({rows}, at::kInt, in);
  const Tensor ws = scratch(brt_hip_route_and_dispatch_workspace_bytes(T, E, cell_bytes), in);
  check(brt_hip_route_and_dispatch(iptr(mask), ptr(in), ptr(out), iptr(indices), iptr(loads), iptr(counts), iptr(tags), T,
                                   E, rows, cell_bytes, iptr(caps.t), caps.n, cap_pad, path_pad, ptr(ws), ws.numel(),
                                   stream_of(in)));
  return tuple(wrap(indices), wrap(loads), wrap(counts), wrap(out), want_tags ? wrap(tags) : none());
}

PyObject* route_by_path(const Args& a) {  // path_ids, paths, capacities, cap_pad, path_pad, max_path_load, rows or None
  const Tensor given = a.tensor(0);
  on_device(given, "path_ids");
  int32(given, "path_ids");
  if (given.dim() != 2) runtime_error("path_ids must be [cells, k]");
  const Tensor ids = dense(given);
  const int64_t T = ids.size(0), k = ids.size(1), E = a.integer(1), mpl = a.integer(5);
  const int64_t rows = !a.none(6) ? a.integer(6) : mpl ? E * mpl : T * k;
  const c10::DeviceGuard guard(ids.device());
  Tensor caps = a.tensor_or_none(2);
  if (caps.defined()) {
    int32(caps, "supported_capacities");
    caps = dense(caps.device() == ids.device() ? caps : caps.to(ids.device()));
  }
  Tensor loads = empty({E}, at::kInt, ids), counts = empty({E}, at::kInt, ids);
  Tensor seat_rows = empty({T, k}, at::kInt, ids), row_entries = empty({rows}, at::kInt, ids);
  const Tensor ws = scratch(brt_hip_route_by_path_workspace_bytes(T, k, E), ids);
  check(brt_hip_route_by_path(iptr(ids), T, k, E, iptr(caps), caps.defined() ? caps.numel() : 0, a.flag(3), a.flag(4), mpl,
                              iptr(loads), iptr(counts), iptr(seat_rows), iptr(row_entries), rows, ptr(ws), ws.numel(),
                              stream_of(ids)));
  return tuple(wrap(loads), wrap(counts), wrap(seat_rows), wrap(row_entries));
}

// ---- host reads --------------------------------------------------------------------------------------
// Whether the word that a kernel sets behind its data is set, within the time that a program's next few launches
// would take; behind more work than that the caller waits for the stream, which does not keep a core busy.
bool seen_within(const int32_t* word, std::chrono::microseconds limit) {
  const auto end = std::chrono::steady_clock::now() + limit;
  do {
    for (int i = 0; i < 64; ++i) {
      if (__atomic_load_n(word, __ATOMIC_ACQUIRE) != 0) return true;
      __builtin_ia32_pause();
    }
  } while (std::chrono::steady_clock::now() < end);
  return false;
}

// Pinned memory for a few words that a kernel on the current stream stores, with a last one behind them that says that they are there
// (other Python threads run while this one waits).  Not watched: more words than a kernel stores quickly, or a stream that
// is being captured (where reading back is an error); these take the runtime's copy and wait.  The memory goes back to its
// allocator, which knows nothing of the stream, only when nothing that is queued stores to it any more, also where an
// exception ends the use between request and read.
struct HostWords {
  at::DataPtr host;
  hipStream_t st;
  size_t bytes;
  const char* what;
  int32_t* seen_from_device = nullptr;  // non-null: watched
  bool queued = false;                  // something that stores here may be

  HostWords(const Tensor& t, size_t n, const char* name) : bytes(n), what(name) {
    constexpr size_t kFewBytes = 4096;
    host = at::getHostAllocator(at::kCUDA)->allocate(bytes + 4);
    st = c10::hip::getCurrentHIPStream(t.get_device()).stream();
    if (bytes > kFewBytes || bytes % 4 != 0) return;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    void* address = nullptr;
    if (hipStreamIsCapturing(st, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone ||
        hipHostGetDevicePointer(&address, host.get(), 0) != hipSuccess) {
      (void)hipGetLastError();  // what asking left behind, if anything
      return;
    }
    seen_from_device = static_cast<int32_t*>(address);
    __atomic_store_n(word(), 0, __ATOMIC_RELEASE);
  }
  HostWords(const HostWords&) = delete;
  ~HostWords() {
    if (!queued) return;
    hipError_t rc;
    Py_BEGIN_ALLOW_THREADS
    rc = hipStreamSynchronize(st);
    Py_END_ALLOW_THREADS
    if (rc != hipSuccess) {
      (void)hipGetLastError();
      (void)host.release_context();  // kept for ever: what became of the stores is not known
    }
  }
  int32_t* word() const { return static_cast<int32_t*>(host.get()) + bytes / 4; }

  // A kernel that copies the words of a watched stream.
  void request(const Tensor& t) {
    if (seen_from_device == nullptr) return;
    ++g_calls;
    queued = true;
    if (brt_hip_copy_to_host(iptr(t), seen_from_device, static_cast<int>(bytes / 4), st) != BRT_OK)
      runtime_error(std::string(what) + ": " + brt_hip_last_error());
  }

  // Waits for the words of a watched stream; of another, copies them from the device first.
  const void* read(const Tensor& t) {
    hipError_t rc = hipSuccess;
    bool seen = false;
    if (seen_from_device != nullptr) {
      Py_BEGIN_ALLOW_THREADS
      seen = seen_within(word(), std::chrono::microseconds(500));
      Py_END_ALLOW_THREADS
    } else {
      queued = true;
      rc = hipMemcpyAsync(host.get(), ptr(t), bytes, hipMemcpyDeviceToHost, st);
    }
    if (rc == hipSuccess && !seen) {
      Py_BEGIN_ALLOW_THREADS
      rc = hipStreamSynchronize(st);
      Py_END_ALLOW_THREADS
    }
    if (rc != hipSuccess) {
      (void)hipGetLastError();  // reported here, not by the next launch that looks for an error
      runtime_error(std::string(what) + ": " + hipGetErrorString(rc));
    }
    queued = false;
    return host.get();
  }
};

// Copies from the device on the current stream into pinned memory and waits for the copy.
at::DataPtr read_back(const Tensor& t, size_t bytes, const char* what) {
  HostWords words(t, bytes, what);
  words.request(t);
  words.read(t);
  return std::move(words.host);
}

PyObject* list_of(const int32_t* values, int64_t n) {
  PyObject* const list = PyList_New(n);
  for (int64_t i = 0; i < n; ++i) PyList_SET_ITEM(list, i, PyLong_FromLong(values[i]));
  return list;
}

// ---- rows --------------------------------------------------------------------------------------------
void take_gates_and_tags(Tensor& gates, Tensor& old_tags, const Tensor& in, const Tensor& route) {
  if (gates.defined()) {
    on_device(gates, "gates");
    if (gates.scalar_type() != in.scalar_type()) runtime_error("gates must have the dtype of in_data");  // router.cc:226
    gates = dense(gates);
  }
  if (old_tags.defined()) {
    on_device(old_tags, "tags");
    if (old_tags.scalar_type() != route.scalar_type()) runtime_error("tags must have the dtype of route_indices");
    old_tags = dense(old_tags);
  }
}

// in_data, route_indices, loads (on the device), counts, gates, old_tags, tags wanted, rows of the output,
// max_path_load, is_1d_routing, is_tag_index, outputs pre-zeroed -> (out, new_tags or None)
PyObject* dispatch(const Args& a) {
  const Tensor given = a.tensor(0), route = dense(a.tensor(1)), loads = a.tensor(2), counts = a.tensor_or_none(3);
  Tensor gates = a.tensor_or_none(4), old_tags = a.tensor_or_none(5);
  const bool want_tags = a.flag(6), one_d = a.flag(9), tag_index = a.flag(10), clear = a.flag(11);
  const int64_t total = a.integer(7), mpl = a.integer(8);
  const Tensor in = dense(given);
  const c10::DeviceGuard guard(in.device());
  const int64_t T = in.size(0), E = route.size(1);
  int64_t cell = divided(in.numel(), T);
  at::DimVector shape(in.sizes().begin(), in.sizes().end());
  if (one_d) {
    shape[0] = total;
  } else {
    cell = divided(cell, E);
    if (shape.size() < 2) index_error("2-d routing needs a [cells, paths, ...] input");
    if (shape.size() == 2) shape.push_back(1);
    shape[1] = total;
    shape.erase(shape.begin());
  }
  Tensor out = clear ? zeros(shape, in.scalar_type(), in) : empty(shape, in.scalar_type(), in);
  if (gates.defined() && !one_d) runtime_error("gates are only supported with 1-d routing");  // route.cu:362
  take_gates_and_tags(gates, old_tags, in, route);
  Tensor tags;
  if (want_tags) tags = clear ? zeros({total}, at::kInt, in) : empty({total}, at::kInt, in);
  check(brt_hip_dispatch(ptr(in), ptr(out), ptr(gates), iptr(route), iptr(loads), iptr(counts), iptr(old_tags), iptr(tags),
                         T, cell, E, total, mpl, one_d, tag_index, code_of(in.scalar_type()), stream_of(in)));
  return tuple(wrap(out), want_tags ? wrap(tags) : none());
}

// in_data, route_indices, loads, counts, gates, old_tags, tags wanted, rows that will do -> (out, new_tags or None, the loads as a list).
// The rows of the output are the sum of the loads, which the host has to wait for.  Meanwhile the rows are moved into room for as many
// as will do by what the caller knows, and the result is cut to the sum; where they did not do, they are moved again, and where the
// device has no memory for the room, they are moved once the sum is known.  (1-d seat routing, packed.)
PyObject* dispatch_and_read(const Args& a) {
  const Tensor given = a.tensor(0), route = dense(a.tensor(1)), loads = dense(a.tensor(2)), counts = a.tensor(3);
  Tensor gates = a.tensor_or_none(4), old_tags = a.tensor_or_none(5), out, tags;
  const bool want_tags = a.flag(6);
  const int64_t room = a.integer(7);
  const Tensor in = dense(given);
  int32(loads, "loads");
  const c10::DeviceGuard guard(in.device());
  const int64_t T = in.size(0), E = route.size(1), cell = divided(in.numel(), T);
  if (loads.numel() != E) runtime_error("loads must have one entry per path");
  take_gates_and_tags(gates, old_tags, in, route);
  auto make_room = [&](int64_t rows) {
    out = tags = Tensor();
    out = empty(rows_of(in, rows), in.scalar_type(), in);
    if (want_tags) tags = empty({rows}, at::kInt, in);
  };
  auto move_rows = [&](int64_t rows) {
    check(brt_hip_dispatch(ptr(in), ptr(out), ptr(gates), iptr(route), iptr(loads), iptr(counts), iptr(old_tags), iptr(tags), T, cell, E, rows, 0,
                           1, 0, code_of(in.scalar_type()), stream_of(in)));
  };
  HostWords words(loads, E * 4, "reading the loads");
  words.request(loads);
  bool ahead = words.seen_from_device != nullptr;
  if (ahead) {
    try {
      make_room(room);
    } catch (const c10::OutOfMemoryError&) {
      ahead = false;
    }
  }
  if (ahead) move_rows(room);
  const int32_t* const v = static_cast<const int32_t*>(words.read(loads));
  int64_t total = 0;
  for (int64_t e = 0; e < E; ++e) total += v[e];
  if (!ahead || total > room) {
    make_room(total);
    move_rows(total);
  } else if (total < room) {  // the storage ends with the rows too: it is saved and compared whole
    auto cut = [](const Tensor& t, at::IntArrayRef shape) {
      t.unsafeGetTensorImpl()->set_sizes_contiguous(shape);
      t.storage().unsafeGetStorageImpl()->set_nbytes(t.nbytes());
    };
    cut(out, rows_of(in, total));
    if (want_tags) cut(tags, {total});
  }
  return tuple(wrap(out), want_tags ? wrap(tags) : none(), list_of(v, E));
}

// in_data, route_indices, loads, gates, out_data, out_dtype, max_path_padding, row_tags (a single-path route whose
// rows carry the tags of the paired dispatch, laid out as in_data is) -> the combined cells
PyObject* combine(const Args& a) {
  const Tensor in = dense(a.tensor(0)), route = dense(a.tensor(1));
  Tensor gates = a.tensor_or_none(3);
  const Tensor residual = a.tensor_or_none(4), given_loads = a.tensor(2);
  int32(route, "route_indices");
  int32(given_loads, "loads");
  const int in_type = data_type(in, "data type");
  const c10::DeviceGuard guard(in.device());
  const int64_t T = route.size(0), E = route.size(1), P = in.size(0), cell = P > 0 ? in.numel() / P : 0;
  const int64_t mpl = a.flag(6) ? divided(P, E) : 0;  // router.cc:427-430
  if (gates.defined()) {
    on_device(gates, "gates");
    data_type(gates, "gate data type");
    gates = dense(gates);
  }
  Tensor out = residual;
  if (residual.defined()) {
    on_device(residual, "out_data");
    if (!residual.is_contiguous()) runtime_error("out_data must be contiguous (it is updated in place)");
  } else {
    at::ScalarType type = in.scalar_type();
    a.dtype(5, &type);
    out = empty(rows_of(in, T), type, in);
  }
  const int out_type = code_of(out.scalar_type());
  if (out_type < 0 || out.numel() != T * cell) runtime_error("out_data does not match [cell_num, *cell_shape]");
  // scatter form (identical rows; cells without a row keep the residual, or become zero)
  const bool scatters = !gates.defined() && !a.none(7) && cell * in.element_size() % 16 == 0 && (out_type == in_type || out_type == BRT_F32);
  if (scatters && residual.defined()) {
    const Tensor tags = a.tensor(7);
    check(brt_hip_combine_by_tags(ptr(in), ptr(out), iptr(tags), P, cell, T, in_type, out_type, stream_of(in)));
    return wrap(out);
  }
  const Tensor loads =
      dense(given_loads.device() == in.device() ? given_loads : given_loads.to(in.options().dtype(at::kInt), /*non_blocking=*/true));
  // Results that fill the last-level cache are written better in order (us, bf16 cells over 8 paths of which all, nine and five of ten have a
  // row, scatter and gather form: 16384 of 8192 elements 109, 105 and 69, and 104, 97 and 63; of 6000, 197 MB, 85, 81 and 53, and
  // 83, 78 and 46; 131072 of 512, 134 MB, 46, 44 and 35, and 56, 43 and 33; 16384 of 2048, 67 MB, 23, 21 and 19, and 24, 23 and 19).
  constexpr int64_t kMostScattered = 5ll << 25;
  if (scatters && E <= 64 && reinterpret_cast<uintptr_t>(ptr(in)) % 16 == 0 && out.numel() * out.element_size() < kMostScattered) {
    const Tensor tags = a.tensor(7);
    check(brt_hip_combine_by_tags_cleared(ptr(in), ptr(out), iptr(tags), iptr(route), iptr(loads), T, cell, E, P, mpl, in_type, out_type,
                                          stream_of(in)));
  } else {
    check(brt_hip_combine(ptr(in), ptr(out), ptr(gates), iptr(route), iptr(loads), T, cell, E, P, mpl, residual.defined(),
                          in_type, out_type, gates.defined() ? code_of(gates.scalar_type()) : BRT_F32, stream_of(in)));
  }
  return wrap(out);
}

PyObject* combine_by_row_tags(const Args& a) {  // in_data, row_tags, cells, out_data, out_dtype
  const Tensor given = a.tensor(0), tags = a.tensor(1), residual = a.tensor_or_none(3);
  on_device(given, "in_data");
  const int in_type = data_type(given, "data type");
  const Tensor in = dense(given);
  const c10::DeviceGuard guard(in.device());
  const int64_t P = in.size(0), cells = a.integer(2), cell = P > 0 ? in.numel() / P : 0;
  Tensor out = residual;
  if (residual.defined()) {
    if (!residual.is_contiguous()) runtime_error("out_data must be contiguous (it is updated in place)");
  } else {
    at::ScalarType type = in.scalar_type();
    a.dtype(4, &type);
    out = zeros(rows_of(in, cells), type, in);
  }
  if (code_of(out.scalar_type()) < 0 || out.numel() != cells * cell)
    runtime_error("out_data does not match [cell_num, *cell_shape]");
  if (tags.numel() < P) runtime_error("one tag per row is needed");
  check(brt_hip_combine_by_tags(ptr(in), ptr(out), iptr(tags), P, cell, cells, in_type, code_of(out.scalar_type()),
                                stream_of(in)));
  return wrap(out);
}

Tensor entry_weights(const Tensor& given, int64_t entries) {
  if (!given.defined()) return given;
  if (given.scalar_type() != at::kFloat || given.numel() != entries) runtime_error("weights must be fp32 [cells, k]");
  return dense(given);
}

PyObject* dispatch_by_rows(const Args& a) {  // in_data, row_entries, k, weights, out
  const Tensor given = a.tensor(0), entries_given = a.tensor(1);
  on_device(given, "in_data"), on_device(entries_given, "row_entries");
  int32(entries_given, "row_entries");
  const int type = data_type(given, "in_data data type");
  const Tensor in = dense(given), entries = dense(entries_given);
  const int64_t T = in.size(0), cell = T > 0 ? in.numel() / T : 0, P = entries.numel(), k = a.integer(2);
  const Tensor weights = entry_weights(a.tensor_or_none(3), T * k);
  const c10::DeviceGuard guard(in.device());
  Tensor out = a.tensor_or_none(4);
  if (!out.defined()) out = empty(rows_of(in, P), in.scalar_type(), in);
  else if (out.scalar_type() != in.scalar_type() || !out.is_contiguous() || out.numel() != P * cell || out.device() != in.device())
    runtime_error("out must be a contiguous [rows, *cell_shape] tensor of the input's type");
  check(brt_hip_dispatch_by_rows(ptr(in), ptr(out), fptr(weights), iptr(entries), P, T, k, cell, type, stream_of(in)));
  return wrap(out);
}

PyObject* combine_by_rows(const Args& a) {  // in_data, path_ids, seat_rows, weights, out_data, out_dtype, gates
  const Tensor given = a.tensor(0), ids_given = a.tensor(1), seats_given = a.tensor(2), residual = a.tensor_or_none(4);
  on_device(given, "in_data"), on_device(ids_given, "path_ids");
  int32(ids_given, "path_ids");
  on_device(seats_given, "seat_rows");
  int32(seats_given, "seat_rows");
  const int in_type = data_type(given, "in_data data type");
  if (ids_given.sizes() != seats_given.sizes() || ids_given.dim() != 2)
    runtime_error("path_ids and seat_rows must both be [cells, k]");
  const Tensor in = dense(given), ids = dense(ids_given), seats = dense(seats_given);
  const int64_t T = ids.size(0), k = ids.size(1), P = in.size(0);
  const int64_t cell = P > 0 ? in.numel() / P : residual.defined() && T > 0 ? residual.numel() / T : 0;
  const Tensor weights = entry_weights(a.tensor_or_none(3), T * k);
  const c10::DeviceGuard guard(in.device());
  Tensor out = residual;
  if (residual.defined()) {
    if (!residual.is_contiguous() || residual.numel() != T * cell) runtime_error("out_data must be a contiguous [cells, ...] tensor");
  } else {
    at::ScalarType type = in.scalar_type();
    a.dtype(5, &type);
    out = empty(rows_of(in, T), type, in);
  }
  const int out_type = code_of(out.scalar_type());
  if (out_type < 0 || (out_type != in_type && out_type != BRT_F32)) not_implemented("output data type is not supported");
  Tensor gates = a.tensor_or_none(6);
  if (gates.defined()) {
    on_device(gates, "gates");
    const int gate_type = data_type(gates, "gate data type");
    if (gates.dim() != 2 || gates.size(0) != T) runtime_error("gates must be [cells, paths]");
    gates = dense(gates);
    check(brt_hip_combine_by_rows_gated(ptr(in), ptr(out), ptr(gates), gate_type, gates.size(1), iptr(ids), iptr(seats), T, k,
                                        cell, P, residual.defined(), in_type, out_type, stream_of(in)));
    return wrap(out);
  }
  check(brt_hip_combine_by_rows(ptr(in), ptr(out), fptr(weights), iptr(ids), iptr(seats), T, k, cell, P, residual.defined(),
                                in_type, out_type, stream_of(in)));
  return wrap(out);
}

// ---- grouped GEMM ------------------------------------------------------------------------------------
Tensor rounded_to_bf16(const Tensor& given) {
  const Tensor in = dense(given);
  const c10::DeviceGuard guard(in.device());
  Tensor out = empty(in.sizes(), at::kBFloat16, in);
  if (in.numel() > 0) check(brt_hip_cast_f32_to_bf16(fptr(in), ptr(out), in.numel(), stream_of(in)));
  return out;
}

// x, out, weight_table, bias_table, loads, in_features, out_features, activation code, tags, gather, scatter,
// rows or None, row_entries, entries_per_cell, row_tags_out, gates
// takes_f32: fp32 rows of x are taken too, rounded to bf16 by the GEMM itself where its kernel does that
PyObject* grouped_linear_of(const Args& a, bool takes_f32) {
  Tensor x = a.tensor(0);
  const bool f32_rows = takes_f32 && x.scalar_type() == at::kFloat && x.is_cuda();
  if (f32_rows) x = dense(x);
  const Tensor out = a.tensor(1), weights = a.tensor(2), biases = a.tensor_or_none(3), loads = a.tensor(4);
  const int64_t K = a.integer(5), N = a.integer(6), act = a.integer(7);
  const Tensor tags = a.tensor_or_none(8), entries = a.tensor_or_none(12), tags_out = a.tensor_or_none(14), gates = a.tensor_or_none(15);
  const bool gather = a.flag(9), scatter = a.flag(10), routed = gather || scatter;
  const int64_t k = a.integer(13);
  if ((x.scalar_type() != at::kBFloat16 && !f32_rows) || (out.scalar_type() != at::kBFloat16 && out.scalar_type() != at::kFloat))
    not_implemented("the grouped GEMM computes in bf16 (fp32 accumulation); the output is bf16 or fp32");
  const bool f32_out = out.scalar_type() == at::kFloat;
  if (gates.defined()) {
    if (!(scatter && f32_out)) runtime_error("gates fold the weighted combine into the store: scatter=True and an fp32 out");
    if (!gates.is_cuda() || gates.scalar_type() != at::kFloat || !gates.is_contiguous())
      runtime_error("gates must be a contiguous fp32 device tensor");
  } else if (f32_out && entries.defined()) {
    not_implemented("the row-entry form writes bf16");
  }
  if (!(x.is_cuda() && out.is_cuda() && loads.is_cuda())) runtime_error("grouped_linear needs device tensors");
  if (loads.scalar_type() != at::kInt) runtime_error("capacities must be int32");
  if (!(x.is_contiguous() && out.is_contiguous())) runtime_error("shared inputs must be contiguous");
  if (x.numel() != x.size(0) * K || out.numel() != out.size(0) * N)
    runtime_error("shared inputs do not match [rows, in_features] / [rows, out_features]");
  int64_t cells = 0, rows = a.none(11) ? -1 : a.integer(11);
  const bool by_rows = routed && entries.defined();
  if (by_rows) {
    if (!entries.is_cuda() || entries.scalar_type() != at::kInt || !entries.is_contiguous())
      runtime_error("row_entries must be a contiguous int32 vector on the device");
    if (gather && scatter && x.size(0) != out.size(0)) runtime_error("a gathered input / scattered output has one row per cell");
    cells = gather ? x.size(0) : out.size(0);
    if (rows < 0) rows = entries.numel();
    else if (rows > entries.numel()) runtime_error("rows exceeds the row-entry vector");
  } else if (routed) {
    if (!tags.defined() || !tags.is_cuda() || tags.scalar_type() != at::kInt || !tags.is_contiguous())
      runtime_error("gather/scatter need the contiguous int32 tag-index matrix on the device");
    cells = tags.size(0);
    if (tags.size(1) != loads.numel()) runtime_error("tags must have one column per branch");
    if ((gather && x.size(0) != cells) || (scatter && out.size(0) != cells))
      runtime_error("a gathered input / scattered output has one row per cell");
  }
  if (rows < 0) {
    // neither side path-major: nothing bounds the rows but the caller (the slots of the tag matrix would
    // launch a grid that is almost all empty row blocks)
    if (gather && scatter) runtime_error("rows (an upper bound of sum(loads)) is needed when x is gathered and out scattered");
    rows = scatter ? x.size(0) : out.size(0);
  } else if ((!gather && rows > x.size(0)) || (!scatter && rows > out.size(0))) {
    runtime_error("rows exceeds the path-major buffer");
  }
  if (!routed && x.size(0) != out.size(0)) runtime_error("shared inputs must have the same number of rows");
  const c10::DeviceGuard guard(x.device());
  void* const st = stream_of(x);
  const void* const* const w = static_cast<const void* const*>(ptr(weights));
  const void* const* const b = static_cast<const void* const*>(ptr(biases));
  const int E = static_cast<int>(loads.numel());
  if (f32_rows) {
    if (!scatter && !gates.defined() && brt_hip_grouped_gemm_f32in_supported(E, rows, cells, K, N, gather) == 1) {
      if (gather && !by_rows && tags_out.defined() && (tags_out.scalar_type() != at::kInt || tags_out.numel() < rows || !tags_out.is_cuda()))
        runtime_error("row_tags_out must be an int32 device vector with one entry per row");
      check(brt_hip_grouped_gemm_f32in(fptr(x), w, b, ptr(out), f32_out, iptr(loads), gather ? iptr(by_rows ? entries : tags) : nullptr,
                                       by_rows ? k : 0, E, rows, cells, K, N, act, gather, by_rows ? nullptr : iptr(tags_out), st));
      return none();
    }
    x = rounded_to_bf16(x);
  }
  if (gates.defined()) {
    if (gates.numel() != cells * (by_rows ? k : E))
      runtime_error("gates must hold one weight per cell and path (tags) or per entry (row_entries)");
    check(brt_hip_grouped_gemm_accumulate(ptr(x), w, b, fptr(out), iptr(loads), iptr(by_rows ? entries : tags), by_rows ? k : 0,
                                          fptr(gates), E, rows, cells, K, N, act, gather, st));
  } else if (by_rows) {
    check(brt_hip_grouped_gemm_by_rows(ptr(x), w, b, ptr(out), iptr(loads), iptr(entries), k, E, rows, cells, K, N, act, gather,
                                       scatter, st));
  } else if (routed) {
    if (tags_out.defined() && (tags_out.scalar_type() != at::kInt || tags_out.numel() < rows || !tags_out.is_cuda()))
      runtime_error("row_tags_out must be an int32 device vector with one entry per row");
    if (f32_out)
      check(brt_hip_grouped_gemm_routed_f32out(ptr(x), w, b, fptr(out), iptr(loads), iptr(tags), E, rows, cells, K, N, act, gather,
                                               scatter, iptr(tags_out), st));
    else
      check(brt_hip_grouped_gemm_routed(ptr(x), w, b, ptr(out), iptr(loads), iptr(tags), E, rows, cells, K, N, act, gather,
                                        scatter, iptr(tags_out), st));
  } else if (f32_out) {
    check(brt_hip_grouped_gemm_f32out(ptr(x), w, b, fptr(out), iptr(loads), E, rows, K, N, act, st));
  } else {
    check(brt_hip_grouped_gemm(ptr(x), w, b, ptr(out), iptr(loads), E, rows, K, N, act, st));
  }
  return none();
}

PyObject* grouped_linear(const Args& a) { return grouped_linear_of(a, false); }
PyObject* grouped_linear_f32(const Args& a) { return grouped_linear_of(a, true); }

// operands (list or tuple), first, step, branches used, what -> (fp32, key): the tensors operands[first::step],
// of which the used ones are all contiguous bf16 or all fp32, and what tells whether they are still the same
// ones as at another call -- for bf16 the addresses of all of them; for fp32 also the object, the version
// counter and the storage of each used one (`.data = ...` swaps the storage without touching the counter).
PyObject* branch_key(const Args& a) {
  PyObject* const seq = a.v[0];
  if (!PyList_Check(seq) && !PyTuple_Check(seq)) throw Raised(PyExc_TypeError, "a list or tuple of branch operands is expected");
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq), first = a.integer(1), step = a.integer(2), used = a.integer(3);
  PyObject* const* const items = PySequence_Fast_ITEMS(seq);
  std::vector<uint64_t> key;
  key.reserve(4 * n / step + 4);
  bool fp32 = false;
  Py_ssize_t b = 0;
  for (Py_ssize_t i = first; i < n; i += step, ++b) {
    if (fp32 && b >= used) break;  // branches past the capacities are never read, nor converted
    if (!THPVariable_Check(items[i])) throw Raised(PyExc_TypeError, "branch operands are tensors");
    const Tensor& t = THPVariable_Unpack(items[i]);
    if (b < used) {
      const bool f = t.scalar_type() == at::kFloat;
      if (b == 0) fp32 = f, key.push_back(f);
      if (f != fp32 || (!f && (t.scalar_type() != at::kBFloat16 || !t.is_contiguous()))) {
        PyObject* const what = PyObject_Str(a.v[4]);
        const std::string name = what != nullptr ? PyUnicode_AsUTF8(what) : "operands";
        Py_XDECREF(what);
        not_implemented("branch " + name + " must be contiguous bf16 or fp32 tensors of one dtype");
      }
    }
    key.push_back(reinterpret_cast<uint64_t>(t.data_ptr()));
    if (fp32) {
      key.push_back(reinterpret_cast<uint64_t>(items[i]));
      key.push_back(static_cast<uint64_t>(t._version()));
      key.push_back(reinterpret_cast<uint64_t>(t.storage().data()));
    }
  }
  return tuple(PyBool_FromLong(fp32), PyBytes_FromStringAndSize(reinterpret_cast<const char*>(key.data()), key.size() * 8));
}

PyObject* cast_f32_to_bf16(const Args& a) {
  const Tensor given = a.tensor(0);
  if (given.scalar_type() != at::kFloat)
    runtime_error(std::string("the cast kernel reads fp32, got ") + c10::toString(given.scalar_type()));
  return wrap(rounded_to_bf16(given));
}

// ---- values on the host ------------------------------------------------------------------------------
// The values of an int32 vector as a list.
PyObject* int_list(const Args& a) {
  const Tensor given = a.tensor(0);
  int32(given, "loads");
  const Tensor t = dense(given);
  const int64_t n = t.numel();
  const int32_t* values = nullptr;
  at::DataPtr host;
  // a tensor that only stands for others (of the meta device, or under a fake-tensor mode) has no values
  if (n > 0 && ptr(t) == nullptr) not_implemented("Cannot copy out of a tensor without data");
  if (n > 0 && t.is_cuda()) {
    const c10::DeviceGuard guard(t.device());
    host = read_back(t, n * 4, "reading the loads");
    values = static_cast<const int32_t*>(host.get());
  } else if (n > 0) {
    values = iptr(t);
  }
  return list_of(values, n);
}

// tags (a vector of 1 to BRT_UNIQUE_WHOLE_MAX int32 or int64 on the device) -> (unique, inverse, lo, hi), the first
// two None where the range is more than one workgroup's table holds
PyObject* unique_tags(const Args& a) {
  const Tensor tags = dense(a.tensor(0));
  on_device(tags, "tags");
  const bool narrow = tags.scalar_type() == at::kInt;
  if (!narrow && tags.scalar_type() != at::kLong) runtime_error("tags must be int32 or int64");
  const c10::DeviceGuard guard(tags.device());
  const int64_t n = tags.numel();
  Tensor unique = empty({n}, tags.scalar_type(), tags), inverse = empty({n}, at::kLong, tags), found = empty({3}, at::kLong, tags);
  check(brt_hip_unique_tags_whole(ptr(tags), narrow ? 32 : 64, n, ptr(unique), static_cast<int64_t*>(ptr(inverse)),
                                  static_cast<int64_t*>(ptr(found)), stream_of(tags)));
  const at::DataPtr host = read_back(found, 24, "reading the number of tags");
  const int64_t* const v = static_cast<const int64_t*>(host.get());
  PyObject *const lo = PyLong_FromLongLong(v[1]), *const hi = PyLong_FromLongLong(v[2]);
  if (v[0] < 0) return tuple(none(), none(), lo, hi);
  return tuple(wrap(unique.narrow(0, 0, v[0])), wrap(inverse), lo, hi);
}

// ---- tensors that carry a route ----------------------------------------------------------------------
// (neither reads the rows: a buffer that is not filled yet stays so)
const Tensor& as_it_is(PyObject* o) {
  if (!THPVariable_Check(o)) throw Raised(PyExc_TypeError, "a tensor is expected");
  return THPVariable_Unpack(o);
}

// Whether a view made here is what the same call from Python makes: no mode or tracer looks on at torch's calls, and
// the tensor does not answer them in Python.  Where not, the entries below leave the work to Python (None).
bool unobserved(const Tensor& t) {
  return !at::impl::torch_function_mode_enabled() && !c10::impl::dispatch_mode_enabled() && !t.key_set().has(c10::DispatchKey::Python);
}

// tensors (or None) -> whether all of them are ordinary ones, and unobserved
PyObject* ordinary(const Args& a) {
  bool all = true;
  for (Py_ssize_t i = 0; i < a.n && all; ++i)
    all = a.none(i) || (THPVariable_CheckExact(a.v[i]) && unobserved(THPVariable_Unpack(a.v[i])));
  return PyBool_FromLong(all);
}

// t.as_subclass(torch.Tensor) without a turn through __torch_function__
PyObject* plain(const Args& a) {
  const Tensor& t = as_it_is(a.v[0]);
  return unobserved(t) ? wrap(t.alias()) : none();
}

// t.as_subclass(class), likewise
PyObject* of_class(const Args& a) {
  if (!PyType_Check(a.v[1])) throw Raised(PyExc_TypeError, "a class is expected");
  const Tensor& t = as_it_is(a.v[0]);
  return unobserved(t) ? THPVariable_Wrap(t.alias(), reinterpret_cast<PyTypeObject*>(a.v[1])) : none();
}

// rows, columns, dtype, like -> an uninitialised [rows, columns] matrix on like's device
PyObject* matrix(const Args& a) {
  const Tensor& like = as_it_is(a.v[3]);
  at::ScalarType type = like.scalar_type();
  a.dtype(2, &type);
  if (!like.is_cuda()) runtime_error("a device tensor is expected");
  return wrap(empty({a.integer(0), a.integer(1)}, type, like));
}

// tensor, class, tag stack, load stack, extra attributes (a dict or None): tensor.as_subclass(class) with the three in
// its dictionary, the last as a copy
PyObject* grid(const Args& a) {
  static PyObject* const keys[3] = {PyUnicode_InternFromString("cell_tag_stack"), PyUnicode_InternFromString("cell_load_stack"),
                                    PyUnicode_InternFromString("cell_extra_attr_dict")};
  if (!PyType_Check(a.v[1])) throw Raised(PyExc_TypeError, "a class is expected");
  const Tensor& t = as_it_is(a.v[0]);
  if (!unobserved(t)) return none();
  PyObject* const made = THPVariable_Wrap(t.alias(), reinterpret_cast<PyTypeObject*>(a.v[1]));
  PyObject* const attrs = made != nullptr ? PyObject_GenericGetDict(made, nullptr) : nullptr;
  PyObject* const extra = attrs == nullptr ? nullptr : PyDict_Check(a.v[4]) ? PyDict_Copy(a.v[4]) : PyDict_New();
  const bool done = extra != nullptr && PyDict_SetItem(attrs, keys[0], a.v[2]) == 0 && PyDict_SetItem(attrs, keys[1], a.v[3]) == 0 &&
                    PyDict_SetItem(attrs, keys[2], extra) == 0;
  Py_XDECREF(extra);
  Py_XDECREF(attrs);
  if (!done) {
    Py_XDECREF(made);
    throw Raised(nullptr, "");
  }
  return made;
}

// data, rows of every path (a list), loads or None, tags or None -> the three as lists of views by path (an empty
// list for None)
PyObject* split_rows(const Args& a) {
  const Tensor data = a.tensor(0), loads = a.tensor_or_none(2), tags = a.tensor_or_none(3);
  if (!PyList_Check(a.v[1])) throw Raised(PyExc_TypeError, "a list of rows is expected");
  const Py_ssize_t paths = PyList_GET_SIZE(a.v[1]);
  std::vector<int64_t> rows(paths);
  for (Py_ssize_t i = 0; i < paths; ++i) {
    rows[i] = PyLong_AsLong(PyList_GET_ITEM(a.v[1], i));
    if (rows[i] == -1 && PyErr_Occurred()) throw Raised(nullptr, "");
  }
  std::vector<Tensor> views[3];
  int64_t start = 0;
  for (Py_ssize_t i = 0; i < paths; ++i) {
    views[0].push_back(data.narrow(0, start, rows[i]));
    if (loads.defined()) views[1].push_back(loads.narrow(0, i, 1));
    if (tags.defined()) views[2].push_back(tags.narrow(0, start, rows[i]));
    start += rows[i];
  }
  PyObject* lists[3];
  for (int k = 0; k < 3; ++k) {
    lists[k] = PyList_New(views[k].size());
    for (size_t i = 0; i < views[k].size(); ++i) PyList_SET_ITEM(lists[k], i, wrap(std::move(views[k][i])));
  }
  return tuple(lists[0], lists[1], lists[2]);
}

// in_data, index, rows of the result: zeros(rows, ...) with in_data's rows added at their index, in ascending row order
PyObject* sum_rows_by_index(const Args& a) {
  const Tensor given = a.tensor(0), index_given = a.tensor(1);
  const Tensor in = dense(given), index = dense(index_given);
  on_device(in, "in_data"), on_device(index, "route_indices");
  const int type = data_type(in, "data type");
  if (index.scalar_type() != at::kInt && index.scalar_type() != at::kLong) runtime_error("route_indices must be int32 or int64");
  const int64_t P = in.size(0), n = a.integer(2);
  if (index.numel() != P) runtime_error("one index per row is needed");
  const c10::DeviceGuard guard(in.device());
  Tensor out = empty(rows_of(in, n), in.scalar_type(), in);
  const size_t bytes = brt_hip_combine_by_index_workspace_bytes(P, n);
  const Tensor ws = scratch(bytes, in);
  check(brt_hip_combine_by_index(ptr(in), ptr(out), ptr(index), index.scalar_type() == at::kInt ? 32 : 64, P, divided(in.numel(), P), n,
                                 ptr(ws), ws.numel(), type, type, stream_of(in)));
  return wrap(out);
}

// The rows of the flows (a list), their tags (a list of vectors) -> (the rows of every tag added up in the order of the flows, the tags
// in ascending order, their number as an int32 vector), (smallest tag, largest tag) where these are too far apart for the launch over the
// flows themselves, or None where it does not take the flows
PyObject* combine_flows(const Args& a) {
  if (!PyList_Check(a.v[0]) || !PyList_Check(a.v[1])) return none();
  const Py_ssize_t count = PyList_GET_SIZE(a.v[0]);
  if (count < 1 || count > BRT_MAX_FLOWS || PyList_GET_SIZE(a.v[1]) != count) return none();
  std::vector<Tensor> datas(count), tags(count);
  std::vector<int32_t> rows(count);
  int64_t n = 0;
  for (Py_ssize_t f = 0; f < count; ++f) {
    PyObject *const d = PyList_GET_ITEM(a.v[0], f), *const t = PyList_GET_ITEM(a.v[1], f);
    if (!THPVariable_CheckExact(d) || !THPVariable_CheckExact(t)) return none();
    datas[f] = THPVariable_Unpack(d), tags[f] = THPVariable_Unpack(t);
    for (const Tensor* x : {&datas[f], &tags[f]})
      if (!unobserved(*x) || !x->is_cuda() || x->layout() != at::kStrided || x->is_neg() || x->dim() < 1 || x->device() != datas[0].device() ||
          x->key_set().has(c10::DispatchKey::FuncTorchBatched))
        return none();
    if (datas[f].scalar_type() != datas[0].scalar_type() || tags[f].scalar_type() != tags[0].scalar_type() ||
        datas[f].sizes().slice(1) != datas[0].sizes().slice(1) || tags[f].dim() != 1 || tags[f].size(0) != datas[f].size(0))
      return none();
    n += datas[f].size(0);
    if (n > BRT_FLOW_ROWS_MAX) return none();
    rows[f] = static_cast<int32_t>(datas[f].size(0));
  }
  const int type = code_of(datas[0].scalar_type());
  const bool narrow = tags[0].scalar_type() == at::kInt;
  const int64_t cell = c10::multiply_integers(datas[0].sizes().slice(1));
  if (n < 2 || type < 0 || (!narrow && tags[0].scalar_type() != at::kLong) || cell < 1 || cell > INT32_MAX) return none();
  const c10::DeviceGuard guard(datas[0].device());
  std::vector<const void*> data_of(count), tags_of(count);
  for (Py_ssize_t f = 0; f < count; ++f) {
    datas[f] = dense(datas[f]), tags[f] = dense(tags[f]);
    data_of[f] = ptr(datas[f]), tags_of[f] = ptr(tags[f]);
    if (rows[f] > 0 && (data_of[f] == nullptr || tags_of[f] == nullptr)) return none();
  }
  const Tensor& like = datas[0];
  Tensor unique = empty({n}, tags[0].scalar_type(), like), number = empty({1}, at::kInt, like);
  const Tensor lists = empty({2 * n}, at::kInt, like), found = empty({3}, at::kLong, like);
  int32_t *const head = iptr(lists), *const next = head + n;
  HostWords words(like, 24, "reading the number of tags");
  words.queued = true;
  check(brt_hip_unique_tags_of_flows(tags_of.data(), rows.data(), count, narrow ? 32 : 64, ptr(unique), head, next, iptr(number),
                                     static_cast<int64_t*>(ptr(found)), words.seen_from_device, words.st));
  const int64_t* const read = static_cast<const int64_t*>(words.read(found));
  const int64_t n_out = read[0];
  if (n_out < 0) return tuple(PyLong_FromLongLong(read[1]), PyLong_FromLongLong(read[2]));
  Tensor out = empty(rows_of(like, n_out), like.scalar_type(), like);
  check(brt_hip_combine_flows(data_of.data(), rows.data(), count, ptr(out), head, next, cell, n_out, type, words.st));
  return tuple(wrap(out), wrap(unique.narrow(0, 0, n_out)), wrap(number));
}

// value, like -> [value] as an int32 vector on like's device, without a wait
PyObject* one_value(const Args& a) {
  const Tensor& like = as_it_is(a.v[1]);
  const c10::DeviceGuard guard(like.device());
  return wrap(at::full({1}, static_cast<int64_t>(a.integer(0)), at::TensorOptions().dtype(at::kInt).device(like.device())));
}

PyObject* calls(const Args&) { return PyLong_FromUnsignedLongLong(g_calls); }

template <PyObject* (*FN)(const Args&), int N>
PyObject* entry(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (n != N) {
    PyErr_Format(PyExc_TypeError, "%d arguments are expected, got %zd", N, n);
    return nullptr;
  }
  try {
    return FN(Args{v, n});
  } catch (const Raised& e) {
    if (e.type != nullptr) PyErr_SetString(e.type, e.what());
  } catch (...) {
    torch::translate_exception_to_python(std::current_exception());
  }
  return nullptr;
}

#define BRT_ENTRY(name, n) \
  { #name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&entry<name, n>)), METH_FASTCALL, nullptr }
PyMethodDef methods[] = {
    BRT_ENTRY(topk_hot_mask, 2),    BRT_ENTRY(gate_topk, 4),           BRT_ENTRY(throttle_hotmask, 3),
    BRT_ENTRY(generate, 5),         BRT_ENTRY(route_and_dispatch, 7),  BRT_ENTRY(route_by_path, 7),
    BRT_ENTRY(dispatch, 12),  BRT_ENTRY(dispatch_and_read, 8),        BRT_ENTRY(combine, 8),             BRT_ENTRY(combine_by_row_tags, 5),
    BRT_ENTRY(top1_to_capacity, 2), BRT_ENTRY(top1_route_to_capacity, 4), BRT_ENTRY(dispatch_by_rows, 5), BRT_ENTRY(combine_by_rows, 7),     BRT_ENTRY(grouped_linear, 16),
    BRT_ENTRY(grouped_linear_f32, 16), BRT_ENTRY(cast_f32_to_bf16, 1), BRT_ENTRY(branch_key, 5),        BRT_ENTRY(int_list, 1),
    BRT_ENTRY(ordinary, 3),         BRT_ENTRY(plain, 1),            BRT_ENTRY(of_class, 2),            BRT_ENTRY(matrix, 4),
    BRT_ENTRY(grid, 5),                BRT_ENTRY(split_rows, 4),
    BRT_ENTRY(sum_rows_by_index, 3), BRT_ENTRY(combine_flows, 2), BRT_ENTRY(one_value, 2),         BRT_ENTRY(unique_tags, 1),      BRT_ENTRY(calls, 0),            {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "brt_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_brt_native() { return PyModule_Create(&module); }

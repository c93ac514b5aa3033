// The host path of the package's torch entry points (fmha_infer_i8, quantize_tensor, dequantize_tensor,
// fmha_infer_from_float): argument checks, output allocation, stream look-up and the call of the C ABI in one native call.
// In Python the same steps took 8 to 10 us per call, more than the kernels of a small problem (B1 H2 S128 d64: 4.2 us on
// the GPU): attribute look-ups on four tensors, two ctypes structures and a ctypes call.  Plain CPython functions taking
// positional arguments; the Python side keeps names, defaults and keyword arguments and turns a returned status into
// FMHAError.
#include <Python.h>

#include <ATen/Functions.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <atomic>
#include <cmath>
#include <mutex>
#include <optional>
#include <thread>
#include <vector>

#include "../../include/fmha_i8.h"
#include "../../include/fmha_quant.h"

namespace {

struct PythonError {};  // a Python exception is set

[[noreturn]] void fail(PyObject* type, const char* text) {
  PyErr_SetString(type, text);
  throw PythonError{};
}

bool on_gpu(PyObject* o) { return THPVariable_Check(o) && THPVariable_Unpack(o).is_cuda(); }

const at::Tensor& int8_on_gpu(PyObject* o, const char* text) {
  if (!on_gpu(o)) fail(PyExc_ValueError, text);
  const at::Tensor& t = THPVariable_Unpack(o);
  if (t.scalar_type() != at::kChar || !t.is_contiguous()) fail(PyExc_ValueError, text);
  return t;
}
const at::Tensor& float_on_gpu(PyObject* o) {
  constexpr const char* text = "x must be a contiguous float32 or bfloat16 tensor on the GPU";
  if (!on_gpu(o)) fail(PyExc_ValueError, text);
  const at::Tensor& t = THPVariable_Unpack(o);
  if ((t.scalar_type() != at::kFloat && t.scalar_type() != at::kBFloat16) || !t.is_contiguous()) fail(PyExc_ValueError, text);
  return t;
}
float number(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw PythonError{};
  return (float)v;
}
// None: torch's current stream of the device; an object with `cuda_stream`, or the handle itself.
hipStream_t stream_of(PyObject* o, const at::Device& device) {
  if (o == Py_None) return c10::hip::getCurrentHIPStream(device.index()).stream();
  PyObject* handle = PyObject_GetAttrString(o, "cuda_stream");
  if (handle == nullptr) {
    if (!PyErr_ExceptionMatches(PyExc_AttributeError)) throw PythonError{};
    PyErr_Clear();
    handle = PyNumber_Index(o);
    if (handle == nullptr) throw PythonError{};
  }
  void* p = PyLong_AsVoidPtr(handle);
  Py_DECREF(handle);
  if (p == nullptr && PyErr_Occurred()) throw PythonError{};
  return static_cast<hipStream_t>(p);
}
// The null stream is that of the current device: a call makes its tensors' device current, and the caller's again when it ends.
// (Where it is current already the guard, whose end asks the runtime for the device's state, costs a call 0.1 us.)
struct OnDevice {
  std::optional<c10::hip::HIPGuard> guard;
  explicit OnDevice(c10::DeviceIndex index) {
    if (c10::hip::current_device() != index) guard.emplace(index);
  }
};
// Memory of torch's caching allocator, ordered by the stream that is current on the device.
at::Tensor empty(c10::IntArrayRef sizes, at::ScalarType type, const at::Device& device) {
  return at::detail::empty_cuda(sizes, type, device, std::nullopt);
}
at::ScalarType float_type(PyObject* o, at::ScalarType otherwise) {
  if (o == Py_None) return otherwise;
  const at::ScalarType t = THPDtype_Check(o) ? reinterpret_cast<THPDtype*>(o)->scalar_type : at::kInt;
  if (t != at::kFloat && t != at::kBFloat16) fail(PyExc_ValueError, "dtype must be float32 or bfloat16");
  return t;
}

// The launches run without the interpreter's lock: a full queue blocks only the calling thread.
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

// Memory that a call needs while it runs and the caller never sees: it belongs to the stream that the kernels are queued on, or
// the current stream could hand it out again while they still use it.
at::Tensor empty_on(hipStream_t stream, int64_t bytes, const at::Device& device) {
  std::optional<c10::hip::HIPStreamGuard> guard;
  if (stream != c10::hip::getCurrentHIPStream(device.index()).stream())
    guard.emplace(c10::hip::getStreamFromExternal(stream, device.index()));
  return empty({bytes}, at::kChar, device);
}

struct AttnShape {
  int b, h, sq, s, d;
};
// The workspace of an attention call, if it has a use for one (a few query rows per head).  The call does without where memory
// is short, and where a stream is being captured into an output of the caller's: torch's allocator keeps what it hands out
// during a capture for the graph only if the capture is torch's own, which a call that allocates its output relies on anyway.
at::Tensor workspace_of(const AttnShape& n, hipStream_t stream, const at::Device& device, bool own_output) {
  constexpr int kMostRows = 32;  // no call of more rows wants any: spares the others the question
  if (n.sq > kMostRows) return {};
  const size_t bytes = FMHAInferI8CrossWorkspaceBytes(FMHACrossAttnDescriptor{n.b, n.sq, n.s, n.h, n.d});
  if (bytes == 0) return {};
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (!own_output && (hipStreamIsCapturing(stream, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone)) return {};
  try {
    return empty_on(stream, (int64_t)bytes, device);
  } catch (const c10::OutOfMemoryError&) {
    return {};
  }
}
int attend(hipStream_t stream, const AttnShape& n, const FMHAParamI8& scales, const void* q, const void* k, const void* v,
           const void* mask, void* out, bool full_range_p, const at::Tensor& workspace) {
  if (workspace.defined())
    return FMHAInferI8CrossWithWorkspace(stream, scales, FMHACrossAttnDescriptor{n.b, n.sq, n.s, n.h, n.d}, q, k, v, mask, out,
                                         full_range_p, workspace.data_ptr(), (size_t)workspace.numel());
  if (!full_range_p && n.sq == n.s)
    return FMHAInferI8Status(stream, scales, AttnDataDescriptor{n.b, n.s, n.h, n.d}, q, k, v, mask, out, true);
  const FMHACrossAttnDescriptor desc{n.b, n.sq, n.s, n.h, n.d};
  return full_range_p ? FMHAInferI8CrossFullRangeP(stream, scales, desc, q, k, v, mask, out)
                      : FMHAInferI8Cross(stream, scales, desc, q, k, v, mask, out);
}
AttnShape shape_of(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& mask) {
  const bool four = q.dim() == 4 && k.dim() == 4;
  if (!four || k.size(0) != q.size(0) || k.size(1) != q.size(1) || k.size(3) != q.size(3) || v.sizes() != k.sizes() ||
      mask.dim() != 2 || mask.size(0) != q.size(0) || mask.size(1) != k.size(2))
    fail(PyExc_ValueError, "shape mismatch: q [B,H,Sq,d], k/v [B,H,S,d] and padding_mask [B,S] expected");
  return {(int)q.size(0), (int)q.size(1), (int)q.size(2), (int)k.size(2), (int)q.size(3)};
}

int dequantize(hipStream_t stream, const int8_t* x, const at::Tensor& out, float amax) {
  return out.scalar_type() == at::kFloat
             ? FMHADequantizeI8(stream, x, out.numel(), amax, out.data_ptr<float>())
             : FMHADequantizeI8BF16(stream, x, out.numel(), amax, static_cast<uint16_t*>(out.data_ptr()));
}

// Pinned words through which the device hands the host the maxima of a running call (FMHAMeasureAndQuantizeI8).  One
// page for the process, in slots of one cache line; a call takes a slot, waits for its words and gives it back, so a
// slot never has two writers, whatever the streams and threads.
class NotePool {
 public:
  static constexpr int kSlots = 64, kWords = 8;
  static NotePool& get() {
    static NotePool* pool = new NotePool;  // (never destroyed: the runtime frees pinned memory when the process ends)
    return *pool;
  }
  unsigned long long* take() {
    for (;;) {
      {
        std::lock_guard<std::mutex> lock(mutex_);
        if (page_ == nullptr) {
          void* p = nullptr;
          if (hipHostMalloc(&p, kSlots * kWords * 8, hipHostMallocPortable) != hipSuccess) return nullptr;
          page_ = static_cast<unsigned long long*>(p);
          for (int i = 0; i < kSlots * kWords; ++i) page_[i] = 0;
          for (int i = 0; i < kSlots; ++i) free_.push_back(page_ + i * kWords);
        }
        if (!free_.empty()) {
          unsigned long long* slot = free_.back();
          free_.pop_back();
          return slot;
        }
      }
      std::this_thread::yield();  // (more than kSlots threads inside a call at once)
    }
  }
  void give_back(unsigned long long* slot) {
    std::lock_guard<std::mutex> lock(mutex_);
    free_.push_back(slot);
  }
  unsigned ticket() { return next_.fetch_add(1, std::memory_order_relaxed); }

 private:
  std::mutex mutex_;
  std::vector<unsigned long long*> free_;
  unsigned long long* page_ = nullptr;
  std::atomic<unsigned> next_{1};
};

// Waits for `count` words that carry this ticket.  The stream is asked now and then, so that a launch that failed, or a
// stream that is being captured, ends the wait.
int wait_for_note(hipStream_t stream, const unsigned long long* note, unsigned ticket, int count, float* amax) {
  int have = 0;
  for (unsigned spin = 1;; ++spin) {
    const bool idle = (spin & 0x3fff) == 0;
    const hipError_t state = idle ? hipStreamQuery(stream) : hipErrorNotReady;
    for (; have < count; ++have) {
      const unsigned long long w = __atomic_load_n(note + have, __ATOMIC_ACQUIRE);
      if ((unsigned)(w >> 32) != ticket) break;
      const unsigned bits = (unsigned)w;
      __builtin_memcpy(&amax[have], &bits, 4);
    }
    if (have == count) return FMHA_I8_OK;
    if (state == hipSuccess) return FMHA_I8_ERR_HIP_BASE + (int)hipErrorUnknown;
    if (state != hipErrorNotReady) return FMHA_I8_ERR_HIP_BASE + (int)state;
    __builtin_ia32_pause();
  }
}

template <typename F>
PyObject* guarded(F f) {
  try {
    return f();
  } catch (const PythonError&) {
    return nullptr;
  }
  catch (const std::exception&) {  // (as torch's own functions raise it: torch.OutOfMemoryError and the others by their types)
    torch::translate_exception_to_python(std::current_exception());
    return nullptr;
  }
}
bool count_is(Py_ssize_t n, Py_ssize_t want) {
  if (n != want) PyErr_Format(PyExc_TypeError, "%zd positional arguments expected, got %zd", want, n);
  return n == want;
}

// (q, k, v, padding_mask, q_amax, k_amax, v_amax, o_amax, out, stream, full_range_p) -> tensor, or the status as an int
PyObject* infer_i8(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!count_is(n, 11)) return nullptr;
  return guarded([&]() -> PyObject* {
    const at::Tensor& q = int8_on_gpu(a[0], "q must be a contiguous int8 tensor on the GPU");
    const at::Tensor& k = int8_on_gpu(a[1], "k must be a contiguous int8 tensor on the GPU");
    const at::Tensor& v = int8_on_gpu(a[2], "v must be a contiguous int8 tensor on the GPU");
    const at::Tensor& mask = int8_on_gpu(a[3], "padding_mask must be a contiguous int8 tensor on the GPU");
    const AttnShape shape = shape_of(q, k, v, mask);
    const FMHAParamI8 scales{number(a[4]), number(a[5]), number(a[6]), number(a[7]), 1.0f};
    const at::Device device = q.device();
    const OnDevice on_device(device.index());
    at::Tensor out;
    if (a[8] == Py_None) {
      out = empty(q.sizes(), at::kChar, device);
    } else {
      constexpr const char* text = "out must be a contiguous int8 tensor on the GPU, shaped like q";
      out = int8_on_gpu(a[8], text);
      if (out.sizes() != q.sizes()) fail(PyExc_ValueError, text);
    }
    const hipStream_t stream = stream_of(a[9], device);
    const int full = PyObject_IsTrue(a[10]);
    if (full < 0) throw PythonError{};
    const at::Tensor workspace = workspace_of(shape, stream, device, a[8] == Py_None);
    int status;
    {
      Unlocked unlocked;
      status = attend(stream, shape, scales, q.data_ptr(), k.data_ptr(), v.data_ptr(), mask.data_ptr(), out.data_ptr(), full != 0, workspace);
    }
    if (status != FMHA_I8_OK) return PyLong_FromLong(status);
    if (a[8] != Py_None) {
      Py_INCREF(a[8]);
      return a[8];
    }
    return THPVariable_Wrap(std::move(out));
  });
}

// (x, amax, stream) -> (int8 tensor, amax tensor), or the status
PyObject* quantize_tensor(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!count_is(n, 3)) return nullptr;
  return guarded([&]() -> PyObject* {
    const at::Tensor& x = float_on_gpu(a[0]);
    const at::Device device = x.device();
    const OnDevice on_device(device.index());
    const hipStream_t stream = stream_of(a[2], device);
    at::Tensor out = empty(x.sizes(), at::kChar, device), amax;
    int status;
    if (a[1] == Py_None) {
      amax = empty({1}, at::kFloat, device);
      const at::Tensor workspace = empty_on(stream, 4 * FMHA_QUANT_WORKSPACE_FLOATS, device);
      const FMHAQuantTensor t{x.data_ptr(), static_cast<int8_t*>(out.data_ptr()), (long long)x.numel()};
      Unlocked unlocked;
      status = FMHAMeasureAndQuantizeI8(stream, &t, 1, x.scalar_type() == at::kFloat ? FMHA_QUANT_F32 : FMHA_QUANT_BF16,
                                        static_cast<float*>(workspace.data_ptr()), amax.data_ptr<float>(), nullptr, 0);
    } else {
      const float value = number(a[1]);
      amax = at::full({1}, value, out.options().dtype(at::kFloat));
      Unlocked unlocked;
      status = x.scalar_type() == at::kFloat
                   ? FMHAQuantizeI8(stream, x.data_ptr<float>(), x.numel(), value, nullptr, static_cast<int8_t*>(out.data_ptr()))
                   : FMHAQuantizeI8BF16(stream, static_cast<const uint16_t*>(x.data_ptr()), x.numel(), value, nullptr,
                                        static_cast<int8_t*>(out.data_ptr()));
    }
    if (status != FMHA_I8_OK) return PyLong_FromLong(status);
    PyObject* first = THPVariable_Wrap(std::move(out));
    PyObject* second = first ? THPVariable_Wrap(std::move(amax)) : nullptr;
    PyObject* pair = second ? PyTuple_Pack(2, first, second) : nullptr;
    Py_XDECREF(first);
    Py_XDECREF(second);
    return pair;
  });
}

// (x, amax, stream, dtype) -> tensor, or the status
PyObject* dequantize_tensor(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!count_is(n, 4)) return nullptr;
  return guarded([&]() -> PyObject* {
    const at::Tensor& x = int8_on_gpu(a[0], "x must be a contiguous int8 tensor on the GPU");
    const at::ScalarType type = float_type(a[3], at::kFloat);
    const float amax = number(a[1]);
    const OnDevice on_device(x.device().index());
    const hipStream_t stream = stream_of(a[2], x.device());
    at::Tensor out = empty(x.sizes(), type, x.device());
    int status;
    {
      Unlocked unlocked;
      status = dequantize(stream, static_cast<const int8_t*>(x.data_ptr()), out, amax);
    }
    if (status != FMHA_I8_OK) return PyLong_FromLong(status);
    return THPVariable_Wrap(std::move(out));
  });
}

// (q, k, v, padding_mask, o_amax, out_dtype, stream, full_range_p) -> (O, int8 O, (q_amax, k_amax, v_amax)), or the status
//
// Launches: abs-max of the three tensors and their quantisation, in one or two, and the attention, which may de-quantise its output too.  The
// attention's scales are call arguments, so the host needs the three maxima in between: the quantising kernel writes them to pinned memory
// as soon as it has them, and the host, which polls for them, has the attention queued while the int8 values are still being written.
PyObject* infer_from_float(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!count_is(n, 8)) return nullptr;
  return guarded([&]() -> PyObject* {
    const at::Tensor* x[3];
    for (int i = 0; i < 3; ++i) x[i] = &float_on_gpu(a[i]);
    const at::Tensor& mask = int8_on_gpu(a[3], "padding_mask must be a contiguous int8 tensor on the GPU");
    const AttnShape shape = shape_of(*x[0], *x[1], *x[2], mask);
    const float o_amax = number(a[4]);
    const at::ScalarType out_type = float_type(a[5], x[0]->scalar_type());
    const at::Device device = x[0]->device();
    const OnDevice on_device(device.index());
    const hipStream_t stream = stream_of(a[6], device);
    const int full = PyObject_IsTrue(a[7]);
    if (full < 0) throw PythonError{};
    // Everything is allocated under the stream that the kernels are queued on.
    std::optional<c10::hip::HIPStreamGuard> guard;
    if (stream != c10::hip::getCurrentHIPStream(device.index()).stream())
      guard.emplace(c10::hip::getStreamFromExternal(stream, device.index()));
    at::Tensor o = empty(x[0]->sizes(), out_type, device), o_i8 = empty(x[0]->sizes(), at::kChar, device);
    auto padded = [](long long bytes) { return (bytes + 255) / 256 * 256; };
    long long at_byte[4] = {0, 0, 0, 0};
    for (int i = 0; i < 3; ++i) at_byte[i + 1] = at_byte[i] + padded(x[i]->numel());
    // the int8 Q, K and V, the partial maxima and the maxima
    at::Tensor scratch = empty({at_byte[3] + 4 * (FMHA_QUANT_WORKSPACE_FLOATS + 4)}, at::kChar, device);
    int8_t* base = static_cast<int8_t*>(scratch.data_ptr());
    float* workspace = reinterpret_cast<float*>(base + at_byte[3]);
    const at::Tensor attend_workspace = workspace_of(shape, stream, device, true);
    FMHAQuantTensor t[3];
    int type[3];
    for (int i = 0; i < 3; ++i) {
      t[i] = {x[i]->data_ptr(), base + at_byte[i], (long long)x[i]->numel()};
      type[i] = x[i]->scalar_type() == at::kFloat ? FMHA_QUANT_F32 : FMHA_QUANT_BF16;
    }
    float amax[3] = {0.f, 0.f, 0.f};
    int status = FMHA_I8_OK;
    {
      Unlocked unlocked;
      NotePool& pool = NotePool::get();
      unsigned long long* note = pool.take();
      if (note == nullptr) status = FMHA_I8_ERR_HIP_BASE + (int)hipErrorOutOfMemory;
      if (status == FMHA_I8_OK) {
        const unsigned ticket = pool.ticket();
        float* maxima = workspace + FMHA_QUANT_WORKSPACE_FLOATS;
        if (type[0] == type[1] && type[1] == type[2]) {
          status = FMHAMeasureAndQuantizeI8(stream, t, 3, type[0], workspace, maxima, note, ticket);
        } else {
          for (int i = 0; i < 3 && status == FMHA_I8_OK; ++i)
            status = FMHAMeasureAndQuantizeI8(stream, t + i, 1, type[i], workspace, maxima + i, note + i, ticket);
        }
        if (status == FMHA_I8_OK) status = wait_for_note(stream, note, ticket, 3, amax);
        pool.give_back(note);
      }
      const bool all_positive = amax[0] > 0.f && amax[1] > 0.f && amax[2] > 0.f;
      const FMHAParamI8 scales{amax[0], amax[1], amax[2], o_amax, 1.0f};
      // The attention kernel de-quantises its output too, which saves a launch and a pass over it; the merge of shared-out key blocks
      // writes int8 only.  Attention with a second launch and fused, us: B4 H16 S1024 d128 30.7 and 26.5 as bfloat16, 32.9 and 28.1 as
      // float32; B8 H12 S512 d64 14.3 and 11.2, 15.0 and 12.5; B1 H32 S4096 d128 157.6 and 153.3, 162.7 and 157.4; B2 H8 S300 d128 9.1
      // and 7.1, 9.5 and 7.5; over at most 128 keys B1 H2 Sq32768 S128 d64 11.3 and 8.2, 11.5 and 9.2, B16 H16 Sq2048 S128 d64 54.4 and
      // 46.4, 63.7 and 52.2, B256 H16 S128 d64 75.5 and 70.4, 84.9 and 82.9.  Over so few keys the call is all memory, and beyond 32 M
      // elements its tensors outgrow the last-level cache, where fused calls take from 13 % less to 8 % more (B512 H16 S128 d128 233 and
      // 217, 290 and 251; B192 79.6 and 85.4, 94.1 and 98.6): those stay with two launches.
      const bool fused = !attend_workspace.defined() && (shape.s > 128 || o.numel() <= 32 << 20);
      if (status == FMHA_I8_OK && all_positive)
        status = fused ? FMHAInferI8CrossToFloat(stream, scales, FMHACrossAttnDescriptor{shape.b, shape.sq, shape.s, shape.h, shape.d},
                                                 t[0].out, t[1].out, t[2].out, mask.data_ptr(), o_i8.data_ptr(), full != 0, o.data_ptr(),
                                                 out_type == at::kBFloat16)
                       : attend(stream, shape, scales, t[0].out, t[1].out, t[2].out, mask.data_ptr(), o_i8.data_ptr(), full != 0,
                                attend_workspace);
      if (status == FMHA_I8_OK && all_positive && !fused) status = dequantize(stream, static_cast<const int8_t*>(o_i8.data_ptr()), o, o_amax);
    }
    if (status != FMHA_I8_OK) return PyLong_FromLong(status);
    PyObject* maxima = Py_BuildValue("(ddd)", (double)amax[0], (double)amax[1], (double)amax[2]);
    if (maxima == nullptr) return nullptr;
    if (!(amax[0] > 0.f && amax[1] > 0.f && amax[2] > 0.f)) {
      PyErr_Format(PyExc_ValueError, "q, k and v must each hold a nonzero value (abs-max %R)", maxima);
      Py_DECREF(maxima);
      return nullptr;
    }
    PyObject* first = THPVariable_Wrap(std::move(o));
    PyObject* second = first ? THPVariable_Wrap(std::move(o_i8)) : nullptr;
    PyObject* triple = second ? PyTuple_Pack(3, first, second, maxima) : nullptr;
    Py_XDECREF(first);
    Py_XDECREF(second);
    Py_DECREF(maxima);
    return triple;
  });
}

template <typename F>
PyCFunction as_cfunction(F f) { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)); }

PyMethodDef methods[] = {
    {"infer_i8", as_cfunction(infer_i8), METH_FASTCALL, nullptr},
    {"quantize_tensor", as_cfunction(quantize_tensor), METH_FASTCALL, nullptr},
    {"dequantize_tensor", as_cfunction(dequantize_tensor), METH_FASTCALL, nullptr},
    {"infer_from_float", as_cfunction(infer_from_float), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fmha_torch", "native host path of the torch entry points", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fmha_torch() { return PyModule_Create(&module); }

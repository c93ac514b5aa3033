// A HIP runtime of two GPUs whose memory is host memory, and the entry points of libfmha_i8.so that the torch host path
// (csrc/fmha_torch.cpp) calls, for tests of that path without a GPU (test_torch_host_path.py): no kernel runs, every call of
// an entry point is noted with the stream it was given and the device that was current.  Loaded with RTLD_GLOBAL before torch,
// its functions stand in front of the real ones.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "../include/fmha_i8.h"
#include "../include/fmha_quant.h"

namespace {
constexpr int kDevices = 2;
constexpr size_t kMemory = 1ull << 30;
thread_local int current = 0;
std::mutex mutex;
std::map<void*, size_t> allocated;
size_t used = 0, limit = kMemory;
struct Call {
  const char* name;
  int device;
  void* stream;
};
std::vector<Call> calls;
char streams[1024];  // handles are addresses in here
int n_streams = 0;

int note(const char* name, hipStream_t stream) {
  std::lock_guard<std::mutex> lock(mutex);
  calls.push_back({name, current, stream});
  return FMHA_I8_OK;
}
}  // namespace

extern "C" {
int fake_calls() { return (int)calls.size(); }
const char* fake_call(int i, int* device, void** stream) {
  *device = calls[i].device;
  *stream = calls[i].stream;
  return calls[i].name;
}
void fake_forget_calls() { calls.clear(); }
void fake_memory_limit(size_t bytes) { limit = bytes; }
int fake_current_device() { return current; }

hipError_t hipGetDeviceCount(int* n) { return *n = kDevices, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = current, hipSuccess; }
hipError_t hipSetDevice(int d) { return d >= 0 && d < kDevices ? (current = d, hipSuccess) : hipErrorInvalidDevice; }
hipError_t hipInit(unsigned) { return hipSuccess; }
hipError_t hipDriverGetVersion(int* v) { return *v = 70000000, hipSuccess; }
hipError_t hipRuntimeGetVersion(int* v) { return *v = 70000000, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof *p);
  strcpy(p->name, "host memory");
  strcpy(p->gcnArchName, "gfx950");
  p->major = 9, p->minor = 5, p->warpSize = 64, p->multiProcessorCount = 256, p->maxThreadsPerBlock = 1024;
  p->maxThreadsPerMultiProcessor = 2048, p->totalGlobalMem = kMemory, p->sharedMemPerBlock = 65536, p->regsPerBlock = 65536;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 0, hipSuccess; }
hipError_t hipDeviceCanAccessPeer(int* v, int, int) { return *v = 0, hipSuccess; }
hipError_t hipDevicePrimaryCtxGetState(hipDevice_t, unsigned* flags, int* active) { return *flags = 0, *active = 1, hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipPeekAtLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "an error of the host-memory runtime"; }
const char* hipGetErrorName(hipError_t) { return "hipError"; }

hipError_t hipMemGetInfo(size_t* free_bytes, size_t* total) { return *free_bytes = limit > used ? limit - used : 0, *total = kMemory, hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> lock(mutex);
  if (used + n > limit) return hipErrorOutOfMemory;
  if (posix_memalign(p, 4096, n ? n : 1) != 0) return hipErrorOutOfMemory;
  memset(*p, 0, n);
  used += allocated[*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lock(mutex);
  used -= allocated[p];
  allocated.erase(p);
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return posix_memalign(p, 4096, n) == 0 ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void* p) { return free(p), hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyWithStream(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return memset(d, v, n), hipSuccess; }

hipError_t hipDeviceGetStreamPriorityRange(int* least, int* greatest) { return *least = *greatest = 0, hipSuccess; }
hipError_t hipStreamCreateWithPriority(hipStream_t* s, unsigned, int) {
  std::lock_guard<std::mutex> lock(mutex);
  if (n_streams == (int)sizeof streams) return hipErrorOutOfMemory;
  return *s = reinterpret_cast<hipStream_t>(streams + n_streams++), hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) { return *s = hipStreamCaptureStatusNone, hipSuccess; }
hipError_t hipStreamGetCaptureInfo_v2(hipStream_t, hipStreamCaptureStatus* s, unsigned long long*, hipGraph_t*, const hipGraphNode_t**, size_t*) {
  return *s = hipStreamCaptureStatusNone, hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = reinterpret_cast<hipEvent_t>(streams), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
// torch's own kernels (a fill)
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) { return *g = *b = dim3(1), *m = 0, *s = nullptr, hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }

int FMHAInferI8Status(hipStream_t s, FMHAParamI8, AttnDataDescriptor, const void*, const void*, const void*, const void*, void*, bool) {
  return note("FMHAInferI8Status", s);
}
int FMHAInferI8Cross(hipStream_t s, FMHAParamI8, FMHACrossAttnDescriptor, const void*, const void*, const void*, const void*, void*) {
  return note("FMHAInferI8Cross", s);
}
int FMHAInferI8CrossFullRangeP(hipStream_t s, FMHAParamI8, FMHACrossAttnDescriptor, const void*, const void*, const void*, const void*, void*) {
  return note("FMHAInferI8CrossFullRangeP", s);
}
int FMHAInferI8CrossWithWorkspace(hipStream_t s, FMHAParamI8, FMHACrossAttnDescriptor, const void*, const void*, const void*, const void*, void*,
                                  int, void*, size_t) {
  return note("FMHAInferI8CrossWithWorkspace", s);
}
int FMHAInferI8CrossToFloat(hipStream_t s, FMHAParamI8, FMHACrossAttnDescriptor, const void*, const void*, const void*, const void*, void*, int,
                            void*, int) {
  return note("FMHAInferI8CrossToFloat", s);
}
int FMHAQuantizeI8(hipStream_t s, const float*, long long, float, const float*, int8_t*) { return note("FMHAQuantizeI8", s); }
int FMHAQuantizeI8BF16(hipStream_t s, const uint16_t*, long long, float, const float*, int8_t*) { return note("FMHAQuantizeI8BF16", s); }
int FMHADequantizeI8(hipStream_t s, const int8_t*, long long, float, float*) { return note("FMHADequantizeI8", s); }
int FMHADequantizeI8BF16(hipStream_t s, const int8_t*, long long, float, uint16_t*) { return note("FMHADequantizeI8BF16", s); }
int FMHAMeasureAndQuantizeI8(hipStream_t s, const FMHAQuantTensor*, int count, int, float*, float* amax, unsigned long long* words,
                             unsigned ticket) {
  for (int i = 0; i < count; ++i) {
    amax[i] = 1.f;
    if (words != nullptr) words[i] = ((unsigned long long)ticket << 32) | 0x3f800000u;
  }
  return note("FMHAMeasureAndQuantizeI8", s);
}
}

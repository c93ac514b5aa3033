// Quantisation front end / back end of the INT8 attention path for gfx950: abs-max, fp32 / bf16 -> int8, int8 -> fp32 / bf16.
// The reference does these on the host, one element at a time (inc/utils.hpp:23-39,53); here they are streaming
// kernels whose cost is memory traffic: 128-bit accesses on the wide side, one wavefront instruction covers 1 KiB of
// contiguous input, a few thousand wavefronts in flight, no LDS except for the block reduction of the maximum.
#include <hip/hip_runtime.h>
#include <atomic>
#include <chrono>
#include <random>
#include <tuple>
#include <stdint.h>

#include "../../include/fmha_quant.h"
#include "fmha_dequant.h"

// Every float operation below must round exactly where the reference's host code rounds: no fused multiply-add that is
// not written out.
#pragma clang fp contract(off)

namespace fmha_i8_gfx950 {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned short v8h __attribute__((ext_vector_type(8)));
typedef int v2i32 __attribute__((ext_vector_type(2)));
typedef int v4i32 __attribute__((ext_vector_type(4)));

constexpr int kQuantThreads = 256;
constexpr int kQuantUnroll = 4;          // 16-byte units per thread and loop trip: 64 B per lane in flight per trip
// Two workgroups of 4 wavefronts per CU: measured best from 8 to 134 MB in each kernel (bf16 de-quantise of 33.5 M elements:
// 15.9 us with 512 workgroups, 17.9 with 1024; 256 lose as much below 16 MB).
constexpr int kQuantMaxBlocks = 256 * 2;
// An input larger than the last-level cache is quantised with loads that bypass it (non-temporal): fp32 62.6 -> 60.0 us at 288
// MiB, 88.3 -> 81.8 at 384, 243 -> 229 at 1 GiB, bf16 75.8 -> 71.8 at 288, 141.5 -> 129.0 at 512; at 256 MiB they lose (fp32 47.0 ->
// 53.2, bf16 57.5 -> 63.3).  Nowhere else: behind an abs-max, which has just read the tensor, they lose up to 700 MiB (fp32 92.9 ->
// 98.2 us at 288, level at 640) and gain 1 to 3 % above; the de-quantisation reads a byte per element (fp32, 268 M elements:
// 208 -> 243 us).
constexpr long long kCacheBytes = 256ll << 20;
// What a kernel writes it never reads again: stores are non-temporal at every size, so that the input - read a second
// time by the quantisation behind the abs-max - keeps the L2 (fp32, abs-max + quantise: 13.6 -> 12.8 us at 8.4 M elements,
// 48.2 -> 45.1 at 33.5 M; de-quantise 7.9 -> 6.4 at 8.4 M; level elsewhere).
// A tensor of up to kSmallElements is measured and quantised by ONE workgroup that keeps it in its registers (32 floats
// per thread): one launch of 3.1 to 4.2 us in place of two that take 5.6 together; above, one CU's bandwidth loses to two launches.
constexpr int kSmallThreads = 1024;
constexpr int kSmallElements = 32768;
// The abs-max without a workspace ends in one atomic per workgroup, all on one address: below this size half the workgroups
// (8.6 against 11.5 us at 12 MB), above it the bandwidth of all of them (27.6 against 24.7 us at 134 MB).
constexpr long long kAtomicBytes = 64ll << 20;

// The element types of the float side.  One 16-byte unit holds kPerUnit of them; a bfloat16 is the upper half of a
// float: widening is exact, so every function below is the float one applied to the widened values.
struct F32 {
  typedef float elem;
  typedef v4f unit;
  typedef int packed;  // the int8 image of one unit
  static constexpr int kPerUnit = 4;
  static __device__ __forceinline__ float widen(float x) { return x; }
};
struct BF16 {
  typedef unsigned short elem;
  typedef v8h unit;
  typedef v2i32 packed;
  static constexpr int kPerUnit = 8;
  static __device__ __forceinline__ float widen(unsigned short h) { return __uint_as_float((unsigned)h << 16); }
};

// One call quantises up to three tensors (the Q, K and V of an attention call) with one launch of each kernel: block b
// belongs to the tensor whose range of blocks holds it.
struct QuantJob {
  const void* x[FMHA_QUANT_MAX_TENSORS];
  int8_t* out[FMHA_QUANT_MAX_TENSORS];
  long long n[FMHA_QUANT_MAX_TENSORS];
  int first_block[FMHA_QUANT_MAX_TENSORS + 1];
};

__device__ __forceinline__ void take_abs(float& m, float v) {
  const float a = fabsf(v);
  m = a > m ? a : m;  // a NaN never compares greater: skipped, as in the reference
}

// The largest |x| of many units in one instruction per element, where take_abs takes three: the largest bit pattern as a signed
// number belongs to the largest positive value, the largest as an unsigned number to the negative one of the largest magnitude.  NaN,
// whose patterns are the largest of all, comes out as a value above infinity's: the caller then goes over its units with take_abs.
typedef short v2s16 __attribute__((ext_vector_type(2)));
typedef unsigned short v2u16 __attribute__((ext_vector_type(2)));
template <typename T>
struct LargestBits;
template <>
struct LargestBits<F32> {
  int positive = 0;
  unsigned negative = 0x80000000u;
  __device__ __forceinline__ void take(const v4f& x) {
#pragma unroll
    for (int e = 0; e < 4; e += 2) {
      const unsigned a = __float_as_uint(x[e]), b = __float_as_uint(x[e + 1]);
      positive = max(max(positive, (int)a), (int)b);
      negative = max(max(negative, a), b);
    }
  }
  __device__ __forceinline__ unsigned bits() const { return max((unsigned)positive, negative & 0x7fffffffu); }
};
template <>
struct LargestBits<BF16> {
  v2s16 positive = {0, 0};
  v2u16 negative = {0x8000, 0x8000};
  __device__ __forceinline__ void take(const v8h& x) {
    const v4i32 w = __builtin_bit_cast(v4i32, x);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int two = w[e];  // (a vector element as the operand of a bit cast comes out as element 0)
      positive = __builtin_elementwise_max(positive, __builtin_bit_cast(v2s16, two));
      negative = __builtin_elementwise_max(negative, __builtin_bit_cast(v2u16, two));
    }
  }
  __device__ __forceinline__ unsigned bits() const {
    const unsigned p = max((int)positive[0], (int)positive[1]), n = max((int)negative[0], (int)negative[1]) & 0x7fff;
    return max(p, n) << 16;
  }
};
__device__ __forceinline__ bool above_infinity(unsigned bits) { return bits > 0x7f800000u; }

// Maximum over the workgroup; every thread gets it.
template <int THREADS>
__device__ __forceinline__ float block_max(float m, float (&part)[THREADS / 64]) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const float o = __shfl_xor(m, off);
    m = o > m ? o : m;
  }
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < THREADS / 64; ++w) m = part[w] > m ? part[w] : m;
  return m;
}

template <typename T>
__device__ __forceinline__ void take_abs_unit(float& m, const typename T::unit& v) {
#pragma unroll
  for (int e = 0; e < T::kPerUnit; ++e) take_abs(m, T::widen(v[e]));
}

// abs-max of this thread's share of a tensor (block `block` of `blocks`).  nan: there is one among its whole units.
template <typename T>
__device__ __forceinline__ float abs_max_share(const typename T::elem* __restrict__ x, long long n, int block, int blocks, bool& nan) {
  const long long units = n / T::kPerUnit;
  const typename T::unit* __restrict__ xu = reinterpret_cast<const typename T::unit*>(x);
  const long long stride = (long long)blocks * kQuantThreads;
  LargestBits<T> largest;
  long long j = (long long)block * kQuantThreads + threadIdx.x;
  for (; j + (kQuantUnroll - 1) * stride < units; j += kQuantUnroll * stride) {
    typename T::unit v[kQuantUnroll];
#pragma unroll
    for (int u = 0; u < kQuantUnroll; ++u) v[u] = xu[j + u * stride];
#pragma unroll
    for (int u = 0; u < kQuantUnroll; ++u) largest.take(v[u]);
  }
  for (; j < units; j += stride) largest.take(xu[j]);
  float m = __uint_as_float(largest.bits());
  nan = above_infinity(largest.bits());
  if (nan) {
    m = 0.f;
    for (j = (long long)block * kQuantThreads + threadIdx.x; j < units; j += stride) take_abs_unit<T>(m, xu[j]);
  }
  if (block == 0 && threadIdx.x < (int)(n - T::kPerUnit * units)) take_abs(m, T::widen(x[T::kPerUnit * units + threadIdx.x]));
  return m;
}

__global__ void zero_float_kernel(float* p) { *p = 0.f; }

// inc/utils.hpp:31-39.  |x| of non-NaN floats orders like its bit pattern, so the grid-wide maximum is an unsigned
// atomic max on *out, which zero_float_kernel has cleared.  A workgroup that finds a larger value there already leaves it:
// the atomics queue up at one address, reads of it do not (12.5 -> 10.5 us at 33 MB).
template <typename T>
__global__ __launch_bounds__(kQuantThreads) void abs_max_kernel(const typename T::elem* __restrict__ x, long long n,
                                                                 float* __restrict__ out) {
  __shared__ float part[kQuantThreads / 64];
  bool nan;
  const float m = block_max<kQuantThreads>(abs_max_share<T>(x, n, blockIdx.x, gridDim.x, nan), part);
  if (threadIdx.x == 0 && m > 0.f && m > __hip_atomic_load(out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    atomicMax(reinterpret_cast<unsigned int*>(out), __float_as_uint(m));
}

// The same with one result per workgroup instead of an atomic on one address; negative where the share has a NaN.
template <typename T>
__global__ __launch_bounds__(kQuantThreads) void abs_max_parts_kernel(QuantJob job, float* __restrict__ parts) {
  __shared__ float part[kQuantThreads / 64];
  int i = 0;
#pragma unroll
  for (int k = 1; k < FMHA_QUANT_MAX_TENSORS; ++k) i += (int)blockIdx.x >= job.first_block[k];
  const int block = blockIdx.x - job.first_block[i], blocks = job.first_block[i + 1] - job.first_block[i];
  bool nan;
  const float m = block_max<kQuantThreads>(
      abs_max_share<T>(static_cast<const typename T::elem*>(job.x[i]), job.n[i], block, blocks, nan), part);
  const bool any_nan = __syncthreads_or(nan);
  if (threadIdx.x == 0) parts[blockIdx.x] = any_nan ? -m : m;
}

// inc/utils.hpp:23-29: floorf(x * (127 / amax) + 0.5) in float arithmetic (the reference's double add is exact and
// floorf takes a float, which is one correctly rounded float add), clamp to [-127, 127]; NaN -> 0.
// v_cvt_i32_f32 saturates out-of-range values and turns NaN into 0, so the clamp can follow on integers (one v_med3_i32)
// and needs no look at NaN: five instructions per element.  (v_cvt_flr_i32_f32 would save the floor, but gives 2^31 - 1
// for NaN.)
__device__ __forceinline__ int quant1(float x, float scale) {
  const float t = floorf(x * scale + 0.5f);
  int q;
  asm("v_cvt_i32_f32 %0, %1" : "=v"(q) : "v"(t));  // (in C++ the conversion of a NaN or of a large value is undefined)
  return min(max(q, -127), 127);
}
__device__ __forceinline__ int pack4(int a, int b, int c, int d) {  // low bytes of four ints
  const int lo = __builtin_amdgcn_perm(b, a, 0x0c0c0400), hi = __builtin_amdgcn_perm(d, c, 0x0c0c0400);
  return __builtin_amdgcn_perm(hi, lo, 0x05040100);
}
__device__ __forceinline__ int quant_unit(const v4f& v, float scale) {
  return pack4(quant1(v[0], scale), quant1(v[1], scale), quant1(v[2], scale), quant1(v[3], scale));
}
__device__ __forceinline__ v2i32 quant_unit(const v8h& v, float scale) {
  auto q = [&](int e) { return quant1(BF16::widen(v[e]), scale); };
  return v2i32{pack4(q(0), q(1), q(2), q(3)), pack4(q(4), q(5), q(6), q(7))};
}
// The same for values that the scale was measured on, 127 / amax with finite amax: no NaN among them and none beyond 127.5, so that
// the rounding instruction, which gives 2^31 - 1 for NaN, can stand for floor and conversion, and the clamp has nothing to do.
__device__ __forceinline__ int quant1_measured(float x, float scale) {
  int q;
  asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(q) : "v"(x * scale + 0.5f));
  return q;
}
__device__ __forceinline__ int quant_unit_measured(const v4f& v, float scale) {
  return pack4(quant1_measured(v[0], scale), quant1_measured(v[1], scale), quant1_measured(v[2], scale), quant1_measured(v[3], scale));
}
__device__ __forceinline__ v2i32 quant_unit_measured(const v8h& v, float scale) {
  auto q = [&](int e) { return quant1_measured(BF16::widen(v[e]), scale); };
  return v2i32{pack4(q(0), q(1), q(2), q(3)), pack4(q(4), q(5), q(6), q(7))};
}
__device__ __forceinline__ bool measured_scale(float amax, float scale) { return amax < __builtin_inff() && scale < __builtin_inff(); }
template <bool NT, typename P>  // (a run-time choice between the two is merged into one plain load, constant or not)
__device__ __forceinline__ P load_unit(const P* p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}
// This thread's share of a tensor.  BACK: from the last trip to the first, behind an abs-max that walked the same share
// forwards: the end of the tensor is what the L2 still holds (50.3 -> 48.2 us at 134 MB, level below 32 MB).
// MEASURED: see quant1_measured.
template <typename T, bool NT, bool BACK, bool MEASURED = false>
__device__ __forceinline__ void quantize_share(const typename T::elem* __restrict__ x, long long n, float scale,
                                               int8_t* __restrict__ out, int block, int blocks) {
  const long long units = n / T::kPerUnit;
  const typename T::unit* __restrict__ xu = reinterpret_cast<const typename T::unit*>(x);
  typename T::packed* __restrict__ ou = reinterpret_cast<typename T::packed*>(out);
  const long long stride = (long long)blocks * kQuantThreads;
  long long j = (long long)block * kQuantThreads + threadIdx.x;
  auto quantised = [&](const typename T::unit& v) { return MEASURED ? quant_unit_measured(v, scale) : quant_unit(v, scale); };
  const long long trip = kQuantUnroll * stride;
  auto trip_at = [&](long long at) {
    typename T::unit v[kQuantUnroll];
#pragma unroll
    for (int u = 0; u < kQuantUnroll; ++u) v[u] = load_unit<NT>(&xu[at + u * stride]);
#pragma unroll
    for (int u = 0; u < kQuantUnroll; ++u) __builtin_nontemporal_store(quantised(v[u]), &ou[at + u * stride]);
  };
  if (BACK) {
    const long long full = units / trip;  // trips in which every thread of the grid has all its units
    for (long long r = full * trip + j; r < units; r += stride) ou[r] = quantised(xu[r]);
    for (long long t = full - 1; t >= 0; --t) trip_at(t * trip + j);
  } else {
    for (; j + (kQuantUnroll - 1) * stride < units; j += trip) trip_at(j);
    for (; j < units; j += stride) ou[j] = quantised(xu[j]);
  }
  if (block == 0 && threadIdx.x < (int)(n - T::kPerUnit * units)) {
    const long long r = T::kPerUnit * units + threadIdx.x;
    out[r] = (int8_t)quant1(T::widen(x[r]), scale);
  }
}

template <typename T, bool NT>
__global__ __launch_bounds__(kQuantThreads) void quantize_i8_kernel(const typename T::elem* __restrict__ x, long long n,
                                                                     float amax_host,
                                                                     const float* __restrict__ amax_dev,
                                                                     int8_t* __restrict__ out) {
  const float amax = amax_dev != nullptr ? *amax_dev : amax_host;
  quantize_share<T, NT, false>(x, n, 127.0f / amax, out, blockIdx.x, gridDim.x);
}

__device__ __forceinline__ void note_amax(unsigned long long* note, int i, float amax, unsigned ticket) {
  if (note != nullptr)
    __hip_atomic_store(note + i, ((unsigned long long)ticket << 32) | __float_as_uint(amax), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Quantisation behind abs_max_parts_kernel: every workgroup reduces its tensor's partial maxima (at most 2 KiB, from the
// cache) before it starts, which replaces both the atomics and the launch that clears their target.  With the same split
// into workgroups as the abs-max, what a workgroup reads here its XCD has read before.
// abs-max + quantise, fp32: 18.8 -> 12.8 us at 8.4 M elements (a clearing kernel, 512 atomics and 9.5 us of abs-max before).
template <typename T>
__global__ __launch_bounds__(kQuantThreads) void quantize_by_parts_kernel(QuantJob job, const float* __restrict__ parts,
                                                                           float* __restrict__ amax_out,
                                                                           unsigned long long* __restrict__ note, unsigned ticket) {
  __shared__ float part[kQuantThreads / 64];
  int i = 0;
#pragma unroll
  for (int k = 1; k < FMHA_QUANT_MAX_TENSORS; ++k) i += (int)blockIdx.x >= job.first_block[k];
  const int first = job.first_block[i], blocks = job.first_block[i + 1] - first;
  float m = 0.f;
  bool nan = false;
  for (int p = threadIdx.x; p < blocks; p += kQuantThreads) {
    const float of_block = parts[first + p];
    m = fmaxf(m, fabsf(of_block));
    nan |= (int)__float_as_uint(of_block) < 0;
  }
  const float amax = block_max<kQuantThreads>(m, part);
  const bool any_nan = __syncthreads_or(nan);
  if ((int)blockIdx.x == first && threadIdx.x == 0) {
    amax_out[i] = amax;
    note_amax(note, i, amax, ticket);
  }
  const typename T::elem* x = static_cast<const typename T::elem*>(job.x[i]);
  const float scale = 127.0f / amax;
  if (!any_nan && measured_scale(amax, scale)) quantize_share<T, false, true, true>(x, job.n[i], scale, job.out[i], blockIdx.x - first, blocks);
  else quantize_share<T, false, true>(x, job.n[i], scale, job.out[i], blockIdx.x - first, blocks);
}

// A tensor that one workgroup holds in its registers: maximum and quantisation in one launch, one workgroup per tensor.
template <typename T>
__global__ __launch_bounds__(kSmallThreads) void quantize_small_kernel(QuantJob job, float* __restrict__ amax_out,
                                                                        unsigned long long* __restrict__ note, unsigned ticket) {
  constexpr int kUnits = kSmallElements / T::kPerUnit / kSmallThreads;
  __shared__ float part[kSmallThreads / 64];
  const int i = blockIdx.x;
  const long long n = job.n[i];
  const int units = (int)(n / T::kPerUnit);
  const typename T::elem* __restrict__ x = static_cast<const typename T::elem*>(job.x[i]);
  const typename T::unit* __restrict__ xu = reinterpret_cast<const typename T::unit*>(x);
  int8_t* __restrict__ out = job.out[i];
  typename T::unit v[kUnits];
#pragma unroll
  for (int u = 0; u < kUnits; ++u) {
    const int j = u * kSmallThreads + threadIdx.x;
    if (j < units) v[u] = xu[j];
    else v[u] = typename T::unit{};
  }
  const int rest = T::kPerUnit * units + threadIdx.x;
  float last = rest < n ? T::widen(x[rest]) : 0.f;
  float m = 0.f;
#pragma unroll
  for (int u = 0; u < kUnits; ++u)
#pragma unroll
    for (int e = 0; e < T::kPerUnit; ++e) take_abs(m, T::widen(v[u][e]));
  take_abs(m, last);
  const float amax = block_max<kSmallThreads>(m, part);
  if (threadIdx.x == 0) {
    amax_out[i] = amax;
    note_amax(note, i, amax, ticket);
  }
  const float scale = 127.0f / amax;
#pragma unroll
  for (int u = 0; u < kUnits; ++u) {
    const int j = u * kSmallThreads + threadIdx.x;
    if (j < units) reinterpret_cast<typename T::packed*>(out)[j] = quant_unit(v[u], scale);
  }
  if (rest < n) out[rest] = (int8_t)quant1(last, scale);
}

// Tensors that the registers and LDS of the chip hold: one launch, one pass over the input.  Every workgroup loads its share, leaves the
// share's maximum in its slot of the workspace, waits for the slots of its tensor's other workgroups (2 us) and quantises what it
// holds.  Two launches read the input twice - the second time from the last-level cache - and the second one starts 2.5 us after the
// first.  Measured, us, two launches and this: fp32 8.4 M elements 13.1 and 10.9, 16.8 M 23.2 and 16.5, 25 M 36.1 and 23.3; bf16
// 0.3 M 6.6 and 5.7, 8.4 M 10.1 and 8.9, 33.5 M 26.7 and 18.8; three of 8.4 M, fp32 36.9 and 23.0, bf16 22.5 and 15.5 (20.9 with three
// and seven instructions per element for maximum and quantisation instead of one and five).  Beyond 104 MB of input two launches remain.
//
// A slot is two 8-byte words, each 48 bits of the call's tag and half of the maximum; the tags of no two calls are alike (TagSource),
// so that what a slot held before is never taken for its maximum and nothing has to be cleared first.
// No workgroup depends on another one's progress: one whose slot has not come after `patience` (ticks of 10 ns) - because other work
// holds its compute unit - is not waited for any longer.  Whoever misses it reads one of the shares that have not come, leaves its
// maximum in its slot, where the others find it, and looks again: what all of them read comes to one pass over those shares or two.
// (Every one reading every missing share for itself: 170, 453 and 810 us for fp32 16.8 M elements beside a kernel of another stream that
// held 16, 64 and 128 compute units; this 44, 54 and 66, two launches 36, 44 and 49.  25 M: 226, 649, 1185; 58, 72, 88; 51, 62, 68.
// Up to 52 MB, where two workgroups fit on a compute unit, at most the two launches' time.  With 240 compute units held by attention the
// call ends with that kernel, 0.6 ms, while the two launches' workgroups fit beside it: 27 to 130 us.)  The patience is what such a call
// loses first; with less than 10 us, calls that nothing disturbs run out of it (25 M with 5 us: 23.3 -> 23.9), on cold inputs too.
struct SlotTag {
  unsigned long long word[2];  // 48 bits each, in the upper ones
};
constexpr int kHeldBlocks = 256;  // one per CU; of 512 threads while they hold the call, so that two such calls fit beside each other
#ifdef FMHA_FORCED_ROUTE
std::atomic<unsigned> kPatience{1000};  // test build only: FMHAQuantDebugPatience
#else
constexpr unsigned kPatience = 1000;
#endif
static_assert(kHeldBlocks * sizeof(SlotTag) <= FMHA_QUANT_WORKSPACE_FLOATS * sizeof(float), "one slot per workgroup");

template <typename T, int THREADS, int UNITS, int IN_LDS>
__global__ __launch_bounds__(THREADS, 4) void quantize_held_kernel(QuantJob job, float* __restrict__ amax_out, unsigned long long* slots,
                                                                     SlotTag tag, unsigned patience, unsigned long long* __restrict__ note,
                                                                     unsigned ticket) {
  __shared__ float part[THREADS / 64];
  __shared__ unsigned long long absent[kHeldBlocks / 64];
  __shared__ __attribute__((aligned(1024))) typename T::unit more[IN_LDS > 0 ? IN_LDS : 1][THREADS];  // a thread's own units only
  int i = 0;
#pragma unroll
  for (int k = 1; k < FMHA_QUANT_MAX_TENSORS; ++k) i += (int)blockIdx.x >= job.first_block[k];
  const int first = job.first_block[i], block = blockIdx.x - first, blocks = job.first_block[i + 1] - first;
  const long long n = job.n[i];
  const int units = (int)(n / T::kPerUnit), stride = blocks * THREADS;
  const typename T::elem* __restrict__ x = static_cast<const typename T::elem*>(job.x[i]);
  const typename T::unit* __restrict__ xu = reinterpret_cast<const typename T::unit*>(x);
  int8_t* __restrict__ out = job.out[i];
  const int tid = threadIdx.x, j0 = block * THREADS + tid;
  typename T::unit v[UNITS];
#pragma unroll
  for (int u = 0; u < UNITS; ++u) v[u] = xu[min(j0 + u * stride, units - 1)];  // (past the end: the last unit again)
  if constexpr (IN_LDS > 0) {
    const unsigned base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) typename T::unit*)&more[0][0] + (tid >> 6) * 1024;
#pragma unroll
    for (int k = 0; k < IN_LDS; ++k) {
      const unsigned dst = __builtin_amdgcn_readfirstlane(base + k * THREADS * 16);
      const long long at = min(j0 + (UNITS + k) * stride, units - 1);
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(xu + at) : "memory");
    }
  }
  const int rest = T::kPerUnit * units + tid;  // the elements behind the last unit, in block 0
  const bool has_rest = block == 0 && rest < n;
  const float last = has_rest ? T::widen(x[rest]) : 0.f;
  LargestBits<T> largest;
#pragma unroll
  for (int u = 0; u < UNITS; ++u) largest.take(v[u]);
  if constexpr (IN_LDS > 0) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int k = 0; k < IN_LDS; ++k) largest.take(more[k][tid]);
  }
  float m = __uint_as_float(largest.bits());
  const bool nan = above_infinity(largest.bits());
  if (nan) {
    m = 0.f;
#pragma unroll
    for (int u = 0; u < UNITS; ++u) take_abs_unit<T>(m, v[u]);
#pragma unroll
    for (int k = 0; k < IN_LDS; ++k) take_abs_unit<T>(m, more[k][tid]);
  }
  take_abs(m, last);
  m = block_max<THREADS>(m, part);
  auto leave = [&](int share, float largest_of_share) {
    if (tid >= 2) return;
    const unsigned bits = __float_as_uint(largest_of_share);
    __hip_atomic_store(slots + 2 * (first + share) + tid, (tid == 0 ? tag.word[0] : tag.word[1]) | (tid == 0 ? bits >> 16 : bits & 0xffffu),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  leave(block, m);
  bool here = tid >= blocks || tid == block;  // thread t < kHeldBlocks: the maximum of share t is in m, or there is no such share
  for (unsigned until = patience;; until = 0) {  // (at most `blocks` times: every time around a share's maximum is added)
    if (tid < kHeldBlocks) {  // whole wavefronts
      const unsigned long long since = __builtin_amdgcn_s_memrealtime();
      for (;;) {
        if (!here) {
          const unsigned long long* slot = slots + 2 * (first + tid);
          const unsigned long long w0 = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          const unsigned long long w1 = __hip_atomic_load(slot + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          if (((w0 ^ tag.word[0]) | (w1 ^ tag.word[1])) >> 16 == 0) {
            m = fmaxf(m, __uint_as_float((unsigned)(w0 & 0xffffu) << 16 | (unsigned)(w1 & 0xffffu)));
            here = true;
          }
        }
        if (__all(here) || __builtin_amdgcn_s_memrealtime() - since >= until) break;
        __builtin_amdgcn_s_sleep(1);
      }
      const unsigned long long of_wave = __ballot(!here);
      if ((tid & 63) == 0) absent[tid >> 6] = of_wave;
    }
    if (!__syncthreads_or(tid < kHeldBlocks && !here)) break;
    // One of the absent shares, as far as they go another one in every workgroup, its maximum left in its slot; then the slots again.
    int count = 0, word = 0;
#pragma unroll
    for (int w = 0; w < kHeldBlocks / 64; ++w) count += __popcll(absent[w]);
    int nth = block % count;
    while (nth >= __popcll(absent[word])) nth -= __popcll(absent[word++]);
    unsigned long long left = absent[word];
    while (nth-- > 0) left &= left - 1;
    const int other = 64 * word + __builtin_ctzll(left);
    // (the very units that its own workgroup takes, the last one again past the end: two workgroups that leave a maximum in one slot
    // must leave the same bits, since a reader may find one word of each)
    float of_share = 0.f;
#pragma unroll 4
    for (int u = 0; u < UNITS + IN_LDS; ++u) take_abs_unit<T>(of_share, xu[min(other * THREADS + tid + u * stride, units - 1)]);
    if (other == 0 && rest < n) take_abs(of_share, T::widen(x[rest]));
    of_share = block_max<THREADS>(of_share, part);
    leave(other, of_share);
    m = fmaxf(m, of_share);
    here |= tid == other;
  }
  const float amax = block_max<THREADS>(m, part);
  if (block == 0 && tid == 0) {
    amax_out[i] = amax;
    note_amax(note, i, amax, ticket);
  }
  const float scale = 127.0f / amax;
  auto write = [&](auto quantised) __attribute__((always_inline)) {
    auto store = [&](int u, const typename T::unit& unit) {
      const int j = j0 + u * stride;
      if (j < units) __builtin_nontemporal_store(quantised(unit), &reinterpret_cast<typename T::packed*>(out)[j]);
    };
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      asm volatile("" : "+v"(v[u]));  // (or widened bfloat16 values are held from the maximum on, twice the registers)
      store(u, v[u]);
    }
#pragma unroll
    for (int k = 0; k < IN_LDS; ++k) store(UNITS + k, more[k][tid]);
  };
  if (!__any(nan) && measured_scale(amax, scale)) write([&](const typename T::unit& unit) { return quant_unit_measured(unit, scale); });
  else write([&](const typename T::unit& unit) { return quant_unit(unit, scale); });
  if (has_rest) out[rest] = (int8_t)quant1(last, scale);
}

__device__ __forceinline__ void dequant_unit(int w, float amax, v4f& r) {
  r = v4f{dequant1((int8_t)(w & 0xff), amax), dequant1((int8_t)((w >> 8) & 0xff), amax), dequant1((int8_t)((w >> 16) & 0xff), amax),
          dequant1(w >> 24, amax)};
}
__device__ __forceinline__ void dequant_unit(const v2i32& w, float amax, v8h& r) {
  v4f a, b;
  dequant_unit(w[0], amax, a);
  dequant_unit(w[1], amax, b);
  r = __builtin_bit_cast(v8h, v4i32{(int)cvt_pk_bf16(a[0], a[1]), (int)cvt_pk_bf16(a[2], a[3]), (int)cvt_pk_bf16(b[0], b[1]),
                                    (int)cvt_pk_bf16(b[2], b[3])});
}

template <typename T>
__global__ __launch_bounds__(kQuantThreads) void dequantize_i8_kernel(const int8_t* __restrict__ x, long long n, float amax,
                                                                       typename T::elem* __restrict__ out) {
  const long long units = n / T::kPerUnit;
  const typename T::packed* __restrict__ xu = reinterpret_cast<const typename T::packed*>(x);
  typename T::unit* __restrict__ ou = reinterpret_cast<typename T::unit*>(out);
  const long long stride = (long long)gridDim.x * kQuantThreads;
  long long j = (long long)blockIdx.x * kQuantThreads + threadIdx.x;
  for (; j + (kQuantUnroll - 1) * stride < units; j += kQuantUnroll * stride) {
    typename T::packed w[kQuantUnroll];
#pragma unroll
    for (int u = 0; u < kQuantUnroll; ++u) w[u] = xu[j + u * stride];
#pragma unroll
    for (int u = 0; u < kQuantUnroll; ++u) {
      typename T::unit r;
      dequant_unit(w[u], amax, r);
      __builtin_nontemporal_store(r, &ou[j + u * stride]);
    }
  }
  for (; j < units; j += stride) {
    typename T::unit r;
    dequant_unit(xu[j], amax, r);
    ou[j] = r;
  }
  if (blockIdx.x == 0 && threadIdx.x < (int)(n - T::kPerUnit * units)) {
    const long long r = T::kPerUnit * units + threadIdx.x;
    const float f = dequant1(x[r], amax);
    if constexpr (T::kPerUnit == 8) out[r] = (unsigned short)cvt_pk_bf16(f, f);
    else out[r] = f;
  }
}

inline int quant_blocks(long long units, int most) {
  const long long per = (long long)kQuantThreads * kQuantUnroll, want = (units + per - 1) / per;
  return (int)(want < 1 ? 1 : (want > most ? most : want));
}
inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
// Launches report the status of the launch itself (what hipLaunchKernel returns), not the calling thread's last
// error: an earlier failure that has nothing to do with this library is neither reported as ours nor cleared.
template <typename... Params, typename... Args>
inline hipError_t launch_kernel(void (*kernel)(Params...), int blocks, int threads, hipStream_t stream, Args... args) {
  std::tuple<Params...> by_value{static_cast<Params>(args)...};
  void* ptrs[sizeof...(Params)];
  int i = 0;
  std::apply([&](auto&... a) { ((ptrs[i++] = static_cast<void*>(&a)), ...); }, by_value);
  return hipLaunchKernel(reinterpret_cast<const void*>(kernel), dim3(blocks), dim3(threads), ptrs, 0, stream);
}
inline int status_of(hipError_t err) { return err == hipSuccess ? FMHA_I8_OK : FMHA_I8_ERR_HIP_BASE + (int)err; }

template <typename T>
int abs_max(hipStream_t stream, const typename T::elem* x, long long n, float* amax_out) {
  if (amax_out == nullptr || (x == nullptr && n > 0) || n < 0) return FMHA_I8_ERR_NULL_POINTER;
  if (!aligned16(x)) return FMHA_I8_ERR_ALIGNMENT;
  hipError_t err = launch_kernel(zero_float_kernel, 1, 1, stream, amax_out);
  if (err == hipSuccess && n > 0)
    err = launch_kernel(abs_max_kernel<T>, quant_blocks(n / T::kPerUnit, (long long)sizeof(*x) * n < kAtomicBytes ? kQuantMaxBlocks / 2 : kQuantMaxBlocks),
                        kQuantThreads, stream, x, n, amax_out);
  return status_of(err);
}

template <typename T>
int quantize(hipStream_t stream, const typename T::elem* x, long long n, float amax_host, const float* amax_dev, int8_t* out) {
  if (n < 0 || ((x == nullptr || out == nullptr) && n > 0)) return FMHA_I8_ERR_NULL_POINTER;
  if (!aligned16(x) || !aligned16(out)) return FMHA_I8_ERR_ALIGNMENT;
  if (amax_dev == nullptr && !(amax_host == amax_host)) return FMHA_I8_ERR_SCALE;
  if (n == 0) return FMHA_I8_OK;
  const int blocks = quant_blocks(n / T::kPerUnit, kQuantMaxBlocks);
  const bool nt = (long long)sizeof(typename T::elem) * n > kCacheBytes;
  return status_of(nt ? launch_kernel(quantize_i8_kernel<T, true>, blocks, kQuantThreads, stream, x, n, amax_host, amax_dev, out)
                      : launch_kernel(quantize_i8_kernel<T, false>, blocks, kQuantThreads, stream, x, n, amax_host, amax_dev, out));
}

// Tags of quantize_held_kernel, 96 bits of which 64 are a bijection of a counter that starts at random: no two calls of a process
// get the same, and memory that holds anything else matches with a chance of 2^-96.
class TagSource {
 public:
  static SlotTag next() {
    static TagSource source;
    const unsigned long long n = source.count_.fetch_add(1, std::memory_order_relaxed);
    const unsigned long long a = mixed(n), b = mixed(n ^ 0x6a09e667f3bcc909ull);
    return SlotTag{{a << 16, (a >> 48 << 48) | (b >> 32 << 16)}};
  }

 private:
  TagSource() noexcept {
    try {
      std::random_device device;
      count_ = (unsigned long long)device() << 32 | device();
    } catch (...) {  // (no source of randomness: the clock, and where this process has its memory)
      count_ = mixed((unsigned long long)std::chrono::steady_clock::now().time_since_epoch().count()) ^ (unsigned long long)reinterpret_cast<uintptr_t>(this);
    }
  }
  static unsigned long long mixed(unsigned long long z) {  // a bijection: the finaliser of SplitMix64 (Steele, Lea, Flood 2014)
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
  }
  std::atomic<unsigned long long> count_{0};
};
// Whether the current device has a compute unit for each of kHeldBlocks workgroups (a partition of a chip has not: they would wait for
// workgroups that cannot start before they end).
bool device_holds_all() {
  constexpr int kDevices = 64;
  static std::atomic<int> units[kDevices];  // 0: not asked yet
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kDevices) return false;
  int n = units[device].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || n <= 0) return false;
    units[device].store(n, std::memory_order_relaxed);
  }
  return n >= kHeldBlocks;
}
// Workgroups per tensor with `per` 16-byte units each, or false where the chip does not hold them all.
bool held_blocks(const long long* units_of, int count, int per, QuantJob& job) {
  long long need[FMHA_QUANT_MAX_TENSORS] = {}, total = 0, blocks = 0;
  for (int i = 0; i < count; ++i) {
    need[i] = units_of[i] > 0 ? (units_of[i] + per - 1) / per : 1;
    total += units_of[i];
    blocks += need[i];
  }
  if (blocks > kHeldBlocks) return false;
  const long long spare = kHeldBlocks - blocks;
  int at = 0;
  for (int i = 0; i < FMHA_QUANT_MAX_TENSORS; ++i) {
    job.first_block[i] = at;
    if (i < count) at += (int)(need[i] + (total > 0 ? spare * units_of[i] / total : 0));
  }
  job.first_block[FMHA_QUANT_MAX_TENSORS] = at;
  return true;
}
// Forms of quantize_held_kernel: threads per workgroup, units per thread in registers (16 take 106 to 124 of them) and in LDS (9: 72 KB
// of 512 threads).  The first that holds a call serves it: the fewer units, the more of the compute units share the work.
template <int THREADS, int UNITS, int IN_LDS = 0>
struct Held {
  static constexpr int kPerBlock = THREADS * (UNITS + IN_LDS);
  template <typename T, typename... Args>
  static hipError_t launch(const QuantJob& job, hipStream_t stream, Args... args) {
    return launch_kernel(quantize_held_kernel<T, THREADS, UNITS, IN_LDS>, job.first_block[FMHA_QUANT_MAX_TENSORS], THREADS, stream, job, args...);
  }
};
template <typename T, typename FORM, typename... FORMS, typename... Args>
bool launch_held(hipError_t& err, QuantJob& job, const long long* units_of, int count, hipStream_t stream, Args... args) {
  if (held_blocks(units_of, count, FORM::kPerBlock, job)) {
    err = FORM::template launch<T>(job, stream, args...);
    return true;
  }
  if constexpr (sizeof...(FORMS) > 0) return launch_held<T, FORMS...>(err, job, units_of, count, stream, args...);
  else return false;
}

template <typename T>
int measure_and_quantize(hipStream_t stream, const FMHAQuantTensor* t, int count, float* workspace, float* amax_out,
                         unsigned long long* note, unsigned ticket) {
  QuantJob job{};
  long long most = 0, least = 0x7fffffffffffffffll, total = 0;
  for (int i = 0; i < count; ++i) {
    if (t[i].n < 0 || ((t[i].x == nullptr || t[i].out == nullptr) && t[i].n > 0)) return FMHA_I8_ERR_NULL_POINTER;
    if (!aligned16(t[i].x) || !aligned16(t[i].out)) return FMHA_I8_ERR_ALIGNMENT;
    job.x[i] = t[i].x;
    job.out[i] = t[i].out;
    job.n[i] = t[i].n;
    most = t[i].n > most ? t[i].n : most;
    least = t[i].n < least ? t[i].n : least;
    total += t[i].n;
  }
  if (most <= kSmallElements)
    return status_of(launch_kernel(quantize_small_kernel<T>, count, kSmallThreads, stream, job, amax_out, note, ticket));
  // One launch, where every tensor has a unit to load; a captured call would be replayed with the tag it was captured with.
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (least >= T::kPerUnit && (reinterpret_cast<uintptr_t>(workspace) & 7) == 0 && device_holds_all() && hipStreamIsCapturing(stream, &capture) == hipSuccess &&
      capture == hipStreamCaptureStatusNone) {
    long long units_of[FMHA_QUANT_MAX_TENSORS] = {};
    for (int i = 0; i < count; ++i) units_of[i] = job.n[i] / T::kPerUnit;
    hipError_t err;
    if (launch_held<T, Held<512, 1>, Held<512, 2>, Held<512, 4>, Held<512, 8>, Held<512, 12>, Held<512, 16>, Held<512, 16, 4>, Held<512, 16, 9>,
                    Held<1024, 16>, Held<1024, 16, 4>, Held<1024, 16, 9>>(err, job, units_of, count, stream, amax_out,
                                                                        reinterpret_cast<unsigned long long*>(workspace), TagSource::next(), (unsigned)kPatience,
                                                                        note, ticket))
      return status_of(err);
  }
  int blocks = 0;
  for (int i = 0; i < FMHA_QUANT_MAX_TENSORS; ++i) {
    job.first_block[i] = blocks;
    if (i < count) blocks += quant_blocks(job.n[i] / T::kPerUnit, (int)((kQuantMaxBlocks * job.n[i] + total - 1) / total));
  }
  job.first_block[FMHA_QUANT_MAX_TENSORS] = blocks;
  hipError_t err = launch_kernel(abs_max_parts_kernel<T>, blocks, kQuantThreads, stream, job, workspace);
  if (err != hipSuccess) return status_of(err);
  return status_of(launch_kernel(quantize_by_parts_kernel<T>, blocks, kQuantThreads, stream, job, workspace, amax_out, note, ticket));
}

template <typename T>
int dequantize(hipStream_t stream, const int8_t* x, long long n, float amax, typename T::elem* out) {
  if (n < 0 || ((x == nullptr || out == nullptr) && n > 0)) return FMHA_I8_ERR_NULL_POINTER;
  if (!aligned16(x) || !aligned16(out)) return FMHA_I8_ERR_ALIGNMENT;
  if (n == 0) return FMHA_I8_OK;
  const int blocks = quant_blocks(n / T::kPerUnit, kQuantMaxBlocks);
  return status_of(launch_kernel(dequantize_i8_kernel<T>, blocks, kQuantThreads, stream, x, n, amax, out));
}

}  // namespace fmha_i8_gfx950

extern "C" {

int FMHAAbsMaxF32(hipStream_t stream, const float* x, long long n, float* amax_out) {
  return fmha_i8_gfx950::abs_max<fmha_i8_gfx950::F32>(stream, x, n, amax_out);
}
int FMHAQuantizeI8(hipStream_t stream, const float* x, long long n, float amax_host, const float* amax_dev, int8_t* out) {
  return fmha_i8_gfx950::quantize<fmha_i8_gfx950::F32>(stream, x, n, amax_host, amax_dev, out);
}
int FMHADequantizeI8(hipStream_t stream, const int8_t* x, long long n, float amax, float* out) {
  return fmha_i8_gfx950::dequantize<fmha_i8_gfx950::F32>(stream, x, n, amax, out);
}
int FMHAAbsMaxBF16(hipStream_t stream, const uint16_t* x, long long n, float* amax_out) {
  return fmha_i8_gfx950::abs_max<fmha_i8_gfx950::BF16>(stream, x, n, amax_out);
}
int FMHAQuantizeI8BF16(hipStream_t stream, const uint16_t* x, long long n, float amax_host, const float* amax_dev,
                       int8_t* out) {
  return fmha_i8_gfx950::quantize<fmha_i8_gfx950::BF16>(stream, x, n, amax_host, amax_dev, out);
}
int FMHADequantizeI8BF16(hipStream_t stream, const int8_t* x, long long n, float amax, uint16_t* out) {
  return fmha_i8_gfx950::dequantize<fmha_i8_gfx950::BF16>(stream, x, n, amax, out);
}

#ifdef FMHA_FORCED_ROUTE
// Test build only: how long quantize_held_kernel waits for the other workgroups, in ticks of 10 ns.
void FMHAQuantDebugPatience(unsigned ticks) { fmha_i8_gfx950::kPatience = ticks; }
#endif

int FMHAMeasureAndQuantizeI8(hipStream_t stream, const FMHAQuantTensor* tensors, int count, int element_type,
                             float* workspace, float* amax_out, unsigned long long* note, unsigned ticket) {
  using namespace fmha_i8_gfx950;
  if (tensors == nullptr || workspace == nullptr || amax_out == nullptr || count < 1 || count > FMHA_QUANT_MAX_TENSORS)
    return FMHA_I8_ERR_NULL_POINTER;
  return element_type == FMHA_QUANT_BF16
             ? measure_and_quantize<BF16>(stream, tensors, count, workspace, amax_out, note, ticket)
             : measure_and_quantize<F32>(stream, tensors, count, workspace, amax_out, note, ticket);
}

}  // extern "C"

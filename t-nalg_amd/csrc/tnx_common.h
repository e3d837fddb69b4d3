// Shared helpers of the gfx950 DMRG kernels: error reporting, dtype access,
// XCD-aware block remapping and wavefront reductions.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <atomic>
#include <string>

#include "../../include/tnalg_hip.h"

#define TNX_VERSION 10000

// thread-local message of the last failure (tnx_last_error)
void tnx_set_error(const char* fmt, ...);

// sampled kernel timing (prof.hip): a Lanczos call asks whether it is
// sampled, switches timing on for its first Krylov step; launch sites bracket
// their kernel with mark/done when timing is on.
enum {
  TNX_PC_GEMM_F64_1 = 0, TNX_PC_GEMM_F64_2, TNX_PC_GEMM_F32_1, TNX_PC_GEMM_F32_2,
  TNX_PC_GEMM_BF16_1, TNX_PC_GEMM_BF16_2, TNX_PC_MIX, TNX_PC_DOTS, TNX_PC_UPDATE_DOTS,
  TNX_PC_UPDATE_NORM
};
bool tnx_prof_call_begin();      // this call is sampled (timing stays off)
void tnx_prof_set(bool on);      // timing on / off for the calling thread
bool tnx_prof_on();
int tnx_prof_mark(int cls, hipStream_t s);                // -1: not timed
unsigned long long* tnx_prof_ts(int mark);                // the launch's stamp slot (or null)
void tnx_prof_done(int mark, hipStream_t s, double work);
void tnx_prof_count(int cls, double work);   // one launch of the class and its work (while armed)

// Launch-span stamps of a timed launch: the slot holds TNX_TS_PAIRS pairs
// (earliest block start, latest block end) of the device's constant wall
// clock; block b updates pair b % TNX_TS_PAIRS with vector atomics (spread
// over pairs, so no address takes more than a few dozen), and the host
// takes the minimum start and maximum end.  A null slot: not timed.
constexpr int TNX_TS_PAIRS = 64;
__device__ __forceinline__ void tnx_stamp_begin(unsigned long long* ts) {
  if (ts != nullptr && threadIdx.x == 0)
    atomicMin(ts + 2 * (blockIdx.x % TNX_TS_PAIRS), (unsigned long long)wall_clock64());
}
__device__ __forceinline__ void tnx_stamp_end(unsigned long long* ts) {
  if (ts != nullptr && threadIdx.x == 0)
    atomicMax(ts + 2 * (blockIdx.x % TNX_TS_PAIRS) + 1, (unsigned long long)wall_clock64());
}
// Grouped GEMM launch with a stamp slot (gemm.hip); tnx_gemm_grouped is this
// with a null slot.
int tnx_gemm_grouped_ts(int mode, const tnx_gemm_problem* prob, int nprob,
                        const tnx_gemm_seg* seg, int ntiles, const int32_t* active,
                        tnx_stream_t stream, unsigned long long* ts);

#define TNX_CHECK_HIP(call)                                                      \
  do {                                                                           \
    hipError_t e_ = (call);                                                      \
    if (e_ != hipSuccess) {                                                      \
      tnx_set_error("%s failed: %s (%s:%d)", #call, hipGetErrorString(e_),       \
                    __FILE__, __LINE__);                                         \
      return TNX_EHIP;                                                           \
    }                                                                            \
  } while (0)

#define TNX_CHECK_LAUNCH()                                                       \
  do {                                                                           \
    hipError_t e_ = hipGetLastError();                                           \
    if (e_ != hipSuccess) {                                                      \
      tnx_set_error("kernel launch failed: %s (%s:%d)", hipGetErrorString(e_),   \
                    __FILE__, __LINE__);                                         \
      return TNX_EHIP;                                                           \
    }                                                                            \
  } while (0)

// Once per kernel and GPU: allow it `bytes` of dynamic LDS (a launch asks for
// more than the default).  `done`: the kernel's bit set of GPUs, static.
inline int tnx_dynamic_lds(const void* kernel, size_t bytes, std::atomic<uint64_t>& done) {
  int dev = 0;
  TNX_CHECK_HIP(hipGetDevice(&dev));
  const uint64_t bit = 1ull << (dev & 63);
  if (done.load(std::memory_order_acquire) & bit) return TNX_OK;
  TNX_CHECK_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
  done.fetch_or(bit, std::memory_order_release);
  return TNX_OK;
}

typedef double tnx_d4 __attribute__((ext_vector_type(4)));
typedef float tnx_f4 __attribute__((ext_vector_type(4)));
typedef __bf16 tnx_bf8 __attribute__((ext_vector_type(8)));

// Pointers of the global address space (the records carry plain integers: a
// generic pointer made from one would be accessed with flat loads, which
// wait on the LDS counter too).
#define TNX_GLOBAL __attribute__((address_space(1)))
template <typename T> __device__ __forceinline__ T TNX_GLOBAL* as_global(uint64_t p) {
  return (T TNX_GLOBAL*)p;
}

// Descriptor records are read through the scalar cache: nothing changes them
// during a launch, and the vector counter then counts operand loads only.
#define TNX_CONST __attribute__((address_space(4)))

// Load element idx of a buffer (global memory) of runtime dtype as double.
__device__ __forceinline__ double tnx_load(const void* p, int dtype, int64_t idx) {
  const uint64_t a = (uint64_t)p;
  if (dtype == TNX_F64) return as_global<const double>(a)[idx];
  if (dtype == TNX_F32) return (double)as_global<const float>(a)[idx];
  return (double)(float)as_global<const __bf16>(a)[idx];
}

__device__ __forceinline__ void tnx_store(void* p, int dtype, int64_t idx, double v) {
  const uint64_t a = (uint64_t)p;
  if (dtype == TNX_F64) as_global<double>(a)[idx] = v;
  else if (dtype == TNX_F32) as_global<float>(a)[idx] = (float)v;
  else as_global<__bf16>(a)[idx] = (__bf16)(float)v;
}

// Workgroups are dispatched round-robin over the 8 XCDs of MI355X, each with
// its own L2.  Remap the hardware block id so that consecutive logical tiles
// (which share operands) land on the same XCD.
__device__ __forceinline__ int tnx_xcd_remap(int bid, int nblocks) {
  const int nx = 8;
  if (nblocks < nx) return bid;
  int x = bid % nx, i = bid / nx;
  int q = nblocks / nx, r = nblocks % nx;
  return x * q + (x < r ? x : r) + i;
}

// Lane exchanges of the butterflies below, all of them VALU operations
// (through the LDS crossbar, __shfl_xor, each took about 120 cycles on the
// path of every reduction).  tnx_row_get: the value that `DPP`, a rotation
// within the 16-lane row, brings from another lane.
template <int DPP> __device__ __forceinline__ double tnx_row_get(double v) {
  const long long x = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)x, DPP, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(x >> 32), DPP, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// Exchange of the odd halves (HALF: lanes 32-63; else the odd 16-lane rows) of
// p with the even ones of q.
template <bool HALF> __device__ __forceinline__ void tnx_swap(double& p, double& q) {
  const long long x = __double_as_longlong(p), y = __double_as_longlong(q);
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  u2 lo, hi;
  if constexpr (HALF) {
    lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  } else {
    lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
    hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  }
  p = __longlong_as_double(((long long)hi[0] << 32) | lo[0]);
  q = __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
}
// Butterfly over lane ^ 32, 16, 8, 4, 2, 1, the same bits in every lane.  In a
// 16-lane row a rotation by d = 8, 4, 2, 1 brings lane ^ d's value, as the
// values repeat with period 2 d by then.
template <typename F> __device__ __forceinline__ double tnx_wave_fold(double v, F f) {
  double p = v, q = v;   // after a swap: the value of the lane with the bit clear, set
  tnx_swap<true>(p, q);
  p = q = f(p, q);
  tnx_swap<false>(p, q);
  v = f(p, q);
  v = f(v, tnx_row_get<0x128>(v));
  v = f(v, tnx_row_get<0x124>(v));
  v = f(v, tnx_row_get<0x122>(v));
  return f(v, tnx_row_get<0x121>(v));
}
__device__ __forceinline__ double tnx_wave_sum(double v) {
  return tnx_wave_fold(v, [](double x, double y) { return x + y; });
}
__device__ __forceinline__ double tnx_wave_min(double v) {
  return tnx_wave_fold(v, [](double x, double y) { return fmin(x, y); });
}

// 1 / d and 1 / sqrt(x) to working accuracy, normal arguments: the hardware's
// approximation and a third-order step, a fraction of a division's or library
// root's chain.
__device__ __forceinline__ double tnx_rcp(double d) {
  const double r = __builtin_amdgcn_rcp(d);
  const double e = fma(-d, r, 1.0);
  return fma(r, fma(e, e, e), r);
}
__device__ __forceinline__ double tnx_rsqrt_step(double x, double y) {   // y ~ 1 / sqrt(x)
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}
__device__ __forceinline__ double tnx_rsqrt(double x) {
  return tnx_rsqrt_step(x, __builtin_amdgcn_rsq(x));
}

// Largest index i in [0, n) whose 32-bit field at byte offset `off` of the
// i-th record (records of `rec` bytes) is <= key.  The fields are prefix
// sums (non-decreasing, first one 0, key >= 0), so i is the record owning
// block `key`.  Called by every lane of a full wavefront with uniform
// arguments: each round the 64 lanes probe 64 evenly spaced records of the
// remaining range [lo, hi] (lane 0 probes lo, known to qualify) and the range
// shrinks to the gap after the last qualifying probe, so up to 4096 records
// cost two dependent loads instead of twelve.
__device__ __forceinline__ int tnx_find_owner(const void* base, int rec, int off, int n,
                                              int key) {
  const char* b = (const char*)base + off;
  const int lane = threadIdx.x & 63;
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int step = (hi - lo + 64) >> 6;  // ceil((hi - lo + 1) / 64)
    const int idx = lo + lane * step;
    bool ok = false;
    if (idx <= hi) ok = *(const int32_t*)(b + (int64_t)idx * rec) <= key;
    const unsigned long long m = __ballot(ok);
    lo += (63 - __clzll((long long)m)) * step;
    hi = min(hi, lo + step - 1);
  }
  return lo;
}

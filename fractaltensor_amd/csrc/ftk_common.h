// Shared helpers for the gfx950 kernels behind include/ftk.h.
#pragma once

#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>

#include <atomic>
#include <type_traits>

#include "../../include/ftk.h"

namespace ftk {

// ---- error reporting ------------------------------------------------------
// One message buffer per host thread; entry points return a code and leave the
// text here.  Kernel launch failures are turned into FTK_ERR_LAUNCH.
char* last_error_buffer();
constexpr int kErrLen = 512;

inline int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(last_error_buffer(), kErrLen, fmt, ap);
  va_end(ap);
  return code;
}

inline int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess)
    return fail(FTK_ERR_LAUNCH, "%s: %s", what, hipGetErrorString(e));
  return FTK_OK;
}

#define FTK_HIP(call)                                                        \
  do {                                                                       \
    hipError_t e_ = (call);                                                  \
    if (e_ != hipSuccess)                                                    \
      return ::ftk::fail(FTK_ERR_LAUNCH, "%s: %s", #call, hipGetErrorString(e_)); \
  } while (0)

// Set-up that a call site owes every device once (a function attribute is kept with the device's copy of the code
// object, so a process that drives two devices has to set it on both).  The set-up is idempotent: two threads that
// both find the device unprepared both do it.
class DeviceOnce {
 public:
  // true while the current device has not been prepared by this call site; *bit then goes to done()
  bool pending(unsigned* bit) const {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev > 31) {
      *bit = 0;
      return true;
    }
    *bit = 1u << dev;
    return !(seen_.load(std::memory_order_acquire) & *bit);
  }
  void done(unsigned bit) { seen_.fetch_or(bit, std::memory_order_release); }

 private:
  std::atomic<unsigned> seen_{0};
};

// The largest dynamic LDS size a call site has set on its kernel, per device: for launchers whose LDS need grows
// with the shape.  Two threads that both find the stored size too small both set the attribute; the larger one wins.
class DeviceMax {
 public:
  // true when the current device has not been given at least `value` by this call site; *dev then goes to raise()
  bool below(int value, int* dev) const {
    *dev = -1;
    int d = 0;
    if (hipGetDevice(&d) != hipSuccess || d < 0 || d >= kDevices) return true;
    *dev = d;
    return max_[d].load(std::memory_order_acquire) < value;
  }
  void raise(int dev, int value) {
    if (dev < 0) return;
    int cur = max_[dev].load(std::memory_order_relaxed);
    while (cur < value && !max_[dev].compare_exchange_weak(cur, value, std::memory_order_release)) {
    }
  }

 private:
  static constexpr int kDevices = 32;
  std::atomic<int> max_[kDevices] = {};
};

// Every workspace a stacked-LSTM entry point takes starts with this block; its first int is the status word
// that ftk_stacked_lstm_status() reads.
constexpr size_t kStatusBytes = 256;

// Device properties, queried once per device id.
struct DeviceProps {
  int cus = 0;
  int lds_optin = 0;
  int clock_khz = 0;
  int wave = 0;
  char arch[32] = {0};
};
int device_props(const DeviceProps** out);

// Launches a kernel whose workgroups wait for each other: `grid` is at most what the device holds at once.  As an
// ordinary launch while that is enough, as a cooperative one otherwise (see ftk_api.hip).
int launch_resident(const void* fn, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t s);
// Whether that is going to be a cooperative launch, as far as can be told before it is made.
bool launch_is_cooperative(hipStream_t s);
// whether s records a graph (or must not be asked because another stream does)
bool stream_records(hipStream_t s);

// ---- vector types for MFMA operands ----------------------------------------
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// Compile-time loop: the body sees its index as a constant expression
// (std::integral_constant), so register arrays indexed by it are promoted to
// registers even when the body sits under a runtime condition.
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (N > 0) {
    static_for<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

// ---- placement
// Workgroups are dealt to the 8 XCDs in turn; the index that makes those of one XCD neighbours, for any grid (XCD x has the
// x-th share of the indexes, the first `total` % 8 shares one more than the others).
__device__ __forceinline__ int xcd_consecutive(int block, int total) {
  const int x = block & 7;
  return x * (total >> 3) + min(x, total & 7) + (block >> 3);
}

// ---- device math ------------------------------------------------------------
// exp through the hardware base-2 exponential (about 1 ulp), reciprocal through
// v_rcp_f32 (1 ulp).  sigmoid is accurate to a few 1e-7 relative everywhere.
__device__ __forceinline__ float fast_exp(float x) {
  return __builtin_amdgcn_exp2f(x * 1.4426950408889634f);
}

__device__ __forceinline__ float sigmoid_f(float x) {
  return __builtin_amdgcn_rcpf(1.0f + fast_exp(-x));
}

// tanh(x) = 1 - 2/(1+e^{2x}) loses relative accuracy near 0 (the result is the difference of two numbers close to 1), so small
// arguments use a polynomial instead; the switch point keeps both branches below 2e-7 relative.  x + x z q(z), z = x^2, with the
// quadratic q whose largest relative error up to the switch is least (2.9e-9; found by weighted least squares): 6.2e-8 in fp32
// arithmetic, where x (1 + z q) with the Taylor series to x^9, an instruction more, had 8.9e-8 (rms 2.3e-8, 2.8e-8).
__device__ __forceinline__ float tanh_exp2x(float x) { return __builtin_amdgcn_exp2f(x * 2.8853900817779268f); }   // e^{2x}
__device__ __forceinline__ float tanh_zq(float z) {
  return z * __builtin_fmaf(z, __builtin_fmaf(z, -0.05143002858f, 0.13324236628f), -0.33333240088f);
}
__device__ __forceinline__ float tanh_f(float x) {
  const float big = 1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + tanh_exp2x(x));
  const float small = __builtin_fmaf(x, tanh_zq(x * x), x);
  return fabsf(x) < 0.25f ? small : big;
}

}  // namespace ftk

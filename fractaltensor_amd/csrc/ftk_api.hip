// Library-wide entry points of include/ftk.h: version, error text, device info.
#include <stdlib.h>
#include <string.h>

#include <mutex>

#include "ftk_common.h"

namespace ftk {

char* last_error_buffer() {
  static thread_local char buf[kErrLen] = {0};
  return buf;
}

int device_props(const DeviceProps** out) {
  constexpr int kMaxDev = 16;
  static DeviceProps cache[kMaxDev];
  static bool ready[kMaxDev] = {false};
  static std::mutex mu;
  int dev = 0;
  FTK_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDev) return fail(FTK_ERR_DEVICE, "device id %d out of range", dev);
  std::lock_guard<std::mutex> lock(mu);
  if (!ready[dev]) {
    hipDeviceProp_t p;
    FTK_HIP(hipGetDeviceProperties(&p, dev));
    DeviceProps d;
    d.cus = p.multiProcessorCount;
    d.lds_optin = (int)p.sharedMemPerBlockOptin;
    if (d.lds_optin <= 0) d.lds_optin = (int)p.sharedMemPerBlock;
    d.clock_khz = p.clockRate;
    d.wave = p.warpSize;
    strncpy(d.arch, p.gcnArchName, sizeof(d.arch) - 1);
    // gfx950 has 160 KB of LDS per compute unit, all of it addressable by one workgroup
    if (strncmp(d.arch, "gfx950", 6) == 0 && d.lds_optin < 163840) d.lds_optin = 163840;
    cache[dev] = d;
    ready[dev] = true;
  }
  *out = &cache[dev];
  return FTK_OK;
}

// A cooperative launch costs about 17 us on the device (it goes through a queue of its own, with barriers to and from
// the stream's): L1 T4 B16 H128, 32.0 -> 14.4 us a call without it.  What it is for is two such kernels that are each
// resident in part and wait for the rest.  Launches on one stream follow each other anyway, so a process that uses one
// stream gets ordinary launches.  When a second stream turns up while a launch of the first may still run, the new launch
// is put behind the first stream's work, and from then on the device gets cooperative launches only; so it does from
// the first stream capture on, whose graph may be replayed on any stream.  Kernels that merely occupy compute
// units end by themselves and need no care.  FTK_COOPERATIVE_LAUNCH=1: cooperative launches always (for processes that share a
// device).
int launch_resident(const void* fn, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t s) {
  constexpr int kDev = 16;
  struct Device {
    bool used = false, cooperative = false;
    hipStream_t stream = nullptr;   // of the ordinary launches so far
  };
  static Device devices[kDev];
  static std::mutex mu;
  static const bool always = [] {
    const char* e = getenv("FTK_COOPERATIVE_LAUNCH");
    return e && e[0] == '1';
  }();
  int dev = 0;
  FTK_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(mu);   // held over the launch: the streams have them in the order decided here
  bool cooperative = always || dev < 0 || dev >= kDev || s == hipStreamPerThread;   // (one handle, a stream per thread)
  if (!cooperative) {
    Device& d = devices[dev];
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (!d.cooperative) {
      if (hipStreamIsCapturing(s, &capture) != hipSuccess) (void)hipGetLastError();
      if (capture != hipStreamCaptureStatusNone) d.cooperative = true;
    }
    if (!d.cooperative && d.used && d.stream != s) {
      // (a stream under capture must not be asked: that would end its capture; nothing can be put behind it either)
      if (hipStreamIsCapturing(d.stream, &capture) != hipSuccess) (void)hipGetLastError();
      const bool capturing = capture != hipStreamCaptureStatusNone;
      const hipError_t e = capturing ? hipSuccess : hipStreamQuery(d.stream);
      if (capturing) {
        d.cooperative = true;
      } else if (e == hipErrorNotReady) {
        (void)hipGetLastError();
        hipEvent_t behind;
        FTK_HIP(hipEventCreateWithFlags(&behind, hipEventDisableTiming));
        hipError_t r = hipEventRecord(behind, d.stream);
        if (r == hipSuccess) r = hipStreamWaitEvent(s, behind, 0);
        (void)hipEventDestroy(behind);
        if (r != hipSuccess) return fail(FTK_ERR_LAUNCH, "launch behind another stream: %s", hipGetErrorString(r));
        d.cooperative = true;
      } else if (e != hipSuccess) {   // the stream is gone; its work may not be
        (void)hipGetLastError();
        FTK_HIP(hipDeviceSynchronize());
      }
    }
    if (!d.cooperative) {
      d.used = true;
      d.stream = s;
    }
    cooperative = d.cooperative;
  }
  if (cooperative) FTK_HIP(hipLaunchCooperativeKernel(fn, grid, block, args, (unsigned)lds, s));
  else FTK_HIP(hipLaunchKernel(fn, grid, block, args, lds, s));
  return FTK_OK;
}

}  // namespace ftk

extern "C" {

int ftk_version(void) { return 100; }

const char* ftk_last_error(void) { return ftk::last_error_buffer(); }

int ftk_device_info_query(ftk_device_info* out) {
  if (!out) return ftk::fail(FTK_ERR_INVALID_ARGUMENT, "ftk_device_info_query: out is NULL");
  const ftk::DeviceProps* d = nullptr;
  int rc = ftk::device_props(&d);
  if (rc) return rc;
  out->compute_units = d->cus;
  out->lds_bytes_per_block = d->lds_optin;
  out->clock_khz = d->clock_khz;
  out->wavefront_size = d->wave;
  out->persistent_slots = d->cus;  // one 256-thread workgroup with all 512 registers per lane fills a CU
  memset(out->arch, 0, sizeof(out->arch));
  strncpy(out->arch, d->arch, sizeof(out->arch) - 1);
  return FTK_OK;
}

}  // extern "C"

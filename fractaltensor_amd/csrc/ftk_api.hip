// Library-wide entry points of include/ftk.h: version, error text, device info.
#include <stdlib.h>
#include <string.h>

#include <mutex>

#include "ftk_common.h"
#include "launch_order.h"

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
// the first stream capture on, whose graph may be replayed on any stream (the first launch after it that is no
// recording is put behind the ordinary ones), and from the first launch on the per-thread handle, which is another stream in
// every thread (launch_order.h).  A replay is not seen here: a program
// lets the launches it made before a capture end before it replays.  Kernels that merely occupy compute units end by themselves and need no care.
// FTK_COOPERATIVE_LAUNCH=1: cooperative launches always (for processes that share a device).
namespace {
struct HipStreams {
  bool capturing(hipStream_t s) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &capture) != hipSuccess) (void)hipGetLastError();
    return capture != hipStreamCaptureStatusNone;
  }
  StreamState state(hipStream_t s) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    const hipError_t c = hipStreamIsCapturing(s, &capture);
    if (c != hipSuccess) (void)hipGetLastError();
    // (the default stream must not be asked either while a stream that waits for it records)
    if (c == hipErrorStreamCaptureImplicit || capture != hipStreamCaptureStatusNone) return StreamState::kCapturing;
    const hipError_t e = hipStreamQuery(s);
    if (e == hipSuccess) return StreamState::kIdle;
    (void)hipGetLastError();
    return e == hipErrorNotReady ? StreamState::kBusy : StreamState::kGone;
  }
  int put_behind(hipStream_t s, hipStream_t of) {
    hipEvent_t behind;
    FTK_HIP(hipEventCreateWithFlags(&behind, hipEventDisableTiming));
    hipError_t r = hipEventRecord(behind, of);
    if (r == hipSuccess) r = hipStreamWaitEvent(s, behind, 0);
    (void)hipEventDestroy(behind);
    if (r != hipSuccess) return fail(FTK_ERR_LAUNCH, "launch behind another stream: %s", hipGetErrorString(r));
    return FTK_OK;
  }
  int wait_for_device() {
    FTK_HIP(hipDeviceSynchronize());
    return FTK_OK;
  }
};

// The launch orders of all devices.
struct Launches {
  static constexpr int kDev = 16;
  LaunchOrder<hipStream_t> devices[kDev];
  std::mutex mu;
  const bool always = [] {
    const char* e = getenv("FTK_COOPERATIVE_LAUNCH");
    return e && e[0] == '1';
  }();
};
Launches& launches() {
  static Launches all;
  return all;
}
}  // namespace

int launch_resident(const void* fn, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t s) {
  Launches& all = launches();
  int dev = 0;
  FTK_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(all.mu);   // held over the launch: the streams have them in the order decided here
  bool cooperative = true;
  if (!all.always && dev >= 0 && dev < Launches::kDev) {
    const int rc = all.devices[dev].next(HipStreams(), s, s == hipStreamPerThread, &cooperative);
    if (rc) return rc;
  }
  if (cooperative) FTK_HIP(hipLaunchCooperativeKernel(fn, grid, block, args, (unsigned)lds, s));
  else FTK_HIP(hipLaunchKernel(fn, grid, block, args, lds, s));
  return FTK_OK;
}

bool stream_records(hipStream_t s) {
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  const hipError_t e = hipStreamIsCapturing(s, &capture);
  if (e != hipSuccess) (void)hipGetLastError();
  return e != hipSuccess || capture != hipStreamCaptureStatusNone;
}

bool launch_is_cooperative(hipStream_t s) {
  Launches& all = launches();
  int dev = 0;
  if (all.always || hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= Launches::kDev) return true;
  std::lock_guard<std::mutex> lock(all.mu);
  return all.devices[dev].cooperative(HipStreams(), s, s == hipStreamPerThread);
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

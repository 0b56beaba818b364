// runtime.hip - library-level state: ABI version, per-device facts and the workspaces.
#include <atomic>
#include <map>
#include <mutex>
#include <utility>

#include "hk_host.h"

extern "C" int hk_abi_version(void) { return HK_ABI_VERSION; }

extern "C" const char* hk_error_string(hipError_t status) { return hipGetErrorString(status); }

namespace hk {

namespace {
struct Workspace {
  void* ptr = nullptr;
  size_t bytes = 0;
  bool captured = false;  // handed out during a stream capture: a graph may hold the address
};
std::mutex g_mu;
// One grow-only workspace per (device, stream): work on one stream is ordered, so a call may
// reuse the buffer the previous call on that stream used; calls on different streams never
// share one. A buffer that a graph may hold is never freed: the buffer that takes its place is at
// least twice as large (while there is memory for that), so those kept add up to less than the one
// in use.
std::map<std::pair<int, hipStream_t>, Workspace> g_ws;
}  // namespace

// Read several times by each call that plans a launch, so without a lock: every thread that finds no
// count yet asks for the same number.
int device_cu_count() {
  constexpr int kDevices = 64;
  static std::atomic<int> count[kDevices];
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 256;
  if (dev < kDevices && (cus = count[dev].load(std::memory_order_relaxed)) > 0) return cus;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus <= 0)
    cus = 256;
  if (dev < kDevices) count[dev].store(cus, std::memory_order_relaxed);
  return cus;
}

bool stream_capturing(hipStream_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &status) != hipSuccess) {
    (void)hipGetLastError();  // the status is unknown, the call's own launch will tell
    return true;
  }
  return status != hipStreamCaptureStatusNone;
}

hipError_t device_workspace(size_t bytes, hipStream_t stream, void** out) {
  std::lock_guard<std::mutex> lk(g_mu);
  int dev = 0;
  HK_RETURN_IF_ERROR(hipGetDevice(&dev));
  Workspace& w = g_ws[std::make_pair(dev, stream)];
  if (bytes > w.bytes) {
    size_t want = bytes < (size_t(1) << 20) ? (size_t(1) << 20) : bytes;
    if (w.captured) {
      void* ptr = nullptr;
      const size_t twice = 2 * w.bytes;
      hipError_t e = hipMalloc(&ptr, want < twice ? twice : want);
      if (e == hipErrorOutOfMemory && want < twice) {
        (void)hipGetLastError();
        e = hipMalloc(&ptr, want);
      } else if (want < twice) {
        want = twice;
      }
      HK_RETURN_IF_ERROR(e);
      w = Workspace{ptr, want, false};
    } else {
      if (w.ptr) {
        // Work already queued on this stream may still read the old buffer.
        HK_RETURN_IF_ERROR(hipStreamSynchronize(stream));
        HK_RETURN_IF_ERROR(hipFree(w.ptr));
        w = Workspace{};
      }
      HK_RETURN_IF_ERROR(hipMalloc(&w.ptr, want));
      w.bytes = want;
    }
  }
  if (!w.captured && stream_capturing(stream)) w.captured = true;
  *out = w.ptr;
  return hipSuccess;
}

size_t device_workspace_bytes(hipStream_t stream) {
  std::lock_guard<std::mutex> lk(g_mu);
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  const auto it = g_ws.find(std::make_pair(dev, stream));
  return it == g_ws.end() ? 0 : it->second.bytes;
}

}  // namespace hk

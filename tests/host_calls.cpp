// A form whose kernel runs on the host (out0 = in0 + in1, out1 = in0 in1), over HIP functions on host memory: the launch
// plumbing of csrc/soa.hpp and csrc/host_arrays.hpp without a GPU (test_host_calls.py).
#include <atomic>
#include <cstdlib>
#include <map>
#include <new>

#include "soa.hpp"

static std::atomic<long> allocations_left{-1};  // the allocation after these fails; never where negative
void* operator new(size_t bytes) {
  if (allocations_left >= 0 && allocations_left-- == 0) throw std::bad_alloc();
  return std::malloc(bytes);
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

namespace {
struct Copy {
  void* to;
  const void* from;
  size_t bytes;
};
std::mutex pending_mutex;
std::map<hipStream_t, std::vector<Copy>> pending;  // queued on a stream, done when it is waited for
void drain(hipStream_t s) {
  std::lock_guard<std::mutex> lock(pending_mutex);
  const auto at = pending.find(s);
  if (at == pending.end()) return;
  for (const Copy& c : at->second) std::memcpy(c.to, c.from, c.bytes);
  pending.erase(at);
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) { return (*p = std::malloc(bytes)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { return hipMalloc(p, bytes); }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpy(void* to, const void* from, size_t bytes, hipMemcpyKind) { return drain(nullptr), std::memcpy(to, from, bytes), hipSuccess; }
hipError_t hipMemcpyAsync(void* to, const void* from, size_t bytes, hipMemcpyKind, hipStream_t) { return std::memcpy(to, from, bytes), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return hipMalloc((void**)s, 1); }
hipError_t hipStreamDestroy(hipStream_t s) { return hipFree(s); }
hipError_t hipStreamSynchronize(hipStream_t s) { return drain(s), hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* c) { return *c = hipStreamCaptureStatusNone, hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipMalloc((void**)e, 1); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipMalloc((void**)e, 1); }
hipError_t hipEventDestroy(hipEvent_t e) { return hipFree(e); }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1, hipSuccess; }
}

namespace combustion::device {
void check(hipError_t e, const char* what) {
  if (e != hipSuccess) throw Error(what);
}
}  // namespace combustion::device

struct HostForm : combustion::SoAForm {
  struct Captured {
    const double* const* in;
    double* const* out;
    size_t n;
  };
  std::vector<Captured> launches;
  std::mutex mutex;
  HostForm() : SoAForm(2, 2) {}
  void launch(const double* const* in, double* const* out, size_t n, const combustion::Launch&) override {
    const Captured c{in, out, n};
    {
      std::lock_guard<std::mutex> lock(mutex);
      launches.push_back(c);
    }
    kernel(c);
  }
  static void kernel(const Captured& c) {
    for (size_t s = 0; s < c.n; s++) {
      const double a = c.in[0][s], b = c.in[1][s];
      c.out[0][s] = a + b;
      c.out[1][s] = a * b;
    }
  }
};

extern "C" {
void* form_new() { return new HostForm; }
void form_free(void* f) { delete (HostForm*)f; }
// 0, or 1 where the call failed.
int form_call(void* f, const double* const* in, size_t n, double* const* out, int on_device, void* stream) {
  try {
    ((HostForm*)f)->call(in, n, out, on_device != 0, (hipStream_t)stream, nullptr);
  } catch (const std::exception&) {
    return 1;
  }
  return 0;
}
void fail_allocation(long n) { allocations_left = n; }
long unused_allocations() { return allocations_left; }
size_t form_launches(void* f) { return ((HostForm*)f)->launches.size(); }
// A launch again with the table it was given, as a captured graph replays it.
void form_replay(void* f, size_t launch) { HostForm::kernel(((HostForm*)f)->launches[launch]); }
void queue_copy(void* stream, void* to, const void* from, size_t bytes) { pending[(hipStream_t)stream].push_back({to, from, bytes}); }
}

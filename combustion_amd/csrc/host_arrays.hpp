// Calls of a module on host arrays: slices of the states through pinned and device staging that the module keeps, two
// slices in flight, so that one's copies run beside the other's kernels and host-side copies.
#pragma once
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

#include "device.hpp"

namespace combustion {

// Copies rows between memory regions on the calling thread and a few helpers that live as long as the team.
class CopyTeam {
 public:
  explicit CopyTeam(int helpers) {
    try {
      threads_.reserve(helpers);
      for (int i = 0; i < helpers; i++) threads_.emplace_back([this] { work(); });
    } catch (const std::exception&) {  // no thread or no memory for one: fewer helpers, or none
    }
  }
  ~CopyTeam() {
    {
      std::lock_guard<std::mutex> lock(mutex_);
      stop_ = true;
    }
    wake_.notify_all();
    for (std::thread& t : threads_) t.join();
  }
  CopyTeam(const CopyTeam&) = delete;
  CopyTeam& operator=(const CopyTeam&) = delete;

  // row(i) for every i < rows, all complete on return.
  void run(int rows, const std::function<void(int)>& row) {
    std::unique_lock<std::mutex> lock(mutex_);
    row_ = &row;
    rows_ = rows;
    next_ = 0;
    left_ = rows;
    if (!threads_.empty() && rows > 1) wake_.notify_all();
    take(lock);
    done_.wait(lock, [&] { return left_ == 0; });
    row_ = nullptr;
  }

 private:
  std::vector<std::thread> threads_;
  std::mutex mutex_;
  std::condition_variable wake_, done_;
  const std::function<void(int)>* row_ = nullptr;
  int rows_ = 0, next_ = 0, left_ = 0;
  bool stop_ = false;

  void take(std::unique_lock<std::mutex>& lock) {
    while (row_ && next_ < rows_) {
      const int i = next_++;
      const auto& row = *row_;
      lock.unlock();
      row(i);
      lock.lock();
      if (--left_ == 0) done_.notify_all();
    }
  }
  void work() {
    std::unique_lock<std::mutex> lock(mutex_);
    while (!stop_) {
      take(lock);
      if (stop_) break;
      wake_.wait(lock);
    }
  }
};

// Staging of one module: two slots of pinned and device memory, allocated with the first call on host arrays, grown to
// at most kSlotBytes each (or one group of 64 states) and given back with the module. The slots' streams live as long
// as a call: streams share the GPU's few hardware queues, and an idle one may sit in the way of another module's.
class HostArrays {
 public:
  static constexpr size_t kSlotBytes = size_t(16) << 20;
  static constexpr size_t kThreadedBytes = size_t(1) << 20;  // below, helpers cost more than they copy

  HostArrays(int n_in, int n_out) : n_in_(n_in), n_out_(n_out) {}
  ~HostArrays() { release(); }
  HostArrays(const HostArrays&) = delete;
  HostArrays& operator=(const HostArrays&) = delete;

  // Whether the arrays may go slice by slice: not where an output overlaps an input at another offset, whose later
  // states it would overwrite before they are read, or another output, where the later one of the two has to end on top.
  bool sliceable(const double* const* inputs, size_t n, double* const* outputs) const {
    for (int o = 0; o < n_out_; o++) {
      for (int i = 0; i < n_in_; i++)
        if (outputs[o] != inputs[i] && outputs[o] < inputs[i] + n && inputs[i] < outputs[o] + n) return false;
      for (int p = 0; p < o; p++)
        if (outputs[o] < outputs[p] + n && outputs[p] < outputs[o] + n) return false;
    }
    return true;
  }

  // run(slot, din, n, dout, stream) launches the module's kernels on a slot's device arrays, on `stream`.
  template <class Run>
  void call(const double* const* inputs, size_t n, double* const* outputs, Run&& run) {
    const size_t rows = (size_t)(n_in_ + n_out_);
    // whole groups of 64 states, as many as a slot holds (one group at the least), evenly over the slices
    const size_t most = std::max<size_t>(64, kSlotBytes / (rows * sizeof(double)) / 64 * 64);
    const size_t slices = (n + most - 1) / most, per = ((n + slices - 1) / slices + 63) / 64 * 64;
    reserve(per);
    struct Streams {
      HostArrays& h;
      void create() {
        for (Slot& s : h.slots_) device::check(hipStreamCreateWithFlags(&s.stream, hipStreamNonBlocking), "hipStreamCreateWithFlags");
      }
      ~Streams() {  // nothing is in flight on return, an exception's included
        for (Slot& s : h.slots_) {
          if (!s.stream) continue;
          (void)hipStreamSynchronize(s.stream);
          (void)hipStreamDestroy(s.stream);
          s.stream = nullptr;
        }
      }
    };
    Streams streams{*this};
    streams.create();
    CopyTeam team(n * rows * sizeof(double) < kThreadedBytes ? 0 : helpers());
    auto finish = [&](size_t slice) {
      Slot& s = slots_[slice % 2];
      const size_t first = slice * per, count = std::min(per, n - first);
      device::check(hipStreamSynchronize(s.stream), "hipStreamSynchronize");
      team.run(n_out_, [&](int i) { std::memcpy(outputs[i] + first, s.pinned + (n_in_ + i) * per, count * sizeof(double)); });
    };
    std::vector<const double*> din(n_in_);
    std::vector<double*> dout(n_out_);
    size_t slice = 0;
    for (size_t first = 0; first < n; first += per, slice++) {
      if (slice >= 2) finish(slice - 2);
      Slot& s = slots_[slice % 2];
      const size_t count = std::min(per, n - first);
      for (int i = 0; i < n_in_; i++) din[i] = s.device + i * per;
      for (int i = 0; i < n_out_; i++) dout[i] = s.device + (n_in_ + i) * per;
      team.run(n_in_, [&](int i) { std::memcpy(s.pinned + i * per, inputs[i] + first, count * sizeof(double)); });
      device::check(hipMemcpyAsync(s.device, s.pinned, n_in_ * per * sizeof(double), hipMemcpyHostToDevice, s.stream), "hipMemcpyAsync H2D");
      run((int)(slice % 2), din.data(), count, dout.data(), s.stream);
      device::check(hipMemcpyAsync(s.pinned + n_in_ * per, s.device + n_in_ * per, n_out_ * per * sizeof(double), hipMemcpyDeviceToHost, s.stream),
                    "hipMemcpyAsync D2H");
    }
    for (size_t i = slice >= 2 ? slice - 2 : 0; i < slice; i++) finish(i);
  }

 private:
  struct Slot {
    double *pinned = nullptr, *device = nullptr;
    hipStream_t stream = nullptr;
  };
  int n_in_, n_out_;
  Slot slots_[2];
  size_t capacity_ = 0;  // states per slot

  static int helpers() { return (int)std::min(7u, std::max(1u, std::thread::hardware_concurrency()) - 1); }

  void reserve(size_t states) {
    if (states <= capacity_) return;
    release();
    const size_t bytes = (size_t)(n_in_ + n_out_) * states * sizeof(double);
    for (Slot& s : slots_) {
      device::check(hipHostMalloc((void**)&s.pinned, bytes, hipHostMallocDefault), "hipHostMalloc");
      device::check(hipMalloc((void**)&s.device, bytes), "hipMalloc staging");
    }
    capacity_ = states;
  }
  void release() {
    for (Slot& s : slots_) {
      if (s.pinned) (void)hipHostFree(s.pinned);
      if (s.device) (void)hipFree(s.device);
      s = Slot{};
    }
    capacity_ = 0;
  }
};

}  // namespace combustion

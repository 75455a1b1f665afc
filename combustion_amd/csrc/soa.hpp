// Launch plumbing shared by every form: SoA pointer tables in device memory, host-buffer staging, the ordering
// of a module's calls across streams and kernel timing with HIP events on the caller's stream.
#pragma once
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <vector>

#include "device.hpp"
#include "forms.hpp"
#include "host_arrays.hpp"

namespace combustion {

class SoAForm : public Form {
 public:
  SoAForm(int n_inputs, int n_outputs) : n_in_(n_inputs), n_out_(n_outputs) {}
  ~SoAForm() override {
    for (void* slab : slabs_) (void)hipFree(slab);
    for (const StagingTable& t : staging_) (void)hipFree(t.table);
    if (start_) (void)hipEventDestroy(start_);
    if (stop_) (void)hipEventDestroy(stop_);
    if (done_) (void)hipEventDestroy(done_);
  }
  int n_inputs() const override { return n_in_; }
  int n_outputs() const override { return n_out_; }

  void call(const double* const* inputs, size_t n, double* const* outputs, bool on_device, hipStream_t stream, float* kernel_ms) override {
    if (n == 0) {
      if (kernel_ms) *kernel_ms = 0;
      return;
    }
    if (!on_device) {
      std::lock_guard<std::mutex> lock(host_mutex_);  // the staging is one for all the threads that share the module
      // Work queued on the default stream (and, through it, on the streams that synchronize with it) and on the caller's
      // may still write the inputs or read the outputs, and the host copies begin at once.
      device::check(hipStreamSynchronize(nullptr), "hipStreamSynchronize");
      if (stream) device::check(hipStreamSynchronize(stream), "hipStreamSynchronize");
      // A form with work memory of its own reports on whole calls (the surrogate's fallback count), so its states go in
      // one slice; the others in slices that stay within the staging.
      if (!host_) host_ = std::make_unique<HostArrays>(n_in_, n_out_);
      if (work_bytes(n) == 0 && host_->sliceable(inputs, n, outputs)) {
        if (kernel_ms) *kernel_ms = 0;
        host_->call(inputs, n, outputs, [&](int slot, const double* const* din, size_t count, double* const* dout, hipStream_t slot_stream) {
          float ms = 0;
          run(staging_table(staging_[slot], pointer_set(din, dout)), count, slot_stream, kernel_ms ? &ms : nullptr);
          if (kernel_ms) *kernel_ms += ms;
        });
        return;
      }
      std::vector<double*> din(n_in_, nullptr), dout(n_out_, nullptr);
      struct Free {
        std::vector<double*>& a;
        std::vector<double*>& b;
        ~Free() {
          for (double* p : a) (void)hipFree(p);
          for (double* p : b) (void)hipFree(p);
        }
      } release{din, dout};
      for (int i = 0; i < n_in_; i++) {
        device::check(hipMalloc(&din[i], n * sizeof(double)), "hipMalloc");
        device::check(hipMemcpy(din[i], inputs[i], n * sizeof(double), hipMemcpyHostToDevice), "hipMemcpy H2D");
      }
      for (int i = 0; i < n_out_; i++) device::check(hipMalloc(&dout[i], n * sizeof(double)), "hipMalloc");
      run(table_for(pointer_set(din.data(), dout.data())), n, stream, kernel_ms);
      device::check(hipStreamSynchronize(stream), "hipStreamSynchronize");
      forget_table(din.data(), dout.data());  // the staging arrays are freed on return
      for (int i = 0; i < n_out_; i++)
        device::check(hipMemcpy(outputs[i], dout[i], n * sizeof(double), hipMemcpyDeviceToHost), "hipMemcpy D2H");
      return;
    }
    run(table_for(pointer_set(inputs, outputs)), n, stream, kernel_ms);
  }

 protected:
  void launch_only(const double* const* in, double* const* out, size_t n, hipStream_t stream, void* work) override {
    if (n) launch(in, out, n, Launch{stream, true, work});
  }

 protected:
  // in/out: device tables of device pointers.
  virtual void launch(const double* const* in, double* const* out, size_t n, const Launch& how) = 0;

  // Orders this call after the module's previous call when the two come on different streams, so that state the
  // module keeps between its kernels (the surrogate's fallback list) is never shared by two calls in flight. Not
  // while the stream is being captured into a graph: the caller orders captured work.
  void order_after_previous_call(hipStream_t stream) {
    if (capturing(stream)) return;
    if (done_ && stream != last_stream_) device::check(hipStreamWaitEvent(stream, done_, 0), "hipStreamWaitEvent");
  }
  void mark_call_done(hipStream_t stream) {
    if (capturing(stream)) return;
    if (!done_) device::check(hipEventCreateWithFlags(&done_, hipEventDisableTiming), "hipEventCreateWithFlags");
    device::check(hipEventRecord(done_, stream), "hipEventRecord");
    last_stream_ = stream;
  }

 private:
  // One device table of the arrays' pointers per distinct set of arrays, written once when the set is first seen and
  // not rewritten until its set is forgotten: a launch still in flight on any stream, or a graph captured from this
  // module, keeps reading the table it was given. Past kMaxTables sets the device is synchronized and the tables
  // are used again (graphs captured before that point must then be captured again).
  static constexpr size_t kMaxTables = 1024;
  int n_in_, n_out_;
  std::map<std::vector<const void*>, void*> tables_;
  hipEvent_t start_ = nullptr, stop_ = nullptr, done_ = nullptr;
  hipStream_t last_stream_ = nullptr;
  std::unique_ptr<HostArrays> host_;
  std::mutex host_mutex_;

  // The null stream is never captured, and asking costs a runtime call.
  static bool capturing(hipStream_t stream) {
    if (!stream) return false;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    device::check(hipStreamIsCapturing(stream, &capture), "hipStreamIsCapturing");
    return capture != hipStreamCaptureStatusNone;
  }

  // Tables come from slabs of kSlabTables (at most kMaxTables in all): a first call on new arrays pays one copy and, at a
  // slab's first table only, an allocation. The copy is complete before the launch, so that any stream or graph may
  // read the table; it is not on a stream of its own, because the few hardware queues would then be shared by the
  // streams that the kernels run on.
  static constexpr size_t kSlabTables = 64;
  std::vector<void*> slabs_, free_tables_;

  void* table_for(const std::vector<const void*>& ptrs) {
    auto it = tables_.find(ptrs);
    if (it != tables_.end()) return it->second;
    const size_t bytes = (ptrs.size() * sizeof(void*) + 255) / 256 * 256;
    if (free_tables_.empty()) {
      if (tables_.size() >= kMaxTables) {
        device::check(hipDeviceSynchronize(), "hipDeviceSynchronize");
        for (auto& t : tables_) free_tables_.push_back(t.second);
        tables_.clear();
      } else {
        void* slab = nullptr;
        device::check(hipMalloc(&slab, kSlabTables * bytes), "hipMalloc tables");
        slabs_.push_back(slab);
        for (size_t i = kSlabTables; i-- > 0;) free_tables_.push_back((char*)slab + i * bytes);
      }
    }
    void* table = free_tables_.back();
    device::check(hipMemcpy(table, ptrs.data(), ptrs.size() * sizeof(void*), hipMemcpyHostToDevice), "hipMemcpy table");
    free_tables_.pop_back();
    tables_.emplace(ptrs, table);
    return table;
  }

  // A staging slot's table, rewritten when the size of a call's slices moves the slot's arrays: every launch of the call
  // before has completed, no graph is captured on host arrays, and the tables of the callers' own arrays stay untouched.
  struct StagingTable {
    void* table = nullptr;
    std::vector<const void*> ptrs;
  };
  StagingTable staging_[2];

  void* staging_table(StagingTable& t, std::vector<const void*> ptrs) {
    if (!t.table) device::check(hipMalloc(&t.table, ptrs.size() * sizeof(void*)), "hipMalloc table");
    if (t.ptrs != ptrs) {
      t.ptrs.clear();
      device::check(hipMemcpy(t.table, ptrs.data(), ptrs.size() * sizeof(void*), hipMemcpyHostToDevice), "hipMemcpy table");
      t.ptrs = std::move(ptrs);
    }
    return t.table;
  }

  std::vector<const void*> pointer_set(const double* const* inputs, double* const* outputs) const {
    std::vector<const void*> ptrs;
    for (int i = 0; i < n_in_; i++) ptrs.push_back(inputs[i]);
    for (int i = 0; i < n_out_; i++) ptrs.push_back(outputs[i]);
    return ptrs;
  }

  // Gives back the table of a pointer set whose launches have completed.
  void forget_table(const double* const* inputs, double* const* outputs) {
    auto it = tables_.find(pointer_set(inputs, outputs));
    if (it == tables_.end()) return;
    free_tables_.push_back(it->second);
    tables_.erase(it);
  }

  void run(void* table, size_t n, hipStream_t stream, float* kernel_ms) {
    auto in = (const double* const*)table;
    auto out = (double* const*)((const void**)table + n_in_);
    order_after_previous_call(stream);
    if (kernel_ms) {
      if (!start_) {
        device::check(hipEventCreate(&start_), "hipEventCreate");
        device::check(hipEventCreate(&stop_), "hipEventCreate");
      }
      device::check(hipEventRecord(start_, stream), "hipEventRecord");
      launch(in, out, n, Launch{stream, false, nullptr});
      device::check(hipEventRecord(stop_, stream), "hipEventRecord");
      mark_call_done(stream);
      device::check(hipEventSynchronize(stop_), "hipEventSynchronize");
      device::check(hipEventElapsedTime(kernel_ms, start_, stop_), "hipEventElapsedTime");
    } else {
      launch(in, out, n, Launch{stream, false, nullptr});
      mark_call_done(stream);
    }
  }
};

}  // namespace combustion

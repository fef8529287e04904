// Large copies between caller memory (pageable) and the device.
//
// hipMemcpy from or to pageable memory goes through the runtime's own staging with one thread, and a fresh result
// array costs a page fault (and the kernel's zeroing) for every page on top: 111 MB of parameters took 11 ms one way,
// where the link moves them in 2.  Here a few threads each take chunks through a pair of pinned buffers of their own, so
// that the link, the copies and the page faults overlap: 10.8 -> 3.1 ms for the 111 MB parameter vector of 3072 variables
// at K = 32, 1.58 -> 0.84 ms for 28 MB, 0.50 -> 0.41 ms for 8 MB (one thread).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <memory>
#include <mutex>
#include <vector>

namespace pcm {

class HostStage {
 public:
  // The current device's stage: made on first use, given back (pinned memory and events) when the last circuit that asked
  // for it is gone.  At most kThreads x 2 x kChunk bytes of pinned memory.
  static std::shared_ptr<HostStage> shared();
  ~HostStage();
  // Both return when the whole copy is done, or with an error when none of it is under way any more.  Ordered behind what
  // `stream` holds, which is waited for first: one transfer at a time goes through the buffers, and calls from several
  // threads queue up for those that are moving, not for a stream that is still at work.
  void to_host(void* dst, const void* d_src, size_t bytes, hipStream_t stream);
  void to_device(void* d_dst, const void* src, size_t bytes, hipStream_t stream);
  // Makes the buffers for a transfer of this size, so that none is made within it.
  void reserve(size_t bytes);

 private:
  static constexpr int kThreads = 6;
  static constexpr size_t kChunk = (size_t)2 << 20;
  static constexpr size_t kSmall = (size_t)1 << 20;   // below: a plain copy
  struct Lane {   // what one thread works with
    char* buf[2] = {nullptr, nullptr};
    hipEvent_t ev[2] = {nullptr, nullptr};
    void make();
    void give_back();
  };
  HostStage() = default;
  int lanes_for(size_t bytes) const;
  template <typename F>
  void run(size_t bytes, hipStream_t stream, F&& lane_work);
  std::mutex mu_;
  Lane lanes_[kThreads];
};

}  // namespace pcm

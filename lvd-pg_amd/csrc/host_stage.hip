#include "host_stage.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <map>
#include <thread>

#include "common.hpp"

namespace pcm {

std::shared_ptr<HostStage> HostStage::shared() {
  static std::mutex mu;
  static std::map<int, std::weak_ptr<HostStage>> held;   // by device
  int dev = 0;
  PCM_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(mu);
  std::shared_ptr<HostStage> s = held[dev].lock();
  if (!s) held[dev] = s = std::shared_ptr<HostStage>(new HostStage);
  return s;
}

HostStage::~HostStage() {
  for (Lane& l : lanes_) l.give_back();
}

void HostStage::Lane::make() {
  for (int i = 0; i < 2; ++i) {
    if (!buf[i]) PCM_HIP(hipHostMalloc((void**)&buf[i], kChunk, hipHostMallocPortable));
    if (!ev[i]) PCM_HIP(hipEventCreateWithFlags(&ev[i], hipEventDisableTiming));
  }
}

void HostStage::Lane::give_back() {
  for (hipEvent_t& e : ev)
    if (e) (void)hipEventDestroy(e);
  for (char*& b : buf)
    if (b) (void)hipHostFree(b);
}

// Every thread has two chunks under way, so a transfer is worth a thread per four; the caller's thread is one of them.
int HostStage::lanes_for(size_t bytes) const {
  const int want = (int)std::min<size_t>(kThreads, std::max<size_t>(1, bytes / (4 * kChunk)));
  return std::max(1, std::min(want, (int)std::thread::hardware_concurrency()));
}

void HostStage::reserve(size_t bytes) {
  if (bytes < kSmall) return;
  std::lock_guard<std::mutex> lock(mu_);
  for (int i = 0; i < lanes_for(bytes); ++i) lanes_[i].make();
}

// lane_work(lane, next): takes chunk numbers from `next` until there are none.
template <typename F>
void HostStage::run(size_t bytes, hipStream_t stream, F&& lane_work) {
  int dev = 0;
  PCM_HIP(hipGetDevice(&dev));
  const int n = lanes_for(bytes);
  for (int i = 0; i < n; ++i) lanes_[i].make();
  std::atomic<size_t> next{0};
  std::atomic<int> failed{0};
  auto work = [&](int i) {
    try {
      lane_work(lanes_[i], next);
    } catch (...) {   // (reported by the caller's thread; the others run out of chunks)
      failed = 1;
      next = bytes;
    }
  };
  std::vector<std::thread> others;
  others.reserve(n);
  try {
    for (int i = 1; i < n; ++i)
      others.emplace_back([&, i] {
        if (hipSetDevice(dev) != hipSuccess) { failed = 1; return; }
        work(i);
      });
  } catch (const std::system_error&) {   // no more threads to be had: those that run take all the chunks
  }
  work(0);
  for (std::thread& t : others) t.join();
  if (failed) {
    (void)hipStreamSynchronize(stream);   // whatever is under way on the buffers or the caller's memory ends before they are free
    fail(PCM_ERR_HIP, "a staged copy of %zu bytes between host and device failed", bytes);
  }
}

void HostStage::to_host(void* dst, const void* d_src, size_t bytes, hipStream_t stream) {
  if (bytes < kSmall) {
    if (bytes) PCM_HIP(hipMemcpyAsync(dst, d_src, bytes, hipMemcpyDeviceToHost, stream));
    PCM_HIP(hipStreamSynchronize(stream));
    return;
  }
  PCM_HIP(hipStreamSynchronize(stream));
  std::lock_guard<std::mutex> lock(mu_);
  run(bytes, stream, [&](Lane& l, std::atomic<size_t>& next) {
    size_t at[2] = {bytes, bytes};
    auto request = [&](int b) {
      at[b] = std::min(bytes, next.fetch_add(1) * kChunk);
      if (at[b] == bytes) return;
      PCM_HIP(hipMemcpyAsync(l.buf[b], static_cast<const char*>(d_src) + at[b], std::min(kChunk, bytes - at[b]),
                             hipMemcpyDeviceToHost, stream));
      PCM_HIP(hipEventRecord(l.ev[b], stream));
    };
    request(0);
    request(1);
    for (int b = 0; at[b] < bytes; b ^= 1) {
      PCM_HIP(hipEventSynchronize(l.ev[b]));
      std::memcpy(static_cast<char*>(dst) + at[b], l.buf[b], std::min(kChunk, bytes - at[b]));
      request(b);
    }
  });
}

void HostStage::to_device(void* d_dst, const void* src, size_t bytes, hipStream_t stream) {
  if (bytes < kSmall) {
    if (bytes) PCM_HIP(hipMemcpyAsync(d_dst, src, bytes, hipMemcpyHostToDevice, stream));
    PCM_HIP(hipStreamSynchronize(stream));
    return;
  }
  PCM_HIP(hipStreamSynchronize(stream));
  std::lock_guard<std::mutex> lock(mu_);
  run(bytes, stream, [&](Lane& l, std::atomic<size_t>& next) {
    bool used[2] = {false, false};
    for (int b = 0;; b ^= 1) {
      const size_t at = next.fetch_add(1) * kChunk;
      if (at >= bytes) break;
      if (used[b]) PCM_HIP(hipEventSynchronize(l.ev[b]));
      const size_t len = std::min(kChunk, bytes - at);
      std::memcpy(l.buf[b], static_cast<const char*>(src) + at, len);
      PCM_HIP(hipMemcpyAsync(static_cast<char*>(d_dst) + at, l.buf[b], len, hipMemcpyHostToDevice, stream));
      PCM_HIP(hipEventRecord(l.ev[b], stream));
      used[b] = true;
    }
  });
  PCM_HIP(hipStreamSynchronize(stream));
}

}  // namespace pcm

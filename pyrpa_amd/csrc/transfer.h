// Copies between the caller's (pageable) arrays and the device.
//
// The runtime's copy of pageable memory goes through one staging thread, which
// also takes the page faults of a freshly allocated result: 5-8 GB/s measured.
// Here a few threads each move 2 MB pieces through pinned buffers of their own,
// so the faults and the host-side copies run in parallel with the transfers.
// The threads live for one copy; the pinned buffers (32 MB) are kept and given
// back by gmod_release_memory.  Callers hold the library's lock.
#pragma once
#include <atomic>
#include <thread>

#include "gmod_common.h"

namespace gmod {

class HostCopy {
 public:
  HostCopy() = default;
  HostCopy(const HostCopy&) = delete;
  HostCopy& operator=(const HostCopy&) = delete;
  ~HostCopy() { join(); }
  // device -> host after the work queued on s; runs beside what s does next
  // (which must not write src) until wait()
  void start(void* dst, const void* src, size_t bytes, hipStream_t s);
  void wait();  // joins; throws if a transfer failed

 private:
  friend void copy_to_device(void* dst, const void* src, size_t bytes, hipStream_t s);
  void run(char* dst, const char* src, size_t bytes, bool to_host, hipStream_t s);
  void join();
  bool owner_ = false;  // of the staging buffers, from run() to join()
  std::vector<std::thread> threads_;
  std::atomic<int> error_{0};
};

// the copy is complete on return (small ones to the device: in stream order)
void copy_to_host(void* dst, const void* src, size_t bytes, hipStream_t s);
void copy_to_device(void* dst, const void* src, size_t bytes, hipStream_t s);
void release_transfer_buffers();

}  // namespace gmod

// Parallel staged copies (see transfer.h).
#include "transfer.h"

#include <algorithm>

namespace gmod {

namespace {
constexpr size_t PIECE = size_t(2) << 20;
// below this one transfer of the runtime is faster than starting the threads
// (8 threads: about 0.2 ms; 8 MB take 1 ms through the runtime)
constexpr size_t SMALL = size_t(8) << 20;
constexpr int MAX_THREADS = 8;

struct Slot {
  void* pin = nullptr;
  hipEvent_t ev = nullptr;
};
Slot g_slots[2 * MAX_THREADS];
hipStream_t g_stream = nullptr;
hipEvent_t g_before = nullptr;
bool g_busy = false;  // one staged copy at a time uses the buffers

// false (and the runtime's own copy is used) when pinned memory is short
bool prepare_slots() {
  auto ok = [](hipError_t e) {
    if (e != hipSuccess) (void)hipGetLastError();
    return e == hipSuccess;
  };
  if (!g_stream && !ok(hipStreamCreateWithFlags(&g_stream, hipStreamNonBlocking))) return false;
  if (!g_before && !ok(hipEventCreateWithFlags(&g_before, hipEventDisableTiming))) return false;
  for (Slot& q : g_slots) {
    if (!q.ev && !ok(hipEventCreateWithFlags(&q.ev, hipEventDisableTiming))) return false;
    if (!q.pin && !ok(hipHostMalloc(&q.pin, PIECE, hipHostMallocDefault))) return false;
  }
  return true;
}
}  // namespace

void release_transfer_buffers() {
  if (g_busy) return;
  for (Slot& q : g_slots)
    if (q.pin) {
      (void)hipHostFree(q.pin);
      q.pin = nullptr;
    }
}

void HostCopy::run(char* dst, const char* src, size_t bytes, bool to_host, hipStream_t s) {
  const size_t n = (bytes + PIECE - 1) / PIECE;
  const unsigned hw = std::max(2u, std::thread::hardware_concurrency());
  const int nt = (int)std::min<size_t>(n, std::min<unsigned>(MAX_THREADS, hw / 2));
  threads_.reserve(nt);
  // both directions wait for what s holds: its kernels write the source, or
  // still use the block that the destination was allocated from
  GMOD_HIP(hipEventRecord(g_before, s));
  GMOD_HIP(hipStreamWaitEvent(g_stream, g_before, 0));
  g_busy = owner_ = true;
  const int dev = ctx().device;
  auto work = [=](int t) {
    auto ok = [&](hipError_t e) {
      if (e != hipSuccess) error_.store((int)e);
      return e == hipSuccess;
    };
    if (!ok(hipSetDevice(dev))) return;
    auto len = [=](size_t i) { return std::min(PIECE, bytes - i * PIECE); };
    Slot* q = g_slots + 2 * t;
    size_t held[2];
    int k = 0, nheld = 0;  // pieces in flight, the oldest in slot (k - nheld) & 1
    auto retire = [&]() {
      const int b = (k - nheld) & 1;
      if (!ok(hipEventSynchronize(q[b].ev))) return false;
      if (to_host) memcpy(dst + held[b] * PIECE, q[b].pin, len(held[b]));
      --nheld;
      return true;
    };
    for (size_t i = t; i < n; i += nt) {
      if (nheld == 2 && !retire()) return;
      const int b = k & 1;
      if (!to_host) memcpy(q[b].pin, src + i * PIECE, len(i));
      if (!ok(to_host ? hipMemcpyAsync(q[b].pin, src + i * PIECE, len(i), hipMemcpyDeviceToHost, g_stream)
                      : hipMemcpyAsync(dst + i * PIECE, q[b].pin, len(i), hipMemcpyHostToDevice, g_stream)) ||
          !ok(hipEventRecord(q[b].ev, g_stream)))
        return;
      held[b] = i;
      ++k;
      ++nheld;
    }
    while (nheld > 0)
      if (!retire()) return;
  };
  for (int t = 0; t < nt; ++t) {
    try {
      threads_.emplace_back(work, t);
    } catch (...) {  // no thread to be had: its pieces are copied here
      work(t);
    }
  }
}

void HostCopy::join() {
  if (!owner_) return;
  for (auto& t : threads_) t.join();
  threads_.clear();
  // a worker that failed leaves its pieces in flight
  if (error_.load()) (void)hipStreamSynchronize(g_stream);
  g_busy = owner_ = false;
}

void HostCopy::start(void* dst, const void* src, size_t bytes, hipStream_t s) {
  if (bytes < SMALL || g_busy || !prepare_slots()) {
    GMOD_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s));
    GMOD_HIP(hipStreamSynchronize(s));
    return;
  }
  run(static_cast<char*>(dst), static_cast<const char*>(src), bytes, true, s);
}

void HostCopy::wait() {
  join();
  if (const int e = error_.exchange(0))
    throw Error(std::string("copy to host memory failed: ") + hipGetErrorString((hipError_t)e));
}

void copy_to_host(void* dst, const void* src, size_t bytes, hipStream_t s) {
  HostCopy c;
  c.start(dst, src, bytes, s);
  c.wait();
}

void copy_to_device(void* dst, const void* src, size_t bytes, hipStream_t s) {
  if (bytes < SMALL || g_busy || !prepare_slots()) {
    GMOD_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s));
    return;
  }
  HostCopy c;
  c.run(static_cast<char*>(dst), static_cast<const char*>(src), bytes, false, s);
  c.join();
  if (const int e = c.error_.exchange(0))
    throw Error(std::string("copy from host memory failed: ") + hipGetErrorString((hipError_t)e));
}

}  // namespace gmod

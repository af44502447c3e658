// Drives transfer.hip's staged copies on the CPU against a small model of the
// runtime: copies of the library's own stream run as late as they may (when an
// event recorded behind them or the stream is waited for), other streams run at
// once, threads and copies can be made to fail.  Prints the failed check.
#include <dlfcn.h>
#include <pthread.h>

#include <cerrno>
#include <cstdio>
#include <deque>
#include <mutex>
#include <numeric>

#include "../../pyrpa_amd/csrc/transfer.h"

namespace {
struct Op { void* dst; const void* src; size_t n; void* ev; };  // a copy, or the record of ev
std::mutex g_mu;
std::deque<Op> g_queue;
std::vector<std::pair<char*, size_t>> g_pinned;
int g_own;  // the library's stream is &g_own
int g_fail_thread = 0, g_fail_copy = -1, g_copies = 0, g_staged = 0, g_freed = 0;

void run_until(void* ev) {  // ev null: all
  while (!g_queue.empty()) {
    const Op o = g_queue.front();
    g_queue.pop_front();
    if (o.dst) memcpy(o.dst, o.src, o.n);
    else if (o.ev == ev) return;
  }
}
bool pinned(const void* p) {
  for (auto& b : g_pinned)
    if ((const char*)p >= b.first && (const char*)p < b.first + b.second) return true;
  return false;
}
bool queued(void* ev) {
  for (auto& o : g_queue)
    if (!o.dst && o.ev == ev) return true;
  return false;
}
}  // namespace

extern "C" {
int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x) {
  if (g_fail_thread) return EAGAIN;
  using F = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  static F real = (F)dlsym(RTLD_NEXT, "pthread_create");
  return real(t, a, f, x);
}
const char* hipGetErrorString(hipError_t) { return "injected"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)&g_own; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t) new int; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = new char[n];
  g_pinned.push_back({(char*)*p, n});
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  for (auto& b : g_pinned)
    if (b.first == p) { b = g_pinned.back(); g_pinned.pop_back(); break; }
  delete[] (char*)p;
  ++g_freed;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
  std::lock_guard<std::mutex> g(g_mu);
  if (g_copies++ == g_fail_copy) return hipErrorUnknown;
  if (pinned(d) || pinned(s)) ++g_staged;
  if ((void*)st == &g_own) g_queue.push_back({d, s, n, nullptr});
  else memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) {
  std::lock_guard<std::mutex> g(g_mu);
  if ((void*)st == &g_own) g_queue.push_back({nullptr, nullptr, 0, e});
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  std::lock_guard<std::mutex> g(g_mu);
  if (queued(e)) run_until(e);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t st) {
  std::lock_guard<std::mutex> g(g_mu);
  if ((void*)st == &g_own) run_until(nullptr);
  return hipSuccess;
}
}

namespace gmod {
Context& ctx() {
  static Context c;
  return c;
}
}  // namespace gmod

static int g_line = 0;
#define CHECK(c) do { if (!(c) && !g_line) { g_line = __LINE__; printf("%s:%d: %s\n", __FILE__, __LINE__, #c); } } while (0)

static std::vector<char> values(size_t n, unsigned seed) {
  std::vector<char> v(n);
  for (size_t i = 0; i < n; ++i) v[i] = (char)((i * 2654435761u + (i >> 12) + seed) >> 7);
  return v;
}
constexpr size_t MB = size_t(1) << 20;
static int other_stream;
static hipStream_t S = (hipStream_t)&other_stream;

static void round_trip(size_t n, unsigned seed) {
  const std::vector<char> a = values(n, seed);
  std::vector<char> d(n), b(n);
  gmod::copy_to_device(d.data(), a.data(), n, S);
  CHECK(d == a);
  gmod::copy_to_host(b.data(), d.data(), n, S);
  CHECK(b == a);
}

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  const size_t big = 37 * MB + 12345;
  if (what == "sizes") {
    unsigned seed = 0;
    for (size_t n : {size_t(1), 8 * MB - 1, 8 * MB, 8 * MB + 1, 16 * MB, 32 * MB + 1, big}) round_trip(n, ++seed);
    CHECK(g_staged > 0);
  } else if (what == "no_threads") {  // the pieces are copied by the caller, and the next copy is staged again
    g_fail_thread = 1;
    round_trip(big, 1);
    g_fail_thread = 0;
    const int before = g_staged;
    round_trip(big, 2);
    CHECK(g_staged == before + 2 * (int)((big + 2 * MB - 1) / (2 * MB)));
  } else if (what == "release") {
    g_fail_thread = 1;
    round_trip(big, 1);
    gmod::release_transfer_buffers();
    CHECK(g_freed == 16 && g_pinned.empty());
    g_fail_thread = 0;
    round_trip(big, 2);
  } else if (what == "failed_copy") {  // an error, nothing left in flight on the buffers, the next copy right
    const std::vector<char> a = values(big, 1);
    std::vector<char> d(big);
    for (int run = 0; run < 8; ++run) {  // with and without threads, a copy in the middle and the last one
      const bool dir = run & 1;
      g_fail_thread = run & 2;
      g_copies = 0;
      g_fail_copy = run & 4 ? 18 : 9;
      bool thrown = false;
      try {
        if (dir) gmod::copy_to_host(d.data(), a.data(), big, S);
        else gmod::copy_to_device(d.data(), a.data(), big, S);
      } catch (gmod::Error&) {
        thrown = true;
      }
      g_fail_copy = -1;
      g_fail_thread = 0;
      CHECK(thrown);
      size_t left = 0;
      for (auto& o : g_queue) left += o.dst != nullptr;
      CHECK(left == 0);
      round_trip(big, 3 + run);
    }
  } else if (what == "background") {  // another copy meanwhile, and an abandoned one
    const std::vector<char> a = values(big, 1);
    std::vector<char> b(big);
    {
      gmod::HostCopy c;
      c.start(b.data(), a.data(), big, S);
      round_trip(big, 2);
      c.wait();
      CHECK(b == a);
    }
    std::fill(b.begin(), b.end(), 0);
    {
      gmod::HostCopy c;
      c.start(b.data(), a.data(), big, S);
    }
    CHECK(b == a);
    const int before = g_staged;
    round_trip(big, 3);
    CHECK(g_staged > before);
    gmod::release_transfer_buffers();
    CHECK(g_pinned.empty());
  } else {
    CHECK(!"a known check");
  }
  return g_line ? 1 : 0;
}

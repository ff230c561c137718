// A stand-in for the HIP runtime in host tests of the transfer code: device
// memory is ordinary memory, a stream is a thread that runs its copies in
// order, some time after they were issued, and an event belongs to the device
// that was current when it was made, as in HIP.
#pragma once
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <thread>

#define __global__ static inline
struct StubDim {
  int x;
};
static StubDim threadIdx{0};

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorInvalidDevice = 101,
                  hipErrorInvalidHandle = 400 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
constexpr unsigned hipHostMallocDefault = 0, hipHostMallocPortable = 1, hipEventDisableTiming = 2;

struct StubStream {
  int dev = 0;
  std::mutex mu;
  std::condition_variable cv;
  std::deque<std::function<void()>> q;
  long put = 0, done = 0;
  bool stop = false;
  std::thread run;
  explicit StubStream(int d) : dev(d), run([this] { loop(); }) {}
  ~StubStream() {
    {
      std::lock_guard<std::mutex> lk(mu);
      stop = true;
    }
    cv.notify_all();
    run.join();
  }
  void loop() {
    unsigned seed = 12345;
    std::unique_lock<std::mutex> lk(mu);
    for (;;) {
      cv.wait(lk, [this] { return stop || !q.empty(); });
      if (q.empty()) return;
      std::function<void()> f = std::move(q.front());
      q.pop_front();
      lk.unlock();
      seed = seed * 1664525u + 1013904223u;
      std::this_thread::sleep_for(std::chrono::microseconds(seed >> 23));   // up to 0.5 ms
      f();
      lk.lock();
      done++;
      cv.notify_all();
    }
  }
  long issue(std::function<void()> f) {
    std::lock_guard<std::mutex> lk(mu);
    q.push_back(std::move(f));
    cv.notify_all();
    return ++put;
  }
  void wait(long t) {
    std::unique_lock<std::mutex> lk(mu);
    cv.wait(lk, [&] { return done >= t; });
  }
};
struct StubEvent {
  int dev;
  std::mutex mu;
  StubStream *s = nullptr;
  long t = 0;
};
using hipStream_t = StubStream *;
using hipEvent_t = StubEvent *;

constexpr int kStubDevices = 2;
inline thread_local int stub_dev = 0;
inline std::atomic<int> stub_no_pinned{0};   // set: hipHostMalloc fails

inline hipError_t hipGetDevice(int *d) {
  *d = stub_dev;
  return hipSuccess;
}
inline hipError_t hipSetDevice(int d) {
  if (d < 0 || d >= kStubDevices) return hipErrorInvalidDevice;
  stub_dev = d;
  return hipSuccess;
}
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = stub_no_pinned.load() ? nullptr : std::malloc(n);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
inline hipError_t hipHostFree(void *p) {
  std::free(p);
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
  long t;
  {
    std::lock_guard<std::mutex> lk(s->mu);
    t = s->put;
  }
  s->wait(t);
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
  st->issue([=] { std::memcpy(d, s, n); });
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  *e = new StubEvent{stub_dev};
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (e->dev != s->dev) return hipErrorInvalidHandle;
  std::lock_guard<std::mutex> a(s->mu), b(e->mu);
  e->s = s;
  e->t = s->put;
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  StubStream *s;
  long t;
  {
    std::lock_guard<std::mutex> lk(e->mu);
    s = e->s;
    t = e->t;
  }
  if (s) s->wait(t);
  return hipSuccess;
}

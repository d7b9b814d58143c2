// A HIP runtime on the CPU for tests of the library's host code: device memory
// is the process's own, a stream is a thread that runs what is queued on it in
// order, and holds still while its gate is shut.  Linked in the runtime's
// place.
#pragma once

#include <hip/hip_runtime_api.h>

#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <thread>

struct ihipStream_t {
  int device = 0;
  std::mutex mu;
  std::condition_variable cv;
  std::deque<std::function<void()>> queue;
  bool open = true, stop = false, busy = false;
  std::thread worker;

  explicit ihipStream_t(int dev) : device(dev), worker([this] { run(); }) {}
  ~ihipStream_t() {
    {
      std::lock_guard<std::mutex> lock(mu);
      open = stop = true;
    }
    cv.notify_all();
    worker.join();
  }
  void run() {
    std::unique_lock<std::mutex> lock(mu);
    for (;;) {
      cv.wait(lock, [this] { return (open && !queue.empty()) || (stop && queue.empty()); });
      if (queue.empty()) return;
      auto op = std::move(queue.front());
      queue.pop_front();
      busy = true;
      lock.unlock();
      op();
      lock.lock();
      busy = false;
      cv.notify_all();
    }
  }
  void push(std::function<void()> op) {
    {
      std::lock_guard<std::mutex> lock(mu);
      queue.push_back(std::move(op));
    }
    cv.notify_all();
  }
  void drain() {
    std::unique_lock<std::mutex> lock(mu);
    cv.wait(lock, [this] { return queue.empty() && !busy; });
  }
  void gate(bool is_open) {
    {
      std::lock_guard<std::mutex> lock(mu);
      open = is_open;
    }
    cv.notify_all();
  }
};

struct ihipEvent_t {
  int device = 0;
  unsigned flags = 0;
  std::mutex mu;
  std::condition_variable cv;
  std::atomic<int> pending{0};
};

namespace fake {

inline thread_local int device = 0;            // the thread's current device
inline std::mutex mu;
inline std::map<char*, size_t> pinned;         // hipHostMalloc
inline std::atomic<int> staged{0}, direct{0};  // copies to pinned and to pageable memory
inline std::function<void(hipEvent_t)> on_event = [](hipEvent_t) {};  // the stream reached it

inline bool is_pinned(const void* p) {
  std::lock_guard<std::mutex> lock(mu);
  auto it = pinned.upper_bound((char*)p);
  if (it == pinned.begin()) return false;
  --it;
  return (char*)p < it->first + it->second;
}

}  // namespace fake

extern "C" {

hipError_t hipGetDevice(int* d) {
  *d = fake::device;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  fake::device = d;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) {
  *d = s->device;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  s->drain();
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::malloc(n ? n : 1);
  std::lock_guard<std::mutex> lock(fake::mu);
  fake::pinned[(char*)*p] = n;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  {
    std::lock_guard<std::mutex> lock(fake::mu);
    fake::pinned.erase((char*)p);
  }
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind kind,
                          hipStream_t s) {
  const bool to_pageable = kind == hipMemcpyDeviceToHost && !fake::is_pinned(dst);
  if (kind == hipMemcpyDeviceToHost) ++(to_pageable ? fake::direct : fake::staged);
  s->push([=] { std::memcpy(dst, src, n); });
  if (to_pageable) s->drain();
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags) {
  *e = new ihipEvent_t;
  (*e)->device = fake::device;
  (*e)->flags = flags;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (e->device != s->device) return hipErrorInvalidHandle;
  ++e->pending;
  s->push([e] {
    fake::on_event(e);
    std::lock_guard<std::mutex> lock(e->mu);
    --e->pending;
    e->cv.notify_all();
  });
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  // as the runtime does: only a blocking event's waiter sleeps
  if (e->flags & hipEventBlockingSync) {
    std::unique_lock<std::mutex> lock(e->mu);
    e->cv.wait(lock, [e] { return e->pending == 0; });
  } else {
    while (e->pending != 0) std::this_thread::yield();
    std::lock_guard<std::mutex> lock(e->mu);  // the notifier is done with it
  }
  return hipSuccess;
}

}  // extern "C"

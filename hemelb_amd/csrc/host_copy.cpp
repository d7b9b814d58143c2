// Device-to-host copies through a ring of pinned chunks, emptied by several
// host threads.
//
// A plain copy into pageable memory runs at about 10 GB/s here whatever its
// size: one thread of the runtime touches (the kernel zeroes) the caller's
// pages and moves the data.  The link delivers more than 50 GB/s into pinned
// memory, so the copy goes into pinned chunks and worker threads move them
// on, each taking the page faults of its own chunks: 420 MB of distributions
// 40 -> 13.9 ms (30 GB/s), 88 MB of density and velocity 8.7 -> 3.3 ms.
#include "host_copy.h"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

namespace hlb {
namespace {

constexpr size_t kChunk = size_t(1) << 20;
constexpr int kSlots = 16;          // 16 MiB of pinned memory per process
constexpr int kMaxWorkers = 8;
// Smaller copies are left to the runtime: starting the workers costs more
// than they save.
constexpr size_t kDirect = size_t(4) << 20;

struct Staging {
  std::mutex mu;       // held by the copy that uses the buffer
  char* pinned = nullptr;
  std::mutex users_mu;
  int users = 0;
};
Staging& staging() {
  static Staging* s = new Staging;   // never destroyed: solvers may outlive statics
  return *s;
}

hipError_t copy_direct(const std::vector<HostSegment>& segments, hipStream_t stream) {
  for (const HostSegment& g : segments) {
    const hipError_t e = hipMemcpyAsync(g.dst, g.src, g.bytes, hipMemcpyDeviceToHost, stream);
    if (e != hipSuccess) return e;
  }
  return hipStreamSynchronize(stream);
}

// The chunks of one copy and the hand-over between the issuing thread and the
// workers: chunk i travels through slot i % kSlots, which is issued again
// only after done[i].  The workers sleep until the stream has reached the copy
// (the steps queued before it may take seconds); the copy itself is short, and
// they poll for its chunks.
struct Job {
  std::vector<HostSegment> chunks;
  std::vector<std::atomic<bool>> done;
  std::atomic<size_t> next{0}, issued{0};
  std::atomic<int> error{(int)hipSuccess};
  hipEvent_t arrived[kSlots] = {}, reached = nullptr;
  char* pinned = nullptr;
  int device;
  std::mutex mu;
  std::condition_variable begun;
  enum { kWaiting, kBegun, kDropped } state = kWaiting;
  std::vector<std::thread> workers;

  Job(std::vector<HostSegment> c, int dev)
      : chunks(std::move(c)), done(chunks.size()), device(dev) {
    for (auto& d : done) d.store(false, std::memory_order_relaxed);
  }
  ~Job() {
    finish();
    for (auto& e : arrived)
      if (e) (void)hipEventDestroy(e);
    if (reached) (void)hipEventDestroy(reached);
  }
  hipError_t create_events() {
    hipError_t e = hipEventCreateWithFlags(&reached, hipEventDisableTiming | hipEventBlockingSync);
    for (int k = 0; k < kSlots && e == hipSuccess; ++k)
      e = hipEventCreateWithFlags(&arrived[k], hipEventDisableTiming);
    return e;
  }
  // As many workers as the system gives, up to `wanted`.
  bool start_workers(size_t wanted) {
    try {
      workers.reserve(wanted);
      for (size_t k = 0; k < wanted; ++k) workers.emplace_back([this] { work(); });
    } catch (const std::exception&) {
    }
    return !workers.empty();
  }
  void begin() {
    {
      std::lock_guard<std::mutex> lock(mu);
      state = kBegun;
    }
    begun.notify_all();
  }
  // Waits for the workers; if the copy has not begun they have nothing to do.
  void finish() {
    {
      std::lock_guard<std::mutex> lock(mu);
      if (state == kWaiting) state = kDropped;
    }
    begun.notify_all();
    for (auto& w : workers) w.join();
    workers.clear();
  }
  void fail(hipError_t e) {
    int none = (int)hipSuccess;
    error.compare_exchange_strong(none, (int)e);
  }
  bool failed() const { return error.load() != (int)hipSuccess; }

  void work() {
    (void)hipSetDevice(device);
    {
      std::unique_lock<std::mutex> lock(mu);
      begun.wait(lock, [this] { return state != kWaiting; });
      if (state == kDropped) return;
    }
    for (;;) {
      const size_t i = next.fetch_add(1);
      if (i >= chunks.size()) return;
      while (issued.load(std::memory_order_acquire) <= i) {
        if (failed()) return;
        std::this_thread::yield();
      }
      const hipError_t e = hipEventSynchronize(arrived[i % kSlots]);
      if (e != hipSuccess) return fail(e);
      std::memcpy(chunks[i].dst, pinned + (i % kSlots) * kChunk, chunks[i].bytes);
      done[i].store(true, std::memory_order_release);
    }
  }
  void issue(hipStream_t stream) {
    for (size_t i = 0; i < chunks.size(); ++i) {
      const int slot = (int)(i % kSlots);
      if (i >= (size_t)kSlots)
        while (!done[i - kSlots].load(std::memory_order_acquire)) {
          if (failed()) return;
          std::this_thread::yield();
        }
      hipError_t e = hipMemcpyAsync(pinned + slot * kChunk, chunks[i].src, chunks[i].bytes,
                                    hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess) e = hipEventRecord(arrived[slot], stream);
      if (e != hipSuccess) return fail(e);
      issued.store(i + 1, std::memory_order_release);
      if (i == 0) begin();
    }
  }
};

// Makes `device` the thread's current one for a scope.
struct CurrentDevice {
  int before = -1;
  hipError_t set(int device) {
    int now = 0;
    hipError_t e = hipGetDevice(&now);
    if (e != hipSuccess || now == device) return e;
    e = hipSetDevice(device);
    if (e == hipSuccess) before = now;
    return e;
  }
  ~CurrentDevice() {
    if (before >= 0) (void)hipSetDevice(before);
  }
};

}  // namespace

hipError_t copy_to_host(const std::vector<HostSegment>& segments, hipStream_t stream) {
  size_t total = 0;
  for (const HostSegment& g : segments) total += g.bytes;
  if (total < kDirect) return copy_direct(segments, stream);
  std::vector<HostSegment> chunks;
  for (const HostSegment& g : segments)
    for (size_t a = 0; a < g.bytes; a += kChunk)
      chunks.push_back({(char*)g.dst + a, (const char*)g.src + a, std::min(kChunk, g.bytes - a)});
  // an event is recorded on streams of the device it was created on alone, and
  // the caller's current device need not be the stream's
  int device = 0;
  hipError_t e = hipStreamGetDevice(stream, &device);
  CurrentDevice current;
  if (e == hipSuccess) e = current.set(device);
  if (e != hipSuccess) return e;
  Job job(std::move(chunks), device);
  e = job.create_events();
  if (e == hipSuccess) e = hipEventRecord(job.reached, stream);
  if (e != hipSuccess) return e;
  const bool workers = job.start_workers(std::min<size_t>(kMaxWorkers, total / (2 * kChunk)));
  // The staging memory is taken once there is something to copy, so that
  // another thread's copy can have it meanwhile.
  e = hipEventSynchronize(job.reached);
  if (e != hipSuccess) return e;
  Staging& st = staging();
  std::unique_lock<std::mutex> lock(st.mu, std::try_to_lock);
  // another thread's copy has the staging buffer: take the runtime's path
  if (!workers || !lock.owns_lock()) return copy_direct(segments, stream);
  // (portable: every device's copies go through it)
  if (!st.pinned && hipHostMalloc((void**)&st.pinned, kSlots * kChunk, hipHostMallocPortable) !=
                        hipSuccess) {
    st.pinned = nullptr;
    (void)hipGetLastError();
    return copy_direct(segments, stream);
  }
  job.pinned = st.pinned;
  job.issue(stream);
  job.finish();
  // no copy may still write the staging buffer or read the source
  e = hipStreamSynchronize(stream);
  return job.failed() ? (hipError_t)job.error.load() : e;
}

void staging_acquire() {
  Staging& st = staging();
  std::lock_guard<std::mutex> lock(st.users_mu);
  ++st.users;
}

void staging_release() {
  Staging& st = staging();
  std::lock_guard<std::mutex> lock(st.users_mu);
  if (--st.users > 0) return;
  std::lock_guard<std::mutex> copy(st.mu);
  if (st.pinned) (void)hipHostFree(st.pinned);
  st.pinned = nullptr;
}

}  // namespace hlb

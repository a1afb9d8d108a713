// readback.cpp -- device arrays to the caller's (pageable) memory.
//
// hipMemcpy into pageable memory moves about 18 GB/s here; DMA into pinned
// memory 57.  So a large array goes through a ring of pinned slots: the DMA
// fills one slot while worker threads copy the others out, each its own
// slice of every slot: a BFS of R-MAT 25 with its 134 MB of levels takes 3.9 ms
// where it took 12.6 (0.85 of them the traversal, 4 the host's count of the
// reached vertices, which the GPU makes now).
#include <algorithm>
#include <atomic>
#include <mutex>
#include <thread>

#include "internal.hpp"

namespace thv {

namespace {

// Whether the runtime knows p (pinned or device memory): DMA reaches it.
bool known_pointer(const void *p) {
  hipPointerAttribute_t at;
  memset(&at, 0, sizeof at);
  const hipError_t e = hipPointerGetAttributes(&at, p);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return at.type != hipMemoryTypeUnregistered;
}

// A ring of pinned slots and an event per slot.
struct Ring {
  HostPinned mem;
  hipEvent_t ev[Readback::SLOTS] = {};
  int device = -1;
  ~Ring() {
    for (auto &e : ev)
      if (e) (void)hipEventDestroy(e);
  }
};

// Rings between copies (a pinned allocation of 12 MB is 2 ms, as long as
// copying 100 MB): at most KEEP of them, none once no graph is open.
struct RingPool {
  static constexpr size_t KEEP = 2;
  std::mutex mu;
  std::vector<std::unique_ptr<Ring>> idle;
  int users = 0;
  static RingPool &get() {
    static RingPool *p = new RingPool();  // never destroyed: HIP may be gone by then
    return *p;
  }
  std::unique_ptr<Ring> take(size_t bytes) {
    int dev = 0;
    HIPC(hipGetDevice(&dev));
    {
      std::lock_guard<std::mutex> lk(mu);
      for (size_t i = 0; i < idle.size(); i++) {
        if (idle[i]->device != dev || idle[i]->mem.bytes < bytes) continue;
        std::unique_ptr<Ring> r = std::move(idle[i]);
        idle.erase(idle.begin() + i);
        return r;
      }
    }
    std::unique_ptr<Ring> r(new Ring());
    r->device = dev;
    r->mem.alloc(bytes);
    for (auto &e : r->ev) HIPC(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    return r;
  }
  void put(std::unique_ptr<Ring> r) {
    std::unique_ptr<Ring> out;  // freed without the lock
    std::lock_guard<std::mutex> lk(mu);
    idle.push_back(std::move(r));
    if (idle.size() <= KEEP) return;
    size_t least = 0;
    for (size_t i = 1; i < idle.size(); i++)
      if (idle[i]->mem.bytes < idle[least]->mem.bytes) least = i;
    out = std::move(idle[least]);
    idle.erase(idle.begin() + least);
  }
};

}  // namespace

Readback::Readback() {
  std::lock_guard<std::mutex> lk(RingPool::get().mu);
  RingPool::get().users++;
}

Readback::~Readback() {
  std::vector<std::unique_ptr<Ring>> out;
  RingPool &p = RingPool::get();
  std::lock_guard<std::mutex> lk(p.mu);
  if (--p.users == 0) out.swap(p.idle);
}

void Readback::copy(void *out, const void *dev, size_t bytes, hipStream_t s) {
  if (!bytes) return;
  // (the core count costs a system call or two: asked for large copies only)
  const size_t T = bytes < MIN_BYTES
                       ? 0
                       : std::min<size_t>(WORKERS, std::thread::hardware_concurrency());
  if (T < 2 || known_pointer(out)) {
    HIPC(hipMemcpy(out, dev, bytes, hipMemcpyDeviceToHost));
    return;
  }
  const size_t slot = bytes >= LARGE ? SLOT_LARGE : bytes >= MEDIUM ? SLOT_MEDIUM : SLOT;
  std::unique_ptr<Ring> held = RingPool::get().take(SLOTS * slot);
  Ring &r = *held;
  const size_t chunks = div_up(bytes, slot);
  std::atomic<size_t> ready{0};             // chunks [0, ready) are in their slots
  std::atomic<bool> stop{false};
  std::unique_ptr<std::atomic<size_t>[]> left(new std::atomic<size_t>[T]);  // chunks copied out
  for (size_t t = 0; t < T; t++) left[t] = 0;
  auto work = [&](size_t t) {
    for (size_t k = 0; k < chunks; k++) {
      while (ready.load(std::memory_order_acquire) <= k) {
        if (stop.load(std::memory_order_relaxed)) return;
        std::this_thread::yield();
      }
      const size_t at = k * slot, len = std::min(slot, bytes - at);
      const size_t a = len * t / T / 64 * 64, b = t + 1 == T ? len : len * (t + 1) / T / 64 * 64;
      memcpy(static_cast<char *>(out) + at + a,
             static_cast<const char *>(r.mem.p) + k % SLOTS * slot + a, b - a);
      left[t].store(k + 1, std::memory_order_release);
    }
  };
  struct Join {  // ends and joins the workers, and the copies, on every way out
    std::vector<std::thread> th;
    std::atomic<bool> &stop;
    hipStream_t s;
    bool done;
    ~Join() {
      stop = true;
      for (auto &t : th) t.join();
      if (!done) (void)hipStreamSynchronize(s);
    }
  } join{{}, stop, s, false};
  size_t issued = 0;
  auto issue = [&] {
    const size_t at = issued * slot, len = std::min(slot, bytes - at);
    HIPC(hipMemcpyAsync(static_cast<char *>(r.mem.p) + issued % SLOTS * slot,
                        static_cast<const char *>(dev) + at, len, hipMemcpyDeviceToHost, s));
    HIPC(hipEventRecord(r.ev[issued % SLOTS], s));
    issued++;
  };
  while (issued < std::min<size_t>(chunks, SLOTS)) issue();
  try {
    for (size_t t = 0; t < T; t++) join.th.emplace_back(work, t);
  } catch (const std::exception &) {  // no threads to be had: the plain copy
    HIPC(hipStreamSynchronize(s));
    HIPC(hipMemcpyAsync(out, dev, bytes, hipMemcpyDeviceToHost, s));
    stop = true;
    for (auto &t : join.th) t.join();
    join.th.clear();
    HIPC(hipStreamSynchronize(s));
    RingPool::get().put(std::move(held));
    return;
  }
  for (size_t k = 0; k < chunks; k++) {
    HIPC(hipEventSynchronize(r.ev[k % SLOTS]));
    ready.store(k + 1, std::memory_order_release);
    // slot k is refilled once every worker has copied its slice of it; the
    // other slots' DMA goes on meanwhile
    if (k >= 1 && issued < chunks) {
      for (size_t t = 0; t < T; t++)
        while (left[t].load(std::memory_order_acquire) < k) std::this_thread::yield();
      issue();
    }
  }
  for (size_t t = 0; t < T; t++)
    while (left[t].load(std::memory_order_acquire) < chunks) std::this_thread::yield();
  join.done = true;
  RingPool::get().put(std::move(held));
}

}  // namespace thv

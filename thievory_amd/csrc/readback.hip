// readback.hip -- device arrays to the caller's (pageable) memory.
//
// hipMemcpy into pageable memory moves about 18 GB/s here; writes into pinned
// memory 56.  So a large array goes through a ring of pinned slots: a kernel
// fills one slot while worker threads copy the others out, each its own
// slice of every slot.  The threads watch the flags, so a copy takes more of the
// host than hipMemcpy did and less time: CC on R-MAT 23 with 1 / 2 / 4 / 8 callers
// at once, each with a graph, 1.04 / 0.85 / 0.79 / 0.91 ms a call (3.57 / 2.08 /
// 2.08 / 2.09) for 6.2 / 6.7 / 10.2 / 12.4 ms of CPU time (3.6 - 3.9); on two
// CPUs 1.3 / 1.4 / 1.5 / 1.7 ms.
#include <algorithm>
#include <atomic>
#include <mutex>
#include <thread>

#include "internal.hpp"
#include "scan.hpp"

namespace thv {

namespace {

constexpr uint64_t WATCH = 1u << 20;  // looks at a flag before the stream is asked

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

// What the GPU tells the host about a slot: the number of the copy it holds,
// and the ring's count after it.  In fine-grained memory, a line each.
struct alignas(128) SlotFlag {
  unsigned long long seq;
  unsigned long long count;
};

// Fill a slot from src[0, n) words (16-byte aligned) and add to *count how many differ from
// `none`.  Bound by the link: 4 MB in 76 us, and 3 more to the next slot's
// kernel, where a copy of the runtime with an event to wait for took 86; and
// the count needs no pass of its own.  The flag is raised by a kernel of its
// own: a system fence in every wave here, for the last block to raise it,
// takes 10 us a slot with 64 blocks and 110 with 512.
constexpr int CBS = 1024, COPY_BLOCKS = 128;
__global__ void __launch_bounds__(CBS) k_copy_out(const uint32_t *src, uint32_t *dst, uint32_t n,
                                                  uint32_t none, unsigned long long *count) {
  __shared__ unsigned long long sh[CBS / 64];
  const uint32_t t = blockIdx.x * CBS + threadIdx.x, T = gridDim.x * CBS;
  const uint4 *s4 = reinterpret_cast<const uint4 *>(src);
  uint4 *d4 = reinterpret_cast<uint4 *>(dst);
  unsigned long long c = 0;
#pragma unroll 4
  for (uint32_t i = t; i < n / 4; i += T) {
    const uint4 x = s4[i];
    d4[i] = x;
    c += (x.x != none) + (x.y != none) + (x.z != none) + (x.w != none);
  }
  for (uint32_t i = n / 4 * 4 + t; i < n; i += T) {
    const uint32_t x = src[i];
    dst[i] = x;
    c += x != none;
  }
  c = block_sum<CBS>(c, sh);
  if (threadIdx.x == 0 && c) atomicAdd(count, c);
}

// After a slot's kernel in its stream: the slot is full.
__global__ void k_raise(const unsigned long long *count, SlotFlag *flag, unsigned long long seq) {
  flag->count = *count;
  __threadfence_system();
  __hip_atomic_store(&flag->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A ring of pinned slots, their flags, and the kernels' counter.
struct Ring {
  char *mem = nullptr;      // SLOTS slots, then SLOTS flags
  char *mem_dev = nullptr;
  size_t bytes = 0;         // of the slots
  DevMem ctr;               // u64
  unsigned long long seq = 0, counted = 0;  // copies into slots, their count
  int device = -1;
  SlotFlag *flags(char *base) const { return reinterpret_cast<SlotFlag *>(base + bytes); }
  ~Ring() {
    if (mem) (void)hipHostFree(mem);
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
        if (idle[i]->device != dev || idle[i]->bytes < bytes) continue;
        std::unique_ptr<Ring> r = std::move(idle[i]);
        idle.erase(idle.begin() + i);
        return r;
      }
    }
    std::unique_ptr<Ring> r(new Ring());
    r->device = dev;
    r->bytes = bytes;
    const size_t all = bytes + Readback::SLOTS * sizeof(SlotFlag);
    HIPC(hipHostMalloc((void **)&r->mem, all, hipHostMallocMapped | hipHostMallocCoherent));
    HIPC(hipHostGetDevicePointer((void **)&r->mem_dev, r->mem, 0));
    memset(r->flags(r->mem), 0, Readback::SLOTS * sizeof(SlotFlag));
    r->ctr.alloc(8);
    HIPC(hipMemset(r->ctr.p, 0, 8));
    HIPC(hipStreamSynchronize(nullptr));
    return r;
  }
  void put(std::unique_ptr<Ring> r) {
    std::unique_ptr<Ring> out;  // freed without the lock
    std::lock_guard<std::mutex> lk(mu);
    idle.push_back(std::move(r));
    if (idle.size() <= KEEP) return;
    size_t least = 0;
    for (size_t i = 1; i < idle.size(); i++)
      if (idle[i]->bytes < idle[least]->bytes) least = i;
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

bool Readback::copy(void *out, const void *dev, size_t bytes, hipStream_t s, uint32_t none,
                    uint64_t *count) {
  if (!bytes) return false;
  // (the core count costs a system call or two: asked for large copies only)
  const size_t T = bytes < MIN_BYTES
                       ? 0
                       : std::min<size_t>(WORKERS, std::thread::hardware_concurrency());
  if (T < 2 || bytes % 4 || reinterpret_cast<uintptr_t>(dev) % 16 || known_pointer(out)) {
    HIPC(hipMemcpy(out, dev, bytes, hipMemcpyDeviceToHost));
    return false;
  }
  const size_t slot = bytes >= LARGE ? SLOT_LARGE : bytes >= MEDIUM ? SLOT_MEDIUM : SLOT;
  std::unique_ptr<Ring> held;
  try {
    held = RingPool::get().take(SLOTS * slot);
  } catch (const std::exception &) {  // no pinned memory to be had: the plain copy
    (void)hipGetLastError();
    HIPC(hipMemcpy(out, dev, bytes, hipMemcpyDeviceToHost));
    return false;
  }
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
             r.mem + k % SLOTS * slot + a, b - a);
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
  const unsigned long long seq0 = r.seq + 1;
  r.seq += chunks;
  auto issue = [&] {
    const size_t at = issued * slot, len = std::min(slot, bytes - at);
    hipLaunchKernelGGL(k_copy_out, dim3(COPY_BLOCKS), dim3(CBS), 0, s,
                       reinterpret_cast<const uint32_t *>(static_cast<const char *>(dev) + at),
                       reinterpret_cast<uint32_t *>(r.mem_dev + issued % SLOTS * slot),
                       (uint32_t)(len / 4), none, r.ctr.as<unsigned long long>());
    hipLaunchKernelGGL(k_raise, dim3(1), dim3(1), 0, s, r.ctr.as<unsigned long long>(),
                       r.flags(r.mem_dev) + issued % SLOTS, seq0 + issued);
    HIPC(hipGetLastError());
    issued++;
  };
  // the slot's flag, watched: a wait on the stream costs 5 us more.  When it
  // does not come, the stream says why.
  auto arrived = [&](size_t k) {
    const SlotFlag *f = r.flags(r.mem) + k % SLOTS;
    for (uint64_t i = 0; __atomic_load_n(&f->seq, __ATOMIC_ACQUIRE) != seq0 + k; i++) {
      if (i < WATCH) {
        __builtin_ia32_pause();
        continue;
      }
      HIPC(hipStreamSynchronize(s));
      if (__atomic_load_n(&f->seq, __ATOMIC_ACQUIRE) != seq0 + k)
        fail(THV_EHIP, "readback did not arrive");
    }
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
    join.done = true;
    return false;  // (the ring is freed: its count is not known)
  }
  for (size_t k = 0; k < chunks; k++) {
    arrived(k);
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
  const unsigned long long all = r.flags(r.mem)[(chunks - 1) % SLOTS].count;
  if (count) *count = all - r.counted;
  r.counted = all;
  RingPool::get().put(std::move(held));
  return count != nullptr;
}

}  // namespace thv

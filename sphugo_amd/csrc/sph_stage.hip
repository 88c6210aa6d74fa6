// Readback staging: device arrays to the caller's (pageable) host arrays
// through pinned blocks, and the counters of a handle in one write.
//
// The runtime's own copy into pageable memory stages or pins per call: 32 us
// for 17 KB, 94 us for 160 KB, 366 us for 800 KB of freshly allocated memory, and
// for 32 MB 3.5 ms, most of it one thread touching new pages.  Here a kernel
// writes the bytes to a pinned block (no copy engine to start), and the host
// copies them on; large arrays go through the slots of a ring, the host copying
// one slot (with up to four threads: new pages cost more than the bytes) while
// the next ones fill: 18, 23, 51 us and 2.1 ms for the same reads.
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "sph_sim.hpp"

namespace sph {

// Larger copies take the slots.  64 KiB, 256 KiB and 1 MiB time alike (a copy of one
// slot is one kernel and one host copy either way).
constexpr size_t kSmallCopy = 256 << 10;
constexpr size_t kSlot = 1 << 20;  // one slot of a large copy
// Slots of a ring.  4, 8 and 16 time alike up to 8 MB; 33.6 MB into fresh memory takes
// 2.45, 2.4 and 1.95 ms, for 4, 8 and 16 MiB of pinned memory per call.
constexpr int kSlots = 8;
static_assert(sizeof(Stage::ev) / sizeof(hipEvent_t) == kSlots, "an event per slot");

namespace {

// Pinned memory of one size, shared by the handles of a process: a call takes what
// it needs and returns it when it ends, so a program with many handles holds as
// many pieces as its calls at one time use and at most kKeep free ones of a size,
// and none once no handle is left.  A block serves the small copies, the flags and
// copies of one slot; a ring, which takes 400 to 650 us to allocate against a
// block's 50 (the first read of 800 KB in a process 534 -> 347 us), those of more,
// which run 2 % faster in one piece than in separate blocks (45 MB of neighbour rows
// 2,470 against 2,530 us).
constexpr size_t kKeep = 16;
struct PinnedPool {
  size_t bytes;
  size_t keep;  // at most kKeep
  void* idle[kKeep];
  size_t n;
};
std::mutex g_mu;
PinnedPool g_blocks = {kSlot, 16, {}, 0}, g_rings = {kSlot * kSlots, 4, {}, 0};
int g_handles = 0;

// null where the runtime has no pinned memory to give: the reads then go through
// its own copy
char* take(PinnedPool& p) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    if (p.n) return (char*)p.idle[--p.n];
  }
  void* b = nullptr;
  if (hipHostMalloc(&b, p.bytes, hipHostMallocPortable | hipHostMallocMapped) == hipSuccess)
    return (char*)b;
  (void)hipGetLastError();  // or the next launch would report it
  return nullptr;
}

void give(PinnedPool& p, char* b) {
  if (!b) return;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    if (p.n < p.keep) {
      p.idle[p.n++] = b;
      return;
    }
  }
  (void)hipHostFree(b);  // teardown
}

// A block or a ring for the length of a call (or null).
struct Pinned {
  PinnedPool& pool;
  char* const p;
  explicit Pinned(PinnedPool& from) : pool(from), p(take(from)) {}
  Pinned(const Pinned&) = delete;
  Pinned& operator=(const Pinned&) = delete;
  ~Pinned() { give(pool, p); }
};

}  // namespace

void stage_open(Stage&) {
  std::lock_guard<std::mutex> lk(g_mu);
  ++g_handles;
}

void stage_close(Stage& s) {
  for (auto& e : s.ev)
    if (e) {
      (void)hipEventDestroy(e);
      e = nullptr;
    }
  give(g_blocks, s.flags);
  s.flags = nullptr;
  void* drop[2 * kKeep];
  size_t n = 0;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    if (--g_handles == 0)
      for (PinnedPool* p : {&g_blocks, &g_rings})
        while (p->n) drop[n++] = p->idle[--p->n];
  }
  while (n) (void)hipHostFree(drop[--n]);
}

static int copy_pageable(sph_sim* s, void* dst, const void* dev, size_t bytes) {
  HIPCHK(hipMemcpyAsync(dst, dev, bytes, hipMemcpyDeviceToHost, s->st));
  HIPCHK(hipStreamSynchronize(s->st));
  return 0;
}

// n16 16-byte words and the tail4 4-byte words after them
__global__ __launch_bounds__(256) void k_copy_out(const char* __restrict__ src,
                                                  char* __restrict__ dst, int64_t n16, int tail4) {
  const int64_t stride = (int64_t)gridDim.x * 256, i0 = (int64_t)blockIdx.x * 256 + threadIdx.x;
  for (int64_t i = i0; i < n16; i += stride) ((u32x4*)dst)[i] = ((const u32x4*)src)[i];
  if (i0 < tail4) ((uint32_t*)(dst + 16 * n16))[i0] = ((const uint32_t*)(src + 16 * n16))[i0];
}

static int enqueue_copy_out(void* pinned, const void* dev, size_t bytes, hipStream_t st) {
  const int64_t n16 = (int64_t)(bytes / 16);
  const int64_t blocks = n16 / 256 + 1;
  hipLaunchKernelGGL(k_copy_out, dim3((unsigned)(blocks < 512 ? blocks : 512)), dim3(256), 0, st,
                     (const char*)dev, (char*)pinned, n16, (int)(bytes % 16 / 4));
  return (int)hipGetLastError();
}

// The host side of a large copy: up to three workers and the caller copy their
// share of every slot the caller announces.  The stream may have much to do before
// the first one (the passes of a server's tick): the workers ask for it, in turns,
// no longer than kAsk and sleep from then on (asleep at once, 32 simulations' fields
// were 2 % slower: a woken thread comes 10 us after its slot).  Every wait ends: the
// caller announces each slot or sets `stop`, and the workers copy without blocking.
constexpr std::chrono::microseconds kAsk{200};
static int copy_slots(sph_sim* s, char* dst, const char* dev, size_t bytes) {
  Stage& sg = s->stage;
  const size_t nslot = (bytes + kSlot - 1) / kSlot;
  const size_t nring = nslot > 1 ? kSlots : 1;
  Pinned ring(nslot > 1 ? g_rings : g_blocks);
  if (!ring.p) return copy_pageable(s, dst, dev, bytes);
  for (size_t i = 0; i < nring; ++i)
    if (!sg.ev[i]) HIPCHK(hipEventCreateWithFlags(&sg.ev[i], hipEventDisableTiming));
  auto length = [&](size_t c) { return c + 1 < nslot ? kSlot : bytes - c * kSlot; };
  auto send = [&](size_t c) -> int {
    if (enqueue_copy_out(ring.p + c % nring * kSlot, dev + c * kSlot, length(c), s->st))
      return fail(SPH_EDEVICE, "readback launch failed");
    HIPCHK(hipEventRecord(sg.ev[c % nring], s->st));
    return 0;
  };
  std::atomic<size_t> ready{0};    // slots filled so far
  std::atomic<bool> stop{false};
  std::atomic<size_t> copied{0};   // shares copied by the workers
  // one, two, four and eight threads: 1 MB 68, 56, 59 and 128 us, 2.1 MB 106, 82, 83 and
  // 140, 4.2 MB 181, 129, 133 and 168, 8.4 MB 343, 225, 226 and 253, 33.6 MB 1,368, 966,
  // 795 and 815 (starting a thread is 10 to 20 us of the caller's time)
  int want = bytes >= (4u << 20) ? 4 : (bytes >= (2u << 20) ? 2 : 1), nthreads = 1;
  auto share = [&](size_t c, int who, int n) {
    const size_t len = length(c), part = (len / n + 63) & ~(size_t)63;
    const size_t a = part * who < len ? part * who : len, b = who + 1 == n || a + part > len ? len : a + part;
    memcpy(dst + c * kSlot + a, ring.p + c % nring * kSlot + a, b - a);
  };
  std::vector<std::thread> pool;
  std::atomic<int> members{0};  // set before the first slot is announced
  std::mutex mu;
  std::condition_variable first;  // the first slot, or `stop`
  auto begun = [&] { return ready.load() > 0 || stop.load(); };
  auto wake = [&] {
    { std::lock_guard<std::mutex> lk(mu); }  // none between its test and its sleep
    first.notify_all();
  };
  auto work = [&](int who) {
    const auto until = std::chrono::steady_clock::now() + kAsk;
    while (!begun() && std::chrono::steady_clock::now() < until) std::this_thread::yield();
    if (!begun()) {
      std::unique_lock<std::mutex> lk(mu);
      first.wait(lk, begun);
    }
    for (size_t c = 0; c < nslot; ++c) {
      while (ready.load(std::memory_order_acquire) <= c) {
        if (stop.load(std::memory_order_relaxed)) return;
        std::this_thread::yield();
      }
      share(c, who, members.load(std::memory_order_relaxed));
      copied.fetch_add(1, std::memory_order_release);
    }
  };
  int rc = 0;
  for (size_t c = 0; c < nslot && c < nring && !rc; ++c) rc = send(c);
  if (!rc) {
    try {
      pool.reserve(want - 1);
      for (; nthreads < want; ++nthreads) pool.emplace_back(work, nthreads);
    } catch (...) {  // no thread to be had: the caller copies more itself
    }
    members.store(nthreads, std::memory_order_relaxed);
  }
  for (size_t c = 0; c < nslot && !rc; ++c) {
    const hipError_t e = hipEventSynchronize(sg.ev[c % nring]);
    if (e != hipSuccess) {
      rc = fail(SPH_EDEVICE, "readback: %s", hipGetErrorString(e));
      break;
    }
    ready.store(c + 1);
    if (c == 0 && nthreads > 1) wake();
    share(c, 0, nthreads);
    if (c + nring < nslot) {
      // the slot is filled again once every worker has taken its share
      while (copied.load(std::memory_order_acquire) < (c + 1) * (size_t)(nthreads - 1))
        std::this_thread::yield();
      rc = send(c + nring);
    }
  }
  if (rc) {
    stop.store(true);
    wake();
  }
  for (auto& t : pool) t.join();
  // what was sent before a failure must not outlive the ring's contents
  if (rc) (void)hipStreamSynchronize(s->st);
  return rc;
}

// The n values of `src` by particle ID: put in order in LDS and written out in
// one piece.  A field of a small simulation leaves in one launch that way, where
// a scatter and a copy were a launch more: 17.4 -> 14.2 us per call at 2,200
// particles, 19.4 -> 17.3 at 8,192 (LDS holds no more).
__global__ __launch_bounds__(1024) void k_read_ordered(const double* __restrict__ src,
                                                       const uint32_t* __restrict__ id, int n,
                                                       double* __restrict__ dst) {
  __shared__ double2 v[kOrderedMax / 2];
#pragma unroll 4
  for (int t = threadIdx.x; t < n; t += 1024) ((double*)v)[id[t]] = src[t];
  __syncthreads();
  for (int i = threadIdx.x; i < n / 2; i += 1024) ((double2*)dst)[i] = v[i];
  if ((n & 1) && threadIdx.x == 0) dst[n - 1] = ((double*)v)[n - 1];
}

int read_ordered(sph_sim* s, double* dst, const double* dev, const uint32_t* id, int n) {
  Pinned b(g_blocks);
  hipLaunchKernelGGL(k_read_ordered, dim3(1), dim3(1024), 0, s->st, dev, id, n,
                     b.p ? (double*)b.p : s->d_scratch);
  if (hipGetLastError() != hipSuccess) return fail(SPH_EDEVICE, "readback launch failed");
  if (!b.p) return copy_pageable(s, dst, s->d_scratch, n * sizeof(double));
  HIPCHK(hipStreamSynchronize(s->st));
  memcpy(dst, b.p, n * sizeof(double));
  return 0;
}

int copy_out(sph_sim* s, void* dst, const void* dev, size_t bytes) {
  if (bytes == 0) return 0;
  if (bytes > kSmallCopy) return copy_slots(s, (char*)dst, (const char*)dev, bytes);
  Pinned b(g_blocks);
  if (!b.p) return copy_pageable(s, dst, dev, bytes);
  if (enqueue_copy_out(b.p, dev, bytes, s->st))
    return fail(SPH_EDEVICE, "readback launch failed");
  HIPCHK(hipStreamSynchronize(s->st));
  memcpy(dst, b.p, bytes);
  return 0;
}

// The error flags (nerr of them) and the kNN counters' sums.
__global__ __launch_bounds__(256) void k_flags(const int* __restrict__ err, int nerr,
                                               const KnnStats* __restrict__ stats,
                                               unsigned long long* __restrict__ sums,
                                               int* __restrict__ err_out) {
  constexpr int kN = sizeof(KnnStats) / sizeof(unsigned long long);
  static_assert(kStatSlots == 64, "a lane per copy");
  const int lane = threadIdx.x & 63;
  if (threadIdx.x < 64) {
    const unsigned long long* p = (const unsigned long long*)(stats + lane);
    for (int i = 0; i < kN; ++i) {
      unsigned long long v = p[i];
      for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
      if (lane == 0) sums[i] = v;
    }
  }
  for (int i = threadIdx.x; i < nerr; i += 256) err_out[i] = err[i];
}

int enqueue_flags(sph_sim* s, int nerr) {
  Stage& sg = s->stage;
  if (sizeof(KnnStats) + (size_t)nerr * sizeof(int) > kSlot) return 0;  // take_flags copies them
  if (!sg.flags && !(sg.flags = take(g_blocks))) return 0;
  hipLaunchKernelGGL(k_flags, dim3(1), dim3(256), 0, s->st, s->pb.err, nerr, s->pb.stats,
                     (unsigned long long*)sg.flags, (int*)(sg.flags + sizeof(KnnStats)));
  if (hipGetLastError() != hipSuccess) return fail(SPH_EDEVICE, "flags launch failed");
  return 0;
}

int take_flags(sph_sim* s, KnnStats* stats, int* err, int nerr) {
  Stage& sg = s->stage;
  if (!sg.flags) {
    KnnStats slot[kStatSlots];
    int rc = copy_pageable(s, slot, s->pb.stats, sizeof slot);
    if (!rc) rc = copy_pageable(s, err, s->pb.err, (size_t)nerr * sizeof(int));
    if (rc) return rc;
    *stats = {};
    for (const KnnStats& v : slot)
      for (size_t i = 0; i < sizeof v / sizeof(unsigned long long); ++i)
        ((unsigned long long*)stats)[i] += ((const unsigned long long*)&v)[i];
    return 0;
  }
  memcpy(stats, sg.flags, sizeof *stats);
  memcpy(err, sg.flags + sizeof *stats, (size_t)nerr * sizeof(int));
  give(g_blocks, sg.flags);
  sg.flags = nullptr;
  return 0;
}

}  // namespace sph

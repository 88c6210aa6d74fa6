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
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "sph_sim.hpp"

namespace sph {

constexpr size_t kSmallBlock = 512 << 10;  // one small copy, or the flags of a full server
constexpr size_t kSmallCopy = 256 << 10;   // larger copies take the slots
constexpr size_t kSlot = 1 << 20;          // one slot of a large copy
constexpr int kSlots = 8;

namespace {

// Pinned blocks of one size, shared by the handles of a process: a handle
// takes one when it first needs it and returns it when it is destroyed.  At
// most `keep` free blocks are held, and none once no handle is left.
struct PinnedPool {
  size_t bytes;
  size_t keep;
  std::vector<void*> idle;
};
std::mutex g_mu;
PinnedPool g_small = {kSmallBlock, 16, {}}, g_ring = {kSlot * kSlots, 4, {}};
int g_handles = 0;

void* take(PinnedPool& p) {
  {
    std::lock_guard<std::mutex> lk(g_mu);
    if (!p.idle.empty()) {
      void* b = p.idle.back();
      p.idle.pop_back();
      return b;
    }
  }
  void* b = nullptr;
  if (hipHostMalloc(&b, p.bytes, hipHostMallocPortable | hipHostMallocMapped) != hipSuccess)
    return nullptr;
  return b;
}

void give(PinnedPool& p, void* b) {
  if (!b) return;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    if (p.idle.size() < p.keep) {
      p.idle.push_back(b);
      return;
    }
  }
  (void)hipHostFree(b);  // teardown
}

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
  give(g_small, s.small);
  give(g_ring, s.ring);
  s.small = s.ring = nullptr;
  std::vector<void*> drop;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    if (--g_handles == 0)
      for (PinnedPool* p : {&g_small, &g_ring}) {
        drop.insert(drop.end(), p->idle.begin(), p->idle.end());
        p->idle.clear();
      }
  }
  for (void* b : drop) (void)hipHostFree(b);
}

static int small_block(Stage& s) {
  if (!s.small && !(s.small = (char*)take(g_small)))
    return fail(SPH_ENOMEM, "pinned host allocation of %zu bytes failed", kSmallBlock);
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

// The host side of a large copy: `workers` threads and the caller copy their
// share of every slot the caller announces.  Every wait ends: the caller
// announces each slot or sets `stop`, and the workers copy without blocking.
static int copy_slots(sph_sim* s, char* dst, const char* dev, size_t bytes) {
  Stage& sg = s->stage;
  if (!sg.ring && !(sg.ring = (char*)take(g_ring)))
    return fail(SPH_ENOMEM, "pinned host allocation of %zu bytes failed", kSlot * kSlots);
  for (auto& e : sg.ev)
    if (!e) HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  const size_t nslot = (bytes + kSlot - 1) / kSlot;
  auto length = [&](size_t c) { return c + 1 < nslot ? kSlot : bytes - c * kSlot; };
  auto send = [&](size_t c) -> int {
    if (enqueue_copy_out(sg.ring + c % kSlots * kSlot, dev + c * kSlot, length(c), s->st))
      return fail(SPH_EDEVICE, "readback launch failed");
    HIPCHK(hipEventRecord(sg.ev[c % kSlots], s->st));
    return 0;
  };
  std::atomic<size_t> ready{0};    // slots filled so far
  std::atomic<bool> stop{false};
  std::atomic<size_t> copied{0};   // shares copied by the workers
  int want = bytes >= (4u << 20) ? 4 : (bytes >= (2u << 20) ? 2 : 1), nthreads = 1;
  auto share = [&](size_t c, int who, int n) {
    const size_t len = length(c), part = (len / n + 63) & ~(size_t)63;
    const size_t a = part * who < len ? part * who : len, b = who + 1 == n || a + part > len ? len : a + part;
    memcpy(dst + c * kSlot + a, sg.ring + c % kSlots * kSlot + a, b - a);
  };
  std::vector<std::thread> pool;
  std::atomic<int> members{0};  // set before the first slot is announced
  auto work = [&](int who) {
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
  for (size_t c = 0; c < nslot && c < (size_t)kSlots && !rc; ++c) rc = send(c);
  if (!rc) {
    try {
      pool.reserve(want - 1);
      for (; nthreads < want; ++nthreads) pool.emplace_back(work, nthreads);
    } catch (...) {  // no thread to be had: the caller copies more itself
    }
    members.store(nthreads, std::memory_order_relaxed);
  }
  for (size_t c = 0; c < nslot && !rc; ++c) {
    const hipError_t e = hipEventSynchronize(sg.ev[c % kSlots]);
    if (e != hipSuccess) {
      rc = fail(SPH_EDEVICE, "readback: %s", hipGetErrorString(e));
      break;
    }
    ready.store(c + 1, std::memory_order_release);
    share(c, 0, nthreads);
    if (c + kSlots < nslot) {
      // the slot is filled again once every worker has taken its share
      while (copied.load(std::memory_order_acquire) < (c + 1) * (size_t)(nthreads - 1))
        std::this_thread::yield();
      rc = send(c + kSlots);
    }
  }
  if (rc) stop.store(true);
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
  if (int rc = small_block(s->stage)) return rc;
  hipLaunchKernelGGL(k_read_ordered, dim3(1), dim3(1024), 0, s->st, dev, id, n,
                     (double*)s->stage.small);
  if (hipGetLastError() != hipSuccess) return fail(SPH_EDEVICE, "readback launch failed");
  HIPCHK(hipStreamSynchronize(s->st));
  memcpy(dst, s->stage.small, n * sizeof(double));
  return 0;
}

int copy_out(sph_sim* s, void* dst, const void* dev, size_t bytes) {
  if (bytes == 0) return 0;
  if (bytes > kSmallCopy) return copy_slots(s, (char*)dst, (const char*)dev, bytes);
  if (int rc = small_block(s->stage)) return rc;
  if (enqueue_copy_out(s->stage.small, dev, bytes, s->st))
    return fail(SPH_EDEVICE, "readback launch failed");
  HIPCHK(hipStreamSynchronize(s->st));
  memcpy(dst, s->stage.small, bytes);
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
  if (sizeof(KnnStats) + (size_t)nerr * sizeof(int) > kSmallBlock)
    return fail(SPH_EINVAL, "too many flags for one block");
  if (int rc = small_block(s->stage)) return rc;
  hipLaunchKernelGGL(k_flags, dim3(1), dim3(256), 0, s->st, s->pb.err, nerr, s->pb.stats,
                     (unsigned long long*)s->stage.small,
                     (int*)(s->stage.small + sizeof(KnnStats)));
  if (hipGetLastError() != hipSuccess) return fail(SPH_EDEVICE, "flags launch failed");
  return 0;
}

void take_flags(sph_sim* s, KnnStats* stats, int* err, int nerr) {
  memcpy(stats, s->stage.small, sizeof *stats);
  memcpy(err, s->stage.small + sizeof *stats, (size_t)nerr * sizeof(int));
}

}  // namespace sph

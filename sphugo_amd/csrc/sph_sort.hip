// Stable LSD radix sort of (cell key, particle index) pairs, 8-bit digits.
//
// Replaces the reference's per-pass Treebuild/Partition permutation
// (sim/core.go:126-224): particles are reordered by the Hilbert-curve
// index of their cell in a uniform 2^lg x 2^lg grid, so that every aligned
// square block of cells, at every level, is one contiguous range of the
// state arrays.
//
// Per pass: (1) block histograms of the digit, (2) one exclusive scan over
// the digit-major [256][blocks] table, (3) a stable scatter in which each
// wave ranks a contiguous quarter of the block's tile, 64 keys at a time, by
// matching digits with 9 ballots against per-wave digit counts in LDS; the
// waves' counts are then scanned once, the tile is gathered in digit order
// in LDS and written out so that each digit's run is contiguous.  Stability
// across passes makes the result independent of launch timing, so runs are
// bitwise reproducible.
#include <type_traits>
#include <utility>

#include "sph_device.hpp"
#include "sph_host.hpp"

namespace sph {

constexpr int kSortThreads = 256;
constexpr int kSortSub = 16;  // sub-tiles of 256 keys per block
constexpr int kSortTile = kSortThreads * kSortSub;

__global__ __launch_bounds__(kSortThreads) void k_sort_hist(
    const uint32_t* __restrict__ keys, int64_t n, int shift,
    uint32_t* __restrict__ counts, int nblocks) {
  __shared__ uint32_t hist[256];
  const int tid = threadIdx.x;
  hist[tid] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * kSortTile;
#pragma unroll 4
  for (int r = 0; r < kSortSub; ++r) {
    int64_t i = base + (int64_t)r * kSortThreads + tid;
    if (i < n) atomicAdd(&hist[(keys[i] >> shift) & 255u], 1u);
  }
  __syncthreads();
  counts[(int64_t)tid * nblocks + blockIdx.x] = hist[tid];
}

// Row d of the digit-major table counts[d][b]: exclusive scan over blocks b
// in place, row total to tot[d].  One block per digit.
__global__ __launch_bounds__(1024) void k_sort_rowscan(uint32_t* __restrict__ counts,
                                                       uint32_t* __restrict__ tot,
                                                       int nblocks) {
  __shared__ uint32_t part[1024];
  const int tid = threadIdx.x;
  uint32_t* row = counts + (int64_t)blockIdx.x * nblocks;
  const int per = (nblocks + 1023) / 1024;
  const int b = tid * per;
  uint32_t s = 0;
  for (int i = 0; i < per; ++i) s += (b + i < nblocks) ? row[b + i] : 0u;
  part[tid] = s;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    uint32_t t = tid >= o ? part[tid - o] : 0u;
    __syncthreads();
    part[tid] += t;
    __syncthreads();
  }
  uint32_t run = part[tid] - s;
  for (int i = 0; i < per && b + i < nblocks; ++i) {
    const uint32_t c = row[b + i];
    row[b + i] = run;
    run += c;
  }
  if (tid == 1023) tot[blockIdx.x] = part[1023];
}

__global__ __launch_bounds__(kSortThreads) void k_sort_scatter(
    const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
    uint32_t* __restrict__ kout, uint32_t* __restrict__ vout, int64_t n,
    int shift, const uint32_t* __restrict__ offsets, const uint32_t* __restrict__ tot,
    int nblocks, int identity_vals) {
  constexpr int kWaves = kSortThreads / 64;
  constexpr int kPerWave = kSortTile / kWaves;  // contiguous keys ranked by one wave
  __shared__ uint32_t wcnt[kWaves][256];  // per wave: keys of digit d so far
  __shared__ uint32_t scan[2][256];
  __shared__ uint32_t gofs[256];    // global position of this block's digit-d keys
  __shared__ uint32_t lstart[256];  // their first position in the block's sorted tile
  __shared__ uint32_t skey[kSortTile];
  __shared__ uint32_t sval[kSortTile];
  const int tid = threadIdx.x;
  const int w = tid >> 6;
  const int lane = tid & 63;
  const int b = blockIdx.x;
#pragma unroll
  for (int q = 0; q < kWaves; ++q) wcnt[q][tid] = 0;
  // exclusive prefix of the digit totals, this block's row offset, and the
  // exclusive prefix of this block's own digit counts
  {
    const uint32_t t = tot[tid];
    const uint32_t o = offsets[(int64_t)tid * nblocks + b];
    const uint32_t cnt = (b + 1 < nblocks ? offsets[(int64_t)tid * nblocks + b + 1] : t) - o;
    scan[0][tid] = t;
    scan[1][tid] = cnt;
    __syncthreads();
    for (int s = 1; s < 256; s <<= 1) {
      const uint32_t a = tid >= s ? scan[0][tid - s] : 0u;
      const uint32_t c = tid >= s ? scan[1][tid - s] : 0u;
      __syncthreads();
      scan[0][tid] += a;
      scan[1][tid] += c;
      __syncthreads();
    }
    gofs[tid] = scan[0][tid] - t + o;
    lstart[tid] = scan[1][tid] - cnt;
  }
  const int64_t base = (int64_t)b * kSortTile;
  const int count = (int)((n - base) < kSortTile ? (n - base) : kSortTile);
  const unsigned long long lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  // the wave's keys and values, all in flight at once
  uint32_t kreg[kSortSub], vreg[kSortSub], loc[kSortSub];
#pragma unroll
  for (int r = 0; r < kSortSub; ++r) {
    const int li = w * kPerWave + r * 64 + lane;
    const int64_t i = base + li;
    kreg[r] = li < count ? kin[i] : 0u;
    vreg[r] = li < count ? (identity_vals ? (uint32_t)i : vin[i]) : 0u;
  }
  // stable ranking within the wave, 64 keys per round in key order: a key's
  // place among its wave's keys of the same digit is the digit's count so
  // far plus the equal-digit lanes below it (matched with 9 ballots); the
  // lowest such lane then advances the count.  One wave's LDS operations
  // complete in order, so every round reads the count the last one left.
#pragma unroll
  for (int r = 0; r < kSortSub; ++r) {
    const int li = w * kPerWave + r * 64 + lane;
    const bool valid = li < count;
    const uint32_t d = valid ? ((kreg[r] >> shift) & 255u) : 256u;
    unsigned long long peers = ~0ull;
#pragma unroll
    for (int bit = 0; bit < 9; ++bit) {
      const bool on = (d >> bit) & 1u;
      const unsigned long long bal = ballot(on);
      peers &= on ? bal : ~bal;
    }
    const unsigned long long below = peers & lt_mask;
    const uint32_t before = valid ? wcnt[w][d] : 0u;
    loc[r] = before + (uint32_t)__popcll(below);
    __builtin_amdgcn_wave_barrier();
    if (valid && below == 0ull) wcnt[w][d] = before + (uint32_t)__popcll(peers);
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  // digit d of wave q starts after the block's earlier digits and the
  // digit-d keys of waves 0 .. q-1
  {
    uint32_t run = lstart[tid];
#pragma unroll
    for (int q = 0; q < kWaves; ++q) {
      const uint32_t c = wcnt[q][tid];
      wcnt[q][tid] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kSortSub; ++r) {
    const int li = w * kPerWave + r * 64 + lane;
    if (li < count) {
      const uint32_t lp = wcnt[w][(kreg[r] >> shift) & 255u] + loc[r];
      skey[lp] = kreg[r];
      sval[lp] = vreg[r];
    }
  }
  __syncthreads();
  // write out in tile order: runs of one digit go to consecutive addresses
  for (int li = tid; li < count; li += kSortThreads) {
    const uint32_t key = skey[li];
    const uint32_t d = (key >> shift) & 255u;
    const uint32_t dst = gofs[d] + ((uint32_t)li - lstart[d]);
    kout[dst] = key;
    vout[dst] = sval[li];
  }
}

// ---- up to kMidMax keys: digits of W = 6 .. 9 bits, two launches per pass;
// up to kOneMax: one launch for the whole sort ----
//
// Below a million keys the three launches of a pass above were mostly launch
// and latency.  Here a block finds its own offsets from the digit counts of all
// blocks, which costs each block a read of the whole table, and tiles are small,
// so that the keys spread over the chip.  The table bounds it: at 262,144 keys
// of 20 bits, 60 us above; 54 with two passes of 10 bits and 256 blocks (a
// 512 KiB table), 39 with 128 of them, 29 with three passes of 7 bits and 256
// blocks (64 KiB).  Hence digits of at most 9 bits in the fewest passes, and the
// fewest keys per thread (2, 4 or 8) that keep 256 blocks.  Against the three
// launches: 30,000 keys (18 bits) 57 -> 18 us, 77,777 (20) 58 -> 23, 524,288 (22)
// 63 -> 45, 1,048,576 (22) 69 -> 64; at 2,000,000 (24) 80 against 106, so kMidMax
// lies at 1,048,576.
constexpr int kMaxW = 9;
constexpr int kMidThreads = 512;
constexpr int kMidBlocks = 256;
constexpr int kMidMax = kMidBlocks * kMidThreads * 8;  // 2, 4 or 8 keys per thread
constexpr int kOneThreads = 1024;
constexpr int kOnePer = 8;
constexpr int kOneMax = kOneThreads * kOnePer;

// Digit counts of each tile, block-major, two to a word (a tile's count fits
// 16 bits).
// MAKE: the keys are made here (of simulation 0) and written out.
template <int PER, bool MAKE>
__global__ __launch_bounds__(kMidThreads) void k_sort_count(uint32_t* __restrict__ keys, KeySrc src,
                                                            int n, int shift, int w,
                                                            uint32_t* __restrict__ counts) {
  __shared__ uint32_t hist[1 << kMaxW];
  const int tid = threadIdx.x, nd = 1 << w;
  const int base = blockIdx.x * kMidThreads * PER;
  uint32_t key[PER];
  if constexpr (MAKE) {
    KeySrc::Raw raw[PER];
#pragma unroll
    for (int r = 0; r < PER; ++r) {
      const int i = base + r * kMidThreads + tid;
      raw[r] = src.load(src.sims, i < n ? i : n - 1);
    }
#pragma unroll
    for (int r = 0; r < PER; ++r) {
      const int i = base + r * kMidThreads + tid;
      key[r] = src.key(src.sims, 0, raw[r]);
      if (i < n) keys[i] = key[r];
    }
  } else {
#pragma unroll
    for (int r = 0; r < PER; ++r) {
      const int i = base + r * kMidThreads + tid;
      key[r] = i < n ? keys[i] : 0u;
    }
  }
  for (int d = tid; d < nd; d += kMidThreads) hist[d] = 0;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < PER; ++r)
    if (base + r * kMidThreads + tid < n)
      atomicAdd(&hist[(key[r] >> shift) & (uint32_t)(nd - 1)], 1u);
  __syncthreads();
  for (int p = tid; p < nd / 2; p += kMidThreads)
    counts[(int64_t)blockIdx.x * (nd / 2) + p] = hist[2 * p] | hist[2 * p + 1] << 16;
  if (MAKE && blockIdx.x == 0 && tid == 0) *src.retry_count = 0u;
}

// exclusive scan of the block's values, one per thread
template <int WAVES>
__device__ inline uint32_t block_scan(uint32_t v, uint32_t* wsum) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint32_t incl = (uint32_t)wave_incl_scan((int)v);
  if (lane == 63) wsum[wv] = incl;
  __syncthreads();
  uint32_t before = 0;
#pragma unroll
  for (int q = 0; q < WAVES; ++q) before += q < wv ? wsum[q] : 0u;
  __syncthreads();
  return before + incl - v;
}

// Stable places of a wave's keys, PER rounds of 64 in key order, against the
// wave's own digit counts (zero at first): loc[r] is the number of its
// earlier keys of the same digit.  A key's peers are matched with one ballot
// per bit; the lowest of them advances the count, and one wave's LDS operations
// complete in order, so every round reads the count the last one left.
template <int W, int PER>
__device__ inline void rank_keys(uint16_t* cnt, const uint32_t* key, int first, int end, int shift,
                                 uint32_t* loc) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    const bool valid = first + r * 64 < end;
    const uint32_t d = (key[r] >> shift) & ((1u << W) - 1u);
    const unsigned long long live = ballot(valid);
    uint32_t lo = (uint32_t)live, hi = (uint32_t)(live >> 32);
    if (live == 0ull) break;  // uniform: the wave's later keys lie past the end too
#pragma unroll
    for (int bit = 0; bit < W; ++bit) {
      const uint32_t mine = (uint32_t)((int32_t)(d << (31 - bit)) >> 31);  // bit in every place
      const unsigned long long b = ballot((d >> bit) & 1u);
      lo &= ~((uint32_t)b ^ mine);
      hi &= ~((uint32_t)(b >> 32) ^ mine);
    }
    const unsigned long long peers = (unsigned long long)hi << 32 | lo;
    const uint32_t before = cnt[d];
    const uint32_t below = (uint32_t)__builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
    loc[r] = before + below;
    __builtin_amdgcn_wave_barrier();
    if (valid && below == 0u) cnt[d] = (uint16_t)(before + (uint32_t)__popcll(peers));
    __builtin_amdgcn_wave_barrier();
  }
}

// One pass's move.  A block sums the counts of the blocks before it and of
// all blocks, scans the digits' totals, ranks its tile and writes it.
template <int W, int PER>
__global__ __launch_bounds__(kMidThreads) void k_sort_move(
    const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
    uint32_t* __restrict__ kout, uint32_t* __restrict__ vout, int n, int shift,
    const uint32_t* __restrict__ counts, int nblocks, int identity_vals) {
  constexpr int kWaves = kMidThreads / 64;
  constexpr int kD = 1 << W, kPairs = kD / 2;
  constexpr int kShare = kMidThreads / kPairs;  // threads per pair of digits
  __shared__ uint16_t cnt[kWaves][kD];
  __shared__ uint32_t start[kD];
  __shared__ uint4 part[kMidThreads];
  __shared__ uint32_t wsum[kWaves];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, b = blockIdx.x;
  const int first = b * (kMidThreads * PER) + wv * (PER * 64) + lane;
  uint32_t key[PER], val[PER], loc[PER];
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    const int i = first + r * 64;
    key[r] = i < n ? kin[i] : 0u;
    val[r] = i < n ? (identity_vals ? (uint32_t)i : vin[i]) : 0u;
  }
  for (int d = tid; d < kWaves * kPairs; d += kMidThreads) ((uint32_t*)cnt)[d] = 0u;
  {
    const int pair = tid & (kPairs - 1);
    uint4 a = make_uint4(0u, 0u, 0u, 0u);  // before, all of the two digits
    // 32 rows' loads in flight at a time
    for (int q0 = tid / kPairs; q0 < nblocks; q0 += 32 * kShare) {
      uint32_t c[32];
#pragma unroll
      for (int u = 0; u < 32; ++u) {
        const int q = q0 + u * kShare;
        c[u] = q < nblocks ? counts[q * kPairs + pair] : 0u;
      }
#pragma unroll
      for (int u = 0; u < 32; ++u) {
        const uint32_t c0 = c[u] & 0xFFFFu, c1 = c[u] >> 16;
        const bool mine = q0 + u * kShare < b;
        a.x += mine ? c0 : 0u;
        a.y += mine ? c1 : 0u;
        a.z += c0;
        a.w += c1;
      }
    }
    part[tid] = a;
    __syncthreads();
    uint4 t = make_uint4(0u, 0u, 0u, 0u);
    if (tid < kPairs)
#pragma unroll
      for (int q = 0; q < kShare; ++q) {
        const uint4 v = part[q * kPairs + tid];
        t.x += v.x;
        t.y += v.y;
        t.z += v.z;
        t.w += v.w;
      }
    const uint32_t ex = block_scan<kWaves>(t.z + t.w, wsum);
    if (tid < kPairs) {
      start[2 * tid] = ex + t.x;
      start[2 * tid + 1] = ex + t.z + t.y;
    }
  }
  rank_keys<W, PER>(cnt[wv], key, first, n, shift, loc);
  __syncthreads();
  for (int d = tid; d < kD; d += kMidThreads) {
    uint32_t run = 0;
#pragma unroll
    for (int q = 0; q < kWaves; ++q) {
      const uint32_t c = cnt[q][d];
      cnt[q][d] = (uint16_t)run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    if (first + r * 64 < n) {
      const uint32_t d = (key[r] >> shift) & (uint32_t)(kD - 1);
      const uint32_t at = start[d] + cnt[wv][d] + loc[r];
      kout[at] = key[r];
      vout[at] = val[r];
    }
  }
}

// The whole sort of at most kOneMax keys by one block: every pass ranks the
// keys in registers and moves them through LDS (2,200 keys of 14 bits: 6.4 us
// against 34 us in six launches).
template <int W>
__global__ __launch_bounds__(kOneThreads) void k_sort_one(const uint32_t* __restrict__ kin,
                                                          uint32_t* __restrict__ kout,
                                                          uint32_t* __restrict__ vout, int n,
                                                          int passes) {
  constexpr int kWaves = kOneThreads / 64;
  constexpr int kD = 1 << W;
  __shared__ uint16_t cnt[kWaves][kD];
  __shared__ uint32_t skey[kOneMax], sval[kOneMax];
  __shared__ uint32_t wsum[kWaves];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  // every wave takes the same number of whole rounds of 64 consecutive keys
  const int rounds = (n + kOneThreads - 1) / kOneThreads;
  const int base = wv * rounds * 64, first = base + lane;
  const int end = base + rounds * 64 < n ? base + rounds * 64 : n;
  uint32_t key[kOnePer], val[kOnePer], loc[kOnePer];
#pragma unroll
  for (int r = 0; r < kOnePer; ++r) key[r] = first + r * 64 < end ? kin[first + r * 64] : 0u;
#pragma unroll
  for (int r = 0; r < kOnePer; ++r) val[r] = (uint32_t)(first + r * 64);
  for (int p = 0; p < passes; ++p) {
    for (int d = tid; d < kWaves * kD / 2; d += kOneThreads) ((uint32_t*)cnt)[d] = 0u;
    __syncthreads();
    rank_keys<W, kOnePer>(cnt[wv], key, first, end, p * W, loc);
    __syncthreads();
    uint32_t all = 0;
    if (tid < kD)
#pragma unroll
      for (int q = 0; q < kWaves; ++q) all += cnt[q][tid];
    uint32_t run = block_scan<kWaves>(all, wsum);
    if (tid < kD)
#pragma unroll
      for (int q = 0; q < kWaves; ++q) {
        const uint32_t c = cnt[q][tid];
        cnt[q][tid] = (uint16_t)run;
        run += c;
      }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kOnePer; ++r) {
      const int i = first + r * 64;
      if (i < end) {
        const uint32_t at =
            (uint32_t)cnt[wv][(key[r] >> (p * W)) & (uint32_t)(kD - 1)] + loc[r];
        skey[at] = key[r];
        sval[at] = val[r];
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kOnePer; ++r) {
      const int i = first + r * 64;
      if (i < end) {
        key[r] = skey[i];
        val[r] = sval[i];
      }
    }
  }
#pragma unroll
  for (int r = 0; r < kOnePer; ++r) {
    const int i = first + r * 64;
    if (i < end) {
      kout[i] = key[r];
      vout[i] = val[r];
    }
  }
}

// Calls f with the digit width w in [6, kMaxW] as a compile-time constant.
template <typename F>
static void with_width(int w, F&& f) {
  if (w <= 6) f(std::integral_constant<int, 6>{});
  else if (w == 7) f(std::integral_constant<int, 7>{});
  else if (w == 8) f(std::integral_constant<int, 8>{});
  else f(std::integral_constant<int, kMaxW>{});
}

// Between the one-block sort (whose single block made 2,200 keys no faster than
// a launch of its own: 4.5 us) and 8 keys per thread (1,048,576 keys: 16.3 us
// against 9.7 + 4.9 us apart); at 77,777 keys 4.8 us against 4.7 + 2.4, at 262,144
// 5.2 against 4.8 + 4.7.
bool sort_makes_keys(int64_t n) { return n > kOneMax && n <= kMidMax / 2; }

int sort_pairs(SortBuffers& sb, int64_t n, int bits, hipStream_t st, const KeySrc* make,
               uint32_t** keys_out, uint32_t** vals_out) {
  const int nblocks = (int)((n + kSortTile - 1) / kSortTile);
  uint32_t* kin = sb.keys;
  uint32_t* vin = sb.vals;
  uint32_t* kout = sb.keys_alt;
  uint32_t* vout = sb.vals_alt;
  if (bits < 1) bits = 1;
  if (n <= kMidMax) {
    const int passes = (bits + kMaxW - 1) / kMaxW;
    with_width((bits + passes - 1) / passes, [&](auto width) {
      constexpr int W = decltype(width)::value;
      const KeySrc src = make ? *make : KeySrc{};
      if (n <= kOneMax) {
        hipLaunchKernelGGL((k_sort_one<W>), dim3(1), dim3(kOneThreads), 0, st, kin, kout, vout,
                           (int)n, passes);
        kin = kout;
        vin = vout;
        return;
      }
      // the fewest keys per thread that keep the count table at kMidBlocks rows
      auto run = [&](auto per) {
        constexpr int P = decltype(per)::value;
        const int nb = (int)((n + kMidThreads * P - 1) / (kMidThreads * P));
        for (int p = 0; p < passes; ++p) {
          if (make && p == 0)
            hipLaunchKernelGGL((k_sort_count<P, true>), dim3(nb), dim3(kMidThreads), 0, st, kin, src,
                               (int)n, p * W, W, sb.counts);
          else
            hipLaunchKernelGGL((k_sort_count<P, false>), dim3(nb), dim3(kMidThreads), 0, st, kin,
                               src, (int)n, p * W, W, sb.counts);
          hipLaunchKernelGGL((k_sort_move<W, P>), dim3(nb), dim3(kMidThreads), 0, st, kin, vin,
                             kout, vout, (int)n, p * W, sb.counts, nb,
                             p == 0 ? 1 : 0);
          std::swap(kin, kout);
          std::swap(vin, vout);
        }
      };
      if (n <= kMidMax / 4) run(std::integral_constant<int, 2>{});
      else if (n <= kMidMax / 2) run(std::integral_constant<int, 4>{});
      else run(std::integral_constant<int, 8>{});
    });
    *keys_out = kin;
    *vals_out = vin;
    return (int)hipGetLastError();
  }
  const int passes = (bits + 7) / 8;
  for (int p = 0; p < passes; ++p) {
    const int shift = 8 * p;
    hipLaunchKernelGGL(k_sort_hist, dim3(nblocks), dim3(kSortThreads), 0, st, kin, n,
                       shift, sb.counts, nblocks);
    hipLaunchKernelGGL(k_sort_rowscan, dim3(256), dim3(1024), 0, st, sb.counts, sb.tot,
                       nblocks);
    hipLaunchKernelGGL(k_sort_scatter, dim3(nblocks), dim3(kSortThreads), 0, st, kin, vin,
                       kout, vout, n, shift, sb.counts, sb.tot, nblocks,
                       p == 0 ? 1 : 0);
    uint32_t* t = kin; kin = kout; kout = t;
    t = vin; vin = vout; vout = t;
  }
  *keys_out = kin;
  *vals_out = vin;
  return (int)hipGetLastError();
}

int64_t sort_counts_size(int64_t n) {
  // of any n' <= n (a serve pool sorts its occupied part).  The count table of
  // the sorts up to kMidMax has at most kMidBlocks rows of two digits a word.
  const int64_t large = (int64_t)256 * ((n + kSortTile - 1) / kSortTile);
  const int64_t rows = (n + 2 * kMidThreads - 1) / (2 * kMidThreads);
  const int64_t mid = (rows < kMidBlocks ? rows : kMidBlocks) << (kMaxW - 1);
  return large > mid ? large : mid;
}

}  // namespace sph

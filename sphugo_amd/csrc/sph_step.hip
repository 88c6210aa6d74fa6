// SPH force pass and integrator kernels for gfx950 (wave64).
//
//   k_keys          cell key of each particle's pass position: Hilbert index
//                   of a power-of-two grid plus the simulation's cell offset
//                   (replaces Treebuild/Partition, sim/core.go:126-224); made by
//                   the sort itself for one simulation of up to a million
//                   particles
//   sort_pairs      stable LSD radix sort of (key, index) (sph_sort.hip)
//   k_permute       gather the state into cell order, apply the drift-1 /
//                   predictor step (sim/sph.go:108-117) or the step-0
//                   initialisation (:96-101); other blocks of the launch
//                   write the cell ranges
//   k_knn           bracketed walk: a wavefront searches groups of 16
//                   consecutive queries, sorting the candidates of each
//                   group's box against every query's bracket around its last
//                   h, then selects the k-th neighbour exactly, sums the
//                   density and writes sound speed and the force record;
//                   misses go to a retry list
//                   (sim/nearest-neighbour.go:28-165, sim/sph.go:306-323,
//                   421-429)
//   k_knn_fallback  exact wavefront-per-query search for the retry list
//   k_force         thread per particle: pressure + artificial viscosity +
//                   EDot over the packed records of its neighbours, fused
//                   with kick, drift 2, periodic wrap and reflection
//                   (sim/sph.go:327-401,122-193), partial sums and the CFL
//                   minimum; in small launches the totals too
//   k_reduce_part,  per-simulation FP64 totals in a fixed order, the next
//   k_reduce        CFL half step and the next kNN walk bracket
//
// All FP64 arithmetic on the parity path is evaluated in the reference's
// association order; the library is compiled with -ffp-contract=off so no
// product is fused into an add there.  Only the FP32C pair terms enable
// contraction, block by block.
#include <algorithm>
#include <type_traits>

#include "sph_device.hpp"
#include "sph_host.hpp"

namespace sph {

// Cell span [a, b] of a search at a level with nc cells per axis, limited to
// the images the reference visits: [-2 nc, 3 nc) on a periodic axis (the
// -L, 0, +L images of positions that may sit up to a box outside it), the
// box itself on an open axis (sim/nearest-neighbour.go:39-55).
__device__ inline void clamp_span(int64_t& a, int64_t& b, int64_t nc, bool open) {
  const int64_t lo = open ? 0 : -2 * nc, hi = open ? nc - 1 : 3 * nc - 1;
  if (a < lo) a = lo;
  if (b > hi) b = hi;
  if (b < a) b = a - 1;  // empty span
}

// Box of each open simulation's pass positions, in two launches: per work
// item the range of the positions k_keys bins (same predictor arithmetic),
// then per simulation the range over its items and the grid box (open_box).
// Periodic simulations and unused pool slots are skipped.
__global__ __launch_bounds__(kItem) void k_bbox(const Item* __restrict__ items, int nitems,
                                                const SimDev* __restrict__ sims,
                                                const double* __restrict__ X,
                                                const double* __restrict__ Y,
                                                const double* __restrict__ VX,
                                                const double* __restrict__ VY, int mode,
                                                double* __restrict__ part) {
  __shared__ double red[4][4];
  const int item_idx = blockIdx.x;
  const Item it = items[item_idx];
  if (it.sim < 0) return;
  const SimDev* S = sims + it.sim;
  if (!S->open) return;
  if (mode < 0) mode = S->pmode;
  double x0 = INFINITY, x1 = -INFINITY, y0 = INFINITY, y1 = -INFINITY;
  if ((int)threadIdx.x < it.count) {
    const int64_t t = it.first + threadIdx.x;
    double x = X[t], y = Y[t];
    if (mode == kPermPredict) {
      const double dt = S->dt_half;
      x = x + VX[t] * dt;
      y = y + VY[t] * dt;
    }
    x0 = x1 = x;
    y0 = y1 = y;
  }
  for (int o = 32; o > 0; o >>= 1) {
    x0 = fmin(x0, __shfl_xor(x0, o, 64));
    x1 = fmax(x1, __shfl_xor(x1, o, 64));
    y0 = fmin(y0, __shfl_xor(y0, o, 64));
    y1 = fmax(y1, __shfl_xor(y1, o, 64));
  }
  const int wv = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    red[wv][0] = x0;
    red[wv][1] = x1;
    red[wv][2] = y0;
    red[wv][3] = y1;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) {
      x0 = fmin(x0, red[w][0]);
      x1 = fmax(x1, red[w][1]);
      y0 = fmin(y0, red[w][2]);
      y1 = fmax(y1, red[w][3]);
    }
    double* p = part + (int64_t)item_idx * kNumRed;
    p[0] = x0;
    p[1] = x1;
    p[2] = y0;
    p[3] = y1;
  }
}

__global__ __launch_bounds__(256) void k_box(SimDev* __restrict__ sims,
                                             const double* __restrict__ part,
                                             const int* __restrict__ item_first,
                                             const int* __restrict__ item_count) {
  __shared__ double red[4][4];
  SimDev* S = sims + blockIdx.x;
  if (S->n == 0 || !S->open) return;
  const int i0 = item_first[blockIdx.x], ni = item_count[blockIdx.x];
  double x0 = INFINITY, x1 = -INFINITY, y0 = INFINITY, y1 = -INFINITY;
  for (int i = threadIdx.x; i < ni; i += 256) {
    const double* p = part + (int64_t)(i0 + i) * kNumRed;
    x0 = fmin(x0, p[0]);
    x1 = fmax(x1, p[1]);
    y0 = fmin(y0, p[2]);
    y1 = fmax(y1, p[3]);
  }
  for (int o = 32; o > 0; o >>= 1) {
    x0 = fmin(x0, __shfl_xor(x0, o, 64));
    x1 = fmax(x1, __shfl_xor(x1, o, 64));
    y0 = fmin(y0, __shfl_xor(y0, o, 64));
    y1 = fmax(y1, __shfl_xor(y1, o, 64));
  }
  const int wv = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    red[wv][0] = x0;
    red[wv][1] = x1;
    red[wv][2] = y0;
    red[wv][3] = y1;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) {
      x0 = fmin(x0, red[w][0]);
      x1 = fmax(x1, red[w][1]);
      y0 = fmin(y0, red[w][2]);
      y1 = fmax(y1, red[w][3]);
    }
    SimDev d = *S;
    open_box(d, x0, x1, y0, y1);
    S->x0 = d.x0;
    S->lx = d.lx;
    S->ivx = d.ivx;
    S->sx = d.sx;
    S->y0 = d.y0;
    S->ly = d.ly;
    S->ivy = d.ivy;
    S->sy = d.sy;
  }
}

__global__ __launch_bounds__(kItem) void k_keys(const Item* __restrict__ items, int nitems,
                                                KeySrc src, uint32_t* __restrict__ keys,
                                                uint32_t hole_cpp) {
  const Item it = items[xcd_item(nitems)];
  if ((int)threadIdx.x >= it.count) return;
  const int64_t t = it.first + threadIdx.x;
  if (it.sim < 0) {
    // unused pool slot: a key of its own position keeps it in place
    keys[t] = (uint32_t)(t * hole_cpp);
    if (blockIdx.x == 0 && threadIdx.x == 0) *src.retry_count = 0u;
    return;
  }
  const SimDev* S = src.sims + it.sim;
  keys[t] = src.key(S, it.sim, src.load(S, t));
  if (blockIdx.x == 0 && threadIdx.x == 0) *src.retry_count = 0u;
}

// Number of keys below `target` in the sorted skeys[lo, hi), plus lo, by one wave:
// 64 probes at a time.
__device__ inline int64_t wave_lower_bound(const uint32_t* __restrict__ skeys, int64_t lo,
                                           int64_t hi, uint32_t target, int lane) {
  while (hi - lo > 64) {
    const int64_t step = (hi - lo + 63) >> 6;
    const int64_t p = lo + lane * step;
    const int below = __popcll(ballot(p < hi && skeys[p] < target));
    const int64_t l = lo;
    lo = below ? l + (below - 1) * step + 1 : l;
    hi = l + below * step < hi ? l + below * step : hi;
    if (hi < lo) hi = lo;
  }
  const int64_t p = lo + lane;
  return lo + __popcll(ballot(p < hi && skeys[p] < target));
}

// The cell ranges of the shares of `nit` consecutive items, from `it` on, of
// their simulation's cells [coff, coff + G^2): cell q starts at the first
// particle whose key is >= q.  The block finds the particles of its cells in the
// sorted keys, counts them per cell in LDS and writes the counts' running sum,
// so every cell and key is touched once wherever the particles are.  Bound by
// latency (two searches, then one chain per 2,048 cells), so it runs beside the
// permuting blocks.  Written by the permuting waves instead, each the cells up
// to its particles' keys, a sparse stretch of the grid held a wave and needed a
// queue and a launch of its own.  Permute with cell ranges, before and now:
// 2,200 particles 10.0 -> 4.7 us, 4,700 in a tube 23.2 -> 6.8, 12 simulations
// served together 24 -> 12.3, 77,777 14 -> 9.1, 262,144 14.4 -> 10.0, 1M clustered
// 42.8 -> 38.7, 4M 144.6 -> 149.5.  Cells outside every simulation's range are
// never read.
constexpr int kCellChunk = 2048;
__device__ inline void item_cells(const Item& it, int nit, const SimDev* S,
                                  const uint32_t* __restrict__ skeys,
                                  uint32_t* __restrict__ cstart) {
  __shared__ uint32_t cnt[kCellChunk];
  __shared__ uint32_t wsum[kItem / 64];
  __shared__ int64_t bound[2];
  constexpr int kOwn = kCellChunk / kItem;  // counters scanned by a thread
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int64_t off = S->off, end = off + S->n;
  const int64_t cells = (int64_t)S->gx * S->gy;
  const int64_t ni = (S->n + kItem - 1) / kItem, li = (it.first - off) / kItem;
  const int64_t c0 = cells * li / ni, c1 = cells * (li + nit) / ni;
  int64_t a = -1;
  for (int64_t c = c0; c < c1; c += kCellChunk) {
    const int nc = (int)(c1 - c < kCellChunk ? c1 - c : kCellChunk);
    // the chunk's particles [a, b); the next chunk goes on at b
    if (wv == 0 && a < 0) {
      const int64_t v = wave_lower_bound(skeys, off, end, (uint32_t)(S->coff + c), lane);
      if (lane == 0) bound[0] = v;
    }
    if (wv == 1) {
      const int64_t v = wave_lower_bound(skeys, off, end, (uint32_t)(S->coff + c + nc), lane);
      if (lane == 0) bound[1] = v;
    }
    for (int i = tid; i < kCellChunk; i += kItem) cnt[i] = 0u;
    __syncthreads();
    if (a < 0) a = bound[0];
    const int64_t b = bound[1];
    // eight loads in flight per thread (a dense chunk holds many particles)
    for (int64_t t = a + tid; t < b; t += 8 * kItem) {
      uint32_t key[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) key[u] = t + u * kItem < b ? skeys[t + u * kItem] : 0u;
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (t + u * kItem < b) atomicAdd(&cnt[key[u] - (uint32_t)(S->coff + c)], 1u);
    }
    __syncthreads();
    uint32_t own[kOwn], sum = 0;
#pragma unroll
    for (int i = 0; i < kOwn; ++i) {
      own[i] = cnt[tid * kOwn + i];
      sum += own[i];
    }
    const uint32_t incl = (uint32_t)wave_incl_scan((int)sum);
    if (lane == 63) wsum[wv] = incl;
    __syncthreads();
    uint32_t run = (uint32_t)a + incl - sum;
#pragma unroll
    for (int q = 0; q < kItem / 64; ++q) run += q < wv ? wsum[q] : 0u;
#pragma unroll
    for (int i = 0; i < kOwn; ++i) {
      cnt[tid * kOwn + i] = run;
      run += own[i];
    }
    __syncthreads();
    for (int i = tid; i < nc; i += kItem) cstart[S->coff + c + i] = cnt[i];
    __syncthreads();
    a = b;
  }
  if (li + nit == ni && tid == 0) cstart[S->coff + cells] = (uint32_t)end;
}

// The first ncells blocks write the cell ranges, per_cells items' shares each;
// the rest permute a work item each.  The ranges come first, so that their
// chains are covered by the permuting blocks: behind them the launch takes 164 us
// at 4M against 147, and 13.6 against 11.9 at 262,144.
__global__ __launch_bounds__(kItem) void k_permute(
    const Item* __restrict__ items_all, int nitems_all, const Item* __restrict__ items, int nitems,
    int ncells, int per_cells, const SimDev* __restrict__ sims, const uint32_t* __restrict__ perm,
    const uint32_t* __restrict__ skeys, int mode, Positions pin, Fields fin,
    double2* __restrict__ xyp, Fields fout, uint8_t* __restrict__ wrap,
    uint32_t* __restrict__ cstart) {
  if ((int)blockIdx.x < ncells) {
    const int i0 = xcd_item(ncells) * per_cells;
    for (int i = i0; i < i0 + per_cells && i < nitems;) {
      // consecutive items of one simulation share their searches
      const Item it = items[i];
      int n = 1;
      while (i + n < i0 + per_cells && i + n < nitems && items[i + n].sim == it.sim) ++n;
      item_cells(it, n, sims + it.sim, skeys, cstart);
      i += n;
    }
    return;
  }
  const Item it = items_all[xcd_item(nitems_all, (int)blockIdx.x - ncells)];
  if (it.sim < 0) return;  // unused pool slot: stays in place
  const SimDev* S = sims + it.sim;
  const bool valid = (int)threadIdx.x < it.count;
  const int64_t t = it.first + (valid ? threadIdx.x : 0);
  if (valid) {
    const uint32_t i = perm[t];
    if (mode < 0) mode = S->pmode;
    double x = pin.x[i], y = pin.y[i];
    const double vx = fin.vx[i], vy = fin.vy[i], e = fin.e[i];
    double vpx, vpy, ep;
    if (mode == kPermPredict) {
      const double dt = S->dt_half;
      x = x + vx * dt;
      y = y + vy * dt;
      const double adx = fin.ax[i] * dt, ady = fin.ay[i] * dt;
      vpx = vx + adx;
      vpy = vy + ady;
      ep = e + fin.edot[i] * dt;
    } else if (mode == kPermInit) {
      vpx = vx; vpy = vy; ep = e;
    } else {
      vpx = fin.vpx[i]; vpy = fin.vpy[i]; ep = fin.ep[i];
    }
    xyp[t] = make_double2(x, y);
    fout.vx[t] = vx;
    fout.vy[t] = vy;
    fout.e[t] = e;
    fout.vpx[t] = vpx;
    fout.vpy[t] = vpy;
    fout.ep[t] = ep;
    fout.h[t] = fin.h[i];
    fout.id[t] = fin.id[i];
    CellIdx c = cell_of(S, x, y);
    const int64_t wx = floordiv_pow2(c.ux, S->lg), wy = floordiv_pow2(c.uy, S->lg);
    wrap[t] = (uint8_t)((wx + 2) | ((wy + 2) << 3));
  }
}

// ------------------------------------------------------------------------
// kNN.
//
// Candidates are the particles of the cells at a coarser level of the
// grid: a coarse cell (X, Y) at level c is one contiguous range of the
// sorted arrays, [cstart[m << 2(lg-c)], cstart[(m+1) << 2(lg-c)]) with m
// its Hilbert index at that level.  Periodic images follow the reference:
// a candidate j is seen through the query offsets o in {-L, 0, L}^2 and its
// squared distance is ((p_i + o) - p_j)^2 (sim/nearest-neighbour.go:57-61,
// 72,76), self excluded at every image (:79).  The k nearest are ordered by
// (d2, ID, image) so ties resolve the same way everywhere.

__device__ inline int level_for(const SimDev* S, double w, double hgt, double ncells) {
  int c = S->lg;
  while (c > 0 && ((double)(1 << c) * w > ncells * S->lx || (double)(1 << c) * hgt > ncells * S->ly))
    --c;
  return c;
}

__device__ inline void cell_range(const SimDev* S, const uint32_t* __restrict__ cstart, int c,
                                  uint32_t xw, uint32_t yw, uint32_t& a, uint32_t& b) {
  const int sh = 2 * (S->lg - c);
  const uint64_t m = (uint64_t)hilbert2(xw, yw, c) << sh;
  a = cstart[S->coff + m];
  b = cstart[S->coff + m + (1ull << sh)];
}

// The Hilbert index (hilbert2) of cell (x, y) at level c <= 15, three levels
// per step: the orientation (swap, complement) entering three levels and their
// three bits of x and y give the six index bits and the orientation that
// leaves them.  The 256 bytes of that table sit in one register per lane
// (lane l: entries 4 l .. 4 l + 3) and are looked up across the lanes.  A
// level of zero bits above the first only flips the swap, so a start
// orientation of their parity pads c to a multiple of three.
struct HilbertTable {
  uint32_t w[64];
};
constexpr HilbertTable make_hilbert_table() {
  HilbertTable t{};
  for (uint32_t i = 0; i < 256; ++i) {
    uint32_t swap = i >> 6 & 1u, comp = i >> 7, d = 0;
    for (int s = 2; s >= 0; --s) {
      const uint32_t bx = (i >> (3 + s)) & 1u, by = (i >> s) & 1u;
      const uint32_t rx = (swap ? by : bx) ^ comp;
      const uint32_t ry = (swap ? bx : by) ^ comp;
      d = (d << 2) | ((3u * rx) ^ ry);
      const uint32_t m = ry ^ 1u;
      swap ^= m;
      comp ^= m & rx;
    }
    t.w[i >> 2] |= (d | swap << 6 | comp << 7) << (8 * (i & 3u));
  }
  return t;
}
__constant__ const HilbertTable kHilbertTable = make_hilbert_table();
__device__ inline uint32_t hilbert_lookup(uint32_t table, uint32_t x, uint32_t y, int c) {
  const int steps = (c + 2) / 3;
  uint32_t d = 0, state = (uint32_t)(3 * steps - c) & 1u;
  for (int s = 3 * (steps - 1); s >= 0; s -= 3) {
    const uint32_t i = state << 6 | ((x >> s) & 7u) << 3 | ((y >> s) & 7u);
    const uint32_t e =
        (uint32_t)__builtin_amdgcn_ds_bpermute((int)i, (int)table) >> (8 * (i & 3u)) & 255u;
    d = d << 6 | (e & 63u);
    state = e >> 6;
  }
  return d;
}

constexpr int kV1Cells = 128;  // coarse cells of one search (<= 9 x 9 used)

// Per-wave scratch of the exact wavefront search.
struct SearchShared {
  double d2[kCandCap];
  uint32_t pk[kCandCap];
  uint32_t pst[kV1Cells];
  int ppref[kV1Cells + 1];
  int8_t ptx[kV1Cells];
  int8_t pty[kV1Cells];
  double sd2[kMaxK];
  uint32_t spk[kMaxK];
  double fterm[kMaxK];
};

struct SearchOut {
  double tau;   // k-th smallest squared distance
  double facc;  // sum of kernel values F(d/h) over the k neighbours
};

// Candidate of a piece: returns false if the reference does not visit
// this (particle, image) pair.
__device__ inline bool cand_image(int ptx, int pty, uint8_t wc, int& ix, int& iy) {
  const int nx = ptx - ((int)(wc & 7) - 2);
  const int ny = pty - ((int)(wc >> 3) - 2);
  ix = -nx;
  iy = -ny;
  return nx >= -1 && nx <= 1 && ny >= -1 && ny <= 1;
}

// Neighbour lists are stored in tiles of 64 consecutive queries: entry e of
// query t lives at tile(t) * kstride * 64 + (e / 4) * 256 + (t % 64) * 4 +
// e % 4 (u32 units), so 64 lanes reading the same 4-entry chunk of their
// rows touch one contiguous 1 KiB segment.  kstride is a multiple of 4.
struct NbrRow {
  uint32_t* base;
  __device__ uint32_t& operator[](int e) const { return base[(e >> 2) * 256 + (e & 3)]; }
  __device__ u32x4* chunk(int c) const { return (u32x4*)(base + c * 256); }
};
__device__ inline NbrRow nbr_row(uint32_t* nbr, int64_t t, int kstride) {
  return NbrRow{nbr + (t >> 6) * (int64_t)kstride * 64 + (t & 63) * 4};
}
__device__ inline NbrRow nbr_row(const uint32_t* nbr, int64_t t, int kstride) {
  return nbr_row(const_cast<uint32_t*>(nbr), t, kstride);
}

// Exact kNN of one query by the whole wavefront, starting from radius R.
// Writes the k entries of `row` (BITWISE: sorted descending by (d2, ID,
// image), the reference's queue order) and returns tau and the density
// kernel sum (BITWISE: summed farthest first, sim/sph.go:313-320).
template <bool BITWISE>
__device__ SearchOut wave_search(const SimDev* S, int64_t t, double xq, double yq, double R,
                                 const double2* __restrict__ XY,
                                 const uint8_t* __restrict__ WR,
                                 const uint32_t* __restrict__ cstart,
                                 const uint32_t* __restrict__ ID, uint32_t table, NbrRow row,
                                 SearchShared& sh, unsigned long long& nretry,
                                 unsigned long long& nties, unsigned long long& nfail) {
  const int lane = lane_id();
  const int k = S->k;
  const double lx = S->lx, ly = S->ly;
  // every image of every particle lies within 2 sqrt(2) max(lx, ly) of the query
  const double rcap = 3.0 * (lx > ly ? lx : ly);
  if (R > rcap) R = rcap;
  double r_lo = 0.0, r_hi = 0.0;
  int cnt = 0;
  double R2 = 0;
  int attempt = 0;
  for (;; ++attempt) {
    R2 = R * R;
    const double Rm = R * (1 + 1e-12) + 1e-15 * (lx + ly);
    const int c = level_for(S, 2 * Rm, 2 * Rm, 8.0);
    const int64_t nc = 1LL << c;
    const double icx = (double)nc / lx, icy = (double)nc / ly;
    const double scx = lx / (double)nc, scy = ly / (double)nc;
    int64_t X0 = (int64_t)floor((xq - S->x0 - Rm) * icx), X1 = (int64_t)floor((xq - S->x0 + Rm) * icx);
    int64_t Y0 = (int64_t)floor((yq - S->y0 - Rm) * icy), Y1 = (int64_t)floor((yq - S->y0 + Rm) * icy);
    clamp_span(X0, X1, nc, S->open & 1);
    clamp_span(Y0, Y1, nc, S->open & 2);
    const int nX = (int)(X1 - X0 + 1), nY = (int)(Y1 - Y0 + 1);
    const int ncell = nX * nY;
    int npieces = 0, ncand = 0;
    for (int cb = 0; cb < ncell; cb += 64) {
      const int ci = cb + lane;
      bool have = false;
      uint32_t a = 0, b = 0;
      int tx = 0, ty = 0;
      // every lane takes part in the lookup
      const int row_ = ci / nX;
      const int Xc = (int)X0 + (ci - row_ * nX), Yc = (int)Y0 + row_;
      const uint32_t hix =
          hilbert_lookup(table, (uint32_t)Xc & (uint32_t)(nc - 1), (uint32_t)Yc & (uint32_t)(nc - 1), c);
      if (ci < ncell) {
        const double bx0 = S->x0 + (double)Xc * scx, by0 = S->y0 + (double)Yc * scy;
        const double dx = xq < bx0 ? bx0 - xq : (xq > bx0 + scx ? xq - (bx0 + scx) : 0.0);
        const double dy = yq < by0 ? by0 - yq : (yq > by0 + scy ? yq - (by0 + scy) : 0.0);
        if (dx * dx + dy * dy <= Rm * Rm) {
          tx = Xc >> c;
          ty = Yc >> c;
          const uint32_t* p = cstart + S->coff + ((uint64_t)hix << (2 * (S->lg - c)));
          a = p[0];
          b = p[1ull << (2 * (S->lg - c))];
          have = b > a;
        }
      }
      const unsigned long long m = ballot(have);
      const int len = have ? (int)(b - a) : 0;
      const int incl = wave_incl_scan(len);
      if (have) {
        const int pos = npieces + lane_prefix(m);
        sh.pst[pos] = a;
        sh.ppref[pos] = ncand + incl - len;
        sh.ptx[pos] = (int8_t)tx;
        sh.pty[pos] = (int8_t)ty;
      }
      npieces += __popcll(m);
      ncand += __shfl(incl, 63, 64);
    }
    if (lane == 0) sh.ppref[npieces] = ncand;
    __builtin_amdgcn_wave_barrier();
    int nsteps = 0;
    while ((1 << nsteps) < npieces) ++nsteps;
    cnt = 0;
    // Stage s takes candidate lane * nst + s: each lane walks a run of
    // consecutive candidates, so its piece is found by a binary search once
    // and then moves at most one step per stage (every piece is non-empty).
    const int nst = (ncand + 63) >> 6;
    int lo = 0;
    {
      const int u0 = lane * nst;
      if (u0 < ncand) {
        int hi = npieces - 1;
        for (int s = 0; s < nsteps; ++s) {
          const int mid = (lo + hi + 1) >> 1;
          if (sh.ppref[mid] <= u0) lo = mid; else hi = mid - 1;
        }
      }
    }
    // three stages' positions are loaded before the first is used
    constexpr int kAhead = 3;
    for (int stage = 0; stage < nst; stage += kAhead) {
      double2 pj[kAhead];
      uint32_t j[kAhead];
      int at[kAhead];
      uint8_t wc[kAhead];
#pragma unroll
      for (int r = 0; r < kAhead; ++r) {
        const int u = lane * nst + stage + r;
        if (u < ncand && stage + r < nst) {
          if (sh.ppref[lo + 1] <= u) ++lo;
          at[r] = lo;
          j[r] = sh.pst[lo] + (uint32_t)(u - sh.ppref[lo]);
          wc[r] = WR[j[r]];
          pj[r] = XY[j[r]];
        }
      }
#pragma unroll
      for (int r = 0; r < kAhead; ++r) {
        if (stage + r >= nst) break;  // uniform
        bool acc = false;
        double d2 = 0;
        uint32_t pk = 0;
        if (lane * nst + stage + r < ncand) {
          int ix, iy;
          const bool vis = cand_image(sh.ptx[at[r]], sh.pty[at[r]], wc[r], ix, iy);
          const bool seen = vis && (int64_t)j[r] != t;
          const double ex = (xq + (double)ix * lx) - pj[r].x;
          const double ey = (yq + (double)iy * ly) - pj[r].y;
          d2 = ex * ex + ey * ey;
          acc = seen && d2 <= R2;
          pk = (j[r] << 4) | img_code(seen ? ix : 0, seen ? iy : 0);
        }
        const unsigned long long m = ballot(acc);
        if (acc) {
          const int pos = cnt + lane_prefix(m);
          if (pos < kCandCap) {
            sh.d2[pos] = d2;
            sh.pk[pos] = pk;
          }
        }
        cnt += __popcll(m);
      }
    }
    __builtin_amdgcn_wave_barrier();
    if (cnt >= k && cnt <= kCandCap) break;
    if (cnt < k) {
      r_lo = R;
      double f = cnt > 0 ? sqrt((1.5 * k) / cnt) : 2.0;
      if (f < 1.25) f = 1.25;
      if (f > 4.0) f = 4.0;
      R = R * f;
      if (r_hi > 0 && R >= r_hi) R = sqrt(r_lo * r_hi);
      if (R > rcap) R = rcap;
    } else {
      r_hi = R;
      double f = sqrt((0.5 * (k + kCandCap)) / cnt);
      if (f > 0.9) f = 0.9;
      R = R * f;
      if (R <= r_lo) R = sqrt(r_lo * r_hi);
    }
    if (attempt > 60 || (cnt < k && r_lo >= rcap)) {
      if (lane == 0) ++nfail;
      break;
    }
  }
  if (attempt > 0 && lane == 0) ++nretry;
  SearchOut out;
  out.tau = 0;
  out.facc = 0;
  if (cnt < k || cnt > kCandCap) return out;
  // k-th smallest squared distance: ballot quickselect
  constexpr int NS = kCandCap / 64;
  double v[NS];
  uint32_t pkr[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int idx = s * 64 + lane;
    v[s] = idx < cnt ? sh.d2[idx] : INFINITY;
    pkr[s] = idx < cnt ? sh.pk[idx] : 0u;
  }
  double lo = -1.0, hi = INFINITY, tau = 0;
  int c_lt = 0, c_le = 0;
  for (;;) {
    int slot = -1, src = 0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if (s * 64 >= cnt) break;
      const unsigned long long b = ballot(v[s] > lo && v[s] < hi);
      if (slot < 0 && b) {
        slot = s;
        src = __builtin_ctzll(b);
      }
    }
    double pv = 0;
#pragma unroll
    for (int s = 0; s < NS; ++s)
      if (s == slot) pv = readlane_d(v[s], src);
    c_lt = 0;
    c_le = 0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if (s * 64 >= cnt) break;  // uniform: most searches fill one or two rounds
      c_lt += __popcll(ballot(v[s] < pv));
      c_le += __popcll(ballot(v[s] <= pv));
    }
    if (c_lt < k && k <= c_le) {
      tau = pv;
      break;
    }
    if (k <= c_lt) hi = pv; else lo = pv;
  }
  // ties at tau keep the smallest (ID, image)
  bool tsel[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) tsel[s] = false;
  if (c_le > k) {
    if (lane == 0) ++nties;
    uint64_t key2[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int idx = s * 64 + lane;
      key2[s] = ~0ull;
      if (idx < cnt && v[s] == tau)
        key2[s] = ((uint64_t)ID[pkr[s] >> 4] << 4) | img_order(pkr[s] & 15u);
    }
    for (int r = 0; r < k - c_lt; ++r) {
      uint64_t mn = ~0ull;
#pragma unroll
      for (int s = 0; s < NS; ++s) mn = key2[s] < mn ? key2[s] : mn;
      for (int o = 32; o > 0; o >>= 1) {
        const uint64_t other = __shfl_xor(mn, o, 64);
        mn = other < mn ? other : mn;
      }
#pragma unroll
      for (int s = 0; s < NS; ++s)
        if (key2[s] == mn) {
          tsel[s] = true;
          key2[s] = ~0ull;
        }
    }
  }
  const double h = sqrt(tau);
  const int kern = S->kernel;
  // The kernel sum is in FP64 in every form: these searches are few and wait
  // on loads, and their rows include the ill-conditioned ones (every neighbour
  // near q = 1, where F(q) = (1 - q)^3 / 3 amplifies a rounding of q by
  // 3 q / (1 - q)).
  double facc = 0.0;
  const double hinv = 1.0 / h;
  int emitted = 0;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int idx = s * 64 + lane;
    const bool sel = idx < cnt && (v[s] < tau || (v[s] == tau && (c_le == k || tsel[s])));
    const unsigned long long m = ballot(sel);
    if (sel) {
      const int pos = emitted + lane_prefix(m);
      if constexpr (!BITWISE) {
        row[pos] = pkr[s];
        facc += kern == kWendland ? WendlandF::F64(sqrt_over(v[s], h, hinv))
                                  : CubicF::F64(sqrt_over(v[s], h, hinv));
      } else {
        sh.sd2[pos] = v[s];
        sh.spk[pos] = pkr[s];
      }
    }
    emitted += __popcll(m);
  }
  if constexpr (!BITWISE) {
    out.facc = group_sum(facc, 64);
  } else {
    __builtin_amdgcn_wave_barrier();
    double dv = lane < k ? sh.sd2[lane] : -1.0;
    uint32_t pv = lane < k ? sh.spk[lane] : 0u;
    uint32_t iv = lane < k ? ID[pv >> 4] : 0u;
    // bitonic sort, descending by (d2, ID, image)
    for (int size = 2; size <= 64; size <<= 1) {
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
        const double od = __shfl_xor(dv, stride, 64);
        const uint32_t op = __shfl_xor(pv, stride, 64);
        const uint32_t oi = __shfl_xor(iv, stride, 64);
        const bool other_greater =
            od > dv || (od == dv && (oi > iv || (oi == iv && img_order(op & 15u) > img_order(pv & 15u))));
        const bool lower = (lane & stride) == 0;
        const bool desc = (lane & size) == 0;
        const bool take = (lower == desc) ? other_greater : !other_greater;
        if (take && (od != dv || oi != iv || op != pv)) {
          dv = od;
          pv = op;
          iv = oi;
        }
      }
    }
    if (lane < k) {
      row[lane] = pv;
      sh.fterm[lane] = kern_F(kern, sqrt(dv) / h);
    }
    __builtin_amdgcn_wave_barrier();
    double acc = 0.0;
    for (int n = 0; n < k; ++n) acc += sh.fterm[n];
    out.facc = acc;
  }
  out.tau = tau;
  __builtin_amdgcn_wave_barrier();
  return out;
}

// Predicted energy and velocity of a query: read where they are used (the
// walk, whose registers are full before), or ahead of the search.
struct PredArr {
  const double *__restrict__ e, *__restrict__ x, *__restrict__ y;
  int64_t t;
  __device__ double ep() const { return e[t]; }
  __device__ double vpx() const { return x[t]; }
  __device__ double vpy() const { return y[t]; }
};
struct PredVal {
  double e, x, y;
  __device__ double ep() const { return e; }
  __device__ double vpx() const { return x; }
  __device__ double vpy() const { return y; }
};

// Density, sound speed, h and the force record of query t.
template <bool FP32C, typename Pred>
__device__ inline void write_result(const SimDev* S, int64_t t, double xq, double yq, double tau,
                                    double facc, const Pred& p, double* __restrict__ H,
                                    double* __restrict__ RHO, double* __restrict__ C,
                                    void* __restrict__ recp) {
  const double h = sqrt(tau);
  const double rho = S->fpref * S->mass * facc / (h * h);
  const double c = sqrt(S->cfac * p.ep());
  H[t] = h;
  RHO[t] = rho;
  C[t] = c;
  const double B = c * c / (S->gamma * rho);
  if constexpr (FP32C) {
    RecF r;
    r.ux = (uint32_t)(int64_t)floor((xq - S->x0) * (4294967296.0 / S->lx));
    r.uy = (uint32_t)(int64_t)floor((yq - S->y0) * (4294967296.0 / S->ly));
    r.vpx = (float)p.vpx();
    r.vpy = (float)p.vpy();
    r.rho = (float)(0.5 * rho);
    r.c = (float)(0.5 * c);
    r.h = (float)(0.5 * h);
    r.B = (float)B;
    ((RecF*)recp)[t] = r;
  } else {
    RecD r;
    r.x = xq;
    r.y = yq;
    r.vpx = p.vpx();
    r.vpy = p.vpy();
    r.rho = 0.5 * rho;
    r.c = 0.5 * c;
    r.h = 0.5 * h;
    r.B = B;
    ((RecD*)recp)[t] = r;
  }
}

// FP32C: may the displacements of a query with support h come from the 32-bit
// fixed-point positions (units of L / 2^32)?  Their 32-bit difference is the
// minimum image while every neighbour lies within half a box (h < 0.45 L).
// The displacement is centred on the query's exact position (centred_step):
// what is left is the neighbour's flooring, uniform within half a step and
// independent between neighbours, below 2^-20 h per component while
// h > 2^-13 L.  Emulated on clusters reaching that threshold the density
// stays within 2e-6 of FP64.  Otherwise the FP64 positions give the
// displacement.
__device__ inline bool fixed_point_ok(double h, double lx, double ly) {
  const double lmin = lx < ly ? lx : ly;
  return h < 0.45 * lmin && h > 0x1p-13 * lmin;
}

// Offset, in fixed-point steps, from a particle's exact position to the
// centre of its fixed-point step (1/2 minus the fraction the floor dropped):
// the displacement to a neighbour j is (u_j - u_i) + this, whose error is
// j's flooring alone, centred on zero.
__device__ inline float centred_step(double x, double x0, double l) {
  const double f = (x - x0) * (4294967296.0 / l);
  return (float)(0.5 - (f - floor(f)));
}

// Search radius of a query without an h: local density from the occupancy of
// the query's cell at a level holding a few particles.
__device__ inline double local_radius(const SimDev* S, const uint32_t* __restrict__ cstart,
                                      double xq, double yq) {
  const CellIdx ci = cell_of(S, xq, yq);
  const int64_t fx = ci.ux - (floordiv_pow2(ci.ux, S->lg) << S->lg);
  const int64_t fy = ci.uy - (floordiv_pow2(ci.uy, S->lg) << S->lg);
  int c = S->lg - 1 > 0 ? S->lg - 1 : 0;
  for (;; --c) {
    const int sh = S->lg - c;
    uint32_t a, b;
    cell_range(S, cstart, c, (uint32_t)(fx >> sh), (uint32_t)(fy >> sh), a, b);
    const double area = (S->lx / (double)(1LL << c)) * (S->ly / (double)(1LL << c));
    if (b - a >= 8 || c == 0) {
      const double dens = (double)(b - a > 0 ? b - a : 1) / area;
      const double r = sqrt(1.3 * S->k / (M_PI * dens));
      return r < S->r_init * 4 ? r : S->r_init * 4;
    }
  }
}

// Block-compensated FP32 sum: the terms of one round (4 or 8 neighbours)
// add up plainly, and each round's partial joins the running sum through a
// Kahan step.  Besides the compensated sum's own error this adds at most
// (B - 1) 2^-24 of the sum of |terms| of a block of B, against four
// operations per term for a Kahan step per term.
struct BlockKahan {
  float s = 0.f, c = 0.f, p = 0.f;
  __device__ void add(float t) { p += t; }
  __device__ void add_mul(float a, float b) { p = __builtin_fmaf(a, b, p); }
  __device__ void flush() {
    const float y = p - c;
    const float tt = s + y;
    c = (tt - s) - y;
    s = tt;
    p = 0.f;
  }
  __device__ double value() const { return (double)s - (double)c; }
};

// ---- the bracketed walk ----
constexpr int kGrp = 16;         // queries searched together (a group)
constexpr int kWalkCand = 240;   // candidates of a group's box, held in LDS
constexpr int kWalkRounds = 4;   // the same in rounds of 64 (one candidate per lane)
constexpr int kWalkRaw = 1024;   // candidates of the box's cells

// Scratch of a walk wave: 10 KiB, so that sixteen waves share a CU's LDS (four
// per SIMD, which its registers allow without spilling).
struct WalkShared {
  double2 xy[kWalkCand];        // candidates inside the group's box
  uint32_t pk[kWalkCand];       // their packed entries
  uint8_t row[kGrp][68];        // per query: candidate slots of its neighbours
  uint8_t annl[kGrp][kAnn];     // per query: candidate slots in its annulus
  union {
    struct {
      uint8_t mark[kWalkRaw];   // first candidate of cell c (lane c): c + 1
      uint2 piece[64];          // per cell: sorted slot minus candidate number, image tile
    } s;
    double ad[kAnn][kGrp];      // annulus squared distances (entry, query)
    struct {                    // one row, bitwise form
      double d2[kMaxK];
      double term[kMaxK];       // kernel values in row order
      uint32_t id[kMaxK];
      uint8_t at[kMaxK];        // lane whose entry took each place
    } b;
  } u;
  // per query of the wave: x, y, then Rlo^2, Rhi^2 until its group is
  // searched, and after it tau and the kernel sum; tau < 0: not found (kMiss*)
  double4 q[64];
};
constexpr double kThinSum = 2e-3;  // FP32C kernel sums below it are redone in FP64
constexpr double kMissWide = -1.0, kMissLo = -2.0, kMissAnn = -3.0, kMissHi = -4.0;
constexpr double kSeeded = -5.0;
// The exact search starts from 1.1 times a query's last h.  One that the walk found
// too few neighbours for, within up to 1.1 h already, starts from the radius
// that would hold 1.2 k at the density inside that (its h is set so that 1.1 h
// is that radius): its first attempt had to fail, 4,700 particles of a tube took
// 15.1 us in the exact search against 11.8, 77,777 11.5 against 10.6.  For k, 1.2 k,
// 1.5 k and 2 k, as timed apart: the tube 16.8, 14.2, 15.0 and 16.2 us, 77,777 14.5,
// 12.4, 12.7 and 13.2, 262,144 16.7, 14.2, 14.5 and 16.1, 1M 26.7, 24.2, 24.9 and 26.8.
constexpr double kFirstReach = 1.1, kMissReach = 1.2;
static_assert(sizeof(WalkShared) == 10240, "sixteen waves per CU");

typedef __attribute__((address_space(3))) uint8_t LdsByte;
__device__ inline uint32_t lds_addr(const uint8_t* p) {
  return (uint32_t)(uintptr_t)(LdsByte*)p;
}
__device__ inline LdsByte* lds_u8(uint32_t a) { return (LdsByte*)(uintptr_t)a; }

// One wave's LDS operations complete in order; this keeps the compiler from
// moving them across.
__device__ inline void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Lane moves within rows of 16 (and, row by row, into the rows after): lanes
// without a source read 0.
template <int CTRL, int ROWS = 0xf>
__device__ inline uint32_t dpp(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, true);
}
// minimum over each row of 16 lanes (every lane ends with it), of values that
// are no NaN
__device__ inline float row_min(float v) {
  auto step = [](float a, uint32_t b) { return __builtin_amdgcn_fmed3f(a, __uint_as_float(b), -INFINITY); };
  v = step(v, dpp<0xB1>(__float_as_uint(v)));   // lane ^ 1
  v = step(v, dpp<0x4E>(__float_as_uint(v)));   // lane ^ 2
  v = step(v, dpp<0x141>(__float_as_uint(v)));  // mirror of 8: the other quad
  return step(v, dpp<0x140>(__float_as_uint(v)));
}
// inclusive scans over the wave: row shifts, then the last lane of each row
// into the rows after it
__device__ inline uint32_t scan_add(uint32_t v) {
  v += dpp<0x111>(v);
  v += dpp<0x112>(v);
  v += dpp<0x114>(v);
  v += dpp<0x118>(v);
  v += dpp<0x142, 0xa>(v);
  v += dpp<0x143, 0xc>(v);
  return v;
}
__device__ inline uint32_t scan_max(uint32_t v) {
  auto mx = [](uint32_t a, uint32_t b) { return a > b ? a : b; };
  v = mx(v, dpp<0x111>(v));
  v = mx(v, dpp<0x112>(v));
  v = mx(v, dpp<0x114>(v));
  v = mx(v, dpp<0x118>(v));
  v = mx(v, dpp<0x142, 0xa>(v));
  v = mx(v, dpp<0x143, 0xc>(v));
  return v;
}

// Squared distance of the candidate in slot `slot` from (xq, yq), in the
// reference's order: ((p_i + o) - p_j)^2.  IMG: some candidate of the group
// is seen through an image (p_i + 0 is p_i).
template <bool IMG>
__device__ inline double slot_d2(const WalkShared& sh, uint32_t slot, double xq, double yq,
                                 double lx, double ly) {
  const double2 pj = sh.xy[slot];
  double ax = xq, ay = yq;
  if constexpr (IMG) {
    const uint32_t im = sh.pk[slot] & 15u;
    ax = xq + (double)img_ix(im) * lx;
    ay = yq + (double)img_iy(im) * ly;
  }
  const double ex = ax - pj.x, ey = ay - pj.y;
  return ex * ex + ey * ey;
}

// Classifies the group's candidates (lane = candidate, NR rounds of 64 in
// registers) for the queries of `gmask` one after the other: the query's
// data is the same in every lane, so a comparison's result is the mask of
// its certain neighbours (inside Rlo) or of its reach (up to Rhi), and a
// candidate's place in the query's list is a prefix count of that mask.  No
// lane waits for another's list, whatever the lists' lengths.  Lanes ql == i
// of every row return query i's counts.  IMG: some candidate is seen through
// an image.
template <int NR, bool IMG>
__device__ inline void classify(WalkShared& sh, const double4* gq, int ncand, uint32_t gmask, uint32_t t0, int k,
                                double lx, double ly, int lane, int& c_lo, int& c_an) {
  double x[NR], y[NR], ox[NR], oy[NR];
  uint32_t j[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int s = r * 64 + lane;
    const bool in = s < ncand;
    const double2 p = sh.xy[in ? s : 0];
    const uint32_t pk = sh.pk[in ? s : 0];
    x[r] = in ? p.x : NAN;  // compares false with everything
    y[r] = p.y;
    j[r] = pk >> 4;
    if constexpr (IMG) {
      ox[r] = (double)img_ix(pk & 15u) * lx;
      oy[r] = (double)img_iy(pk & 15u) * ly;
    }
  }
  const int ql = lane & (kGrp - 1);
  // LDS addresses as numbers: a list's base folds into its prefix count
  const uint32_t rows = lds_addr(&sh.row[0][0]), anns = lds_addr(&sh.annl[0][0]);
  for (uint32_t rem = gmask; rem; rem &= rem - 1u) {
    const int i = __builtin_ctz(rem);
    const double4 q = gq[i];
    const uint32_t ti = t0 + (uint32_t)i;
    unsigned long long mc[NR], ma[NR];
    int nc = 0, na = 0;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      double ex, ey;
      if constexpr (IMG) {
        ex = (q.x + ox[r]) - x[r];
        ey = (q.y + oy[r]) - y[r];
      } else {
        ex = q.x - x[r];
        ey = q.y - y[r];
      }
      const double d2 = ex * ex + ey * ey;
      // one comparison per ballot: combined on the scalar unit.  Every image
      // of the query itself is excluded.
      const unsigned long long other = ballot(j[r] != ti);
      const unsigned long long in = ballot(d2 < q.z) & other;
      ma[r] = ballot(d2 <= q.w) & other & ~in;
      mc[r] = in;
      nc += __popcll(mc[r]);
      na += __popcll(ma[r]);
    }
    if (nc < k && na <= kAnn && nc + na >= k) {
      uint32_t at = rows + (uint32_t)i * 68u;
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const uint32_t pos = __builtin_amdgcn_mbcnt_hi((uint32_t)(mc[r] >> 32),
                                 __builtin_amdgcn_mbcnt_lo((uint32_t)mc[r], at));
        if (__builtin_amdgcn_inverse_ballot_w64(mc[r])) *lds_u8(pos) = (uint8_t)(r * 64 + lane);
        at += (uint32_t)__popcll(mc[r]);
      }
      at = anns + (uint32_t)i * kAnn;
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const uint32_t pos = __builtin_amdgcn_mbcnt_hi((uint32_t)(ma[r] >> 32),
                                 __builtin_amdgcn_mbcnt_lo((uint32_t)ma[r], at));
        if (__builtin_amdgcn_inverse_ballot_w64(ma[r])) *lds_u8(pos) = (uint8_t)(r * 64 + lane);
        at += (uint32_t)__popcll(ma[r]);
      }
    }
    c_lo = ql == i ? nc : c_lo;
    c_an = ql == i ? na : c_an;
  }
}

// The lists of the queries of `todo`, whose annulus holds more than kAnn, by
// narrower brackets: the bracket of the squared distance is halved until it does
// not.  (Equal distances are never parted: the exact search takes more than kAnn of
// them.)  Few queries, but at k = 64 nine of ten of those that the exact search
// took, 4M clustered 22,900 per pass -> 3,400: that search 104 -> 43 us, and 34 ->
// 20 at 1M, while the walk's time stays (halving in classify's own loop, whose
// registers are full, made it 5 % slower).  Queries with k certain neighbours are
// left to the exact search: they are few in every size, and where launches are
// short the wave that stays for one costs more than the search (2,200 particles 46.2
// -> 46.9 us per step).
template <bool IMG>
__device__ inline void tighten(WalkShared& sh, const double4* gq, int ncand, uint32_t todo,
                               uint32_t t0, int k, double lx, double ly, int lane, int& c_lo,
                               int& c_an) {
  constexpr int NR = (kWalkCand + 63) / 64;
  for (uint32_t rem = todo; rem; rem &= rem - 1u) {
    const int i = __builtin_ctz(rem);
    const double4 q = gq[i];
    const uint32_t ti = t0 + (uint32_t)i;
    double d2[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int s = r * 64 + lane;
      const bool in = s < ncand && (sh.pk[s] >> 4) != ti;
      d2[r] = in ? slot_d2<IMG>(sh, (uint32_t)s, q.x, q.y, lx, ly) : INFINITY;
    }
    auto below = [&](double v) {
      int n = 0;
#pragma unroll
      for (int r = 0; r < NR; ++r) n += __popcll(ballot(d2[r] < v));
      return n;
    };
    // nlo of them lie below lo, fewer than k; nhi below hi, k or more
    double lo = q.z, hi = q.w;
    int nlo = below(lo), nhi = k + kAnn;
    for (int it = 0; it < 24 && nhi - nlo > kAnn; ++it) {
      const double mid = 0.5 * (lo + hi);
      const int n = below(mid);
      if (n >= k) {
        hi = mid;
        nhi = n;
      } else {
        lo = mid;
        nlo = n;
      }
    }
    int nc = 0, na = 0;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const unsigned long long mc = ballot(d2[r] < lo), ma = ballot(d2[r] < hi) & ~mc;
      // (past kAnn the counts say so and the lists are not read)
      if (d2[r] < lo) sh.row[i][nc + lane_prefix(mc)] = (uint8_t)(r * 64 + lane);
      else if (d2[r] < hi && na + lane_prefix(ma) < kAnn)
        sh.annl[i][na + lane_prefix(ma)] = (uint8_t)(r * 64 + lane);
      nc += __popcll(mc);
      na += __popcll(ma);
    }
    const int ql = lane & (kGrp - 1);
    c_lo = ql == i ? nc : c_lo;
    c_an = ql == i ? na : c_an;
  }
}

// The k-th distance of a group's queries, and their rows completed: lane
// (ql, part) holds four of query ql's annulus entries (e = 4 part + i).  The
// k - c_lo smallest by (d2, entry) are taken; an exact tie at the k-th
// distance is resolved by (ID, image order).  Returns tau in the four lanes
// of each query, and counts the queries with a tie.
template <bool IMG>
__device__ inline double select_annulus(WalkShared& sh, bool ok, int k, int c_lo, int c_an,
                                        double xq, double yq, double lx, double ly, int ql,
                                        int part, const uint32_t* __restrict__ ID,
                                        unsigned& nties) {
  const int need = k - c_lo;
  uint32_t slot[4];
  double ad[4], nx[4];
  {
    const uint32_t ids = *(const uint32_t*)&sh.annl[ql][4 * part];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool in = ok && 4 * part + i < c_an;
      slot[i] = in ? (ids >> (8 * i)) & 255u : 0u;
      const double d2 = slot_d2<IMG>(sh, slot[i], xq, yq, lx, ly);
      ad[i] = in ? d2 : INFINITY;
      // the next double: x < next(d2) is x <= d2
      nx[i] = __longlong_as_double(__double_as_longlong(ad[i]) + 1);
      sh.u.ad[4 * part + i][ql] = ad[i];
    }
  }
  wave_fence();
  // entries before each in the order (d2, entry): those of earlier quarters
  // up to and including its distance, the others below it; ties inside the
  // quarter by place
  int before[4] = {0, 0, 0, 0};
  const int most = ballot(ok && c_an > 12) ? 4 : ballot(ok && c_an > 8) ? 3
                 : ballot(ok && c_an > 4)  ? 2 : 1;
  for (int f4 = 0; f4 < most; ++f4) {
    const bool earlier = f4 < part;
    const double th0 = earlier ? nx[0] : ad[0], th1 = earlier ? nx[1] : ad[1];
    const double th2 = earlier ? nx[2] : ad[2], th3 = earlier ? nx[3] : ad[3];
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const double v = sh.u.ad[4 * f4 + f][ql];
      before[0] += v < th0;
      before[1] += v < th1;
      before[2] += v < th2;
      before[3] += v < th3;
    }
  }
#pragma unroll
  for (int i = 1; i < 4; ++i)
#pragma unroll
    for (int f = 0; f < i; ++f) before[i] += ad[f] == ad[i];
  double tau = -1.0;
  bool sel[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    sel[i] = ok && 4 * part + i < c_an && before[i] < need;
    if (sel[i]) sh.row[ql][c_lo + before[i]] = (uint8_t)slot[i];
    tau = sel[i] && ad[i] > tau ? ad[i] : tau;
  }
  {
    const double o1 = __shfl_xor(tau, 16, 64);
    tau = o1 > tau ? o1 : tau;
    const double o2 = __shfl_xor(tau, 32, 64);
    tau = o2 > tau ? o2 : tau;
  }
  // an entry left out at exactly the k-th distance (the others left out lie
  // beyond it)
  bool tie = false;
#pragma unroll
  for (int i = 0; i < 4; ++i) tie = tie || (ok && 4 * part + i < c_an && !sel[i] && ad[i] == tau);
  const unsigned long long tied = ballot(tie);
  if (tied) {
    const uint32_t tq = (uint32_t)(tied | tied >> 16 | tied >> 32 | tied >> 48) & 0xFFFFu;
    nties += __builtin_popcount(tq);
    wave_fence();
    if (part == 0 && ((tq >> ql) & 1u)) {
      int below = 0;
      for (int e = 0; e < c_an; ++e) below += sh.u.ad[e][ql] < tau ? 1 : 0;
      // the slots after the entries below tau take the tied entries with the
      // smallest (ID, image order)
      uint64_t prev = 0;
      bool first = true;
      for (int p = c_lo + below; p < k; ++p) {
        uint64_t best = ~0ull;
        uint32_t bslot = 0;
        for (int e = 0; e < c_an; ++e) {
          if (sh.u.ad[e][ql] != tau) continue;
          const uint32_t sl = sh.annl[ql][e], pk = sh.pk[sl];
          const uint64_t key = ((uint64_t)ID[pk >> 4] << 4) | img_order(pk & 15u);
          if ((first || key > prev) && key < best) {
            best = key;
            bslot = sl;
          }
        }
        sh.row[ql][p] = (uint8_t)bslot;
        prev = best;
        first = false;
      }
    }
  }
  wave_fence();
  return tau;
}

// The kernel sum over the k neighbours of a group's queries, and their rows'
// entries to memory: lane (ql, part) takes every fourth chunk of four
// entries of query ql's row, so that the 16 queries' chunks leave as 256
// contiguous bytes.  Returns the sum in the four lanes of each query.
template <bool FP32C, bool IMG, typename KT>
__device__ inline double row_density(const WalkShared& sh, NbrRow row, int k, double tau, double xq,
                                     double yq, double lx, double ly, int ql, int part) {
  double acc = 0.0;
  BlockKahan fk;
  // FP32C: q^2 = d^2 / tau formed in FP64 before the FP32 square root: a
  // rounded 1 / h shared by every term would move all q together, and a
  // particle whose neighbours all sit near q = 1 would lose 1e-5 of its density
  const double itau = FP32C ? 1.0 / tau : 0.0;
  const double h = FP32C ? 0.0 : sqrt(tau), hinv = FP32C ? 0.0 : rcp64(h);
  auto visit = [&](int ch, int n) {
    const uint32_t ids = *(const uint32_t*)&sh.row[ql][4 * ch];
    uint32_t pk[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool in = i < n;
      const uint32_t sl = in ? (ids >> (8 * i)) & 255u : 0u;
      pk[i] = sh.pk[sl];
      const double d2 = slot_d2<IMG>(sh, sl, xq, yq, lx, ly);
      if constexpr (FP32C) {
        // the k-th neighbour's q may round to a few ulp past 1, where F is of
        // order ulp^3 (no clamp needed)
        const float f = KT::F(__builtin_amdgcn_sqrtf((float)(d2 * itau)));
        fk.add(in ? f : 0.f);
      } else {
        const double f = KT::F64(sqrt_over(d2, h, hinv));
        acc += in ? f : 0.0;
      }
    }
    if constexpr (FP32C) fk.flush();
    *row.chunk(ch) = u32x4{pk[0], pk[1], pk[2], pk[3]};
  };
  int ch = part;
  for (; 4 * ch + 4 <= k; ch += 4) visit(ch, 4);
  if (4 * ch < k) visit(ch, k - 4 * ch);
  if constexpr (FP32C) acc = fk.value();
  acc += __shfl_xor(acc, 16, 64);
  acc += __shfl_xor(acc, 32, 64);
  return acc;
}

// Bitwise form: the row of one query at a time, lane = entry.  Each lane counts
// the entries farther than its own; where two claim a place (equal distances)
// the whole order (d2, ID, image) counts.  The row leaves in that order, and its
// kernel values are added farthest first, as the reference's queue is read
// (sim/sph.go:313-320).  `todo`: the queries of the group; lanes ql == i of every
// row return query i's sum.  About 400 vector instructions per query, against
// some 2,300 in the exact search that every query of this form took before
// (30,011 clustered, k = 32: 773 us, now 83 us and 16 us for the misses).
template <bool IMG>
__device__ inline double rows_bitwise(WalkShared& sh, const double4* gq, uint32_t todo, uint32_t t0,
                                      int k, int kern, double tau, double lx, double ly, int lane,
                                      const uint32_t* __restrict__ ID, uint32_t* __restrict__ nbr,
                                      int kstride) {
  const int ql = lane & (kGrp - 1);
  double facc = 0.0;
  for (uint32_t rem = todo; rem; rem &= rem - 1u) {
    const int i = __builtin_ctz(rem);
    const double xq = gq[i].x, yq = gq[i].y;
    const double h = sqrt(readlane_d(tau, i));
    const bool in = lane < k;
    const uint32_t slot = in ? sh.row[i][lane] : 0u;
    const uint32_t pk = sh.pk[slot];
    const double d2 = in ? slot_d2<IMG>(sh, slot, xq, yq, lx, ly) : -1.0;
    const uint32_t id = ID[pk >> 4];
    wave_fence();
    sh.u.b.d2[lane] = d2;
    sh.u.b.id[lane] = id;
    wave_fence();
    int at = 0;
    for (int m = 0; m < k; ++m) at += sh.u.b.d2[m] > d2;
    if (in) sh.u.b.at[at] = (uint8_t)lane;
    wave_fence();
    if (ballot(in && sh.u.b.at[at] != lane)) {
      at = 0;
      for (int m = 0; m < k; ++m) {
        const double v = sh.u.b.d2[m];
        const uint32_t w = sh.u.b.id[m];
        const uint32_t im = img_order(sh.pk[sh.row[i][m]] & 15u);
        at += v > d2 || (v == d2 && (w > id || (w == id && im > img_order(pk & 15u))));
      }
    }
    if (in) {
      sh.u.b.term[at] = kern_F(kern, sqrt(d2) / h);
      nbr_row(nbr, (int64_t)t0 + i, kstride)[at] = pk;
    }
    wave_fence();
    double acc = 0.0;
    for (int n = 0; n < k; ++n) acc += sh.u.b.term[n];
    facc = ql == i ? acc : facc;
  }
  wave_fence();
  return facc;
}

// Distance to the k-th neighbour of each query of `gmask` among the group's
// staged candidates, by bisection of the squared distance (lane = candidate,
// FP32; to within 1 %, a fraction of the walk's bracket).  gq[i].w is the radius
// R that the group's box was made for and becomes the answer: up to R it is the
// distance, beyond it (candidates outside the box are missing) it is negative,
// an upper limit to search again within; gq[i].z becomes kSeeded.
template <bool IMG>
__device__ inline void seed_radii(WalkShared& sh, double4* gq, int ncand, uint32_t gmask,
                                  uint32_t t0, int k, double lx, double ly, int lane) {
  constexpr int NR = (kWalkCand + 63) / 64;
  for (uint32_t rem = gmask; rem; rem &= rem - 1u) {
    const int i = __builtin_ctz(rem);
    const double4 q = gq[i];
    const uint32_t ti = t0 + (uint32_t)i;
    float d2[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int s = r * 64 + lane;
      const bool in = s < ncand && (sh.pk[s] >> 4) != ti;
      d2[r] = in ? (float)slot_d2<IMG>(sh, (uint32_t)s, q.x, q.y, lx, ly) : INFINITY;
    }
    auto count = [&](float v) {
      int n = 0;
#pragma unroll
      for (int r = 0; r < NR; ++r) n += __popcll(ballot(d2[r] <= v));
      return n;
    };
    const float R2 = (float)(q.w * q.w);
    const bool inside = count(R2) >= k;
    float lo = inside ? 0.f : R2, hi = inside ? R2 : 16.f * R2;
    double h = -2.0 * q.w;
    if (inside || count(hi) >= k) {
      for (int it = 0; it < 24 && hi - lo > 0.02f * hi; ++it) {
        const float mid = 0.5f * (lo + hi);
        if (count(mid) >= k) hi = mid; else lo = mid;
      }
      h = sqrt(0.5 * ((double)lo + (double)hi));
      if (!inside) h = -1.02 * h;
    }
    if (lane == 0) {
      gq[i].z = kSeeded;
      gq[i].w = h;
    }
  }
  wave_fence();
}

// kNN + density + sound speed + force record of the queries that have an h
// from the last pass.  A wave takes up to 64 consecutive (Hilbert-ordered)
// queries, lane = query, and searches groups of 16 of them one after the
// other:
//
//   box       the box around the group's search circles (radius
//             h_prev (1 + delta)), in cells of the finest grid; the cells of
//             the coarsest level that covers it with at most nsub x nsub
//             cells are looked up one per lane
//   stage     the cells' particles, 64 at a time, filtered against the box
//             and packed into LDS (position, packed entry)
//   classify  lane = candidate: per query, certain neighbours (nearer than
//             h_prev (1 - delta)) and the annulus up to h_prev (1 + delta)
//   select    lane = (query, quarter of its annulus): exact distances, the
//             k-th distance
//   density   lane = (query, every fourth chunk of its row): the kernel sum
//             from the LDS positions, the row to memory (bitwise form: a row at
//             a time, in the reference's order)
//
// A group whose cells hold more than 24 * split candidates (576: a box of 16
// queries at k = 64 usually holds 250 in its cells; staging a few hundred more
// costs less than two half groups: 4M 1.17 -> 1.12 ms against 384), or whose box
// more than kWalkCand, is halved (cell order can put two distant regions in one
// group), with kWalkRaw in place of 24 * split from then on.  Groups of 4 that
// are still too wide go to the exact search, as queries without an h and
// queries whose bracket misses do: its waves take one such query each, side by
// side, where halving down to single queries kept one wave busy (30,000
// clustered: 196 against 136 us per step).
//
// What bounds it: vector issue, 75 % of all issue slots at 4M clustered, k = 64
// (124 vector instructions per query; 1.31 GB written, 0.29 GB read).
// One query's candidates side by side in the lanes need no per-query lists and
// no lane waits for the longest of 64 lists, and a group of 16 queries is a
// short chain of loads, so small launches finish early.  Against the walk with
// a query per lane and its separate selection and density kernel that this
// replaced: 4M FP32C 1.40 -> 1.12 ms, 1M FP64 0.45 -> 0.33 ms, 77,777 at k = 19
// 108 -> 31 us, 2,200 at k = 32 55 -> 15 us.  One wave per block: a wave that
// ends frees its LDS at once (1.54 -> 1.39 ms); 10 KiB per wave and four waves
// per SIMD without a spilled register, where five spilled 40 (1.39 -> 1.17 ms).
//
// SEED: finds an h for the queries that have none (a simulation's first pass)
// in place of their neighbours, from the same staging: `seed` 1 for the queries
// without an h (2: for all), searching within local_radius, and 0 for those that
// the first search left with a limit (negative).  The walk then takes them like
// any other; before, all of them went to the exact search, a wave each.  kNN of
// a first pass, before and now: 2,200 particles at k = 32 586 -> 69 us, 100,000 in
// an open box 853 -> 138, 30,011 clustered at k = 64 in the bitwise form 980 -> 300;
// a first call of 20 steps at 4M clustered 73.3 -> 60.0 ms.
template <bool FP32C, bool BITWISE, bool SEED>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void k_knn(
    const Item* __restrict__ items, int nitems, const SimDev* __restrict__ sims,
    const double2* __restrict__ XY, const uint8_t* __restrict__ WR,
    const uint32_t* __restrict__ cstart, double* __restrict__ H, const double* __restrict__ EP,
    const double* __restrict__ VPX, const double* __restrict__ VPY,
    const uint32_t* __restrict__ ID, uint32_t* __restrict__ nbr, int kstride,
    double* __restrict__ RHO, double* __restrict__ C, void* __restrict__ recp,
    KnnStats* __restrict__ stats, uint2* __restrict__ retry, uint32_t* __restrict__ retry_count,
    WalkKnobs kn, uint32_t* __restrict__ walk_miss, int wpi, int seed) {
  __shared__ WalkShared sh;
  const int lane0 = threadIdx.x;
  // wpi blocks (of one wave) per item (4, 8 or 16), each taking 256 / wpi
  // queries
  const int blk = xcd_item(nitems * wpi);
  const int item_idx = blk / wpi;
  const Item it = items[item_idx];
  const int per = kItem / wpi;
  const int w0 = (blk - item_idx * wpi) * per;
  if (w0 >= it.count) return;
  const int nq = it.count - w0 < per ? it.count - w0 : per;
  const SimDev* S = sims + it.sim;
  const int k = S->k;
  const double lx = S->lx, ly = S->ly;
  const int lg = S->lg;
  const int raw_cap = kn.split * 24 < kWalkRaw ? kn.split * 24 : kWalkRaw;
  // ---- this lane's own query ----
  const bool valid = lane0 < nq;
  const uint32_t tw = (uint32_t)(it.first + w0);
  const uint32_t t = tw + (valid ? lane0 : 0);
  unsigned long long can;
  const uint32_t wrap = WR[t];
  // the search circle's box in finest cells, widened by 1/64 of a cell (far
  // beyond the rounding to float of at most 6 * 2^13 cells)
  float qx0, qx1, qy0, qy1;
  {
    const double2 pq = XY[t];
    double hp = H[t];
    const double delta = SEED ? 0.0 : S->walk_delta;
    if constexpr (SEED) {
      // every image lies within 3 boxes
      const double rcap = 3.0 * (lx > ly ? lx : ly);
      const bool todo = valid && (seed == 0 ? hp < 0 : seed == 2 || !(hp > 0));
      if (todo) hp = seed ? local_radius(S, cstart, pq.x, pq.y) : -hp;
      if (hp > rcap) hp = rcap;
      can = ballot(todo && hp > 0);
    } else {
      can = ballot(valid && hp > 0);
    }
    const double Rlo = hp * (1 - delta), Rhi = hp * (1 + delta);
    const double Rm = Rhi * (1 + 1e-12) + 1e-15 * (lx + ly);
    const double fx = (pq.x - S->x0) * S->ivx, fy = (pq.y - S->y0) * S->ivy;
    const double rx = Rm * S->ivx + 0.015625, ry = Rm * S->ivy + 0.015625;
    qx0 = (float)(fx - rx);
    qx1 = -(float)(fx + rx);
    qy0 = (float)(fy - ry);
    qy1 = -(float)(fy + ry);
    sh.q[lane0] = make_double4(pq.x, pq.y, Rlo * Rlo, SEED ? Rhi : Rhi * Rhi);
  }
  unsigned nties = 0, ntight = 0;
  const uint32_t table = kHilbertTable.w[lane0];
  const uint32_t* cells = cstart + S->coff;

  for (int g = 0; g * kGrp < nq; ++g) {
    const uint32_t t0 = tw + (uint32_t)(g * kGrp);
    double4* gq = sh.q + g * kGrp;
    uint32_t pending = (uint32_t)(can >> (g * kGrp)) & 0xFFFFu;
    int gsz = kGrp;
    while (pending) {
      // per iteration, so that no address made of it is kept in a register
      // across the groups
      int lane = lane0;
      asm("" : "+v"(lane));
      const int ql = lane & (kGrp - 1), part = lane >> 4;
      const int l0 = __builtin_ctz(pending);
      // of the block of gsz queries that holds l0, those in l0's own image tile:
      // a query that drifted over a periodic boundary stays a box length away
      // from its slot's neighbours until the wrap
      const unsigned long long tile = ballot(wrap == readlane_u(wrap, g * kGrp + l0));
      const uint32_t gmask = pending & (((1u << gsz) - 1u) << (l0 & ~(gsz - 1))) &
                             (uint32_t)(tile >> (g * kGrp));
      const bool grp = (gmask >> ql) & 1u;  // of the row's query ql
      auto row_box = [&](float v) {  // row g holds the group's own lanes
        return __int_as_float(__builtin_amdgcn_readlane(
            __float_as_int(row_min(grp ? v : INFINITY)), g * kGrp));
      };
      const float bx0 = row_box(qx0), bx1 = -row_box(qx1);
      const float by0 = row_box(qy0), by1 = -row_box(qy1);
      // cells of 2^s finest cells: the box spans at most nsub of them per axis
      int s = 0;
      {
        const float m =
            __builtin_fmaxf(bx1 - bx0, by1 - by0) * (kn.nsub == 4 ? 1.f / 2.99f : 1.f / 6.99f);
        if (m > 1.f) s = __builtin_amdgcn_frexp_expf(m);
        s = __builtin_amdgcn_readfirstlane(s < lg ? s : lg);
      }
      const int c = lg - s, nc = 1 << c;
      const float down = __int_as_float((127 - s) << 23);  // 2^-s
      int64_t X0 = (int)floorf(bx0 * down), X1 = (int)floorf(bx1 * down);
      int64_t Y0 = (int)floorf(by0 * down), Y1 = (int)floorf(by1 * down);
      clamp_span(X0, X1, nc, S->open & 1);
      clamp_span(Y0, Y1, nc, S->open & 2);
      uint32_t pa = 0, pb = 0;
      const int xc = (int)X0 + (lane & 7), yc = (int)Y0 + (lane >> 3);
      const int tx = xc >> c, ty = yc >> c;
      const uint32_t hix =
          hilbert_lookup(table, (uint32_t)(xc & (nc - 1)), (uint32_t)(yc & (nc - 1)), c);
      if ((lane & 7) <= (int)(X1 - X0) && (lane >> 3) <= (int)(Y1 - Y0)) {
        const uint32_t* p = cells + ((uint64_t)hix << (2 * s));
        pa = p[0];
        pb = p[1ull << (2 * s)];
      }
      const int len = (int)(pb - pa);
      const int incl = (int)scan_add((uint32_t)len);
      const int nraw = __builtin_amdgcn_readlane(incl, 63);
      int ncand = 0;
      unsigned long long images = 0ull;
      bool fits = nraw <= (gsz == kGrp ? raw_cap : kWalkRaw);
      if (fits) {
        wave_fence();
        ((u32x4*)sh.u.s.mark)[lane] = u32x4{0u, 0u, 0u, 0u};
        wave_fence();
        if (len > 0) {
          sh.u.s.mark[incl - len] = (uint8_t)(lane + 1);
          sh.u.s.piece[lane] = make_uint2(pa - (uint32_t)(incl - len),
                                          (uint32_t)((tx + 2) | ((ty + 2) << 3)));
        }
        wave_fence();
        const double gw = (double)S->gx;
        const double dbx0 = bx0, dbx1 = bx1, dby0 = by0, dby1 = by1;
        uint32_t carry = 0;
        // four rounds' positions are loaded before the first is used
        for (int base = 0; base < nraw && ncand <= kWalkCand; base += 64 * kWalkRounds) {
          uint32_t j[kWalkRounds], tile[kWalkRounds];
          double2 pj[kWalkRounds];
          uint8_t wc[kWalkRounds];
#pragma unroll
          for (int r = 0; r < kWalkRounds; ++r) {
            if (base + r * 64 < nraw) {  // uniform
              const int u = base + r * 64 + lane < nraw ? base + r * 64 + lane : nraw - 1;
              // the last mark at or before u: lanes past the end see u's own,
              // which the scan has passed already
              const uint32_t sc = scan_max((uint32_t)sh.u.s.mark[u]);
              const uint32_t id = sc > carry ? sc : carry;
              carry = readlane_u(id, 63);
              const uint2 pc = sh.u.s.piece[id - 1];
              j[r] = pc.x + (uint32_t)u;
              tile[r] = pc.y;
              wc[r] = WR[j[r]];
              pj[r] = XY[j[r]];
            }
          }
#pragma unroll
          for (int r = 0; r < kWalkRounds; ++r) {
            const int rest = nraw - base - r * 64;
            if (rest > 0) {
              unsigned long long in = rest >= 64 ? ~0ull : (1ull << rest) - 1ull;
              double px = (pj[r].x - S->x0) * S->ivx;
              double py = (pj[r].y - S->y0) * S->ivy;
              uint32_t pk = (j[r] << 4) | 5u;
              // a particle in the search's own tile is seen directly
              const unsigned long long im = ballot(wc[r] != tile[r]);
              if (im) {
                int ix, iy;
                const bool vis = cand_image((int)(tile[r] & 7u) - 2, (int)(tile[r] >> 3) - 2, wc[r],
                                            ix, iy);
                px -= (double)ix * gw;
                py -= (double)iy * gw;
                pk = (j[r] << 4) | img_code(ix, iy);
                in &= ballot(vis);
              }
              in &= ballot(px >= dbx0) & ballot(px <= dbx1) & ballot(py >= dby0) & ballot(py <= dby1);
              images |= in & im;
              const int pos = ncand + lane_prefix(in);
              ncand += __popcll(in);
              if (ncand <= kWalkCand) {
                if (__builtin_amdgcn_inverse_ballot_w64(in)) {
                  sh.xy[pos] = pj[r];
                  sh.pk[pos] = pk;
                }
              } else {
                ncand = kWalkCand + 1;
              }
            }
          }
        }
        fits = ncand <= kWalkCand;
      }
      if (!fits) {
        if (gsz > 4) {
          gsz >>= 1;
        } else {
          if (grp && part == g) gq[ql].z = kMissWide;
          pending &= ~gmask;
          gsz = kGrp;
        }
        continue;
      }
      wave_fence();
      if constexpr (SEED) {
        if (images) seed_radii<true>(sh, gq, ncand, gmask, t0, k, lx, ly, lane);
        else seed_radii<false>(sh, gq, ncand, gmask, t0, k, lx, ly, lane);
        pending &= ~gmask;
        gsz = kGrp;
        continue;
      }
      int c_lo = 0, c_an = 0;
      const int nr = (ncand + 63) >> 6;
#define SPH_CLASSIFY(NR)                                                                        \
  {                                                                                             \
    if (images) classify<NR, true>(sh, gq, ncand, gmask, t0, k, lx, ly, lane, c_lo, c_an);          \
    else classify<NR, false>(sh, gq, ncand, gmask, t0, k, lx, ly, lane, c_lo, c_an);                \
  }
      if (nr == 3) SPH_CLASSIFY(3)
      else if (nr == 4) SPH_CLASSIFY(4)
      else if (nr == 2) SPH_CLASSIFY(2)
      else SPH_CLASSIFY(1)
#undef SPH_CLASSIFY
      const uint32_t dense =
          (uint32_t)ballot(grp && c_lo < k && c_an > kAnn && c_lo + c_an >= k) & 0xFFFFu;
      if (dense) {
        wave_fence();
        if (images) tighten<true>(sh, gq, ncand, dense, t0, k, lx, ly, lane, c_lo, c_an);
        else tighten<false>(sh, gq, ncand, dense, t0, k, lx, ly, lane, c_lo, c_an);
        // those that it resolved: the others count as misses below
        ntight += (unsigned)__builtin_popcount(
            dense & (uint32_t)ballot(c_an <= kAnn && c_lo + c_an >= k));
      }
      wave_fence();
      const double xq = gq[ql].x, yq = gq[ql].y;
      const bool ok = grp && c_lo < k && c_an <= kAnn && c_lo + c_an >= k;
      auto finish = [&](auto img) {
        constexpr bool IMG = decltype(img)::value;
        const double tau =
            select_annulus<IMG>(sh, ok, k, c_lo, c_an, xq, yq, lx, ly, ql, part, ID, nties);
        if constexpr (BITWISE) {
          const uint32_t todo = (uint32_t)ballot(ok) & 0xFFFFu;
          const double facc = rows_bitwise<IMG>(sh, gq, todo, t0, k, S->kernel, tau, lx, ly, lane,
                                                ID, nbr, kstride);
          if (ok && part == 0) {
            gq[ql].z = tau;
            gq[ql].w = facc;
          }
        } else if (ok) {
          const NbrRow row = nbr_row(nbr, (int64_t)t0 + ql, kstride);
          double facc = 0.0;
          kern_visit(S->kernel, [&](auto kt) {
            facc = row_density<FP32C, IMG, decltype(kt)>(sh, row, k, tau, xq, yq, lx, ly, ql, part);
            // FP32C: a rounding of q of 2^-24 moves F(q) ~ (1 - q)^3 by
            // 3 q / (1 - q) times that, at most 2^-24 2.1 (k / sum)^(1/3) of
            // the sum: beyond 6e-6 where 64 terms add to less than kThinSum
            // (every neighbour near q = 1: the edge of a compact clump, tiny
            // k).  Those few are summed in FP64.
            if constexpr (FP32C) {
              if (facc < kThinSum)
                facc = row_density<false, IMG, decltype(kt)>(sh, row, k, tau, xq, yq, lx, ly, ql, part);
            }
          });
          if (part == 0) {
            gq[ql].z = tau;
            gq[ql].w = facc;
          }
        }
      };
      if (images) finish(std::true_type{}); else finish(std::false_type{});
      if (grp && !ok && part == 0) {
        gq[ql].z = c_lo >= k ? kMissLo : (c_an > kAnn ? kMissAnn : kMissHi);
        // a radius for the exact search from the neighbours inside Rhi
        const double more = kMissReach * k / (c_lo + c_an > 0 ? c_lo + c_an : 1);
        gq[ql].w = __builtin_amdgcn_sqrt(gq[ql].w * (more < 4.0 ? more : 4.0));
      }
      pending &= ~gmask;
      gsz = kGrp;
    }
  }
  wave_fence();
  const double4 out = sh.q[lane0];
  const bool tried = (can >> lane0) & 1ull;
  if constexpr (SEED) {
    // a limit only for a second search
    if (tried) H[t] = out.z == kSeeded && (seed || out.w > 0) ? out.w : 0.0;
    return;
  }
  const bool resolved = tried && out.z >= 0.0;
  if (resolved)
    write_result<FP32C>(S, t, out.x, out.y, out.z, out.w, PredArr{EP, VPX, VPY, t}, H, RHO, C, recp);
  // what is left goes to the exact search
  const bool left = valid && !resolved;
  const unsigned long long m = ballot(left);
  if (m) {
    uint32_t base = 0;
    if (lane0 == 0) base = atomicAdd(retry_count, (uint32_t)__popcll(m));
    base = readlane_u(base, 0);
    if (left) {
      retry[base + lane_prefix(m)] = make_uint2(t, (uint32_t)item_idx);
      if (tried && out.z == kMissHi) H[t] = out.w * (1.0 / kFirstReach);
    }
  }
  // counters: queries with an h that needed the exact search, and why
  const unsigned nfall = __popcll(m & can);
  const unsigned nlo = __popcll(can & ballot(out.z == kMissLo));
  const unsigned nann = __popcll(can & ballot(out.z == kMissAnn));
  const unsigned nhi = __popcll(can & ballot(out.z == kMissHi));
  const unsigned nsplit = __popcll(can & ballot(out.z == kMissWide));
  if (lane0 == 0) {
    // the simulation's bracket misses (set_totals adapts its delta)
    uint32_t* ms = walk_miss + ((int64_t)it.sim * kMissSlots + (blockIdx.x & (kMissSlots - 1))) *
                                   kMissStride;
    if (nlo + nhi) atomicAdd(ms, nlo + nhi);
    if (nann + ntight) atomicAdd(ms + 1, nann + ntight);
    KnnStats* sp = stat_slot(stats);
    stat_add(&sp->retries, nfall);
    stat_add(&sp->ties, nties);
    stat_add(&sp->miss_lo, nlo);
    stat_add(&sp->miss_hi, nhi);
    stat_add(&sp->miss_ann, nann);
    stat_add(&sp->split_fallback, nsplit);
  }
}

// Waves per item of the walk: each takes group / 16 groups of queries, and
// where that would leave fewer than 16384 waves (four per SIMD resident on
// 1024 SIMDs, four rounds of them) down to one group each, so that a small
// launch is as short as one group's search.  Results do not depend on it (a
// group's search knows nothing of the others).
inline int walk_waves_per_item(int nitems, int group) {
  int wpi = 4 * (64 / group);
  while (wpi < 16 && (int64_t)nitems * wpi < 16384) wpi *= 2;
  return wpi;
}

// Byte offset of record j of an array of T, from a packed entry
// pk = j << 4 | image (pk & ~15 is 16 j): one shift at most, so that the
// address is one shift-add on the array base.
template <typename T>
__device__ inline uint64_t rec_off(uint32_t pk) {
  constexpr int sz = (int)sizeof(T);
  static_assert(sz == 32 || sz == 64, "record size");
  return (uint64_t)(pk & ~15u) << (sz == 32 ? 1 : 2);
}

// Source of the neighbour gathers, indexed by packed entry.  A gather runs
// in three steps over a round's entries: near() issues the first load and
// says whether it is the value, pin() waits for those loads, far() loads the
// rest.
//
// An array read through a block's LDS window: entries [wb, wb + W)
// (indices mod 2^32) come from the staged copy, the rest from the array.
// Particles are in Hilbert order, so most neighbours of a block's 256
// consecutive queries lie within a few hundred slots of them.  Every lane
// reads the window (slot 0 when outside it) and pin() passes the values
// through an empty asm statement, so that the compiler cannot fold the two
// loads into one flat load: a flat load completes out of order with the
// global loads, and every wait for a gather would also wait for the row
// chunk loaded behind it.
//
// The window is stored by 16-byte quarters, quarter q of entry i at q W + i: the
// lanes of a wave read the same quarter of arbitrary entries, which spreads
// over all of LDS's banks, where whole entries of 64 (32) bytes would put every
// first quarter into a quarter (half) of them (FP64 force, 1M clustered: 211 ->
// 207 us; bank conflicts -40 %).
template <typename T, int W>
struct WinSrc {
  static constexpr int kQ = (int)sizeof(T) / 16;
  const T* __restrict__ g;
  const u32x4* lds;
  uint32_t wb;
  __device__ bool near(uint32_t pk, T& v) const {
    const uint32_t wj = (pk >> 4) - wb;
    const bool in = wj < (uint32_t)W;
    const uint32_t at = in ? wj : 0u;
#pragma unroll
    for (int q = 0; q < kQ; ++q) ((u32x4*)&v)[q] = lds[q * W + at];
    return in;
  }
  __device__ void pin(T& v) const {
    uint32_t* w = (uint32_t*)&v;
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) / 4); ++i) asm("" : "+v"(w[i]));
  }
  __device__ T far(uint32_t pk) const { return *(const T*)((const char*)g + rec_off<T>(pk)); }
};

// Gathers the sources of n packed entries.
template <int N, typename S, typename T>
__device__ inline void gather(const S& src, const uint32_t* pks, T* pj) {
  bool in[N];
#pragma unroll
  for (int u = 0; u < N; ++u) in[u] = src.near(pks[u], pj[u]);
#pragma unroll
  for (int u = 0; u < N; ++u) src.pin(pj[u]);
#pragma unroll
  for (int u = 0; u < N; ++u)
    if (!in[u]) pj[u] = src.far(pks[u]);
}

// Stages entries [wb, wb + W) of `g` that lie in [lo, hi) into `lds` (the
// block's threads together; the caller synchronises).
template <typename T, int W>
__device__ inline void stage_window(u32x4* lds, const T* __restrict__ g, int64_t wb, int64_t lo,
                                    int64_t hi) {
  constexpr int kQ = (int)sizeof(T) / 16;
  for (int i = threadIdx.x; i < W; i += blockDim.x) {
    const int64_t j = wb + i;
    if (j >= lo && j < hi)
#pragma unroll
      for (int q = 0; q < kQ; ++q) lds[q * W + i] = ((const u32x4*)(g + j))[q];
  }
}

// Visits the entries [n0, k) of a neighbour row (n0 a multiple of 4) in rounds of
// four: their sources (src's records of the entries) are gathered together and
// the next row chunk is loaded before the current one is processed, so that the
// row and gather latencies overlap; the row is read for the last time
// (non-temporal loads).  Full rounds gather their entries as they are; a last
// partial round gathers the query's own slot `self` for the entries past k.
// IMAGES: `body` is told (as a type) whether an entry of the wave's round may be an
// image, which few waves' are.  `flush` runs after each round, with the next
// round's first entry.
template <bool IMAGES = false, typename S, typename Body, typename Flush>
__device__ inline void row_visit(const NbrRow row, int n0, int k, uint32_t self, const S& src,
                                 Body body, Flush flush) {
  constexpr int N = 4;
  if (n0 >= k) return;
  using T = std::remove_cv_t<std::remove_reference_t<decltype(src.far(0u))>>;
  auto ld = [&](int c) { return __builtin_nontemporal_load(row.chunk(c)); };
  u32x4 q = ld(n0 >> 2);
  for (; n0 + N <= k; n0 += N) {
    const uint32_t pks[N] = {q.x, q.y, q.z, q.w};
    T pj[N];
    gather<N>(src, pks, pj);
    if (n0 + N < k) q = ld((n0 + N) >> 2);
    auto round = [&](auto img) {
#pragma unroll
      for (int u = 0; u < N; ++u) body(pks[u], pj[u], img);
    };
    if constexpr (IMAGES) {
      uint32_t im = 0;  // code 5: no image
#pragma unroll
      for (int u = 0; u < N; ++u) im |= pks[u] ^ 5u;
      if (ballot(im & 15u)) round(std::true_type{}); else round(std::false_type{});
    } else {
      round(std::true_type{});
    }
    flush(n0 + N);
  }
  if (n0 < k) {
    const uint32_t spk = self << 4;
    const uint32_t pks[N] = {q.x, q.y, q.z, q.w};
    uint32_t gpk[N];
#pragma unroll
    for (int u = 0; u < N; ++u) gpk[u] = n0 + u < k ? pks[u] : spk;
    T pj[N];
    gather<N>(src, gpk, pj);
#pragma unroll
    for (int u = 0; u < N; ++u) {
      if (n0 + u >= k) break;
      body(pks[u], pj[u], std::true_type{});
    }
    flush(n0 + N);
  }
}

// Exact wavefront search for the queries of the retry list.  Waves stride over
// the list, so the slow searches spread over the GPU.
// Bound by latency, a chain of dependent loads per query, with four waves per
// SIMD to hide it.  What can be loaded ahead is: the next list entry and the
// query's predicted fields before the search, three stages' candidates together;
// the query is a scalar, so its simulation's parameters come by scalar loads, and
// a cell's Hilbert index takes a third of the steps from the table.  Before and now,
// us: 2,200 particles 10.1 -> 9.4, 77,777 12.4 -> 11.4, 262,144 14.3 -> 12.6, 32
// batched simulations 14.9 -> 13.3; with the queries of full annuli, which the walk
// has taken since (tighten), 1M clustered 37.6 -> 34.3, 4M 119 -> 104.
template <bool BITWISE, bool FP32C>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_knn_fallback(
    const Item* __restrict__ items, const SimDev* __restrict__ sims, const double2* __restrict__ XY,
    const uint8_t* __restrict__ WR, const uint32_t* __restrict__ cstart,
    double* __restrict__ H, const double* __restrict__ EP, const double* __restrict__ VPX,
    const double* __restrict__ VPY, const uint32_t* __restrict__ ID,
    uint32_t* __restrict__ nbr, int kstride, double* __restrict__ RHO,
    double* __restrict__ C, void* __restrict__ recp, KnnStats* __restrict__ stats,
    const uint2* __restrict__ retry, const uint32_t* __restrict__ retry_count, int64_t np,
    int* __restrict__ err) {
  __shared__ SearchShared wsh[4];
  // the wave's query as a scalar: its data and its simulation's come by scalar
  // loads, whose registers the search does not need
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  SearchShared& sh = wsh[wv];
  const int64_t nw = (int64_t)gridDim.x * 4;
  const int64_t q0 = (int64_t)blockIdx.x * 4 + wv;
  const int64_t total = (int64_t)(*retry_count);
  uint2 next = retry[q0 < np ? q0 : 0];  // beside the count, and below beside the search
  const uint32_t table = kHilbertTable.w[lane];
  unsigned long long nretry = 0, nties = 0, nfail = 0;
  for (int64_t q = q0; q < total; q += nw) {
    const int64_t t = (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)next.x);
    const int sim = items[__builtin_amdgcn_readfirstlane((int)next.y)].sim;
    next = retry[q + nw < np ? q + nw : 0];
    const SimDev* S = sims + sim;
    const double2 pq = XY[t];
    const double xq = pq.x, yq = pq.y, hp = H[t];
    const PredVal pred = {EP[t], VPX[t], VPY[t]};
    const double R0 = hp > 0 ? hp * kFirstReach : local_radius(S, cstart, xq, yq);
    const unsigned long long nfail0 = nfail;
    const SearchOut so = wave_search<BITWISE>(S, t, xq, yq, R0, XY, WR, cstart, ID, table,
                                              nbr_row(nbr, t, kstride), sh, nretry, nties, nfail);
    if (lane == 0 && nfail != nfail0) atomicOr(err + 1 + sim, 2);
    if (lane == 0 && so.tau > 0)
      write_result<FP32C>(S, t, xq, yq, so.tau, so.facc, pred, H, RHO, C, recp);
  }
  if (lane == 0) {
    KnnStats* sp = stat_slot(stats);
    stat_add(&sp->retries, nretry);
    stat_add(&sp->ties, nties);
    stat_add(&sp->failures, nfail);
  }
}

// ------------------------------------------------------------------------
// Force: one thread per particle, neighbours summed in list order (the
// reference's order when the list is sorted, BITWISE), then kick, drift 2,
// periodic wrap and reflection (sim/sph.go:327-401,122-193).
//
// What bounds it: at 1M clustered, k = 64, FP64, a wave's chain of window reads,
// far gathers and arithmetic with three waves per SIMD to overlap: the vector
// units are busy 55 % of the time, LDS 40 %, the vector L1 50 %.  Halving the FP64
// form's vector instructions (offsets only where a round holds an image,
// viscosity and the spline's derivative without branches, third-order root and
// reciprocal steps: 80 -> 37 per pair) took 50,021 particles at k = 32 from 21.2 to
// 18.6 us, 100,000 from 25.8 to 22.9 and 262,144 from 40.5 to 39.2; 1M, whose
// rows leave the window more often, stayed at 208.
//
// A row's terms are added up in four sections of whole chunks, and the four
// sums in order (the bitwise form: straight through, as the reference), so that
// both splits of the work give the same bits.  PARTS 1: a thread per particle,
// the block's 256 particles sharing a window.  PARTS 4: a block takes 64
// particles and each of its waves one section of their rows, for launches whose
// time is one thread's chain of gathers: 2,200 particles at k = 32 FP64 16 -> 8 us,
// at k = 64 27 -> 11; FP32C 13 -> 7 and 20 -> 9.
inline constexpr int kSections = 4;
// The most items for PARTS 4, whose smaller windows hold fewer of the
// neighbours and are staged four times as often.  FP64 force (with the event
// records' 2 us) by PARTS 1 and 4, us: k = 16 24,576 particles 14.0 and 12.4,
// 32,768 13.9 and 14.3; k = 32 32,768 19.4 and 16.0, 49,152 20.0 and 19.9; k = 64 49,152
// 30.5 and 23.5; 262,144 at k = 32 38 and 60.
inline int force_split_items(int kmax) { return 64 + 2 * kmax; }
int64_t partial_rows(int nitems, int kmax) {
  return std::max<int64_t>(nitems, (int64_t)kSections * std::min(nitems, force_split_items(kmax)));
}
__host__ __device__ inline int section_begin(int k, int s) { return 4 * (((k + 3) / 4 * s) >> 2); }

// The sum of the sections done, and the entry after the current one.
struct SectionSum {
  double x = 0.0, y = 0.0, e = 0.0;
  int end, s = 0;
  __device__ explicit SectionSum(int k) : end(0) { next(k); }
  __device__ void next(int k) {  // past empty sections (k < 13)
    const int at = end;
    do end = section_begin(k, ++s); while (end == at && s < kSections);
  }
};

// ---- totals ----
// From a simulation's sums: the totals, the next CFL half step and the next walk
// bracket (move, wide: the walk's misses of this pass).
__device__ inline void set_totals(SimDev* S, const double* sum, double cfl_min, uint32_t move,
                                  uint32_t wide, bool per_sim, int mode) {
#pragma unroll
  for (int r = 0; r < kNumRed; ++r) S->red[r] = sum[r];
  if (mode == kForceKick) S->dt_last = S->dt_half;
  if (per_sim) {  // regular steps after a job's first pass
    S->pmode = kPermPredict;
    S->fmode = kForceKick;
  }
  S->walk_delta = adapt_delta(S->walk_delta, S->walk_delta0, move, wide, S->n);
  S->dt_half = S->use_cfl ? 0.5 * (S->cfl * cfl_min) : S->dt_fixed;
  S->cfl_min_bits = (unsigned long long)__double_as_longlong(INFINITY);
}

// In launches of up to kFinishItems work items the totals come from the force's
// own launch: the block of a simulation that ends last adds its items' partial
// sums up, in k_reduce's order.  Bound by latency: a launch of its own (k_reduce)
// takes 4.7 us per pass, this adds 2.4 us to the force at 2,200 particles and 3.5
// at 77,777 (304 items).  From about two blocks per CU on, every block's wait for its
// stores and its counter lasts into the next block's time: 262,144 particles (1024
// items) 38.2 -> 45.6 us against 6.4 for the launch, 1M 215 -> 225.6 against 10.5.
inline constexpr int kFinishItems = 512;

// Values that blocks of one launch hand to each other: stored and loaded past
// the caches that their XCDs do not share.
__device__ inline void put_shared(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline double get_shared(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Called by one wave of each of `of` blocks after its put_shared's: true for the
// last of them, which may then get_shared what the others put.  The counter is
// zero again for the next launch.
__device__ inline bool last_of(uint32_t* counter, uint32_t of, int lane) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // what was put has arrived
  uint32_t v = 0;
  if (lane == 0) {
    v = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
    if (v == of) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  v = readlane_u(v, 0);
  asm volatile("" ::: "memory");
  return v == of;
}

// By one wave of each of the simulation's blocks, `parts` of them per item; i0 is
// its first item, ni their number (at most kFinishItems).
__device__ inline void finish_totals(SimDev* S, int sim, int i0, int ni, int parts,
                                     const double* __restrict__ partials,
                                     uint32_t* __restrict__ done,
                                     uint32_t* __restrict__ walk_miss, bool per_sim, int mode,
                                     int lane) {
  if (!last_of(done + (int64_t)sim * kDoneStride, (uint32_t)(ni * parts), lane)) return;
  // the walk's miss counts of this pass (copy q by lane q), read and cleared for
  // the next pass
  int move = 0, wide = 0;
  if (lane < kMissSlots) {
    uint32_t* wm = walk_miss + ((int64_t)sim * kMissSlots + lane) * kMissStride;
    move = (int)wm[0];
    wide = (int)wm[1];
    wm[0] = 0u;
    wm[1] = 0u;
  }
  const double cfl_min = __longlong_as_double((long long)__hip_atomic_load(
      &S->cfl_min_bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  // lane l stands for k_reduce's threads l, l + 64, l + 128 and l + 192
  double v[4][kNumRed];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
#pragma unroll
    for (int r = 0; r < kNumRed; ++r) v[q][r] = 0.0;
    for (int i = q * 64 + lane; i < ni; i += 256) {
      const double* p = partials + (int64_t)(i0 + i) * parts * kNumRed;
#pragma unroll
      for (int r = 0; r < kNumRed; ++r)
        v[q][r] += parts == 1 ? get_shared(p + r)
                              : (get_shared(p + r) + get_shared(p + kNumRed + r)) +
                                    (get_shared(p + 2 * kNumRed + r) + get_shared(p + 3 * kNumRed + r));
    }
  }
  double sum[kNumRed];
#pragma unroll
  for (int r = 0; r < kNumRed; ++r)
    sum[r] = group_sum((v[0][r] + v[2][r]) + (v[1][r] + v[3][r]), 64);
  for (int o = kMissSlots / 2; o > 0; o >>= 1) {
    move += __shfl_xor(move, o, 64);
    wide += __shfl_xor(wide, o, 64);
  }
  if (lane == 0) set_totals(S, sum, cfl_min, (uint32_t)move, (uint32_t)wide, per_sim, mode);
}

// FINISH: the totals too (finish_totals).
template <bool FP32C, bool EXACT, int PARTS, bool FINISH>
__global__ __launch_bounds__(256) void k_force(
    const Item* __restrict__ items, int nitems, SimDev* __restrict__ sims,
    const void* __restrict__ recp, Fields f, const uint32_t* __restrict__ nbr, int kstride,
    int mode, Positions pout, double* __restrict__ partials, const double2* __restrict__ XY,
    uint32_t* __restrict__ red_done, uint32_t* __restrict__ walk_miss) {
  static_assert(PARTS == 1 || (PARTS == kSections && !EXACT));
  constexpr int kParticles = kItem / PARTS;  // of a block
  __shared__ double red[4][kNumRed + 1];
  const int blk = xcd_item(nitems * PARTS);
  const int item_idx = blk / PARTS;
  const Item it = items[item_idx];
  SimDev* S = sims + it.sim;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int slot = PARTS == 1 ? (int)threadIdx.x : (blk % PARTS) * kParticles + lane;
  const bool valid = slot < it.count;
  const int64_t t = it.first + (valid ? slot : 0);
  const int k = S->k;
  const double mass = S->mass;
  const double lx = S->lx, ly = S->ly;
  const int kern = S->kernel;
  const double dt = S->dt_half;
  const bool per_sim = mode < 0;
  if (per_sim) mode = S->fmode;
  // The block's window of neighbour records in LDS, which holds most of the
  // neighbours of Hilbert-ordered particles; the rest are gathered from memory.
  // As wide as its registers' waves leave room for in LDS: 640 slots from first -
  // 192 in FP64 (40 KB, three waves per SIMD), 896 from first - 320 in FP32C (28 KB,
  // five; the bitwise form, four, 512).  Against 512 from first - 128: 1M clustered at k = 64 FP64 208 -> 206 us,
  // 4M FP32C 473 -> 458; 1,024 in FP32C (LDS for four waves) 501.  Around 64
  // particles 256 slots.
  constexpr int kWin = PARTS > 1 ? 256 : (FP32C ? 896 : (EXACT ? 512 : 640));
  constexpr int kBack = PARTS > 1 ? 96 : (FP32C ? 320 : (EXACT ? 128 : 192));
  using Rec = std::conditional_t<FP32C, RecF, RecD>;
  __shared__ u32x4 wrec[kWin * sizeof(Rec) / 16];
  const int64_t wb = it.first + (PARTS == 1 ? 0 : (blk % PARTS) * kParticles) - kBack;
  stage_window<Rec, kWin>(wrec, (const Rec*)recp, wb, S->off, S->off + S->n);
  __syncthreads();
  const WinSrc<Rec, kWin> wsrc{(const Rec*)recp, wrec, (uint32_t)wb};
  double xi, yi, hi, ci, rhoi, A;
  double sx = 0.0, sy = 0.0, se = 0.0;
  const NbrRow row = nbr_row(nbr, t, kstride);
  // this thread's entries: the whole row, or its wave's section
  const int n0 = PARTS == 1 ? 0 : section_begin(k, wv);
  const int n1 = PARTS == 1 || wv == PARTS - 1 ? k : section_begin(k, wv + 1);
  SectionSum total(k);
  if constexpr (!FP32C) {
    const RecD* rec = (const RecD*)recp;
    const RecD me = rec[t];
    xi = me.x; yi = me.y; hi = 2.0 * me.h; ci = 2.0 * me.c; rhoi = 2.0 * me.rho; A = me.B;
    const double hih = me.h, cih = me.c, rhoih = me.rho;  // halves, for the pair means
    const double vpxi = me.vpx, vpyi = me.vpy;
    const double alpha = S->alpha, beta = S->beta, eta2 = S->eta2;
    const double hinv = EXACT ? 0.0 : 1.0 / hi;
    // 4 records (64 B each) in flight per lane, the next row chunk behind them
    auto flush = [&](int n) {
      if (!EXACT && PARTS == 1 && n == total.end) {
        total.x += sx;
        total.y += sy;
        total.e += se;
        sx = sy = se = 0.0;
        total.next(k);
      }
    };
    if constexpr (EXACT) {
      row_visit(row, n0, n1, (uint32_t)t, wsrc, [&](uint32_t pk, const RecD& nb, auto) {
        // the reference's arithmetic, operation for operation
        const double ox = (double)img_ix(pk & 15u) * lx, oy = (double)img_iy(pk & 15u) * ly;
        const double rABx = (nb.x - ox) - xi, rABy = (nb.y - oy) - yi;
        const double ex = (xi + ox) - nb.x, ey = (yi + oy) - nb.y;
        const double vABx = nb.vpx - vpxi, vABy = nb.vpy - vpyi;
        const double d2 = ex * ex + ey * ey;
        const double dot = vABx * rABx + vABy * rABy;
        const double d = sqrt(d2);
        const double q = d / hi;
        const double dR = kern_DF(kern, q);
        double piAB = 0.0;
        if (dot < 0) {
          const double cAB = cih + nb.c;
          const double rhoAB = rhoih + nb.rho;
          const double hAB = hih + nb.h;
          const double muAB = dot * hAB / ((rABx * rABx + rABy * rABy) + eta2);
          piAB = (-alpha * cAB * muAB + beta * muAB * muAB) / rhoAB;
        }
        sx += rABx * (piAB + A + nb.B) * dR / d;
        sy += rABy * (piAB + A + nb.B) * dR / d;
        se += dot * dR;
      }, flush);
    } else {
      // within the 1e-12 contract of this form: the distance from r_AB (one
      // rounding away from the query-side difference) and fused multiply-adds
      // throughout
      const double acih = alpha * cih;
      kern_visit(kern, [&](auto kt) {
        row_visit<true>(row, n0, n1, (uint32_t)t, wsrc, [&](uint32_t pk, const RecD& nb,
                                                                     auto img) {
#pragma clang fp contract(fast)
          double rABx = nb.x - xi, rABy = nb.y - yi;
          if constexpr (decltype(img)::value) {
            rABx = (nb.x - (double)img_ix(pk & 15u) * lx) - xi;
            rABy = (nb.y - (double)img_iy(pk & 15u) * ly) - yi;
          }
          const double vABx = nb.vpx - vpxi, vABy = nb.vpy - vpyi;
          const double r2 = rABx * rABx + rABy * rABy;
          const double dot = vABx * rABx + vABy * rABy;
          const double rinv = rsq64(r2);
          const double q = (r2 * rinv) * hinv;
          const double dR = decltype(kt)::DF64(q);
          // viscosity where the pair approaches, for every pair from
          // min(dot, 0): pi = mu (beta mu - alpha cAB) / rhoAB with one
          // reciprocal, t = mu / rhoAB = dot hAB / ((r^2 + eta2) rhoAB)
          const double rhoAB = rhoih + nb.rho;
          const double v = __builtin_fmin(dot, 0.0) * (hih + nb.h) * rcp64((r2 + eta2) * rhoAB);
          const double x = beta * (v * rhoAB) - (alpha * nb.c + acih);
          const double w = (x * v + (A + nb.B)) * dR * rinv;
          sx += rABx * w;
          sy += rABy * w;
          se += dot * dR;
        }, flush);
      });
    }
    if constexpr (!EXACT && PARTS == 1) {
      sx = total.x;
      sy = total.y;
      se = total.e;
    }
  } else {
    const RecF* rec = (const RecF*)recp;
    const RecF me = rec[t];
    const double2 pme = XY[t];
    xi = pme.x; yi = pme.y;
    hi = 2.0 * (double)me.h;
    // displacements from the fixed-point difference (the minimum image) hold
    // while every neighbour lies within half a box and h spans enough steps
    // of L / 2^32; otherwise from FP64
    const bool fixed = fixed_point_ok(hi, lx, ly);
    const float fsx = (float)(lx * 0x1p-32), fsy = (float)(ly * 0x1p-32);
    const float csx = centred_step(xi, S->x0, lx) * fsx, csy = centred_step(yi, S->y0, ly) * fsy;
    ci = 2.0 * (double)me.c;
    rhoi = 2.0 * (double)me.rho;
    A = (double)me.B;
    // own rho, c, h halved as stored (the pair means are sums of halves)
    const float vpxi = me.vpx, vpyi = me.vpy, rhoif = me.rho, hif = me.h, Af = me.B;
    const float hinv = __builtin_amdgcn_rcpf(2.0f * hif);
    const float alpha = (float)S->alpha, beta = (float)S->beta, eta2 = (float)S->eta2;
    const float acif = alpha * me.c;
    // block-compensated sums (a Kahan step per round of 4 neighbours)
    BlockKahan ax_, ay_, ae_;
    auto flush = [&](int n) {
      ax_.flush();
      ay_.flush();
      ae_.flush();
      if (PARTS == 1 && n == total.end) {
        total.x += ax_.value();
        total.y += ay_.value();
        total.e += ae_.value();
        ax_ = ay_ = ae_ = BlockKahan();
        total.next(k);
      }
    };
    kern_visit(kern, [&](auto kt) {
      using KT = decltype(kt);
      auto pair = [&](float rx, float ry, const RecF& nb) {
#pragma clang fp contract(fast)
        const float d2 = rx * rx + ry * ry;
        // Two particles within one fixed-point step (L / 2^32) can get a zero
        // displacement here (or one from the FP64 positions of coincident
        // particles); their pair term vanishes with the distance (DF(q) ~ q
        // and dot ~ r as r -> 0): the reciprocal square root of at least
        // FLT_MIN keeps it 0 (q = 0, DF(0) = 0, r = 0) rather than the
        // 0 * inf of rsq(0).
        const float dinv = __builtin_amdgcn_rsqf(__builtin_fmaxf(d2, 0x1p-126f));
        // q of the k-th neighbour may round to a few ulp past 1, where DF is
        // of order ulp^2 (no clamp needed)
        const float q = (d2 * dinv) * hinv;
        const float dR = KT::DF(q);
        const float vx_ = nb.vpx - vpxi, vy_ = nb.vpy - vpyi;
        const float dot = vx_ * rx + vy_ * ry;
        // viscosity where the pair approaches (dot < 0), for every pair from
        // min(dot, 0) (mu and pi vanish otherwise; the lanes of a wave take
        // both sides anyway): mu = dot hAB / (r^2 + eta2),
        // pi = mu (beta mu - alpha cAB) / rhoAB, with one reciprocal of
        // (r^2 + eta2) rhoAB
        const float acAB = __builtin_fmaf(alpha, nb.c, acif);
        const float rhoAB = rhoif + nb.rho;
        const float hAB = hif + nb.h;
        const float a_ = __builtin_fminf(dot, 0.f) * hAB;
        const float inv = __builtin_amdgcn_rcpf((d2 + eta2) * rhoAB);
        const float muAB = a_ * inv * rhoAB;
        const float piAB = __builtin_fmaf(beta, muAB, -acAB) * (a_ * inv);
        const float w = (piAB + (Af + nb.B)) * dR * dinv;
        ax_.add_mul(rx, w);
        ay_.add_mul(ry, w);
        ae_.add_mul(dot, dR);
      };
      // 4 records (32 B each) in flight per lane: with most of them in the LDS
      // window, the registers of more buy less than a fifth wave per SIMD.  A
      // wave whose queries all take fixed-point displacements (the usual case)
      // runs a loop without the FP64 form, so every record loads whole.
      if (__all(fixed)) {
        row_visit(row, n0, n1, (uint32_t)t, wsrc, [&](uint32_t, const RecF& nb, auto) {
          pair(__builtin_fmaf((float)(int32_t)(nb.ux - me.ux), fsx, csx),
               __builtin_fmaf((float)(int32_t)(nb.uy - me.uy), fsy, csy), nb);
        }, flush);
      } else {
        row_visit(row, n0, n1, (uint32_t)t, wsrc, [&](uint32_t pk, const RecF& nb, auto) {
          float rx, ry;
          if (fixed) {
            rx = __builtin_fmaf((float)(int32_t)(nb.ux - me.ux), fsx, csx);
            ry = __builtin_fmaf((float)(int32_t)(nb.uy - me.uy), fsy, csy);
          } else {
            const double ox = (double)img_ix(pk & 15u) * lx, oy = (double)img_iy(pk & 15u) * ly;
            const double2 pj = XY[pk >> 4];
            rx = (float)((pj.x - ox) - xi);
            ry = (float)((pj.y - oy) - yi);
          }
          pair(rx, ry, nb);
        }, flush);
      }
    });
    sx = PARTS == 1 ? total.x : ax_.value();
    sy = PARTS == 1 ? total.y : ay_.value();
    se = PARTS == 1 ? total.e : ae_.value();
  }
  if constexpr (PARTS > 1) {
    __shared__ double sec[3][PARTS][64];
    sec[0][wv][lane] = sx;
    sec[1][wv][lane] = sy;
    sec[2][wv][lane] = se;
    __syncthreads();
    if (wv) return;
    sx = sy = se = 0.0;
#pragma unroll
    for (int p = 0; p < PARTS; ++p) {
      sx += sec[0][p][lane];
      sy += sec[1][p][lane];
      se += sec[2][p][lane];
    }
  }
  double r_e = 0, r_rho = 0, r_E = 0, r_px = 0, r_py = 0, r_cfl = INFINITY;
  if (valid) {
    const double fac = mass * S->dfpref / (hi * hi * hi);
    const double ax = sx * fac + S->gxa;
    const double ay = sy * fac + S->gya;
    const double edot = A * se * mass;
    f.ax[t] = ax;
    f.ay[t] = ay;
    f.edot[t] = edot;
    double vx = f.vx[t], vy = f.vy[t], e = f.e[t];
    double x = xi, y = yi;
    if (mode == kForceKick) {
      // kick, sim/sph.go:122-127
      const double adx = ax * (2 * dt), ady = ay * (2 * dt);
      vx = vx + adx;
      vy = vy + ady;
      e = e + edot * 2 * dt;
      // drift 2, :130-135
      const double vdx = vx * dt, vdy = vy * dt;
      x = x + vdx;
      y = y + vdy;
      // periodic wrap, :147-167 (an X wrap skips the Y wrap)
      if (x < S->hor0) {
        x += (S->hor1 - S->hor0);
      } else if (x > S->hor1) {
        x -= (S->hor1 - S->hor0);
      } else if (y < S->vert0) {
        y += (S->vert1 - S->vert0);
      } else if (y > S->vert1) {
        y -= (S->vert1 - S->vert0);
      }
      // reflection, :170-193
      if (x < S->refl[0]) { x -= x - S->refl[0]; vx = -vx; }
      if (x > S->refl[1]) { x -= x - S->refl[1]; vx = -vx; }
      if (y < S->refl[2]) { y -= y - S->refl[2]; vy = -vy; }
      if (y > S->refl[3]) { y -= y - S->refl[3]; vy = -vy; }
      f.vx[t] = vx;
      f.vy[t] = vy;
      f.e[t] = e;
    }
    pout.x[t] = x;
    pout.y[t] = y;
    const double sp2 = vx * vx + vy * vy;
    r_cfl = (0.5 * hi) / (ci + sqrt(sp2));
    r_e = e;
    r_rho = rhoi;
    r_E = mass * (e + 0.5 * sp2);
    r_px = mass * vx;
    r_py = mass * vy;
    // the TotalMomentum quirk value
    if (FINISH && t == S->off + S->n - 1) S->last_speed = sqrt(sp2);
  }
  // block reductions in a fixed order
  r_e = group_sum(r_e, 64);
  r_rho = group_sum(r_rho, 64);
  r_E = group_sum(r_E, 64);
  r_px = group_sum(r_px, 64);
  r_py = group_sum(r_py, 64);
  for (int o = 32; o > 0; o >>= 1) {
    const double other = __shfl_xor(r_cfl, o, 64);
    r_cfl = other < r_cfl ? other : r_cfl;
  }
  auto put = [](double* p, double v) {
    if constexpr (FINISH) put_shared(p, v);
    else *p = v;
  };
  if constexpr (PARTS == 1) {
    if (lane == 0) {
      red[wv][0] = r_e;
      red[wv][1] = r_rho;
      red[wv][2] = r_E;
      red[wv][3] = r_px;
      red[wv][4] = r_py;
      red[wv][5] = r_cfl;
    }
    __syncthreads();
    if (wv) return;
    if (lane < kNumRed)
      put(partials + (int64_t)item_idx * kNumRed + lane,
          (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]));
#pragma unroll
    for (int w = 0; w < 4; ++w) r_cfl = red[w][5] < r_cfl ? red[w][5] : r_cfl;
  } else if (lane == 0) {
    double* p = partials + (int64_t)blk * kNumRed;
    put(p, r_e);
    put(p + 1, r_rho);
    put(p + 2, r_E);
    put(p + 3, r_px);
    put(p + 4, r_py);
  }
  if (lane == 0 && r_cfl < INFINITY)
    atomicMin(&S->cfl_min_bits, (unsigned long long)__double_as_longlong(r_cfl));
  if constexpr (FINISH) {
    const int li = (int)((it.first - S->off) / kItem);
    const int ni = (int)((S->n + kItem - 1) / kItem);
    finish_totals(S, it.sim, item_idx - li, ni, PARTS, partials, red_done, walk_miss, per_sim, mode,
                  lane);
  }
}

// Totals over a simulation's work items in a fixed order.  A simulation of
// more than 1024 items is summed in two stages: red_parts blocks each sum a
// contiguous share of its items (k_reduce_part), then k_reduce adds those
// sums in block order; a smaller one is summed by k_reduce alone.  The order
// of every addition depends only on the simulation's own item count, so
// totals are reproducible and the same alone, batched and served.
__device__ inline void block_sum(double (*sh)[256], double (&acc)[kNumRed]) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int r = 0; r < kNumRed; ++r) sh[r][tid] = acc[r];
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (tid < o)
#pragma unroll
      for (int r = 0; r < kNumRed; ++r) sh[r][tid] += sh[r][tid + o];
    __syncthreads();
  }
}

__global__ __launch_bounds__(256) void k_reduce_part(const SimDev* __restrict__ sims,
                                                     const double* __restrict__ partials,
                                                     const int* __restrict__ item_first,
                                                     const int* __restrict__ item_count,
                                                     double* __restrict__ red_part,
                                                     int parts_max) {
  __shared__ double sh[kNumRed][256];
  const int sim = blockIdx.x / parts_max, part = blockIdx.x % parts_max;
  if (sims[sim].n == 0) return;  // unused slot
  const int i0 = item_first[sim], ni = item_count[sim];
  const int nparts = red_parts(ni);
  if (nparts == 1 || part >= nparts) return;
  const int chunk = (ni + nparts - 1) / nparts;
  const int ia = part * chunk, ib = ia + chunk < ni ? ia + chunk : ni;
  double acc[kNumRed];
#pragma unroll
  for (int r = 0; r < kNumRed; ++r) acc[r] = 0.0;
#pragma unroll 4
  for (int i = ia + (int)threadIdx.x; i < ib; i += 256)
#pragma unroll
    for (int r = 0; r < kNumRed; ++r) acc[r] += partials[(int64_t)(i0 + i) * kNumRed + r];
  block_sum(sh, acc);
  if (threadIdx.x < kNumRed)
    red_part[((int64_t)sim * kRedSplit + part) * kNumRed + threadIdx.x] = sh[threadIdx.x][0];
}

// One block per simulation: the totals from the first stage's sums, the
// TotalMomentum quirk value and what follows from them.
__global__ __launch_bounds__(256) void k_reduce(SimDev* __restrict__ sims,
                                                const double* __restrict__ partials,
                                                const double* __restrict__ red_part,
                                                const int* __restrict__ item_first,
                                                const int* __restrict__ item_count, Fields f,
                                                int mode, uint32_t* __restrict__ walk_miss) {
  __shared__ double sh[kNumRed][256];
  __shared__ uint32_t miss[2][kMissSlots];
  SimDev* S = sims + blockIdx.x;
  if (S->n == 0) return;  // unused slot
  const bool per_sim = mode < 0;
  if (per_sim) mode = S->fmode;
  const int tid = threadIdx.x;
  // the walk's miss counts of this pass (copy q by thread q), read and
  // cleared for the next pass
  if (tid < kMissSlots) {
    uint32_t* wm = walk_miss + ((int64_t)blockIdx.x * kMissSlots + tid) * kMissStride;
    miss[0][tid] = wm[0];
    miss[1][tid] = wm[1];
    wm[0] = 0u;
    wm[1] = 0u;
  }
  const int64_t last = S->off + S->n - 1;
  const double vx_last = tid == 0 ? f.vx[last] : 0.0, vy_last = tid == 0 ? f.vy[last] : 0.0;
  const int i0 = item_first[blockIdx.x], ni = item_count[blockIdx.x];
  const int nparts = red_parts(ni);
  double acc[kNumRed];
#pragma unroll
  for (int r = 0; r < kNumRed; ++r) acc[r] = 0.0;
  if (nparts == 1) {
    // unrolled so that many items' loads are in flight; the additions keep
    // their order
#pragma unroll 8
    for (int i = tid; i < ni; i += 256)
#pragma unroll
      for (int r = 0; r < kNumRed; ++r) acc[r] += partials[(int64_t)(i0 + i) * kNumRed + r];
  } else if (tid < nparts) {
#pragma unroll
    for (int r = 0; r < kNumRed; ++r)
      acc[r] = red_part[((int64_t)blockIdx.x * kRedSplit + tid) * kNumRed + r];
  }
  block_sum(sh, acc);
  if (tid == 0) {
    double sum[kNumRed];
#pragma unroll
    for (int r = 0; r < kNumRed; ++r) sum[r] = sh[r][0];
    S->last_speed = sqrt(vx_last * vx_last + vy_last * vy_last);
    uint32_t move = 0u, wide = 0u;
    for (int q = 0; q < kMissSlots; ++q) {
      move += miss[0][q];
      wide += miss[1][q];
    }
    set_totals(S, sum, __longlong_as_double((long long)S->cfl_min_bits), move, wide, per_sim, mode);
  }
}

__global__ void k_init_sims(SimDev* sims, int nsims) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nsims) return;
  sims[s].cfl_min_bits = (unsigned long long)__double_as_longlong(INFINITY);
}

// ------------------------------------------------------------------------
int enqueue_pass(PassBuffers& b, int perm_mode, int force_mode, hipStream_t st,
                 hipEvent_t* ev) {
  b.timed = 0;
  auto mark = [&](int slot, int end) {
    if (!ev) return;
    (void)hipEventRecord(ev[2 * slot + end], st);  // timing only
    b.timed |= 1u << slot;
  };
  const dim3 blk(kItem);
  const dim3 grd(b.nitems);
  const dim3 grd_all(b.nitems_all);
  const KeySrc src = {b.sims, b.pos_cur.x, b.pos_cur.y, b.fcur.vx, b.fcur.vy, perm_mode, b.err,
                      b.retry_count};
  // one simulation: the sort's first read of the keys makes them
  const bool fused = b.nsims == 1 && b.hole_cpp == 0 && sort_makes_keys(b.np);
  if (!fused || b.any_open) mark(0, 0);
  if (b.any_open) {
    hipLaunchKernelGGL(k_bbox, grd, blk, 0, st, b.items, b.nitems, b.sims, b.pos_cur.x,
                       b.pos_cur.y, b.fcur.vx, b.fcur.vy, perm_mode, b.partials);
    hipLaunchKernelGGL(k_box, dim3(b.nsims), dim3(256), 0, st, b.sims, b.partials, b.red_first,
                       b.red_count);
  }
  if (!fused)
    hipLaunchKernelGGL(k_keys, grd_all, blk, 0, st, b.items_all, b.nitems_all, src, b.sort.keys,
                       b.hole_cpp);
  if (!fused || b.any_open) mark(0, 1);
  mark(1, 0);
  uint32_t *skeys = nullptr, *perm = nullptr;
  sort_pairs(b.sort, b.np, b.key_bits, st, fused ? &src : nullptr, &skeys, &perm);
  mark(1, 1);
  mark(2, 0);
  // as many cell blocks as fit at once, beside which the permuting ones follow
  // (permute at 1M / 4M: 1,024 blocks 46.1 / 148.4 us, 2,048 40.3 / 146.6, 4,096
  // 37.4 / 151.9)
  const int per_cells = (b.nitems + 2047) / 2048;
  const int ncells = (b.nitems + per_cells - 1) / per_cells;
  hipLaunchKernelGGL(k_permute, dim3(b.nitems_all + ncells), blk, 0, st, b.items_all, b.nitems_all,
                     b.items, b.nitems, ncells, per_cells, b.sims, perm, skeys, perm_mode,
                     b.pos_cur, b.fcur, b.xyp, b.fnew, b.wrap, b.cstart);
  mark(2, 1);
  mark(3, 0);
  {
    const int wpi = walk_waves_per_item(b.nitems, b.walk.group);
#define SPH_KNN(F32, BW, SEED, seed)                                                          \
  hipLaunchKernelGGL((k_knn<F32, BW, SEED>), dim3(b.nitems * wpi), dim3(64), 0, st, b.items,    \
                     b.nitems, b.sims, b.xyp, b.wrap, b.cstart, b.fnew.h, b.fnew.ep,           \
                     b.fnew.vpx, b.fnew.vpy, b.fnew.id, b.nbr, b.kmax, b.fnew.rho, b.fnew.c,   \
                     b.rec, b.stats, b.retry, b.retry_count, b.walk, b.walk_miss, wpi, seed)
    // the retry list: four times as many blocks as fit at once, so that blocks
    // that drew quick searches make room for others (a few % faster than
    // one resident round); four queries per block
    const int fb_grid = b.nitems < 64 ? 64 * b.nitems : 4096;
#define SPH_FB(BW, F32)                                                                       \
  hipLaunchKernelGGL((k_knn_fallback<BW, F32>), dim3(fb_grid), dim3(256), 0, st, b.items,     \
                     b.sims, b.xyp, b.wrap, b.cstart, b.fnew.h,               \
                     b.fnew.ep, b.fnew.vpx, b.fnew.vpy, b.fnew.id, b.nbr, b.kmax, b.fnew.rho,   \
                     b.fnew.c, b.rec, b.stats, b.retry, b.retry_count, b.np, b.err)
    mark(6, 0);
    if (!b.have_h || b.some_new) {
      SPH_KNN(false, false, true, b.have_h ? 1 : 2);
      SPH_KNN(false, false, true, 0);
    }
    if (b.bitwise) SPH_KNN(false, true, false, 0);
    else if (b.prec == kPrecFP32C) SPH_KNN(true, false, false, 0);
    else SPH_KNN(false, false, false, 0);
    mark(6, 1);
    mark(8, 0);
    if (b.bitwise) SPH_FB(true, false);
    else if (b.prec == kPrecFP32C) SPH_FB(false, true);
    else SPH_FB(false, false);
    mark(8, 1);
#undef SPH_KNN
#undef SPH_FB
  }
  mark(3, 1);
  mark(4, 0);
  const int parts = b.bitwise || b.nitems > force_split_items(b.kmax) ? 1 : kSections;
  const bool finish = b.nitems <= kFinishItems;
#define SPH_FORCE_(F32, EX, P, FIN)                                                            \
  hipLaunchKernelGGL((k_force<F32, EX, P, FIN>), dim3(b.nitems * P), dim3(256), 0, st, b.items, \
                     b.nitems, b.sims, (const void*)b.rec, b.fnew, b.nbr, b.kmax, force_mode,  \
                     b.pos_cur, b.partials, b.xyp, b.red_done, b.walk_miss)
#define SPH_FORCE(F32, EX)                                                                     \
  {                                                                                            \
    if (finish) SPH_FORCE_(F32, EX, 1, true); else SPH_FORCE_(F32, EX, 1, false);              \
  }
  static_assert(64 + 2 * kMaxK <= kFinishItems, "launches that split rows finish in the force");
  if (b.bitwise) SPH_FORCE(false, true)
  else if (b.prec == kPrecFP32C && parts > 1) SPH_FORCE_(true, false, kSections, true);
  else if (b.prec == kPrecFP32C) SPH_FORCE(true, false)
  else if (parts > 1) SPH_FORCE_(false, false, kSections, true);
  else SPH_FORCE(false, false)
#undef SPH_FORCE_
#undef SPH_FORCE
  mark(4, 1);
  if (!finish) {
    mark(5, 0);
    if (b.red_parts_max > 1)
      hipLaunchKernelGGL(k_reduce_part, dim3(b.nsims * b.red_parts_max), dim3(256), 0, st, b.sims,
                         b.partials, b.red_first, b.red_count, b.red_part, b.red_parts_max);
    hipLaunchKernelGGL(k_reduce, dim3(b.nsims), dim3(256), 0, st, b.sims, b.partials, b.red_part,
                       b.red_first, b.red_count, b.fnew, force_mode, b.walk_miss);
    mark(5, 1);
  }
  return (int)hipGetLastError();
}

// ------------------------------------------------------------------------
// readback / upload by particle ID
__host__ __device__ inline double* field_ptr(const Positions& p, const Fields& f, int field) {
  switch (field) {
    case 0: return p.x;
    case 1: return p.y;
    case 2: return f.vx;
    case 3: return f.vy;
    case 4: return f.rho;
    case 5: return f.c;
    case 6: return f.e;
    case 7: return f.edot;
    case 8: return f.ax;
    case 9: return f.ay;
    case 10: return f.ep;
    case 11: return f.vpx;
    case 12: return f.vpy;
    case 13: return f.h;
    default: return nullptr;
  }
}

// Field readback / upload by particle ID.  Row of particle t is
// off(sim) + ID(t); `sim` < 0 selects every simulation, otherwise rows are
// relative to that simulation's first particle.
__global__ void k_scatter_by_id(const Item* __restrict__ items, int nitems,
                                const SimDev* __restrict__ sims, Positions p, Fields f,
                                int field, int sim, double* __restrict__ out) {
  const Item it = items[blockIdx.x];
  if ((int)threadIdx.x >= it.count || (sim >= 0 && it.sim != sim)) return;
  const int64_t t = it.first + threadIdx.x;
  const int64_t base = sim >= 0 ? 0 : sims[it.sim].off;
  out[base + f.id[t]] = field_ptr(p, f, field)[t];
}

__global__ void k_gather_by_id(const Item* __restrict__ items, int nitems,
                               const SimDev* __restrict__ sims, Positions p, Fields f,
                               int field, int sim, const double* __restrict__ in) {
  const Item it = items[blockIdx.x];
  if ((int)threadIdx.x >= it.count || (sim >= 0 && it.sim != sim)) return;
  const int64_t t = it.first + threadIdx.x;
  const int64_t base = sim >= 0 ? 0 : sims[it.sim].off;
  field_ptr(p, f, field)[t] = in[base + f.id[t]];
}

double* field_data(const PassBuffers& b, int field) { return field_ptr(b.pos_cur, b.fcur, field); }

int enqueue_read_field(const PassBuffers& b, int field, int sim, double* dev_out, hipStream_t st) {
  hipLaunchKernelGGL(k_scatter_by_id, dim3(b.nitems), dim3(kItem), 0, st, b.items, b.nitems, b.sims,
                     b.pos_cur, b.fcur, field, sim, dev_out);
  return (int)hipGetLastError();
}

int enqueue_write_field(PassBuffers& b, int field, int sim, const double* dev_in, hipStream_t st) {
  hipLaunchKernelGGL(k_gather_by_id, dim3(b.nitems), dim3(kItem), 0, st, b.items, b.nitems, b.sims,
                     b.pos_cur, b.fcur, field, sim, dev_in);
  return (int)hipGetLastError();
}

// Neighbour rows by ID: IDs of the neighbours, recomputed squared distances
// (same formula as the search) and, if px is not null, the neighbours'
// positions seen through the query's image offset o (NNPos = p_j - o,
// sim/nearest-neighbour.go:81,152), sorted ascending by (d2, ID), equal ones (one
// particle through several images) in list order.  Entries of a row past the
// simulation's k (batches of mixed k) read ID 0xFFFFFFFF and NaN, so every
// output entry is written.
//
// Lane = entry, G = 32 or 64 lanes per row: each counts the entries before its
// own in that order (k broadcast reads from LDS) and writes to that place of the
// row, so that a row leaves as one contiguous piece.  With a thread per row,
// sorting by insertion in global memory, 50,021 rows of 32 took 262 us (521 us
// with positions).
constexpr int kReadRows = 32;  // rows of a block
template <int G>
__global__ __launch_bounds__(256) void k_read_nbrs(const Item* __restrict__ items, int nitems,
                                                   const SimDev* __restrict__ sims,
                                                   const double2* __restrict__ XY, Fields f,
                                                   const uint32_t* __restrict__ nbr, int kstride,
                                                   int kout, uint32_t* __restrict__ ids,
                                                   double* __restrict__ d2o,
                                                   double* __restrict__ px,
                                                   double* __restrict__ py) {
  constexpr int kRows = 256 / G;  // rows at once
  __shared__ double sd[kRows][G];
  __shared__ uint32_t sid[kRows][G];
  const int item_idx = blockIdx.x / (kItem / kReadRows);
  const int q0 = blockIdx.x % (kItem / kReadRows) * kReadRows;
  const Item it = items[item_idx];
  const SimDev* S = sims + it.sim;
  const int k = S->k;
  const double lx = S->lx, ly = S->ly;
  const int r = threadIdx.x / G, e = threadIdx.x % G;
  // a row's lanes lie in one wave, whose LDS operations complete in order
  for (int q = q0 + r; q < q0 + kReadRows && q < it.count; q += kRows) {
    const int64_t t = it.first + q;
    const double2 pi = XY[t];
    double d2 = NAN, x = NAN, y = NAN;
    uint32_t id = 0xFFFFFFFFu;
    if (e < k) {
      const uint32_t pk = nbr_row(nbr, t, kstride)[e];
      const uint32_t j = pk >> 4;
      const double ox = (double)img_ix(pk & 15u) * lx;
      const double oy = (double)img_iy(pk & 15u) * ly;
      const double2 pj = XY[j];
      const double ex = (pi.x + ox) - pj.x, ey = (pi.y + oy) - pj.y;
      d2 = ex * ex + ey * ey;
      id = f.id[j];
      x = pj.x - ox;
      y = pj.y - oy;
    }
    // what the row is ordered by: a distance that is no number (a particle of a state
    // gone bad) comes last, so that every place is taken once
    const double by = d2 == d2 ? d2 : INFINITY;
    wave_fence();
    sd[r][e] = by;
    sid[r][e] = id;
    wave_fence();
    int at = e;
    if (e < k) {
      at = 0;
      for (int m = 0; m < k; ++m) {
        const double v = sd[r][m];
        const uint32_t w = sid[r][m];
        at += v < by || (v == by && (w < id || (w == id && m < e)));
      }
    }
    if (e < kout) {
      const int64_t o = ((int64_t)f.id[t] + S->off) * kout + at;
      ids[o] = id;
      d2o[o] = d2;
      if (px) {
        px[o] = x;
        py[o] = y;
      }
    }
  }
}

int enqueue_read_neighbours(const PassBuffers& b, uint32_t* dev_ids, double* dev_d2,
                            double* dev_px, double* dev_py, hipStream_t st) {
  const dim3 grd(b.nitems * (kItem / kReadRows));
#define SPH_READ(G)                                                                               \
  hipLaunchKernelGGL((k_read_nbrs<G>), grd, dim3(256), 0, st, b.items, b.nitems, b.sims, b.xyp,   \
                     b.fcur, b.nbr, b.kmax, b.kout, dev_ids, dev_d2, dev_px, dev_py)
  if (b.kout <= 32) SPH_READ(32);
  else SPH_READ(64);
#undef SPH_READ
  return (int)hipGetLastError();
}

int enqueue_init_sims(PassBuffers& b, hipStream_t st) {
  hipLaunchKernelGGL(k_init_sims, dim3((b.nsims + 255) / 256), dim3(256), 0, st, b.sims,
                     b.nsims);
  return (int)hipGetLastError();
}

}  // namespace sph

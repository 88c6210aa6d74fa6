// Internal handle of the C ABI (include/sphugo.h), shared by the batch
// path and the serve loop.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdio>
#include <string>
#include <utility>
#include <vector>

#include "sph_host.hpp"
#include "sphugo.h"

namespace sph {

int fail(int code, const char* fmt, ...);

#define HIPCHK(call)                                                                \
  do {                                                                              \
    hipError_t e_ = (call);                                                         \
    if (e_ != hipSuccess)                                                           \
      return sph::fail(SPH_EDEVICE, "%s: %s", #call, hipGetErrorString(e_));        \
  } while (0)

}  // namespace sph

using sph::Fields;
using sph::Item;
using sph::KnnStats;
using sph::PassBuffers;
using sph::Positions;
using sph::SimDev;

namespace sph {
// What a handle keeps for its readbacks (sph_stage.hip).
struct Stage {
  char* flags = nullptr;   // pinned block (or none) from enqueue_flags to take_flags
  hipEvent_t ev[8] = {};   // per slot of a large copy: filled
};
void stage_open(Stage& s);
void stage_close(Stage& s);
}  // namespace sph

struct sph_sim {
  int device = 0;
  std::vector<SimDev> hsims;
  std::vector<sph_params> hparams;  // creation parameters, per simulation
  std::vector<int64_t> sim_n;
  std::vector<Item> hitems;
  int64_t np = 0;
  int kmax = 0;
  int prec = 0;
  int bitwise = 0;
  bool timing = false;
  hipStream_t st = nullptr;
  hipEvent_t ev[2 * SPH_NTIMERS] = {};
  double t_ms[SPH_NTIMERS] = {};
  int64_t t_cnt[SPH_NTIMERS] = {};
  int cur = 0;
  Fields F[2] = {};
  Positions P[2] = {};
  PassBuffers pb = {};
  int64_t step = 0;
  std::vector<void*> allocs;
  double* d_scratch = nullptr;     // np doubles for readback
  uint32_t* d_nids = nullptr;      // neighbour readback (lazy)
  double* d_nd2 = nullptr;
  double* d_npx = nullptr;         // neighbour image positions (lazy)
  double* d_npy = nullptr;
  KnnStats last_stats = {};
  // graph replay of a regular step, one per field-buffer parity
  bool graph_on = false;
  hipGraphExec_t gexec[2] = {nullptr, nullptr};
  double grid_cpp = 4.0;        // cells per particle of the cell grid
  int64_t cell_capacity = 0;    // cstart entries allocated
  sph::Stage stage;

  sph_sim() { sph::stage_open(stage); }
  sph_sim(const sph_sim&) = delete;
  sph_sim& operator=(const sph_sim&) = delete;

  template <class T>
  int alloc(T** p, int64_t count) {
    void* q = nullptr;
    size_t bytes = (size_t)(count > 0 ? count : 1) * sizeof(T);
    if (hipMalloc(&q, bytes) != hipSuccess)
      return sph::fail(SPH_ENOMEM, "hipMalloc of %zu bytes failed", bytes);
    allocs.push_back(q);
    *p = (T*)q;
    return 0;
  }
  void drop_graphs() {
    for (auto& g : gexec)
      if (g) {
        (void)hipGraphExecDestroy(g);
        g = nullptr;
      }
  }
  ~sph_sim() {
    drop_graphs();
    // teardown: nothing is left to report a failure to
    for (void* q : allocs) (void)hipFree(q);
    for (auto& e : ev)
      if (e) (void)hipEventDestroy(e);
    if (st) (void)hipStreamDestroy(st);
    sph::stage_close(stage);
  }
  void bind() {
    pb.fcur = F[cur];
    pb.fnew = F[cur ^ 1];
    pb.pos_cur = P[0];
  }
  // Exchange everything with another handle (a handle rebuilt in place:
  // the caller's pointer stays valid).  Lists every member above.
  void swap_state(sph_sim& o) {
    std::swap(device, o.device);
    hsims.swap(o.hsims);
    hparams.swap(o.hparams);
    sim_n.swap(o.sim_n);
    hitems.swap(o.hitems);
    std::swap(np, o.np);
    std::swap(kmax, o.kmax);
    std::swap(prec, o.prec);
    std::swap(bitwise, o.bitwise);
    std::swap(timing, o.timing);
    std::swap(st, o.st);
    std::swap(ev, o.ev);
    std::swap(t_ms, o.t_ms);
    std::swap(t_cnt, o.t_cnt);
    std::swap(cur, o.cur);
    std::swap(F, o.F);
    std::swap(P, o.P);
    std::swap(pb, o.pb);
    std::swap(step, o.step);
    allocs.swap(o.allocs);
    std::swap(d_scratch, o.d_scratch);
    std::swap(d_nids, o.d_nids);
    std::swap(d_nd2, o.d_nd2);
    std::swap(d_npx, o.d_npx);
    std::swap(d_npy, o.d_npy);
    std::swap(last_stats, o.last_stats);
    std::swap(graph_on, o.graph_on);
    std::swap(gexec, o.gexec);
    std::swap(grid_cpp, o.grid_cpp);
    std::swap(cell_capacity, o.cell_capacity);
    std::swap(stage, o.stage);
  }
};

namespace sph {
// shared helpers (sph_api.hip)
void fill_simdev(SimDev& d, const sph_params* p, int64_t n, int lg);
void set_grid(SimDev& d, int lg);
// box of the open axes around host positions (creation guess; the device
// sets it again before every pass) and the first-pass radius guess
void init_open_box(SimDev& d, const double* x, const double* y, int64_t n);
int check_params(const sph_params* p, int64_t n);
int fetch_sims(sph_sim* s);
// readback staging (sph_stage.hip): copy `bytes` (a multiple of 4) of a device
// array to the host after the stream's work so far; returns when they are there
int copy_out(sph_sim* s, void* dst, const void* dev, size_t bytes);
// the same of at most kOrderedMax doubles in the order of their IDs 0..n-1
inline constexpr int kOrderedMax = 8192;
int read_ordered(sph_sim* s, double* dst, const double* dev, const uint32_t* id, int n);
// write the first nerr error flags and the counters' sums to a pinned block
// (enqueue_flags), and read them there once the stream is done (take_flags, which
// copies them itself where there is no block)
int enqueue_flags(sph_sim* s, int nerr);
int take_flags(sph_sim* s, sph::KnnStats* stats, int* err, int nerr);
int check_device_flags(sph_sim* s);
int alloc_state(sph_sim* h, int64_t np, int nitems);
// Cells per particle of a grid (at least; at most four times as many, as a
// grid's size is a power of four) unless tuning chose another.  The walk looks
// at cells of several particles, so the finest ones serve regions denser than
// the mean, and their number costs key bits and cell ranges: per pass with 4
// and 2 per particle, us: 77,777 uniform 114 and 107, 100,000 clustered at k = 64
// 167 and 163, 524,288 clustered 356 and 346; sizes whose grid is the same either
// way (262,144, 1,048,576) alike.  With 1, 1,048,576 clustered take 634 against 603.
inline constexpr double kGridCpp = 2.0;
int grid_log2(int64_t n, double cpp);
}  // namespace sph

// pyfds_amd C-ABI: contexts, uploads, per-tile event lists, the step loop and HIP graphs.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <limits>
#include <deque>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "../../include/pyfds_amd.h"
#include "fds_common.h"
#include "fds_kernels.h"
#include "fds_lbc.h"
#include "fds_line1d.h"
#include "fds_step2d.h"
#include "fds_step_nl.h"

namespace {

thread_local std::string g_last_error;

int fail(int code, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

#define HIP_TRY(expr)                                                                        \
  do {                                                                                       \
    hipError_t err_ = (expr);                                                                \
    if (err_ != hipSuccess)                                                                  \
      return fail(FDS_E_HIP, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(err_),       \
                  __FILE__, __LINE__);                                                       \
  } while (0)

// Owned device allocation.
struct DevBuf {
  void *p = nullptr;
  size_t bytes = 0;
  DevBuf() = default;
  DevBuf(const DevBuf &) = delete;
  DevBuf &operator=(const DevBuf &) = delete;
  DevBuf(DevBuf &&o) noexcept : p(o.p), bytes(o.bytes) {
    o.p = nullptr;
    o.bytes = 0;
  }
  DevBuf &operator=(DevBuf &&o) noexcept {
    if (this != &o) {
      release();
      p = o.p;
      bytes = o.bytes;
      o.p = nullptr;
      o.bytes = 0;
    }
    return *this;
  }
  ~DevBuf() { release(); }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
  }
  hipError_t ensure(size_t b) {
    if (b <= bytes && p) return hipSuccess;
    release();
    if (b == 0) b = 16;
    hipError_t e = hipMalloc(&p, b);
    if (e == hipSuccess) bytes = b;
    return e;
  }
  template <typename U>
  U *as() const { return static_cast<U *>(p); }
};

// Pinned host memory (hipHostMalloc), grown on demand: the staging area that asynchronous
// runs copy their recorded outputs into.
struct HostBuf {
  void *p = nullptr;
  size_t bytes = 0;
  HostBuf() = default;
  HostBuf(const HostBuf &) = delete;
  HostBuf &operator=(const HostBuf &) = delete;
  ~HostBuf() { release(); }
  void release() {
    if (p) (void)hipHostFree(p);
    p = nullptr;
    bytes = 0;
  }
  hipError_t ensure(size_t b) {
    if (b <= bytes && p) return hipSuccess;
    release();
    hipError_t e = hipHostMalloc(&p, std::max<size_t>(b, 16), hipHostMallocDefault);
    if (e == hipSuccess) bytes = std::max<size_t>(b, 16);
    return e;
  }
};

// A run enqueued by fds_run_async / fds_batch_run_async whose outputs are not taken yet:
// its step count and the staging slot (and event set) it uses.
struct Flight {
  int64_t rows = 0;
  int slot = 0;
};
constexpr int kMaxFlights = 2;

template <typename U>
hipError_t upload(DevBuf &d, const std::vector<U> &h, hipStream_t s) {
  hipError_t e = d.ensure(std::max<size_t>(h.size() * sizeof(U), 16));
  if (e != hipSuccess) return e;
  if (h.empty()) return hipSuccess;
  e = hipMemcpyAsync(d.p, h.data(), h.size() * sizeof(U), hipMemcpyHostToDevice, s);
  if (e != hipSuccess) return e;
  return hipStreamSynchronize(s);
}

int64_t floordiv(int64_t a, int64_t b) {
  int64_t q = a / b;
  if ((a % b != 0) && ((a < 0) != (b < 0))) --q;
  return q;
}

int64_t ceildiv(int64_t a, int64_t b) { return -floordiv(-a, b); }

// Where a component's values live inside a tile's LDS arrays: rows [rmin, rmax] x cols
// [cmin, cmax] of the tile (relative to its origin), stored row-major with row width w.
struct Region {
  int rmin, rmax, cmin, cmax, w;
  int pos(int r, int c) const { return (r - rmin) * w + (c - cmin); }
};

struct Events {
  std::vector<int32_t> ptr, pos, id;
};

struct Comp {
  bool present = false;
  bool accumulated = false;   // updated with -= (Kahan compensation applies)
  DevBuf buf[2], cbuf[2];
  // boundary program (host copy kept for validation and event building)
  std::vector<int64_t> cells;
  std::vector<int32_t> ptr;
  std::vector<double> a, table;
  std::vector<int64_t> off, stride, len;
  DevBuf d_ptr, d_a, d_off, d_stride, d_table;
  DevBuf ev_ptr, ev_pos, ev_id;
  // outputs
  std::vector<int64_t> out_cells;
  DevBuf oev_ptr, oev_pos, oev_id;
  DevBuf lhead, ohead;   // resident 1D engine: per-thread first boundary cell / output point
  DevBuf lput, oput;     // and the heads of the threads that have any
  DevBuf obuf;
  int64_t obuf_rows = 0;
  HostBuf stage[kMaxFlights];   // outputs of asynchronous runs, one slot per run in flight
};

enum Family { kAcoustic, kThermal, kNonlinear };

}  // namespace

struct fds_ctx {
  int model = 0, form = 0, device = 0;
  int64_t nx = 0, ny = 0, n = 0;
  Family family = kAcoustic;
  bool one_d = false;     // 1D linear model run on the 2D kernels (nx = n, ny = 1)
  bool axi = false;
  hipStream_t stream = nullptr;
  Comp comp[3];
  int parity = 0;
  DevBuf coef[FDS_NUM_COEFF];
  bool coef_set[FDS_NUM_COEFF] = {};
  DevBuf zeros;           // n zeros of the state type (1D y coefficients, absent slots)
  double s[FDS_NUM_SCALARS] = {};
  bool lossy = false, iso_b = true, iso_k = true;
  bool committed = false;
  int tile = -1;          // requested shape index (-1: default)
  int shape = 0;          // shape index in use (tile table, then the streaming table)
  bool streaming = false; // row-streaming engine in use
  int strip_rows = 0;     // streaming strip height override (0: from the shape and the grid)
  int num_cu = 256;       // compute units of the device
  int fuse = 1;           // time steps per launch of the streaming shape
  int ghost = 0;          // ghost columns per side of a streaming tile (fuse - 1; lossy: 1)
  int ghost_rows = 0;     // ghost rows per side of a streaming strip (fuse - 1; lossy: 0)
  int sx = 0;             // x stride of the tiles (tx - 2*ghost)
  bool fused = false;     // fused engine in use (a row-streaming engine: streaming is set too)
  bool coupled = false;   // stepped one step per launch by a coupling (until it runs alone again)
  int fused_stages = 0, fused_rows = 0;   // layout a batch asked for (0: by the grid)
  // the layout (stages, strip height) whose tiles cannot hold the event lists (0: none known)
  int over_stages = 0, over_rows = 0;
  DevBuf fev_tables;         // its event tables, one after the other (`fused_ev` points into it)
  fds::FusedEv fused_ev{};
  DevBuf pal_idx, pal;    // material classes of the cells and their coefficients
  int npal = 0;           // classes, the zero class included (0: none known)
  bool line = false;      // resident 1D engine in use (one workgroup, many steps per launch)
  int line_var = 0;       // its variant: index into fds::kLineCpt
  int line_threads = 0;   // its workgroup size
  int line_wgs = 1;       // workgroups (segments of the line)
  int line_seg = 0;       // cells owned per segment
  int line_ghost = 0;     // ghost cells per segment side = most steps per launch (0: one segment)
  int line_cfg_threads = -1, line_cfg_ghost = 0;  // requested segmentation (-1: automatic)
  int tx = 0, ty = 0, tiles_x = 0, tiles_y = 0, ntiles = 0;
  bool events_dirty = true;
  DevBuf dyn;
  DevBuf zero_ptr;        // ntiles+1 zeros: empty event lists
  const fds::KernelSet *ks = nullptr;
  size_t elem = 8;
  // graphs: key (chunk, parity) -> exec
  std::map<std::pair<int, int>, hipGraphExec_t> graphs;
  int graph_chunk = 0;              // steps of a full graph chunk (other graphs: run tails)
  uint64_t generation = 0, graph_generation = ~0ull;
  std::vector<hipGraph_t> graph_objs;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;   // bracket the launches of the last run
  double last_run_ms = 0.0;
  // asynchronous runs in flight (oldest first), the next staging slot, and per slot the
  // events after the run's first launch, its last launch and its output copies
  std::deque<Flight> flights;
  int next_slot = 0;
  int batch_flights = 0;          // asynchronous batch runs in flight that include this context
  hipEvent_t fev[kMaxFlights][3] = {};
  // flow along x (AcousticFlow2D): per-row shift period, applied after every step
  DevBuf flow_period;
  bool flow = false;
  // ThermoAcoustic1D loss coupling (acoustic context): density, loss factor, accumulator
  DevBuf couple_rho, couple_loss, couple_acc;
  // learned absorbing boundary (caller-owned bf16 weights), applied after every step
  const uint16_t *lbc_w1 = nullptr, *lbc_w2 = nullptr;
  int lbc_layer = 0;
  float lbc_cs[3] = {1.f, 1.f, 1.f};
  bool lbc_ring = false;      // several steps per launch (fds_lbc_ring.hip)
  DevBuf lbc_rec, lbc_cells, lbc_packed;   // recorded points of its band, its cells, its weights
  int lbc_nrec = 0;
  // non-finite detection: scans in every graph chunk and after every run; the result
  // (dyn[kDynNonfinite]) is copied to nf_stage[slot] (slot kMaxFlights: synchronous runs)
  bool nf_check = false;
  HostBuf nf_stage;
};

// What a batch's kernels and tables assume of a member.
struct MemberLayout {
  int shape, fuse, ghost, ghost_rows, tx, ty, ntiles;
  bool fused, line, lossy;
  bool operator==(const MemberLayout &o) const {
    return shape == o.shape && fuse == o.fuse && ghost == o.ghost && ghost_rows == o.ghost_rows &&
           tx == o.tx && ty == o.ty && ntiles == o.ntiles && fused == o.fused && line == o.line &&
           lossy == o.lossy;
  }
};

struct fds_batch {
  std::vector<fds_ctx *> ctxs;
  int device = 0, form = 0, tile = -1;
  size_t elem = 8;
  hipStream_t stream = nullptr;
  const fds::KernelSet *ks = nullptr;
  int shape = 0;
  bool streaming = false;
  bool fused = false, fused_any = false;   // fused engine; some member is not acoustic iso / axi
  DevBuf ev_inst, ev_slot;                 // its tiles with events
  int nev = 0;
  int fuse = 1;
  int tx = 0, ty = 0, ntiles = 0;
  std::vector<MemberLayout> layouts;       // the members as its tables and kernels take them
  size_t lds = 0;
  DevBuf descs[2][2];          // [parity][store]
  DevBuf tile_inst, inst_base, dyn;
  std::map<std::pair<int, int>, hipGraphExec_t> graphs;
  std::vector<hipGraph_t> graph_objs;
  std::vector<uint64_t> build_gen;   // member generations the descriptors were built for
  std::vector<int> build_parity;     // member parities at build time
  int flip = 0;                      // members flipped this many times (mod 2) since build
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  double last_run_ms = 0.0;
  std::deque<Flight> flights;     // asynchronous batch runs in flight (oldest first)
  int next_slot = 0;
  hipEvent_t fev[kMaxFlights][3] = {};
  // tile scheduling of streaming batches: 0 the hardware dispatcher (one workgroup per tile,
  // XCD-banded), 1 a persistent grid taking tiles from a work queue in `order`
  int schedule = 0;
  DevBuf order, queue;
  int nq = 0;             // work-queue counters the queue buffer holds (one per launch)
};

namespace {

bool is_kahan(const fds_ctx *c) { return c->form == FDS_FP32_KAHAN; }

void drop_graphs(fds_ctx *c) {
  for (auto &kv : c->graphs) (void)hipGraphExecDestroy(kv.second);
  for (auto g : c->graph_objs) (void)hipGraphDestroy(g);
  c->graphs.clear();
  c->graph_objs.clear();
}

void touch(fds_ctx *c) { c->generation++; }

Region region_of(const fds_ctx *c, int k) {
  const int tx = c->tx, ty = c->ty;
  if (c->family == kNonlinear) {
    if (k == 0) return Region{0, 0, -1, tx, tx + 2};
    if (k == 1) return Region{0, 0, 0, tx, tx + 1};
    return Region{0, 0, 0, tx - 1, tx};
  }
  // rows of all fused stages: G ghost rows above and below the strip
  const int G = c->ghost_rows;
  if (k == 0) return Region{-G - 1, ty + G, -1, tx, tx + 2};
  if (k == 1) return Region{-G, ty - 1 + G, 0, tx, tx + 1};
  return Region{-G, ty + G, 0, tx - 1, tx};
}

// One entry of a tile's event list.
struct TileEvent {
  int32_t tile, pos, id;
};

// The entries by tile, in order of (pos, id) within a tile.  (Counted into place: cells mostly come
// in order of their index, so few tiles need sorting.  1000 x 800 cells, a fifth of them on a
// boundary of both velocities: first pass 109 ms with all entries sorted, 41 ms so.)
void group_events(const std::vector<TileEvent> &all, int ntiles, Events &ev) {
  ev.ptr.assign(ntiles + 1, 0);
  for (const auto &e : all) ev.ptr[e.tile + 1]++;
  for (int t = 0; t < ntiles; ++t) ev.ptr[t + 1] += ev.ptr[t];
  ev.pos.resize(all.size());
  ev.id.resize(all.size());
  std::vector<int32_t> at(ev.ptr.begin(), ev.ptr.end() - 1);
  for (const auto &e : all) {
    const int32_t q = at[e.tile]++;
    ev.pos[q] = e.pos;
    ev.id[q] = e.id;
  }
  std::vector<std::pair<int32_t, int32_t>> tmp;
  for (int t = 0; t < ntiles; ++t) {
    const int32_t e0 = ev.ptr[t], e1 = ev.ptr[t + 1];
    const auto before = [&](int32_t a, int32_t b) {
      return ev.pos[a] < ev.pos[b] || (ev.pos[a] == ev.pos[b] && ev.id[a] <= ev.id[b]);
    };
    int32_t e = e0 + 1;
    while (e < e1 && before(e - 1, e)) ++e;
    if (e >= e1) continue;
    tmp.clear();
    for (e = e0; e < e1; ++e) tmp.push_back({ev.pos[e], ev.id[e]});
    std::sort(tmp.begin(), tmp.end());
    for (e = e0; e < e1; ++e) {
      ev.pos[e] = tmp[e - e0].first;
      ev.id[e] = tmp[e - e0].second;
    }
  }
}

void build_bound_events(const fds_ctx *c, int k, Events &ev) {
  const Comp &cp = c->comp[k];
  const Region R = region_of(c, k);
  // tile (txi, tyi) has its column 0 at absolute column txi*sx - g and row 0 at tyi*ty
  const int64_t nx = c->nx, sx = c->sx, ty = c->ty, g = c->ghost;
  std::vector<TileEvent> all;
  const int64_t cmin_abs = R.cmin - g;
  const int64_t cmax_abs = (int64_t)(c->tiles_x - 1) * sx + R.cmax - g;
  const int64_t rmax_abs = (int64_t)(c->tiles_y - 1) * ty + R.rmax;
  for (size_t u = 0; u < cp.cells.size(); ++u) {
    const int64_t j = cp.cells[u];
    // absolute row Rw and column C with Rw*nx + C = j, C in [cmin_abs, cmax_abs]
    const int64_t rlo = std::max<int64_t>(R.rmin, ceildiv(j - cmax_abs, nx));
    const int64_t rhi = std::min<int64_t>(rmax_abs, floordiv(j - cmin_abs, nx));
    for (int64_t Rw = rlo; Rw <= rhi; ++Rw) {
      const int64_t C = j - Rw * nx;
      const int64_t ty_lo = std::max<int64_t>(0, ceildiv(Rw - R.rmax, ty));
      const int64_t ty_hi = std::min<int64_t>(c->tiles_y - 1, floordiv(Rw - R.rmin, ty));
      const int64_t tx_lo = std::max<int64_t>(0, ceildiv(C + g - R.cmax, sx));
      const int64_t tx_hi = std::min<int64_t>(c->tiles_x - 1, floordiv(C + g - R.cmin, sx));
      for (int64_t tyi = ty_lo; tyi <= ty_hi; ++tyi)
        for (int64_t txi = tx_lo; txi <= tx_hi; ++txi) {
          const int r = (int)(Rw - tyi * ty), col = (int)(C - txi * sx + g);
          all.push_back({(int32_t)(tyi * c->tiles_x + txi), R.pos(r, col), (int32_t)u});
        }
    }
  }
  group_events(all, c->ntiles, ev);
}

void build_output_events(const fds_ctx *c, int k, Events &ev) {
  const Comp &cp = c->comp[k];
  const Region R = region_of(c, k);
  std::vector<TileEvent> all;
  for (size_t s = 0; s < cp.out_cells.size(); ++s) {
    const int64_t j = cp.out_cells[s];
    // the tile that owns the cell (owned columns of a streaming tile start at its ghost)
    const int64_t iy = j / c->nx, ix = j % c->nx;
    const int64_t tyi = iy / c->ty, txi = ix / c->sx;
    const int r = (int)(iy - tyi * c->ty), col = (int)(ix - txi * c->sx + c->ghost);
    all.push_back({(int32_t)(tyi * c->tiles_x + txi), R.pos(r, col), (int32_t)s});
  }
  group_events(all, c->ntiles, ev);
}

// Shape index -> (tx, ty); indices from kNumTiles on name the streaming shapes.
void shape_of(int t, int *tx, int *ty) {
  if (t < fds::kNumTiles) {
    *tx = fds::kTileShapes[t][0];
    *ty = fds::kTileShapes[t][1];
  } else {
    *tx = fds::kStreamShapes[t - fds::kNumTiles][0];
    *ty = fds::kStreamShapes[t - fds::kNumTiles][1];
  }
}

// The streaming engine covers the 2D models (lossy acoustics one step per launch); 1D models
// run on the resident engine or tiles.  Batches stream lossless members only.
bool can_stream(const fds_ctx *c) {
  return c->family != kNonlinear && c->ny > 1;
}

bool can_stream_batch(const fds_ctx *c) { return can_stream(c) && !c->lossy; }

// The fused engines cover the 2D models whose arrays a buffer descriptor spans (32-bit byte
// offsets, rows past either end included), lossy ones if their material classes are known.
bool fuse_reach(const fds_ctx *c) {
  const int64_t reach = c->n + (fds::kFusedStrip + 4 * fds::kFusedMax) * c->nx + 1024;
  return can_stream(c) && reach * (int64_t)c->elem < (int64_t)1 << 32;
}

bool can_fuse(const fds_ctx *c) {
  return fuse_reach(c) && (!(c->lossy && c->family == kAcoustic) || c->npal > 0);
}

// Resident 1D engine variant for n cells: `cpt` cells per thread if given, else the fewest
// cells per thread that fit (the most threads: a step is bound by the one CU's issue rate, so
// spreading the line over more waves wins; measured on 2000 cells: 0.59 us per step with 2
// cells per thread, 0.62 with 4, 0.70 with 8).  Returns the variant index or -1.
int line_variant(int64_t n, int cpt, int fam) {
  for (int i = 0; i < fds::kNumLineCpt; ++i) {
    const int64_t thr = (n + fds::kLineCpt[i] - 1) / fds::kLineCpt[i];
    if (thr > fds::line_max_threads(fam, i)) continue;
    if (cpt <= 0 || fds::kLineCpt[i] == cpt) return i;
  }
  return -1;
}

// Depth of a cell from the rim of a square grid.
int rim_depth(const fds_ctx *c, int64_t cell) {
  const int64_t x = cell % c->nx, y = cell / c->nx;
  return (int)std::min(std::min(x, c->nx - 1 - x), std::min(y, c->ny - 1 - y));
}

// Whether a learned boundary can take S steps per launch (fds_lbc_ring.hip): FP32, isotropic
// lossless, no boundary cell where the frame is computed anew, no recorded point in the layer and
// few in the band.  Any other field steps one by one (1056^2: 19.8 us a step then, 7.9 so).
bool can_ring(const fds_ctx *c, int S) {
  if (is_kahan(c) || c->lossy || c->flow || c->coupled || !c->iso_b || !c->iso_k ||
      !fds::lbc_ring_fits(c->nx, S))
    return false;
  int records = 0;
  for (int k = 0; k < 3; ++k) {
    for (int64_t q : c->comp[k].cells)
      if (rim_depth(c, q) < fds::kLbcDepth + fds::kLbcBand + S) return false;
    for (int64_t q : c->comp[k].out_cells) {
      const int d = rim_depth(c, q);
      if (d < fds::kLbcDepth) return false;
      if (d < fds::kLbcDepth + fds::kLbcBand) ++records;
    }
  }
  return records <= fds::kRingRecords;
}

// Layout of the fused engine: stages per launch and strip height.
//
// Stages: a launch's time grows slowly with them (2048^2 FP64 acoustics: 38 us at 4, 42 us at 6),
// so all kFusedMax, except on small grids, where a launch is bound by the latency of one strip
// and the iterations it takes: 401 x 301 FP64 2.3 us a step at 4 stages, 2.4 at 6; from 800 x 600
// on 6 are ahead (FP64 3.0 and 2.9).  One where something follows every step.
//
// Lossy acoustics: a stage holds 15 values a column, so three stages (2000 x 1500 FP64 11 us a
// step at 3, 14 at 2; 3000^2 38 at 3 and 4), four for large fields of the FP32 forms (3000^2 FP32
// 13.4 at 4, 15.0 at 3), and with the radius' coefficients on top two (2000 x 1500 FP64 15.8 at
// 2, 15.6 at 3, 301 x 901 5.3 and 5.4), three for large ones (3000^2 FP64 53 at 2, 46 at 3).
//
// Height: short strips make enough waves to fill the chip, tall ones waste fewer ghost rows
// (2S a strip, lossy 3S).  Two rounds of resident waves: two a SIMD for FP64, lossy fields and
// AXI (its stage's chain is the longest), so 16 strips a CU, three for the FP32 forms, 24.  us a
// step at 16 and 24: FP64 1200 x 1100 3.70 and 4.14, 2048^2 7.0 and 7.0, 3000 x 2500 16.7 and
// 16.3, thermal 1500^2 3.47 and 3.64, AXI 1024 x 1536 3.99 and 4.79, Kahan AXI 4.13 and 4.92;
// Kahan 2048^2 7.45 and 7.29, thermal 1500^2 3.16 and 2.94; FP32 1500 x 1203 3.23 and 3.02,
// 2500^2 5.8 and 5.3.  Rows beyond 64 or below 4 gained nothing at any size.  (Not the best at
// every size: 2048^2 FP64 takes 43.7 us a launch at the rule's height, 40.5 in strips of 12.)
//
// 1: no such layout, the tiles of this one cannot hold the event lists.
int choose_fused(fds_ctx *c) {
  const bool lossy = c->lossy && c->family == kAcoustic;
  int S = c->n < (1 << 18) ? 4 : fds::kFusedMax;
  if (lossy && c->axi) S = c->n < (1 << 22) ? 2 : 3;
  else if (lossy) S = c->elem == 4 && c->n >= (1 << 20) ? fds::kFusedLossyMax : 3;
  if (c->fused_stages) S = c->fused_stages;
  c->lbc_ring = c->lbc_w1 && can_ring(c, S);
  if ((c->lbc_w1 && !c->lbc_ring) || c->flow || c->coupled) S = 1;
  const int64_t sx = 64 - 2 * S - (lossy ? 1 : 0), across = (c->nx + sx - 1) / sx;
  const int64_t strips = (lossy || c->axi || c->elem == 8 ? 16 : 24) * (int64_t)c->num_cu;
  const int64_t want = (across * c->ny + strips / 2) / strips;
  const int H = c->strip_rows > 0 ? std::min(c->strip_rows, fds::kFusedStrip)
                : c->fused_rows   ? c->fused_rows
                                  : (int)std::min<int64_t>(std::max<int64_t>(want, 4), 64);
  if (S == c->over_stages && H == c->over_rows) {
    c->lbc_ring = false;
    return 1;
  }
  c->fused = c->streaming = true;
  c->fuse = S;
  c->ghost = S;
  c->ghost_rows = lossy ? 2 * S - 1 : S - 1;
  c->tx = 64;
  c->ty = H;
  c->sx = (int)sx;
  c->shape = fds::kDefaultLossless2D;
  c->tiles_x = (int)((c->nx + c->sx - 1) / c->sx);
  c->tiles_y = (int)((c->ny + c->ty - 1) / c->ty);
  const int64_t nt = (int64_t)c->tiles_x * c->tiles_y;
  if (nt > (int64_t)std::numeric_limits<int32_t>::max() / 2)
    return fail(FDS_E_ARG, "grid too large for the tile index (%lld tiles)", (long long)nt);
  c->ntiles = (int)nt;
  c->events_dirty = true;
  return 0;
}

int choose_tiles(fds_ctx *c) {
  c->streaming = false;
  c->fused = false;
  c->lbc_ring = false;
  c->line = false;
  c->fuse = 1;
  c->ghost = 0;
  c->ghost_rows = 0;
  if ((c->one_d || c->family == kNonlinear) && c->tile < 0 && c->n <= fds::kLineMaxResident) {
    // automatic layout (no line shape set): one wave, else segments by line_layout
    int cfg_threads = c->line_cfg_threads, cfg_ghost = c->line_cfg_ghost, cpt_req = c->strip_rows;
    if (cfg_threads < 0) {
      cfg_threads = 0;
      if (c->strip_rows <= 0 && c->n > fds::kLineWave) {
        const fds::LineLayout l = fds::line_layout(
            c->n, c->lossy && c->family == kAcoustic, c->family == kNonlinear,
            c->family == kThermal, is_kahan(c));
        cfg_threads = fds::kLineWave;
        cfg_ghost = l.ghost;
        cpt_req = l.cpt;
      }
    }
    int v = -1;
    if (cfg_threads > 0) {
      for (int i = 0; i < fds::kNumLineCpt; ++i)
        if (fds::kLineCpt[i] == cpt_req) v = i;
    } else {
      v = line_variant(c->n, cpt_req,
                       c->family == kNonlinear ? fds::kLineNonlinear : fds::kLineAcoustic);
    }
    if (v < 0 && c->strip_rows > 0)
      return fail(FDS_E_ARG, "the resident 1D engine has no %d-cell-per-thread variant for %lld "
                  "cells", c->strip_rows, (long long)c->n);
    if (v >= 0) {
      // event lists are indexed by thread over all segments, like tiles
      c->line = true;
      c->line_var = v;
      const int cpt = fds::kLineCpt[v];
      if (cfg_threads > 0) {
        // W workgroups of cfg_threads threads: L owned + 2 G ghost cells each
        c->line_threads = cfg_threads;
        c->line_ghost = cfg_ghost;
        c->line_seg = c->line_threads * cpt - 2 * c->line_ghost;
        c->line_wgs = (int)((c->n + c->line_seg - 1) / c->line_seg);
      } else {
        c->line_threads = (int)(((c->n + cpt - 1) / cpt + 63) / 64 * 64);
        c->line_ghost = 0;
        c->line_seg = (int)c->n;
        c->line_wgs = 1;
      }
      c->shape = -1;
      c->tx = (int)c->n;
      c->ty = 1;
      c->sx = c->tx;
      c->tiles_x = c->ntiles = c->line_threads * c->line_wgs;
      c->tiles_y = 1;
      c->events_dirty = true;
      return 0;
    }
  }
  if (c->family == kNonlinear) {
    c->tx = fds::kNlTile;
    c->ty = 1;
    c->shape = 0;
  } else {
    if (c->tile < 0 && can_fuse(c))
      if (const int rc = choose_fused(c); rc <= 0) return rc;
    int t = c->tile;
    if (t < 0) t = (c->ny == 1) ? fds::kTileRow : (c->lossy ? fds::kDefaultLossy2D
                                                             : fds::kDefaultLossless2D);
    if (t >= fds::kNumTiles && !can_stream(c))
      t = (c->ny == 1) ? fds::kTileRow : fds::kDefaultTile2D;
    // lossy acoustics streams one step per launch with its own row ring: shapes with deeper
    // prefetch have no lossy kernels
    if (t >= fds::kNumTiles && c->lossy && c->family == kAcoustic &&
        fds::stream_single_only(t - fds::kNumTiles))
      return fail(FDS_E_ARG, "shape %d (prefetch %d rows) serves lossless fields only", t,
                  fds::kStreamShapes[t - fds::kNumTiles][4]);
    c->shape = t;
    c->streaming = t >= fds::kNumTiles;
    shape_of(t, &c->tx, &c->ty);
    if (c->streaming) {
      // lossy acoustics: one step per launch, one ghost column per side, no ghost rows
      const bool lossy = c->lossy && c->family == kAcoustic;
      c->fuse = lossy ? 1 : fds::kStreamShapes[t - fds::kNumTiles][2];
      c->ghost = lossy ? 1 : c->fuse - 1;
      c->ghost_rows = lossy ? 0 : c->ghost;
      if (c->strip_rows > 0) {
        c->ty = c->strip_rows;
      } else {
        // a strip is walked row by row by its waves: small grids get shorter strips so that
        // there are enough waves to cover the memory latency (~4 per SIMD)
        const int64_t sx = c->tx - 2 * c->ghost;
        const int64_t waves = ((c->nx + sx - 1) / sx) * (c->tx / 64);
        const int64_t want = 4 * 4 * (int64_t)c->num_cu;
        const int64_t h = (c->ny * waves + want - 1) / want;
        const int hmin = 2 * c->fuse + 2;
        if (h < c->ty) c->ty = (int)std::max<int64_t>(hmin, h);
      }
    }
  }
  c->sx = c->tx - 2 * c->ghost;
  c->tiles_x = (int)((c->nx + c->sx - 1) / c->sx);
  c->tiles_y = (int)((c->ny + c->ty - 1) / c->ty);
  const int64_t nt = (int64_t)c->tiles_x * c->tiles_y;
  if (nt > (int64_t)std::numeric_limits<int32_t>::max() / 2)
    return fail(FDS_E_ARG, "grid too large for the tile index (%lld tiles)", (long long)nt);
  c->ntiles = (int)nt;
  c->events_dirty = true;
  return 0;
}

size_t lds_bytes(const fds_ctx *c) {
  if (c->family == kNonlinear || c->streaming || c->line) return 0;   // static LDS only
  const bool sep_k = c->axi || !c->iso_k;
  fds::Lds2D L = fds::lds2d_layout(c->tx, c->ty, !c->iso_b, sep_k, is_kahan(c));
  return (size_t)L.total * c->elem;
}

// Event lists of the resident 1D engine, sorted by thread (over the threads of all segments):
// pos = register slot of the cell in its thread's block of cpt cells; id = unique boundary cell or
// output slot.  Boundary cells go to every segment whose ghost-extended range holds them (ghost
// cells must evolve like the owner's), recorded points only to their owner.
struct LineEvents {
  std::vector<int32_t> thread, pos, id;
};

void build_line_events(const fds_ctx *c, const std::vector<int64_t> &cells, bool outputs,
                       LineEvents &ev) {
  const int64_t cpt = fds::kLineCpt[c->line_var];
  const int64_t L = c->line_seg, G = c->line_ghost, E = (int64_t)c->line_threads * cpt;
  const int64_t W = c->line_wgs;
  std::vector<std::pair<int32_t, std::pair<int32_t, int32_t>>> all;
  for (size_t u = 0; u < cells.size(); ++u) {
    const int64_t j = cells[u];
    const int64_t w_lo = outputs ? j / L : std::max<int64_t>(0, ceildiv(j + G - E + 1, L));
    const int64_t w_hi = outputs ? j / L : std::min<int64_t>(W - 1, floordiv(j + G, L));
    for (int64_t w = w_lo; w <= w_hi; ++w) {
      const int64_t local = j - (w * L - G);
      all.push_back({(int32_t)(w * c->line_threads + local / cpt),
                     {(int32_t)(local % cpt), (int32_t)u}});
    }
  }
  std::sort(all.begin(), all.end());
  for (auto &t : all) {
    ev.thread.push_back(t.first);
    ev.pos.push_back(t.second.first);
    ev.id.push_back(t.second.second);
  }
}

// A head and its thread.  Most threads of a line have none: the table is filled on the device and
// only these go there from the host.
template <typename H>
struct LinePut {
  H h;
  int32_t thread;
};

template <typename H>
__global__ __launch_bounds__(256) void k_line_fill(H *h, int n, H none) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t < n) h[t] = none;
}

template <typename H>
__global__ __launch_bounds__(256) void k_line_put(H *h, const LinePut<H> *put, int n) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t < n) h[put[t].thread] = put[t].h;
}

template <typename H>
int upload_heads(fds_ctx *c, DevBuf &heads, DevBuf &list, const std::vector<LinePut<H>> &put,
                 const H &none) {
  const int n = c->ntiles, m = (int)put.size();
  HIP_TRY(heads.ensure((size_t)n * sizeof(H)));
  hipLaunchKernelGGL(k_line_fill<H>, dim3((n + 255) / 256), dim3(256), 0, c->stream,
                     heads.as<H>(), n, none);
  if (m) {
    HIP_TRY(upload(list, put, c->stream));
    hipLaunchKernelGGL(k_line_put<H>, dim3((m + 255) / 256), dim3(256), 0, c->stream,
                       heads.as<H>(), list.as<const LinePut<H>>(), m);
  }
  HIP_TRY(hipGetLastError());
  return 0;
}

// Per-thread heads of the resident 1D engine's event lists: the first boundary cell with its
// program entry (when the program has one entry), the first recorded point.
int rebuild_line_heads(fds_ctx *c, Comp &cp, const LineEvents &ev, const LineEvents &oe) {
  std::vector<LinePut<fds::LineEvHead>> bh;
  std::vector<LinePut<fds::LineOutHead>> oh;
  for (size_t e0 = 0, e1; e0 < ev.thread.size(); e0 = e1) {
    for (e1 = e0; e1 < ev.thread.size() && ev.thread[e1] == ev.thread[e0];) ++e1;
    const int u = ev.id[e0], q0 = cp.ptr[u];
    fds::LineEvHead h{0x1ff, 0, 0, 0.0, (int32_t)e0, (int32_t)e1};
    if (cp.ptr[u + 1] - q0 == 1)
      h = fds::LineEvHead{ev.pos[e0] | (e1 - e0 > 1 ? 0x100 : 0), (int32_t)cp.stride[q0],
                          cp.off[q0], cp.a[q0], (int32_t)e0 + 1, (int32_t)e1};
    bh.push_back({h, ev.thread[e0]});
  }
  for (size_t e0 = 0, e1; e0 < oe.thread.size(); e0 = e1) {
    for (e1 = e0; e1 < oe.thread.size() && oe.thread[e1] == oe.thread[e0];) ++e1;
    oh.push_back({fds::LineOutHead{oe.pos[e0] | (e1 - e0 > 1 ? 0x100 : 0), oe.id[e0],
                                   (int32_t)e0 + 1, (int32_t)e1},
                  oe.thread[e0]});
  }
  if (int rc = upload_heads(c, cp.lhead, cp.lput, bh, fds::LineEvHead{0xff, 0, 0, 0.0, 0, 0}))
    return rc;
  return upload_heads(c, cp.ohead, cp.oput, oh, fds::LineOutHead{0xff, 0, 0, 0});
}

// Event tables of the fused engine (fds::FusedEv) from the components' boundary event lists
// `bev` and output event lists `oev`.  Boundary programs become classes: a tile's distinct
// programs, each a chain of entries.  Returns 1 when some tile has more entries than the kernels
// hold (the caller then leaves the fused engine).
int build_fused_events(fds_ctx *c, const Events *bev, const Events *oev) {
  const int g = c->ghost_rows + 1, rows = c->ty + 2 * g;
  std::vector<int32_t> slot(c->ntiles, -1), cls_ptr(1, 0), tiles;
  std::vector<uint32_t> words;
  std::vector<fds::FusedClass> cls;
  std::vector<fds::FusedPoint> points;
  std::vector<int32_t> point_rows;
  // distinct programs of each component, by their entries (-1: one without entries, which does
  // nothing and has no class)
  std::vector<int32_t> prog[3];
  std::vector<std::pair<int32_t, int32_t>> first[3];   // entries of a distinct program
  for (int k = 0; k < 3; ++k) {
    const Comp &cp = c->comp[k];
    std::map<std::vector<int64_t>, int32_t> seen;
    std::vector<int64_t> key;
    for (size_t u = 0; u < cp.cells.size(); ++u) {
      if (cp.ptr[u] == cp.ptr[u + 1]) {
        prog[k].push_back(-1);
        continue;
      }
      key.clear();
      for (int32_t e = cp.ptr[u]; e < cp.ptr[u + 1]; ++e) {
        int64_t bits;
        std::memcpy(&bits, &cp.a[e], 8);
        key.insert(key.end(), {bits, cp.off[e], cp.stride[e]});
      }
      const auto it = seen.emplace(key, (int32_t)first[k].size());
      if (it.second) first[k].push_back({cp.ptr[u], cp.ptr[u + 1]});
      prog[k].push_back(it.first->second);
    }
  }
  int nslots = 0;
  std::vector<int32_t> local[3], known[3];   // a program's entry in tile known[..]
  for (int k = 0; k < 3; ++k) {
    local[k].assign(first[k].size(), 0);
    known[k].assign(first[k].size(), -1);
  }
  for (int t = 0; t < c->ntiles; ++t) {
    bool any = false;
    for (int k = 0; k < 3; ++k)
      any = any || bev[k].ptr[t + 1] > bev[k].ptr[t] || oev[k].ptr[t + 1] > oev[k].ptr[t];
    if (!any) continue;
    slot[t] = nslots++;
    tiles.push_back(t);
    words.resize((size_t)nslots * rows * 64, 0u);
    uint32_t *w = words.data() + (size_t)(nslots - 1) * rows * 64;
    const size_t base = cls.size();
    for (int k = 0; k < 3; ++k) {
      const Region R = region_of(c, k);
      for (int32_t e = bev[k].ptr[t]; e < bev[k].ptr[t + 1]; ++e) {
        const int r = bev[k].pos[e] / R.w + R.rmin + g, col = bev[k].pos[e] % R.w + R.cmin;
        if (r < 0 || r >= rows || col < 0 || col >= 64) continue;
        const int32_t p = prog[k][bev[k].id[e]];
        if (p < 0) continue;
        if (known[k][p] != t) {
          known[k][p] = t;
          local[k][p] = (int32_t)(cls.size() - base + 1);
          const auto [e0, e1] = first[k][p];
          for (int32_t q = e0; q < e1; ++q)
            cls.push_back(fds::FusedClass{c->comp[k].a[q], c->comp[k].off[q],
                                          c->comp[k].stride[q], k,
                                          q + 1 < e1 ? (int32_t)(cls.size() - base + 2) : 0});
          if (cls.size() - base >= (size_t)fds::kFusedClasses) return 1;
        }
        w[r * 64 + col] |= (uint32_t)local[k][p] << (8 * k);
      }
      // recorded points: owned cells, the list is sorted by row
      int32_t e = oev[k].ptr[t];
      for (int r = 0; r <= c->ty; ++r) {
        point_rows.push_back((int32_t)points.size());
        for (; e < oev[k].ptr[t + 1] && oev[k].pos[e] / R.w + R.rmin == r; ++e) {
          const int col = oev[k].pos[e] % R.w + R.cmin;
          points.push_back(fds::FusedPoint{(uint32_t)(col | k << 6 | r << 8), oev[k].id[e]});
          w[(r + g) * 64 + col] |= fds::kFusedRecord << k;
        }
      }
    }
    cls_ptr.push_back((int32_t)cls.size());
  }
  if (c->lbc_ring) {
    std::vector<fds::LbcRec> rec;
    for (int k = 0; k < 3; ++k)
      for (size_t q = 0; q < c->comp[k].out_cells.size(); ++q)
        if (rim_depth(c, c->comp[k].out_cells[q]) < fds::kLbcDepth + fds::kLbcBand)
          rec.push_back(fds::LbcRec{(int32_t)c->comp[k].out_cells[q], k, (int32_t)q});
    c->lbc_nrec = (int)rec.size();
    HIP_TRY(upload(c->lbc_rec, rec, c->stream));
    fds::LbcRing r{};
    r.g = (int)c->nx;
    r.depth = c->fuse;
    r.rec = c->lbc_rec.as<const fds::LbcRec>();
    r.nrec = c->lbc_nrec;
    HIP_TRY(c->lbc_cells.ensure(fds::lbc_ring_cells_bytes(r)));
    HIP_TRY(c->lbc_packed.ensure(fds::lbc_ring_packed_bytes()));
    fds::launch_ring_cells(r, c->lbc_cells.p, c->stream);
    HIP_TRY(hipGetLastError());
  }
  // one buffer and one copy: each costs more than what is in it
  std::vector<uint8_t> blob;
  const auto put = [&](const auto &v) {
    const size_t at = blob.size(), n = v.size() * sizeof(v[0]);
    blob.resize((at + n + 15) / 16 * 16);
    if (n) std::memcpy(blob.data() + at, v.data(), n);
    return at;
  };
  const size_t at[7] = {put(slot), put(tiles), put(words), put(cls_ptr), put(cls), put(points),
                        put(point_rows)};
  HIP_TRY(upload(c->fev_tables, blob, c->stream));
  const uint8_t *base = c->fev_tables.as<const uint8_t>();
  c->fused_ev = fds::FusedEv{reinterpret_cast<const int32_t *>(base + at[0]),
                        reinterpret_cast<const int32_t *>(base + at[1]),
                        reinterpret_cast<const uint32_t *>(base + at[2]),
                        reinterpret_cast<const int32_t *>(base + at[3]),
                        reinterpret_cast<const fds::FusedClass *>(base + at[4]),
                        reinterpret_cast<const fds::FusedPoint *>(base + at[5]),
                        reinterpret_cast<const int32_t *>(base + at[6]), rows, nslots};
  return 0;
}

int rebuild_events(fds_ctx *c) {
  if (!c->events_dirty) return 0;
  if (c->fused) {
    Events bev[3], oev[3];
    for (int k = 0; k < 3; ++k) {
      build_bound_events(c, k, bev[k]);
      build_output_events(c, k, oev[k]);
    }
    const int rc = build_fused_events(c, bev, oev);
    if (rc < 0) return rc;
    if (rc == 0) {
      c->events_dirty = false;
      touch(c);
      return 0;
    }
    c->over_stages = c->fuse;    // until the boundaries change
    c->over_rows = c->ty;
    if (int rc2 = choose_tiles(c)) return rc2;
  }
  if (!c->line) {
    std::vector<int32_t> zp(c->ntiles + 1, 0);
    HIP_TRY(upload(c->zero_ptr, zp, c->stream));
  }
  for (int k = 0; k < 3; ++k) {
    Comp &cp = c->comp[k];
    if (!cp.present) continue;
    if (c->line) {
      LineEvents ev, oe;
      build_line_events(c, cp.cells, false, ev);
      HIP_TRY(upload(cp.ev_pos, ev.pos, c->stream));
      HIP_TRY(upload(cp.ev_id, ev.id, c->stream));
      build_line_events(c, cp.out_cells, true, oe);
      HIP_TRY(upload(cp.oev_pos, oe.pos, c->stream));
      HIP_TRY(upload(cp.oev_id, oe.id, c->stream));
      if (int rc = rebuild_line_heads(c, cp, ev, oe)) return rc;
      continue;
    }
    Events ev;
    build_bound_events(c, k, ev);
    HIP_TRY(upload(cp.ev_ptr, ev.ptr, c->stream));
    HIP_TRY(upload(cp.ev_pos, ev.pos, c->stream));
    HIP_TRY(upload(cp.ev_id, ev.id, c->stream));
    Events oe;
    build_output_events(c, k, oe);
    HIP_TRY(upload(cp.oev_ptr, oe.ptr, c->stream));
    HIP_TRY(upload(cp.oev_pos, oe.pos, c->stream));
    HIP_TRY(upload(cp.oev_id, oe.id, c->stream));
  }
  c->events_dirty = false;
  touch(c);
  return 0;
}

// ---- host float64 arrays <-> device arrays of the form's type (FP32 forms convert on the device;
// Kahan: the pair (x, c) with x - c = the value)
__global__ __launch_bounds__(256) void k_from_double(const double *__restrict__ d, float *x,
                                                     float *c, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float f = (float)d[i];
  x[i] = f;
  if (c) c[i] = (float)((double)f - d[i]);
}

__global__ __launch_bounds__(256) void k_to_double(double *__restrict__ d, const float *x,
                                                   const float *c, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) d[i] = c ? (double)x[i] - (double)c[i] : (double)x[i];
}

// One piece of a transfer on the context's stream: n values at `at` of the device array(s),
// through the conversion scratch `conv` (FP32 forms).
hipError_t move_piece(fds_ctx *c, bool up, double *host, void *dev, void *comp, double *conv,
                      int64_t at, int64_t n) {
  const unsigned grid = (unsigned)((n + 255) / 256);
  if (c->elem == 8) {
    double *d = static_cast<double *>(dev) + at;
    return up ? hipMemcpyAsync(d, host, n * 8, hipMemcpyHostToDevice, c->stream)
              : hipMemcpyAsync(host, d, n * 8, hipMemcpyDeviceToHost, c->stream);
  }
  float *x = static_cast<float *>(dev) + at;
  float *k = comp ? static_cast<float *>(comp) + at : nullptr;
  if (up) {
    const hipError_t e = hipMemcpyAsync(conv, host, n * 8, hipMemcpyHostToDevice, c->stream);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_from_double, dim3(grid), dim3(256), 0, c->stream, conv, x, k, n);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_to_double, dim3(grid), dim3(256), 0, c->stream, conv, x, k, n);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return hipMemcpyAsync(host, conv, n * 8, hipMemcpyDeviceToHost, c->stream);
}

// Small arrays: converted here (a launch more costs what it saves) and copied by the runtime.
int transfer_small(fds_ctx *c, bool up, double *host, void *dev, void *comp, int64_t n) {
  const hipMemcpyKind kind = up ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost;
  if (c->elem == 8) {
    HIP_TRY(hipMemcpyAsync(up ? dev : host, up ? host : dev, n * 8, kind, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return 0;
  }
  std::vector<float> x(n), k(comp ? n : 0);
  if (up) {
    for (int64_t i = 0; i < n; ++i) {
      x[i] = (float)host[i];
      if (comp) k[i] = (float)((double)x[i] - host[i]);
    }
  }
  hipError_t e = hipMemcpyAsync(up ? dev : x.data(), up ? x.data() : dev, n * 4, kind, c->stream);
  if (e == hipSuccess && comp)
    e = hipMemcpyAsync(up ? comp : k.data(), up ? k.data() : comp, n * 4, kind, c->stream);
  const hipError_t done = hipStreamSynchronize(c->stream);   // (the vectors are in use until then)
  HIP_TRY(e);
  HIP_TRY(done);
  if (!up)
    for (int64_t i = 0; i < n; ++i) host[i] = comp ? (double)x[i] - (double)k[i] : (double)x[i];
  return 0;
}

// Large arrays go in chunks through pinned memory, copied by a few host threads and converted on
// the device: the runtime's own staging of pageable memory, and the conversion, are one thread's
// work.  Each thread owns two chunks, so one is copied while the other's transfer runs.  1000 steps
// of Thermal2D 4096^2 FP32-Kahan with the state there and back: 87.7 ms before, 22.8 ms so (16.5
// in the kernels); below 2^20 values a pass got up to 9 % slower.
constexpr int64_t kXferChunk = 1 << 18;      // values (2 MB)
constexpr int kXferThreads = 4;              // two chunks each
constexpr int kXferSlots = 2 * kXferThreads;
constexpr int64_t kXferLarge = 1 << 20;      // values from which an array takes this path
constexpr size_t kXferKept = 2;              // idle workspaces a device keeps

// What one large transfer works in: pinned chunks (16 MB), conversion scratch (FP32 forms, 16 MB)
// and the events after the chunks' copies.
struct Xfer {
  HostBuf pinned;
  DevBuf conv;
  hipEvent_t ev[kXferSlots] = {};
  ~Xfer() {
    for (auto e : ev)
      if (e) (void)hipEventDestroy(e);
  }
  hipError_t ready(bool convert) {
    constexpr size_t bytes = kXferSlots * kXferChunk * 8;
    hipError_t e = pinned.ensure(bytes);
    if (e == hipSuccess && convert) e = conv.ensure(bytes);
    for (auto &v : ev)
      if (e == hipSuccess && !v) e = hipEventCreateWithFlags(&v, hipEventDisableTiming);
    return e;
  }
};

// The workspaces between transfers.  A sweep of many large fields transfers one or two of them at
// a time, so they belong to the device and not to each field, and are freed with its last context.
// (The pool itself is never destroyed: the runtime may be gone when the process ends.)
struct XferPool {
  struct PerDevice {
    int contexts = 0;
    std::vector<Xfer *> idle;
  };
  std::mutex mu;
  std::map<int, PerDevice> devices;
};

XferPool &xfer_pool() {
  static XferPool *pool = new XferPool;
  return *pool;
}

void count_context(int device, int by) {
  std::vector<Xfer *> gone;
  XferPool &pool = xfer_pool();
  {
    std::lock_guard<std::mutex> lock(pool.mu);
    XferPool::PerDevice &d = pool.devices[device];
    d.idle.reserve(kXferKept);
    d.contexts += by;
    if (d.contexts == 0) gone.swap(d.idle);
  }
  for (auto *x : gone) delete x;
}

// A workspace, or null where its memory is not to be had.
Xfer *take_xfer(const fds_ctx *c) {
  Xfer *x = nullptr;
  XferPool &pool = xfer_pool();
  {
    std::lock_guard<std::mutex> lock(pool.mu);
    auto &idle = pool.devices[c->device].idle;
    if (!idle.empty()) {
      x = idle.back();
      idle.pop_back();
    }
  }
  if (!x) x = new Xfer;
  if (x->ready(c->elem == 4) == hipSuccess) return x;
  (void)hipGetLastError();
  delete x;
  return nullptr;
}

void give_xfer(const fds_ctx *c, Xfer *x) {
  XferPool &pool = xfer_pool();
  {
    std::lock_guard<std::mutex> lock(pool.mu);
    auto &idle = pool.devices[c->device].idle;
    if (idle.size() < kXferKept) {
      idle.push_back(x);
      return;
    }
  }
  delete x;
}

int transfer(fds_ctx *c, bool up, double *host, void *dev, void *comp, int64_t n) {
  if (n < kXferLarge) return transfer_small(c, up, host, dev, comp, n);
  Xfer *const ws = take_xfer(c);
  if (!ws) return transfer_small(c, up, host, dev, comp, n);
  double *const pinned = static_cast<double *>(ws->pinned.p), *const conv = ws->conv.as<double>();
  const int64_t chunks = (n + kXferChunk - 1) / kXferChunk;
  std::atomic<int> err{(int)hipSuccess};
  const auto worker = [&](int w) {
    hipError_t e = hipSetDevice(c->device);
    int64_t prev = -1;        // the chunk whose transfer is in flight
    int i = 0, before = 0;    // its slot: before
    const auto count = [&](int64_t k) { return std::min(kXferChunk, n - k * kXferChunk); };
    const auto finish = [&]() {     // (down) the chunk in flight to the caller's array
      if (prev < 0 || e != hipSuccess) return;
      e = hipEventSynchronize(ws->ev[before]);
      if (e == hipSuccess)
        std::memcpy(host + prev * kXferChunk, pinned + before * kXferChunk, count(prev) * 8);
    };
    for (int64_t k = w; k < chunks && e == hipSuccess; k += kXferThreads, ++i) {
      const int slot = 2 * w + (i & 1);
      double *pin = pinned + slot * kXferChunk;
      if (up) {
        if (i >= 2) e = hipEventSynchronize(ws->ev[slot]);
        std::memcpy(pin, host + k * kXferChunk, count(k) * 8);
      }
      if (e == hipSuccess)
        e = move_piece(c, up, pin, dev, comp, conv + slot * kXferChunk, k * kXferChunk, count(k));
      if (e == hipSuccess) e = hipEventRecord(ws->ev[slot], c->stream);
      if (!up) finish();
      prev = k;
      before = slot;
    }
    if (!up) finish();
    if (e != hipSuccess) err = (int)e;
  };
  std::vector<std::thread> extra;
  int started = 1;
  try {
    extra.reserve(kXferThreads - 1);
    for (; started < kXferThreads; ++started) extra.emplace_back(worker, started);
  } catch (...) {        // no more threads: the caller's does their chunks
  }
  worker(0);
  for (int w = started; w < kXferThreads; ++w) worker(w);
  for (auto &t : extra) t.join();
  const hipError_t done = hipStreamSynchronize(c->stream);     // (the workspace is in use until then)
  give_xfer(c, ws);
  HIP_TRY((hipError_t)err.load());
  HIP_TRY(done);
  return 0;
}

int to_device(fds_ctx *c, void *dst, const double *src, int64_t n) {
  return transfer(c, true, const_cast<double *>(src), dst, nullptr, n);
}

template <typename T>
void fill_args(const fds_ctx *c, fds::StepArgs<T> &a, int parity) {
  std::memset(&a, 0, sizeof a);
  a.nx = (int32_t)c->nx;
  a.ny = (int32_t)c->ny;
  a.n = c->n;
  a.tiles_x = c->tiles_x;
  a.ntiles = c->ntiles;
  for (int k = 0; k < 3; ++k) {
    const Comp &cp = c->comp[k];
    const bool pp = cp.accumulated || c->family != kThermal || k == 0;
    const int rd = pp ? parity : 0, wr = pp ? parity ^ 1 : 0;
    a.in[k] = cp.buf[rd].as<const T>();
    a.out[k] = cp.buf[wr].as<T>();
    a.cin[k] = cp.cbuf[rd].as<const T>();
    a.cout[k] = cp.cbuf[wr].as<T>();
    const bool has_b = !cp.cells.empty();
    a.bev[k].ptr = has_b ? cp.ev_ptr.as<const int32_t>() : c->zero_ptr.as<const int32_t>();
    a.bev[k].pos = cp.ev_pos.as<const int32_t>();
    a.bev[k].id = cp.ev_id.as<const int32_t>();
    a.prog[k].ptr = cp.d_ptr.as<const int32_t>();
    a.prog[k].a = cp.d_a.as<const double>();
    a.prog[k].off = cp.d_off.as<const int64_t>();
    a.prog[k].stride = cp.d_stride.as<const int64_t>();
    a.prog[k].table = cp.d_table.as<const double>();
    const bool has_o = !cp.out_cells.empty();
    a.outp[k].ev.ptr = has_o ? cp.oev_ptr.as<const int32_t>() : c->zero_ptr.as<const int32_t>();
    a.outp[k].ev.pos = cp.oev_pos.as<const int32_t>();
    a.outp[k].ev.id = cp.oev_id.as<const int32_t>();
    a.outp[k].buf = cp.obuf.as<double>();
    a.outp[k].m = (int32_t)cp.out_cells.size();
    a.lhead[k] = cp.lhead.p;
    a.ohead[k] = cp.ohead.p;
  }
  for (int s = 0; s < FDS_NUM_COEFF; ++s)
    a.coef[s] = c->coef_set[s] ? c->coef[s].as<const T>() : c->zeros.as<const T>();
  if (c->family != kNonlinear) {
    // cleared y slots alias their x slot, except for 1D models whose y terms are zero
    const int pairs[3][2] = {{0, 1}, {2, 3}, {4, 5}};
    for (auto &pr : pairs)
      if (!c->coef_set[pr[1]]) a.coef[pr[1]] = c->one_d ? c->zeros.as<const T>() : a.coef[pr[0]];
  }
  for (int s = 0; s < FDS_NUM_SCALARS; ++s) a.s[s] = c->s[s];
  a.dyn = c->dyn.as<const int64_t>();
  a.flags = (c->iso_b ? fds::kFlagIsoB : 0) | (c->iso_k ? fds::kFlagIsoK : 0);
  a.strip_h = c->ty;
  a.ghost = c->ghost;
  a.ghost_rows = c->ghost_rows;
  a.sx = c->sx;
  if (c->fused) {
    a.fev = c->fused_ev;
    a.pal_idx = c->pal_idx.as<const uint8_t>();
    a.pal = c->pal.as<const T>();
    a.npal = c->npal;
  }
}

// ring_ok: the arrays suit an LDS-ring shape's 16-byte row loads (else its register-path twin
// runs, same bits).
fds::LaunchFn pick_launch(const fds_ctx *c, int stages, bool ring_ok = true) {
  const int t = c->shape;
  if (c->fused && c->lossy && c->family == kAcoustic)
    return c->ks->fused_lossy[c->axi ? 1 : (c->iso_b && c->iso_k && !c->coef_set[FDS_C_MY]) ? 2 : 0]
                             [stages - 1];
  if (c->fused) {
    const int v = c->axi ? 1 : (c->iso_b && c->iso_k) ? 2 : 0;
    return c->ks->fused[c->family == kThermal ? 1 : 0][c->npal > 0 ? 1 : 0][v][stages - 1];
  }
  if (c->streaming && c->lossy) {
    // variant: axial-symmetric, isotropic (B, K and M y slots alias the x ones), plain
    const int v = c->axi ? 1 : (c->iso_b && c->iso_k && !c->coef_set[FDS_C_MY]) ? 2 : 0;
    const int s0 = t - fds::kNumTiles;
    return c->ks->stream_lossy[ring_ok ? s0 : fds::ring_fallback(s0)][v];
  }
  if (c->streaming) {
    const int s0 = t - fds::kNumTiles, f = stages - 1;
    const int s = ring_ok ? s0 : fds::ring_fallback(s0);
    // variant: axial-symmetric, isotropic (y coefficient slots alias the x ones), plain
    const int v = c->axi ? 1 : (c->iso_b && c->iso_k) ? 2 : 0;
    return c->family == kThermal ? c->ks->stream_thermal[s][v][f]
                                 : c->ks->stream_acoustic[s][v][f];
  }
  switch (c->family) {
    case kAcoustic: return c->ks->acoustic[t][c->axi ? 1 : 0][c->lossy ? 1 : 0];
    case kThermal: return c->ks->thermal[t][c->axi ? 1 : 0];
    default: return c->ks->nonlinear;
  }
}

// Flow along x (pyfds/acoustic_flow.py:49-57): after the step at `step`, every row r whose
// period divides the step (period 0 always; numpy's int % 0 is 0) moves one cell to +x and
// takes a zero at its start, in every state array (and compensation array) of the step's
// output.  One workgroup per row shifts it in place, chunk by chunk from the right end, so
// each chunk reads its left neighbour before that neighbour is overwritten.
template <typename T>
__global__ __launch_bounds__(256) void k_flow_shift(T *a0, T *a1, T *a2, T *c0, T *c1, T *c2,
                                                    int nx, const int64_t *__restrict__ period,
                                                    const int64_t *__restrict__ dyn, int k) {
  const int r = blockIdx.x;
  const int64_t step = dyn[0] + k;
  const int64_t p = period[r];
  const int64_t ap = p < 0 ? -p : p;
  if (!(ap == 0 || step % ap == 0)) return;
  T *rows[6] = {a0, a1, a2, c0, c1, c2};
  for (int q = 0; q < 6; ++q) {
    T *row = rows[q];
    if (!row) continue;
    row += (int64_t)r * nx;
    for (int s = ((nx - 1) / 256) * 256; s >= 0; s -= 256) {
      const int i = s + (int)threadIdx.x;
      const T v = (i >= 1 && i < nx) ? row[i - 1] : T(0);
      __syncthreads();
      if (i < nx) row[i] = v;
      __syncthreads();
    }
  }
}

// Step counters at the start of a run, written in stream order (no host round trip, so a run
// may be enqueued behind one still executing).
__global__ void k_set_dyn(int64_t *dyn, int64_t start) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    dyn[0] = start;
    dyn[1] = 0;
  }
}

__global__ void k_advance(int64_t *dyn, int64_t by) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    dyn[0] += by;
    dyn[1] += by;
  }
}

// Zero the first n work-queue counters (one per launch of a run).
__global__ __launch_bounds__(256) void k_queue_reset(unsigned *q, int n) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) q[i] = 0u;
}

// Non-finite detection.  dyn[kDynNonfinite] holds the smallest (step * 4 + component) over the
// scans that met a NaN or an infinity in a component's state (all bits set: none), where step
// counts the steps done when the scan ran.  A scan reads the state once (grid-stride loop);
// only lanes that meet a non-finite value touch the flag.
constexpr int kDynNonfinite = 4;
constexpr uint64_t kNoNonfinite = ~0ull;
constexpr int64_t kNonfiniteEvery = 50;   // resident 1D engine: steps between scans (at least)

__global__ void k_nonfinite_reset(int64_t *dyn) {
  if (threadIdx.x == 0 && blockIdx.x == 0)
    reinterpret_cast<unsigned long long *>(dyn)[kDynNonfinite] = kNoNonfinite;
}

template <typename T>
__global__ __launch_bounds__(256) void k_nonfinite_scan(const T *__restrict__ x, int64_t n,
                                                        int comp,
                                                        const int64_t *__restrict__ base,
                                                        int64_t add, int64_t *flag_dyn) {
  bool bad = false;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    bad |= !__builtin_isfinite(x[i]);
  if (bad)
    atomicMin(reinterpret_cast<unsigned long long *>(flag_dyn) + kDynNonfinite,
              (unsigned long long)((base[0] + add) * 4 + comp));
}

// Launch one step: reads state buffer `parity`, writes parity^1.
template <typename T>
void launch_lbc(fds_ctx *, const fds::StepArgs<T> &) {}

template <>
void launch_lbc<float>(fds_ctx *c, const fds::StepArgs<float> &a) {
  fds::LbcStep st;
  for (int k = 0; k < 3; ++k) {
    st.prev[k] = a.in[k];
    st.cur[k] = a.out[k];
    st.cur_comp[k] = is_kahan(c) ? a.cout[k] : nullptr;
    st.cs[k] = c->lbc_cs[k];
  }
  st.w1 = c->lbc_w1;
  st.w2 = c->lbc_w2;
  st.g = (int)c->nx;
  st.l = c->lbc_layer;
  fds::launch_lbc_step(st, c->stream);
}

template <typename T>
void launch_ring(fds_ctx *, const fds::StepArgs<T> &, int) {}

template <>
void launch_ring<float>(fds_ctx *c, const fds::StepArgs<float> &a, int stages) {
  fds::LbcRing r{};
  for (int k = 0; k < 3; ++k) {
    r.in[k] = a.in[k];
    r.out[k] = a.out[k];
    r.rows[k] = a.outp[k].buf;
    r.m[k] = a.outp[k].m;
    r.cs[k] = c->lbc_cs[k];
  }
  r.b = a.coef[FDS_C_BX];
  r.k = a.coef[FDS_C_KX];
  r.packed = c->lbc_packed.p;
  r.cells = c->lbc_cells.p;
  r.rec = c->lbc_rec.as<const fds::LbcRec>();
  r.nrec = c->lbc_nrec;
  r.dyn = a.dyn;
  r.row = a.k;
  r.g = (int)c->nx;
  r.stages = stages;
  r.depth = c->fuse;
  fds::launch_lbc_ring(r, c->stream);
}

// Time steps per launch: the streaming shapes' fused stage count (one step per launch when a
// per-step learned boundary follows the step kernel).
int step_group(const fds_ctx *c) {
  return (c->streaming && (!c->lbc_w1 || c->lbc_ring) && !c->flow) ? c->fuse : 1;
}

// Launch `stages` fused steps (1 <= stages <= step_group(c)) starting at step k of the launch
// sequence: reads state buffer `parity`, writes parity^1.
template <typename T>
int launch_step(fds_ctx *c, int parity, int k, bool store, int stages) {
  fds::StepArgs<T> a;
  fill_args<T>(c, a, parity);
  a.k = k;
  if (store) a.flags |= fds::kFlagStore;
  bool ring_ok = true;
  if (c->streaming && !c->fused && fds::kStreamShapes[c->shape - fds::kNumTiles][5]) {
    // LDS-ring kernels load 16-byte chunks of rows: rows must start on 16-byte boundaries and
    // every array they read must be 16-byte aligned (whole device allocations are); otherwise
    // the register-path kernel of the same tiling runs
    ring_ok = c->nx % (16 / (int)c->elem) == 0;
    for (int k = 0; k < 3; ++k)
      ring_ok = ring_ok && ((uintptr_t)a.in[k] & 15) == 0 && ((uintptr_t)a.cin[k] & 15) == 0;
    for (int q = 0; q < FDS_NUM_COEFF; ++q) ring_ok = ring_ok && ((uintptr_t)a.coef[q] & 15) == 0;
  }
  const int nb = fds::xcd_grid(c->ntiles) + (c->fused ? fds::xcd_grid(c->fused_ev.nslots) : 0);
  pick_launch(c, stages, ring_ok)(&a, nb, lds_bytes(c), c->stream);
  HIP_TRY(hipGetLastError());
  if (c->flow) {
    hipLaunchKernelGGL(k_flow_shift<T>, dim3((unsigned)c->ny), dim3(256), 0, c->stream,
                       a.out[0], a.out[1], a.out[2], a.cout[0], a.cout[1], a.cout[2],
                       (int)c->nx, c->flow_period.as<const int64_t>(), a.dyn, k);
    HIP_TRY(hipGetLastError());
  }
  if (c->lbc_w1) {
    if (stages > 1) launch_ring<T>(c, a, stages);
    else launch_lbc<T>(c, a);
    HIP_TRY(hipGetLastError());
  }
  return 0;
}

// Launch the resident 1D kernel for `steps` steps starting at step k of the run.
template <typename T>
int launch_line(fds_ctx *c, int parity, int k, int steps) {
  fds::StepArgs<T> a;
  fill_args<T>(c, a, parity);
  a.k = k;
  a.steps = steps;
  a.strip_h = c->line_seg;
  a.ghost = c->line_ghost;
  const int fam = c->family == kNonlinear ? fds::kLineNonlinear
                  : c->family == kThermal ? fds::kLineThermal
                  : (c->lossy ? fds::kLineAcousticLossy : fds::kLineAcoustic);
  c->ks->line[c->line_var][fam](&a, c->line_wgs, c->line_threads, c->stream);
  HIP_TRY(hipGetLastError());
  return 0;
}

int launch_step_any(fds_ctx *c, int parity, int k, bool store, int stages = 1) {
  return c->elem == 8 ? launch_step<double>(c, parity, k, store, stages)
                      : launch_step<float>(c, parity, k, store, stages);
}

// Scan component k's state (buffer `parity` where the component ping-pongs) for non-finite
// values on `stream`; a hit records step base[0] + add in flag_dyn.
int scan_nonfinite(const fds_ctx *c, int k, int parity, const int64_t *base, int64_t add,
                   int64_t *flag_dyn, hipStream_t stream) {
  const Comp &cp = c->comp[k];
  if (!cp.present) return 0;
  const bool pp = cp.accumulated || c->family != kThermal || k == 0;
  const void *x = cp.buf[pp ? parity : 0].p;
  const unsigned nb = (unsigned)std::min<int64_t>((c->n + 1023) / 1024, 2048);
  if (c->elem == 8)
    hipLaunchKernelGGL(k_nonfinite_scan<double>, dim3(nb), dim3(256), 0, stream,
                       static_cast<const double *>(x), c->n, k, base, add, flag_dyn);
  else
    hipLaunchKernelGGL(k_nonfinite_scan<float>, dim3(nb), dim3(256), 0, stream,
                       static_cast<const float *>(x), c->n, k, base, add, flag_dyn);
  HIP_TRY(hipGetLastError());
  return 0;
}

int scan_all_nonfinite(const fds_ctx *c, int parity, const int64_t *base, int64_t add,
                       hipStream_t stream) {
  for (int k = 0; k < 3; ++k)
    if (int rc = scan_nonfinite(c, k, parity, base, add, c->dyn.as<int64_t>(), stream))
      return rc;
  return 0;
}

// Copy the context's non-finite result to staging slot `slot` (stream order).
int stage_nonfinite(fds_ctx *c, int slot, hipStream_t stream) {
  if (!c->nf_check) return 0;
  HIP_TRY(c->nf_stage.ensure((kMaxFlights + 1) * sizeof(uint64_t)));
  HIP_TRY(hipMemcpyAsync(static_cast<uint64_t *>(c->nf_stage.p) + slot,
                         c->dyn.as<uint64_t>() + kDynNonfinite, sizeof(uint64_t),
                         hipMemcpyDeviceToHost, stream));
  return 0;
}

// After the copy of stage_nonfinite(c, slot) completed: FDS_E_NONFINITE if a scan met a NaN
// or an infinity.
int check_nonfinite(const fds_ctx *c, int slot) {
  if (!c->nf_check || !c->nf_stage.p) return 0;
  const uint64_t v = static_cast<const uint64_t *>(c->nf_stage.p)[slot];
  if (v == kNoNonfinite) return 0;
  return fail(FDS_E_NONFINITE, "non-finite value in component %d, found after step %lld",
              (int)(v & 3), (long long)(v >> 2));
}

int get_graph(fds_ctx *c, int chunk, int parity, hipGraphExec_t *out) {
  if (c->graph_generation != c->generation) {
    drop_graphs(c);
    c->graph_generation = c->generation;
  }
  auto key = std::make_pair(chunk, parity);
  auto it = c->graphs.find(key);
  if (it != c->graphs.end()) {
    *out = it->second;
    return 0;
  }
  // capture on an idle stream (an asynchronous run may still be executing)
  HIP_TRY(hipStreamSynchronize(c->stream));
  HIP_TRY(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
  int rc = 0;
  const int grp = step_group(c);   // chunk is a multiple of grp
  for (int k = 0; k < chunk && rc == 0; k += grp)
    rc = launch_step_any(c, parity ^ ((k / grp) & 1), k, false, grp);
  if (rc == 0 && c->nf_check)       // the first component after the chunk
    rc = scan_nonfinite(c, 0, parity ^ ((chunk / grp) & 1), c->dyn.as<const int64_t>(), chunk,
                        c->dyn.as<int64_t>(), c->stream);
  if (rc == 0) {
    hipLaunchKernelGGL(k_advance, dim3(1), dim3(64), 0, c->stream, c->dyn.as<int64_t>(),
                       (int64_t)chunk);
  }
  hipGraph_t g = nullptr;
  hipError_t e = hipStreamEndCapture(c->stream, &g);
  if (rc) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  if (e != hipSuccess) return fail(FDS_E_HIP, "graph capture failed: %s", hipGetErrorString(e));
  hipGraphExec_t ex = nullptr;
  e = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
  if (e != hipSuccess) {
    (void)hipGraphDestroy(g);
    return fail(FDS_E_HIP, "graph instantiate failed: %s", hipGetErrorString(e));
  }
  c->graph_objs.push_back(g);
  c->graphs[key] = ex;
  // the graph's device-side copy now, not on its first launch inside a run
  HIP_TRY(hipGraphUpload(ex, c->stream));
  *out = ex;
  return 0;
}

// Material classes.  Cells with the same coefficients (by their bits) are one class; a field whose
// cells form fewer than kPalMax classes gets an array of class numbers, one byte a cell, and a
// table of the classes' coefficients.  The table is a hash table of the classes' first cells found:
// a wave looks the coefficients of its first cell without a class up, gives the class to all its
// cells that have them, and goes on with the next such cell.  A class that finds no slot ends the
// search: the field has too many.
//
// One pass over the coefficients, and one launch whatever the number of classes: bound by the
// latency of its lookups on small fields.  A commit takes 39 us with it, 50000 cells of one
// material or of 200 (0.7 ms for the latter with a pass a class; 65 us with the slots of a lookup
// tried one after the other).
template <typename T>
struct PalCoefs {
  const T *c[fds::kPalSlots];   // in the table's order
};

constexpr int kPalClasses = fds::kPalMax - 1;     // slots; tab[kPalClasses]: too many classes
static_assert(kPalClasses == 63, "a slot a lane");

__device__ __forceinline__ uint32_t lane_bits(uint32_t v, int lane) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
}
__device__ __forceinline__ uint64_t lane_bits(uint64_t v, int lane) {
  return (uint64_t)lane_bits((uint32_t)(v >> 32), lane) << 32 | lane_bits((uint32_t)v, lane);
}

template <typename T, int NC>
__global__ __launch_bounds__(256) void k_classes(PalCoefs<T> pc, int64_t n, uint8_t *idx, T *pal,
                                                 unsigned *tab) {
  using B = std::conditional_t<sizeof(T) == 8, uint64_t, uint32_t>;
  const int lane = threadIdx.x & 63;
  const int64_t stride = (int64_t)gridDim.x * 256;
  B last[NC] = {};       // the class looked up last (0: none)
  int cls = 0;
  for (int64_t i0 = (int64_t)blockIdx.x * 256 + (threadIdx.x & ~63); i0 < n; i0 += stride) {
    const int64_t i = i0 + lane;
    const bool in = i < n;
    B own[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) own[k] = in ? __builtin_bit_cast(B, pc.c[k][i]) : B(0);
    int mine = 0;
    for (uint64_t left = __ballot(in); left;) {
      const int lead = __builtin_ctzll(left);
      B key[NC];
      bool same = cls != 0;
#pragma unroll
      for (int k = 0; k < NC; ++k) {
        key[k] = lane_bits(own[k], lead);
        same = same && key[k] == last[k];
      }
      if (!same) {
        uint64_t h = 0;
#pragma unroll
        for (int k = 0; k < NC; ++k) {
          h = (h ^ key[k]) * 0x9e3779b97f4a7c15ull;      // (the golden ratio's bits, odd)
          h ^= h >> 29;
          last[k] = key[k];
        }
        const int home = (int)(((h >> 32) * kPalClasses) >> 32);
        // all slots at a time, one a lane (the last lane: too many); each turn without a class has
        // at least one slot more to compare, which another wave took meanwhile
        cls = 0;
        unsigned f = 0;
        while (!cls) {
          if (f == 0)
            f = __hip_atomic_load(tab + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          if (lane_bits(f, kPalClasses)) return;
          bool eq = f != 0 && lane < kPalClasses;
          if (eq) {
#pragma unroll
            for (int k = 0; k < NC; ++k)
              eq = eq && __builtin_bit_cast(B, pc.c[k][f - 1]) == key[k];
          }
          const uint64_t hit = __ballot(eq), empty = __ballot(f == 0 && lane < kPalClasses);
          if (hit) {
            cls = __builtin_ctzll(hit) + 1;
          } else if (!empty) {
            if (lane == lead)
              __hip_atomic_store(tab + kPalClasses, 1u, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
            return;
          } else {
            // the first empty slot from the key's own on: waves with one key try one slot
            const uint64_t after = empty >> home << home;
            const int s = __builtin_ctzll(after ? after : empty);
            unsigned was = 0;
            if (lane == lead) was = atomicCAS(tab + s, 0u, (unsigned)i + 1);
            was = lane_bits(was, lead);
            if (was) {
              if (lane == s) f = was;
              continue;
            }
            cls = s + 1;
            if (lane == lead) {
#pragma unroll
              for (int k = 0; k < NC; ++k)
                pal[cls * fds::kPalSlots + k] = __builtin_bit_cast(T, own[k]);
            }
          }
        }
      }
      bool eq = in;
#pragma unroll
      for (int k = 0; k < NC; ++k) eq = eq && own[k] == key[k];
      if (eq) mine = cls;
      left &= ~__ballot(eq);
    }
    if (in) idx[i] = (uint8_t)mine;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_pal_init(T *pal, int coefs, unsigned *tab, int slots) {
  for (int i = threadIdx.x; i < coefs; i += 256) pal[i] = T(0);
  for (int i = threadIdx.x; i < slots; i += 256) tab[i] = 0u;
}

template <typename T>
int find_classes(fds_ctx *c) {
  const bool lossy = c->lossy && c->family == kAcoustic;
  const auto slot = [&](int k, int alias) {
    return c->coef_set[k] ? c->coef[k].as<const T>()
                          : alias >= 0 ? c->coef[alias].as<const T>() : c->zeros.as<const T>();
  };
  // (thermal: Q, G in the places of B, K)
  const PalCoefs<T> pc{{slot(2, -1), slot(0, -1), slot(3, 2), slot(1, 0), slot(4, -1), slot(5, 4),
                        slot(6, -1), slot(7, -1)}};
  constexpr int kCoefs = fds::kPalMax * fds::kPalSlots;
  HIP_TRY(c->pal_idx.ensure(c->n));
  HIP_TRY(c->pal.ensure(kCoefs * sizeof(T) + (kPalClasses + 1) * sizeof(unsigned)));
  unsigned *const tab = reinterpret_cast<unsigned *>(c->pal.as<T>() + kCoefs);
  hipLaunchKernelGGL(k_pal_init<T>, dim3(1), dim3(256), 0, c->stream, c->pal.as<T>(), kCoefs, tab,
                     kPalClasses + 1);
  const unsigned nb = (unsigned)std::min<int64_t>((c->n + 1023) / 1024, 2048);
  hipLaunchKernelGGL((lossy ? k_classes<T, 8> : k_classes<T, 4>), dim3(nb), dim3(256), 0, c->stream,
                     pc, c->n, c->pal_idx.as<uint8_t>(), c->pal.as<T>(), tab);
  HIP_TRY(hipGetLastError());
  unsigned over = 0;
  HIP_TRY(hipMemcpyAsync(&over, tab + kPalClasses, sizeof over, hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  if (!over) c->npal = fds::kPalMax;
  return 0;
}

// The material classes of a field that may run on the fused engines.
int ready_classes(fds_ctx *c) {
  c->npal = 0;
  if (c->tile >= 0 || c->family == kNonlinear || !fuse_reach(c)) return 0;
  return c->elem == 8 ? find_classes<double>(c) : find_classes<float>(c);
}

// A field that a coupling stepped last (one step per launch, coefficients cell by cell) runs by
// itself again: the layout and classes of its coefficients as the coupling left them.
int leave_coupling(fds_ctx *c) {
  if (!c->coupled) return 0;
  c->coupled = false;
  if (c->tile >= 0 || !fuse_reach(c)) return 0;      // (its engine is the same either way)
  if (!c->npal)
    if (int rc = ready_classes(c)) return rc;
  if (int rc = choose_tiles(c)) return rc;
  touch(c);
  return 0;
}

int check_ctx(fds_ctx *c) {
  if (!c) return fail(FDS_E_ARG, "null context");
  hipError_t e = hipSetDevice(c->device);
  if (e != hipSuccess) return fail(FDS_E_HIP, "hipSetDevice: %s", hipGetErrorString(e));
  return 0;
}

// Setters, synchronous runs and output reads wait until the asynchronous runs are taken.
int check_idle(fds_ctx *c) {
  if (int rc = check_ctx(c)) return rc;
  if (!c->flights.empty() || c->batch_flights)
    return fail(FDS_E_STATE, "asynchronous runs in flight: take them first");
  return 0;
}

int check_comp(fds_ctx *c, int comp) {
  if (comp < 0 || comp > 2 || !c->comp[comp].present)
    return fail(FDS_E_ARG, "component %d does not exist for this model", comp);
  return 0;
}

}  // namespace

extern "C" {

const char *fds_last_error(void) { return g_last_error.c_str(); }

const char *fds_version(void) { return "pyfds_amd 0.1 (gfx950)"; }

int fds_tile_count(void) { return fds::kNumTiles + fds::kNumStream; }

int fds_engine(fds_ctx *c) {
  if (int rc = check_ctx(c)) return rc;
  if (c->line) return 2;
  if (c->family == kNonlinear) return 3;
  return c->streaming ? 1 : 0;
}

int fds_steps_per_launch(fds_ctx *c) {
  if (int rc = check_ctx(c)) return rc;
  return step_group(c);
}

int fds_tile_engine(int i) {
  if (i < 0 || i >= fds::kNumTiles + fds::kNumStream)
    return fail(FDS_E_ARG, "tile index %d out of range", i);
  return i >= fds::kNumTiles ? 1 : 0;
}

int fds_tile_traits(int i, int *steps, int *nontemporal, int *prefetch, int *lds_ring) {
  if (i < 0 || i >= fds::kNumTiles + fds::kNumStream)
    return fail(FDS_E_ARG, "tile index %d out of range", i);
  if (!steps || !nontemporal || !prefetch || !lds_ring) return fail(FDS_E_ARG, "null argument");
  const bool st = i >= fds::kNumTiles;
  *steps = st ? fds::kStreamShapes[i - fds::kNumTiles][2] : 1;
  *nontemporal = st ? fds::kStreamShapes[i - fds::kNumTiles][3] : 0;
  *prefetch = st ? fds::kStreamShapes[i - fds::kNumTiles][4] : 0;
  *lds_ring = st ? fds::kStreamShapes[i - fds::kNumTiles][5] : 0;
  return 0;
}

int fds_tile_shape(int i, int *tx, int *ty) {
  if (i < 0 || i >= fds::kNumTiles + fds::kNumStream)
    return fail(FDS_E_ARG, "tile index %d out of range", i);
  shape_of(i, tx, ty);
  return 0;
}

int fds_create(fds_ctx **out, int model, int form, int64_t nx, int64_t ny, int device) {
  g_last_error.clear();
  if (!out) return fail(FDS_E_ARG, "null output pointer");
  *out = nullptr;
  if (form < FDS_FP64 || form > FDS_FP32_KAHAN) return fail(FDS_E_ARG, "unknown form %d", form);
  if (nx < 1 || ny < 1) return fail(FDS_E_ARG, "grid must be at least 1x1");
  // kernels index cells with 32-bit ints, including look-ahead rows past the last strip
  if (nx * (ny + 40) + 1024 > (int64_t)std::numeric_limits<int32_t>::max())
    return fail(FDS_E_ARG, "grid of %lld cells exceeds the 32-bit cell index",
                (long long)(nx * ny));
  auto *c = new fds_ctx();
  c->model = model;
  c->form = form;
  c->device = device;
  c->n = nx * ny;
  c->nx = nx;
  c->ny = ny;
  switch (model) {
    case FDS_ACOUSTIC1D: c->family = kAcoustic; c->one_d = true; break;
    case FDS_ACOUSTIC2D: c->family = kAcoustic; break;
    case FDS_ACOUSTIC_AXI: c->family = kAcoustic; c->axi = true; break;
    case FDS_THERMAL1D: c->family = kThermal; c->one_d = true; break;
    case FDS_THERMAL2D: c->family = kThermal; break;
    case FDS_THERMAL_AXI: c->family = kThermal; c->axi = true; break;
    case FDS_IDEALGAS1D:
    case FDS_ACOUSTIC2ND1D: c->family = kNonlinear; break;
    default: delete c; return fail(FDS_E_ARG, "unknown model %d", model);
  }
  if ((c->one_d || c->family == kNonlinear) && ny != 1) {
    delete c;
    return fail(FDS_E_ARG, "1D models need ny = 1");
  }
  if (c->one_d || c->family == kNonlinear) {
    c->nx = c->n;
    c->ny = 1;
  }
  c->elem = (form == FDS_FP64) ? 8 : 4;
  c->ks = form == FDS_FP64 ? &fds::kernels_f64()
                           : (form == FDS_FP32 ? &fds::kernels_f32() : &fds::kernels_k32());
  hipError_t e = hipSetDevice(device);
  if (e != hipSuccess) {
    delete c;
    return fail(FDS_E_HIP, "hipSetDevice(%d): %s", device, hipGetErrorString(e));
  }
  e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
  if (e != hipSuccess) {
    delete c;
    return fail(FDS_E_HIP, "hipStreamCreate: %s", hipGetErrorString(e));
  }
  count_context(device, 1);
  int cus = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess &&
      cus > 0)
    c->num_cu = cus;
  // components: all three exist for every model (1D linear models carry an inert third one)
  for (int k = 0; k < 3; ++k) {
    Comp &cp = c->comp[k];
    cp.present = true;
    cp.accumulated = (c->family != kThermal) ? !(c->family == kNonlinear && k == 0) : (k == 0);
    const int nbuf = (c->family == kThermal && k > 0) ? 1 : 2;
    for (int b = 0; b < nbuf; ++b) {
      if (cp.buf[b].ensure(c->n * c->elem) != hipSuccess ||
          hipMemsetAsync(cp.buf[b].p, 0, c->n * c->elem, c->stream) != hipSuccess) {
        fds_destroy(c);
        return fail(FDS_E_HIP, "out of device memory for %lld cells", (long long)c->n);
      }
      if (form == FDS_FP32_KAHAN && cp.accumulated) {
        if (cp.cbuf[b].ensure(c->n * c->elem) != hipSuccess ||
            hipMemsetAsync(cp.cbuf[b].p, 0, c->n * c->elem, c->stream) != hipSuccess) {
          fds_destroy(c);
          return fail(FDS_E_HIP, "out of device memory (compensation)");
        }
      }
    }
  }
  if (c->zeros.ensure(c->n * c->elem) != hipSuccess ||
      hipMemsetAsync(c->zeros.p, 0, c->n * c->elem, c->stream) != hipSuccess ||
      c->dyn.ensure(64) != hipSuccess) {
    fds_destroy(c);
    return fail(FDS_E_HIP, "out of device memory");
  }
  c->s[FDS_S_DX] = 1.0;
  c->s[FDS_S_HALF_DX] = 0.5;
  int rc = choose_tiles(c);
  if (rc) {
    fds_destroy(c);
    return rc;
  }
  if (hipStreamSynchronize(c->stream) != hipSuccess) {
    fds_destroy(c);
    return fail(FDS_E_HIP, "stream synchronize failed");
  }
  *out = c;
  return 0;
}

int fds_destroy(fds_ctx *c) {
  if (!c) return 0;
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  drop_graphs(c);
  if (c->ev0) (void)hipEventDestroy(c->ev0);
  if (c->ev1) (void)hipEventDestroy(c->ev1);
  for (auto &set : c->fev)
    for (auto e : set)
      if (e) (void)hipEventDestroy(e);
  if (c->stream) {
    (void)hipStreamDestroy(c->stream);
    count_context(c->device, -1);
  }
  delete c;
  return 0;
}

int fds_set_scalars(fds_ctx *c, const double *s, int n) {
  if (int rc = check_idle(c)) return rc;
  if (n < 0 || n > FDS_NUM_SCALARS) return fail(FDS_E_ARG, "bad scalar count %d", n);
  for (int i = 0; i < n; ++i) c->s[i] = s[i];
  touch(c);
  return 0;
}

int fds_set_coeff(fds_ctx *c, int slot, const double *data, int64_t n) {
  if (int rc = check_idle(c)) return rc;
  if (slot < 0 || slot >= FDS_NUM_COEFF) return fail(FDS_E_ARG, "bad coefficient slot %d", slot);
  if (n == 0) {
    c->coef[slot].release();
    c->coef_set[slot] = false;
  } else {
    if (n != c->n) return fail(FDS_E_ARG, "coefficient needs %lld values, got %lld",
                               (long long)c->n, (long long)n);
    HIP_TRY(c->coef[slot].ensure(n * c->elem));
    if (int rc = to_device(c, c->coef[slot].p, data, n)) return rc;
    c->coef_set[slot] = true;
  }
  c->committed = false;
  touch(c);
  return 0;
}

int fds_commit(fds_ctx *c) {
  if (int rc = check_idle(c)) return rc;
  if (c->family == kAcoustic) {
    if (!c->coef_set[FDS_C_KX] || !c->coef_set[FDS_C_BX])
      return fail(FDS_E_STATE, "acoustic coefficients K and B must be set");
    c->lossy = c->coef_set[FDS_C_MX];
    if (c->axi && c->lossy && (!c->coef_set[FDS_C_MC] || !c->coef_set[FDS_C_MT]))
      return fail(FDS_E_STATE, "lossy Axi field needs the MC and MT coefficients");
  } else if (c->family == kThermal) {
    if (!c->coef_set[FDS_C_GX] || !c->coef_set[FDS_C_QX])
      return fail(FDS_E_STATE, "thermal coefficients G and Q must be set");
  } else {
    if (!c->coef_set[FDS_C_RHO0]) return fail(FDS_E_STATE, "static density must be set");
  }
  c->coupled = false;
  c->fused_stages = c->fused_rows = 0;
  c->iso_b = !c->one_d && !c->coef_set[FDS_C_BY];   // (thermal: QY)
  c->iso_k = !c->one_d && !c->coef_set[FDS_C_KY];   // (thermal: GY)
  if (c->family != kNonlinear) {
    // the engine depends on the lossy flag just derived and on the material classes
    if (int rc = ready_classes(c)) return rc;
    if (int rc = choose_tiles(c)) return rc;
    const size_t lds = lds_bytes(c);
    if (lds > 65536) {
      // fall back to the default shape, which always fits
      c->tile = -1;
      if (int rc = choose_tiles(c)) return rc;
    }
  }
  c->committed = true;
  touch(c);
  return 0;
}

int fds_set_state(fds_ctx *c, int comp, const double *data, int64_t n) {
  if (int rc = check_idle(c)) return rc;
  if (int rc = check_comp(c, comp)) return rc;
  if (n != c->n) return fail(FDS_E_ARG, "state needs %lld values", (long long)c->n);
  Comp &cp = c->comp[comp];
  const int b = (cp.buf[1].p && (cp.accumulated || c->family != kThermal || comp == 0)) ? c->parity : 0;
  return transfer(c, true, const_cast<double *>(data), cp.buf[b].p,
                  c->form == FDS_FP32_KAHAN && cp.accumulated ? cp.cbuf[b].p : nullptr, n);
}

int fds_get_state(fds_ctx *c, int comp, double *data, int64_t n) {
  if (int rc = check_ctx(c)) return rc;
  if (int rc = check_comp(c, comp)) return rc;
  // the context's own runs in flight are ordered before the copy on its stream; a batch run
  // in flight is on the batch's stream
  if (c->batch_flights) return fail(FDS_E_STATE, "a batch run of this context is in flight");
  if (n != c->n) return fail(FDS_E_ARG, "state holds %lld values", (long long)c->n);
  Comp &cp = c->comp[comp];
  const int b = (cp.buf[1].p && (cp.accumulated || c->family != kThermal || comp == 0)) ? c->parity : 0;
  return transfer(c, false, data, cp.buf[b].p,
                  c->form == FDS_FP32_KAHAN && cp.accumulated ? cp.cbuf[b].p : nullptr, n);
}

int fds_set_boundaries(fds_ctx *c, int comp, int64_t ncell, const int64_t *cells,
                       const int32_t *ptr, int64_t nent, const double *a, const int64_t *off,
                       const int64_t *stride, const int64_t *len, int64_t ntable,
                       const double *table) {
  if (int rc = check_idle(c)) return rc;
  if (int rc = check_comp(c, comp)) return rc;
  Comp &cp = c->comp[comp];
  if (ncell < 0 || nent < 0 || ntable < 0) return fail(FDS_E_ARG, "negative size");
  if (ncell > 0 && (int64_t)ptr[ncell] != nent) return fail(FDS_E_ARG, "ptr[ncell] != nent");
  for (int64_t u = 0; u < ncell; ++u) {
    if (cells[u] < 0 || cells[u] >= c->n)
      return fail(FDS_E_INDEX, "boundary cell %lld out of range", (long long)cells[u]);
    if (ptr[u] > ptr[u + 1]) return fail(FDS_E_ARG, "ptr not monotone");
  }
  for (int64_t e = 0; e < nent; ++e) {
    if (off[e] < 0 || stride[e] < 0 || len[e] < 1 ||
        (stride[e] > 0 && off[e] + (len[e] - 1) * stride[e] >= ntable) ||
        (stride[e] == 0 && off[e] >= ntable))
      return fail(FDS_E_ARG, "boundary entry %lld addresses outside the table", (long long)e);
  }
  cp.cells.assign(cells, cells + ncell);
  cp.ptr.assign(ptr, ptr + (ncell > 0 ? ncell + 1 : 0));
  cp.a.assign(a, a + nent);
  cp.off.assign(off, off + nent);
  cp.stride.assign(stride, stride + nent);
  cp.len.assign(len, len + nent);
  cp.table.assign(table, table + ntable);
  HIP_TRY(upload(cp.d_ptr, cp.ptr, c->stream));
  HIP_TRY(upload(cp.d_a, cp.a, c->stream));
  HIP_TRY(upload(cp.d_off, cp.off, c->stream));
  HIP_TRY(upload(cp.d_stride, cp.stride, c->stream));
  HIP_TRY(upload(cp.d_table, cp.table, c->stream));
  if (c->over_stages || c->lbc_w1) {
    c->over_stages = c->over_rows = 0;
    if (int rc = choose_tiles(c)) return rc;
  }
  c->events_dirty = true;
  touch(c);
  return 0;
}

int fds_set_outputs(fds_ctx *c, int comp, int64_t m, const int64_t *cells) {
  if (int rc = check_idle(c)) return rc;
  if (int rc = check_comp(c, comp)) return rc;
  if (m < 0) return fail(FDS_E_ARG, "negative output count");
  for (int64_t k = 0; k < m; ++k)
    if (cells[k] < 0 || cells[k] >= c->n)
      return fail(FDS_E_INDEX, "output cell %lld out of range", (long long)cells[k]);
  Comp &cp = c->comp[comp];
  cp.out_cells.assign(cells, cells + m);
  if (c->lbc_w1)
    if (int rc = choose_tiles(c)) return rc;
  c->events_dirty = true;
  touch(c);
  return 0;
}

int fds_set_tile(fds_ctx *c, int t) {
  if (int rc = check_idle(c)) return rc;
  if (t < -1 || t >= fds::kNumTiles + fds::kNumStream)
    return fail(FDS_E_ARG, "tile index %d out of range", t);
  const int old = c->tile;
  c->tile = t;
  if (c->committed && t < 0 && old >= 0 && !c->coupled)
    if (int rc = ready_classes(c)) return rc;
  if (int rc = choose_tiles(c)) return rc;
  if (c->committed && lds_bytes(c) > 65536) {
    c->tile = old;
    choose_tiles(c);
    return fail(FDS_E_ARG, "tile %d needs more than 64 KiB of LDS for this field", t);
  }
  touch(c);
  return 0;
}

int fds_set_line_shape(fds_ctx *c, int cells_per_thread, int threads, int ghost) {
  if (int rc = check_idle(c)) return rc;
  if (!c->one_d && c->family != kNonlinear)
    return fail(FDS_E_ARG, "the resident engine serves 1D models only");
  const int fam = c->family == kNonlinear ? fds::kLineNonlinear : fds::kLineAcoustic;
  int v = -1;
  for (int i = 0; i < fds::kNumLineCpt; ++i)
    if (fds::kLineCpt[i] == cells_per_thread) v = i;
  if (v < 0) return fail(FDS_E_ARG, "cells per thread must be 1, 2, 4 or 8");
  if (threads != 0) {
    if (threads < 64 || threads % 64 || threads > fds::line_max_threads(fam, v))
      return fail(FDS_E_ARG, "segment workgroup of %d threads: a multiple of 64 up to %d",
                  threads, fds::line_max_threads(fam, v));
    if (ghost < 2 || threads * cells_per_thread - 2 * ghost < 1)
      return fail(FDS_E_ARG, "ghost cells must be at least 2 and leave owned cells");
  }
  const int o_rows = c->strip_rows, o_t = c->line_cfg_threads, o_g = c->line_cfg_ghost;
  c->strip_rows = cells_per_thread;
  c->line_cfg_threads = threads;
  c->line_cfg_ghost = threads ? ghost : 0;
  if (int rc = choose_tiles(c)) {
    c->strip_rows = o_rows;
    c->line_cfg_threads = o_t;
    c->line_cfg_ghost = o_g;
    choose_tiles(c);
    return rc;
  }
  touch(c);
  return 0;
}

int fds_set_strip_height(fds_ctx *c, int rows) {
  if (int rc = check_idle(c)) return rc;
  if (rows < 0 || rows > 65536) return fail(FDS_E_ARG, "strip height %d out of range", rows);
  const int old = c->strip_rows;
  c->strip_rows = rows;
  if (int rc = choose_tiles(c)) {
    c->strip_rows = old;
    choose_tiles(c);
    return rc;
  }
  touch(c);
  return 0;
}

}  // extern "C"

namespace {

// Common start of a run of nsteps steps from `start`: signal lengths, event lists, output
// rows, the device step counter.
int prepare_run(fds_ctx *c, int64_t start, int64_t nsteps) {
  // every boundary entry must have a value for every step of the run
  for (int k = 0; k < 3; ++k) {
    const Comp &cp = c->comp[k];
    for (size_t e = 0; e < cp.len.size(); ++e)
      if (start + nsteps > cp.len[e])
        return fail(FDS_E_INDEX, "boundary signal of component %d has %lld samples, step %lld "
                    "requested", k, (long long)cp.len[e], (long long)(start + nsteps - 1));
  }
  if (int rc = rebuild_events(c)) return rc;
  // output rows for this run
  for (int k = 0; k < 3; ++k) {
    Comp &cp = c->comp[k];
    const size_t need = std::max<size_t>(cp.out_cells.size() * nsteps * 8, 16);
    if (cp.obuf.bytes < need) {
      // grow geometrically (and to at least 4096 rows) so repeated runs keep their graphs
      const size_t rows = std::max<int64_t>(nsteps, 4096);
      HIP_TRY(cp.obuf.ensure(std::max(std::max(need, cp.obuf.bytes * 2),
                                      cp.out_cells.size() * rows * 8)));
      touch(c);
    }
    cp.obuf_rows = cp.out_cells.empty() ? 0 : nsteps;
  }
  hipLaunchKernelGGL(k_set_dyn, dim3(1), dim3(64), 0, c->stream, c->dyn.as<int64_t>(), start);
  HIP_TRY(hipGetLastError());
  if (c->lbc_ring) {       // the caller may have trained on since the last run
    fds::launch_ring_pack(c->lbc_w1, c->lbc_w2, c->lbc_packed.p, c->stream);
    HIP_TRY(hipGetLastError());
  }
  if (c->nf_check) {
    hipLaunchKernelGGL(k_nonfinite_reset, dim3(1), dim3(64), 0, c->stream, c->dyn.as<int64_t>());
    HIP_TRY(hipGetLastError());
  }
  if (!c->ev0) HIP_TRY(hipEventCreate(&c->ev0));
  if (!c->ev1) HIP_TRY(hipEventCreate(&c->ev1));
  if (c->line) {
    // resident 1D engine: the signal table is addressed with 32-bit indices
    for (int k = 0; k < 3; ++k)
      if (c->comp[k].table.size() > (size_t)std::numeric_limits<int32_t>::max())
        return fail(FDS_E_ARG, "boundary table of component %d too large for the resident 1D "
                    "engine (select tile %d)", k, fds::kTileRow);
  }
  return 0;
}

template <typename T>
int launch_couple(fds_ctx *ac, fds_ctx *th, int k, int steps, int threads,
                  const fds::LineCouple<T> &cp) {
  fds::StepArgs<T> a, h;
  fill_args<T>(ac, a, ac->parity);
  fill_args<T>(th, h, th->parity);
  a.k = h.k = k;
  a.steps = h.steps = steps;
  a.strip_h = h.strip_h = ac->line_seg;
  a.ghost = h.ghost = ac->line_ghost;
  ac->ks->couple[ac->line_var][ac->lossy ? 1 : 0](&a, &h, &cp, ac->line_wgs, threads,
                                                   ac->stream);
  HIP_TRY(hipGetLastError());
  return 0;
}

template <typename T>
int couple_run(fds_ctx *ac, fds_ctx *th, const double *rho, const double *loss, double dt,
               int64_t stepping, int accumulate, double *accum, int64_t start, int64_t nsteps,
               int threads) {
  const int64_t n = ac->n;
  std::vector<T> r(n), l(n);
  for (int64_t i = 0; i < n; ++i) {
    r[i] = (T)rho[i];
    l[i] = (T)loss[i];
  }
  std::vector<double> acc(accumulate ? accum : nullptr, accumulate ? accum + n : nullptr);
  if (acc.empty()) acc.assign(1, 0.0);
  HIP_TRY(upload(ac->couple_rho, r, ac->stream));
  HIP_TRY(upload(ac->couple_loss, l, ac->stream));
  HIP_TRY(upload(ac->couple_acc, acc, ac->stream));
  fds::LineCouple<T> cp;
  cp.rho = ac->couple_rho.as<const T>();
  cp.loss = ac->couple_loss.as<const T>();
  cp.acc = ac->couple_acc.as<double>();
  cp.dt = (T)dt;
  cp.stepping = stepping;
  cp.accumulate = accumulate ? 1 : 0;
  HIP_TRY(hipEventRecord(ac->ev0, ac->stream));
  // segments: the loss transfer reads the velocity's left neighbour, so wrong values reach
  // one cell further into the temperature than into the fields: ghost - 2 steps per launch
  const int per = ac->line_wgs > 1 ? std::min(ac->line_ghost - 2, fds::kLineSteps)
                                   : fds::kLineSteps;
  int64_t done = 0;
  while (done < nsteps) {
    const int st = (int)std::min<int64_t>(nsteps - done, per);
    if (int rc = launch_couple<T>(ac, th, (int)done, st, threads, cp)) return rc;
    ac->parity ^= 1;
    th->parity ^= 1;
    done += st;
  }
  HIP_TRY(hipEventRecord(ac->ev1, ac->stream));
  HIP_TRY(hipStreamSynchronize(ac->stream));
  if (accumulate)
    HIP_TRY(hipMemcpy(accum, ac->couple_acc.p, n * sizeof(double), hipMemcpyDeviceToHost));
  float ms = 0.f;
  HIP_TRY(hipEventElapsedTime(&ms, ac->ev0, ac->ev1));
  ac->last_run_ms = th->last_run_ms = ms;
  return 0;
}

// The steps of a prepared run (prepare_run) enqueued on the context's stream, between events
// e0 and e1.
// Capture the chunk graphs a run of nsteps steps replays (at most two: one per buffer parity
// it starts a chunk on).  Capturing is set-up: it waits for the stream to be idle, then builds
// the graph on the host.
// Graph of the whole launches before the last one of a run's tail of `rest` steps (at most one
// chunk): rest - 1 rounded down to whole launches, when that is at least two launches.  0: the
// tail runs as plain launches (also once kMaxShortGraphs tail lengths hold graphs).
constexpr int kMaxShortGraphs = 8;

int short_graph_steps(const fds_ctx *c, int64_t rest, int parity) {
  const int g = step_group(c);
  const int64_t len = (rest - 1) / g * g;
  if (len < 2 * g) return 0;
  if (c->graphs.count(std::make_pair((int)len, parity))) return (int)len;
  int shorts = 0;
  for (const auto &kv : c->graphs) shorts += kv.first.first != c->graph_chunk;
  return shorts < 2 * kMaxShortGraphs ? (int)len : 0;
}

// both_parities: also the graphs a run starting from the other state buffer replays (runs
// prepared ahead of other runs of odd launch counts).
int capture_run_graphs(fds_ctx *c, int64_t nsteps, int chunk, bool both_parities = false) {
  if (c->line || chunk <= 0) return 0;
  if (both_parities) {
    c->parity ^= 1;
    const int rc = capture_run_graphs(c, nsteps, chunk);
    c->parity ^= 1;
    if (rc) return rc;
  }
  const int g = step_group(c);
  const int ch = std::max(g, chunk - chunk % g);
  c->graph_chunk = ch;
  int parity = c->parity;
  for (int64_t left = nsteps, n = 0; left > ch && n < 2; left -= ch, ++n) {
    hipGraphExec_t ex;
    if (int rc = get_graph(c, ch, parity, &ex)) return rc;
    parity ^= ((ch / g) & 1);
  }
  // the tail after the full chunks (a run shorter than a chunk is all tail)
  const int64_t tail = (nsteps - 1) % ch + 1, full = (nsteps - tail) / ch;
  parity = c->parity ^ (int)((full * (ch / g)) & 1);
  if (const int len = short_graph_steps(c, tail, parity)) {
    hipGraphExec_t ex;
    if (int rc = get_graph(c, len, parity, &ex)) return rc;
  }
  return 0;
}

int enqueue_steps(fds_ctx *c, int64_t nsteps, int chunk, hipEvent_t e0, hipEvent_t e1) {
  // graphs first, so that the events bracket the steps only
  if (int rc = capture_run_graphs(c, nsteps, chunk)) return rc;
  HIP_TRY(hipEventRecord(e0, c->stream));
  int64_t done = 0;
  if (c->line) {
    // one segment: up to kLineSteps steps per launch.  Several: a wrong value enters each
    // segment from its open ends, one cell per step from the left and, where the update of
    // the second component reads its right neighbour's old value (viscous and convective
    // terms, the nonlinear mass flux), one more cell on the right: ghost - 1 steps per launch.
    const int per = c->line_wgs > 1 ? std::min(c->line_ghost - 1, fds::kLineSteps)
                                    : fds::kLineSteps;
    int64_t scanned = 0;
    while (done < nsteps) {
      const int st = (int)std::min<int64_t>(nsteps - done, per);
      const int rc = c->elem == 8 ? launch_line<double>(c, c->parity, (int)done, st)
                                  : launch_line<float>(c, c->parity, (int)done, st);
      if (rc) return rc;
      c->parity ^= 1;
      done += st;
      // the first component every kNonfiniteEvery steps or more (launch granularity)
      if (c->nf_check && done < nsteps && done - scanned >= kNonfiniteEvery) {
        if (int rc2 = scan_nonfinite(c, 0, c->parity, c->dyn.as<const int64_t>(), done,
                                     c->dyn.as<int64_t>(), c->stream))
          return rc2;
        scanned = done;
      }
    }
    chunk = 0;
  }
  const int g = step_group(c);
  int64_t graph_done = 0;    // steps the device step counter advanced by (graph chunks)
  if (chunk > 0) {
    // graph-replayed full chunks (whole launches of g steps), never including the run's last
    // step (which stores the assigned components)
    chunk = std::max(g, chunk - chunk % g);
    while (nsteps - done > chunk) {
      hipGraphExec_t ex;
      if (int rc = get_graph(c, chunk, c->parity, &ex)) return rc;
      HIP_TRY(hipGraphLaunch(ex, c->stream));
      c->parity ^= ((chunk / g) & 1);
      done += chunk;
      graph_done += chunk;
    }
    // the tail's whole launches but the last as one graph too (one launch call, not several)
    if (const int len = short_graph_steps(c, nsteps - done, c->parity)) {
      hipGraphExec_t ex;
      if (int rc = get_graph(c, len, c->parity, &ex)) return rc;
      HIP_TRY(hipGraphLaunch(ex, c->stream));
      c->parity ^= ((len / g) & 1);
      done += len;
      graph_done += len;
    }
  }
  // the rest as plain launches of g stages, then one launch of the remaining stages (k counts
  // from the device step counter's current base)
  for (int64_t k = 0; done + k < nsteps;) {
    const int st = (int)std::min<int64_t>(g, nsteps - done - k);
    if (int rc = launch_step_any(c, c->parity, (int)k, done + k + st == nsteps, st)) return rc;
    c->parity ^= 1;
    k += st;
  }
  if (c->nf_check)   // every component after the run
    if (int rc = scan_all_nonfinite(c, c->parity, c->dyn.as<const int64_t>(),
                                    nsteps - graph_done, c->stream))
      return rc;
  HIP_TRY(hipEventRecord(e1, c->stream));
  return 0;
}

// True when prepare_run(c, ., nsteps) neither rebuilds the event tables nor grows an output
// buffer (so it frees no device memory a run in flight may use).
bool run_steady(const fds_ctx *c, int64_t nsteps) {
  if (c->events_dirty || (!c->graphs.empty() && c->graph_generation != c->generation))
    return false;
  for (int k = 0; k < 3; ++k) {
    const Comp &cp = c->comp[k];
    if (cp.obuf.bytes < std::max<size_t>(cp.out_cells.size() * nsteps * 8, 16)) return false;
  }
  return true;
}

int ensure_events(hipEvent_t (&ev)[3]) {
  for (int i = 0; i < 3; ++i)
    if (!ev[i]) HIP_TRY(hipEventCreate(&ev[i]));
  return 0;
}

// Enqueue the copy of a run's recorded outputs (rows x outputs per component) into staging
// slot `slot` on stream s.
int stage_outputs(fds_ctx *c, int slot, int64_t rows, hipStream_t s) {
  for (int k = 0; k < 3; ++k) {
    Comp &cp = c->comp[k];
    const size_t bytes = cp.out_cells.size() * (size_t)rows * 8;
    if (!bytes) continue;
    HIP_TRY(cp.stage[slot].ensure(bytes));
    HIP_TRY(hipMemcpyAsync(cp.stage[slot].p, cp.obuf.p, bytes, hipMemcpyDeviceToHost, s));
  }
  return 0;
}

// Copy a finished run's staged outputs to the caller (null destinations are skipped).
void take_outputs(fds_ctx *c, const Flight &f, double *const *dst) {
  for (int k = 0; k < 3; ++k) {
    const Comp &cp = c->comp[k];
    const size_t bytes = cp.out_cells.size() * (size_t)f.rows * 8;
    if (bytes && dst[k]) std::memcpy(dst[k], cp.stage[f.slot].p, bytes);
  }
}

}  // namespace

extern "C" {

int fds_couple_loss_run(fds_ctx *ac, fds_ctx *th, const double *rho, const double *loss,
                        double dt, int64_t stepping, int accumulate, double *accum,
                        int64_t start, int64_t nsteps) {
  if (int rc = check_idle(ac)) return rc;
  if (int rc = check_idle(th)) return rc;
  if (ac->model != FDS_ACOUSTIC1D || th->model != FDS_THERMAL1D)
    return fail(FDS_E_ARG, "the loss coupling joins an Acoustic1D and a Thermal1D context");
  if (ac->device != th->device || ac->form != th->form || ac->n != th->n)
    return fail(FDS_E_ARG, "coupled contexts must share device, form and cell count");
  if (!ac->committed || !th->committed) return fail(FDS_E_STATE, "coefficients not committed");
  if (ac->tile >= 0 || th->tile >= 0)
    return fail(FDS_E_ARG, "coupled contexts must use the resident 1D engine (tile -1)");
  if (!rho || !loss || (accumulate && !accum)) return fail(FDS_E_ARG, "null coupling input");
  if (stepping < 1) return fail(FDS_E_ARG, "coupling stepping must be at least 1");
  if (nsteps < 0 || start < 0) return fail(FDS_E_ARG, "negative step count");
  if (nsteps == 0) return 0;
  // one layout for both contexts: one workgroup of one cell per thread for short lines (the
  // coupled kernel holds two fields, so it has half the single-field threads from 2 cells per
  // thread on), else the single-field default segments
  const bool seg = ac->n > fds::kLineSegmentAbove;
  const int cpt = seg ? fds::kLineSegCpt : 1;
  const int cfg_t = seg ? fds::kLineSegThreads : 0, cfg_g = seg ? fds::kLineSegGhost : 0;
  static_assert(fds::kLineSegThreads <= fds::kCoupleMaxThreads[1] && fds::kLineSegCpt == 2 &&
                    fds::kLineSegmentAbove <= fds::kCoupleMaxThreads[0] &&
                    fds::kLineSegGhost > 2,
                "coupled layouts must fit the coupled kernel's launch bounds");
  for (fds_ctx *c : {ac, th}) {
    if (!c->line || c->strip_rows != cpt || c->line_cfg_threads != cfg_t ||
        c->line_cfg_ghost != cfg_g) {
      c->strip_rows = cpt;
      c->line_cfg_threads = cfg_t;
      c->line_cfg_ghost = cfg_g;
      if (int rc = choose_tiles(c)) return rc;
      touch(c);
    }
    if (!c->line)
      return fail(FDS_E_ARG, "coupled runs hold at most %lld cells",
                  (long long)fds::kLineMaxResident);
    if (int rc = prepare_run(c, start, nsteps)) return rc;
  }
  // the coupled kernel runs on the acoustic context's stream and reads the thermal context's
  // step counters, which prepare_run wrote on the thermal stream
  HIP_TRY(hipStreamSynchronize(th->stream));
  const int threads = ac->line_threads;
  return ac->elem == 8 ? couple_run<double>(ac, th, rho, loss, dt, stepping, accumulate, accum,
                                            start, nsteps, threads)
                       : couple_run<float>(ac, th, rho, loss, dt, stepping, accumulate, accum,
                                           start, nsteps, threads);
}

int fds_run(fds_ctx *c, int64_t start, int64_t nsteps, int chunk) {
  if (int rc = check_idle(c)) return rc;
  if (!c->committed) return fail(FDS_E_STATE, "coefficients not committed");
  if (nsteps < 0 || start < 0) return fail(FDS_E_ARG, "negative step count");
  if (nsteps == 0) return 0;
  if (int rc = leave_coupling(c)) return rc;
  if (int rc = prepare_run(c, start, nsteps)) return rc;
  if (int rc = enqueue_steps(c, nsteps, chunk, c->ev0, c->ev1)) return rc;
  if (int rc = stage_nonfinite(c, kMaxFlights, c->stream)) return rc;
  HIP_TRY(hipStreamSynchronize(c->stream));
  float ms = 0.f;
  HIP_TRY(hipEventElapsedTime(&ms, c->ev0, c->ev1));
  c->last_run_ms = ms;
  return check_nonfinite(c, kMaxFlights);
}

int fds_prepare_run(fds_ctx *c, int64_t start, int64_t nsteps, int chunk) {
  if (int rc = check_idle(c)) return rc;
  if (!c->committed) return fail(FDS_E_STATE, "coefficients not committed");
  if (nsteps < 1 || start < 0) return fail(FDS_E_ARG, "a run needs steps");
  if (int rc = leave_coupling(c)) return rc;
  if (int rc = prepare_run(c, start, nsteps)) return rc;
  if (int rc = capture_run_graphs(c, nsteps, chunk, true)) return rc;
  // the fused engines' stage counts are code objects of their own, loaded on their first launch
  // (1.3 ms): those of the launches outside the graphs
  if (c->fused)
    for (const int st : {step_group(c), (int)(nsteps % step_group(c))})
      if (st > 0) pick_launch(c, st)(nullptr, 0, 0, c->stream);
  // pinned staging and events of asynchronous runs of this length (both slots)
  for (int slot = 0; slot < kMaxFlights; ++slot) {
    if (int rc = ensure_events(c->fev[slot])) return rc;
    for (int k = 0; k < 3; ++k) {
      const size_t bytes = c->comp[k].out_cells.size() * (size_t)nsteps * 8;
      if (bytes) HIP_TRY(c->comp[k].stage[slot].ensure(bytes));
    }
  }
  HIP_TRY(hipStreamSynchronize(c->stream));
  return 0;
}

int fds_run_async(fds_ctx *c, int64_t start, int64_t nsteps, int chunk) {
  if (int rc = check_ctx(c)) return rc;
  if (!c->committed) return fail(FDS_E_STATE, "coefficients not committed");
  if (nsteps < 1 || start < 0) return fail(FDS_E_ARG, "an asynchronous run needs steps");
  if (c->batch_flights) return fail(FDS_E_STATE, "a batch run of this context is in flight");
  if ((int)c->flights.size() >= kMaxFlights)
    return fail(FDS_E_STATE, "%d runs in flight: take the oldest first", kMaxFlights);
  if (int rc = leave_coupling(c)) return rc;     // (a coupled run left none in flight)
  // a run that rebuilds tables or grows the output rows frees device memory the runs in
  // flight may read: let them finish first
  if (!run_steady(c, nsteps)) HIP_TRY(hipStreamSynchronize(c->stream));
  if (int rc = prepare_run(c, start, nsteps)) return rc;
  const int slot = c->next_slot;
  if (int rc = ensure_events(c->fev[slot])) return rc;
  if (int rc = enqueue_steps(c, nsteps, chunk, c->fev[slot][0], c->fev[slot][1])) return rc;
  if (int rc = stage_outputs(c, slot, nsteps, c->stream)) return rc;
  if (int rc = stage_nonfinite(c, slot, c->stream)) return rc;
  HIP_TRY(hipEventRecord(c->fev[slot][2], c->stream));
  if (c->flights.empty()) c->last_run_ms = 0.0;   // a new sequence of asynchronous runs
  c->flights.push_back(Flight{nsteps, slot});
  c->next_slot = (slot + 1) % kMaxFlights;
  return 0;
}

int fds_run_take(fds_ctx *c, double *dst0, double *dst1, double *dst2) {
  if (int rc = check_ctx(c)) return rc;
  if (c->flights.empty()) return fail(FDS_E_STATE, "no asynchronous run in flight");
  const Flight f = c->flights.front();
  HIP_TRY(hipEventSynchronize(c->fev[f.slot][2]));
  c->flights.pop_front();
  double *dst[3] = {dst0, dst1, dst2};
  take_outputs(c, f, dst);
  float ms = 0.f;
  HIP_TRY(hipEventElapsedTime(&ms, c->fev[f.slot][0], c->fev[f.slot][1]));
  c->last_run_ms += ms;
  return check_nonfinite(c, f.slot);
}

int fds_set_nonfinite_check(fds_ctx *c, int enable) {
  if (int rc = check_idle(c)) return rc;
  if (c->nf_check != (enable != 0)) {
    c->nf_check = enable != 0;
    touch(c);   // the chunk graphs hold the scans
  }
  return 0;
}

int fds_set_flow(fds_ctx *c, const int64_t *period, int64_t nrows) {
  if (int rc = check_idle(c)) return rc;
  if (!period || nrows == 0) {
    c->flow = false;
    if (int rc = choose_tiles(c)) return rc;
    touch(c);
    return 0;
  }
  if (c->family != kAcoustic || c->one_d)
    return fail(FDS_E_ARG, "flow is implemented for the 2D acoustic models");
  if (nrows != c->ny) return fail(FDS_E_ARG, "flow needs %lld row periods, got %lld",
                                  (long long)c->ny, (long long)nrows);
  std::vector<int64_t> p(period, period + nrows);
  HIP_TRY(upload(c->flow_period, p, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  c->flow = true;
  if (int rc = choose_tiles(c)) return rc;
  touch(c);
  return 0;
}

int fds_set_learned_boundary(fds_ctx *c, const uint16_t *w1, const uint16_t *w2, int layer,
                             const float *comp_scale) {
  if (int rc = check_idle(c)) return rc;
  if (!w1) {
    c->lbc_w1 = c->lbc_w2 = nullptr;
    if (int rc = choose_tiles(c)) return rc;
    touch(c);
    return 0;
  }
  if (!w2 || !comp_scale) return fail(FDS_E_ARG, "weights and component scales are required");
  if (c->family != kAcoustic || c->axi || c->one_d)
    return fail(FDS_E_ARG, "the learned boundary is implemented for Acoustic2D");
  if (c->elem != 4) return fail(FDS_E_ARG, "the learned boundary needs an FP32 form");
  if (c->nx != c->ny) return fail(FDS_E_ARG, "the learned boundary needs a square grid");
  if (layer != fds::kLbcDepth || c->nx < 2 * layer + fds::kLbcBand + 1)
    return fail(FDS_E_ARG, "layer depth must be %d on a grid wider than %d", fds::kLbcDepth,
                2 * fds::kLbcDepth + fds::kLbcBand);
  for (int k = 0; k < 3; ++k)
    if (!(comp_scale[k] > 0.f)) return fail(FDS_E_ARG, "component scales must be positive");
  c->lbc_w1 = w1;
  c->lbc_w2 = w2;
  c->lbc_layer = layer;
  for (int k = 0; k < 3; ++k) c->lbc_cs[k] = comp_scale[k];
  if (int rc = choose_tiles(c)) return rc;
  touch(c);
  return 0;
}

int fds_last_run_ms(fds_ctx *c, double *ms) {
  if (int rc = check_ctx(c)) return rc;
  if (!ms) return fail(FDS_E_ARG, "null output pointer");
  *ms = c->last_run_ms;
  return 0;
}

int fds_read_outputs(fds_ctx *c, int comp, int64_t row0, int64_t nrows, double *dst) {
  if (int rc = check_idle(c)) return rc;
  if (int rc = check_comp(c, comp)) return rc;
  Comp &cp = c->comp[comp];
  const int64_t m = (int64_t)cp.out_cells.size();
  if (m == 0 || nrows == 0) return 0;
  if (row0 < 0 || nrows < 0 || row0 + nrows > cp.obuf_rows)
    return fail(FDS_E_INDEX, "output rows [%lld, %lld) not recorded", (long long)row0,
                (long long)(row0 + nrows));
  HIP_TRY(hipMemcpyAsync(dst, cp.obuf.as<double>() + row0 * m, nrows * m * 8,
                         hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  return 0;
}

}  // extern "C"

namespace {

bool batch_stale(const fds_batch *b) {
  if (b->build_gen.size() != b->ctxs.size()) return true;
  for (size_t i = 0; i < b->ctxs.size(); ++i) {
    const fds_ctx *c = b->ctxs[i];
    if (c->generation != b->build_gen[i] || (c->parity ^ b->build_parity[i]) != b->flip)
      return true;
  }
  return false;
}

void batch_drop_graphs(fds_batch *b) {
  for (auto &kv : b->graphs) (void)hipGraphExecDestroy(kv.second);
  for (auto g : b->graph_objs) (void)hipGraphDestroy(g);
  b->graphs.clear();
  b->graph_objs.clear();
}

MemberLayout layout_of(const fds_ctx *c) {
  return MemberLayout{c->shape, c->fuse,   c->ghost, c->ghost_rows, c->tx,
                      c->ty,    c->ntiles, c->fused, c->line,       c->lossy};
}

// Lay a batch out: every member on the fused engine (try_fused, where it covers them all) or on
// one shape of the tile table, and the tables that map the launch's tiles to members.
int batch_layout(fds_batch *b, bool try_fused) {
  // (runs in flight elsewhere read the members' tables)
  for (auto *c : b->ctxs)
    if (!c->flights.empty() || c->batch_flights) {
      HIP_TRY(hipDeviceSynchronize());
      break;
    }
  b->fused = false;
  if (try_fused && b->tile < 0 && b->schedule == 0) {
    int64_t cells = 0, across = 0;
    bool ok = true;
    for (auto *c : b->ctxs) {
      c->tile = -1;
      if (int rc = leave_coupling(c)) return rc;
      if (!(can_stream_batch(c) && fuse_reach(c))) ok = false;
      if (ok && !c->npal)
        if (int rc = ready_classes(c)) return rc;
      ok = ok && c->npal > 0;
      cells += c->n;
    }
    // The stages by the rule of one field (choose_fused) on the whole batch; the height for 24
    // strips a CU in every form: a launch ends with the tiles that hold sources and recorded points,
    // which every member has, and short strips shorten those.  us a step at 16, 20, 24 and 28, with
    // a source line and 8 points a member: 40 plane and axial members, 128 to 640 cells a side,
    // FP64 13.7, 13.3, 13.8, 13.8, FP32 8.4, 8.0, 7.0, 6.9, Kahan 14.5, 14.1, 14.3, 14.3; 12 of
    // 500 x 480 FP64 7.1, 6.5, 6.2, 6.3, FP32 5.6, 5.3, 4.9, 4.8; 60 of 100 to 200 FP64 5.9, 5.7,
    // 6.0, 6.4, Kahan 6.1, 6.1, 6.3, 6.8; 4 of 1500 x 1400 FP64 19.7, 19.2, 20.1, 19.6, FP32 11.1,
    // 9.9, 9.3, 9.2; 64 of 128 to 1024 level.  (Without any source or point 16 is 3 to 10 % ahead.)
    const int S = cells < (1 << 18) ? 4 : fds::kFusedMax, sx = 64 - 2 * S;
    for (auto *c : b->ctxs) across += (c->nx + sx - 1) / sx * c->ny;
    const int64_t strips = 24 * (int64_t)b->ctxs[0]->num_cu;
    const int64_t want = (across + strips / 2) / strips;
    for (auto *c : b->ctxs) {
      if (!ok) break;
      c->fused_stages = S;
      c->fused_rows = (int)std::min<int64_t>(std::max<int64_t>(want, 4), 64);
      if (int rc = choose_tiles(c)) return rc;
      touch(c);
      if (int rc = rebuild_events(c)) return rc;   // (may leave the fused engine)
      ok = c->fused && c->fuse == S;
    }
    b->fused = ok;
    b->fuse = S;
  }
  bool all_stream = true;
  for (auto *c : b->ctxs) all_stream = all_stream && can_stream_batch(c);
  int t = b->tile < 0 ? (all_stream ? fds::kDefaultLossless2D : fds::kDefaultTile2D) : b->tile;
  if (t >= fds::kNumTiles + fds::kNumStream || t < 0)
    return fail(FDS_E_ARG, "tile index %d out of range", t);
  if (t >= fds::kNumTiles && !all_stream) t = fds::kDefaultTile2D;
  if (t >= fds::kNumTiles && fds::stream_single_only(t - fds::kNumTiles))
    return fail(FDS_E_ARG, "shape %d (prefetch %d rows) serves single fields only", t,
                fds::kStreamShapes[t - fds::kNumTiles][4]);
  std::vector<int32_t> tinst, base;
  size_t lds = 0;
  b->layouts.clear();
  const int n = (int)b->ctxs.size();
  for (int i = 0; i < n; ++i) {
    fds_ctx *c = b->ctxs[i];
    if (!b->fused) {
      c->fused_stages = c->fused_rows = 0;
      c->tile = t;
      if (int rc = choose_tiles(c)) return rc;
      touch(c);
      lds = std::max(lds, lds_bytes(c));
    }
    base.push_back((int32_t)tinst.size());
    b->layouts.push_back(layout_of(c));
    for (int k = 0; k < c->ntiles; ++k) tinst.push_back(i);
  }
  if (lds > 65536)
    return fail(FDS_E_ARG, "tile %d needs more than 64 KiB of LDS for some member", t);
  b->shape = t;
  b->streaming = t >= fds::kNumTiles;
  if (!b->fused) b->fuse = b->streaming ? fds::kStreamShapes[t - fds::kNumTiles][2] : 1;
  shape_of(t, &b->tx, &b->ty);
  b->lds = lds;
  b->ntiles = (int)tinst.size();
  // work-queue order: largest tiles first (owned cells plus ghosts; edge tiles are smaller)
  std::vector<int64_t> cost(b->ntiles);
  for (int g = 0; g < b->ntiles; ++g) {
    const fds_ctx *c = b->ctxs[tinst[g]];
    const int t = g - base[tinst[g]];
    const int64_t ty = t / std::max(1, c->tiles_x), tx = t - ty * c->tiles_x;
    const int64_t sx = std::max(1, c->sx), h = std::max(1, c->ty);
    const int64_t cols = std::min<int64_t>(sx, c->nx - tx * sx);
    const int64_t rows = std::min<int64_t>(h, c->ny - ty * h);
    cost[g] = (cols + 2 * c->ghost) * (rows + 2 * c->ghost_rows);
  }
  std::vector<int32_t> order(b->ntiles);
  for (int g = 0; g < b->ntiles; ++g) order[g] = g;
  std::stable_sort(order.begin(), order.end(),
                   [&](int32_t x, int32_t y) { return cost[x] > cost[y]; });
  if (upload(b->tile_inst, tinst, b->stream) != hipSuccess ||
      upload(b->inst_base, base, b->stream) != hipSuccess || b->dyn.ensure(64) != hipSuccess ||
      upload(b->order, order, b->stream) != hipSuccess)
    return fail(FDS_E_HIP, "out of device memory for the batch tables");
  batch_drop_graphs(b);
  b->build_gen.clear();
  return 0;
}

// Whether the members are still as the batch was laid out (a member may have been given another
// tile, strip height, or coefficients of another kind since).
bool batch_laid_out(const fds_batch *b) {
  for (size_t i = 0; i < b->ctxs.size(); ++i) {
    const fds_ctx *c = b->ctxs[i];
    if (!(layout_of(c) == b->layouts[i]) || lds_bytes(c) > b->lds || (b->fused && !c->npal))
      return false;
  }
  return true;
}

template <typename T>
int batch_build(fds_batch *b, int64_t nsteps) {
  for (auto *c : b->ctxs)
    if (int rc = rebuild_events(c)) return rc;
  if (!batch_laid_out(b))
    if (int rc = batch_layout(b, true)) return rc;
  for (auto *c : b->ctxs) {
    if (int rc = rebuild_events(c)) return rc;
    for (int k = 0; k < 3; ++k) {
      Comp &cp = c->comp[k];
      const size_t need = std::max<size_t>(cp.out_cells.size() * nsteps * 8, 16);
      if (cp.obuf.bytes < need) {
        const size_t rows = std::max<int64_t>(nsteps, 4096);
        HIP_TRY(cp.obuf.ensure(std::max(std::max(need, cp.obuf.bytes * 2),
                                        cp.out_cells.size() * rows * 8)));
        touch(c);
      }
      cp.obuf_rows = cp.out_cells.empty() ? 0 : nsteps;
    }
  }
  if (!batch_stale(b)) return 0;
  const int ni = (int)b->ctxs.size();
  for (int parity = 0; parity < 2; ++parity)
    for (int store = 0; store < 2; ++store) {
      std::vector<fds::StepArgs<T>> d(ni);
      for (int i = 0; i < ni; ++i) {
        fds_ctx *c = b->ctxs[i];
        // members flip in lock step: descriptor set `parity` reads each member's buffer
        // (its parity at build time) ^ parity
        fill_args<T>(c, d[i], c->parity ^ parity);
        d[i].dyn = b->dyn.as<const int64_t>();
        if (c->axi) d[i].flags |= fds::kFlagAxi;
        if (c->lossy) d[i].flags |= fds::kFlagLossy;
        if (c->family == kThermal) d[i].flags |= fds::kFlagThermal;
        if (store) d[i].flags |= fds::kFlagStore;
      }
      HIP_TRY(upload(b->descs[parity][store], d, b->stream));
    }
  if (b->fused) {
    // (a member's new coefficients may be of another kind than those the batch was laid out for)
    b->fused_any = false;
    std::vector<int32_t> inst, slot;
    for (int i = 0; i < ni; ++i) {
      const fds_ctx *c = b->ctxs[i];
      b->fused_any = b->fused_any || c->family != kAcoustic || !(c->axi || (c->iso_b && c->iso_k));
      for (int s = 0; s < c->fused_ev.nslots; ++s) {
        inst.push_back(i);
        slot.push_back(s);
      }
    }
    b->nev = (int)inst.size();
    HIP_TRY(upload(b->ev_inst, inst, b->stream));
    HIP_TRY(upload(b->ev_slot, slot, b->stream));
  }
  batch_drop_graphs(b);
  b->build_gen.clear();
  b->build_parity.clear();
  for (auto *c : b->ctxs) {
    b->build_gen.push_back(c->generation);
    b->build_parity.push_back(c->parity);
  }
  b->flip = 0;
  return 0;
}

int batch_launch(fds_batch *b, int rel_parity, int k, bool store, int stages = 1) {
  fds::BatchLaunch L;
  L.descs = b->descs[rel_parity][store ? 1 : 0].p;
  L.tile_inst = b->tile_inst.as<const int32_t>();
  L.inst_base = b->inst_base.as<const int32_t>();
  L.ntiles = b->ntiles;
  L.k = k;
  L.order = b->order.as<const int32_t>();
  L.queue = b->queue.as<unsigned>();
  L.nq = b->nq;
  L.spl = b->fuse;
  L.num_cu = b->ctxs[0]->num_cu;
  L.ev_inst = b->ev_inst.as<const int32_t>();
  L.ev_slot = b->ev_slot.as<const int32_t>();
  L.nev = b->nev;
  if (b->fused) {
    b->ks->fused_batch[b->fused_any ? 1 : 0][stages - 1](L, 0, 0, b->stream);
    HIP_TRY(hipGetLastError());
    return 0;
  }
  // the work queue serves full launches; remainder launches (fewer stages) and other shapes
  // run on the dispatcher kernels
  if (b->streaming && b->schedule == 1 && stages == b->fuse)
    b->ks->stream_batch_wq[b->shape - fds::kNumTiles][stages - 1](L, fds::xcd_grid(b->ntiles),
                                                                    0, b->stream);
  else if (b->streaming)
    b->ks->stream_batch[b->shape - fds::kNumTiles][stages - 1](L, fds::xcd_grid(b->ntiles), 0,
                                                                 b->stream);
  else
    b->ks->batch[b->shape](L, fds::xcd_grid(b->ntiles), b->lds, b->stream);
  HIP_TRY(hipGetLastError());
  return 0;
}

int batch_graph(fds_batch *b, int chunk, int rel_parity, hipGraphExec_t *out) {
  auto key = std::make_pair(chunk, rel_parity);
  auto it = b->graphs.find(key);
  if (it != b->graphs.end()) {
    *out = it->second;
    return 0;
  }
  HIP_TRY(hipStreamSynchronize(b->stream));
  HIP_TRY(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
  int rc = 0;
  const int grp = b->fuse;   // chunk is a multiple of grp
  for (int k = 0; k < chunk && rc == 0; k += grp)
    rc = batch_launch(b, rel_parity ^ ((k / grp) & 1), k, false, grp);
  if (rc == 0)
    hipLaunchKernelGGL(k_advance, dim3(1), dim3(64), 0, b->stream, b->dyn.as<int64_t>(),
                       (int64_t)chunk);
  hipGraph_t g = nullptr;
  hipError_t e = hipStreamEndCapture(b->stream, &g);
  if (rc) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  if (e != hipSuccess) return fail(FDS_E_HIP, "graph capture failed: %s", hipGetErrorString(e));
  hipGraphExec_t ex = nullptr;
  e = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
  if (e != hipSuccess) {
    (void)hipGraphDestroy(g);
    return fail(FDS_E_HIP, "graph instantiate failed: %s", hipGetErrorString(e));
  }
  b->graph_objs.push_back(g);
  b->graphs[key] = ex;
  HIP_TRY(hipGraphUpload(ex, b->stream));
  *out = ex;
  return 0;
}

// Checks a batch run's members, (re)builds the descriptors and output rows for nsteps steps
// and enqueues the step counters' start.
int batch_prepare(fds_batch *b, int64_t start, int64_t nsteps) {
  for (auto *c : b->ctxs) {
    if (!c->committed) return fail(FDS_E_STATE, "coefficients not committed");
    if (!c->flights.empty()) return fail(FDS_E_STATE, "a member has asynchronous runs in flight");
    for (int k = 0; k < 3; ++k)
      for (size_t e = 0; e < c->comp[k].len.size(); ++e)
        if (start + nsteps > c->comp[k].len[e])
          return fail(FDS_E_INDEX, "boundary signal too short for step %lld",
                      (long long)(start + nsteps - 1));
    HIP_TRY(hipStreamSynchronize(c->stream));
    if (int rc = leave_coupling(c)) return rc;
  }
  int rc = b->elem == 8 ? batch_build<double>(b, nsteps) : batch_build<float>(b, nsteps);
  if (rc) return rc;
  hipLaunchKernelGGL(k_set_dyn, dim3(1), dim3(64), 0, b->stream, b->dyn.as<int64_t>(), start);
  HIP_TRY(hipGetLastError());
  if (b->schedule == 1) {   // one empty counter per launch of the run
    const int64_t need = nsteps / std::max(1, b->fuse) + 2;
    if (need > std::numeric_limits<int32_t>::max())
      return fail(FDS_E_ARG, "run too long for the work queue");
    if (b->nq < need) {
      // a larger buffer (batch_steady made runs in flight finish first)
      HIP_TRY(b->queue.ensure((size_t)need * 2 * sizeof(unsigned)));
      b->nq = (int)(b->queue.bytes / sizeof(unsigned));
      batch_drop_graphs(b);   // captured launches hold the old buffer
    }
    const unsigned grid = (unsigned)std::min<int64_t>((need + 255) / 256, 1024);
    hipLaunchKernelGGL(k_queue_reset, dim3(grid), dim3(256), 0, b->stream,
                       b->queue.as<unsigned>(), (int)need);
    HIP_TRY(hipGetLastError());
  }
  for (auto *c : b->ctxs)
    if (c->nf_check) {
      hipLaunchKernelGGL(k_nonfinite_reset, dim3(1), dim3(64), 0, b->stream,
                         c->dyn.as<int64_t>());
      HIP_TRY(hipGetLastError());
    }
  return 0;
}

// True when batch_prepare rebuilds nothing (no device memory freed under a run in flight).
bool batch_steady(const fds_batch *b, int64_t nsteps) {
  for (const auto *c : b->ctxs)
    if (!run_steady(c, nsteps)) return false;
  if (b->schedule == 1 && b->nq < nsteps / std::max(1, b->fuse) + 2) return false;
  return !batch_stale(b);
}

// The steps of a prepared batch run between events e0 and e1; the members' buffer parities
// follow the launches.
int batch_enqueue(fds_batch *b, int64_t nsteps, int chunk, hipEvent_t e0, hipEvent_t e1) {
  HIP_TRY(hipEventRecord(e0, b->stream));
  int rel = b->flip;
  int64_t done = 0;
  const int g = b->fuse;
  if (chunk > 0) {
    chunk = std::max(g, chunk - chunk % g);
    while (nsteps - done > chunk) {
      hipGraphExec_t ex;
      if (int rc2 = batch_graph(b, chunk, rel, &ex)) return rc2;
      HIP_TRY(hipGraphLaunch(ex, b->stream));
      rel ^= ((chunk / g) & 1);
      done += chunk;
    }
  }
  const int64_t graph_done = done;   // steps the batch step counter advanced by
  // full launches, then the remainder: one launch on the fused engine, else one stage at a time
  // (batch kernels exist for the shape's stage count and for one stage)
  for (int64_t k = 0; done + k < nsteps;) {
    const int64_t rest = nsteps - done - k;
    const int st = rest >= g ? g : b->fused ? (int)rest : 1;
    if (int rc2 = batch_launch(b, rel, (int)k, done + k + st == nsteps, st)) return rc2;
    rel ^= 1;
    k += st;
  }
  HIP_TRY(hipEventRecord(e1, b->stream));
  // members advanced nsteps steps in lock step, flipping buffers once per launch
  if (rel != b->flip) {
    for (auto *c : b->ctxs) c->parity ^= 1;
    b->flip ^= 1;
  }
  // members that check for non-finite values: every component after the run
  for (auto *c : b->ctxs)
    if (c->nf_check)
      if (int rc2 = scan_all_nonfinite(c, c->parity, b->dyn.as<const int64_t>(),
                                       nsteps - graph_done, b->stream))
        return rc2;
  return 0;
}

// The first member whose non-finite check of staging slot `slot` failed, or 0.
int batch_check_nonfinite(const fds_batch *b, int slot) {
  for (size_t i = 0; i < b->ctxs.size(); ++i)
    if (int rc = check_nonfinite(b->ctxs[i], slot)) {
      const std::string msg = g_last_error;
      return fail(rc, "batch member %d: %s", (int)i, msg.c_str());
    }
  return 0;
}

}  // namespace

extern "C" {

int fds_batch_create(fds_batch **out, fds_ctx *const *ctxs, int n, int tile) {
  if (!out || !ctxs || n < 1) return fail(FDS_E_ARG, "batch needs at least one context");
  *out = nullptr;
  auto *b = new fds_batch();
  b->ctxs.assign(ctxs, ctxs + n);
  fds_ctx *c0 = ctxs[0];
  b->device = c0->device;
  b->form = c0->form;
  b->elem = c0->elem;
  b->ks = c0->ks;
  b->tile = tile;
  for (auto *c : b->ctxs) {
    if (!c || !c->committed) { delete b; return fail(FDS_E_STATE, "batch member not committed"); }
    if (!c->flights.empty() || c->batch_flights) {
      delete b;
      return fail(FDS_E_STATE, "a batch member has asynchronous runs in flight");
    }
    if (c->device != b->device || c->form != b->form) {
      delete b;
      return fail(FDS_E_ARG, "batch members must share device and form");
    }
    if (c->family == kNonlinear) {
      delete b;
      return fail(FDS_E_ARG, "nonlinear 1D models cannot be batched");
    }
    // the batch launches only the step kernels: a member's per-step flow shift or learned
    // boundary would be skipped
    if (c->flow || c->lbc_w1) {
      delete b;
      return fail(FDS_E_ARG, "members with flow (AcousticFlow2D) or a learned boundary "
                             "cannot be batched");
    }
  }
  hipError_t e = hipSetDevice(b->device);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking);
  if (e != hipSuccess) { delete b; return fail(FDS_E_HIP, "stream: %s", hipGetErrorString(e)); }
  if (int rc = batch_layout(b, true)) {
    fds_batch_destroy(b);
    return rc;
  }
  *out = b;
  return 0;
}

int fds_batch_set_schedule(fds_batch *b, int schedule) {
  if (!b) return fail(FDS_E_ARG, "null batch");
  if (schedule != 0 && schedule != 1) return fail(FDS_E_ARG, "schedule is 0 or 1");
  if (!b->flights.empty()) return fail(FDS_E_STATE, "asynchronous runs in flight");
  if (schedule == 1 && !b->streaming)
    return fail(FDS_E_ARG, "the work-queue schedule needs a streaming shape");
  if (b->schedule != schedule) {
    HIP_TRY(hipSetDevice(b->device));
    HIP_TRY(hipStreamSynchronize(b->stream));
    batch_drop_graphs(b);
    // (the fused engine has no work-queue kernels: such a batch goes to its streaming shape)
    b->schedule = schedule;
    if (b->fused || (schedule == 0 && b->tile < 0))
      if (int rc = batch_layout(b, true)) return rc;
  }
  return 0;
}

int fds_batch_destroy(fds_batch *b) {
  if (!b) return 0;
  (void)hipSetDevice(b->device);
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  batch_drop_graphs(b);
  if (b->ev0) (void)hipEventDestroy(b->ev0);
  if (b->ev1) (void)hipEventDestroy(b->ev1);
  for (auto &set : b->fev)
    for (auto e : set)
      if (e) (void)hipEventDestroy(e);
  // members no longer wait for this batch's runs
  for (size_t i = 0; i < b->flights.size(); ++i)
    for (auto *c : b->ctxs) c->batch_flights--;
  if (b->stream) (void)hipStreamDestroy(b->stream);
  delete b;
  return 0;
}

int fds_batch_run(fds_batch *b, int64_t start, int64_t nsteps, int chunk) {
  if (!b) return fail(FDS_E_ARG, "null batch");
  HIP_TRY(hipSetDevice(b->device));
  if (nsteps < 0 || start < 0) return fail(FDS_E_ARG, "negative step count");
  if (nsteps == 0) return 0;
  if (!b->flights.empty()) return fail(FDS_E_STATE, "asynchronous runs in flight: take them first");
  if (int rc = batch_prepare(b, start, nsteps)) return rc;
  if (!b->ev0) HIP_TRY(hipEventCreate(&b->ev0));
  if (!b->ev1) HIP_TRY(hipEventCreate(&b->ev1));
  if (int rc = batch_enqueue(b, nsteps, chunk, b->ev0, b->ev1)) return rc;
  for (auto *c : b->ctxs)
    if (int rc = stage_nonfinite(c, kMaxFlights, b->stream)) return rc;
  HIP_TRY(hipStreamSynchronize(b->stream));
  float ms = 0.f;
  HIP_TRY(hipEventElapsedTime(&ms, b->ev0, b->ev1));
  b->last_run_ms = ms;
  return batch_check_nonfinite(b, kMaxFlights);
}

int fds_batch_run_async(fds_batch *b, int64_t start, int64_t nsteps, int chunk) {
  if (!b) return fail(FDS_E_ARG, "null batch");
  HIP_TRY(hipSetDevice(b->device));
  if (nsteps < 1 || start < 0) return fail(FDS_E_ARG, "an asynchronous run needs steps");
  if ((int)b->flights.size() >= kMaxFlights)
    return fail(FDS_E_STATE, "%d runs in flight: take the oldest first", kMaxFlights);
  if (!batch_steady(b, nsteps)) HIP_TRY(hipStreamSynchronize(b->stream));
  if (int rc = batch_prepare(b, start, nsteps)) return rc;
  const int slot = b->next_slot;
  if (int rc = ensure_events(b->fev[slot])) return rc;
  if (int rc = batch_enqueue(b, nsteps, chunk, b->fev[slot][0], b->fev[slot][1])) return rc;
  for (auto *c : b->ctxs) {
    if (int rc = stage_outputs(c, slot, nsteps, b->stream)) return rc;
    if (int rc = stage_nonfinite(c, slot, b->stream)) return rc;
  }
  HIP_TRY(hipEventRecord(b->fev[slot][2], b->stream));
  if (b->flights.empty()) b->last_run_ms = 0.0;
  b->flights.push_back(Flight{nsteps, slot});
  for (auto *c : b->ctxs) c->batch_flights++;
  b->next_slot = (slot + 1) % kMaxFlights;
  return 0;
}

int fds_batch_take(fds_batch *b, double *const *dst) {
  if (!b) return fail(FDS_E_ARG, "null batch");
  HIP_TRY(hipSetDevice(b->device));
  if (b->flights.empty()) return fail(FDS_E_STATE, "no asynchronous run in flight");
  const Flight f = b->flights.front();
  HIP_TRY(hipEventSynchronize(b->fev[f.slot][2]));
  b->flights.pop_front();
  for (size_t i = 0; i < b->ctxs.size(); ++i) {
    b->ctxs[i]->batch_flights--;
    if (dst) take_outputs(b->ctxs[i], f, dst + 3 * i);
  }
  float ms = 0.f;
  HIP_TRY(hipEventElapsedTime(&ms, b->fev[f.slot][0], b->fev[f.slot][1]));
  b->last_run_ms += ms;
  return batch_check_nonfinite(b, f.slot);
}

int fds_batch_last_run_ms(fds_batch *b, double *ms) {
  if (!b || !ms) return fail(FDS_E_ARG, "null argument");
  *ms = b->last_run_ms;
  return 0;
}

int fds_batch_steps_per_launch(fds_batch *b) {
  if (!b) return fail(FDS_E_ARG, "null batch");
  return b->fuse;
}

}  // extern "C"

namespace {

template <typename TA, typename TB>
__global__ __launch_bounds__(256) void k_window_sq_diff(const TA *__restrict__ a, int anx,
                                                        const TB *__restrict__ b, int bnx,
                                                        int wx, int wy, int ax0, int ay0,
                                                        int bx0, int by0,
                                                        double *__restrict__ out) {
  __shared__ double r0[256], r1[256];
  double num = 0.0, den = 0.0;
  const int64_t n = (int64_t)wx * wy;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const int iy = (int)(i / wx), ix = (int)(i % wx);
    const double va = (double)a[(int64_t)(ay0 + iy) * anx + ax0 + ix];
    const double vb = (double)b[(int64_t)(by0 + iy) * bnx + bx0 + ix];
    const double d = va - vb;
    num += d * d;
    den += vb * vb;
  }
  r0[threadIdx.x] = num;
  r1[threadIdx.x] = den;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      r0[threadIdx.x] += r0[threadIdx.x + s];
      r1[threadIdx.x] += r1[threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[2 * blockIdx.x] = r0[0];
    out[2 * blockIdx.x + 1] = r1[0];
  }
}

const void *current_state(const fds_ctx *c, int comp) {
  const Comp &cp = c->comp[comp];
  const int b = (cp.buf[1].p && (cp.accumulated || c->family != kThermal || comp == 0)) ? c->parity : 0;
  return cp.buf[b].p;
}

}  // namespace

namespace {

constexpr int kWindowBlocks = 512;   // workgroups of the window reduction (partial sums each)

// Partial sums of the no-allocation window reduction: one array per GPU, held by the process
// until it ends.  Host code uses its device address from hipGetSymbolAddress (window_scratch),
// never the array's name.
static __device__ __align__(256) double scratch[2 * kWindowBlocks];

// Device address of `scratch` on `device`, looked up once per device (with it current).
int window_scratch(int device, double **out) {
  static std::mutex mu;
  static std::map<int, double *> ptrs;
  std::lock_guard<std::mutex> lock(mu);
  auto it = ptrs.find(device);
  if (it == ptrs.end()) {
    double *p = nullptr;
    HIP_TRY(hipSetDevice(device));
    const hipError_t e = hipGetSymbolAddress(reinterpret_cast<void **>(&p), HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(FDS_E_HIP, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
    it = ptrs.emplace(device, p).first;
  }
  *out = it->second;
  return 0;
}

// The window reduction of fds_window_sq_diff into `part` (2 * kWindowBlocks doubles, device),
// summed on the host in block order.
int window_sq_diff(fds_ctx *a, int comp_a, fds_ctx *b, int comp_b, int wx, int wy, int ax0,
                   int ay0, int bx0, int by0, double *part, double *num, double *den) {
  const int blocks = kWindowBlocks;
  const void *pa = current_state(a, comp_a), *pb = current_state(b, comp_b);
  const int anx = (int)a->nx, bnx = (int)b->nx;
  double *o = part;
  if (a->elem == 8 && b->elem == 8)
    hipLaunchKernelGGL((k_window_sq_diff<double, double>), dim3(blocks), dim3(256), 0, a->stream,
                       (const double *)pa, anx, (const double *)pb, bnx, wx, wy, ax0, ay0, bx0, by0, o);
  else if (a->elem == 4 && b->elem == 4)
    hipLaunchKernelGGL((k_window_sq_diff<float, float>), dim3(blocks), dim3(256), 0, a->stream,
                       (const float *)pa, anx, (const float *)pb, bnx, wx, wy, ax0, ay0, bx0, by0, o);
  else if (a->elem == 4)
    hipLaunchKernelGGL((k_window_sq_diff<float, double>), dim3(blocks), dim3(256), 0, a->stream,
                       (const float *)pa, anx, (const double *)pb, bnx, wx, wy, ax0, ay0, bx0, by0, o);
  else
    hipLaunchKernelGGL((k_window_sq_diff<double, float>), dim3(blocks), dim3(256), 0, a->stream,
                       (const double *)pa, anx, (const float *)pb, bnx, wx, wy, ax0, ay0, bx0, by0, o);
  HIP_TRY(hipGetLastError());
  double h[2 * kWindowBlocks];
  HIP_TRY(hipMemcpyAsync(h, o, sizeof h, hipMemcpyDeviceToHost, a->stream));
  HIP_TRY(hipStreamSynchronize(a->stream));
  double s0 = 0, s1 = 0;
  for (int i = 0; i < blocks; ++i) {
    s0 += h[2 * i];
    s1 += h[2 * i + 1];
  }
  *num = s0;
  *den = s1;
  return 0;
}

int window_checks(fds_ctx *a, int comp_a, fds_ctx *b, int comp_b, int wx, int wy, int ax0,
                  int ay0, int bx0, int by0, double *num, double *den) {
  if (int rc = check_idle(a)) return rc;
  if (!b || b->device != a->device) return fail(FDS_E_ARG, "contexts must share a device");
  if (int rc = check_idle(b)) return rc;
  if (int rc = check_comp(a, comp_a)) return rc;
  if (int rc = check_comp(b, comp_b)) return rc;
  if (!num || !den) return fail(FDS_E_ARG, "null output");
  if (wx < 1 || wy < 1 || ax0 < 0 || ay0 < 0 || bx0 < 0 || by0 < 0 || ax0 + wx > a->nx ||
      ay0 + wy > a->ny || bx0 + wx > b->nx || by0 + wy > b->ny)
    return fail(FDS_E_INDEX, "window outside a grid");
  HIP_TRY(hipStreamSynchronize(b->stream));
  return 0;
}

}  // namespace

extern "C" int fds_window_sq_diff(fds_ctx *a, int comp_a, fds_ctx *b, int comp_b, int wx, int wy,
                                  int ax0, int ay0, int bx0, int by0, double *num, double *den) {
  if (int rc = window_checks(a, comp_a, b, comp_b, wx, wy, ax0, ay0, bx0, by0, num, den))
    return rc;
  DevBuf part;
  HIP_TRY(part.ensure(2 * kWindowBlocks * sizeof(double)));
  return window_sq_diff(a, comp_a, b, comp_b, wx, wy, ax0, ay0, bx0, by0, part.as<double>(),
                        num, den);
}

extern "C" int fds_window_sq_diff_static(fds_ctx *a, int comp_a, fds_ctx *b, int comp_b, int wx,
                                         int wy, int ax0, int ay0, int bx0, int by0, double *num,
                                         double *den) {
  if (int rc = window_checks(a, comp_a, b, comp_b, wx, wy, ax0, ay0, bx0, by0, num, den))
    return rc;
  double *part = nullptr;
  if (int rc = window_scratch(a->device, &part)) return rc;
  return window_sq_diff(a, comp_a, b, comp_b, wx, wy, ax0, ay0, bx0, by0, part, num, den);
}

extern "C" int fds_output_device_ptr(fds_ctx *c, int comp, double **ptr, int64_t *rows, int64_t *m) {
  if (int rc = check_idle(c)) return rc;
  if (int rc = check_comp(c, comp)) return rc;
  *ptr = c->comp[comp].obuf.as<double>();
  *rows = c->comp[comp].obuf_rows;
  *m = (int64_t)c->comp[comp].out_cells.size();
  return 0;
}

#include "fds_couple.inc"

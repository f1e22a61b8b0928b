// Fused step kernels of the lossless 2D models (Acoustic2D / Acoustic3DAxi and Thermal2D /
// Thermal3DAxi): S time steps per launch on one-wave strips, the default engine.
//
// A workgroup is one wave.  It owns a strip of H rows and 64 - 2G columns (G >= S ghost columns
// on each side) and marches down the rows.  Stage s (0 .. S-1) advances the field from step
// n + s to n + s + 1 and takes one row per iteration: from row r of its input it forms the
// velocities (fluxes) of row r and, with those of row r - 1 kept from the iteration before, the
// pressure (temperature) of row r - 1.  So a stage hands on row r - 1 complete, the next stage
// takes it in the same iteration, and only the last stage's rows are stored.  A strip of H rows
// takes H + 2S iterations; the first 2S are unrolled with the stages that have no row yet left
// out, each of the H others stores one row.
//
// What bounds it: at one step per launch the step moves 48 B (acoustics, FP64) a cell and HBM is
// the bound; S steps per launch divide that by S, until the ghost rows and columns and the
// instructions of the stages cost as much.  Acoustic2D 2048^2 FP64, a launch: S = 1 32 us, S = 4
// 36 us, S = 6 42 us (205 MB of state read and written once: 4.9 TB/s), so 7.0 us a step against
// 45 us for two steps per launch on register-path strips (fds_stream2d.h, the engine before).
// Eight stages would not fit the registers of two waves per SIMD in FP64.
//
// Columns: lane t holds column x0 + t, the x neighbours come by DPP wave shifts.  The outermost
// lanes miss a neighbour, and each stage makes one more column per side wrong; only the columns
// at least G from the edges are stored.  (Loading the missing neighbour columns would save two
// columns of 64 and cost every row five loads and the edge selects.)
//
// Rows are read and written through buffer descriptors whose range is the array: a read outside
// it returns zero, which is the reference's zero ghost, and a lane that must not store gets an
// offset outside it.  Rows therefore need no bounds tests, no alignment and no branches, and
// the loop body is one straight line: the compiler counts the loads in flight exactly, so PF
// rows of loads stay in flight across the waits (FP64 acoustics, S = 4: 92 instructions a row,
// against 228 for three stages of the LDS-ring strips).
//
// Coefficients: a field of few materials (PAL) reads one byte a cell, the cell's material class,
// and takes the class's coefficients from LDS; others read the coefficient arrays.
//
// Arithmetic: the tile kernel's expressions, term by term, in the same order, so FP64 results
// are bit-identical to the reference whatever S, H and PF are.
//
// Events: a tile with boundary cells or recorded points carries a word per cell of its region
// (class of each component's boundary program, recorded-point flags; FusedEv), which travels
// with its row.  A class is a chain of (factor, value of each stage) in LDS, evaluated once per
// launch, so applying it is one LDS lookup per lane, however many cells the row has.  Such a
// tile takes about twice a plain one's time (iterations with such a row in a stage four times),
// so these tiles are launched first: 2048^2, S = 4, rigid wall on one side: 57 us a launch in
// tile order, 38 us with them first (36 us without events).
#pragma once

#include <type_traits>

#include "fds_common.h"
#include "fds_step2d.h"
#include "fds_stream2d.h"
#include "../../include/pyfds_amd.h"

namespace fds {

using BufRsrc = __amdgpu_buffer_rsrc_t;

// Descriptor of an array of n elements (raw buffer, stride 0, 32-bit data format).
template <typename T>
__device__ __forceinline__ BufRsrc buf_rsrc(const T *p, int64_t n) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(p), 0, (int)(n * (int64_t)sizeof(T)),
                                           0x00027000);
}

constexpr uint32_t kBufOutside = 0xffffff00u;   // byte offset outside every descriptor's range

template <typename T>
__device__ __forceinline__ T buf_load(BufRsrc r, uint32_t off) {
  if constexpr (sizeof(T) == 8) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0);
    return __builtin_bit_cast(T, v);
  } else {
    const auto v = __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
    return __builtin_bit_cast(T, v);
  }
}

template <typename T>
__device__ __forceinline__ void buf_store(BufRsrc r, uint32_t off, T v) {
  if constexpr (sizeof(T) == 8) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), r, (int)off, 0, 0);
  } else {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, (int)off, 0, 0);
  }
}

// One boundary class entry at one stage: x = a*x + v.
struct FusedTerm {
  double a, v;
};

// LDS of a fused workgroup: the material classes' coefficients (PAL) and the tile's boundary
// classes (entry 0: none): term[s] at stage s, then the entry `next` (0: last).
template <typename T, bool ISO, int S>
struct FusedLds {
  static constexpr int NC = ISO ? 2 : 4;   // bx, kx[, by, ky]
  __attribute__((aligned(16))) T pal[kPalMax][NC];
  FusedTerm term[S][kFusedClasses];
  uint8_t next[kFusedClasses];
};

// One row of one column.
template <typename T>
struct FuRow {
  T p, cp, vx, cvx, vy, cvy;
};

template <typename T>
struct FuCoef {
  T bx, by, kx, ky;
};

// What a stage keeps of the row before.
template <typename T>
struct FuCarry {
  T p, cp, bpy, kvy, kvd, vx, cvx, vy, cvy;
};

// The tile's events: classes in LDS, recorded points by row.
struct FusedEvents {
  const FusedTerm *term;    // [stage][class]
  const uint8_t *next;
  const OutView *out;
  const FusedPoint *point;
  bool chained;             // some class has a next entry
  bool few;                 // the tile has at most 64 recorded points, one a lane:
  uint32_t where;           // this lane's (FusedPoint; none: all bits)
  int32_t id;
  const int32_t *rows;      // first point of (component, row of the strip), rows + 1 a component
  int stride;
  int64_t row;              // output row of stage 0
};

// What a row's event words hold (bits of a uniform mask): boundary cells of component k
// (1 << k), its recorded points (8 << k).
constexpr uint32_t kRowRecord = 0x38u;

// Entry of component K's boundary class in event word w.
template <int K>
__device__ __forceinline__ uint32_t fused_class(uint32_t w) {
  return (w >> (8 * K)) & 0xffu;
}

// Component K's boundary at stage s for the cell with event word w, whose class's first entry is
// m (a cell without one: class 0).
template <typename T, bool KAHAN, int K>
__device__ __forceinline__ void fused_bound(const FusedEvents &E, const FusedTerm &m, int s,
                                            uint32_t w, T &x, T &c) {
  const bool hit = fused_class<K>(w) != 0;
  double v = KAHAN ? (double)x - (double)c : (double)x;
  {
    const double ax = m.a * v;
    v = ax + m.v;
  }
  if (E.chained) {          // (uniform) some cell of the tile has more than one entry
    uint32_t cls = E.next[fused_class<K>(w)];
    while (__any(cls != 0)) {
      if (cls != 0) {
        const FusedTerm q = E.term[s * kFusedClasses + cls];
        const double ax = q.a * v;
        v = ax + q.v;
        cls = E.next[cls];
      }
    }
  }
  if (hit) {
    x = (T)v;
    if (KAHAN) c = (T)((double)x - v);
  }
}

// The first entries of the row's boundary classes, read ahead of their use.
__device__ __forceinline__ void fused_terms(const FusedEvents &E, int s, uint32_t w, uint32_t any,
                                            FusedTerm (&m)[3]) {
  if (any & 7u) {
    m[0] = E.term[s * kFusedClasses + fused_class<0>(w)];
    m[1] = E.term[s * kFusedClasses + fused_class<1>(w)];
    m[2] = E.term[s * kFusedClasses + fused_class<2>(w)];
  } else {
    m[0] = m[1] = m[2] = FusedTerm{1.0, 0.0};
  }
}

// Recorded points of row r of the strip at stage s (components K0 .. K1 - 1; `any`: what the row
// holds).  A point's value comes from the lane of its column.  The points of the usual tile are in
// its lanes' registers; lists are read only for more than 64 of them.  (With lists for all, a row
// with a point cost three dependent lookups a stage, and the addresses of all stages 30 registers
// that every tile paid for in occupancy: 1056^2 FP32 with a source and four points 19.2 us a
// launch of six steps then, 17.6 so; 4096^2 Thermal2D Kahan 16.5 us a step and 13.5.)
template <typename T, bool KAHAN, int K0 = 0, int K1 = 3>
__device__ __forceinline__ void fused_record(const FusedEvents &E, int s, int r, uint32_t any, T p,
                                             T cp, T vx, T cvx, T vy, T cvy) {
  const int t = threadIdx.x;
#pragma unroll
  for (int k = K0; k < K1; ++k) {
    if (!(any & (8u << k))) continue;
    const T x = k == 0 ? p : k == 1 ? vx : vy, c = k == 0 ? cp : k == 1 ? cvx : cvy;
    int64_t row = E.row;
    __asm__ volatile("" : "+v"(row));     // (else the addresses of all stages stay in registers)
    double *buf = E.out[k].buf + (row + s) * E.out[k].m;
    if (E.few) {
      const int col = E.where & 63;
      const T xv = __shfl(x, col), cv = KAHAN ? __shfl(c, col) : T(0);
      int32_t id = E.id;
      __asm__ volatile("" : "+v"(id));
      if (E.where >> 6 == (uint32_t)(k | r << 2)) buf[id] = out_value<T, KAHAN>(xv, cv);
      continue;
    }
    const int e0 = E.rows[k * E.stride + r], e1 = E.rows[k * E.stride + r + 1];
    for (int e = e0; e < e1; e += 64) {
      const bool in = e + t < e1;
      const FusedPoint q = E.point[in ? e + t : e0];
      const int col = q.where & 63;
      const T xv = __shfl(x, col), cv = KAHAN ? __shfl(c, col) : T(0);
      if (in) buf[q.id] = out_value<T, KAHAN>(xv, cv);
    }
  }
}

// The events of the tile in word slot `slot`; its classes go to LDS, lane q evaluates entry q for
// every stage.
template <int S, typename T>
__device__ __forceinline__ FusedEvents fused_events(const StepArgs<T> &a, int slot, int64_t step,
                                                    int64_t row,
                                                    FusedTerm (&term)[S][kFusedClasses],
                                                    uint8_t (&next)[kFusedClasses]) {
  const FusedEv &fe = a.fev;
  const int t = threadIdx.x, stride = a.strip_h + 1;
  FusedEvents E;
  E.term = &term[0][0];
  E.next = next;
  E.out = a.outp;
  E.point = fe.points;
  E.stride = stride;
  E.rows = fe.point_rows + (int64_t)slot * 3 * stride;
  E.row = row;
  const int p0 = E.rows[0], np = E.rows[3 * stride - 1] - p0;
  E.few = np <= 64;
  E.where = ~0u;
  E.id = 0;
  if (E.few && t < np) {
    E.where = fe.points[p0 + t].where;
    E.id = fe.points[p0 + t].id;
  }
  const int e0 = fe.cls_ptr[slot], e1 = fe.cls_ptr[slot + 1];
  bool chained = false;
  if (t == 0) {
    next[0] = 0;
    for (int s = 0; s < S; ++s) term[s][0] = FusedTerm{1.0, 0.0};
  }
  for (int q = t; q < e1 - e0; q += 64) {
    const FusedClass cl = fe.cls[e0 + q];
    next[q + 1] = (uint8_t)cl.next;
    chained = chained || cl.next != 0;
#pragma unroll
    for (int s = 0; s < S; ++s)
      term[s][q + 1] = FusedTerm{cl.a, a.prog[cl.comp].table[cl.off + (step + s) * cl.stride]};
  }
  E.chained = __any(chained);
  __syncthreads();
  return E;
}

// What the row with event words w holds.
__device__ __forceinline__ uint32_t fused_row_flags(uint32_t w) {
  if (!__any(w != 0)) return 0;
  return (__any(fused_class<0>(w) != 0) ? 1u : 0u) | (__any(fused_class<1>(w) != 0) ? 2u : 0u) |
         (__any(fused_class<2>(w) != 0) ? 4u : 0u) | (__any(w & kFusedRecord) ? 8u : 0u) |
         (__any(w & kFusedRecord << 1) ? 16u : 0u) | (__any(w & kFusedRecord << 2) ? 32u : 0u);
}

// One stage of the lossless acoustic step: takes row r in x, leaves row r - 1 of the next time
// level in x.  kr = kx / rad (AXI).
template <typename T, bool KAHAN, bool AXI, bool ISO, bool EV>
__device__ __forceinline__ void fused_acoustic_stage(FuCarry<T> &c, FuRow<T> &x,
                                                     const FuCoef<T> &k, T rad, int s,
                                                     uint32_t w, uint32_t any, int r,
                                                     const FusedEvents &E) {
  FusedTerm m[3];
  if constexpr (EV) fused_terms(E, s, w, any, m);
  if constexpr (EV) {
    if (any & 1u) fused_bound<T, KAHAN, 0>(E, m[0], s, w, x.p, x.cp);
  }
  const T bpx = k.bx * x.p;
  const T bpy = ISO ? bpx : k.by * x.p;
  const T left = wave_from_left(bpx);
  const T dvx = (-left) + bpx;
  T vx = x.vx, cvx = x.cvx;
  if (KAHAN) kahan_sub(vx, cvx, dvx); else vx = vx - dvx;
  if constexpr (EV) {
    if (any & 2u) fused_bound<T, KAHAN, 1>(E, m[1], s, w, vx, cvx);
  }
  const T kvx = AXI ? k.kx * (vx * rad) : k.kx * vx;
  const T right = wave_from_right(kvx);
  const T kvd = (-kvx) + right;
  const T dvy = (-c.bpy) + bpy;
  T vy = x.vy, cvy = x.cvy;
  if (KAHAN) kahan_sub(vy, cvy, dvy); else vy = vy - dvy;
  if constexpr (EV) {
    if (any & 4u) fused_bound<T, KAHAN, 2>(E, m[2], s, w, vy, cvy);
  }
  if constexpr (EV) {
    if (any & kRowRecord) fused_record<T, KAHAN>(E, s, r, any, x.p, x.cp, vx, cvx, vy, cvy);
  }
  const T kvy = k.ky * vy;
  const T dy = (-c.kvy) + kvy;
  const T d = c.kvd + dy;
  T p = c.p, cp = c.cp;
  if (KAHAN) kahan_sub(p, cp, d); else p = p - d;
  const FuRow<T> out{p, cp, c.vx, c.cvx, c.vy, c.cvy};
  c = FuCarry<T>{x.p, x.cp, bpy, kvy, kvd, vx, cvx, vy, cvy};
  x = out;
}

// One stage of the thermal step (p: temperature; vx, vy: the fluxes, assigned, of row r - 1 on
// return).  Coefficients: bx, by = Qx, Qy; kx, ky = Gx (over the radius: AXI), Gy.
template <typename T, bool KAHAN, bool AXI, bool ISO, bool EV>
__device__ __forceinline__ void fused_thermal_stage(FuCarry<T> &c, FuRow<T> &x, const FuCoef<T> &k,
                                                    T rad, int s, uint32_t w, uint32_t any,
                                                    int r, const FusedEvents &E) {
  FusedTerm m[3];
  if constexpr (EV) fused_terms(E, s, w, any, m);
  if constexpr (EV) {
    if (any & 1u) fused_bound<T, KAHAN, 0>(E, m[0], s, w, x.p, x.cp);
  }
  T none = T(0);
  const T qtx = k.bx * x.p;
  const T qty = ISO ? qtx : k.by * x.p;
  const T left = wave_from_left(qtx);
  T fx = -((-left) + qtx);
  if constexpr (EV) {
    if (any & 2u) fused_bound<T, false, 1>(E, m[1], s, w, fx, none);
  }
  const T gqx = AXI ? k.kx * (fx * rad) : k.kx * fx;
  const T right = wave_from_right(gqx);
  const T gqd = (-gqx) + right;
  T fy = -((-c.bpy) + qty);
  if constexpr (EV) {
    if (any & 4u) fused_bound<T, false, 2>(E, m[2], s, w, fy, none);
  }
  if constexpr (EV) {
    if (any & kRowRecord) fused_record<T, KAHAN>(E, s, r, any, x.p, x.cp, fx, T(0), fy, T(0));
  }
  const T gqy = k.ky * fy;
  const T dy = (-c.kvy) + gqy;
  const T d = c.kvd + dy;
  T p = c.p, cp = c.cp;
  if (KAHAN) kahan_sub(p, cp, d); else p = p - d;
  const FuRow<T> out{p, cp, c.vx, T(0), c.vy, T(0)};
  c = FuCarry<T>{x.p, x.cp, qty, gqy, gqd, fx, T(0), fy, T(0)};
  x = out;
}

// A copy of v in a register of its own.
template <typename T>
__device__ __forceinline__ T fused_copy(T v) {
  __asm__ volatile("" : "+v"(v));
  return v;
}

// The strip of tile `tile`: S stages, PF rows of loads in flight.
template <typename T, bool KAHAN, bool THERMAL, bool AXI, bool ISO, bool PAL, bool EV, int S,
          int PF>
__device__ __forceinline__ void fused_strip(const StepArgs<T> &a, int tile, int slot, int64_t step,
                                            int64_t row, FusedLds<T, ISO, S> &L) {
  constexpr int RS = PF + 1;          // row slots of the loads in flight
  const int G = a.ghost, sx = a.sx, H = a.strip_h;
  const int t = threadIdx.x;
  const int ty = tile / a.tiles_x, tx = tile - ty * a.tiles_x;
  const int x0 = tx * sx - G, y0 = ty * H;
  const int nx = a.nx;
  const int rows = a.ny - y0 < H ? a.ny - y0 : H;      // rows this strip stores
  const bool owned = t >= G && t < G + sx && x0 + t < nx;
  const bool store = (a.flags & kFlagStore) != 0;
  constexpr int CB = THERMAL ? FDS_C_QX : FDS_C_BX, CK = THERMAL ? FDS_C_GX : FDS_C_KX;
  const BufRsrc in0 = buf_rsrc(a.in[0], a.n), in1 = buf_rsrc(a.in[1], a.n),
                in2 = buf_rsrc(a.in[2], a.n);
  const BufRsrc out0 = buf_rsrc(a.out[0], a.n), out1 = buf_rsrc(a.out[1], a.n),
                out2 = buf_rsrc(a.out[2], a.n);
  const BufRsrc cin0 = buf_rsrc(KAHAN ? a.cin[0] : a.in[0], a.n),
                cin1 = buf_rsrc(KAHAN ? a.cin[1] : a.in[0], a.n),
                cin2 = buf_rsrc(KAHAN ? a.cin[2] : a.in[0], a.n);
  const BufRsrc cout0 = buf_rsrc(KAHAN ? a.cout[0] : a.out[0], a.n),
                cout1 = buf_rsrc(KAHAN ? a.cout[1] : a.out[0], a.n),
                cout2 = buf_rsrc(KAHAN ? a.cout[2] : a.out[0], a.n);
  const BufRsrc rbx = buf_rsrc(a.coef[CB], a.n), rby = buf_rsrc(a.coef[CB + 1], a.n),
                rkx = buf_rsrc(a.coef[CK], a.n), rky = buf_rsrc(a.coef[CK + 1], a.n);
  const BufRsrc ridx = buf_rsrc(PAL ? a.pal_idx : (const uint8_t *)a.in[0], a.n);
  if constexpr (PAL) {
    if (t < a.npal) {
      constexpr int NC = FusedLds<T, ISO, S>::NC;
#pragma unroll
      for (int q = 0; q < NC; ++q) L.pal[t][q] = a.pal[t * kPalSlots + q];
    }
    __syncthreads();
  }
  T rad = T(1);
  if (AXI) rad = radius<T>(wrap_any(x0 + t, nx), a.s[FDS_S_DX], a.s[FDS_S_HALF_DX]);

  // ghost_rows + 1 rows above the strip come first
  const BufRsrc words = EV ? buf_rsrc(a.fev.words + (int64_t)slot * a.fev.rows * 64,
                                      (int64_t)a.fev.rows * 64)
                           : buf_rsrc((const uint32_t *)a.in[0], 0);
  FusedEvents E{};
  if constexpr (EV) E = fused_events<S>(a, slot, step, row, L.term, L.next);

  struct Slot {
    FuRow<T> x;
    FuCoef<T> k;
    uint32_t w, m;
  };
  Slot in[RS];
  // row ordinal o of the launch is row o - S of the strip; rows past the last one needed are
  // that row again
  const int last = rows + S - 1;
  auto load = [&](int o, Slot &d) __attribute__((always_inline)) {
    const int rho = o - S < last ? o - S : last;
    const uint32_t off = (uint32_t)((y0 + rho) * nx + x0 + t) * (uint32_t)sizeof(T);
    d.x.p = buf_load<T>(in0, off);
    if constexpr (PAL) {
      d.m = __builtin_amdgcn_raw_buffer_load_b8(ridx, (y0 + rho) * nx + x0 + t, 0, 0);
    } else {
      d.k.bx = buf_load<T>(rbx, off);
      d.k.kx = buf_load<T>(rkx, off);
      if (!ISO) {
        d.k.by = buf_load<T>(rby, off);
        d.k.ky = buf_load<T>(rky, off);
      }
    }
    if (!THERMAL) {
      d.x.vx = buf_load<T>(in1, off);
      d.x.vy = buf_load<T>(in2, off);
    } else {
      d.x.vx = d.x.vy = T(0);
    }
    if (KAHAN) {
      d.x.cp = buf_load<T>(cin0, off);
      if (!THERMAL) {
        d.x.cvx = buf_load<T>(cin1, off);
        d.x.cvy = buf_load<T>(cin2, off);
      }
    }
    if (!KAHAN || THERMAL) d.x.cvx = d.x.cvy = T(0);
    if (!KAHAN) d.x.cp = T(0);
    d.w = EV ? buf_load<uint32_t>(words, (uint32_t)((rho + a.ghost_rows + 1) * 64 + t) * 4u) : 0u;
  };
  static_for<PF>([&](auto Oc) __attribute__((always_inline)) {
    load(decltype(Oc)::value, in[decltype(Oc)::value]);
  });

  FuCarry<T> c[S] = {};
  // of the rows in the stages: coefficients (PAL: only AXI's kx / rad, the others come from
  // LDS), material classes, event words
  FuCoef<T> kc[S] = {};
  uint32_t mc[S] = {};
  uint32_t wc[S] = {};
  uint32_t ac[S] = {};       // what the rows hold (uniform)
  int busy = 0;              // iterations until no row with events is in a stage
  // iteration i: stage s takes row i - S - s; `FIRST` stages have a row
  auto iterate = [&](auto Wc, auto NSc, int i) __attribute__((always_inline)) -> FuRow<T> {
    constexpr int W = decltype(Wc)::value, NS = decltype(NSc)::value;
    load(i + PF, in[(W + PF) % RS]);
    const uint32_t above = mc[0];
    static_for<S - 1, true>([&](auto Sc) __attribute__((always_inline)) {
      constexpr int s = decltype(Sc)::value + 1;
      kc[s] = kc[s - 1];
      mc[s] = mc[s - 1];
      wc[s] = wc[s - 1];
      ac[s] = ac[s - 1];
    });
    FuRow<T> x = in[W].x;
    if constexpr (PAL) {
      mc[0] = in[W].m;
      // the quotient again only where a row brings another class
      if (AXI && __any(mc[0] != above)) kc[0].kx = L.pal[mc[0]][1] / rad;
    } else {
      // copies: the slots are loaded again while the rows' coefficients are still in use
      kc[0].bx = fused_copy(in[W].k.bx);
      kc[0].kx = fused_copy(in[W].k.kx);
      kc[0].by = ISO ? kc[0].bx : fused_copy(in[W].k.by);
      kc[0].ky = ISO ? kc[0].kx : fused_copy(in[W].k.ky);
      if (AXI) kc[0].kx = kc[0].kx / rad;
    }
    if constexpr (EV) {
      wc[0] = in[W].w;
      ac[0] = fused_row_flags(wc[0]);
      if (ac[0]) busy = S;
    }
    auto stages = [&](auto EVc) __attribute__((always_inline)) {
      constexpr bool E1 = decltype(EVc)::value;
      static_for<NS>([&](auto Sc) __attribute__((always_inline)) {
        constexpr int s = decltype(Sc)::value;
        FuCoef<T> k = kc[s];
        if constexpr (PAL) {
          const T *m = L.pal[mc[s]];
          k.bx = m[0];
          if (!AXI) k.kx = m[1];
          k.by = ISO ? k.bx : m[2];
          k.ky = ISO ? k.kx : m[3];
        }
        if constexpr (THERMAL)
          fused_thermal_stage<T, KAHAN, AXI, ISO, E1>(c[s], x, k, rad, s, wc[s], ac[s], i - S - s,
                                                      E);
        else
          fused_acoustic_stage<T, KAHAN, AXI, ISO, E1>(c[s], x, k, rad, s, wc[s], ac[s],
                                                       i - S - s, E);
      });
    };
    if constexpr (EV) {
      // rows without events run the plain stages, one straight line
      if (busy > 0) {
        --busy;
        stages(std::true_type{});
      } else {
        stages(std::false_type{});
      }
    } else {
      stages(std::false_type{});
    }
    return x;
  };
  // tiles with events (their stages are long code): the first 2S rows go through the loop too,
  // all stages active (what a stage makes of a row it does not have yet reaches no row it has)
  constexpr int P = EV ? 0 : 2 * S;
  static_for<P>([&](auto Ic) __attribute__((always_inline)) {
    constexpr int i = decltype(Ic)::value;
    constexpr int NS = i / 2 + 1 < S ? i / 2 + 1 : S;
    (void)iterate(std::integral_constant<int, i % RS>{}, std::integral_constant<int, NS>{}, i);
  });
  auto put = [&](int m, const FuRow<T> &x) __attribute__((always_inline)) {
    const uint32_t o = (uint32_t)((y0 + m) * nx + x0 + t) * (uint32_t)sizeof(T);
    const uint32_t off = owned ? o : kBufOutside;
    buf_store<T>(out0, off, x.p);
    if (KAHAN) buf_store<T>(cout0, off, x.cp);
    if (!THERMAL) {
      buf_store<T>(out1, off, x.vx);
      buf_store<T>(out2, off, x.vy);
      if (KAHAN) {
        buf_store<T>(cout1, off, x.cvx);
        buf_store<T>(cout2, off, x.cvy);
      }
    } else if (store) {
      buf_store<T>(out1, off, x.vx);
      buf_store<T>(out2, off, x.vy);
    }
  };
  // one row; true: it was the strip's last
  auto one = [&](auto Jc, int m) __attribute__((always_inline)) -> bool {
    constexpr int J = decltype(Jc)::value;
    const FuRow<T> x = iterate(std::integral_constant<int, (P + J) % RS>{},
                               std::integral_constant<int, S>{}, 2 * S + m + J);
    if (!EV || m + J >= 0) put(m + J, x);
    return m + J + 1 >= rows;
  };
  static_assert(RS <= 6, "the row loop is written out for at most six slots");
  for (int m = P - 2 * S;; m += RS) {
    if (one(std::integral_constant<int, 0>{}, m)) break;
    if constexpr (RS > 1) if (one(std::integral_constant<int, 1>{}, m)) break;
    if constexpr (RS > 2) if (one(std::integral_constant<int, 2>{}, m)) break;
    if constexpr (RS > 3) if (one(std::integral_constant<int, 3>{}, m)) break;
    if constexpr (RS > 4) if (one(std::integral_constant<int, 4>{}, m)) break;
    if constexpr (RS > 5) if (one(std::integral_constant<int, 5>{}, m)) break;
  }
}

// The tile of this workgroup.  The first `first` workgroups take the tiles with events, which run
// longest (a single such tile started late would end the launch alone), the others all tiles
// in XCD bands, leaving out those.
template <typename T, bool KAHAN, bool THERMAL, bool AXI, bool ISO, bool PAL, int S, int PF>
__device__ __forceinline__ void fused_tile(const StepArgs<T> &a, int64_t step, int64_t row,
                                           FusedLds<T, ISO, S> &L) {
  const int first = (a.fev.nslots + kNumXcd - 1) / kNumXcd * kNumXcd;
  const int b = blockIdx.x;
  if (b < first) {
    if (b >= a.fev.nslots) return;
    const int tile = __builtin_amdgcn_readfirstlane(a.fev.tiles[b]);
    fused_strip<T, KAHAN, THERMAL, AXI, ISO, PAL, true, S, 1>(a, tile, b, step, row, L);
  } else {
    const int tile = xcd_tile(b - first, gridDim.x - first, a.ntiles);
    if (tile < 0 || a.fev.slot[tile] >= 0) return;
    fused_strip<T, KAHAN, THERMAL, AXI, ISO, PAL, false, S, PF>(a, tile, -1, step, row, L);
  }
}

// LDS of a batch's workgroup, for any of its members' models.
template <typename T, int S>
union FusedBatchLds {
  FusedLds<T, true, S> iso;
  FusedLds<T, false, S> plain;
  __device__ FusedBatchLds() {}
};

// One tile of instance `a` in a batched launch, a tile with events (EV: word slot `slot`) or one
// without.  ANY: every lossless model; else acoustics with isotropic coefficients or axial
// symmetry (a sweep of those is the usual batch, and the kernel's registers are the largest
// member model's).  All members have material classes.
template <typename T, bool KAHAN, bool ANY, bool EV, int S, int PF>
__device__ __forceinline__ void fused_any(const StepArgs<T> &a, int tile, int slot, int64_t step,
                                          int64_t row, FusedBatchLds<T, S> &L) {
  const int f = __builtin_amdgcn_readfirstlane(a.flags);
  const bool iso = (f & kFlagIsoB) && (f & kFlagIsoK);
  if (!ANY || !(f & kFlagThermal)) {
    if (f & kFlagAxi)
      fused_strip<T, KAHAN, false, true, false, true, EV, S, PF>(a, tile, slot, step, row, L.plain);
    else if (!ANY || iso)
      fused_strip<T, KAHAN, false, false, true, true, EV, S, PF>(a, tile, slot, step, row, L.iso);
    else if constexpr (ANY)
      fused_strip<T, KAHAN, false, false, false, true, EV, S, PF>(a, tile, slot, step, row,
                                                                  L.plain);
  } else if constexpr (ANY) {
    if (f & kFlagAxi)
      fused_strip<T, KAHAN, true, true, false, true, EV, S, PF>(a, tile, slot, step, row, L.plain);
    else if (iso)
      fused_strip<T, KAHAN, true, false, true, true, EV, S, PF>(a, tile, slot, step, row, L.iso);
    else
      fused_strip<T, KAHAN, true, false, false, true, EV, S, PF>(a, tile, slot, step, row,
                                                                 L.plain);
  }
}

}  // namespace fds

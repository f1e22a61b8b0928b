// Fused step kernels for lossy acoustics (Acoustic2D / Acoustic3DAxi with absorption) on fields of
// few materials: S time steps per launch on one-wave strips, as fds_fused2d.h, plus the viscous
// operator on both velocities (fds_stream_lossy.h has the expressions and their order):
//   vx <- vx - (((Dbwd(Bx) p) - V vx) [+ (Mt vx) / r^2])      vy <- vy - ((Dbwd(By) p) - V vy)
//   V f at j = (((My f)[j-nx] + (cm f)[j-1]) + (c0 f)[j]) + (cp f)[j+1]) + (My f)[j+nx]
//
// V reads the old velocities of the rows above and below, so a stage that takes row r forms the
// velocities of row r - 1 and the pressure of row r - 2, and hands on row r - 2: two rows a
// stage instead of one.  Everything of V but the row below is summed when a row arrives and kept
// as one value, in the reference's order.  A strip of H rows takes H + 3S iterations and reads S
// rows above and 2S below; a stage makes one column wrong on the left and, as the new pressure
// needs the new velocity on its right and that the old one beyond, one more on the right in the
// last stage: S ghost columns on the left, S + 1 on the right.
//
// What bounds it: a stage keeps 15 values a column (a lossless one 6), so FP64 holds three
// stages at two waves per SIMD; the step is then bound by its instructions and their latency
// rather than by HBM, which bounds the one-step kernels.  Lossy 2000 x 1500 FP64, us a step: 50 on
// the register-path strips (one step per launch), here 26, 14, 11 and 11 at 1 to 4 stages; AXI,
// with a division a stage left, 26, 16, 16 and 18; FP32 14, 8.2, 7.1 and 6.6.
//
// Coefficients come from the material classes' table in LDS.  AXI's quotients by the radius are
// kept per stage and formed again only where a row brings another class.
#pragma once

#include "fds_fused2d.h"

namespace fds {

// LDS: the classes' coefficients (ISO: bx, kx, M, c0; else the table's eight) and the tile's
// boundary classes.
template <typename T, bool ISO, int S>
struct LossyFusedLds {
  static constexpr int NC = ISO ? 4 : kPalSlots;
  __attribute__((aligned(16))) T pal[kPalMax][NC];
  FusedTerm term[S][kFusedClasses];
  uint8_t next[kFusedClasses];
};

// What a stage keeps: of the row that arrived last (the centre) its state, its differences of B p,
// its My v and the part of V that needs no row below; of the row before the new velocities, the
// differences of K v and the old pressure.
template <typename T>
struct LfCarry {
  T p, cp, vx, cvx, vy, cvy, dbx, dby, bpy, ux, uy, sx, sy, term;
  T pp, cpp, kvd, kvy, nvx, ncvx, nvy, ncvy;
};

template <typename T>
struct LfCoef {
  T bx, by, kx, ky, mx, my, c0;
  T cm, cp;      // AXI: x factors of V at the left and right neighbour
  T mt;          // AXI
};

// One stage: takes row r in x, leaves row r - 2 of the next time level in x.  ka, wa, fa:
// coefficients, event words and flags of row r; kx, ky, wc, fc: of row r - 1.
template <typename T, bool KAHAN, bool AXI, bool ISO, bool EV>
__device__ __forceinline__ void fused_lossy_stage(LfCarry<T> &c, FuRow<T> &x, const LfCoef<T> &ka,
                                                  T kx, T ky, T rad, int s, uint32_t wa,
                                                  uint32_t fa, uint32_t wc, uint32_t fc, int r,
                                                  const FusedEvents &E) {
  FusedTerm ma[3], mc[3];
  if constexpr (EV) {
    fused_terms(E, s, wa, fa & 1u, ma);
    fused_terms(E, s, wc, fc & 6u, mc);
    if (fa & 1u) fused_bound<T, KAHAN, 0>(E, ma[0], s, wa, x.p, x.cp);
    if (fa & 8u)
      fused_record<T, KAHAN, 0, 1>(E, s, r, fa, x.p, x.cp, T(0), T(0), T(0), T(0));
  }
  // ---- row r
  const T bpx = ka.bx * x.p;
  const T bpy = ISO ? bpx : ka.by * x.p;
  const T left = wave_from_left(bpx);
  const T dbx = (-left) + bpx;
  const T dby = (-c.bpy) + bpy;
  T qlx, qrx, qly, qry, ux, uy;
  if constexpr (AXI) {
    qlx = wave_from_left(ka.cm * x.vx);
    qrx = wave_from_right(ka.cp * x.vx);
    qly = wave_from_left(ka.cm * x.vy);
    qry = wave_from_right(ka.cp * x.vy);
    ux = ka.my * x.vx;
    uy = ka.my * x.vy;
  } else {
    const T qx = ka.mx * x.vx, qy = ka.mx * x.vy;
    qlx = wave_from_left(qx);
    qrx = wave_from_right(qx);
    qly = wave_from_left(qy);
    qry = wave_from_right(qy);
    ux = ISO ? qx : ka.my * x.vx;
    uy = ISO ? qy : ka.my * x.vy;
  }
  // ---- row r - 1: its velocities, now that the row below is here
  T vx = c.vx, cvx = c.cvx;
  {
    const T y = c.sx + ux;
    T d = c.dbx - y;
    if (AXI) d = d + c.term;
    if (KAHAN) kahan_sub(vx, cvx, d); else vx = vx - d;
  }
  if constexpr (EV) {
    if (fc & 2u) fused_bound<T, KAHAN, 1>(E, mc[1], s, wc, vx, cvx);
  }
  const T kvx = AXI ? kx * (vx * rad) : kx * vx;
  const T right = wave_from_right(kvx);
  const T kvd = (-kvx) + right;
  T vy = c.vy, cvy = c.cvy;
  {
    const T y = c.sy + uy;
    const T d = c.dby - y;
    if (KAHAN) kahan_sub(vy, cvy, d); else vy = vy - d;
  }
  if constexpr (EV) {
    if (fc & 4u) fused_bound<T, KAHAN, 2>(E, mc[2], s, wc, vy, cvy);
    if (fc & kRowRecord & ~8u)
      fused_record<T, KAHAN, 1, 3>(E, s, r - 1, fc, T(0), T(0), vx, cvx, vy, cvy);
  }
  const T kvy = ky * vy;
  // ---- row r - 2: its pressure
  const T dy = (-c.kvy) + kvy;
  const T d = c.kvd + dy;
  T p = c.pp, cp = c.cpp;
  if (KAHAN) kahan_sub(p, cp, d); else p = p - d;
  const FuRow<T> out{p, cp, c.nvx, c.ncvx, c.nvy, c.ncvy};
  // ---- row r as the next iteration's centre: V without the row below
  T sx = T(0), sy = T(0);
  sx = sx + c.ux;
  sx = sx + qlx;
  { const T u = ka.c0 * x.vx; sx = sx + u; }
  sx = sx + qrx;
  sy = sy + c.uy;
  sy = sy + qly;
  { const T u = ka.c0 * x.vy; sy = sy + u; }
  sy = sy + qry;
  const T term = AXI ? (ka.mt * x.vx) / (rad * rad) : T(0);
  c = LfCarry<T>{x.p, x.cp, x.vx, x.cvx, x.vy, x.cvy, dbx, dby,  bpy, ux,  uy,
                 sx,  sy,   term, c.p,   c.cp, kvd,   kvy, vx,   cvx, vy,  cvy};
  x = out;
}

template <typename T, bool KAHAN, bool AXI, bool ISO, bool EV, int S, int PF>
__device__ __forceinline__ void fused_lossy_strip(const StepArgs<T> &a, int tile, int slot,
                                                  int64_t step, int64_t row,
                                                  LossyFusedLds<T, ISO, S> &L) {
  constexpr int RS = PF + 1, D = 2 * S;   // D: rows between a launch's first and last stage
  const int G = a.ghost, sx = a.sx, H = a.strip_h;
  const int t = threadIdx.x;
  const int ty = tile / a.tiles_x, tx = tile - ty * a.tiles_x;
  const int x0 = tx * sx - G, y0 = ty * H;
  const int nx = a.nx;
  const int rows = a.ny - y0 < H ? a.ny - y0 : H;
  const bool owned = t >= G && t < G + sx && x0 + t < nx;
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
  const BufRsrc ridx = buf_rsrc(a.pal_idx, a.n);
  if (t < a.npal) {
    const T *q = a.pal + t * kPalSlots;
    if constexpr (ISO) {
      L.pal[t][0] = q[0];
      L.pal[t][1] = q[1];
      L.pal[t][2] = q[4];
      L.pal[t][3] = (T(-2) * q[4]) + (T(-2) * q[4]);
    } else {
#pragma unroll
      for (int k = 0; k < kPalSlots; ++k) L.pal[t][k] = q[k];
    }
  }
  __syncthreads();
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
    uint32_t w, m;
  };
  Slot in[RS];
  // row ordinal o of the launch is row o - S of the strip
  const int last = rows + D - 1;
  auto load = [&](int o, Slot &d) __attribute__((always_inline)) {
    const int rho = o - S < last ? o - S : last;
    const int j = (y0 + rho) * nx + x0 + t;
    const uint32_t off = (uint32_t)j * (uint32_t)sizeof(T);
    d.x.p = buf_load<T>(in0, off);
    d.x.vx = buf_load<T>(in1, off);
    d.x.vy = buf_load<T>(in2, off);
    d.m = __builtin_amdgcn_raw_buffer_load_b8(ridx, j, 0, 0);
    if (KAHAN) {
      d.x.cp = buf_load<T>(cin0, off);
      d.x.cvx = buf_load<T>(cin1, off);
      d.x.cvy = buf_load<T>(cin2, off);
    } else {
      d.x.cp = d.x.cvx = d.x.cvy = T(0);
    }
    d.w = EV ? buf_load<uint32_t>(words, (uint32_t)((rho + a.ghost_rows + 1) * 64 + t) * 4u) : 0u;
  };
  static_for<PF>([&](auto Oc) __attribute__((always_inline)) {
    load(decltype(Oc)::value, in[decltype(Oc)::value]);
  });

  LfCarry<T> c[S] = {};
  struct Radial {        // AXI: quotients of the stage's rows, formed again at another class
    T kr, cm, cp;        // kx / rad of the centre row's class; x factors of V
  };
  Radial q[S] = {};
  T krc[S] = {};         // AXI: kx / rad of the centre row
  uint32_t mc[D] = {};   // of the row that arrived d iterations ago: material class,
  uint32_t wc[D] = {};   // event words, what the words hold
  uint32_t ac[D] = {};
  int busy = 0;
  auto iterate = [&](auto Wc, auto NSc, int i) __attribute__((always_inline)) -> FuRow<T> {
    constexpr int W = decltype(Wc)::value, NS = decltype(NSc)::value;
    load(i + PF, in[(W + PF) % RS]);
    static_for<D - 1, true>([&](auto Dc) __attribute__((always_inline)) {
      constexpr int d = decltype(Dc)::value + 1;
      mc[d] = mc[d - 1];
      wc[d] = wc[d - 1];
      ac[d] = ac[d - 1];
    });
    FuRow<T> x = in[W].x;
    mc[0] = in[W].m;
    if constexpr (EV) {
      wc[0] = in[W].w;
      ac[0] = fused_row_flags(wc[0]);
      if (ac[0]) busy = D;
    }
    auto stages = [&](auto EVc) __attribute__((always_inline)) {
      constexpr bool E1 = decltype(EVc)::value;
      static_for<NS>([&](auto Sc) __attribute__((always_inline)) {
        constexpr int s = decltype(Sc)::value;
        const T *m = L.pal[mc[2 * s]], *mp = L.pal[mc[2 * s + 1]];   // row r, row r - 1
        LfCoef<T> k;
        T kx, ky;
        k.bx = m[0];
        if constexpr (ISO) {
          k.by = m[0];
          k.mx = k.my = m[2];
          k.c0 = m[3];
          kx = mp[1];
          ky = kx;
        } else {
          k.by = m[2];
          k.mx = m[4];
          k.my = m[5];
          k.c0 = (T(-2) * m[4]) + (T(-2) * m[5]);
          kx = mp[1];
          ky = mp[3];
        }
        if constexpr (AXI) {
          krc[s] = q[s].kr;
          // (row r - 1's class is known to the quotients: they are the last row's)
          if (__any(mc[2 * s] != mc[2 * s + 1]) || i == 3 * s) {
            const T f = m[6] / rad;
            q[s].cm = m[4] + (-f) / T(2);
            q[s].cp = m[4] + f / T(2);
            q[s].kr = m[1] / rad;
          }
          k.cm = q[s].cm;
          k.cp = q[s].cp;
          k.mt = m[7];
          kx = krc[s];
        }
        fused_lossy_stage<T, KAHAN, AXI, ISO, E1>(c[s], x, k, kx, ky, rad, s, wc[2 * s],
                                                  ac[2 * s], wc[2 * s + 1], ac[2 * s + 1],
                                                  i - S - 2 * s, E);
      });
    };
    if constexpr (EV) {
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
  // tiles with events: the first 3S rows go through the loop too, all stages active
  constexpr int P = EV ? 0 : 3 * S;
  static_for<P>([&](auto Ic) __attribute__((always_inline)) {
    constexpr int i = decltype(Ic)::value;
    constexpr int NS = i / 3 + 1 < S ? i / 3 + 1 : S;
    (void)iterate(std::integral_constant<int, i % RS>{}, std::integral_constant<int, NS>{}, i);
  });
  auto put = [&](int m, const FuRow<T> &x) __attribute__((always_inline)) {
    const uint32_t o = (uint32_t)((y0 + m) * nx + x0 + t) * (uint32_t)sizeof(T);
    const uint32_t off = owned ? o : kBufOutside;
    buf_store<T>(out0, off, x.p);
    buf_store<T>(out1, off, x.vx);
    buf_store<T>(out2, off, x.vy);
    if (KAHAN) {
      buf_store<T>(cout0, off, x.cp);
      buf_store<T>(cout1, off, x.cvx);
      buf_store<T>(cout2, off, x.cvy);
    }
  };
  // one row; true: it was the strip's last
  auto one = [&](auto Jc, int m) __attribute__((always_inline)) -> bool {
    constexpr int J = decltype(Jc)::value;
    const FuRow<T> x = iterate(std::integral_constant<int, (P + J) % RS>{},
                               std::integral_constant<int, S>{}, 3 * S + m + J);
    if (!EV || m + J >= 0) put(m + J, x);
    return m + J + 1 >= rows;
  };
  static_assert(RS <= 4, "the row loop is written out for at most four slots");
  for (int m = P - 3 * S;; m += RS) {
    if (one(std::integral_constant<int, 0>{}, m)) break;
    if constexpr (RS > 1) if (one(std::integral_constant<int, 1>{}, m)) break;
    if constexpr (RS > 2) if (one(std::integral_constant<int, 2>{}, m)) break;
    if constexpr (RS > 3) if (one(std::integral_constant<int, 3>{}, m)) break;
  }
}

// The tile of this workgroup (tiles with events first, as fused_tile).
template <typename T, bool KAHAN, bool AXI, bool ISO, int S, int PF>
__device__ __forceinline__ void fused_lossy_tile(const StepArgs<T> &a, int64_t step, int64_t row,
                                                 LossyFusedLds<T, ISO, S> &L) {
  const int first = (a.fev.nslots + kNumXcd - 1) / kNumXcd * kNumXcd;
  const int b = blockIdx.x;
  if (b < first) {
    if (b >= a.fev.nslots) return;
    const int tile = __builtin_amdgcn_readfirstlane(a.fev.tiles[b]);
    fused_lossy_strip<T, KAHAN, AXI, ISO, true, S, 1>(a, tile, b, step, row, L);
  } else {
    const int tile = xcd_tile(b - first, gridDim.x - first, a.ntiles);
    if (tile < 0 || a.fev.slot[tile] >= 0) return;
    fused_lossy_strip<T, KAHAN, AXI, ISO, false, S, PF>(a, tile, -1, step, row, L);
  }
}

}  // namespace fds

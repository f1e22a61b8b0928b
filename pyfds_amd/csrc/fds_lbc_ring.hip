// Learned absorbing boundary, several steps per launch.
//
// The network touches only the outer frame of the grid, and a step carries its influence one cell
// further in.  So the S steps of a launch of the fused engine (fds_fused2d.h), run with the layer
// as it was before them, are right for every cell kLbcDepth + S - 1 or more cells from the rim,
// and this kernel, next on the stream, computes the frame outside that anew: stencil and network
// alternate in LDS on overlapping segments of the frame, and the owned part of each segment
// overwrites what the fused launch left there, recorded points included.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "fds_common.h"
#include "fds_lbc.h"
#include "fds_lbc_dev.h"

namespace fds {

namespace {

// Depth from the rim: 0-15 the layer, 16-23 the band the network reads.  A segment keeps depths
// 15 .. 23 + S: what lies outside 15 reaches nothing inside, and each step spoils one more row at
// the inner edge.  Along the frame, a step spoils one position at either end and the network four
// (its two convolutions' reach): 4 S + 1 in all are computed beyond the owned ones.  Corner
// segments own a square and both its networks, side segments kRingSeg positions: 112 with their
// halo at six steps, whole MFMA tiles.
constexpr int R = kLbcTaps / 2;
constexpr int kRingThreads = 768, kRingWaves = kRingThreads / 64;
constexpr int kRingCells = 3;                         // a thread's cells
constexpr int kRingCellsMax = 51 * 51;                // corner square at six steps
constexpr int kRingRows = 160;                        // output rows of a segment's networks
constexpr int kRingX = kRingRows + 8;                 // input and hidden rows
constexpr int SX = 3 * kLbcBand, SH = kLbcHidden + 4; // LDS row strides
constexpr int N1 = kLbcTaps * (kLbcCin / 16), N2 = kLbcTaps * (kLbcHidden / 16);  // products

// One cell of a thread.
struct __attribute__((aligned(16))) RingCell {
  int32_t at;                // flat index in the grid
  uint16_t lc, net;          // place in the segment (none: 0xffff); row of its network's output + 1
  uint16_t in[2];            // row * SX + band row of the networks' inputs, + 1 (0: not read)
  int32_t flags;             // 1: stored, 2: has a recorded point
};

// The weights in the order the waves' products take them, per side: layer 1 [2][N1][64], layer 2
// [3][N2][64], of layer 2 what a next step reads [N2][64] (columns 0-2: depth 15 of p, vx, vy).
constexpr int kRingPacked = (2 * N1 + 4 * N2) * 64;

__global__ __launch_bounds__(256) void k_ring_pack(const uint16_t *__restrict__ w1,
                                                   const uint16_t *__restrict__ w2, s4 *out) {
  const int i = blockIdx.x * 256 + threadIdx.x, s = blockIdx.y;
  if (i >= kRingPacked) return;
  const int l = i & 63, m = l & 15, g = l >> 4, r = i >> 6;
  const uint16_t *src;
  if (r < 2 * N1) {
    const int nt = r / N1, j = r % N1;
    src = w1 + ((size_t)(s * kLbcHidden + 16 * nt + m) * kLbcTaps + j / 3) * kLbcCin + 16 * (j % 3);
  } else {
    const int q = r - 2 * N1, nt = q / N2, j = q % N2;
    const int co = nt < 3 ? 16 * nt + m : (m < 3 ? 16 * m : 0) + kLbcDepth - 1;
    src = w2 + ((size_t)(s * kLbcCout + co) * kLbcTaps + j / 2) * kLbcHidden + 16 * (j % 2);
  }
  out[(size_t)s * kRingPacked + i] = ld4(src + 4 * g);
}

// Segment `blk`: cells [X0, X1) x [Y0, Y1), owned positions [lo, hi) of its networks' sides.
struct RingSegment {
  bool corner;
  int X0, X1, Y0, Y1, nets, side[2], lo[2], hi[2];
  int w, n, bar;             // row length, size of the square or strip, depths
  int h0[2];                 // hidden row r of network q: position h0[q] + r, output row r: R more
  int tiles, xrows;          // row tiles and input rows of a network

  __device__ __forceinline__ RingSegment(const LbcRing &A, int blk) {
    const int G = A.g, L = kLbcDepth, h = A.halo, C = L + h, D = L + kLbcBand + A.depth;
    corner = blk < 4;
    if (corner) {
      const bool right = blk & 1, bottom = blk & 2;
      X0 = right ? G - C - h : L - 1;
      X1 = right ? G - L + 1 : C + h;
      Y0 = bottom ? G - C - h : L - 1;
      Y1 = bottom ? G - L + 1 : C + h;
      side[0] = bottom ? 1 : 0;
      side[1] = right ? 3 : 2;
      lo[0] = right ? G - C : 0;
      hi[0] = right ? G : C;
      lo[1] = bottom ? G - C : L;
      hi[1] = bottom ? G - L : C;
      nets = 2;
    } else {
      const int q = blk - 4, s = q / A.segs;
      const int o = C + (q - s * A.segs) * kRingSeg, e = min(o + kRingSeg, G - C);
      const int d0 = s == 0 || s == 2 ? L - 1 : G - D, d1 = s == 0 || s == 2 ? D : G - L + 1;
      X0 = s < 2 ? o - h : d0;
      X1 = s < 2 ? e + h : d1;
      Y0 = s < 2 ? d0 : o - h;
      Y1 = s < 2 ? d1 : e + h;
      side[0] = side[1] = s;
      lo[0] = lo[1] = o;
      hi[0] = hi[1] = e;
      nets = 1;
    }
    w = X1 - X0;
    n = w * (Y1 - Y0);
    bar = D - L + 1;
    // corner networks see the rim of the frame (position -R on)
    h0[0] = side[0] < 2 ? X0 : Y0;
    h0[1] = side[1] < 2 ? X0 : Y0;
    if (corner && X0 == L - 1) h0[0] = -R;
    if (corner && Y0 == L - 1) h0[1] = -R;
    const int span = corner ? C + h + 2 * R : hi[0] - lo[0] + 2 * h;      // hidden rows
    tiles = (span + 15) / 16;
    xrows = 16 * tiles + 2 * R;
  }
};

// The cells of every segment's threads ([segment][kRingCells][kRingThreads]): a corner's are the
// two bars of depths below D.  (Formed by each launch they took a quarter of its time.)
__global__ __launch_bounds__(kRingThreads) void k_ring_cells(LbcRing A, RingCell *cells) {
  const RingSegment S(A, blockIdx.x);
  const int G = A.g, L = kLbcDepth, C = L + A.halo, c = threadIdx.x + kRingThreads * blockIdx.y;
  const int count = S.corner ? S.w * S.bar + (S.w - S.bar) * S.bar : S.n;
  RingCell r{0, 0xffff, 0, {0, 0}, 0};
  if (c < count) {
    int ly = c / S.w, lx = c - ly * S.w;
    if (S.corner) {
      if (c < S.w * S.bar) {
        if (S.side[0] == 1) ly += S.w - S.bar;
      } else {
        const int q = c - S.w * S.bar;
        ly = q / S.bar;
        lx = q - ly * S.bar + (S.side[1] == 3 ? S.w - S.bar : 0);
        if (S.side[0] == 0) ly += S.bar;
      }
    }
    const int x = S.X0 + lx, y = S.Y0 + ly;
    r.at = y * G + x;
    r.lc = (uint16_t)(ly * S.w + lx);
    bool band = false;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if (q >= S.nets) continue;
      const int s = S.side[q], a = s < 2 ? x : y;
      const int d = s == 0 ? y : s == 1 ? G - 1 - y : s == 2 ? x : G - 1 - x;
      if (a < L || a >= G - L) continue;
      if (d >= L && d < L + kLbcBand) {
        const int row = a - S.h0[q] + R;
        if (row >= 0 && row < S.xrows) r.in[q] = (uint16_t)((q * S.xrows + row) * SX + d - L + 1);
        band = true;
      }
      const int row = a - S.h0[q] - R;
      if (d == L - 1 && row >= 0 && row < 16 * S.tiles)
        r.net = (uint16_t)(q * 16 * S.tiles + row + 1);
    }
    const bool own = S.corner ? (S.side[1] == 2 ? x < C : x >= G - C) &&
                                    (S.side[0] == 0 ? y < C : y >= G - C)
                     : S.side[0] < 2 ? x >= S.lo[0] && x < S.hi[0]
                                     : y >= S.lo[0] && y < S.hi[0];
    if (band && own) {
      r.flags = 1;
      for (int q = 0; q < A.nrec; ++q)
        if (A.rec[q].cell == r.at) r.flags = 3;
    }
  }
  cells[((size_t)blockIdx.x * kRingCells + blockIdx.y) * kRingThreads + threadIdx.x] = r;
}

// What bounds it: the issue rate and latency of one CU.  A step is four phases with a barrier
// after each (velocities; pressure and the network's input; hidden layer; layer), and of the 68
// segments of a 1056^2 grid the corners take longest.  12 waves share a phase, each keeping its
// weights in registers; a step's row tiles are those that still reach an owned cell.
__global__ __launch_bounds__(kRingThreads) void k_lbc_ring(LbcRing A) {
  __shared__ float bp[kRingCellsMax], kvx[kRingCellsMax], kvy[kRingCellsMax];
  __shared__ __attribute__((aligned(16))) uint16_t xin[2][kRingX * SX];
  __shared__ __attribute__((aligned(16))) uint16_t hid[kRingX * SH];
  __shared__ float net[3][kRingRows];     // the network's p, vx, vy at depth 15
  __shared__ float b15[kRingRows];        // its cells' coefficient ...
  __shared__ int cell15[kRingRows];       // ... and place in the segment (-1: outside)
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63, m = l & 15, g = l >> 4;
  RingCell cell[kRingCells];
#pragma unroll
  for (int i = 0; i < kRingCells; ++i)
    cell[i] = static_cast<const RingCell *>(
        A.cells)[((size_t)blockIdx.x * kRingCells + i) * kRingThreads + tid];
  const RingSegment S(A, blockIdx.x);
  const int G = A.g, L = kLbcDepth, w = S.w, n = S.n, tiles = S.tiles, xrows = S.xrows;

  // weights: a wave's column of channels of layer 1 (n1); of layer 2 a column too (n2, a
  // component) after the last step, before it only what the next step reads, a row tile a wave
  // (q3)
  const int n1 = wave & 1, q1 = S.corner ? (wave >> 1) & 1 : 0, sub1 = wave >> (S.corner ? 2 : 1),
            step1 = S.corner ? kRingWaves / 4 : kRingWaves / 2;
  const int n2 = wave % 3, q2 = S.corner ? wave / 3 & 1 : 0, sub2 = wave / (S.corner ? 6 : 3),
            step2 = S.corner ? kRingWaves / 6 : kRingWaves / 3;
  const int q3 = wave >= tiles ? 1 : 0;
  const int s2 = q2 ? S.side[1] : S.side[0];
  s4 w1[N1], w2[N2];
  const s4 *packed = static_cast<const s4 *>(A.packed) + l;
  {
    const s4 *p1 = packed + (q1 ? S.side[1] : S.side[0]) * kRingPacked + n1 * N1 * 64;
    const s4 *p2 = packed + (q3 ? S.side[1] : S.side[0]) * kRingPacked + (2 * N1 + 3 * N2) * 64;
#pragma unroll
    for (int j = 0; j < N1; ++j) w1[j] = p1[64 * j];
#pragma unroll
    for (int j = 0; j < N2; ++j) w2[j] = p2[64 * j];
  }
  for (int i = tid; i < 2 * kRingX * SX / 2; i += kRingThreads)
    reinterpret_cast<uint32_t *>(&xin[0][0])[i] = 0u;
  for (int i = tid; i < kRingRows; i += kRingThreads) cell15[i] = -1;
  if (S.corner)          // (its inside)
    for (int i = tid; i < n; i += kRingThreads) bp[i] = kvx[i] = kvy[i] = 0.f;
  for (int i = tid; i < kRingX * SH / 2; i += kRingThreads)
    reinterpret_cast<uint32_t *>(hid)[i] = 0u;

  float p[kRingCells], vx[kRingCells], vy[kRingCells], b[kRingCells], k[kRingCells];
#pragma unroll
  for (int i = 0; i < kRingCells; ++i) {
    const int at = cell[i].at;
    p[i] = A.in[0][at];
    vx[i] = A.in[1][at];
    vy[i] = A.in[2][at];
    b[i] = A.b[at];
    k[i] = A.k[at];
  }
  __syncthreads();
  const float cs0 = A.cs[0], cs1 = A.cs[1], cs2 = A.cs[2];
  auto inputs = [&](uint16_t *x, int i) __attribute__((always_inline)) {
    if (cell[i].in[0] == 0 && cell[i].in[1] == 0) return;
    const uint16_t u0 = f2bf(p[i] * cs0), u1 = f2bf(vx[i] * cs1), u2 = f2bf(vy[i] * cs2);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if (cell[i].in[q] == 0) continue;
      uint16_t *d = x + cell[i].in[q] - 1;
      d[0] = u0;
      d[kLbcBand] = u1;
      d[2 * kLbcBand] = u2;
    }
  };
#pragma unroll
  for (int i = 0; i < kRingCells; ++i) {
    const int c = cell[i].lc;
    if (c == 0xffff) continue;
    bp[c] = b[i] * p[i];
    inputs(xin[1], i);
    if (cell[i].net) {
      b15[cell[i].net - 1] = b[i];
      cell15[cell[i].net - 1] = c;
    }
  }
  __syncthreads();

  for (int st = 0; st < A.stages; ++st) {
    // (taken apart anew in each step: the parts in registers of their own are too many)
#pragma unroll
    for (int i = 0; i < kRingCells; ++i) {
      uint32_t u[2];
      __builtin_memcpy(u, &cell[i].lc, 8);
      __asm__ volatile("" : "+v"(u[0]), "+v"(u[1]));
      __builtin_memcpy(&cell[i].lc, u, 8);
    }
    // velocities (a missing neighbour's zero spoils only what the halo gives up)
#pragma unroll
    for (int i = 0; i < kRingCells; ++i) {
      const int c = cell[i].lc;
      if (c == 0xffff) continue;
      if (st > 0 && cell[i].net) {
        p[i] = net[0][cell[i].net - 1];
        vx[i] = net[1][cell[i].net - 1];
        vy[i] = net[2][cell[i].net - 1];
      }
      const float own = b[i] * p[i];
      const float left = c > 0 ? bp[c - 1] : 0.f, above = c >= w ? bp[c - w] : 0.f;
      vx[i] = vx[i] - ((-left) + own);
      vy[i] = vy[i] - ((-above) + own);
      kvx[c] = k[i] * vx[i];
      kvy[c] = k[i] * vy[i];
      if (cell[i].flags & 2) {
        const int64_t row = A.dyn[1] + A.row + st;
        for (int q = 0; q < A.nrec; ++q) {
          const LbcRec rec = A.rec[q];
          if (rec.cell == cell[i].at)
            A.rows[rec.comp][row * A.m[rec.comp] + rec.id] =
                (double)(rec.comp == 0 ? p[i] : rec.comp == 1 ? vx[i] : vy[i]);
        }
      }
    }
    __syncthreads();
    // pressure; what the network reads
    uint16_t *cur = xin[st & 1];
    const uint16_t *prev = xin[(st & 1) ^ 1];
#pragma unroll
    for (int i = 0; i < kRingCells; ++i) {
      const int c = cell[i].lc;
      if (c == 0xffff) continue;
      const float right = c + 1 < n ? kvx[c + 1] : 0.f, below = c + w < n ? kvy[c + w] : 0.f;
      const float dx = (-(k[i] * vx[i])) + right, dy = (-(k[i] * vy[i])) + below;
      p[i] = p[i] - (dx + dy);
      bp[c] = b[i] * p[i];
      inputs(cur, i);
    }
    __syncthreads();
    // hidden layer: the rows whose outputs reach an owned cell in the steps left
    const bool last = st + 1 == A.stages;
    const int reach = 4 * (A.stages - 1 - st) + 1;
    const int r0 = (q1 ? S.lo[1] - S.h0[1] : S.lo[0] - S.h0[0]) - reach - R,
              r1 = (q1 ? S.hi[1] - S.h0[1] : S.hi[0] - S.h0[0]) + reach + R;
    const uint16_t *xa = cur + 4 * g, *xb = g < 2 ? cur + 16 + 4 * g : prev + 4 * g - 8,
                   *xc = prev + 8 + 4 * g;
    const int t1 = min((r1 + 15) >> 4, tiles);
#pragma unroll 1
    for (int t = (max(r0, 0) >> 4) + sub1; t < t1; t += step1) {
      f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < N1; ++j) {
        const int row = q1 * xrows + 16 * t + m + j / 3;
        acc = mfma(ld4((j % 3 == 0 ? xa : j % 3 == 1 ? xb : xc) + row * SX), w1[j], acc);
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = 16 * t + 4 * g + v, a = (q1 ? S.h0[1] : S.h0[0]) + r;
        hid[(q1 * xrows + r) * SH + 16 * n1 + m] = a >= 0 && a < G ? f2bf(acc[v]) : (uint16_t)0;
      }
    }
    if (last) {          // the whole layer's weights, for after the barrier
      const s4 *p2 = packed + s2 * kRingPacked + (2 * N1 + n2 * N2) * 64;
#pragma unroll
      for (int j = 0; j < N2; ++j) w2[j] = p2[64 * j];
    }
    __syncthreads();
    const auto layer2 = [&](int row) __attribute__((always_inline)) {
      f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < N2; ++j)
        acc = mfma(ld4(hid + (row + m + j / 2) * SH + 16 * (j % 2) + 4 * g), w2[j], acc);
      return acc;
    };
    if (!last) {
      const int t = wave - q3 * tiles, o0 = (q3 ? S.h0[1] : S.h0[0]) + R + 16 * t;
      if (wave < S.nets * tiles && o0 + 16 > (q3 ? S.lo[1] : S.lo[0]) - reach &&
          o0 < (q3 ? S.hi[1] : S.hi[0]) + reach) {
        const f4 acc = layer2(q3 * xrows + 16 * t);
        if (m < 3) {
          const float cs = m == 0 ? cs0 : m == 1 ? cs1 : cs2;
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int row = 16 * wave + 4 * g + v;
            const float x = acc[v] / cs;
            net[m][row] = x;
            if (m == 0 && cell15[row] >= 0) bp[cell15[row]] = b15[row] * x;
          }
        }
      }
      __syncthreads();
      continue;
    }
    // after the last step the whole layer
    const float cs = n2 == 0 ? cs0 : n2 == 1 ? cs1 : cs2;
    float *dst = n2 == 0 ? A.out[0] : n2 == 1 ? A.out[1] : A.out[2];
    const int a0 = (q2 ? S.h0[1] : S.h0[0]) + R;
    const int lo = q2 ? S.lo[1] : S.lo[0], hi = q2 ? S.hi[1] : S.hi[0];
#pragma unroll 1
    for (int t = sub2; t < tiles; t += step2) {
      if (a0 + 16 * t >= hi || a0 + 16 * t + 16 <= lo) continue;
      const f4 acc = layer2(q2 * xrows + 16 * t);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int a = a0 + 16 * t + 4 * g + v;
        if (a >= lo && a < hi) dst[lbc_cell(s2, m, a, G)] = acc[v] / cs;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < kRingCells; ++i)
    if (cell[i].flags & 1) {
      A.out[0][cell[i].at] = p[i];
      A.out[1][cell[i].at] = vx[i];
      A.out[2][cell[i].at] = vy[i];
    }
}

void ring_layout(LbcRing &a) {
  a.halo = 4 * a.depth + 1;
  a.segs = (a.g - 2 * (kLbcDepth + a.halo) + kRingSeg - 1) / kRingSeg;
}

}  // namespace

bool lbc_ring_fits(int64_t g, int stages) {
  const int halo = 4 * stages + 1, side = 2 * halo + 1;
  const int bar = kLbcBand + 1 + stages;
  return stages >= 2 && side * side <= kRingCellsMax &&
         std::max(side * bar + (side - bar) * bar, (kRingSeg + 2 * halo) * bar) <=
             kRingCells * kRingThreads &&
         g >= 2 * (kLbcDepth + halo);
}

size_t lbc_ring_cells_bytes(LbcRing a) {
  ring_layout(a);
  return (size_t)(4 + 4 * a.segs) * kRingCells * kRingThreads * sizeof(RingCell);
}

size_t lbc_ring_packed_bytes() { return (size_t)4 * kRingPacked * sizeof(s4); }

void launch_ring_cells(LbcRing a, void *cells, hipStream_t s) {
  ring_layout(a);
  hipLaunchKernelGGL(k_ring_cells, dim3(4 + 4 * a.segs, kRingCells), dim3(kRingThreads), 0, s, a,
                     static_cast<RingCell *>(cells));
}

void launch_ring_pack(const uint16_t *w1, const uint16_t *w2, void *packed, hipStream_t s) {
  hipLaunchKernelGGL(k_ring_pack, dim3((kRingPacked + 255) / 256, 4), dim3(256), 0, s, w1, w2,
                     static_cast<s4 *>(packed));
}

void launch_lbc_ring(LbcRing a, hipStream_t s) {
  ring_layout(a);
  hipLaunchKernelGGL(k_lbc_ring, dim3(4 + 4 * a.segs), dim3(kRingThreads), 0, s, a);
}

}  // namespace fds

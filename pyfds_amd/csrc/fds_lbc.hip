// Learned absorbing boundary: BF16 MFMA (v_mfma_f32_16x16x16_bf16) kernels with FP32
// accumulation for training (1D convolution forward, backward-data, backward-weight, MSE loss,
// Adam) and the fused per-step inference kernel that writes the boundary layer.
//
// MFMA 16x16x16 lane layout used throughout (l = lane, m = l % 16, g = l / 16):
//   A (16 x 16, rows x k):  lane holds A[m][4g .. 4g+3]
//   B (16 x 16, k x cols):  lane holds B[4g .. 4g+3][m]
//   D (16 x 16, f32):       lane holds D[4g + v][m], v = 0..3
// A 1D convolution y[p, co] = sum_k sum_ci w[co, k, ci] x[p + k - K/2, ci] (zero outside the
// strip) is a GEMM over (k, ci): rows are positions, and for a fixed tap the 16 ci of a k-chunk
// are contiguous in the [position][channel] layout, so each lane loads 4 bf16 (8 bytes).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/pyfds_amd.h"
#include "fds_lbc.h"
#include "fds_lbc_dev.h"

namespace fds {
namespace {

__device__ __forceinline__ s4 ld4_strided(const uint16_t *p, int stride, int n_valid) {
  s4 r;
  r[0] = n_valid > 0 ? (short)p[0] : (short)0;
  r[1] = n_valid > 1 ? (short)p[stride] : (short)0;
  r[2] = n_valid > 2 ? (short)p[2 * stride] : (short)0;
  r[3] = n_valid > 3 ? (short)p[3 * stride] : (short)0;
  return r;
}

// ---------------------------------------------------------------- training kernels
// x [B][P][Ci] bf16, w [S][Co][K][Ci] bf16, side [B] -> y [B][P][Co] f32 (+ bf16 copy)
__global__ __launch_bounds__(64) void k_conv_fwd(const uint16_t *__restrict__ x,
                                                 const uint16_t *__restrict__ w,
                                                 const int32_t *__restrict__ side,
                                                 float *__restrict__ y, uint16_t *__restrict__ yb,
                                                 int P, int Ci, int Co, int K) {
  const int p0 = blockIdx.x * 16, co0 = blockIdx.y * 16, b = blockIdx.z;
  const int l = threadIdx.x, m = l & 15, g = l >> 4, R = K / 2;
  const uint16_t *xb = x + (size_t)b * P * Ci;
  const uint16_t *ws = w + (size_t)side[b] * Co * K * Ci;
  f4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < K; ++k) {
    const int pa = p0 + m + k - R;
    const bool in = pa >= 0 && pa < P;
    for (int c0 = 0; c0 < Ci; c0 += 16) {
      const s4 av = in ? ld4(xb + (size_t)pa * Ci + c0 + 4 * g) : s4{0, 0, 0, 0};
      const s4 bv = ld4(ws + ((size_t)(co0 + m) * K + k) * Ci + c0 + 4 * g);
      acc = mfma(av, bv, acc);
    }
  }
  for (int v = 0; v < 4; ++v) {
    const int p = p0 + 4 * g + v;
    if (p < P) {
      const size_t o = ((size_t)b * P + p) * Co + co0 + m;
      y[o] = acc[v];
      if (yb) yb[o] = f2bf(acc[v]);
    }
  }
}

// dy [B][P][Co] bf16, wt [S][Ci][K][Co] bf16 -> dx [B][P][Ci] f32 (+ bf16 copy)
__global__ __launch_bounds__(64) void k_conv_bwd_data(const uint16_t *__restrict__ dy,
                                                      const uint16_t *__restrict__ wt,
                                                      const int32_t *__restrict__ side,
                                                      float *__restrict__ dx,
                                                      uint16_t *__restrict__ dxb, int P, int Ci,
                                                      int Co, int K) {
  const int q0 = blockIdx.x * 16, ci0 = blockIdx.y * 16, b = blockIdx.z;
  const int l = threadIdx.x, m = l & 15, g = l >> 4, R = K / 2;
  const uint16_t *dyb = dy + (size_t)b * P * Co;
  const uint16_t *ws = wt + (size_t)side[b] * Ci * K * Co;
  f4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < K; ++k) {
    const int pa = q0 + m - k + R;
    const bool in = pa >= 0 && pa < P;
    for (int c0 = 0; c0 < Co; c0 += 16) {
      const s4 av = in ? ld4(dyb + (size_t)pa * Co + c0 + 4 * g) : s4{0, 0, 0, 0};
      const s4 bv = ld4(ws + ((size_t)(ci0 + m) * K + k) * Co + c0 + 4 * g);
      acc = mfma(av, bv, acc);
    }
  }
  for (int v = 0; v < 4; ++v) {
    const int q = q0 + 4 * g + v;
    if (q < P) {
      const size_t o = ((size_t)b * P + q) * Ci + ci0 + m;
      dx[o] = acc[v];
      if (dxb) dxb[o] = f2bf(acc[v]);
    }
  }
}

// dw partial per sample: part[b][co][k][ci] = sum_p dy[b, p, co] * x[b, p + k - R, ci]
__global__ __launch_bounds__(64) void k_conv_bwd_weight(const uint16_t *__restrict__ dy,
                                                        const uint16_t *__restrict__ x,
                                                        float *__restrict__ part, int P, int Ci,
                                                        int Co, int K) {
  const int k = blockIdx.x, b = blockIdx.z;
  const int nci = Ci / 16;
  const int co0 = (blockIdx.y / nci) * 16, ci0 = (blockIdx.y % nci) * 16;
  const int l = threadIdx.x, m = l & 15, g = l >> 4, R = K / 2;
  const uint16_t *dyb = dy + (size_t)b * P * Co;
  const uint16_t *xb = x + (size_t)b * P * Ci;
  f4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int p0 = 0; p0 < P; p0 += 16) {
    // A[m][kk] = dy[p0 + kk, co0 + m]; B[kk][n] = x[p0 + kk + k - R, ci0 + n]
    const int pa = p0 + 4 * g;
    const s4 av = ld4_strided(dyb + (size_t)pa * Co + co0 + m, Co, P - pa);
    s4 bv;
    for (int v = 0; v < 4; ++v) {
      const int px = pa + v + k - R;
      bv[v] = (pa + v < P && px >= 0 && px < P) ? (short)xb[(size_t)px * Ci + ci0 + m] : (short)0;
    }
    acc = mfma(av, bv, acc);
  }
  float *pb = part + (size_t)b * Co * K * Ci;
  for (int v = 0; v < 4; ++v)
    pb[((size_t)(co0 + 4 * g + v) * K + k) * Ci + ci0 + m] = acc[v];
}

// dw[s][i] = sum over samples b with side[b] == s of part[b][i]
__global__ void k_reduce_weight(const float *__restrict__ part, const int32_t *__restrict__ side,
                                float *__restrict__ dw, int B, int S, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int s = blockIdx.y;
  if (i >= n) return;
  float acc = 0.f;
  for (int b = 0; b < B; ++b)
    if (side[b] == s) acc += part[(size_t)b * n + i];
  dw[(size_t)s * n + i] = acc;
}

// Weighted MSE over positions [lo[b], hi[b]) of each sample: loss partial sums per block and
// dy = 2 w_c (y - t) * norm as bf16.
__global__ __launch_bounds__(256) void k_mse(const float *__restrict__ y,
                                             const float *__restrict__ t,
                                             const int32_t *__restrict__ lo,
                                             const int32_t *__restrict__ hi,
                                             const float *__restrict__ wch,
                                             uint16_t *__restrict__ dyb,
                                             float *__restrict__ loss_part, int B, int P, int C,
                                             float norm) {
  __shared__ float red[256];
  const size_t total = (size_t)B * P * C;
  float acc = 0.f;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
    const int c = (int)(i % C);
    const size_t bp = i / C;
    const int p = (int)(bp % P), b = (int)(bp / P);
    float d = 0.f;
    if (p >= lo[b] && p < hi[b]) {
      const float e = y[i] - t[i];
      acc += wch[c] * e * e;
      d = 2.f * wch[c] * e * norm;
    }
    dyb[i] = f2bf(d);
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) loss_part[blockIdx.x] = red[0] * norm;
}

__global__ void k_adam(float *__restrict__ w, float *__restrict__ m1, float *__restrict__ m2,
                       const float *__restrict__ gr, int n, float lr, float b1, float b2,
                       float eps, float c1, float c2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = gr[i];
  const float a = b1 * m1[i] + (1.f - b1) * gi;
  const float v = b2 * m2[i] + (1.f - b2) * gi * gi;
  m1[i] = a;
  m2[i] = v;
  w[i] -= lr * (a / c1) / (sqrtf(v / c2) + eps);
}

// master f32 [S][Co][K][Ci] -> bf16 same layout and bf16 transposed [S][Ci][K][Co]
__global__ void k_pack(const float *__restrict__ w, uint16_t *__restrict__ wb,
                       uint16_t *__restrict__ wtb, int S, int Co, int K, int Ci) {
  const int n = S * Co * K * Ci;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int ci = i % Ci, k = (i / Ci) % K, co = (i / (Ci * K)) % Co, s = i / (Ci * K * Co);
  const uint16_t h = f2bf(w[i]);
  wb[i] = h;
  if (wtb) wtb[(((size_t)s * Ci + ci) * K + k) * Co + co] = h;
}

// frames [F][3][4][D][G] f32 (F = runs * T steps).  Sample b = (run, step, side):
//   x[b][a][h*24 + c*8 + j] = frames[run*T + step - h][c][side][L + j][a] * cs[c] * scale[b]
//                             (zero for a outside [L, G-L))
//   t[b][a][c*16 + d]       = frames[run*T + step][c][side][d][a] * cs[c] * scale[b]
__global__ __launch_bounds__(256) void k_gather(const float *__restrict__ frames,
                                                const int32_t *__restrict__ run,
                                                const int32_t *__restrict__ step,
                                                const int32_t *__restrict__ side,
                                                const float *__restrict__ scale,
                                                uint16_t *__restrict__ x, float *__restrict__ t,
                                                int T, int D, int G, int L, float cs0, float cs1,
                                                float cs2) {
  const int b = blockIdx.y;
  const int a = blockIdx.x * 256 + threadIdx.x;
  if (a >= G) return;
  const float cs[3] = {cs0, cs1, cs2};
  const int s = side[b];
  const size_t f0 = (size_t)run[b] * T + step[b];
  const float sc = scale[b];
  const bool band = a >= L && a < G - L;
  uint16_t *xo = x + ((size_t)b * G + a) * kLbcCin;
  for (int h = 0; h < 2; ++h)
    for (int c = 0; c < 3; ++c)
      for (int j = 0; j < kLbcBand; ++j) {
        float v = 0.f;
        if (band)
          v = frames[((((f0 - h) * 3 + c) * 4 + s) * D + L + j) * G + a] * cs[c] * sc;
        xo[h * 24 + c * 8 + j] = f2bf(v);
      }
  float *to = t + ((size_t)b * G + a) * kLbcCout;
  for (int c = 0; c < 3; ++c)
    for (int d = 0; d < kLbcDepth; ++d)
      to[c * kLbcDepth + d] = frames[(((f0 * 3 + c) * 4 + s) * D + d) * G + a] * cs[c] * sc;
}

// ---------------------------------------------------------------- fused training iteration
// Three launches per iteration.  One kernel per operation, enqueued one by one with six sample
// lists copied in between, was bound by the host and by those copies: 20 iterations of 32 samples
// on 1056 positions 6.9 ms, 1.0 ms so.
//   k_train_grads    gather, both convolutions, loss and the gradient at the hidden layer of a
//                    segment of a sample, in LDS;
//   k_train_weights  the weight gradients of one sample, one 16 x 16 tile for all taps a wave;
//   k_train_update   sum over the samples, Adam, and the bf16 copies of the weights.
// Sums run in the order of the separate kernels (k_conv_fwd, ...): the same bits.
// Between the first two, x, the hidden layer and both gradients stand channel-major
// ([B][C][pitch] bf16, position p at kPad + p, zeros around), so that the reduction over the
// positions reads whole vectors.
constexpr int kPad = 4;
constexpr int kTrainSeg = 64;     // positions a workgroup of k_train_grads hands on
constexpr int kChunk = 8;         // 16-position products of k_train_weights in flight

struct TrainStep {
  const float *frames, *scale, *wch;
  const int32_t *run, *step, *side;
  const uint16_t *w1b, *w2b, *w2t;
  uint16_t *x, *h, *dy, *dh;
  float *part1, *part2, *loss;
  int T, D, G, L, pitch;
  float cs[3], norm;
};

__host__ __device__ inline int train_pitch(int G) { return (G + 127) / 128 * 128 + 2 * kPad; }

// Zeros around the rows of the four channel-major arrays (k_train_grads writes the rest).
__global__ __launch_bounds__(64) void k_train_pads(uint16_t *rows, int G, int pitch) {
  uint16_t *r = rows + (size_t)blockIdx.x * pitch;
  if (threadIdx.x < kPad) r[threadIdx.x] = 0;
  for (int i = kPad + G + threadIdx.x; i < pitch; i += 64) r[i] = 0;
}

// Bound by latency: a chain of loads, three products and three barriers; 64 positions a
// workgroup give 544 of them for 32 samples of 1056 positions (two a CU), and the 12 rows
// computed twice on the way cost a fifth.  The weights stay in registers: a wave keeps one
// column of 16 output channels for all its rows.  24.7 us at that size (26.9 with the input
// cells dealt out by element, whose index arithmetic every lane did).
__global__ __launch_bounds__(256) void k_train_grads(TrainStep A) {
  constexpr int R = kLbcTaps / 2;
  constexpr int NT = 5;                            // row tiles of the hidden layer and of dy
  constexpr int NR = 16 * NT, NXR = NR + 2 * R;    // rows; input rows the tiles read
  constexpr int SX = kLbcCin + 4, SH = kLbcHidden + 4, SY = kLbcCout + 4;  // (LDS banks)
  static_assert(kTrainSeg + 8 * R <= NR, "hidden rows cover the segment and its reach");
  // row 0 of the hidden layer and of dy is position a0 - 2R, of the input a0 - 3R; hid has R
  // rows more on both sides, which only rows of dy that nothing reads look at
  __shared__ __attribute__((aligned(16))) uint16_t xin[NXR * SX];
  __shared__ __attribute__((aligned(16))) uint16_t hid[(NR + 2 * R) * SH];
  __shared__ __attribute__((aligned(16))) uint16_t dyl[NR * SY];
  __shared__ float red[4];
  const int G = A.G, L = A.L, b = blockIdx.y, a0 = blockIdx.x * kTrainSeg;
  const int tid = threadIdx.x, wave = tid >> 6, l = tid & 63, m = l & 15, g = l >> 4;
  const int s = A.side[b];
  const size_t f0 = (size_t)A.run[b] * A.T + A.step[b];
  const float sc = A.scale[b];
  constexpr int N1 = kLbcTaps * (kLbcCin / 16), N2 = kLbcTaps * (kLbcHidden / 16),
                NB = kLbcTaps * (kLbcCout / 16);

  // inputs, targets and the weights of both layers, all in flight together.  A wave takes 12
  // input channels: of each the first 64 rows, then the other 20 rows of three at a time.
  constexpr int WC = kLbcCin / 4, NL = NXR - 64, NP = 64 / NL;
  static_assert(NL > 0 && WC % NP == 0, "the rows past a wave's lanes go by whole groups");
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  const auto source = [&](int ci) {
    const int h = ci / 24, c = (ci % 24) / kLbcBand, j = ci % kLbcBand;
    return A.frames + ((((f0 - h) * 3 + c) * 4 + s) * A.D + L + j) * G;
  };
  const int al = a0 - 3 * R + l, row2 = 64 + l % NL, ah = a0 - 3 * R + row2, q2 = l / NL;
  const bool in1 = al >= L && al < G - L, in2 = q2 < NP && ah >= L && ah < G - L;
  float r1[WC], r2[WC / NP];
#pragma unroll
  for (int i = 0; i < WC; ++i) r1[i] = in1 ? source(wv * WC + i)[al] : 0.f;
#pragma unroll
  for (int i = 0; i < WC / NP; ++i) r2[i] = in2 ? source(wv * WC + NP * i + q2)[ah] : 0.f;
  // layer 2: waves 0-2 take a column of channels each (a component), rows of tiles 0-3; wave 3
  // the last tile of all three
  float tg[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int nt = wave < 3 ? wave : i, mt = wave < 3 ? i : NT - 1;
    const int a = a0 - 2 * R + 16 * mt + 4 * g;
    const bool job = wave < 3 || i < 3;
    const float *t = A.frames + (((f0 * 3 + nt) * 4 + s) * A.D + m) * G + a;
    if (job && a >= 0 && a + 3 < G) {
      typedef float f4a __attribute__((ext_vector_type(4), aligned(4)));
      const f4a v = *reinterpret_cast<const f4a *>(t);
      tg[i][0] = v[0], tg[i][1] = v[1], tg[i][2] = v[2], tg[i][3] = v[3];
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v) tg[i][v] = job && a + v >= 0 && a + v < G ? t[v] : 0.f;
    }
  }
  s4 b1[N1], b2[N2];
  const uint16_t *g1 = A.w1b + (size_t)s * kLbcHidden * kLbcTaps * kLbcCin;
  const uint16_t *g2 = A.w2b + (size_t)s * kLbcCout * kLbcTaps * kLbcHidden;
  const auto load2 = [&](int nt) {
#pragma unroll
    for (int i = 0; i < N2; ++i)
      b2[i] = ld4(g2 + ((16 * nt + m) * kLbcTaps + i / 2) * kLbcHidden + 16 * (i % 2) + 4 * g);
  };
#pragma unroll
  for (int i = 0; i < N1; ++i)
    b1[i] = ld4(g1 + ((16 * (wave & 1) + m) * kLbcTaps + i / 3) * kLbcCin + 16 * (i % 3) + 4 * g);
  load2(wave < 3 ? wave : 0);

  const auto input = [&](int ci, int row, int a, float v) {
    const int c = (ci % 24) / kLbcBand;
    const uint16_t u = f2bf(v * (c == 0 ? A.cs[0] : c == 1 ? A.cs[1] : A.cs[2]) * sc);
    xin[row * SX + ci] = u;
    if (a >= a0 && a < a0 + kTrainSeg && a < G)
      A.x[((size_t)b * kLbcCin + ci) * A.pitch + kPad + a] = u;
  };
#pragma unroll
  for (int i = 0; i < WC; ++i) input(wv * WC + i, l, al, r1[i]);
  if (q2 < NP) {
#pragma unroll
    for (int i = 0; i < WC / NP; ++i) input(wv * WC + NP * i + q2, row2, ah, r2[i]);
  }
  for (int e = tid; e < R * SH; e += 256) {
    hid[e] = 0;
    hid[(NR + R) * SH + e] = 0;
  }
  __syncthreads();

  // layer 1
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int nt = wave & 1, mt = (wave >> 1) + 2 * i;
    if (mt >= NT) break;
    f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < N1; ++j)
      acc = mfma(ld4(xin + (16 * mt + m + j / 3) * SX + 16 * (j % 3) + 4 * g), b1[j], acc);
    s4 o;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int hp = 16 * mt + 4 * g + v, a = a0 - 2 * R + hp;
      o[v] = a >= 0 && a < G ? (short)f2bf(acc[v]) : (short)0;
      hid[(hp + R) * SH + 16 * nt + m] = (uint16_t)o[v];
    }
    const int a = a0 - 2 * R + 16 * mt + 4 * g;
    if (a >= a0 && a < a0 + kTrainSeg)
      *reinterpret_cast<s4 *>(A.h + ((size_t)b * kLbcHidden + 16 * nt + m) * A.pitch + kPad + a) = o;
  }
  __syncthreads();

  // layer 2, the loss and its gradient; the weights of the way back are under way meanwhile
  s4 bb[NB];
  const uint16_t *gt = A.w2t + (size_t)s * kLbcHidden * kLbcTaps * kLbcCout;
#pragma unroll
  for (int i = 0; i < NB; ++i)
    bb[i] = ld4(gt + ((16 * (wave & 1) + m) * kLbcTaps + i / 3) * kLbcCout + 16 * (i % 3) + 4 * g);
  const int lo = s < 2 ? 0 : L, hi = s < 2 ? G : G - L;
  float lsum = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int nt = wave < 3 ? wave : i, mt = wave < 3 ? i : NT - 1;
    if (wave == 3) {
      if (i == 3) break;
      if (i > 0) load2(nt);
    }
    f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < N2; ++j)
      acc = mfma(ld4(hid + (16 * mt + m + j / 2) * SH + 16 * (j % 2) + 4 * g), b2[j], acc);
    const float wc = A.wch[16 * nt + m], cs = nt == 0 ? A.cs[0] : nt == 1 ? A.cs[1] : A.cs[2];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int hp = 16 * mt + 4 * g + v, p = a0 - 2 * R + hp;
      float d = 0.f;
      if (p >= lo && p < hi) {
        const float e = acc[v] - tg[i][v] * cs * sc;
        if (p >= a0 && p < a0 + kTrainSeg) lsum += wc * e * e;
        d = 2.f * wc * e * A.norm;
      }
      dyl[hp * SY + 16 * nt + m] = f2bf(d);
    }
  }
  for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o);
  if (l == 0) red[wave] = lsum;
  __syncthreads();
  if (tid == 0)
    A.loss[(size_t)b * gridDim.x + blockIdx.x] = (red[0] + red[1] + red[2] + red[3]) * A.norm;

  // dy and the gradient at the hidden layer, channel-major (rows past the strip are zeros)
#pragma unroll
  for (int i = 0; i < kLbcCout * kTrainSeg / 4 / 256; ++i) {
    const int e = tid + 256 * i, ch = e / (kTrainSeg / 4), q = e % (kTrainSeg / 4) * 4;
    s4 o;
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = (short)dyl[(2 * R + q + v) * SY + ch];
    *reinterpret_cast<s4 *>(A.dy + ((size_t)b * kLbcCout + ch) * A.pitch + kPad + a0 + q) = o;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int nt = wave & 1, mt = (wave >> 1) * 2 + i;
    f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NB; ++j)
      acc = mfma(ld4(dyl + (16 * mt + m + 3 * R - j / 3) * SY + 16 * (j % 3) + 4 * g), bb[j], acc);
    const int a = a0 + 16 * mt + 4 * g;
    s4 o;
#pragma unroll
    for (int v = 0; v < 4; ++v) o[v] = a + v < G ? (short)f2bf(acc[v]) : (short)0;
    *reinterpret_cast<s4 *>(A.dh + ((size_t)b * kLbcHidden + 16 * nt + m) * A.pitch + kPad + a) = o;
  }
}

// part[b][co][k][ci] = sum_p d[b, p, co] * in[b, p + k - R, ci] of both layers: one wave takes
// a 16 x 16 tile for all taps over the whole strip, so that the sum keeps its order and the
// taps are independent products.  A lane's four positions of the five taps lie in 16 bytes.
// Bound by the memory's latency over the positions, hence kChunk products' operands ahead.
__global__ __launch_bounds__(64) void k_train_weights(TrainStep A) {
  typedef uint32_t u4a __attribute__((ext_vector_type(4), aligned(4)));
  const int tile = blockIdx.x % 6, b = blockIdx.y;
  const bool first = blockIdx.x < 6;
  const int Co = first ? kLbcHidden : kLbcCout, Ci = first ? kLbcCin : kLbcHidden;
  const int nci = Ci / 16, co0 = tile / nci * 16, ci0 = tile % nci * 16;
  const int l = threadIdx.x, m = l & 15, g = l >> 4;
  const uint16_t *ra = (first ? A.dh : A.dy) + ((size_t)b * Co + co0 + m) * A.pitch + kPad + 4 * g;
  const uint16_t *rb = (first ? A.x : A.h) + ((size_t)b * Ci + ci0 + m) * A.pitch + kPad + 4 * g -
                       kLbcTaps / 2;
  struct Operands {
    s4 a[kChunk];
    u4a b[kChunk];
  };
  const auto load = [&](Operands &o, int c) {
#pragma unroll
    for (int i = 0; i < kChunk; ++i) {
      o.a[i] = ld4(ra + 16 * (kChunk * c + i));
      o.b[i] = *reinterpret_cast<const u4a *>(rb + 16 * (kChunk * c + i));
    }
  };
  f4 acc[kLbcTaps] = {};
  const auto multiply = [&](const Operands &o) {
#pragma unroll
    for (int i = 0; i < kChunk; ++i) {
      const u4a w = o.b[i];
      const uint32_t o0 = __builtin_amdgcn_alignbit(w[1], w[0], 16),
                     o1 = __builtin_amdgcn_alignbit(w[2], w[1], 16),
                     o2 = __builtin_amdgcn_alignbit(w[3], w[2], 16);
      const uint32_t v[kLbcTaps][2] = {{w[0], w[1]}, {o0, o1}, {w[1], w[2]}, {o1, o2}, {w[2], w[3]}};
#pragma unroll
      for (int k = 0; k < kLbcTaps; ++k) {
        s4 bv;
        __builtin_memcpy(&bv, v[k], 8);
        acc[k] = mfma(o.a[i], bv, acc[k]);
      }
    }
  };
  const int chunks = (A.G + 16 * kChunk - 1) / (16 * kChunk);
  Operands even, odd;
  load(even, 0);
  for (int c = 0; c < chunks; c += 2) {     // (loads past the end read the last chunk again)
    load(odd, min(c + 1, chunks - 1));
    __builtin_amdgcn_sched_barrier(0);
    multiply(even);
    if (c + 1 >= chunks) break;
    load(even, min(c + 2, chunks - 1));
    __builtin_amdgcn_sched_barrier(0);
    multiply(odd);
  }
  float *pb = (first ? A.part1 : A.part2) + (size_t)b * Co * kLbcTaps * Ci;
#pragma unroll
  for (int k = 0; k < kLbcTaps; ++k)
#pragma unroll
    for (int v = 0; v < 4; ++v)
      pb[((size_t)(co0 + 4 * g + v) * kLbcTaps + k) * Ci + ci0 + m] = acc[k][v];
}

struct TrainLayer {
  float *w, *m1, *m2;
  uint16_t *wb, *wt;
  const float *part;
  int Co, Ci;
};

// One weight a thread: its samples' gradients in order (four loads in flight), Adam, the copies.
__global__ __launch_bounds__(256) void k_train_update(TrainLayer first, TrainLayer second,
                                                      const int32_t *__restrict__ side, int B,
                                                      float lr, float b1, float b2, float eps,
                                                      float c1, float c2) {
  const TrainLayer &Y = blockIdx.z == 0 ? first : second;
  const int n = Y.Co * kLbcTaps * Y.Ci, i = blockIdx.x * 256 + threadIdx.x;
  const int s = blockIdx.y, l = threadIdx.x & 63;
  const int at = min(i, n - 1);
  float gi = 0.f;
  for (int b0 = 0; b0 < B; b0 += 64) {
    uint64_t mine = __ballot(b0 + l < B && side[min(b0 + l, B - 1)] == s);
    while (mine) {
      float v[4];
      int got = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (!mine) break;
        const int b = b0 + __builtin_ctzll(mine);
        mine &= mine - 1;
        v[j] = Y.part[(size_t)b * n + at];
        got = j + 1;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j < got) gi += v[j];
    }
  }
  if (i >= n) return;
  const size_t q = (size_t)s * n + i;
  const float a = b1 * Y.m1[q] + (1.f - b1) * gi;
  const float v = b2 * Y.m2[q] + (1.f - b2) * gi * gi;
  Y.m1[q] = a;
  Y.m2[q] = v;
  const float w = Y.w[q] - lr * (a / c1) / (sqrtf(v / c2) + eps);
  Y.w[q] = w;
  const int ci = i % Y.Ci, k = i / Y.Ci % kLbcTaps, co = i / (Y.Ci * kLbcTaps);
  const uint16_t h = f2bf(w);
  Y.wb[q] = h;
  Y.wt[(((size_t)s * Y.Ci + ci) * kLbcTaps + k) * Y.Co + co] = h;
}

// RMS of the pressure band of every frame and side: rms[f][s]
__global__ __launch_bounds__(256) void k_band_rms(const float *__restrict__ frames,
                                                  float *__restrict__ rms, int D, int G, int L) {
  __shared__ float red[256];
  const int f = blockIdx.x, s = blockIdx.y;
  float acc = 0.f;
  const int n = kLbcBand * (G - 2 * L);
  for (int e = threadIdx.x; e < n; e += 256) {
    const int j = e / (G - 2 * L), a = L + e % (G - 2 * L);
    const float v = frames[((((size_t)f * 3 + 0) * 4 + s) * D + L + j) * G + a];
    acc += v * v;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) rms[(size_t)f * 4 + s] = sqrtf(red[0] / (float)n);
}

// ---------------------------------------------------------------- fused inference, one step
__global__ __launch_bounds__(256) void k_lbc_step(LbcStep A) {
  constexpr int R = kLbcTaps / 2;
  constexpr int NX = kLbcSeg + 4 * R;                       // input positions
  constexpr int NH = (kLbcSeg + 2 * R + 15) / 16 * 16;      // hidden rows (whole MFMA tiles)
  constexpr int NXP = NH + 2 * R;                           // input rows the tiles read
  constexpr int NW1 = kLbcHidden * kLbcTaps * kLbcCin;
  constexpr int NW2 = kLbcCout * kLbcTaps * kLbcHidden;
  // input rows past NX feed only hidden rows past kLbcSeg + 2R, which layer 2 never reads;
  // they are zeroed so that every tile reads its operands without a bounds test
  __shared__ __attribute__((aligned(16))) uint16_t xin[NXP * kLbcCin];
  __shared__ __attribute__((aligned(16))) uint16_t hid[NH * kLbcHidden];
  __shared__ __attribute__((aligned(16))) uint16_t sw1[NW1];
  __shared__ __attribute__((aligned(16))) uint16_t sw2[NW2];
  __shared__ float outs[kLbcSeg * kLbcCout];
  const LbcStep &st = A;
  const int G = st.g, L = st.l;
  const int s = blockIdx.y, a0 = blockIdx.x * kLbcSeg;
  const int tid = threadIdx.x, wave = tid >> 6, l = tid & 63, m = l & 15, g = l >> 4;
  // top and bottom rows run along a (contiguous in memory), left and right columns along the
  // depth: the gather and the scatter let consecutive lanes walk the contiguous direction
  const bool along = s < 2;

  // this side's weights and the band inputs into LDS: every global load is issued before the
  // first LDS store, so the workgroup waits for one memory round trip, not one per element.
  // Components are picked by selects among the argument block's pointers: indexing the block
  // with a lane-varying component makes the compiler load the pointer itself first, one
  // dependent round trip per element
  constexpr int N1 = NW1 / 4, N2 = NW2 / 4, NI = NX * kLbcCin;
  constexpr int I1 = (N1 + 255) / 256, I2 = (N2 + 255) / 256, II = (NI + 255) / 256;
  s4 r1[I1], r2[I2];
  float rx[II];
  {
    const s4 *g1 = reinterpret_cast<const s4 *>(st.w1 + (size_t)s * NW1);
    const s4 *g2 = reinterpret_cast<const s4 *>(st.w2 + (size_t)s * NW2);
    // loads past the end re-read the last element (the LDS store below skips them): a load
    // under a branch would make the compiler wait for it where the branches join
#pragma unroll
    for (int i = 0; i < I1; ++i) r1[i] = g1[min(tid + 256 * i, N1 - 1)];
#pragma unroll
    for (int i = 0; i < I2; ++i) r2[i] = g2[min(tid + 256 * i, N2 - 1)];
    const float *cur0 = st.cur[0], *cur1 = st.cur[1], *cur2 = st.cur[2];
    const float *prv0 = st.prev[0], *prv1 = st.prev[1], *prv2 = st.prev[2];
#pragma unroll
    for (int i = 0; i < II; ++i) {
      const int e = tid + 256 * i;
      float v = 0.f;
      if (e < NI) {
        const int row = along ? e % NX : e / kLbcCin, ci = along ? e / NX : e % kLbcCin;
        const int a = a0 - 2 * R + row;
        if (a >= L && a < G - L) {
          const int h = ci / 24, c = (ci % 24) / kLbcBand, j = ci % kLbcBand;
          const float *src = h == 0 ? (c == 0 ? cur0 : c == 1 ? cur1 : cur2)
                                    : (c == 0 ? prv0 : c == 1 ? prv1 : prv2);
          v = src[lbc_cell(s, L + j, a, G)];
        }
      }
      rx[i] = v;
    }
    s4 *l1 = reinterpret_cast<s4 *>(sw1);
    s4 *l2 = reinterpret_cast<s4 *>(sw2);
#pragma unroll
    for (int i = 0; i < I1; ++i) {
      const int e = tid + 256 * i;
      if (e < N1) l1[e] = r1[i];
    }
#pragma unroll
    for (int i = 0; i < I2; ++i) {
      const int e = tid + 256 * i;
      if (e < N2) l2[e] = r2[i];
    }
    const float cs0 = A.cs[0], cs1 = A.cs[1], cs2 = A.cs[2];
    for (int e = NI + tid; e < NXP * kLbcCin; e += 256) xin[e] = 0;
#pragma unroll
    for (int i = 0; i < II; ++i) {
      const int e = tid + 256 * i;
      if (e < NI) {
        const int row = along ? e % NX : e / kLbcCin, ci = along ? e / NX : e % kLbcCin;
        const int c = (ci % 24) / kLbcBand;
        xin[row * kLbcCin + ci] = f2bf(rx[i] * (c == 0 ? cs0 : c == 1 ? cs1 : cs2));
      }
    }
  }
  __syncthreads();

  // layer 1: hid[hp][co], hidden position a = a0 - R + hp (zero outside the strip)
  const uint16_t *w1 = sw1;
  for (int t = wave; t < (NH / 16) * (kLbcHidden / 16); t += 4) {
    const int mt = t / (kLbcHidden / 16), nt = t % (kLbcHidden / 16);
    // all operands of the tile first, then the MFMA chain: one LDS round trip per tile
    constexpr int NC = kLbcCin / 16;
    s4 av[kLbcTaps * NC], bv[kLbcTaps * NC];
#pragma unroll
    for (int k = 0; k < kLbcTaps; ++k)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        av[k * NC + c] = ld4(xin + (16 * mt + m + k) * kLbcCin + 16 * c + 4 * g);
        bv[k * NC + c] = ld4(w1 + ((16 * nt + m) * kLbcTaps + k) * kLbcCin + 16 * c + 4 * g);
      }
    f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < kLbcTaps * NC; ++i) acc = mfma(av[i], bv[i], acc);
    for (int v = 0; v < 4; ++v) {
      const int hp = 16 * mt + 4 * g + v;
      const int a = a0 - R + hp;
      hid[hp * kLbcHidden + 16 * nt + m] = (a >= 0 && a < G) ? f2bf(acc[v]) : (uint16_t)0;
    }
  }
  __syncthreads();

  // layer 2: outs[op][co] at a = a0 + op
  const uint16_t *w2 = sw2;
  for (int t = wave; t < (kLbcSeg / 16) * (kLbcCout / 16); t += 4) {
    const int mt = t / (kLbcCout / 16), nt = t % (kLbcCout / 16);
    constexpr int NC = kLbcHidden / 16;
    s4 av[kLbcTaps * NC], bv[kLbcTaps * NC];
#pragma unroll
    for (int k = 0; k < kLbcTaps; ++k)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        av[k * NC + c] = ld4(hid + (16 * mt + m + k) * kLbcHidden + 16 * c + 4 * g);
        bv[k * NC + c] = ld4(w2 + ((16 * nt + m) * kLbcTaps + k) * kLbcHidden + 16 * c + 4 * g);
      }
    f4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < kLbcTaps * NC; ++i) acc = mfma(av[i], bv[i], acc);
    for (int v = 0; v < 4; ++v) outs[(16 * mt + 4 * g + v) * kLbcCout + 16 * nt + m] = acc[v];
  }
  __syncthreads();

  static_assert(kLbcSeg * kLbcCout % 256 == 0, "scatter covers the outputs in whole passes");
  float *const cur[3] = {st.cur[0], st.cur[1], st.cur[2]};
  float *const comp[3] = {st.cur_comp[0], st.cur_comp[1], st.cur_comp[2]};
  const float cs[3] = {A.cs[0], A.cs[1], A.cs[2]};
#pragma unroll
  for (int i = 0; i < kLbcSeg * kLbcCout / 256; ++i) {
    const int e = tid + 256 * i;
    const int op = along ? e % kLbcSeg : e / kLbcCout, co = along ? e / kLbcSeg : e % kLbcCout;
    const int a = a0 + op;
    if (a >= G || (!along && (a < L || a >= G - L))) continue;
    const int c = co / kLbcDepth, d = co % kLbcDepth;
    const int cell = lbc_cell(s, d, a, G);
    const float v = outs[op * kLbcCout + co];
    // one branch per component with a compile-time index keeps the pointers in scalar
    // registers (along the top and bottom rows c is uniform over each wave)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      if (c != k) continue;
      cur[k][cell] = v / cs[k];
      if (comp[k]) comp[k][cell] = 0.f;
    }
  }
}

}  // namespace

void launch_lbc_step(const LbcStep &st, hipStream_t s) {
  const int segs = (st.g + kLbcSeg - 1) / kLbcSeg;
  hipLaunchKernelGGL(k_lbc_step, dim3(segs, 4), dim3(256), 0, s, st);
}

}  // namespace fds

// ---------------------------------------------------------------- C-ABI (training side)
namespace {

hipStream_t as_stream(void *s) { return static_cast<hipStream_t>(s); }

int last_launch() { return hipGetLastError() == hipSuccess ? 0 : FDS_E_HIP; }

bool bad_dims(int Ci, int Co) { return Ci <= 0 || Co <= 0 || Ci % 16 || Co % 16; }

}  // namespace

extern "C" {

int fds_lbc_conv_fwd(const uint16_t *x, const uint16_t *w, const int32_t *side, float *y,
                     uint16_t *yb, int B, int P, int Ci, int Co, int K, void *stream) {
  if (bad_dims(Ci, Co) || B < 1 || B > 65535 || P < 1 || K < 1 || K % 2 == 0) return FDS_E_ARG;
  hipLaunchKernelGGL(fds::k_conv_fwd, dim3((P + 15) / 16, Co / 16, B), dim3(64), 0,
                     as_stream(stream), x, w, side, y, yb, P, Ci, Co, K);
  return last_launch();
}

int fds_lbc_conv_bwd_data(const uint16_t *dy, const uint16_t *wt, const int32_t *side,
                          float *dx, uint16_t *dxb, int B, int P, int Ci, int Co, int K,
                          void *stream) {
  if (bad_dims(Ci, Co) || B < 1 || B > 65535 || P < 1 || K < 1 || K % 2 == 0) return FDS_E_ARG;
  hipLaunchKernelGGL(fds::k_conv_bwd_data, dim3((P + 15) / 16, Ci / 16, B), dim3(64), 0,
                     as_stream(stream), dy, wt, side, dx, dxb, P, Ci, Co, K);
  return last_launch();
}

int fds_lbc_conv_bwd_weight(const uint16_t *dy, const uint16_t *x, float *part, int B, int P,
                            int Ci, int Co, int K, void *stream) {
  if (bad_dims(Ci, Co) || B < 1 || B > 65535 || P < 1 || K < 1 || K % 2 == 0) return FDS_E_ARG;
  hipLaunchKernelGGL(fds::k_conv_bwd_weight, dim3(K, (Co / 16) * (Ci / 16), B), dim3(64), 0,
                     as_stream(stream), dy, x, part, P, Ci, Co, K);
  return last_launch();
}

int fds_lbc_reduce_weight(const float *part, const int32_t *side, float *dw, int B, int S,
                          int n, void *stream) {
  if (B < 1 || S < 1 || n < 1) return FDS_E_ARG;
  hipLaunchKernelGGL(fds::k_reduce_weight, dim3((n + 255) / 256, S), dim3(256), 0,
                     as_stream(stream), part, side, dw, B, S, n);
  return last_launch();
}

int fds_lbc_mse(const float *y, const float *t, const int32_t *lo, const int32_t *hi,
                const float *wch, uint16_t *dyb, float *loss_part, int nblocks, int B, int P,
                int C, float norm, void *stream) {
  if (B < 1 || P < 1 || C < 1 || nblocks < 1) return FDS_E_ARG;
  hipLaunchKernelGGL(fds::k_mse, dim3(nblocks), dim3(256), 0, as_stream(stream), y, t, lo, hi,
                     wch, dyb, loss_part, B, P, C, norm);
  return last_launch();
}

int fds_lbc_adam(float *w, float *m1, float *m2, const float *g, int n, float lr, float b1,
                 float b2, float eps, int step, void *stream) {
  if (n < 1 || step < 1) return FDS_E_ARG;
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(fds::k_adam, dim3((n + 255) / 256), dim3(256), 0, as_stream(stream), w, m1,
                     m2, g, n, lr, b1, b2, eps, c1, c2);
  return last_launch();
}

int fds_lbc_pack(const float *w, uint16_t *wb, uint16_t *wtb, int S, int Co, int K, int Ci,
                 void *stream) {
  const int n = S * Co * K * Ci;
  if (n < 1) return FDS_E_ARG;
  hipLaunchKernelGGL(fds::k_pack, dim3((n + 255) / 256), dim3(256), 0, as_stream(stream), w, wb,
                     wtb, S, Co, K, Ci);
  return last_launch();
}

int fds_lbc_gather(const float *frames, const int32_t *run, const int32_t *step,
                   const int32_t *side, const float *scale, uint16_t *x, float *t, int B, int T,
                   int D, int G, int L, const float *comp_scale, void *stream) {
  if (B < 1 || B > 65535 || T < 2 || G < 2 * L + 1 || L != fds::kLbcDepth ||
      D < L + fds::kLbcBand)
    return FDS_E_ARG;
  hipLaunchKernelGGL(fds::k_gather, dim3((G + 255) / 256, B), dim3(256), 0, as_stream(stream),
                     frames, run, step, side, scale, x, t, T, D, G, L, comp_scale[0],
                     comp_scale[1], comp_scale[2]);
  return last_launch();
}

int fds_lbc_train_workspace(int B, int G, int64_t *bytes) {
  if (B < 1 || B > 65535 || G < 1) return FDS_E_ARG;
  const int64_t rows = (int64_t)B * 2 * (fds::kLbcCin + fds::kLbcHidden);
  const int64_t part = (int64_t)B * 2 * fds::kLbcCin * fds::kLbcTaps * fds::kLbcHidden;
  *bytes = rows * fds::train_pitch(G) * 2 + part * 4;
  return 0;
}

int fds_lbc_train(const float *frames, const int32_t *run, const int32_t *step,
                  const int32_t *side, const float *scale, const float *wch,
                  const fds_lbc_layer *layers, void *work, float *loss, int iters, int B, int T,
                  int D, int G, int L, const float *comp_scale, float lr, float b1, float b2,
                  float eps, int first_step, void *stream) {
  if (iters < 1 || B < 1 || B > 65535 || T < 2 || G < 2 * L + 1 || L != fds::kLbcDepth ||
      D < L + fds::kLbcBand || first_step < 1)
    return FDS_E_ARG;
  const hipStream_t q = as_stream(stream);
  const int segs = (G + fds::kTrainSeg - 1) / fds::kTrainSeg;
  constexpr int n = fds::kLbcCin * fds::kLbcTaps * fds::kLbcHidden;
  fds::TrainStep a{};
  a.frames = frames;
  a.wch = wch;
  a.w1b = layers[0].wb;
  a.w2b = layers[1].wb;
  a.w2t = layers[1].wt;
  a.T = T, a.D = D, a.G = G, a.L = L;
  a.pitch = fds::train_pitch(G);
  for (int c = 0; c < 3; ++c) a.cs[c] = comp_scale[c];
  a.norm = (float)(1.0 / ((double)B * G * 4.0));
  a.part1 = static_cast<float *>(work);
  a.part2 = a.part1 + (size_t)B * n;
  a.x = reinterpret_cast<uint16_t *>(a.part2 + (size_t)B * n);
  a.h = a.x + (size_t)B * fds::kLbcCin * a.pitch;
  a.dy = a.h + (size_t)B * fds::kLbcHidden * a.pitch;
  a.dh = a.dy + (size_t)B * fds::kLbcCout * a.pitch;
  a.loss = loss;
  const fds::TrainLayer y[2] = {
      {layers[0].w, layers[0].m, layers[0].v, layers[0].wb, layers[0].wt, a.part1,
       fds::kLbcHidden, fds::kLbcCin},
      {layers[1].w, layers[1].m, layers[1].v, layers[1].wb, layers[1].wt, a.part2,
       fds::kLbcCout, fds::kLbcHidden}};
  hipLaunchKernelGGL(fds::k_train_pads, dim3(B * 2 * (fds::kLbcCin + fds::kLbcHidden)), dim3(64),
                     0, q, a.x, G, a.pitch);
  for (int it = 0; it < iters; ++it) {
    a.run = run + (size_t)it * B;
    a.step = step + (size_t)it * B;
    a.side = side + (size_t)it * B;
    a.scale = scale + (size_t)it * B;
    const float t = (float)(first_step + it), c1 = 1.f - powf(b1, t), c2 = 1.f - powf(b2, t);
    hipLaunchKernelGGL(fds::k_train_grads, dim3(segs, B), dim3(256), 0, q, a);
    hipLaunchKernelGGL(fds::k_train_weights, dim3(12, B), dim3(64), 0, q, a);
    hipLaunchKernelGGL(fds::k_train_update, dim3((n + 255) / 256, 4, 2), dim3(256), 0, q, y[0],
                       y[1], a.side, B, lr, b1, b2, eps, c1, c2);
  }
  return last_launch();
}

int fds_lbc_band_rms(const float *frames, float *rms, int F, int D, int G, int L, void *stream) {
  if (F < 1 || F > 65535 || G < 2 * L + 1 || D < L + fds::kLbcBand) return FDS_E_ARG;
  hipLaunchKernelGGL(fds::k_band_rms, dim3(F, 4), dim3(256), 0, as_stream(stream), frames, rms,
                     D, G, L);
  return last_launch();
}

}  // extern "C"

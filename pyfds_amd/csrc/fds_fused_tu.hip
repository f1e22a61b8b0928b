// Fused step kernels of one numeric form and one stage count.  The build compiles this file
// once per form (FDS_FORM 0: float64, 1: float32, 2: float32 + Kahan) and stage count
// (FDS_STAGES), so they compile in parallel.
#include "fds_fused2d.h"
#include "fds_fused_lossy.h"
#include "fds_kernels.h"

#if !defined(FDS_FORM) || !defined(FDS_STAGES)
#error "compile with -DFDS_FORM=<0|1|2> -DFDS_STAGES=<count>"
#endif

#if FDS_FORM == 0
#define FDS_FORM_NS f64
#define FDS_T double
#define FDS_KAHAN false
#elif FDS_FORM == 1
#define FDS_FORM_NS f32
#define FDS_T float
#define FDS_KAHAN false
#else
#define FDS_FORM_NS k32
#define FDS_T float
#define FDS_KAHAN true
#endif

#define FDS_CAT2(a, b) a##b
#define FDS_CAT(a, b) FDS_CAT2(a, b)

namespace fds {
namespace FDS_FORM_NS {

using T = FDS_T;
constexpr bool K = FDS_KAHAN;

// Rows of loads in flight: 3 keep the memory busy at two or three waves per SIMD; 2 and 5
// measured within 3 % (5 takes the registers of one more wave).
constexpr int kRowsAhead = 3;
constexpr int kLossyRowsAhead = 2;   // (a stage holds more: 1 and 2 take the same registers)

template <int S, bool THERMAL, bool AXI, bool ISO, bool PAL>
__global__ __launch_bounds__(64) void k_fused(StepArgs<T> a) {
  __shared__ FusedLds<T, ISO, S> L;
  fused_tile<T, K, THERMAL, AXI, ISO, PAL, S, kRowsAhead>(a, a.dyn[0] + a.k, a.dyn[1] + a.k, L);
}

// (no workgroups: the kernel's code is loaded onto the device, which its first launch would do)
template <typename F>
void load_kernel(F *kernel) {
  hipFuncAttributes attr;
  (void)hipFuncGetAttributes(&attr, reinterpret_cast<const void *>(kernel));
}

template <int S, bool THERMAL, bool AXI, bool ISO, bool PAL>
void launch_fused(const void *args, int nblocks, size_t, hipStream_t s) {
  if (nblocks == 0) return load_kernel(k_fused<S, THERMAL, AXI, ISO, PAL>);
  hipLaunchKernelGGL((k_fused<S, THERMAL, AXI, ISO, PAL>), dim3(nblocks), dim3(64), 0, s,
                     *static_cast<const StepArgs<T> *>(args));
}

template <int S, bool AXI, bool ISO>
__global__ __launch_bounds__(64) void k_fused_lossy(StepArgs<T> a) {
  __shared__ LossyFusedLds<T, ISO, S> L;
  fused_lossy_tile<T, K, AXI, ISO, S, kLossyRowsAhead>(a, a.dyn[0] + a.k, a.dyn[1] + a.k, L);
}

template <int S, bool AXI, bool ISO>
void launch_fused_lossy(const void *args, int nblocks, size_t, hipStream_t s) {
  if (nblocks == 0) return load_kernel(k_fused_lossy<S, AXI, ISO>);
  hipLaunchKernelGGL((k_fused_lossy<S, AXI, ISO>), dim3(nblocks), dim3(64), 0, s,
                     *static_cast<const StepArgs<T> *>(args));
}

// Batched launch: the members' tiles with events first (they take longest), then all tiles in XCD
// bands.  40 FP32 members, 128 to 640 cells a side, 300 steps: 27.1 ms a pass with two steps per
// launch of the streaming shape, 14.0 ms here, the members' state transfers included.
template <int S, bool ANY>
__global__ __launch_bounds__(64) void k_fused_batch(const StepArgs<T> *__restrict__ descs,
                                                    const int32_t *__restrict__ tile_inst,
                                                    const int32_t *__restrict__ inst_base,
                                                    const int32_t *__restrict__ ev_inst,
                                                    const int32_t *__restrict__ ev_slot, int nev,
                                                    int ntiles, int k) {
  __shared__ FusedBatchLds<T, S> L;
  const int first = (nev + kNumXcd - 1) / kNumXcd * kNumXcd;
  const int b = blockIdx.x;
  if (b < first) {
    if (b >= nev) return;
    const StepArgs<T> &a = descs[ev_inst[b]];
    const int slot = __builtin_amdgcn_readfirstlane(ev_slot[b]);
    fused_any<T, K, ANY, true, S, 1>(a, __builtin_amdgcn_readfirstlane(a.fev.tiles[slot]), slot,
                                     a.dyn[0] + k, a.dyn[1] + k, L);
  } else {
    const int g = xcd_tile(b - first, gridDim.x - first, ntiles);
    if (g < 0) return;
    const int inst = tile_inst[g];
    const StepArgs<T> &a = descs[inst];
    const int tile = g - inst_base[inst];
    if (a.fev.slot[tile] >= 0) return;
    fused_any<T, K, ANY, false, S, kRowsAhead>(a, tile, -1, a.dyn[0] + k, a.dyn[1] + k, L);
  }
}

template <int S, bool ANY>
void launch_fused_batch(const BatchLaunch &b, int, size_t, hipStream_t s) {
  const int grid = xcd_grid(b.nev) + xcd_grid(b.ntiles);
  hipLaunchKernelGGL((k_fused_batch<S, ANY>), dim3(grid), dim3(64), 0, s,
                     static_cast<const StepArgs<T> *>(b.descs), b.tile_inst, b.inst_base,
                     b.ev_inst, b.ev_slot, b.nev, b.ntiles, b.k);
}

template <int S, bool THERMAL, bool PAL>
void fill_family(KernelSet &ks) {
  auto &f = ks.fused[THERMAL ? 1 : 0][PAL ? 1 : 0];
  f[0][S - 1] = launch_fused<S, THERMAL, false, false, PAL>;
  f[1][S - 1] = launch_fused<S, THERMAL, true, false, PAL>;
  f[2][S - 1] = launch_fused<S, THERMAL, false, true, PAL>;
}

void FDS_CAT(fill_fused_, FDS_STAGES)(KernelSet &ks) {
  constexpr int S = FDS_STAGES;
  static_assert(S >= 1 && S <= kFusedMax, "stage count out of range");
  fill_family<S, false, false>(ks);
  fill_family<S, false, true>(ks);
  fill_family<S, true, false>(ks);
  fill_family<S, true, true>(ks);
  ks.fused_batch[0][S - 1] = launch_fused_batch<S, false>;
  ks.fused_batch[1][S - 1] = launch_fused_batch<S, true>;
  if constexpr (S <= kFusedLossyMax) {
    // (four stages: the FP32 forms' plane fields only, see choose_fused)
    if constexpr (S < kFusedLossyMax) ks.fused_lossy[1][S - 1] = launch_fused_lossy<S, true, false>;
    if constexpr (S < kFusedLossyMax || sizeof(T) == 4) {
      ks.fused_lossy[0][S - 1] = launch_fused_lossy<S, false, false>;
      ks.fused_lossy[2][S - 1] = launch_fused_lossy<S, false, true>;
    }
  }
}

}  // namespace FDS_FORM_NS
}  // namespace fds

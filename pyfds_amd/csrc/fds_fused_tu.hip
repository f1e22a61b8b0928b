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

template <int S, bool THERMAL, bool AXI, bool ISO, bool PAL>
void launch_fused(const void *args, int nblocks, size_t, hipStream_t s) {
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
  hipLaunchKernelGGL((k_fused_lossy<S, AXI, ISO>), dim3(nblocks), dim3(64), 0, s,
                     *static_cast<const StepArgs<T> *>(args));
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
  if constexpr (S <= kFusedLossyMax) {
    ks.fused_lossy[0][S - 1] = launch_fused_lossy<S, false, false>;
    ks.fused_lossy[1][S - 1] = launch_fused_lossy<S, true, false>;
    ks.fused_lossy[2][S - 1] = launch_fused_lossy<S, false, true>;
  }
}

}  // namespace FDS_FORM_NS
}  // namespace fds

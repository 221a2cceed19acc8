// sxc_scan_kernels.h -- the diagonal scan's kernel as a template over the transform length and
// the kind of pair (bits 5 and 6 of NB, see ScanSmem), and its launch.  One translation unit
// per kind (sxc_scan_pure.hip, sxc_scan_n.hip, sxc_scan_general.hip), so they compile side by side.
#pragma once
#include "sxc_fft_kernels.h"
#include "sxc_kernels.h"

namespace sxc {

struct NoRegs {};

// The pure-A/C/G/T scan kernel gets a register budget for as many of its 4-wave
// workgroups per CU as its LDS plan admits, up to 8 waves per SIMD (measured on the 4096-pair
// workload at N = 8192 with byte-parallel flags: 5 waves 1.05 ms, 6: 1.00 ms, 7: 0.94 ms,
// 8: 0.93 ms; the spills the budget costs are cheaper than the latency the extra waves hide).
template <int NB>
constexpr int scan_waves() {
  if constexpr (!ScanSmem<NB>::PURE) {
    return 1;
  } else {
    constexpr int wg = 163840 / ScanSmem<NB>::BYTES;
    return wg < 1 ? 1 : (wg > 8 ? 8 : wg);
  }
}
static_assert(scan_waves<13 | 32>() == 8, "the pure scan's LDS plan at N = 8192 fits 8 workgroups per CU");

template <int NB>
__global__ __launch_bounds__(SCAN_NT) __attribute__((amdgpu_waves_per_eu(scan_waves<NB>()))) void k_scan(ScanArgs a) {
  __shared__ __align__(16) char sm[ScanSmem<NB>::BYTES];
  NoRegs r;
  DevExec<NoRegs> ex{r};
  scan_body<NB>(ex, sm, a, (int)blockIdx.x);
}

// The scan of one kind (KIND: 32, 64 or 0) over `grid` workgroups.
template <int KIND>
hipError_t launch_scan_kind(int nb, const ScanArgs& a, int grid, hipStream_t s) {
  switch (nb) {
#define SXC_SCAN_CASE(X)                                                          \
  case X:                                                                         \
    hipLaunchKernelGGL(k_scan<(X) | KIND>, dim3(grid), dim3(SCAN_NT), 0, s, a);    \
    break;
    SXC_SCAN_CASE(9)
    SXC_SCAN_CASE(10)
    SXC_SCAN_CASE(11)
    SXC_SCAN_CASE(12)
    SXC_SCAN_CASE(13)
    SXC_SCAN_CASE(14)
    SXC_SCAN_CASE(15)
#undef SXC_SCAN_CASE
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace sxc

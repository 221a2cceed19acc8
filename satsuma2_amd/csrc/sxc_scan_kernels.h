// sxc_scan_kernels.h -- the diagonal scan's kernel as a template over the transform length and
// the kind of pair (bits 5 and 6 of NB, see ScanSmem), and its launch.  One translation unit
// per kind (sxc_scan_pure.hip, sxc_scan_n.hip, sxc_scan_general.hip), so they compile side by side.
#pragma once
#include "sxc_fft_kernels.h"
#include "sxc_kernels.h"

namespace sxc {

struct NoRegs {};

// Waves per SIMD the register budget is set for.  The sliced scan (pure A/C/G/T) keeps 32 words of
// a slice and their counts in registers: 6 waves (80 registers, 6 spilled) take 0.507 ms for 8192
// strands at N = 8192 and 1.47 for 24000 at 2048, 5 waves 0.529 and 1.53, 8 (26 spilled) 0.515 and
// 1.40.  The general scan is compiled for 5 waves also where its LDS plan admits fewer workgroups (4 at
// N = 8192, 2 at 16384): it then has the same registers (106, none spilled), but compiled for as many as fit
// it took 276 instead of 224 us for 128 strands with one other letter at N = 8192 and 559 instead of 446
// at 16384.  The A/C/G/T/N scan gets as many of its 4-wave workgroups per CU as its LDS plan admits,
// up to 8 waves (the spills the budget costs are cheaper than the latency the waves hide).
template <int NB>
constexpr int scan_waves() {
  if constexpr (ScanSmem<NB>::SLICED) {
    return 6;
  } else if constexpr (!ScanSmem<NB>::PURE) {
    return 5;
  } else {
    constexpr int wg = 163840 / ScanSmem<NB>::BYTES;
    return wg < 1 ? 1 : (wg > 8 ? 8 : wg);
  }
}

// Workgroups that a CU holds at once.
template <int NB>
constexpr int scan_resident() {
  constexpr int wg = 163840 / ScanSmem<NB>::BYTES;
  return wg < scan_waves<NB>() ? wg : scan_waves<NB>();
}
static_assert(scan_resident<12>() == 5 && scan_resident<13>() == 4 && scan_resident<14>() == 2, "");
static_assert(scan_resident<15>() == 1 && scan_resident<15 | 64>() == 2, "");

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

// sxc_kernels_parts.hip -- the pair and spectra kernels with a workgroup per channel, for launches
// too small to fill the device (CHANNEL_SPLIT).
//
// Such a launch takes as long as one workgroup, and a workgroup's time is latency: four channels
// in a row, each a chain of LDS rounds with barriers between.  Here each channel has a workgroup
// (which repeats the chunk's preparation, about a fifth of its time), and a second kernel adds the
// four correlations in their order and looks for the peaks.  One 4096-bp pair, both strands: target
// spectra 46 -> 24 us, pair kernel 68 -> 38 us with the sum; 64 pairs with resident query
// spectra 36 -> 28 us.  One geometry per length: the default, whose 16-wide
// stage A gives a transform twice the threads of the 32-wide one and so the shorter chain.
#include "sxc_fft_kernels.h"
#include "sxc_kernels.h"

namespace sxc {

template <int NB>
__global__ __launch_bounds__(Geo<NB>::NT) void k_correlate_part(PairArgs a) {
  __shared__ __align__(16) char sm[Smem<NB>::BYTES];
  Regs<NB> r;
  DevExec<Regs<NB>> ex{r};
  const int b = (int)blockIdx.x;
  correlate_body<NB, true>(ex, sm, a, b >> 2, b & 3, (b & 3) + 1);
}

template <int NB>
__global__ __launch_bounds__(Geo<NB>::NT) void k_sum_peaks(PairArgs a) {
  __shared__ __align__(16) char sm[Smem<NB>::BYTES];
  Regs<NB> r;
  DevExec<Regs<NB>> ex{r};
  sum_peaks_body<NB>(ex, sm, a, (int)blockIdx.x);
}

template <int NB>
__global__ __launch_bounds__(Geo<NB>::NT) void k_spectra_part(SpecArgs a) {
  __shared__ __align__(16) char sm[Smem<NB>::BYTES];
  Regs<NB> r;
  DevExec<Regs<NB>> ex{r};
  const int b = (int)blockIdx.x;
  spectra_body<NB>(ex, sm, a, b >> 2, b & 3, (b & 3) + 1);
}

#define SXC_NB_SWITCH(NB, CALL)      \
  switch (NB) {                      \
    case 9: CALL(9); break;          \
    case 10: CALL(10); break;        \
    case 11: CALL(11); break;        \
    case 12: CALL(12); break;        \
    case 13: CALL(13); break;        \
    case 14: CALL(14); break;        \
    case 15: CALL(15); break;        \
    default: return hipErrorInvalidValue; \
  }

hipError_t launch_correlate_parts(int nb, const PairArgs& a, int total, hipStream_t s) {
#define CALL(X)                                                                              \
  hipLaunchKernelGGL(k_correlate_part<X>, dim3(4 * total), dim3(Geo<X>::NT), 0, s, a);        \
  hipLaunchKernelGGL(k_sum_peaks<X>, dim3(total), dim3(Geo<X>::NT), 0, s, a)
  SXC_NB_SWITCH(nb, CALL)
#undef CALL
  return hipGetLastError();
}

hipError_t launch_spectra_parts(int nb, const SpecArgs& a, hipStream_t s) {
#define CALL(X) hipLaunchKernelGGL(k_spectra_part<X>, dim3(4 * a.n), dim3(Geo<X>::NT), 0, s, a)
  SXC_NB_SWITCH(nb, CALL)
#undef CALL
  return hipGetLastError();
}

}  // namespace sxc

// sxc_scan_pure.hip -- the diagonal scan of pairs whose two chunks are pure A/C/G/T.
#include "sxc_scan_kernels.h"

namespace sxc {

hipError_t launch_scan_pure(int nb, const ScanArgs& a, int grid, hipStream_t s) {
  return launch_scan_kind<32>(nb, a, grid, s);
}

}  // namespace sxc

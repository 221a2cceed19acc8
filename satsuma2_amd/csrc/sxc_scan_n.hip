// sxc_scan_n.hip -- the diagonal scan of pairs of A/C/G/T/N chunks with an N.
#include "sxc_scan_kernels.h"

namespace sxc {

hipError_t launch_scan_n(int nb, const ScanArgs& a, int grid, hipStream_t s) {
  return launch_scan_kind<64>(nb, a, grid, s);
}

}  // namespace sxc

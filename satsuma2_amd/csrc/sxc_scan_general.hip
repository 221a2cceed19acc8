// sxc_scan_general.hip -- the diagonal scan of pairs with any other letter.
#include "sxc_scan_kernels.h"

namespace sxc {

hipError_t launch_scan_general(int nb, const ScanArgs& a, int grid, hipStream_t s) {
  return launch_scan_kind<0>(nb, a, grid, s);
}

}  // namespace sxc

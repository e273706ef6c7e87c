// Scan kernels of the long-context summon: 4 subspaces.
#include "summon_wide.cuh"

namespace sva {
namespace wide {

int launch_scan_4(const WideArgs& a, int64_t items, bool masked, int kp, hipStream_t stream) {
  return launch_wide_s<4, false>(a, items, masked, kp, stream);
}

}  // namespace wide
}  // namespace sva

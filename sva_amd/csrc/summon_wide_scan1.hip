// Scan kernels of the long-context summon: 1 subspace.
#include "summon_wide.cuh"

namespace sva {
namespace wide {

int launch_scan_1(const WideArgs& a, int64_t items, bool masked, int kp, hipStream_t stream) {
  return launch_wide_s<1, false>(a, items, masked, kp, stream);
}

}  // namespace wide
}  // namespace sva

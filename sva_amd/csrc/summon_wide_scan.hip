// Scan of the long-context summon: the code widths S, one translation unit
// each (summon_wide_scan<S>.hip), for every table width and masking.
#include "summon_wide.cuh"

namespace sva {
namespace wide {

int launch_scan(const WideArgs& a, int64_t items, bool masked, int kp, hipStream_t stream) {
  switch (a.p.S) {
    case 1: return launch_scan_1(a, items, masked, kp, stream);
    case 2: return launch_scan_2(a, items, masked, kp, stream);
    case 4: return launch_scan_4(a, items, masked, kp, stream);
    default: return launch_scan_8(a, items, masked, kp, stream);
  }
}

int launch_scan_8(const WideArgs& a, int64_t items, bool masked, int kp, hipStream_t stream) {
  return launch_wide_s<8, false>(a, items, masked, kp, stream);
}

}  // namespace wide
}  // namespace sva

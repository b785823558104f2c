// The selective scan of channels with 9 - 16 states (selective_scan.hip), taken by launch_selective_scan. Same contract: capturable,
// no allocation.
#pragma once

#include "rec_launchers.h"

namespace die {

hipError_t launch_scan_lanes(const SelectiveScanArgs& a, RaggedRows r, hipStream_t s);

}  // namespace die

// zwalk_map.hip -- map (hit-count) walks on the unfolded image (zwalk_launch.h).
#include "zwalk_launch.h"

namespace rwnmr {

template hipError_t launch_z_mode<0>(const WalkArgs &, const LaunchShape &, uint32_t, hipStream_t);

}  // namespace rwnmr

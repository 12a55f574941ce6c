// zwalk_cpmg.hip -- CPMG walks on the unfolded image (zwalk_launch.h).
#include "zwalk_launch.h"

namespace rwnmr {

template hipError_t launch_z_mode<1>(const WalkArgs &, const LaunchShape &, uint32_t, hipStream_t);

}  // namespace rwnmr

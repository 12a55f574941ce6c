// zwalk_mirror.hip -- mirror CPMG, map and per-label walks with reflection
// flags on the unfolded image (zwalk_launch.h).
#include "zwalk_launch.h"

namespace rwnmr {

template <int EMODE>
hipError_t launch_z_mirror(const WalkArgs &a, const LaunchShape &ls, uint32_t blocks, hipStream_t st)
{
    if (a.zcache == 5) {   // 8-byte chunk cache
        if (EMODE < 2 && ls.threads >= 1024)
            return a.zl.wrapfix ? launch_z<EMODE, true, 64, 3, false, true>(a, ls, blocks, st)
                                : launch_z<EMODE, false, 64, 3, false, true>(a, ls, blocks, st);
        return a.zl.wrapfix ? launch_z<EMODE, true, 64, 2, false, true>(a, ls, blocks, st)
                            : launch_z<EMODE, false, 64, 2, false, true>(a, ls, blocks, st);
    }
    // CPMG and map walks of 1024-thread blocks read the flag-keyed
    // tables (58 KiB of LDS: two blocks per CU, 8 waves per SIMD)
    if (EMODE < 2 && ls.threads >= 1024)
        return a.zl.wrapfix ? launch_z<EMODE, true, 128, 3, false, true>(a, ls, blocks, st)
                            : launch_z<EMODE, false, 128, 3, false, true>(a, ls, blocks, st);
    return a.zl.wrapfix ? launch_z<EMODE, true, 128, 2, false, true>(a, ls, blocks, st)
                        : launch_z<EMODE, false, 128, 2, false, true>(a, ls, blocks, st);
}

#if !defined(RWNMR_MIRROR_EMODE)
#error "compiled once per energy mode"
#endif
template hipError_t launch_z_mirror<RWNMR_MIRROR_EMODE>(const WalkArgs &, const LaunchShape &, uint32_t, hipStream_t);

}  // namespace rwnmr

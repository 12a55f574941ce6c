// zwalk_spec.hip -- the speculative CPMG walk (zwalk_tile_spec) for runs of
// few walkers.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "walk_common.h"
#include "walk_device.h"
#include "zwalk_device.h"
#include "zwalk_kernels.h"

namespace rwnmr {

// Speculative CPMG walk (zwalk_tile_spec): one walker per lane, for runs
// too small to hide the chunk-load latency of a step.
template <bool WRAPFIX, bool NOFLUX, bool MFLAGS>
__global__ __launch_bounds__(1024) void zwalk_spec_kernel(const WalkArgs a)
{
    __shared__ double lds[kEchoChunk][kEchoCols];
    __shared__ uint4 tab[MFLAGS ? 8 * kZFlagStride / 16 : (NOFLUX ? 12 : 6)];
    __shared__ uint2 fix[MFLAGS ? 8 * kZFlagStride / 16 : 6];
    __shared__ uint8_t keys[kZKeyEntries];
    const uint64_t tile = tile_of_block(a);
    if (a.tile_map && tile >= a.n_tiles)
        return;  // spare workgroup of the XCD-striped grid (whole block leaves together)
    if (NOFLUX)
        zbuild_table_noflux(a.zl, tab);
    else if (MFLAGS)
        zbuild_table_flags(a.zl, tab, fix);
    else
        zbuild_table(a.zl, tab, fix);
    zbuild_key_table(keys, NOFLUX ? 32u : 16u);
    __syncthreads();
    zwalk_tile_spec<WRAPFIX, NOFLUX, MFLAGS>(a, tile, a.partials ? a.partials + tile : nullptr, a.partial_stride,
                                             lds, tab, fix, keys);
}

template <bool WRAPFIX, bool NOFLUX, bool MFLAGS>
static hipError_t launch_spec(const WalkArgs &a, const LaunchShape &ls, uint32_t blocks, hipStream_t st)
{
    hipLaunchKernelGGL((zwalk_spec_kernel<WRAPFIX, NOFLUX, MFLAGS>), dim3(blocks), dim3(ls.threads), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_z_spec(const WalkArgs &a, const LaunchShape &ls, uint32_t blocks, hipStream_t st)
{
    if (a.znoflux)
        return launch_spec<false, true, false>(a, ls, blocks, st);
    if (a.zmflags)
        return a.zl.wrapfix ? launch_spec<true, false, true>(a, ls, blocks, st)
                            : launch_spec<false, false, true>(a, ls, blocks, st);
    return a.zl.wrapfix ? launch_spec<true, false, false>(a, ls, blocks, st)
                        : launch_spec<false, false, false>(a, ls, blocks, st);
}

}  // namespace rwnmr

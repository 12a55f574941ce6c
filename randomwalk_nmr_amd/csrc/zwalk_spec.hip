// zwalk_spec.hip -- the speculative CPMG and map walks (zwalk_tile_spec) for
// runs of few walkers.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "walk_common.h"
#include "walk_device.h"
#include "zwalk_device.h"
#include "zwalk_kernels.h"

namespace rwnmr {

template <int EMODE, bool WRAPFIX, bool NOFLUX, bool MFLAGS, bool SUB>
__global__ __launch_bounds__(1024) void zwalk_spec_kernel(const WalkArgs a)
{
    extern __shared__ double zrows[];   // kZRowEchoes x kZRowStride per wave
    __shared__ double lds[kEchoChunk][kEchoCols];
    __shared__ uint4 tab[MFLAGS ? 8 * kZFlagStride / 16 : (NOFLUX ? 12 : 6)];
    __shared__ uint2 fix[MFLAGS ? 8 * kZFlagStride / 16 : 6];
    __shared__ __align__(16) uint8_t keys[kZKeyEntries];
    const uint64_t tile = tile_of_block(a);
    if (a.tile_map && tile >= a.n_tiles)
        return;  // spare workgroup of the XCD-striped grid (whole block leaves together)
    if (NOFLUX)
        zbuild_table_noflux(a.zl, tab, SUB ? (uint32_t)a.shift : 0u);
    else if (MFLAGS)
        zbuild_table_flags(a.zl, tab, fix);
    else
        zbuild_table(a.zl, tab, fix);
    zbuild_key_table(keys, NOFLUX ? 32u : 16u);
    __syncthreads();
    zwalk_tile_spec<EMODE, WRAPFIX, NOFLUX, MFLAGS, SUB>(a, tile, a.partials ? a.partials + tile : nullptr,
                                                         a.partial_stride, lds, zrows, tab, fix, keys);
}

template <int EMODE, bool SUB>
static hipError_t launch_spec(const WalkArgs &a, uint32_t threads, uint32_t blocks, hipStream_t st)
{
    const dim3 g(blocks), t(threads);
    const size_t rows = (size_t)(threads / kWave) * kZRowEchoes * kZRowStride * sizeof(double);
    if (a.znoflux)
        hipLaunchKernelGGL((zwalk_spec_kernel<EMODE, false, true, false, SUB>), g, t, rows, st, a);
    else if (a.zmflags && a.zl.wrapfix)
        hipLaunchKernelGGL((zwalk_spec_kernel<EMODE, true, false, true, SUB>), g, t, rows, st, a);
    else if (a.zmflags)
        hipLaunchKernelGGL((zwalk_spec_kernel<EMODE, false, false, true, SUB>), g, t, rows, st, a);
    else if (a.zl.wrapfix)
        hipLaunchKernelGGL((zwalk_spec_kernel<EMODE, true, false, false, SUB>), g, t, rows, st, a);
    else
        hipLaunchKernelGGL((zwalk_spec_kernel<EMODE, false, false, false, SUB>), g, t, rows, st, a);
    return hipGetLastError();
}

hipError_t launch_z_spec(const WalkArgs &a, int emode, const LaunchShape &ls, uint32_t blocks, hipStream_t st)
{
    if (emode == 0)
        return a.shift ? launch_spec<0, true>(a, ls.threads, blocks, st) : launch_spec<0, false>(a, ls.threads, blocks, st);
    return a.shift ? launch_spec<1, true>(a, ls.threads, blocks, st) : launch_spec<1, false>(a, ls.threads, blocks, st);
}

}  // namespace rwnmr

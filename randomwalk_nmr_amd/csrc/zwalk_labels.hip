// zwalk_labels.hip -- per-label CPMG walks on the unfolded image
// (zwalk_launch.h): the labelled walk, the label-set walk and the Jacobian
// forward.
#include "zwalk_launch.h"

namespace rwnmr {

template hipError_t launch_z_mode<2>(const WalkArgs &, const LaunchShape &, uint32_t, hipStream_t);

// Label-set CPMG: 8 sets of label deltas evaluated on one trajectory (one
// walker per lane; zwalk_tile with NS = 8).  Unused sets (a.n_label_sets <
// 8) carry deltas of 1.
template <bool WRAPFIX, bool NOFLUX, bool MFLAGS>
__global__ __launch_bounds__(1024) void zwalk_sets_kernel(const WalkArgs a)
{
    extern __shared__ double lds8[];   // kEchoChunk x 8 sets x waves of the block
    __shared__ uint4 tab[MFLAGS ? 8 * kZFlagStride / 16 : (NOFLUX ? 12 : 6)];
    __shared__ uint2 fix[MFLAGS ? 8 * kZFlagStride / 16 : 6];
    __shared__ __align__(16) uint8_t keys[kZKeyEntries];
    __shared__ double ldelta[8 * kMaxLabels];
    const uint64_t tile = tile_of_block(a);
    if (a.tile_map && tile >= a.n_tiles)
        return;
    if (NOFLUX)
        zbuild_table_noflux(a.zl, tab);
    else if (MFLAGS)
        zbuild_table_flags(a.zl, tab, fix);
    else
        zbuild_table(a.zl, tab, fix);
    zbuild_key_table(keys, NOFLUX ? 32u : 16u);
    for (uint32_t t = threadIdx.x; t < 8u * kMaxLabels; t += blockDim.x) {
        const uint32_t q = t / kMaxLabels, l = t % kMaxLabels;
        ldelta[t] = (q < a.n_label_sets && (int)l < a.n_labels) ? a.label_delta[q * (uint32_t)a.n_labels + l] : 1.0;
    }
    __syncthreads();
    zwalk_tile<2, 1, WRAPFIX, 128, 2, NOFLUX, MFLAGS, 8>(a, tile, a.partials ? a.partials + tile : nullptr,
                                                         a.partial_stride, nullptr, tab, fix, ldelta, keys, nullptr,
                                                         lds8);
}

// Jacobian forward: the per-label CPMG walk (zwalk_tile EMODE 2, one walker
// per lane, per-label hit counts in LDS) that also sums h_l E per label and
// echo (zwalk_tile JAC).  Dynamic LDS: the 8-label echo staging (kEchoChunk
// x 8 x waves doubles), then the hit-count rows (blockDim x kLhStride).
template <bool WRAPFIX, bool NOFLUX, bool MFLAGS>
__global__ __launch_bounds__(1024) void zwalk_jac_kernel(const WalkArgs a)
{
    extern __shared__ double zjdyn[];
    __shared__ double lds[kEchoChunk][kEchoCols];
    __shared__ uint4 tab[MFLAGS ? 8 * kZFlagStride / 16 : (NOFLUX ? 12 : 6)];
    __shared__ uint2 fix[MFLAGS ? 8 * kZFlagStride / 16 : 6];
    __shared__ __align__(16) uint8_t keys[kZKeyEntries];
    __shared__ double ldelta[kMaxLabels];
    const uint64_t tile = tile_of_block(a);
    if (a.tile_map && tile >= a.n_tiles)
        return;
    double *lds8 = zjdyn;
    uint32_t *zlh = reinterpret_cast<uint32_t *>(zjdyn + (size_t)kEchoChunk * 8 * (blockDim.x / kWave));
    if (NOFLUX)
        zbuild_table_noflux(a.zl, tab);
    else if (MFLAGS)
        zbuild_table_flags(a.zl, tab, fix);
    else
        zbuild_table(a.zl, tab, fix);
    zbuild_key_table(keys, NOFLUX ? 32u : 16u);
    if (threadIdx.x < kMaxLabels)
        ldelta[threadIdx.x] = (int)threadIdx.x < a.n_labels ? a.label_delta[threadIdx.x] : 1.0;
    __syncthreads();
    zwalk_tile<2, 1, WRAPFIX, 128, 2, NOFLUX, MFLAGS, 1, true>(a, tile, a.partials ? a.partials + tile : nullptr,
                                                               a.partial_stride, lds, tab, fix, ldelta, keys, zlh,
                                                               lds8);
}

hipError_t launch_zwalk_sets(const WalkArgs &a, uint32_t threads, hipStream_t st)
{
    if (a.n == 0)
        return hipSuccess;
    if (a.shift != 0 || !a.zwords || !a.zlabels || !a.label_delta || a.n_labels <= 0 || a.n_labels > kMaxLabels ||
        a.n_label_sets == 0 || a.n_label_sets > 8 || threads == 0 || threads > 1024 || threads % 64 != 0)
        return hipErrorInvalidValue;
    const uint64_t tiles = (a.n + threads - 1) / threads;
    if (tiles > 0x7FFFFFF0ull || (a.tile_map && a.n_tiles != tiles))
        return hipErrorInvalidValue;
    const uint32_t blocks = a.tile_map ? (uint32_t)(((tiles + kXcds - 1) / kXcds) * kXcds) : (uint32_t)tiles;
    // the per-set echo staging, sized for this block's waves
    const size_t lds8_bytes = (size_t)kEchoChunk * 8 * (threads / kWave) * sizeof(double);
    const dim3 g(blocks), b(threads);
#define RW_SETS(WF, NF, MF) hipLaunchKernelGGL((zwalk_sets_kernel<WF, NF, MF>), g, b, lds8_bytes, st, a)
    if (a.znoflux)
        RW_SETS(false, true, false);
    else if (a.zmflags && a.zl.wrapfix)
        RW_SETS(true, false, true);
    else if (a.zmflags)
        RW_SETS(false, false, true);
    else if (a.zl.wrapfix)
        RW_SETS(true, false, false);
    else
        RW_SETS(false, false, false);
#undef RW_SETS
    return hipGetLastError();
}

hipError_t launch_zwalk_jac(const WalkArgs &a, uint32_t threads, hipStream_t st)
{
    if (a.n == 0)
        return hipSuccess;
    if (a.shift != 0 || !a.zwords || !a.zlabels || !a.label_delta || !a.partials || !a.jac_partials ||
        a.n_labels <= 0 || a.n_labels > kMaxLabels || threads == 0 || threads > 1024 || threads % 64 != 0)
        return hipErrorInvalidValue;
    const uint64_t tiles = (a.n + threads - 1) / threads;
    if (tiles > 0x7FFFFFF0ull || (a.tile_map && a.n_tiles != tiles))
        return hipErrorInvalidValue;
    const uint32_t blocks = a.tile_map ? (uint32_t)(((tiles + kXcds - 1) / kXcds) * kXcds) : (uint32_t)tiles;
    const size_t dyn = (size_t)kEchoChunk * 8 * (threads / kWave) * sizeof(double) +
                       (size_t)kLhStride * threads * sizeof(uint32_t);
    const dim3 g(blocks), b(threads);
#define RW_JAC(WF, NF, MF) hipLaunchKernelGGL((zwalk_jac_kernel<WF, NF, MF>), g, b, dyn, st, a)
    if (a.znoflux)
        RW_JAC(false, true, false);
    else if (a.zmflags && a.zl.wrapfix)
        RW_JAC(true, false, true);
    else if (a.zmflags)
        RW_JAC(false, false, true);
    else if (a.zl.wrapfix)
        RW_JAC(true, false, false);
    else
        RW_JAC(false, false, false);
#undef RW_JAC
    return hipGetLastError();
}

}  // namespace rwnmr

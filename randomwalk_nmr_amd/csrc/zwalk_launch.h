// zwalk_launch.h -- the CPMG / map / per-label walk kernel on the unfolded
// image (step described in zwalk_device.h) and the choice of its instance.
// Included by one source per energy mode (zwalk_map.hip, zwalk_cpmg.hip,
// zwalk_labels.hip), which compile side by side.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "walk_common.h"
#include "walk_device.h"
#include "zwalk_device.h"
#include "zwalk_kernels.h"

namespace rwnmr {

// The speculative CPMG (emode 1) and map (0) walks (zwalk_spec.hip), one
// walker per lane.
hipError_t launch_z_spec(const WalkArgs &a, int emode, const LaunchShape &ls, uint32_t blocks, hipStream_t st);

template <int EMODE, int K, bool WRAPFIX, int CACHE, int TAB, bool NOFLUX = false, bool MFLAGS = false,
          bool ADISP = false, bool HITS = true, bool SUB = false>
// 80 SGPRs: with 16 more kept for the trap handler a wave then takes 96 of the
// SIMD's 800, so 8 waves fit; with 82 it takes 112, and of two 1024-thread
// blocks per CU only one is resident (512^3 walk: 1.07e12 against 1.25e12
// walker-steps/s).
__global__ __launch_bounds__(max_threads_for_k(K)) __attribute__((amdgpu_num_sgpr(80))) void zwalk_kernel(
    const WalkArgs a)
{
    __shared__ double lds[kEchoChunk][kEchoCols];
    __shared__ uint4 tab[TAB == 1 ? kZWideEntries
                                  : (TAB == 3 ? kZFlippedEntries : (MFLAGS ? 8 * kZFlagStride / 16 : (NOFLUX ? 12 : 6)))];
    __shared__ uint4 small[6];
    __shared__ uint2 fix[TAB == 3 ? kZFlippedEntries : (MFLAGS ? 8 * kZFlagStride / 16 : 6)];
    __shared__ __align__(16) uint32_t keys[TAB == 3 ? kZFlagKeyEntries / 4 : (TAB == 2 ? kZKeyEntries / 4 : 1)];
    __shared__ double ldelta[kMaxLabels];
    extern __shared__ uint32_t zlh[];   // EMODE 2, K == 1: per-label hit counts (blockDim x kLhStride)
    const uint64_t tile = tile_of_block(a);
    if (a.tile_map && tile >= a.n_tiles)
        return;  // spare workgroup of the XCD-striped grid (whole block leaves together)
    uint8_t *key_bytes = reinterpret_cast<uint8_t *>(keys);
    if (NOFLUX)
        zbuild_table_noflux(a.zl, tab, SUB ? (uint32_t)a.shift : 0u);
    else if (TAB == 3)
        zbuild_table_flipped(a.zl, tab, fix);
    else if (MFLAGS)
        zbuild_table_flags(a.zl, tab, fix);
    else
        zbuild_table(a.zl, TAB == 1 ? small : tab, fix);
    if (TAB == 3)
        zbuild_flag_key_table(keys);
    if (TAB == 2)
        zbuild_key_table(key_bytes, NOFLUX ? 32u : 16u);
    if (EMODE == 2 && threadIdx.x < kMaxLabels)
        ldelta[threadIdx.x] = (int)threadIdx.x < a.n_labels ? a.label_delta[threadIdx.x] : 1.0;
    __syncthreads();
    if (TAB == 1) {
        zbuild_table_wide(small, tab);
        __syncthreads();
    }
    zwalk_tile<EMODE, K, WRAPFIX, CACHE, TAB, NOFLUX, MFLAGS, 1, false, ADISP, HITS, SUB>(
        a, tile, a.partials ? a.partials + tile : nullptr, a.partial_stride, lds, tab, fix, ldelta, key_bytes,
        EMODE == 2 && K == 1 ? zlh : nullptr);
}

// ONE: ls.k is 1, and only that instance is built.
template <int EMODE, bool WRAPFIX, int CACHE, int TAB, bool NOFLUX = false, bool MFLAGS = false, bool ONE = false>
static hipError_t launch_z(const WalkArgs &a, const LaunchShape &ls, uint32_t blocks, hipStream_t st)
{
    // EMODE 2 with one walker per lane keeps the per-label hit counts in LDS
    const size_t lh_bytes = EMODE == 2 ? (size_t)kLhStride * ls.threads * sizeof(uint32_t) : 0;
    // CPMG and map walks of one walker per lane on images of periods of 128 and
    // more: unbounded moves from address displacements; hits counted only when
    // asked for.  CPMG outside the flag-keyed tables pairs them with masks,
    // which more waves per SIMD outrun: up to kZMaskWalkers.
    if constexpr (EMODE < 2 && CACHE >= 64 && TAB >= 2 && !NOFLUX) {
        const bool few = EMODE == 0 || TAB == 3 || a.n <= kZMaskWalkers;
        if (few && ls.k == 1 && zaddress_displacement_ok(a.zl)) {
            if (EMODE == 0 || a.hits)
                hipLaunchKernelGGL((zwalk_kernel<EMODE, 1, WRAPFIX, CACHE, TAB, NOFLUX, MFLAGS, true>), dim3(blocks),
                                   dim3(ls.threads), 0, st, a);
            else
                hipLaunchKernelGGL((zwalk_kernel<EMODE, 1, WRAPFIX, CACHE, TAB, NOFLUX, MFLAGS, true, EMODE == 0>),
                                   dim3(blocks), dim3(ls.threads), 0, st, a);
            return hipGetLastError();
        }
    }
    if constexpr (ONE) {
        hipLaunchKernelGGL((zwalk_kernel<EMODE, 1, WRAPFIX, CACHE, TAB, NOFLUX, MFLAGS>), dim3(blocks), dim3(ls.threads), lh_bytes, st, a);
        return hipGetLastError();
    }
    switch (ls.k) {
    case 1: hipLaunchKernelGGL((zwalk_kernel<EMODE, 1, WRAPFIX, CACHE, TAB, NOFLUX, MFLAGS>), dim3(blocks), dim3(ls.threads), lh_bytes, st, a); break;
    case 2: hipLaunchKernelGGL((zwalk_kernel<EMODE, 2, WRAPFIX, CACHE, TAB, NOFLUX, MFLAGS>), dim3(blocks), dim3(ls.threads), 0, st, a); break;
    case 4:
        // the flag-keyed tables run in 1024-thread blocks, four walkers per lane in at most 512
        if constexpr (TAB == 3)
            return hipErrorInvalidValue;
        else
            hipLaunchKernelGGL((zwalk_kernel<EMODE, 4, WRAPFIX, CACHE, TAB, NOFLUX, MFLAGS>), dim3(blocks), dim3(ls.threads), 0, st, a);
        break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// Voxel division (a.shift > 0): one walker per lane, whatever ls.k says, and
// the 8-byte chunk, which a sub-voxel step leaves less often.
template <int EMODE, bool WRAPFIX, bool NOFLUX, bool MFLAGS>
static hipError_t launch_z_sub(const WalkArgs &a, const LaunchShape &ls, uint32_t blocks, hipStream_t st)
{
    const size_t lh_bytes = EMODE == 2 ? (size_t)kLhStride * ls.threads * sizeof(uint32_t) : 0;
    constexpr bool ADISP = EMODE < 2 && !NOFLUX;
    if (ADISP && zaddress_displacement_ok(a.zl))
        hipLaunchKernelGGL((zwalk_kernel<EMODE, 1, WRAPFIX, 64, 2, NOFLUX, MFLAGS, ADISP, true, true>),
                           dim3(blocks), dim3(ls.threads), lh_bytes, st, a);
    else
        hipLaunchKernelGGL((zwalk_kernel<EMODE, 1, WRAPFIX, 64, 2, NOFLUX, MFLAGS, false, true, true>), dim3(blocks),
                           dim3(ls.threads), lh_bytes, st, a);
    return hipGetLastError();
}

// Mirror walks with reflection flags (a.zmflags, a.zcache >= 2), instantiated
// apart from the rest (zwalk_mirror.hip): they are the larger half to compile.
template <int EMODE>
hipError_t launch_z_mirror(const WalkArgs &a, const LaunchShape &ls, uint32_t blocks, hipStream_t st);

// a.zcache: 0 no chunk cache; 1 128-bit chunk with word select; 2 and 3 a
// 128-bit chunk with the shift test and the direction drawn one step ahead,
// through the byte-key table (2) or, for power-of-two periods, the wide
// direction table (3; the 6-entry table otherwise); 4 the speculative CPMG
// and map walks; 5 as 2 with a 64-bit (4 x 4 x 4 voxel) chunk, mirror walks with
// reflection flags and other walks of one walker per lane (the rest run 2).
template <int EMODE>
hipError_t launch_z_mode(const WalkArgs &a, const LaunchShape &ls, uint32_t blocks, hipStream_t st)
{
    // a.zcache 4: the speculative CPMG and map walks (one walker per lane);
    // other modes and lane shapes take the pipelined chunk-cache walk
    if (a.zcache == 4 && EMODE < 2 && (ls.k == 1 || a.shift))
        return launch_z_spec(a, EMODE, ls, blocks, st);
    if (a.shift) {
        if (a.znoflux)
            return launch_z_sub<EMODE, false, true, false>(a, ls, blocks, st);
        if (a.zmflags)
            return a.zl.wrapfix ? launch_z_sub<EMODE, true, false, true>(a, ls, blocks, st)
                                : launch_z_sub<EMODE, false, false, true>(a, ls, blocks, st);
        return a.zl.wrapfix ? launch_z_sub<EMODE, true, false, false>(a, ls, blocks, st)
                            : launch_z_sub<EMODE, false, false, false>(a, ls, blocks, st);
    }
    if (a.zcache == 4) {
        WalkArgs b = a;
        b.zcache = 2;
        return launch_z_mode<EMODE>(b, ls, blocks, st);
    }
    if (a.zcache == 5 && ls.k == 1 && !a.zmflags) {   // noflux and periodic, 8-byte chunk cache
        if (a.znoflux)
            return launch_z<EMODE, false, 64, 2, true, false, true>(a, ls, blocks, st);
        return a.zl.wrapfix ? launch_z<EMODE, true, 64, 2, false, false, true>(a, ls, blocks, st)
                            : launch_z<EMODE, false, 64, 2, false, false, true>(a, ls, blocks, st);
    }
    if (a.znoflux)   // noflux on the periodic image: pipelined byte-key walk only
        return a.zcache >= 2 ? launch_z<EMODE, false, 128, 2, true>(a, ls, blocks, st) : hipErrorInvalidValue;
    if (a.zmflags && a.zcache >= 2)   // mirror, walkers folded to the first octant with reflection flags
        return launch_z_mirror<EMODE>(a, ls, blocks, st);
    if (a.zcache == 5) {
        WalkArgs b = a;
        b.zcache = 2;
        return launch_z_mode<EMODE>(b, ls, blocks, st);
    }
    if (a.zl.wrapfix) {
        switch (a.zcache) {
        case 0: return launch_z<EMODE, true, 0, 0>(a, ls, blocks, st);
        case 1: return launch_z<EMODE, true, 1, 0>(a, ls, blocks, st);
        case 2: return launch_z<EMODE, true, 128, 2>(a, ls, blocks, st);
        case 3: return launch_z<EMODE, true, 128, 0>(a, ls, blocks, st);
        default: return hipErrorInvalidValue;
        }
    }
    switch (a.zcache) {
    case 0: return launch_z<EMODE, false, 0, 0>(a, ls, blocks, st);
    case 1: return launch_z<EMODE, false, 1, 0>(a, ls, blocks, st);
    case 2: return launch_z<EMODE, false, 128, 2>(a, ls, blocks, st);
    case 3: return launch_z<EMODE, false, 128, 1>(a, ls, blocks, st);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace rwnmr

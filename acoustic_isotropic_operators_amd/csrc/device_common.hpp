// device_common.hpp -- what the HIP translation units share: the stencil
// constants, the workgroup-to-XCD mapping and the global-memory views.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace aiso {

constexpr int FAT = 5;
constexpr int NT = 256;
// The step kernels address a slice as a 64-bit base plus a 32-bit element
// offset; their launchers refuse larger slices.
constexpr long kMaxSlicePoints = 0x7fffffffL;

__device__ __forceinline__ int imin(int a, int b) { return a < b ? a : b; }

// Linear workgroup ids go round-robin over the 8 XCDs; give each XCD a
// contiguous run of (shot, tile) work so neighbouring tiles share its L2.
__device__ __forceinline__ int xcd_logical(int bid, int gridPadded)
{
    const int per = gridPadded >> 3;
    return (bid & 7) * per + (bid >> 3);
}

// Global-memory views: pointers read from the ShotSlot table are generic to
// the compiler; casting them lets it emit global (not flat) loads and stores
// with a uniform 64-bit base and a 32-bit per-lane offset.
#define GBL __attribute__((address_space(1)))
using gf = GBL float;
using cgf = const GBL float;
__device__ __forceinline__ gf* G(float* p) { return (gf*)p; }
__device__ __forceinline__ cgf* G(const float* p) { return (cgf*)p; }

}  // namespace aiso

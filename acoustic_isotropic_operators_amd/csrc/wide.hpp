// wide.hpp -- 16-byte accesses of the kernels with four z-points per lane.
#pragma once

#include "device_common.hpp"

namespace aiso {

// Four floats at any 4-byte aligned address.
typedef float f4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float f4a __attribute__((ext_vector_type(4)));
using gf4 = GBL f4;
using cgf4 = const GBL f4;

// base + a 32-bit byte offset: one scalar base and one vector register.
__device__ __forceinline__ cgf4* at4(cgf* base, unsigned byteOff) { return (cgf4*)((const GBL char*)base + byteOff); }
__device__ __forceinline__ gf4* at4(gf* base, unsigned byteOff) { return (gf4*)((GBL char*)base + byteOff); }
__device__ __forceinline__ cgf* at1(cgf* base, unsigned byteOff) { return (cgf*)((const GBL char*)base + byteOff); }
__device__ __forceinline__ f4 ld4(cgf* base, unsigned byteOff) { return *at4(base, byteOff); }
__device__ __forceinline__ f4 ld4s(cgf* base, unsigned byteOff, int nt)
{
    return nt ? __builtin_nontemporal_load(at4(base, byteOff)) : *at4(base, byteOff);
}
__device__ __forceinline__ void st4(gf* base, unsigned byteOff, f4 v) { *at4(base, byteOff) = v; }
__device__ __forceinline__ void st4s(gf* base, unsigned byteOff, f4 v, int nt)
{
    if (nt) __builtin_nontemporal_store(v, at4(base, byteOff));
    else *at4(base, byteOff) = v;
}

}  // namespace aiso

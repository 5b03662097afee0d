// What csrc/steps.hip needs of the HIP headers, for a CPU build of its kernels
// (tests/test_steps_schedule.py): a workgroup is a set of fibers of one
// process, and __syncthreads gives the scheduler of fibers.hpp its turn.
#pragma once

#include <algorithm>
#include <cmath>

struct int2 { int x, y; };
struct dim3 {
    unsigned x, y, z;
    dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
using hipError_t = int;
using hipStream_t = void*;
using hipEvent_t = void*;
constexpr hipError_t hipSuccess = 0, hipErrorInvalidValue = 1;
inline hipError_t hipGetLastError() { return hipSuccess; }

#define __global__
#define __device__
#define __shared__ static
#define __launch_bounds__(...)
#undef __forceinline__
#define __forceinline__ inline

extern dim3 threadIdx, blockIdx, gridDim;
void __syncthreads();

#include "fibers.hpp"
#define hipLaunchKernelGGL(kernel, grid, threads, lds, stream, ...) \
    fibers::launch((grid).x, (threads).x, [&] { kernel(__VA_ARGS__); })
#define hipExtLaunchKernelGGL(kernel, grid, threads, lds, stream, e0, e1, flags, ...) \
    hipLaunchKernelGGL(kernel, grid, threads, lds, stream, __VA_ARGS__)

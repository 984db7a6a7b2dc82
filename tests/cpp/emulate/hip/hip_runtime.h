// Stand-in for the HIP runtime header that lets a device source run on the CPU: the threads of a
// block take turns as fibers of one thread (run_blocks, emulate.h), __syncthreads yields to the next
// one, and one array serves as the dynamic LDS of the running block.
#pragma once
#include <cmath>
#include <cstddef>
#include <cstdint>

#define __device__
#define __host__
#define __global__
#define __shared__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n) __attribute__((aligned(n)))

struct float2 { float x, y; };
struct double2 { double x, y; };
struct uint2 { unsigned x, y; };
struct uint4 { unsigned x, y, z, w; };
inline float2 make_float2(float x, float y) { return {x, y}; }
inline double2 make_double2(double x, double y) { return {x, y}; }
struct dim3 {
    unsigned x, y, z;
    dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
extern dim3 threadIdx, blockIdx, blockDim, gridDim;
void emulate_yield();
inline void __syncthreads() { emulate_yield(); }
inline unsigned __umulhi(unsigned a, unsigned b) { return (unsigned)(((unsigned long long)a * b) >> 32); }

using hipError_t = int;
using hipStream_t = void *;
enum : int { hipSuccess = 0, hipErrorInvalidValue = 1 };
using hipEvent_t = void *;

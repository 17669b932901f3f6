// hp_reduce.h -- reductions into the status block shared by the sweep, speed
// and particle kernels.  Atomics on one address are served one at a time,
// about 12 ns each across the XCDs, so a launch of many short waves ends on
// them: a block meets in LDS first, and a maximum is raised only when it
// exceeds the value in memory.  A maximum only grows between its resets (by
// other kernels of the stream), so a stale read costs a needless atomic and
// never a lost one.
#pragma once
#include <hip/hip_runtime.h>

#include "hp_kernels.h"

namespace hp {

// Non-negative doubles order as their bit patterns, with NaN above them all.
__device__ __forceinline__ void raise_velmax(DevStatus* st, unsigned long long bits)
{
    if (bits > __hip_atomic_load(&st->velmax_bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(&st->velmax_bits, bits);
}

// The largest of the per-lane maxima v of a block of at most 256 threads, as
// a bit pattern, valid on thread 0; every thread must call it.
__device__ __forceinline__ unsigned long long block_max_bits(double v)
{
    __shared__ unsigned long long s_max[4];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
    unsigned long long bits = (unsigned long long)__double_as_longlong(v);
    if ((threadIdx.x & 63) == 0) s_max[threadIdx.x >> 6] = bits;
    __syncthreads();
    const int nw = (blockDim.x + 63) >> 6;
    for (int k = 1; k < nw; ++k) bits = max(bits, s_max[k]);
    return bits;
}

}  // namespace hp

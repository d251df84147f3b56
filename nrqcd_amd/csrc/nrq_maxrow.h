// nrq_maxrow.h -- the maximum of a quantity >= 0 over a whole launch, for loops
// whose next launch (and later the host) needs it: a row of 64 slots that the
// blocks raise with atomic maxima (64 slots, so that thousands of blocks do not
// queue at one address) and that any wavefront folds in one load.  The bit
// patterns of non-negative doubles order like unsigned integers, and a maximum
// does not depend on the order of the blocks: the result is deterministic.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nrq {

constexpr int MAXROW = 64; // slots per row, one per lane

__device__ __forceinline__ double lane_max(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
    return v;
}

// Maximum of a row, in every lane (all 64 lanes must call).
__device__ __forceinline__ double row_max(const double *__restrict__ row) { return lane_max(row[threadIdx.x & 63]); }

// Raises the row to at least v >= 0 (one lane per block or wavefront calls); a
// NaN raises nothing, as fmax ignores it everywhere else.
__device__ __forceinline__ void row_raise(double *row, double v)
{
    atomicMax((unsigned long long *)row + blockIdx.x % MAXROW, (unsigned long long)__double_as_longlong(fmax(v, 0.0)));
}

} // namespace nrq

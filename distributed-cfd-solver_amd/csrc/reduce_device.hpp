// Reductions inside a workgroup and the hand-over of their results to the host,
// shared by the kernels that end in sums.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels_linalg.hpp"

namespace cfdg {

__device__ __forceinline__ double wave_sum(double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

// Sums over the workgroup of the first ncomp components, each in a fixed tree
// order (the waves' sums in wave order); sum j valid in thread j.  lds: 5 per wave.
__device__ __forceinline__ double block_sums(const double v[5], int ncomp, double* lds) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int j = 0; j < 5; ++j) {
        if (j >= ncomp) break;
        const double s = wave_sum(v[j]);
        if (lane == 0) lds[wid * 5 + j] = s;
    }
    __syncthreads();
    double s = 0.0;
    if (static_cast<int>(threadIdx.x) < ncomp)
        for (int w = 0; w < static_cast<int>(blockDim.x >> 6); ++w) s += lds[w * 5 + static_cast<int>(threadIdx.x)];
    return s;
}

// Sums of nblocks partial 5-vectors: thread t adds blocks t,
// t + blockDim, ... in order, then the threads' sums as block_sums; sum j in thread j.
// Bound by latency: the components' loads are in flight together and their trees share
// the barriers (one component after the other took 7 us for five components of 1,024
// partials).
__device__ __forceinline__ double sum_partials(int nblocks, int ncomp, const double* partial, double* lds) {
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    for (int b = threadIdx.x; b < nblocks; b += static_cast<int>(blockDim.x))
#pragma unroll
        for (int j = 0; j < 5; ++j)
            if (j < ncomp) acc[j] += partial[b * 5 + j];
    return block_sums(acc, ncomp, lds);
}

// The workgroup's values in host memory are complete: seq becomes visible to the host
// after them.  Every thread of the (single) workgroup calls it.
__device__ __forceinline__ void publish_seq(const Publish& p) {
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(&p.host->seq, p.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace cfdg

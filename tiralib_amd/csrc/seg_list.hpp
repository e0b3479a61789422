// seg_list.hpp -- starts of the runs of a compacted list: exclusive sums of
// per-segment counts in two levels, shared by the listed gathers of the 3D
// learned plate (plate_sparse.hip) and of the 2D search session (vote2.hip).
// After k_seg_scan and k_seg_scan_top, segment i starts at seg_start(cnt, tot, i).
#pragma once
#include <hip/hip_runtime.h>

namespace th {

constexpr unsigned kScanSegs = 1024;  // segments per scan block

// Exclusive sums of 1024 consecutive counts in place, their total to tot[block].
static __global__ __launch_bounds__(256) void k_seg_scan(unsigned* __restrict__ cnt, unsigned n,
                                                         unsigned* __restrict__ tot) {
    __shared__ unsigned s[256];
    const unsigned i0 = blockIdx.x * kScanSegs + threadIdx.x * 4;
    unsigned v[4], sum = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        v[k] = i0 + k < n ? cnt[i0 + k] : 0u;
        sum += v[k];
    }
    s[threadIdx.x] = sum;
    __syncthreads();
    for (int d = 1; d < 256; d <<= 1) {
        const unsigned a = (int)threadIdx.x >= d ? s[threadIdx.x - d] : 0u;
        __syncthreads();
        s[threadIdx.x] += a;
        __syncthreads();
    }
    unsigned run = s[threadIdx.x] - sum;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        if (i0 + k < n) cnt[i0 + k] = run;
        run += v[k];
    }
    if (threadIdx.x == 255) tot[blockIdx.x] = s[255];
}

// Exclusive sums of the block totals (one block); *next (optional) is zeroed.
static __global__ __launch_bounds__(1024) void k_seg_scan_top(unsigned* __restrict__ tot, unsigned n,
                                                              unsigned* __restrict__ next) {
    __shared__ unsigned s[1024];
    unsigned carry = 0;
    for (unsigned b = 0; b < n; b += 1024) {
        const unsigned i = b + threadIdx.x, v = i < n ? tot[i] : 0u;
        s[threadIdx.x] = v;
        __syncthreads();
        for (int d = 1; d < 1024; d <<= 1) {
            const unsigned a = (int)threadIdx.x >= d ? s[threadIdx.x - d] : 0u;
            __syncthreads();
            s[threadIdx.x] += a;
            __syncthreads();
        }
        if (i < n) tot[i] = carry + s[threadIdx.x] - v;
        carry += s[1023];
        __syncthreads();
    }
    if (next && threadIdx.x == 0) *next = 0u;
}

__device__ __forceinline__ unsigned seg_start(const unsigned* __restrict__ cnt, const unsigned* __restrict__ tot,
                                              unsigned seg) {
    return cnt[seg] + tot[seg / kScanSegs];
}

// v of lane j (wave-uniform j), as a scalar.
__device__ __forceinline__ float lane_f(float v, int j) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j));
}

}  // namespace th

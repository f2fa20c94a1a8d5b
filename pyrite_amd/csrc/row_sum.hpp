// row_sum.hpp -- adds the partial rows of a reduction in a fixed order.
#pragma once

#include "hr_common.hpp"

namespace hr {
namespace {

// out[k] += sum_b partial[b][k] over n_rows rows of n values: 16 threads share a
// value, thread g adding rows g, g + 16, ... and the 16 sums then added in
// order, so the result is the same for every launch.  Latency bound: the rows
// sit in the L2, and what counts is how many loads are in flight.  One thread per
// value (in two levels of 64 rows) took 22 us for 1,024 rows of 2,000 values and
// 100 us for the 512 of 16,384 of a coherent field; a bremsstrahlung call got
// 20 us shorter with this, a coherent one with two fields 190 us.
constexpr int kRowLanes = 16;
__global__ void __launch_bounds__(256) row_sum_kernel(const double *__restrict__ partial, int64_t n_rows, int64_t n,
                                                      double *__restrict__ out) {
    __shared__ double s_part[kRowLanes][kRowLanes + 1];
    const int v = threadIdx.x & (kRowLanes - 1), g = threadIdx.x / kRowLanes;
    const int64_t k = (int64_t)blockIdx.x * kRowLanes + v;
    double s = 0.0;
    if (k < n) {
#pragma unroll 8
        for (int64_t b = g; b < n_rows; b += kRowLanes) s += partial[b * n + k];
    }
    s_part[g][v] = s;
    __syncthreads();
    if (g == 0 && k < n) {
#pragma unroll
        for (int i = 1; i < kRowLanes; ++i) s += s_part[i][v];
        out[k] += s;
    }
}

inline hr_status row_sum(const double *partial, int64_t n_rows, int64_t n, double *out, hipStream_t s) {
    const int64_t grid = (n + kRowLanes - 1) / kRowLanes;
    HR_REQUIRE(grid < (1LL << 31), "%lld values exceed one row-sum launch", (long long)n);
    hipLaunchKernelGGL(row_sum_kernel, dim3((unsigned)grid), dim3(256), 0, s, partial, n_rows, n, out);
    HR_CHECK_HIP(hipGetLastError());
    return HR_OK;
}

}  // namespace
}  // namespace hr

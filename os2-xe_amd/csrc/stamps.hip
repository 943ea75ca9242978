// stamps.hip - stage times of a region of many launches.
#include "kernels.hpp"

namespace oz2 {
namespace k {
namespace {

// one thread a launch; then one wave a stage adds them up
__global__ void __launch_bounds__(kStampSlots) sum_stamps_kernel(const uint64_t* __restrict__ ts, StampStages stages, uint32_t n,
                                                                 double* __restrict__ sums, bool first) {
    __shared__ double part[kStageSums][kStampSlots];
    const uint32_t i = threadIdx.x;
    double t[kStageSums] = {};
    if (i < n) add_stage_ticks(ts + static_cast<size_t>(i) * kStampWords, stages.s[i], t);
    for (int g = 0; g < kStageSums; ++g) part[g][i] = t[g];
    __syncthreads();
    static_assert(kStampSlots == 64 * kStageSums);
    const uint32_t g = i >> 6, lane = i & 63;
    double sum = 0.0;
    for (uint32_t j = lane; j < kStampSlots; j += 64) sum += part[g][j];
    for (int o = 32; o >= 1; o >>= 1) sum += __shfl_xor(sum, o, 64);
    if (lane == 0) sums[g] = first ? sum : sums[g] + sum;
}

}  // namespace

void sum_stamps(hipStream_t st, const uint64_t* ts, const StampStages& stages, uint32_t n, double* sums, bool first) {
    hipLaunchKernelGGL(sum_stamps_kernel, dim3(1), dim3(kStampSlots), 0, st, ts, stages, n, sums, first);
}

}  // namespace k
}  // namespace oz2

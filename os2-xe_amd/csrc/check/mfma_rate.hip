// mfma_rate.hip - sustained INT8 MFMA rate of the GPU with no memory traffic: every
// wave runs 16 independent v_mfma_i32_32x32x32_i8 accumulator chains held in
// registers (the instruction and wave tile of the library's INT8 GEMM), one wave per
// SIMD, and stores one word per lane at the end.  The rate depends on the operands'
// data: with a few constant words the clock stays near its peak, with random words,
// four of A by four of B as in the GEMM's wave tile, the power limit lowers it.
// Measurement harness only, not part of liboz2.so; the rate on random words is the
// practical MFMA ceiling that the GEMM's rate is read against (bench.py --mfma-rate).
#include <hip/hip_runtime.h>

#include <cstdint>

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

__device__ v4i random_words(uint32_t x) {  // any mixing of the bits does
    v4i r;
    for (int i = 0; i < 4; ++i) {
        x = (x ^ (x >> 16)) * 0x7FEB352Du;
        x = (x ^ (x >> 15)) * 0x846CA68Bu;
        x ^= x >> 16;
        r[i] = static_cast<int>(x);
        x += 0x9E3779B9u;
    }
    return r;
}

template <bool RANDOM>
__global__ void __launch_bounds__(256, 1) mfma_loop_kernel(int iters, int* __restrict__ out) {
    v4i a[4], b[4];
    for (int i = 0; i < 4; ++i) {
        const uint32_t seed = (blockIdx.x * 256 + threadIdx.x) * 8 + i;
        a[i] = RANDOM ? random_words(seed) : v4i{static_cast<int>(threadIdx.x), 3, 5, 7};
        b[i] = RANDOM ? random_words(seed + 4) : v4i{1, static_cast<int>(blockIdx.x), 2, 9};
    }
    v16i acc[16];
#pragma unroll
    for (int j = 0; j < 16; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[j][v] = 0;
    for (int it = 0; it < iters; ++it) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {  // columns back and forth under the rows, as in the GEMM
            const int r = j / 4, c = r % 2 ? 3 - j % 4 : j % 4;
            acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[r], b[c], acc[j], 0, 0, 0);
        }
    }
    int s = 0;
#pragma unroll
    for (int j = 0; j < 16; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) s += acc[j][v];
    out[static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x] = s;
}

}  // namespace

// blocks workgroups of 256 threads, each running iters x 16 MFMAs per wave (4 waves):
// 2 * 32768 * 16 * iters * 4 * blocks int8 operations; out needs blocks * 256 ints
static int mfma_rate(void (*kernel)(int, int*), void* stream, int blocks, int iters, int* out) {
    if (blocks <= 0 || iters <= 0) return 1;
    if (!out) return 1;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, static_cast<hipStream_t>(stream), iters, out);
    return hipGetLastError() == hipSuccess ? 0 : 2;
}
extern "C" int oz2chk_mfma_rate(void* stream, int blocks, int iters, int* out) {
    return mfma_rate(mfma_loop_kernel<false>, stream, blocks, iters, out);
}
// the same with random operands
extern "C" int oz2chk_mfma_rate_random(void* stream, int blocks, int iters, int* out) {
    return mfma_rate(mfma_loop_kernel<true>, stream, blocks, iters, out);
}

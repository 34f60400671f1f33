// Re-codes A for the tile kernel on 6-bit floats, and adds its rows up.
#pragma once
#include "qm_fp6.hpp"

namespace qm {

struct Expand6Args {
    const uint8_t *A;  // [M, K/2] packed s4, rows 16-byte aligned, K a multiple of 32 and at least 256
    uint8_t *codes;
    int *sums;
    int M, K, kt, groups;
};

// One workgroup re-codes 16 rows over FP6_PART_STEPS K-steps (blockIdx.y), eight waves of two K-steps at a
// time: 128 bytes of every row, whole lines.  Two K-steps that a row does not fill are its last 128
// bytes, as the GEMM loads them of B, with zeros where the steps before have been.
__global__ void __launch_bounds__(512) expand_a6_kernel(const Expand6Args q)
{
    __shared__ int red[8][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const int half = blockIdx.x, row = half * 16 + r, Kb = q.K >> 1;
    const uint8_t *src = q.A + (size_t)min(row, q.M - 1) * Kb + 16 * g;
    uint8_t *out = q.codes + (size_t)(half >> 1) * q.kt * FP6_GROUP_BYTES;
    constexpr int PAIRS = FP6_PART_STEPS / 16;  // per wave
    v4i v[PAIRS][2];
#pragma unroll
    for (int t = 0; t < PAIRS; ++t) {
        const int step = blockIdx.y * FP6_PART_STEPS + 2 * (wave + 8 * t), at = min(step * 64, Kb - 128);
#pragma unroll
        for (int u = 0; u < 2; ++u) v[t][u] = *reinterpret_cast<const v4i *>(src + at + 64 * u);
    }
    int sum = 0;
#pragma unroll
    for (int t = 0; t < PAIRS; ++t) {
        const int step = blockIdx.y * FP6_PART_STEPS + 2 * (wave + 8 * t), at = min(step * 64, Kb - 128);
        if (step >= q.kt) break;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            v4i w = v[t][u];
            if (row >= q.M || at + 64 * u + 16 * g < step * 64) w = v4i{0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 4; ++e) sum = __builtin_amdgcn_sdot8(w[e], 0x11111111, sum, false);
            uint32_t lo[3], hi[3];
            fp6_signed((uint32_t)w.x, (uint32_t)w.y, lo);
            fp6_signed((uint32_t)w.z, (uint32_t)w.w, hi);
            uint8_t *o = out + (size_t)(step + u) * FP6_GROUP_BYTES;
            *reinterpret_cast<v4i *>(o + (half & 1) * 1024 + lane * 16) = v4i{(int)lo[0], (int)lo[1], (int)lo[2], (int)hi[0]};
            *reinterpret_cast<v2i *>(o + 2048 + (half & 1) * 512 + lane * 8) = v2i{(int)hi[1], (int)hi[2]};
        }
    }
    sum += __shfl_xor(sum, 16);
    sum += __shfl_xor(sum, 32);
    if (lane < 16) red[wave][lane] = sum;
    __syncthreads();
    if (threadIdx.x < 16) {
        int total = 0;
#pragma unroll
        for (int w = 0; w < 8; ++w) total += red[w][threadIdx.x];
        q.sums[((size_t)blockIdx.y * q.groups * 2 + half) * 16 + threadIdx.x] = total;
    }
}

}  // namespace qm

// Re-codes A for the tile kernel on 6-bit floats, and adds its rows up; or quantises it straight to those codes.
#pragma once
#include "qm_aux.hpp"
#include "qm_fp6.hpp"

namespace qm {

struct Expand6Args {
    const uint8_t *A;  // [M, K/2] packed s4; rows 16-byte aligned and K a multiple of 32, unless ANY
    uint8_t *codes;
    int *sums;
    int M, K, kt, groups;
    // ANY only: B [N, K/2], and its copy with rows of Kp / 2 bytes, Kp a multiple of 128
    const uint8_t *B;
    v4i *b_copy;
    int N, Kp;
};

// 16 bytes of a row of Kb from byte `at` on, zeros past its end
__device__ __forceinline__ v4i row_piece(const uint8_t *row, const int at, const int Kb)
{
    const int left = Kb - at;  // bytes of the row from there on
    v4i v = *reinterpret_cast<const v4i_any_aligned *>(row + min(at, Kb - 16));
    if (left < 16) {
        // the row's last 16 bytes: the wanted ones are its last `left`
        const int down = 8 * (16 - max(left, 0));
        uint64_t lo = (uint32_t)v.x | (uint64_t)(uint32_t)v.y << 32, hi = (uint32_t)v.z | (uint64_t)(uint32_t)v.w << 32;
        if (down >= 64) {
            lo = down < 128 ? hi >> (down - 64) : 0;
            hi = 0;
        } else {
            lo = lo >> down | hi << (64 - down);
            hi >>= down;
        }
        v = v4i{(int)lo, (int)(lo >> 32), (int)hi, (int)(hi >> 32)};
    }
    return v;
}

// One workgroup re-codes 16 rows over FP6_PART_STEPS K-steps (blockIdx.y), eight waves of two K-steps at a
// time: 128 bytes of every row, whole lines.  Two K-steps that a row does not fill are its last 128
// bytes, as the GEMM loads them of B, with zeros where the steps before have been.
// ANY: rows of any K and at any address, as if padded with zeros to Kp; the workgroups beyond A's (blockIdx.y past the
// parts) copy B with its rows padded, one 16-byte piece per thread, in the same launch.
template <bool ANY>
__global__ void __launch_bounds__(512) expand_a6_kernel(const Expand6Args q)
{
    __shared__ int red[8][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const int Kb = q.K >> 1;
    if constexpr (ANY) {
        const int parts = (q.kt + FP6_PART_STEPS - 1) / FP6_PART_STEPS;
        if ((int)blockIdx.y >= parts) {
            const uint32_t per_row = (uint32_t)q.Kp >> 5, piece = ((blockIdx.y - parts) * gridDim.x + blockIdx.x) * 512u + threadIdx.x;  // (below 2^28)
            const uint32_t n = piece / per_row;
            if (n < (uint32_t)q.N) q.b_copy[piece] = row_piece(q.B + (size_t)n * Kb, 16 * (int)(piece - n * per_row), Kb);
            return;
        }
    }
    const int row_bytes = ANY ? q.Kp >> 1 : Kb;
    const int half = blockIdx.x, row = half * 16 + r;
    const uint8_t *src = q.A + (size_t)min(row, q.M - 1) * Kb;
    uint8_t *out = q.codes + (size_t)(half >> 1) * q.kt * FP6_GROUP_BYTES;
    constexpr int PAIRS = FP6_PART_STEPS / 16;  // per wave
    v4i v[PAIRS][2];
#pragma unroll
    for (int t = 0; t < PAIRS; ++t) {
        const int step = blockIdx.y * FP6_PART_STEPS + 2 * (wave + 8 * t), at = min(step * 64, row_bytes - 128);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if constexpr (ANY) v[t][u] = row_piece(src, at + 64 * u + 16 * g, Kb);
            else v[t][u] = *reinterpret_cast<const v4i *>(src + at + 64 * u + 16 * g);
        }
    }
    int sum = 0;
#pragma unroll
    for (int t = 0; t < PAIRS; ++t) {
        const int step = blockIdx.y * FP6_PART_STEPS + 2 * (wave + 8 * t), at = min(step * 64, row_bytes - 128);
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

struct Quant6Args {
    const uint8_t *x;  // [M, K] fp16 / bf16 / fp32, K a multiple of 32 and at least 256
    uint8_t *codes;
    int *sums;         // (one part)
    float *scales;
    int M, K, kt;
};

// The rows of x quantised by the rule of quantize_pack_kernel, with the same arithmetic, and written as 6-bit codes: the linear
// layer's activations on their way to the tile kernel, without the packed rows in between and the launch that re-codes
// them.  Eight rows per workgroup, a wave on each, NC chunks of eight elements per lane (k <= 512 NC) in registers between
// the maximum and the quantisation; the nibbles meet in the LDS, so that eight rows' codes leave as whole 128-byte lines.
constexpr int QUANT6_ROWS = 8, QUANT6_THREADS = 64 * QUANT6_ROWS;
inline int quant6_lds_bytes(int k) { return QUANT6_ROWS * (k / 2 + 16); }  // rows 16 bytes apart in banks
template <int IN, int NC>
__global__ void __launch_bounds__(QUANT6_THREADS, 2) quantize_a6_kernel(const Quant6Args q)
{
    extern __shared__ __align__(16) uint8_t nibbles[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = blockIdx.x * QUANT6_ROWS + wave, Kb = q.K >> 1, pitch = Kb + 16, nchunks = q.K >> 3;
    const uint8_t *src = q.x + (size_t)min(row, q.M - 1) * q.K * QuantIn<IN>::BYTES;
    Chunk8<IN> v[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) v[i].load(src + (size_t)min(lane + i * 64, nchunks - 1) * 8 * QuantIn<IN>::BYTES);
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < NC; ++i) amax = v[i].amax(amax);
    amax = row_max<1>(amax, nullptr);
    const float inv = amax > 0.0f ? 7.0f / amax : 0.0f;
    int sum = 0;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        const int c = lane + i * 64;
        // (the elements as loaded: widened for the maximum, the compiler would keep all of them as floats)
#pragma unroll
        for (int w = 0; w < QuantIn<IN>::WORDS / 4; ++w) asm volatile("" : "+v"(v[i].w[w]));
        const uint32_t n8 = quant8(v[i], inv);
        if (c < nchunks) {
            sum = __builtin_amdgcn_sdot8((int)n8, 0x11111111, sum, false);
            *reinterpret_cast<uint32_t *>(nibbles + wave * pitch + 4 * c) = n8;
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off);
    if (lane == 0) {
        q.sums[row] = sum;  // (of the last group's rows beyond M too: nobody reads what comes of them)
        if (row < q.M) q.scales[row] = amax / 7.0f;
    }
    __syncthreads();
    // rows 8 (b & 3) .. of group b >> 2: as expand_a6_kernel writes them
    const int in_group = (blockIdx.x & 3) * QUANT6_ROWS, half = in_group >> 4;
    uint8_t *out = q.codes + (size_t)(blockIdx.x >> 2) * q.kt * FP6_GROUP_BYTES;
    for (int u = threadIdx.x; u < q.kt * 32; u += QUANT6_THREADS) {
        const int r8 = u & 7, g = (u >> 3) & 3, step = u >> 5, pair = (step & ~1) * 64;
        const int at = min(pair, Kb - 128) + 64 * (step & 1) + 16 * g, to = (in_group & 15) + r8 + 16 * g;
        v4i w = *reinterpret_cast<const v4i *>(nibbles + r8 * pitch + at);
        if (at < pair) w = v4i{0, 0, 0, 0};
        uint32_t lo[3], hi[3];
        fp6_signed((uint32_t)w.x, (uint32_t)w.y, lo);
        fp6_signed((uint32_t)w.z, (uint32_t)w.w, hi);
        uint8_t *o = out + (size_t)step * FP6_GROUP_BYTES;
        *reinterpret_cast<v4i *>(o + half * 1024 + to * 16) = v4i{(int)lo[0], (int)lo[1], (int)lo[2], (int)hi[0]};
        *reinterpret_cast<v2i *>(o + 2048 + half * 512 + to * 8) = v2i{(int)hi[1], (int)hi[2]};
    }
}

template <int IN, int NC>
static hipError_t launch_quantize_a6(const Quant6Args &q, int groups, hipStream_t s)
{
    quantize_a6_kernel<IN, NC><<<dim3(groups * 32 / QUANT6_ROWS), dim3(QUANT6_THREADS), quant6_lds_bytes(q.K), s>>>(q);
    return hipGetLastError();
}
// The K it holds: 64 KiB of LDS, and for fp32 128 registers of one wave per row.
inline bool quant6_fits(int k, int in) { return quant6_lds_bytes(k) <= 64 * 1024 && (in != QM_IN_F32 || k <= 8192); }
template <int IN>
static hipError_t launch_quantize_a6(const Quant6Args &q, int groups, hipStream_t s)
{
    if (q.K <= 2048) return launch_quantize_a6<IN, 4>(q, groups, s);
    if (q.K <= 4096) return launch_quantize_a6<IN, 8>(q, groups, s);
    if (q.K <= 8192) return launch_quantize_a6<IN, 16>(q, groups, s);
    if constexpr (IN != QM_IN_F32) return launch_quantize_a6<IN, 32>(q, groups, s);
    return hipErrorInvalidValue;
}

}  // namespace qm

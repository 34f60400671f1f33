// Re-codes A for the tile kernel on 6-bit floats, and adds its rows up; or quantises it straight to those codes.
#pragma once
#include "qm_aux.hpp"
#include "qm_fp6.hpp"

namespace qm {

struct Expand6Args {
    const uint8_t *A;  // [M, K/2] packed s4; rows 16-byte aligned and K a multiple of 32, unless ANY
    uint8_t *codes;
    int *sums;
    int M, K, kt, groups, parts;
    // ANY only: B [N, K/2], and its copy with rows of Kp / 2 bytes, Kp a multiple of 128
    const uint8_t *B;
    v4i *b_copy;
    int N, Kp;
};

// 16 bytes of a row of Kb from byte `at` on, zeros past its end.  Loaded by row_load -- SHIFT: rows that do not lie on multiples of four --
// and put right once it is there.
template <bool SHIFT>
using RowPiece = std::conditional_t<SHIFT, Shifted16, v4i>;
template <bool SHIFT>
__device__ __forceinline__ void row_load(RowPiece<SHIFT> &v, const DwordSpan &s, const uint32_t row, const int at, const int Kb)
{
    const uint32_t from = row * (uint32_t)Kb + (uint32_t)min(at, Kb - 16);
    if constexpr (SHIFT) v.load(s, from);
    else v = *reinterpret_cast<const v4i_any_aligned *>(s.base + (s.lead + from));
}
template <bool SHIFT>
__device__ __forceinline__ v4i row_value(const RowPiece<SHIFT> &piece, const int at, const int Kb)
{
    const int left = Kb - at;  // bytes of the row from there on
    v4i v;
    if constexpr (SHIFT) v = piece.value();
    else v = piece;
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

// The rows of a workgroup: half of them from r0 on and the other half 16 further in a group of 32, both halves of every 16 bytes of codes that they
// share: of eight rows 64 contiguous bytes of codes at a time, of sixteen 128, whole lines.  (Eight: workgroups of a group, which share 128-byte lines of codes, on
// one XCD: 8192 x 8192 16.9 us, 2048 x 11008 6.5, against 14.8 and 6.0 with neighbours of any kind.)
// Eight fill the device where there is little to do; where the codes do not stay in the L2s with what else is there, half lines leave them twice: 11008 x
// 8192 traced in front of its GEMM 23.6 us by sixteen neighbouring rows, 34.0 by eight, and the whole product on 4096 columns, us, 191.7, 198.1, 189.8 by sixteen
// as here.  The whole product over 686 sizes, by eight / by sixteen over sixteen neighbouring ones: 0.961 / 0.971 below 4 million
// elements of A, 0.978 / 0.983 to 32 million, 0.983 / 0.978 beyond.
constexpr int CODE_ROWS = 8;
inline int expand_rows(int m, int k) { return (long long)m * k >= 32000000 ? 16 : 8; }
template <int ROWS>
__device__ __forceinline__ void code_rows(const int block, int &group, int &r0)
{
    group = block / (32 / ROWS);
    r0 = (block & (32 / ROWS - 1)) * (ROWS / 2);
}

// One workgroup re-codes ROWS rows over FP6_PART_STEPS K-steps, eight waves of two K-steps at a time: 128 bytes of every row,
// whole lines.  Two K-steps that a row does not fill are its last 128
// bytes, as the GEMM loads them of B, with zeros where the steps before have been.
// ANY: rows of any K and at any address, as if padded with zeros to Kp; the workgroups beyond A's
// copy B with its rows padded, one 16-byte piece per thread, in the same launch.
// Bound: HBM on large operands, the launch and one round trip on small ones.  us in a graph, by sixteen
// neighbouring rows to a workgroup / by eight as here: 512 x 8192 3.9 / 3.2, 1536 x 4096 4.1 / 3.4, 4096 x 4096 5.8 / 5.7, 8192 x 8192 17.0 / 14.8 (5.7 TB/s).
// SHIFT (rows of A off the multiples of four): with B's copy 1531 x 3307 x 4100 6.8 -> 5.0, the whole product 35.6 -> 32.7 with A's new split.
constexpr int EXPAND6_THREADS = 512;
template <bool ANY, bool SHIFT, int ROWS>
__global__ void __launch_bounds__(EXPAND6_THREADS) expand_a6_kernel(const Expand6Args q)
{
    constexpr int WAVES = EXPAND6_THREADS / 64, PAIRS = FP6_PART_STEPS / 2 / WAVES;  // (pairs of K-steps: per wave)
    constexpr int HALF = ROWS / 2, U = ROWS / 8;  // rows of a fragment, K-steps of a pair that a lane has
    __shared__ int red[WAVES][ROWS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int Kb = q.K >> 1;
    const unsigned blocks = (unsigned)q.groups * (32 / ROWS);
    const int part = blockIdx.x / blocks;
    if constexpr (ANY) {
        if (part >= q.parts) {
            const uint32_t per_row = (uint32_t)q.Kp >> 5, piece = (blockIdx.x - q.parts * blocks) * (uint32_t)EXPAND6_THREADS + threadIdx.x;  // (below 2^28 and a workgroup)
            const uint32_t n = piece / per_row;
            if (n < (uint32_t)q.N) {
                const int at = 16 * (int)(piece - n * per_row);
                // (one load per thread, as it is also where that is four accesses: shifted dwords are no faster here)
                const v4i w = *reinterpret_cast<const v4i_any_aligned *>(q.B + (n * (uint32_t)Kb + (uint32_t)min(at, Kb - 16)));
                q.b_copy[piece] = row_value<false>(w, at, Kb);
            }
            return;
        }
    }
    int group, r0;
    code_rows<ROWS>(blockIdx.x - part * blocks, group, r0);
    // lane: row, 16 bytes of a K-step, step of the two
    const int h = (lane / HALF) & 1, r = r0 + (lane & (HALF - 1)), g = (lane / ROWS) & 3;
    const auto step_of = [&](int u) { return U == 2 ? u : lane >> 5; };
    const int row = group * 32 + h * 16 + r, row_bytes = ANY ? q.Kp >> 1 : Kb;
    const DwordSpan span = dword_span(q.A, (uint32_t)q.M * (uint32_t)Kb);
    RowPiece<SHIFT> v[PAIRS][U];
#pragma unroll
    for (int t = 0; t < PAIRS; ++t)
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int at = min((part * FP6_PART_STEPS + 2 * (wave + WAVES * t)) * 64, row_bytes - 128) + 64 * step_of(u) + 16 * g;
            if constexpr (ANY) row_load<SHIFT>(v[t][u], span, min(row, q.M - 1), at, Kb);
            else v[t][u] = *reinterpret_cast<const v4i *>(q.A + (size_t)min(row, q.M - 1) * Kb + at);
        }
    int sum = 0;
#pragma unroll
    for (int t = 0; t < PAIRS; ++t) {
        const int step = part * FP6_PART_STEPS + 2 * (wave + WAVES * t);
        if (step >= q.kt) break;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int at = min(step * 64, row_bytes - 128) + 64 * step_of(u) + 16 * g;
            v4i w;
            if constexpr (ANY) w = row_value<SHIFT>(v[t][u], at, Kb);
            else w = v[t][u];
            if (row >= q.M || at < step * 64) w = v4i{0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 4; ++e) sum = __builtin_amdgcn_sdot8(w[e], 0x11111111, sum, false);
            uint32_t f[6];
            fp6_fragment(w, f);
            uint8_t *const o = q.codes + ((size_t)group * q.kt + step + step_of(u)) * FP6_GROUP_BYTES + (r + 16 * g) * 16;
            const v4i four = h == 0 ? v4i{(int)f[0], (int)f[1], (int)f[2], (int)f[3]} : v4i{(int)f[2], (int)f[3], (int)f[4], (int)f[5]};
            const v2i two = h == 0 ? v2i{(int)f[4], (int)f[5]} : v2i{(int)f[0], (int)f[1]};
            *reinterpret_cast<v4i *>(o + h * 2048) = four;
            *reinterpret_cast<v2i *>(o + 1024 + h * 8) = two;
        }
    }
#pragma unroll
    for (int apart = ROWS; apart < 64; apart <<= 1) sum += __shfl_xor(sum, apart);
    if (lane < ROWS) red[wave][lane] = sum;
    __syncthreads();
    if (threadIdx.x < ROWS) {
        int total = 0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) total += red[w][threadIdx.x];
        q.sums[((size_t)part * q.groups + group) * 32 + h * 16 + r] = total;
    }
}

// the codes of a lane of a pair of fragments, at its place in the first of the three pieces
__device__ __forceinline__ void put_pair(uint8_t *at, const uint32_t (&f)[2][6])
{
    v4i *const o = reinterpret_cast<v4i *>(at);
    o[0] = v4i{(int)f[0][0], (int)f[0][1], (int)f[0][2], (int)f[0][3]};
    o[64] = v4i{(int)f[0][4], (int)f[0][5], (int)f[1][0], (int)f[1][1]};
    o[128] = v4i{(int)f[1][2], (int)f[1][3], (int)f[1][4], (int)f[1][5]};
}

struct Quant6Args {
    const uint8_t *x;  // [M, K] fp16 / bf16 / fp32, K a multiple of 32 and at least 256
    uint8_t *codes;
    int *sums;         // (one part)
    float *scales;
    int M, K, kt, groups;
};

// The rows of x quantised by the rule of quantize_pack_kernel, with the same arithmetic, and written as 6-bit codes: the linear
// layer's activations on their way to the tile kernel, without the packed rows in between and the launch that re-codes
// them.  Eight rows per workgroup, a wave on each, NC chunks of eight elements per lane (k <= 512 NC) in registers between
// the maximum and the quantisation; the nibbles meet in the LDS, so that their
// codes leave 64 contiguous bytes at a time.
constexpr int QUANT6_ROWS = CODE_ROWS, QUANT6_THREADS = 64 * QUANT6_ROWS;
inline int quant6_lds_bytes(int k) { return QUANT6_ROWS * (k / 2 + 16); }  // rows 16 bytes apart in banks
template <int IN, int NC>
__global__ void __launch_bounds__(QUANT6_THREADS, 2) quantize_a6_kernel(const Quant6Args q)
{
    extern __shared__ __align__(16) uint8_t nibbles[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int group, r0;
    code_rows<CODE_ROWS>(blockIdx.x, group, r0);
    const int row = group * 32 + r0 + (wave & 3) + (wave >> 2) * 16, Kb = q.K >> 1, pitch = Kb + 16, nchunks = q.K >> 3;
    const uint8_t *src = q.x + (size_t)min(row, q.M - 1) * q.K * QuantIn<IN>::BYTES;
    Chunk8<IN> v[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) v[i].load(src + (size_t)min(lane + i * 64, nchunks - 1) * 8 * QuantIn<IN>::BYTES);
    bool plain;
    const float amax = row_max<1>(chunks_amax(v, plain), nullptr);
    const float inv = amax > 0.0f ? 7.0f / amax : 0.0f;
    int sum = 0;
    quantise_chunks<IN>(plain, amax, inv, [&](auto quant) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int c = lane + i * 64;
            // (the elements as loaded: widened for the maximum, the compiler would keep all of them as floats)
#pragma unroll
            for (int w = 0; w < QuantIn<IN>::WORDS / 4; ++w) asm volatile("" : "+v"(v[i].w[w]));
            const uint32_t n8 = quant(v[i]);
            if (c < nchunks) {
                sum = __builtin_amdgcn_sdot8((int)n8, 0x11111111, sum, false);
                *reinterpret_cast<uint32_t *>(nibbles + wave * pitch + 4 * c) = n8;
            }
        }
    });
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off);
    if (lane == 0) {
        q.sums[row] = sum;  // (of the last group's rows beyond M too: nobody reads what comes of them)
        if (row < q.M) q.scales[row] = amax / 7.0f;
    }
    __syncthreads();
    uint8_t *const out = q.codes + (size_t)group * q.kt * FP6_GROUP_BYTES;
    for (int u = threadIdx.x; u < q.kt * 16; u += QUANT6_THREADS) {
        // (eight lanes together: four rows, 16 bytes apart in banks, of two steps, 64 bytes apart)
        const int r4 = u & 3, g = (u >> 3) & 3, step = (u >> 5) * 2 + ((u >> 2) & 1), pair = (step & ~1) * 64;
        const int at = min(pair, Kb - 128) + 64 * (step & 1) + 16 * g;
        uint32_t f[2][6];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            v4i w = *reinterpret_cast<const v4i *>(nibbles + (h * 4 + r4) * pitch + at);
            if (at < pair) w = v4i{0, 0, 0, 0};
            fp6_fragment(w, f[h]);
        }
        put_pair(out + (size_t)step * FP6_GROUP_BYTES + (r0 + r4 + 16 * g) * 16, f);
    }
}

template <int IN, int NC>
static hipError_t launch_quantize_a6_rows(const Quant6Args &q, hipStream_t s)
{
    return enqueue(&quantize_a6_kernel<IN, NC>, dim3(q.groups * (32 / CODE_ROWS)), dim3(QUANT6_THREADS), quant6_lds_bytes(q.K), s, q);
}
// The K it holds: 64 KiB of LDS, and for fp32 128 registers of one wave per row.
inline bool quant6_fits(int k, int in) { return quant6_lds_bytes(k) <= 64 * 1024 && (in != QM_IN_F32 || k <= 8192); }
template <int IN>
static hipError_t launch_quantize_a6(const Quant6Args &q, hipStream_t s)
{
    if (q.K <= 2048) return launch_quantize_a6_rows<IN, 4>(q, s);
    if (q.K <= 4096) return launch_quantize_a6_rows<IN, 8>(q, s);
    if (q.K <= 8192) return launch_quantize_a6_rows<IN, 16>(q, s);
    if constexpr (IN != QM_IN_F32) return launch_quantize_a6_rows<IN, 32>(q, s);
    return hipErrorInvalidValue;
}

}  // namespace qm

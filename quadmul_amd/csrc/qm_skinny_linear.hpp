// The int4 linear layer for 3 to 16 rows of 16-bit activations, in one launch.
#pragma once
#include "qm_aux.hpp"
#include "qm_launch.hpp"
#include "qm_skinny_dma.hpp"

namespace qm {

// gemm_skinny_stream_dma_kernel with the quantisation of its rows in front: every workgroup quantises all of x by itself, with the
// arithmetic of quantize_pack_kernel, into the LDS, from where its waves take their fragments of A, and then walks over its blocks of sixteen
// columns.  A row belongs to one wave (16 rows), two (8) or four (4), which hold it in registers between the maximum and the
// quantisation; the first loads of B go out as soon as x is there, ahead of the arithmetic.
// Bound: the launch, and on more rows or a longer K the vector arithmetic: 256 workgroups each quantise all of x, 0.5 us for 4 x 4096
// elements and 2 for 16 x 4096, where the quantisation as a launch of its own takes 2.1 and the gap between dependent kernels.
template <int IN_, int ROWS_, int NC_, int R_, int D_>
struct SkinnyLinearCfg {
    static constexpr int IN = IN_, ROWS = ROWS_, NC = NC_, R = R_, D = D_;  // NC chunks of eight elements per lane and row, R runs of 256 nibbles per wave, D of them of B in flight
    static constexpr int NW = 16, THREADS = 64 * NW, BN = 16, WPR = NW / ROWS;
    static constexpr int MAX_K = NW * R * 256 < NC * WPR * 512 ? NW * R * 256 : NC * WPR * 512;
    static constexpr int UNIT_BYTES = 2048, RUN_BYTES = ROWS * 128;  // of a run of B, and of A
    static constexpr int RING_BYTES = NW * D * UNIT_BYTES, RED_BYTES = 2 * 1024;
    static int lds_bytes(int k) { return RING_BYTES + RED_BYTES + (k / 2 + 127) / 128 * RUN_BYTES; }
    static_assert(ROWS == 4 || ROWS == 8 || ROWS == 16, "rows of a fragment");
    static_assert(RING_BYTES + RED_BYTES + NW * R * RUN_BYTES <= 159 * 1024, "LDS budget of a gfx950 CU");
};

template <class Cfg>
__global__ void __launch_bounds__(Cfg::THREADS)
skinny_linear_kernel(const uint8_t *x, const uint8_t *B, int32_t *Y, const int grid_rows_out, const int N, const int K, const float *col_scale, const uint16_t *bias)
{
    // (grid_rows_out as in gemm_skinny_stream_dma_kernel)
    GemmArgs p{nullptr, B, Y, (grid_rows_out >> 2) & 63, N, K};
    p.col_scale = col_scale;
    p.bias = bias;
    p.out = grid_rows_out & 3;
    constexpr int IN = Cfg::IN, ROWS = Cfg::ROWS, NC = Cfg::NC, R = Cfg::R, D = Cfg::D, NW = Cfg::NW, WPR = Cfg::WPR, LPU = 2;
    extern __shared__ __align__(16) uint8_t smem[];
    int32_t *const red = reinterpret_cast<int32_t *>(smem + Cfg::RING_BYTES);  // [2][register][lane]
    uint8_t *const a_rows = smem + Cfg::RING_BYTES + Cfg::RED_BYTES;           // [run][row][128 bytes], 16-byte pieces permuted as B's
    __shared__ float wave_max[NW], row_scale[ROWS];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int Kb = p.K >> 1, nruns = (Kb + 127) >> 7, xchunks = p.K >> 3;
    const int cnt = wave < nruns ? (nruns - wave + NW - 1) / NW : 0;  // this wave's runs: wave, wave + NW, ... (at most R)

    // ---- x ----
    const int row = wave / WPR, c0 = lane + 64 * (wave % WPR);
    Chunk8<IN> v[NC];
    float amax = 0.0f;
    bool plain = true;
    if (row < p.M) {
        const uint8_t *const xr = x + (size_t)row * p.K * QuantIn<IN>::BYTES;
#pragma unroll
        for (int t = 0; t < NC; ++t) v[t].load(xr + (uint32_t)min(c0 + t * 64 * WPR, xchunks - 1) * (8 * QuantIn<IN>::BYTES));
        amax = chunks_amax(v, plain);
    }
    asm volatile("" : "+v"(amax));  // (x is there: a wait for it further down would be one for B too, whose loads the compiler does not see)

    // ---- B: as in gemm_skinny_stream_dma_kernel ----
    const int row8 = lane >> 3, pos = lane & 7;
    uint32_t piece_off[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) piece_off[h] = (uint32_t)((pos ^ (((8 * h + row8) >> 1) & 7)) * 16);
    const uint32_t last16 = (uint32_t)(Kb - 16);
    const uint32_t ring_lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem + wave * D * Cfg::UNIT_BYTES);
    const int G = grid_rows_out >> 8, nblocks = (N + Cfg::BN - 1) / Cfg::BN;
    const int my_blocks = (int)blockIdx.x >= nblocks ? 0 : (G >= nblocks ? 1 : (nblocks - (int)blockIdx.x + G - 1) / G);
    const int units = my_blocks * cnt;  // (block, run) pairs of this wave, block-major
    int ld_u = 0, ld_blk = blockIdx.x, ld_run = 0;
    auto issue_unit = [&]() __attribute__((always_inline)) {
        const int slot = ld_u % D, run = wave + ld_run * NW, n0 = ld_blk * Cfg::BN;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t dst = ring_lds + slot * Cfg::UNIT_BYTES + h * 1024;
            const uint32_t goff = row_bytes24(min(n0 + 8 * h + row8, p.N - 1), Kb) + min((uint32_t)run * 128u + piece_off[h], last16);
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(dst), "v"(goff), "s"(p.B) : "memory", "m0");
        }
        ++ld_u;
        if (++ld_run == cnt) { ld_run = 0; ld_blk += G; }
    };
    const int ahead = min(D, units);
    for (int d = 0; d < ahead; ++d) issue_unit();

    // ---- maxima, nibbles, scales ----
    amax = row_max<1>(amax, nullptr);
    for (int idx = tid; idx < 2 * 256; idx += Cfg::THREADS) red[idx] = 0;
    if constexpr (WPR > 1) {
        if (lane == 0) wave_max[wave] = amax;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < WPR; ++w) amax = fmaxf(amax, wave_max[row * WPR + w]);
    }
    if (row < p.M) {
        const float inv = amax > 0.0f ? 7.0f / amax : 0.0f;
        if (lane == 0 && wave % WPR == 0) row_scale[row] = amax / 7.0f;
        const int at = row * 128;
        quantise_chunks<IN>(plain, amax, inv, [&](auto quant) __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < NC; ++t) {
                // (the elements as loaded: widened for the maximum, the compiler would keep all of them as floats)
                asm volatile("" : "+v"(v[t].w[0]));
                const int c = c0 + t * 64 * WPR;
                const uint32_t n8 = quant(v[t]);
                if (c < xchunks) *reinterpret_cast<uint32_t *>(a_rows + (c >> 5) * Cfg::RUN_BYTES + at + ((((c >> 2) & 7) ^ ((row >> 1) & 7)) << 4) + (c & 3) * 4) = n8;
            }
        });
    }
    __syncthreads();

    // ---- fragments of A: lane (r, g), chunk j of the run -> logical piece 4 j + g (rows from ROWS on are rows 0 .. again) ----
    const int ra = r & (ROWS - 1), a_at = ra * 128, a_sw = (ra >> 1) & 7;
    v4i aev[R][2], aod[R][2];
#pragma unroll
    for (int q = 0; q < R; ++q)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            x16_expand_pairs(*reinterpret_cast<const v4i *>(a_rows + min(wave + q * NW, nruns - 1) * Cfg::RUN_BYTES + a_at + (((4 * j + g) ^ a_sw) << 4)), aev[q][j], aod[q][j]);
        }
    const float rs = row_scale[min(r, p.M - 1)];

    const int rd_row = (r >> 3) * 1024 + (r & 7) * 128, rd_sw = (r >> 1) & 7;
    const int rd_at[2] = {rd_row + ((g ^ rd_sw) << 4), rd_row + (((4 + g) ^ rd_sw) << 4)};
    auto wait_b = [&](const int younger) __attribute__((always_inline)) {
        if (younger <= 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        else if (younger == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPU) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LPU) : "memory");
    };
    static_assert(D <= 3, "wait_b");

    int u = 0;
    for (int b = 0, half = 0; b < my_blocks; ++b, half ^= 1) {
        const int blk = blockIdx.x + b * G;
        v4i acc = {0, 0, 0, 0};
#pragma unroll
        for (int q = 0; q < R; ++q) {
            if (q < cnt) {
                const int slot = u % D, run = wave + q * NW;
                wait_b(min(D - 1, units - 1 - u));
                const uint8_t *const at = smem + (wave * D + slot) * Cfg::UNIT_BYTES;
                v4i bpk[2];
#pragma unroll
                for (int c = 0; c < 2; ++c) bpk[c] = *reinterpret_cast<const v4i *>(at + rd_at[c]);
                if (u + D < units) {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    issue_unit();
                }
                ++u;
                if (run == nruns - 1 && (Kb & 127) != 0) {
#pragma unroll
                    for (int c = 0; c < 2; ++c) bpk[c] = run * 128 + (4 * c + g) * 16 < Kb ? bpk[c] : v4i{0, 0, 0, 0};
                }
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    v4i bev, bod;
                    x16_expand_pairs(bpk[c], bev, bod);
                    acc = mfma16(bev, aev[q][c], acc);
                    acc = mfma16(bod, aod[q][c], acc);
                }
            }
        }
        int32_t *const rh = red + half * 256;
        if (cnt > 0) {
#pragma unroll
            for (int e = 0; e < 4; ++e) __hip_atomic_fetch_add(&rh[e * 64 + lane], acc[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        __syncthreads();
        // One wave stores the block and clears its sums for the block after next; another one for the next block, since the loads of
        // its scales wait for those of B that it has in flight
        if (wave == (b & (NW - 1))) {
            v4i s;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s[e] = rh[e * 64 + lane] >> 8;
                rh[e * 64 + lane] = 0;
            }
            const int n = blk * Cfg::BN + 4 * g;
            if (r < p.M && n < p.N) {
                uint16_t *const d = reinterpret_cast<uint16_t *>(p.C) + (size_t)r * p.N + n;
                uint16_t h[4];
                finish16x4(p, s, rs, n, h);
                if (n + 3 < p.N) {
                    *reinterpret_cast<v2i_half_aligned *>(d) = v2i{(int)(h[0] | ((uint32_t)h[1] << 16)), (int)(h[2] | ((uint32_t)h[3] << 16))};
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (n + e < p.N) d[e] = h[e];
                }
            }
        }
    }
}

template <int IN, int ROWS, int NC, int R, int D>
static hipError_t ready_skinny_linear()
{
    using Cfg = SkinnyLinearCfg<IN, ROWS, NC, R, D>;
    static std::atomic<bool> lds_ok[QM_MAX_DEVICES] = {};
    return ensure_dynamic_lds(&skinny_linear_kernel<Cfg>, Cfg::lds_bytes(Cfg::MAX_K), lds_ok);
}
template <int IN, int ROWS, int NC, int R, int D>
static hipError_t launch_skinny_linear(const void *x, const void *B, void *Y, int m, int n, int k, const float *col_scale, const uint16_t *bias, int out, hipStream_t s)
{
    using Cfg = SkinnyLinearCfg<IN, ROWS, NC, R, D>;
    // (of a longer row the kernel would leave the rest out, of more rows all but ROWS)
    if (m > Cfg::ROWS || k > Cfg::MAX_K) return hipErrorInvalidValue;
    hipError_t e = ready_skinny_linear<IN, ROWS, NC, R, D>();
    if (e != hipSuccess) return e;
    int cus = 0;
    e = device_cus(&cus);
    if (e != hipSuccess) return e;
    const int blocks = (n + Cfg::BN - 1) / Cfg::BN, grid = blocks < cus ? blocks : cus;
    return enqueue(&skinny_linear_kernel<Cfg>, dim3(grid), dim3(Cfg::THREADS), Cfg::lds_bytes(k), s,
        static_cast<const uint8_t *>(x), static_cast<const uint8_t *>(B), static_cast<int32_t *>(Y), grid << 8 | m << 2 | out, n, k, col_scale, bias);
}
template <int IN>
static hipError_t launch_skinny_linear(const void *x, const void *B, void *Y, int m, int n, int k, const float *col_scale, const uint16_t *bias, int out, hipStream_t s)
{
    if (m > 8) return launch_skinny_linear<IN, 16, 4, 1, 3>(x, B, Y, m, n, k, col_scale, bias, out, s);
    if (m > 4) return launch_skinny_linear<IN, 8, 4, 1, 3>(x, B, Y, m, n, k, col_scale, bias, out, s);
    if (k <= 4096) return launch_skinny_linear<IN, 4, 2, 1, 3>(x, B, Y, m, n, k, col_scale, bias, out, s);
    return launch_skinny_linear<IN, 4, 4, 2, 3>(x, B, Y, m, n, k, col_scale, bias, out, s);
}
template <int IN>
static hipError_t ready_skinny_linear()
{
    for (const auto ready : {&ready_skinny_linear<IN, 16, 4, 1, 3>, &ready_skinny_linear<IN, 8, 4, 1, 3>, &ready_skinny_linear<IN, 4, 2, 1, 3>, &ready_skinny_linear<IN, 4, 4, 2, 3>}) {
        const hipError_t e = ready();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
// What the kernels that launch_skinny_linear has can do, whether it pays or not
constexpr bool skinny_linear_fits(int m, int k, int in)
{
    if (in == QM_IN_F32 || m < 1 || m > 16) return false;
    return k <= (m > 8 ? SkinnyLinearCfg<QM_IN_F16, 16, 4, 1, 3>::MAX_K : m > 4 ? SkinnyLinearCfg<QM_IN_F16, 8, 4, 1, 3>::MAX_K : SkinnyLinearCfg<QM_IN_F16, 4, 4, 2, 3>::MAX_K);
}
// Against two launches, in a graph with the weights from HBM, one / two over 75 sizes and both types (us: 4 x 4096 x 4096 5.9 -> 4.5,
// 8 x 6144 x 4096 7.1 -> 6.2, 16 x 2048 x 2048 5.1 -> 4.7); called eagerly they gain more, the host half of a call:
//   3, 4 rows    K <= 4096 to 12288 columns 0.73 .. 0.97, beyond 0.90 .. 1.27; K <= 8192 to 4096 0.85 .. 0.94, beyond 0.96 .. 1.11
//   5 .. 8       K <= 4096 to 8192 columns 0.79 .. 1.00, beyond 0.96 .. 1.33
//   9 .. 16      K <= 2048 to 8192 columns 0.75 .. 0.94, beyond 0.94 .. 1.34
// A longer K has no kernel (skinny_linear_fits).  (Below 1024 columns nothing was measured.  fp32 has twice the bytes of x and no shorter arithmetic.)
constexpr bool skinny_linear_pays(int m, int n, int k, int in)
{
    if (in == QM_IN_F32 || m < 3 || m > 16 || n < 1024) return false;
    if (m > 8) return k <= 2048 && n <= 8192;
    if (m > 4) return k <= 4096 && n <= 8192;
    return k <= 4096 ? n <= 12288 : k <= 8192 && n <= 4096;
}

}  // namespace qm

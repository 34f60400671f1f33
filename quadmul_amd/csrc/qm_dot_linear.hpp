// The int4 linear layer for one or two rows of activations, in one launch.
#pragma once
#include "qm_aux.hpp"
#include "qm_skinny.hpp"

namespace qm {

// gemm_dot_kernel with the quantisation of its rows in front: every workgroup quantises x by itself, with the arithmetic of
// quantize_pack_kernel, while the first of its loads of B are on their way.  That is a few elements per
// thread out of the L2; as a kernel of its own it is a second launch, 2.4 us and the gap between dependent kernels, in front of a
// GEMM of 2 to 3 (1 x 4096 x 4096), and on the host half of a call.  From three rows on: qm_skinny_linear.hpp.
template <int IN, int MR_, int NW_, int U_>
struct DotLinearCfg {
    static constexpr int MR = MR_, NW = NW_, U = U_, THREADS = 64 * NW, BN = 16;
    static constexpr int NC = 4;  // chunks of eight elements per thread and row that stay in registers between the maximum and the quantisation
};
inline int dot_linear_lds_bytes(int mr, int k) { return mr * (k / 2); }
// Against two launches, by the columns of one round of workgroups: every workgroup quantises x again, which costs little beside
// its own B while it runs once, and the launch and more where the device takes a second round of them.  A
// round is what registers leave room for (fp16 56, else 72 on 16 waves and one row: two workgroups of 1024
// threads per CU, or one).  Some way into a second round the calls stay in one launch while that takes the GPU less than two take the
// host, 8 to 9 us: called eagerly they then win by what the host saves, in a graph they lose the rest.
// GPU time, one launch / two inside a graph, weights from HBM, the range over 2500 sizes in all, and eager calls in turn:
//   one row   K > 4096         fp16 to 8192 columns 0.81 .. 1.02, else to 4096 0.83 .. 0.92; beyond 0.91 .. 1.11 and 1.04 .. 1.38
//             2048 < K <= 4096 0.83 .. 1.01 to 65536
//             K <= 2048        fp16 to 16384 0.69 .. 1.01, else to 12288 0.69 .. 0.95; to 24576 0.93 .. 1.16, eager 0.65 .. 0.97
//                              (24576 x 512 8.0 -> 6.2 us); beyond 1.0 .. 2.1
//   two rows  K > 4096         to 4096 0.85 .. 1.00; beyond 1.17 .. 1.31
//             K <= 4096        to 8192 0.74 .. 1.02 (fp16 from a K of 3072, 12288: 0.92 .. 1.00); below 3072 to 12288 (10240 below
//                              1024) 0.96 .. 1.18 (1.30), eager 0.71 .. 0.90 (10240 x 1024 8.0 -> 5.8 us); beyond to 3.5
// us, two / one: 1 x 1024 x 1024 4.46 / 3.18, 1 x 4096 x 4096 5.54 / 4.46, 1 x 28672 x 4096 14.2 / 13.1, but 1 x 10240 x 8192 12.2 / 15.0
// and 2 x 174481 x 64 17 / 60.  Above a K of 16384 a row takes more turns than hide their loads: 1 x 8192 x 28672 27.1 / 28.2.
inline bool dot_linear_pays(int m, int n, int k, int in)
{
    const bool f16 = in == QM_IN_F16;
    if (k > 16384) return false;
    if (m == 2) {
        if (k > 4096) return n <= 4096;
        if (k >= 3072) return n <= (f16 ? 12288 : 8192);
        return n <= (k >= 1024 ? 12288 : 10240);
    }
    if (k > 4096) return n <= (f16 ? 8192 : 4096);
    return n <= (k > 2048 ? 65536 : 24576);
}

template <int IN, class Cfg, bool ROUND>
__global__ void __launch_bounds__(Cfg::THREADS)
dot_linear_kernel(const uint8_t *x, const uint8_t *B, int32_t *D, const int rows_out, const int N, const int K, const float *col_scale, const uint16_t *bias)
{
    GemmArgs p{nullptr, B, D, packed_rows(rows_out), N, K};
    p.col_scale = col_scale;
    p.bias = bias;
    p.out = packed_out(rows_out);
    constexpr int MR = Cfg::MR, NW = Cfg::NW, U = Cfg::U, THREADS = Cfg::THREADS, NC = Cfg::NC;
    extern __shared__ __align__(16) uint8_t rows[];  // [MR][K / 2] packed
    __shared__ float red_max[MR][NW];
    __shared__ int32_t red[NW][MR][16];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n0 = blockIdx.x * Cfg::BN, Kb = p.K >> 1, nchunks = (p.K + 127) >> 7, xchunks = p.K >> 3;
    // x first: the counter of outstanding loads is in order, and these are needed first
    const auto x_at = [&](int i, int c) __attribute__((always_inline)) { return x + ((size_t)min(i, p.M - 1) * p.K + (size_t)min(c, xchunks - 1) * 8) * QuantIn<IN>::BYTES; };
    Chunk8<IN> v[MR][NC];
#pragma unroll
    for (int i = 0; i < MR; ++i)
#pragma unroll
        for (int t = 0; t < NC; ++t)
            if (t == 0 || t * THREADS < xchunks) v[i][t].load(x_at(i, tid + t * THREADS));
            else v[i][t] = v[i][0];
    // as in gemm_dot_kernel: 8 lanes per row of B, 128 contiguous bytes, 8 rows per load
    const int ld_row = lane >> 3, ld_ch = lane & 7;
    uint32_t b_off[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) b_off[h] = row_bytes24(min(n0 + 8 * h + ld_row, p.N - 1), Kb) + ld_ch * 16;
    v4i bq[U / 2][2];
    const auto load_b = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
        for (int pu = 0; pu < U / 2; ++pu) {
            const int kofs = (c0 + 2 * pu) * 64;
            const bool ok = kofs + ld_ch * 16 < Kb;
#pragma unroll
            for (int h = 0; h < 2; ++h) bq[pu][h] = ok ? __builtin_nontemporal_load(reinterpret_cast<const v4i *>(p.B + b_off[h] + kofs)) : v4i{0, 0, 0, 0};
        }
    };
    // (ROUND: as in gemm_dot_kernel; us in a graph, before -> now: 1 x 4096 x 8192 6.59 -> 6.35, 2 x 4096 x 8192 7.48 -> 6.87, 1 x 8192 x 8192
    // fp16 8.68 -> 8.00)
    const int first = ROUND ? wave * U + first_of_runs(nchunks / (NW * U), NW) * NW * U : wave * U;
    load_b(first);
    __builtin_amdgcn_sched_barrier(0);

    float scale[MR];
#pragma unroll
    for (int i = 0; i < MR; ++i) {
        float amax = 0.0f;
#pragma unroll
        for (int t = 0; t < NC; ++t) amax = v[i][t].amax(amax);
        for (int c = tid + NC * THREADS; c < xchunks; c += THREADS) {
            Chunk8<IN> w;
            w.load(x_at(i, c));
            amax = w.amax(amax);
        }
        amax = row_max<1>(amax, nullptr);
        if (lane == 0) red_max[i][wave] = amax;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MR; ++i) {
        float amax = red_max[i][0];
#pragma unroll
        for (int w = 1; w < NW; ++w) amax = fmaxf(amax, red_max[i][w]);
        const float inv = amax > 0.0f ? 7.0f / amax : 0.0f;
        scale[i] = amax / 7.0f;
        uint32_t *row = reinterpret_cast<uint32_t *>(rows + i * Kb);
#pragma unroll
        for (int t = 0; t < NC; ++t) {
            const uint32_t n8 = quant8(v[i][t], inv);
            if (tid + t * THREADS < xchunks) row[tid + t * THREADS] = n8;
        }
        for (int c = tid + NC * THREADS; c < xchunks; c += THREADS) {
            Chunk8<IN> w;
            w.load(x_at(i, c));
            row[c] = quant8(w, inv);
        }
    }
    __syncthreads();

    int32_t acc[MR][2];
#pragma unroll
    for (int i = 0; i < MR; ++i) acc[i][0] = acc[i][1] = 0;
    for (int part = 0; part < (ROUND ? 2 : 1); ++part)
        for (int c0 = part == 0 ? first : wave * U; c0 < (part == 0 ? nchunks : first); c0 += NW * U) {
            if (c0 != first) load_b(c0);
#pragma unroll
            for (int pu = 0; pu < U / 2; ++pu) {
                const int kofs = (c0 + 2 * pu) * 64 + ld_ch * 16;
#pragma unroll
                for (int i = 0; i < MR; ++i) {
                    const v4i a = *reinterpret_cast<const v4i *>(rows + i * Kb + min(kofs, Kb - 16));  // (past the row's end B is zero)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[i][h] = __builtin_amdgcn_sdot8(a[e], bq[pu][h][e], acc[i][h], false);
                }
            }
        }
#pragma unroll
    for (int i = 0; i < MR; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            int32_t s = acc[i][h];
            s += __builtin_amdgcn_update_dpp(0, s, 0xB1, 0xF, 0xF, true);
            s += __builtin_amdgcn_update_dpp(0, s, 0x4E, 0xF, 0xF, true);
            s += __builtin_amdgcn_update_dpp(0, s, 0x141, 0xF, 0xF, true);
            if (ld_ch == 0) red[wave][i][8 * h + ld_row] = s;
        }
    __syncthreads();
    if (tid < MR * 16) {
        const int m = tid >> 4, n = n0 + (tid & 15);
        if (m < p.M && n < p.N) {
            int32_t s = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) s += red[w][m][tid & 15];
            reinterpret_cast<uint16_t *>(D)[(size_t)m * p.N + n] = finish16(p, s, MR == 1 || m == 0 ? scale[0] : scale[MR - 1], n);
        }
    }
}

// Waves and chunks in flight by K as for the GEMM alone (heuristic() in qm_select.hpp).
template <int IN, int MR, int NW, int U>
static hipError_t launch_dot_linear(const void *x, const void *B, void *D, int m, int n, int k, const float *col_scale, const uint16_t *bias, int out, hipStream_t s)
{
    using Cfg = DotLinearCfg<IN, MR, NW, U>;
    // (the rows that go round are longer than those of the others)
    constexpr bool CAN_ROUND = NW == 16;
    static_assert(8192 / 128 % (NW * U) == 0, "whole turns");
    return enqueue(CAN_ROUND && goes_round(m, n, k) ? &dot_linear_kernel<IN, Cfg, CAN_ROUND> : &dot_linear_kernel<IN, Cfg, false>, dim3((n + Cfg::BN - 1) / Cfg::BN), dim3(Cfg::THREADS), dot_linear_lds_bytes(MR, k), s,
        static_cast<const uint8_t *>(x), static_cast<const uint8_t *>(B), static_cast<int32_t *>(D), pack_rows_out(m, out), n, k, col_scale, bias);
}
template <int IN>
static hipError_t launch_dot_linear(const void *x, const void *B, void *D, int m, int n, int k, const float *col_scale, const uint16_t *bias, int out, hipStream_t s)
{
    if (m == 2) return k <= 4096 ? launch_dot_linear<IN, 2, 8, 4>(x, B, D, m, n, k, col_scale, bias, out, s) : launch_dot_linear<IN, 2, 16, 2>(x, B, D, m, n, k, col_scale, bias, out, s);
    if (k <= 2048) return launch_dot_linear<IN, 1, 8, 4>(x, B, D, m, n, k, col_scale, bias, out, s);
    if (k <= 4096) return launch_dot_linear<IN, 1, 4, 8>(x, B, D, m, n, k, col_scale, bias, out, s);
    return launch_dot_linear<IN, 1, 16, 2>(x, B, D, m, n, k, col_scale, bias, out, s);
}

}  // namespace qm

// Wave-level split-K int4 GEMM for operands the 16-byte-aligned kernels cannot take: any even
// K from 32 up (rows may start at any byte), A and B at any address.
//
// The reference has no such path (its shapes are the rows of a table, kernel.cu:340-385).
// Without it these calls ran on one thread per element of C (small products) or on
// zero-padded copies of both operands (2 x (M + N) K / 2 bytes of extra traffic, which is
// most of the time while M is small).  Bound: where rows do not lie on multiples of four bytes the L1, which
// takes the 16 bytes of such a lane in four accesses, one access per clock (16 x 65536 x 4100: 4.07 accesses per
// lane and load, 0.99 per clock and CU; 78 us): those rows are loaded as aligned dwords, four and the one after them, and shifted (SHIFT; us, before ->
// now: 16 x 5001 x 2050 7.5 -> 4.3, 17 x 3307 x 4100 8.9 -> 5.2, 9 x 7085 x 7390 13.4 -> 9.0, 143 x 1003 x 1788 7.7 -> 4.6); where they
// do (0.87 per lane and
// load), HBM on a wide B (16 x 65536 x 8200 77 us, 3.5 TB/s; 3 x 9000 x 9000 12 us, 3.4 TB/s), the latency
// of a wave's K loop otherwise.  The decomposition is that of gemm_skinny_kernel: a
// workgroup owns 16*FM rows of A (grid.y walks over blocks of them) and 16*FN rows of B, its
// NW waves split K in 128-nibble chunks, partial blocks meet in the LDS.  Lane (r, g) loads the
// 16 bytes it feeds to the matrix core itself -- row r, bytes 16 g .. + 15 of the chunk's 64 --
// as one global_load_dwordx4, or that and a dword.  (Direct global -> LDS loads, which
// the aligned kernels use, want aligned addresses.)  U chunks are in flight per wave, no more than it has: with every wave
// loading U chunks whether or not they exist, 1 x 5001 x 2050 -- seventeen chunks on sixteen waves --
// took 10.5 us instead of 6.7.
//
// The end of a row: a lane whose 16 bytes would run past the end of the row loads the row's
// last 16 bytes instead -- in bounds, Kb >= 16 -- from A and from B alike, and the bytes of
// them that another lane has already (all of them for a lane wholly past the end) are zeroed in
// B.  No byte outside the operands is read.
#pragma once
#include "qm_common.hpp"

namespace qm {

template <int FM_, int FN_, int NW_, int U_>
struct RaggedCfg {
    static constexpr int FM = FM_, FN = FN_, NW = NW_, U = U_;
    static constexpr int THREADS = 64 * NW;
    static constexpr int MAX_M = 16 * FM, BN = 16 * FN;
    static_assert((FM + FN) * U <= 16, "staging registers: four per load in flight");
};

template <class Cfg, bool SHIFT>
__global__ void __launch_bounds__(Cfg::THREADS)
gemm_ragged_kernel(const uint8_t *A, const uint8_t *B, int32_t *C, const int M, const int N, const int K, const int ldc, const int out,
                   const float *row_scale, const float *col_scale, const uint16_t *bias)
{
    GemmArgs p{A, B, C, M, N, K};
    p.row_scale = row_scale;
    p.col_scale = col_scale;
    p.bias = bias;
    p.out = out;
    p.ldc = ldc;
    constexpr int FM = Cfg::FM, FN = Cfg::FN, NW = Cfg::NW, U = Cfg::U;
    __shared__ int32_t red[FM * FN * 256];  // the sum of the waves' blocks: [block][register][lane]

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * Cfg::BN, m0 = blockIdx.y * Cfg::MAX_M;
    const int Kb = K >> 1;                // bytes per row, any number from 16 up
    const int nchunks = (Kb + 63) >> 6;   // 64-byte chunks per row, the last one possibly short

    // (32-bit offsets: the host side keeps each operand below 2 GiB)
    uint32_t a_off[FM], b_off[FN];
#pragma unroll
    for (int i = 0; i < FM; ++i) a_off[i] = (uint32_t)min(m0 + i * 16 + r, M - 1) * (uint32_t)Kb;
#pragma unroll
    for (int j = 0; j < FN; ++j) b_off[j] = (uint32_t)min(n0 + j * 16 + r, N - 1) * (uint32_t)Kb;

    for (int idx = tid; idx < FM * FN * 256; idx += Cfg::THREADS) red[idx] = 0;
    __syncthreads();

    v4i acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = v4i{0, 0, 0, 0};

    const DwordSpan a_span = dword_span(A, (uint32_t)M * (uint32_t)Kb), b_span = dword_span(B, (uint32_t)N * (uint32_t)Kb);
    // chunks wave, wave + NW, ... of this wave, U at a time
    for (int c0 = wave; c0 < nchunks; c0 += NW * U) {
        v4i aq[U][FM], bq[U][FN];
        Shifted16 as[SHIFT ? U : 1][FM], bs[SHIFT ? U : 1][FN];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (c0 + u * NW >= nchunks) break;  // (wave-uniform)
            const uint32_t at = (uint32_t)min((c0 + u * NW) * 64 + g * 16, Kb - 16);
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                if constexpr (SHIFT) bs[u][j].load(b_span, b_off[j] + at);
                else bq[u][j] = *reinterpret_cast<const v4i_any_aligned *>(B + (b_off[j] + at));
            }
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                if constexpr (SHIFT) as[u][i].load(a_span, a_off[i] + at);
                else aq[u][i] = *reinterpret_cast<const v4i_any_aligned *>(A + (a_off[i] + at));
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = c0 + u * NW;
            if (c >= nchunks) break;
            if constexpr (SHIFT) {
#pragma unroll
                for (int j = 0; j < FN; ++j) bq[u][j] = bs[u][j].value();
#pragma unroll
                for (int i = 0; i < FM; ++i) aq[u][i] = as[u][i].value();
            }
            if ((c + 1) * 64 > Kb) {
                // the short last chunk: of the 16 bytes loaded the first `seen` belong to lanes
                // before this one
                const int seen = max(c * 64 + g * 16 - (Kb - 16), 0);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int s = min(max(seen - 4 * e, 0), 4);
                    const uint32_t keep = s >= 4 ? 0u : 0xFFFFFFFFu << (8 * s);
#pragma unroll
                    for (int j = 0; j < FN; ++j) bq[u][j][e] = (int)((uint32_t)bq[u][j][e] & keep);
                }
            }
            v4i bev[FN], bod[FN];
#pragma unroll
            for (int j = 0; j < FN; ++j) x16_expand_pairs(bq[u][j], bev[j], bod[j]);
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                v4i aev, aod;
                x16_expand_pairs(aq[u][i], aev, aod);
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[i][j] = mfma16(bev[j], aev, acc[i][j]);
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[i][j] = mfma16(bod[j], aod, acc[i][j]);
            }
        }
    }

    if (wave < nchunks) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    __hip_atomic_fetch_add(&red[((i * FN + j) * 4 + e) * 64 + lane], acc[i][j][e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __syncthreads();
    // one element per thread and pass, 16 consecutive threads in one row of C (whose rows are
    // not aligned either, as a rule)
    for (int idx = tid; idx < FM * FN * 256; idx += Cfg::THREADS) {
        const int blk = idx >> 8, ml = (idx >> 4) & 15, nl = idx & 15;
        const int32_t s = red[blk * 256 + (nl & 3) * 64 + ml + 16 * (nl >> 2)] >> 8;
        const int m = m0 + (blk / FN) * 16 + ml, n = n0 + (blk % FN) * 16 + nl;
        if (m < M && n < N) {
            const size_t at = (size_t)m * c_stride(p) + n;
            if (out == OUT_I32) C[at] = s;
            else reinterpret_cast<uint16_t *>(C)[at] = finish16(p, s, scale_at(row_scale, m, M), n);
        }
    }
}

}  // namespace qm

// int4 GEMM tile kernel on v_mfma_f32_16x16x128_f8f6f4 with 6-bit floats (gfx950).
//
// A 6-bit E2M3 float with the upper exponent bit clear is a sign and a four-bit magnitude in
// units of 1/8, so every int4 value is one of its codes, and the matrix core takes 128 of them per
// instruction in the time it takes 64 int8: 7.3 to 7.9 against 4.4 to 4.5 POP/s, card to card, on a loop of the
// instruction alone (quadmul_amd/probe.py; on one pair of operand registers, which do not toggle, 8.4 to 8.9).  Products are multiples of 1/64; the fp32 accumulators start from 1.5 * 2^17, where
// one unit in the last place is 1/64, so their bit patterns count those units as an integer would
// and every sum is exact (|C| <= 64 K < 2^22, K < 65536; checked on the
// extremes, in closed form, up to K = 65504).
//
// The price is the re-coding, and each operand pays it where it is cheaper:
//   * A is re-coded ahead of the GEMM by expand_a6_kernel into the caller's workspace, exactly
//     (sign and magnitude), in the order the LDS wants it, every row padded with zeros to an even
//     number of K-steps, together with the sum of each row;
//   * B stays packed in memory and in the LDS, and a wave re-codes its own fragments in registers:
//     seven instructions for 16 nibbles, as b + 8 (the nibble with its top bit flipped), a code
//     without a sign.  The 8 that every b has too much is 8 * (sum of the row of A) in C, taken out
//     where an item's accumulators get their start value.
//
// What bounds it: no unit is full, the LDS nearest to it.  The schedule is the int8 tile's (qm_tile16.hpp) -- slots of one matrix
// instruction each, the loads running ahead through item boundaries, the write-out inside an item's last
// K-step.  8192 x 8192 x 8192 runs at 1.8 to 1.9 GHz (int8: 2.15) in 469 thousand cycles: 264 of its matrix instructions, 16 each; fragments of
// 34.7 MB per CU read out of the LDS, 271 at 128 bytes a cycle, and 10.5 MB loaded into it, 82; no bank conflicts; a wave issues for a third of its time and waits to issue
// for 39 % (counters of the traced kernel).  Without its loads into the LDS the clock rises to 2.13 GHz and
// the cycles stay (taken before A was read as it is now, see read_a).  us, this kernel / int8: 8192 x 8192 x 8192 262 / 336,
// 2048 x 11008 x 4096 60 / 77, 4096 x 4096 x 4096 39.3 / 48.5; the kernel that re-codes A takes 22.6, 7.9 and 7.2 traced in front of it.
//
// Eight waves, two per SIMD: a wave by itself issues a vector instruction every eight cycles (two every four),
// and the 56 re-coding instructions per wave and K-step then take longer than the matrix ones (four waves
// with 128 x 128 each: 281 us instead of 262).
//
// Registers: the 256 x 256 tile keeps none of them in scratch memory (int32), 10 (scaled) or 24 (scaled, bias), all of it
// around an item's start and write-out: no reload, whose wait would drain the counted loads, lies in the loop over K.
//
// Tiles of 256 x 128 (4 x 2 waves) halve the grain where 256 x 256 leaves most of a round idle: per K-step and round 0.53 us
// against 0.82, per round 5.8 against 13.8; their LDS has room for a write-out area of its own, where the large tile borrows a stage of B.
#pragma once
#include <type_traits>

#include "qm_fp6.hpp"
#include "qm_tile16.hpp"

namespace qm {

__device__ __forceinline__ void mfma6_acc(v4i &acc, const v6i &s0, const v6i &s1)
{
    asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0 cbsz:2 blgp:2" : "+a"(acc) : "v"(s0), "v"(s1));
}
// The start value of a lane's four accumulators -- one row of A, four columns -- whatever they held: 1.0 * start + 0
// in the outer product of 16 blocks of 4 x 4, whose layout gives a lane its own column.  (An addend in
// vector registers is not to be had for a result in accumulator ones.  Two wait states: vector instructions may
// have worked `start` out just before.)
__device__ __forceinline__ void mfma6_start(v4i &acc, const float &one, const int &start)
{
    asm volatile("s_nop 1\n\tv_mfma_f32_4x4x1_16b_f32 %0, %1, %2, 0" : "+a"(acc) : "v"(one), "v"(start));
}

__device__ __forceinline__ v2i shl2_pair(const int lo, const int hi)
{
    v2i in = {lo, hi}, out;
    asm("v_lshlrev_b64 %0, 2, %1" : "=v"(out) : "v"(in));
    return out;
}
__device__ __forceinline__ int bit_select(const uint32_t mask, const int one, const int zero)
{
    return (int)__builtin_amdgcn_bitop3_b32(mask, (uint32_t)one, (uint32_t)zero, 0xca);
}
__device__ __forceinline__ int and_xor(const int y, const uint32_t keep, const uint32_t flip)
{
    return (int)__builtin_amdgcn_bitop3_b32((uint32_t)y, keep, flip, 0x6a);
}
__device__ __forceinline__ void keep_here6(const v6i &x) { asm volatile("" ::"v"(x)); }
__device__ __forceinline__ void keep_here1(const int &x) { asm volatile("" ::"v"(x)); }
__device__ __forceinline__ void acc_to_lds(const uint32_t at, const v4i &acc) { asm volatile("ds_write_b128 %0, %1" ::"v"(at), "a"(acc) : "memory"); }

template <int BM_, int BN_, int WGM_, int WGN_>
struct Tile6Cfg {
    static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_;
    static constexpr int WAVES = WGM * WGN, THREADS = 64 * WAVES;
    static constexpr int WM = BM / WGM, WN = BN / WGN, FM = WM / 16, FN = WN / 16;
    // A K-step of A per stage; B two K-steps at a time, whole 128-byte lines of its rows
    static constexpr int A_STAGES = 4, B_STAGES = 2, A_BYTES = BM * FP6_STEP_BYTES, B_BYTES = BN * 128;
    static constexpr int RING_BYTES = A_STAGES * A_BYTES + B_STAGES * B_BYTES;
    static constexpr int XHALF_BYTES = 16 * 128;           // the write-out's area, per wave, as in Tile16Cfg
    static constexpr int SCALE_BYTES = WM * 4 + WN * 6;   // ... and its scales and biases, beside them
    // Where the ring leaves no room for them they are in the stage of B that is free in an item's last step.
    static constexpr bool OWN_AREA = RING_BYTES + WAVES * (XHALF_BYTES + SCALE_BYTES) <= 160 * 1024;
    static constexpr int LDS_BYTES = RING_BYTES + (OWN_AREA ? WAVES * (XHALF_BYTES + SCALE_BYTES) : 0);
    static constexpr int A_GROUPS = BM / 32 / WAVES, A_PIECES = 3 * A_GROUPS, B_PIECES = BN / 8 / WAVES;
    static_assert(BM % (32 * WAVES) == 0 && BN % (8 * WAVES) == 0 && WAVES % 2 == 0, "loads divide evenly among the waves");
    static_assert(WM % 64 == 0 && WN % 64 == 0 && (OWN_AREA || WAVES * (XHALF_BYTES + SCALE_BYTES) <= B_BYTES), "the write-out fits the stage it borrows");
    static_assert(LDS_BYTES <= 160 * 1024, "LDS budget of a gfx950 CU");
    static_assert(FM % 4 == 0 && FN >= 4 && FN % 2 == 0, "two pairs of fragments of A in rotation; blocks leave in pairs");
};

template <class Cfg, int OUT = OUT_I32, bool BIAS = false>
__global__ void __launch_bounds__(Cfg::THREADS, Cfg::THREADS / 256)
gemm_tile6_kernel(const GemmArgs p, const uint8_t *const a6, const int *const row_sums, const int parts, const int kt_all, const int tiles_m, const int tiles_n, const int group_m)
{
    constexpr int BM = Cfg::BM, BN = Cfg::BN, FM = Cfg::FM, FN = Cfg::FN, WAVES = Cfg::WAVES;
    constexpr int A_PIECES = Cfg::A_PIECES, B_PIECES = Cfg::B_PIECES;
    constexpr int ESZ = OUT == OUT_I32 ? 4 : 2;
    extern __shared__ __align__(16) uint8_t smem[];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave / Cfg::WGN, wn = wave % Cfg::WGN;
    const int r = lane & 15, g = lane >> 4;
    const int G = gridDim.x;
    const int nitems = tiles_m * tiles_n;
    const int Kb = p.K >> 1;
    const int ldc = c_stride(p);
    const bool vec_ok = (ldc & 3) == 0 && ((uintptr_t)p.C & (4 * ESZ - 1)) == 0;
    const int last_n0 = vec_ok ? p.N : p.N - BN;
    const int full_m = p.M / BM, full_n = p.N / BN;
    const int nwhole = __builtin_amdgcn_readfirstlane(full_m * full_n);
    auto locate = [&](const int item, int &m0, int &n0) __attribute__((always_inline)) {
        const int rows = nwhole ? full_m : tiles_m, cols = nwhole ? full_n : tiles_n;
        const int pid = xcd_contiguous_id(nwhole ? min(item, nwhole - 1) : item, nwhole ? nwhole : nitems);
        const int width = group_m * cols;
        const int first_m = (pid / width) * group_m;
        const int gsz = min(rows - first_m, group_m);
        const int tm_a = __builtin_amdgcn_readfirstlane(first_m + (pid % width) % gsz);
        const int tn_a = __builtin_amdgcn_readfirstlane((pid % width) / gsz);
        const bool ragged = nwhole != 0 && item >= nwhole;
        const int nr = max(nitems - nwhole, 1), right = tiles_n > full_n ? tiles_m : 0;
        const int e8 = max(item - nwhole, 0) + (nwhole & 7), x8 = e8 & 7, s8 = nwhole & 7;
        const int f_hi = ((s8 + nr) >> 3) * x8 + min((s8 + nr) & 7, x8), f_lo = min(s8, x8);
        const int q = __builtin_amdgcn_readfirstlane(min(f_hi - f_lo + (e8 >> 3) - (x8 < s8 ? 1 : 0), nr - 1));
        const int r0 = __builtin_amdgcn_readfirstlane(q * right / nr), r1 = __builtin_amdgcn_readfirstlane((q + 1) * right / nr);
        const int tm_b = r1 > r0 ? r0 : full_m, tn_b = r1 > r0 ? full_n : q - r0;
        m0 = (ragged ? tm_b : tm_a) * BM;
        n0 = min((ragged ? tn_b : tn_a) * BN, last_n0);
    };

    // ---- global -> LDS ----
    // (piece c of row n of a stage of B lies at c ^ ((n >> 1) & 7): the 16 rows of a fragment read are then in
    // different banks)
    const int dma_row = lane >> 3;
    const uint32_t dma_col = ((lane & 7) ^ ((dma_row >> 1) | ((wave & 1) << 2))) * 16;
    const int groups = (p.M + 31) >> 5;
    uint32_t a_goff[Cfg::A_GROUPS], b_goff[B_PIECES];
    int d_item = blockIdx.x, d_kt = 0;
    auto cursor_load = [&]() __attribute__((always_inline)) {
        int m0, n0;
        locate(d_item, m0, n0);
#pragma unroll
        for (int q = 0; q < Cfg::A_GROUPS; ++q)
            a_goff[q] = (uint32_t)min((m0 >> 5) + q * WAVES + wave, groups - 1) * (uint32_t)(kt_all * FP6_GROUP_BYTES) + lane * 16;
#pragma unroll
        for (int q = 0; q < B_PIECES; ++q)
            b_goff[q] = (uint32_t)min(n0 + (q * WAVES + wave) * 8 + dma_row, p.N - 1) * (uint32_t)Kb + dma_col;
    };
    const uint8_t *a_src, *b_src;
    // (two steps that the row of B does not fill read the row's last 128 bytes; what of them is not these steps'
    // own has zeros in A.  b_src counts at the first of two steps only)
    auto cursor_point = [&]() __attribute__((always_inline)) {
        a_src = a6 + d_kt * FP6_GROUP_BYTES;
        b_src = p.B + min(d_kt * 64, Kb - 128);
    };
    auto cursor_advance = [&]() __attribute__((always_inline)) {
        if (++d_kt == kt_all) {
            if (d_item + G < nitems) {
                d_item += G;
                d_kt = 0;
                cursor_load();
            } else {
                d_kt = kt_all - 1;
            }
        }
        cursor_point();
    };
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
    const uint32_t dma_lds_a = __builtin_amdgcn_readfirstlane(lds0 + wave * FP6_GROUP_BYTES);
    const uint32_t dma_lds_b = __builtin_amdgcn_readfirstlane(lds0 + wave * 1024);
    // piece q of B, and the three KiB of A, which follow each other in memory and in the LDS (the
    // instruction's offset counts on both sides)
    auto dma_setup_b = [&](int q, int stage) __attribute__((always_inline)) {
        asm volatile("s_mov_b32 m0, %0" ::"s"(dma_lds_b + stage + q * WAVES * 1024) : "memory", "m0");
    };
    auto dma_setup_a = [&](int q, int stage) __attribute__((always_inline)) {
        asm volatile("s_mov_b32 m0, %0" ::"s"(dma_lds_a + stage + q / 3 * WAVES * FP6_GROUP_BYTES) : "memory", "m0");
    };
    auto dma_issue_b = [&](int q) __attribute__((always_inline)) { asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(b_goff[q]), "s"(b_src) : "memory"); };
    auto dma_issue_a = [&](int q) __attribute__((always_inline)) {
        if (q % 3 == 0) asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(a_goff[q / 3]), "s"(a_src) : "memory");
        else if (q % 3 == 1) asm volatile("global_load_lds_dwordx4 %0, %1 offset:1024" ::"v"(a_goff[q / 3]), "s"(a_src) : "memory");
        else asm volatile("global_load_lds_dwordx4 %0, %1 offset:2048" ::"v"(a_goff[q / 3]), "s"(a_src) : "memory");
    };

    // ---- fragment reads ----
    constexpr int B_BASE = Cfg::A_STAGES * Cfg::A_BYTES;
    // A: two fragments, 32 rows, are three reads of 16 bytes per lane into twelve registers, the second fragment behind the
    // first.  (As a read of 16 and one of 8 bytes per fragment, which the LDS serves at less than its full rate, the same bytes took
    // longer: us, before -> now, 8192 x 8192 x 8192 266 -> 262, 2048 x 11008 x 4096 62.3 -> 60.4, 2048 x 4096 x 11008 62.5 -> 59.7, all on 256 x 256.)
    const int a_rd = wm * (Cfg::WM / 32) * FP6_GROUP_BYTES + lane * 16;
    const int b_row = wn * Cfg::WN + r;
    const int b_rd = b_row * 128 + ((g ^ ((b_row >> 1) & 7)) << 4);  // of the first of two steps; the second's differs in bit 6
    typedef int v12i __attribute__((ext_vector_type(12)));
    auto read_a = [&](int stage, int q, int t, v12i &pair) __attribute__((always_inline)) {  // third t of pair q
        const v4i x = *reinterpret_cast<const v4i *>(smem + stage + a_rd + q * FP6_GROUP_BYTES + t * 1024);
        pair[4 * t] = x.x; pair[4 * t + 1] = x.y; pair[4 * t + 2] = x.z; pair[4 * t + 3] = x.w;
    };
    const int b_rd2 = b_rd ^ 64;
    auto read_b = [&](int stage, bool second, int j) __attribute__((always_inline)) -> v4i {
        return *reinterpret_cast<const v4i *>(smem + stage + (second ? b_rd2 : b_rd) + j * 16 * 128);
    };

    v4i acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = v4i{0, 0, 0, 0};

    // re-coding of B: masks in scalar registers, what is flipped in vector ones (an instruction reads one scalar register)
    uint32_t pick[3], keep[3], flip[3];
#pragma unroll
    for (int t = 0; t < 3; ++t) {
        asm volatile("s_mov_b32 %0, %1" : "=s"(pick[t]) : "s"(FP6_PICK[t]));
        asm volatile("s_mov_b32 %0, %1" : "=s"(keep[t]) : "s"(FP6_KEEP[t]));
        asm volatile("v_mov_b32 %0, %1" : "=v"(flip[t]) : "s"(FP6_TOP[t]));
    }
    constexpr int W = 14;  // instructions per fragment
    v2i sh;
    auto code_op = [&](auto k_, const v4i &pk, v6i &f) __attribute__((always_inline)) {
        constexpr int k = decltype(k_)::value, h = k / 7, part = k % 7, t = (part - 1) / 2;
        if constexpr (part == 0) sh = shl2_pair(pk[2 * h], pk[2 * h + 1]);
        else if constexpr (part % 2 == 1) f[3 * h + t] = bit_select(pick[t], t == 1 ? pk[2 * h + 1] : pk[2 * h], t == 0 ? sh.x : sh.y);
        else f[3 * h + t] = and_xor(f[3 * h + t], keep[t], flip[t]);
    };

    // ---- writing a finished tile (see qm_tile16.hpp, the half-size area) ----
    int c_item = blockIdx.x, c_m0, c_n0;
    char *tile_c = nullptr;
    typedef float v4f __attribute__((ext_vector_type(4)));
    constexpr int NH = FN / 2;  // half groups of 32 columns
    // Scaled output: a wave's scales and biases wait in a few registers, one value per lane, while an item's K-steps run,
    // and go to an area of its own beside the write-out's in its last step, to be read back in the order of the stores
    // (held per lane in that order they are twenty registers too many).
    constexpr bool SCALED = OUT != OUT_I32;
    float rs_reg[SCALED ? Cfg::WM / 64 : 1], cs_reg[SCALED ? Cfg::WN / 64 : 1];
    uint16_t bias_reg[BIAS ? Cfg::WN / 64 : 1];
    int sc = 0;  // byte offset of the area: row scales, column scales, biases
    float rs_now[2];
    v4f cs_now;
    v2i bias_now;
    int rows_left = 0, cols_left = 0;
    v4i xr[2];
    const uint32_t lane_half = ((uint32_t)(wm * Cfg::WM + (lane >> 3)) * (uint32_t)ldc + (uint32_t)(wn * Cfg::WN + (lane & 7) * 4)) * (uint32_t)ESZ;
    int xh = 0;  // this wave's area: byte offset in the LDS
    const int xh_wr = r * 128 + ((g ^ (r & 7)) << 4);
    const int xh_rd = (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 3)) << 4);
    auto store_lanes = [&](char *const base, const uint32_t lane_off, const auto v, auto row_, auto col_) __attribute__((always_inline)) {
        constexpr int row = decltype(row_)::value, col = decltype(col_)::value;
        const int rl = rows_left, cl = cols_left;
        uint64_t saved, on;
        if constexpr (sizeof(v) == 16)
            asm volatile("s_nop 4\n\tv_cmp_lt_i32_e32 vcc, %7, %5\n\ts_mov_b64 %1, vcc\n\tv_cmp_lt_i32_e32 vcc, %8, %6\n\ts_and_b64 %1, %1, vcc\n\t"
                         "s_mov_b64 %0, exec\n\ts_mov_b64 exec, %1\n\tglobal_store_dwordx4 %2, %3, %4\n\ts_mov_b64 exec, %0"
                         : "=&s"(saved), "=&s"(on) : "v"(lane_off), "v"(v), "s"(base), "v"(rl), "v"(cl), "n"(row), "n"(col) : "memory", "vcc", "scc");
        else
            asm volatile("s_nop 4\n\tv_cmp_lt_i32_e32 vcc, %7, %5\n\ts_mov_b64 %1, vcc\n\tv_cmp_lt_i32_e32 vcc, %8, %6\n\ts_and_b64 %1, %1, vcc\n\t"
                         "s_mov_b64 %0, exec\n\ts_mov_b64 exec, %1\n\tglobal_store_dwordx2 %2, %3, %4\n\ts_mov_b64 exec, %0"
                         : "=&s"(saved), "=&s"(on) : "v"(lane_off), "v"(v), "s"(base), "v"(rl), "v"(cl), "n"(row), "n"(col) : "memory", "vcc", "scc");
    };
    auto store_half = [&](auto ib_, auto h_, auto k_, auto edge_) __attribute__((always_inline)) {
        constexpr bool edge = decltype(edge_)::value;
        constexpr int ib = decltype(ib_)::value, h = decltype(h_)::value, k = decltype(k_)::value;
        char *const at = tile_c + ((size_t)(ib * 16 + 8 * k) * ldc + h * 32) * ESZ;  // wave-uniform
        using Row = std::integral_constant<int, ib * 16 + 8 * k>;
        using Col = std::integral_constant<int, h * 32>;
        if constexpr (OUT == OUT_I32) {
            v4i v = xr[k];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] -= (int)FP6_START;
            if constexpr (edge) store_lanes(at, lane_half, v, Row{}, Col{});
            else *reinterpret_cast<v4i_elem_aligned *>(at + lane_half) = v;
        } else {
            const int e0 = xr[k][0], e1 = xr[k][1], e2 = xr[k][2], e3 = xr[k][3];
            constexpr int start = (int)FP6_START;
            const float rs = rs_now[k];
            v2i o{(int)round16_pair<SCALED ? OUT : OUT_F16>(scaled(e0 - start, rs, cs_now[0]), scaled(e1 - start, rs, cs_now[1])),
                  (int)round16_pair<SCALED ? OUT : OUT_F16>(scaled(e2 - start, rs, cs_now[2]), scaled(e3 - start, rs, cs_now[3]))};
            if constexpr (BIAS) o = v2i{(int)add16_pair<OUT>((uint32_t)o.x, (uint32_t)bias_now.x), (int)add16_pair<OUT>((uint32_t)o.y, (uint32_t)bias_now.y)};
            if constexpr (edge) store_lanes(at, lane_half, o, Row{}, Col{});
            else *reinterpret_cast<v2i_half_aligned *>(at + lane_half) = o;
        }
    };
    // part t = 0..3 of blocks (ib, 2h) and (ib, 2h + 1)
    auto write_half = [&](auto ib_, auto h_, auto t_, auto edge_) __attribute__((always_inline)) {
        constexpr int ib = decltype(ib_)::value, h = decltype(h_)::value, t = decltype(t_)::value;
        constexpr int pib = h > 0 ? ib : ib - 1, ph = h > 0 ? h - 1 : NH - 1;  // the half group before this one
        if constexpr (t < 2) {
            const int at = t == 0 ? xh_wr : xh_wr ^ 64;
            acc_to_lds(lds0 + xh + at, acc[ib][2 * h + t]);
            if constexpr (pib >= 0) store_half(std::integral_constant<int, pib>{}, std::integral_constant<int, ph>{}, t_, edge_);
        }
        if constexpr (t >= 2) {
            xr[t - 2] = *reinterpret_cast<const v4i *>(smem + xh + xh_rd + 1024 * (t - 2));
            if constexpr (SCALED) rs_now[t - 2] = *reinterpret_cast<const float *>(smem + sc + (ib * 16 + 8 * (t - 2) + (lane >> 3)) * 4);
            if constexpr (SCALED && t == 2) cs_now = *reinterpret_cast<const v4f *>(smem + sc + Cfg::WM * 4 + (h * 32 + (lane & 7) * 4) * 4);
            if constexpr (BIAS && t == 2) bias_now = *reinterpret_cast<const v2i *>(smem + sc + Cfg::WM * 4 + Cfg::WN * 4 + (h * 32 + (lane & 7) * 4) * 2);
        }
    };

    // During step s, a_ring[t] holds A of step s + t (t = 3: is being filled).  Even s: b_ring[0] holds B of steps s and s + 1
    // -- of s + 1 only, B of s went into registers during step s - 1 -- and b_ring[1] of s + 2 and s + 3; odd s: b_ring[0] is free
    // and is filled again, with steps s + 3 and s + 4.
    int a_ring[Cfg::A_STAGES], b_ring[2] = {B_BASE, B_BASE + Cfg::B_BYTES};
#pragma unroll
    for (int t = 0; t < Cfg::A_STAGES; ++t) a_ring[t] = t * Cfg::A_BYTES;
    auto load_b = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < B_PIECES; ++q) {
            dma_setup_b(q, stage);
            asm volatile("s_nop 0" ::: "memory");
            dma_issue_b(q);
        }
    };
    int start_reg[FM];
    // where an item lies, and the sums of its rows of A on their way (a lane has every fourth part of them)
    auto next_item = [&](const int item) __attribute__((always_inline)) {
        locate(item, c_m0, c_n0);
        const int row = c_m0 + wm * Cfg::WM + r;
#pragma unroll
        for (int ib = 0; ib < FM; ++ib) start_reg[ib] = row_sums[min(g, parts - 1) * groups * 32 + min(row + ib * 16, groups * 32 - 1)];
    };
    cursor_load();
    cursor_point();
#pragma unroll
    for (int t = 0; t < 3; ++t) {
        if (t != 1) load_b(b_ring[t >> 1]);
#pragma unroll
        for (int q = 0; q < A_PIECES; ++q) {
            dma_setup_a(q, a_ring[t]);
            asm volatile("s_nop 0" ::: "memory");
            dma_issue_a(q);
        }
        cursor_advance();
    }
    next_item(blockIdx.x);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(A_PIECES + B_PIECES) : "memory");
    __syncthreads();

    v6i bf[2][FN];
    v12i ap[2];
    constexpr int NPK = FM * FN >= 32 ? 2 : FN;  // packed fragments of B between their read and their re-coding
    v4i b_pk[NPK];
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const v4i q = read_b(b_ring[0], false, j);
        static_for<0, W>([&](auto k_) __attribute__((always_inline)) { code_op(k_, q, bf[0][j]); });
    }
#pragma unroll
    for (int t = 0; t < 3; ++t) read_a(a_ring[0], 0, t, ap[0]);
    // (one register tuple, before its halves are used: else the compiler gives each half one of its own and copies)
    asm volatile("" : "+v"(ap[0]));
    auto frag_a = [&](auto i_) __attribute__((always_inline)) -> v6i {
        constexpr int i = decltype(i_)::value, q = (i >> 1) & 1;
        if constexpr (i & 1) return __builtin_shufflevector(ap[q], ap[q], 6, 7, 8, 9, 10, 11);
        else return __builtin_shufflevector(ap[q], ap[q], 0, 1, 2, 3, 4, 5);
    };
    float one;
    asm volatile("v_mov_b32 %0, 1.0" : "=v"(one));

    auto swap_b = [&]() __attribute__((always_inline)) {
        const int t = b_ring[0];
        b_ring[0] = b_ring[1];
        b_ring[1] = t;
    };
    // One K-step: contracts the step in a_ring[0] with its B fragments in register set bs, reads and re-codes
    // the B fragments of the step after it, and issues the cursor's loads.  `first`: the accumulators
    // start over.  `last` as in gemm_tile16_kernel: 1 a whole tile, 2 one that sticks out of C.
    auto k_step = [&](auto bs_tag, auto first_tag, auto last_tag) __attribute__((always_inline)) {
        constexpr int bs = decltype(bs_tag)::value;
        constexpr bool first = decltype(first_tag)::value, last = decltype(last_tag)::value != 0, edge = decltype(last_tag)::value == 2;
        constexpr int SLOTS = FM * FN, OPS = W * FN;
        constexpr bool loads_b = bs == 1 && (!last || Cfg::OWN_AREA);  // (else the stage is the write-out's)
        constexpr int LEAD = FN;               // the first fragment read in slot 0 is there by then
        static_for<0, SLOTS>([&](auto s_) __attribute__((always_inline)) {
            constexpr int s = decltype(s_)::value, i = s / FN, j = s % FN;
            mfma6_acc(acc[i][j], bf[bs][j], frag_a(std::integral_constant<int, i>{}));
            if constexpr (first && i + 1 < FM) mfma6_start(acc[i + 1][j], one, start_reg[i + 1]);
            if constexpr (i % 2 == 0 && j < 3) read_a(i + 2 >= FM ? a_ring[1] : a_ring[0], (i + 2) % FM / 2, j, ap[(i / 2 + 1) & 1]);
            if constexpr (i % 2 == 1 && j == FN - 1) asm volatile("" : "+v"(ap[(i / 2 + 1) & 1]));
            // fragment q of B is re-coded in ops [W q, W (q + 1)), which begin at slot LEAD + W q (SLOTS - LEAD) / OPS
            static_for<0, FN>([&](auto q_) __attribute__((always_inline)) {
                constexpr int q = decltype(q_)::value;
                constexpr int begin = LEAD + W * q * (SLOTS - LEAD) / OPS;
                if constexpr (s == begin - LEAD) b_pk[q % NPK] = read_b(b_ring[bs], bs == 0, q);
            });
            if constexpr (s >= LEAD) {
                constexpr int lo = (s - LEAD) * OPS / (SLOTS - LEAD), hi = (s - LEAD + 1) * OPS / (SLOTS - LEAD);
                static_for<lo, hi>([&](auto o_) __attribute__((always_inline)) {
                    constexpr int o = decltype(o_)::value, q = o / W;
                    code_op(std::integral_constant<int, o % W>{}, b_pk[q % NPK], bf[bs ^ 1][q]);
                });
            }
            // write-out of the accumulator row finished one sub-step ago: 4 NH parts over FN slots
            if constexpr (last && i >= 1) {
                static_for<j * 4 * NH / FN, (j + 1) * 4 * NH / FN>([&](auto t_) __attribute__((always_inline)) {
                    constexpr int t = decltype(t_)::value;
                    write_half(std::integral_constant<int, i - 1>{}, std::integral_constant<int, t / 4>{}, std::integral_constant<int, t % 4>{}, std::integral_constant<bool, edge>{});
                });
            }
            // the loads, spread over the step, M0 written two slots ahead
            constexpr int NB = loads_b ? B_PIECES : 0;
            static_for<0, NB + A_PIECES>([&](auto q_) __attribute__((always_inline)) {
                constexpr int q = decltype(q_)::value, at = 3 + q * (SLOTS - 6) / (NB + A_PIECES);
                if constexpr (s == at - 2 && q < NB) dma_setup_b(q, b_ring[0]);
                if constexpr (s == at - 2 && q >= NB && (q - NB) % 3 == 0) dma_setup_a(q - NB, a_ring[3]);
                if constexpr (s == at && q < NB) dma_issue_b(q);
                if constexpr (s == at && q >= NB) dma_issue_a(q - NB);
            });
            __builtin_amdgcn_sched_barrier(0);
        });
#pragma unroll
        for (int j = 0; j < FN; ++j) keep_here6(bf[bs ^ 1][j]);
        // What the step after this one reads -- its A, the B of the step after it -- must be there: everything but this
        // step's own loads.  The counter is in order of issue and counts stores too: a last step's are all
        // younger, and may stay in flight (`edge`: a store without lanes may not count).
        constexpr int pending = A_PIECES + (loads_b ? B_PIECES : 0) + (last && !edge ? (FM - 1) * FN - 2 : 0);
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(pending > 63 ? 63 : pending) : "memory");
        const int ta = a_ring[0];
#pragma unroll
        for (int u = 0; u + 1 < Cfg::A_STAGES; ++u) a_ring[u] = a_ring[u + 1];
        a_ring[Cfg::A_STAGES - 1] = ta;
        if constexpr (loads_b) swap_b();
        if constexpr (!last || loads_b) cursor_advance();
    };

    auto run_item = [&](auto mode_) __attribute__((always_inline)) {
        constexpr int mode = decltype(mode_)::value;
        constexpr bool edge = mode == 2;
        using No = std::integral_constant<int, 0>;
        if constexpr (edge) {
            rows_left = p.M - c_m0 - wm * Cfg::WM - (lane >> 3);
            cols_left = p.N - c_n0 - wn * Cfg::WN - (lane & 7) * 4;
        }
#pragma unroll
        for (int ib = 0; ib < FM; ++ib) {
            int sum = g < parts ? start_reg[ib] : 0;
            for (int t = g + 4; t < parts; t += 4) sum += row_sums[t * groups * 32 + min(c_m0 + wm * Cfg::WM + r + ib * 16, groups * 32 - 1)];
            sum += __shfl_xor(sum, 16);
            sum += __shfl_xor(sum, 32);
            start_reg[ib] = (int)FP6_START - 8 * sum;
        }
        if constexpr (SCALED) {
#pragma unroll
            for (int q = 0; q < Cfg::WM / 64; ++q) rs_reg[q] = scale_at(p.row_scale, c_m0 + wm * Cfg::WM + q * 64 + lane, p.M);
#pragma unroll
            for (int q = 0; q < Cfg::WN / 64; ++q) cs_reg[q] = scale_at(p.col_scale, c_n0 + wn * Cfg::WN + q * 64 + lane, p.N);
            if constexpr (BIAS) {
#pragma unroll
                for (int q = 0; q < Cfg::WN / 64; ++q) {
                    const int n = c_n0 + wn * Cfg::WN + q * 64 + lane;
                    bias_reg[q] = n < p.N ? p.bias[n] : (uint16_t)0x8000u;
                }
            }
#pragma unroll
            for (int q = 0; q < Cfg::WM / 64; ++q) keep_here_f(rs_reg[q]);
#pragma unroll
            for (int q = 0; q < Cfg::WN / 64; ++q) keep_here_f(cs_reg[q]);
        }
        static_for<0, FN>([&](auto j_) __attribute__((always_inline)) { mfma6_start(acc[0][decltype(j_)::value], one, start_reg[0]); });
        asm volatile("s_nop 7" ::: "memory");
        k_step(std::integral_constant<int, 0>{}, std::true_type{}, No{});
        for (int kt = 2; kt < kt_all; kt += 2) {
            k_step(std::integral_constant<int, 1>{}, std::false_type{}, No{});
            k_step(std::integral_constant<int, 0>{}, std::false_type{}, No{});
        }
        const int area = Cfg::OWN_AREA ? Cfg::RING_BYTES : b_ring[0];
        xh = area + wave * Cfg::XHALF_BYTES;
        if constexpr (SCALED) {
            sc = area + WAVES * Cfg::XHALF_BYTES + wave * Cfg::SCALE_BYTES;
#pragma unroll
            for (int q = 0; q < Cfg::WM / 64; ++q) *reinterpret_cast<float *>(smem + sc + (q * 64 + lane) * 4) = rs_reg[q];
#pragma unroll
            for (int q = 0; q < Cfg::WN / 64; ++q) *reinterpret_cast<float *>(smem + sc + Cfg::WM * 4 + (q * 64 + lane) * 4) = cs_reg[q];
            if constexpr (BIAS) {
#pragma unroll
                for (int q = 0; q < Cfg::WN / 64; ++q) *reinterpret_cast<uint16_t *>(smem + sc + Cfg::WM * 4 + Cfg::WN * 4 + (q * 64 + lane) * 2) = bias_reg[q];
            }
        }
        tile_c = reinterpret_cast<char *>(p.C) + ((size_t)c_m0 * ldc + c_n0) * ESZ;
        k_step(std::integral_constant<int, 1>{}, std::false_type{}, std::integral_constant<int, mode>{});
        static_for<0, FN>([&](auto j_) __attribute__((always_inline)) { mfma16_settle(acc[FM - 1][decltype(j_)::value]); });
        static_for<0, 4 * NH>([&](auto t_) __attribute__((always_inline)) {
            constexpr int t = decltype(t_)::value;
            write_half(std::integral_constant<int, FM - 1>{}, std::integral_constant<int, t / 4>{}, std::integral_constant<int, t % 4>{}, std::integral_constant<bool, edge>{});
            __builtin_amdgcn_sched_barrier(0);
        });
        store_half(std::integral_constant<int, FM - 1>{}, std::integral_constant<int, NH - 1>{}, std::integral_constant<int, 0>{}, std::integral_constant<bool, edge>{});
        store_half(std::integral_constant<int, FM - 1>{}, std::integral_constant<int, NH - 1>{}, std::integral_constant<int, 1>{}, std::integral_constant<bool, edge>{});
        if constexpr (!Cfg::OWN_AREA) {
            // every wave is done with its area: the loads of B that the last step left out
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            load_b(b_ring[0]);
            swap_b();
            cursor_advance();
        }
        next_item(min(c_item + G, nitems - 1));
    };
    for (; c_item < nwhole; c_item += G) run_item(std::integral_constant<int, 1>{});
    for (; c_item < nitems; c_item += G) run_item(std::integral_constant<int, 2>{});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

}  // namespace qm

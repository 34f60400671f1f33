// C ABI of libqm_hip.so (include/qm_abi.h): argument checks, configuration
// choice and launches.  Takes the place of the reference's host side:
// wrapper (kernel.cu:334-385), LAUNCH_KERNEL_IF_CONDITION (kernel.cu:321-332)
// and launch_igemm (kernel.cu:268-289).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <mutex>

#include "../../include/qm_abi.h"
#include "qm_launch.hpp"
#include "qm_skinny.hpp"
#include "qm_skinny_dma.hpp"
#include "qm_ragged.hpp"
#include "qm_aux.hpp"
#include "qm_expand6.hpp"
#include "qm_dot_linear.hpp"
#include "qm_skinny_linear.hpp"

#define QM_EXPORT extern "C" __attribute__((visibility("default")))

namespace qm {

// --------------------------------------------------------------------------
// Launchers of the skinny and dot kernels
// --------------------------------------------------------------------------
template <class Cfg>
static hipError_t launch_skinny(const GemmArgs &p, hipStream_t stream, int opt)
{
    if (opt & QM_OPT_PREPARE) return hipSuccess;  // static LDS, nothing to set up
    const int blocks = (p.N + Cfg::BN - 1) / Cfg::BN;
    // More column blocks than two workgroups per CU can hold at once, and K within one turn
    // of the waves: workgroups that walk over several blocks each, evenly.
    constexpr int resident = 2 * 256;
    if constexpr (Cfg::U % 2 == 0) {
        if (blocks > resident && (p.K + 127) / 128 <= Cfg::NW * Cfg::U) {
            const int turns = (blocks + resident - 1) / resident;
            return enqueue(&gemm_skinny_stream_kernel<Cfg>, dim3((blocks + turns - 1) / turns), dim3(Cfg::THREADS), 0, stream, p, blocks);
        }
    }
    return enqueue(&gemm_skinny_kernel<Cfg>, dim3(blocks), dim3(Cfg::THREADS), 0, stream, p);
}
#define QM_SKINNY(FM, FN, NW, U) \
    hipError_t QM_SKINNY_FN(FM, FN, NW, U)(const GemmArgs &p, hipStream_t s, int gm) { return launch_skinny<SkinnyCfg<FM, FN, NW, U>>(p, s, gm); }
template <class Cfg>
static hipError_t launch_dot(const GemmArgs &p, hipStream_t stream, int opt)
{
    if (opt & QM_OPT_PREPARE) return hipSuccess;
    const int blocks = (p.N + Cfg::BN - 1) / Cfg::BN;
    static_assert(8192 / 128 % (Cfg::NW * Cfg::U) == 0, "rows that go round are whole turns");
    const auto kernel = goes_round(p.M, p.N, p.K) ? &gemm_dot_kernel<Cfg, true> : &gemm_dot_kernel<Cfg, false>;
    static_assert(kernarg_bytes(&gemm_dot_kernel<Cfg, false>) <= 64, "see pack_rows_out");
    return enqueue(kernel, dim3(blocks), dim3(Cfg::THREADS), 0, stream, p.A, p.B, p.C, pack_rows_out(p.M, p.out), p.N, p.K, p.ldc, p.row_scale, p.col_scale, p.bias);
}
#define QM_DOT(MR, FN, NW, U) \
    hipError_t QM_DOT_FN(MR, FN, NW, U)(const GemmArgs &p, hipStream_t s, int gm) { return launch_dot<DotCfg<MR, FN, NW, U>>(p, s, gm); }
template <class Cfg>
static hipError_t launch_skinny_dma(const GemmArgs &p, hipStream_t stream, int opt)
{
    static std::atomic<bool> lds_ok[2][QM_MAX_DEVICES] = {};
    const bool prepare = (opt & QM_OPT_PREPARE) != 0, round = goes_round(p.M, p.N, p.K);
    const auto kernel = round ? &gemm_skinny_dma_kernel<Cfg, true> : &gemm_skinny_dma_kernel<Cfg, false>;
    hipError_t e = ensure_dynamic_lds(kernel, Cfg::LDS_BYTES, lds_ok[round]);
    if (e == hipSuccess && prepare) e = ensure_dynamic_lds(round ? &gemm_skinny_dma_kernel<Cfg, false> : &gemm_skinny_dma_kernel<Cfg, true>, Cfg::LDS_BYTES, lds_ok[!round]);
    if (e != hipSuccess || prepare) return e;
    const int blocks = (p.N + Cfg::BN - 1) / Cfg::BN, row_blocks = (p.M + Cfg::MAX_M - 1) / Cfg::MAX_M;
    if (row_blocks > 65535) return hipErrorInvalidValue;
    static_assert(kernarg_bytes(&gemm_skinny_dma_kernel<Cfg, true>) <= 64, "see pack_rows_out");
    return enqueue(kernel, dim3(skinny_dma_columns(blocks, row_blocks), row_blocks), dim3(Cfg::THREADS), Cfg::LDS_BYTES, stream,
        p.A, p.B, p.C, pack_rows_out(p.M, p.out), p.N, p.K, p.ldc, p.row_scale, p.col_scale, p.bias);
}
template <class Cfg>
static hipError_t launch_skinny_stream_dma(const GemmArgs &p, hipStream_t stream, int opt)
{
    // (rows of 4096 bytes fit the waves of some only)
    constexpr bool CAN_ROUND = Cfg::MAX_K >= 8192;
    static std::atomic<bool> lds_ok[2][QM_MAX_DEVICES] = {};
    const bool round = CAN_ROUND && goes_round(p.M, p.N, p.K);
    const auto kernel = round ? &gemm_skinny_stream_dma_kernel<Cfg, CAN_ROUND> : &gemm_skinny_stream_dma_kernel<Cfg, false>;
    hipError_t e = ensure_dynamic_lds(kernel, Cfg::LDS_BYTES, lds_ok[round]);
    if (e == hipSuccess && CAN_ROUND && (opt & QM_OPT_PREPARE))
        e = ensure_dynamic_lds(round ? &gemm_skinny_stream_dma_kernel<Cfg, false> : &gemm_skinny_stream_dma_kernel<Cfg, CAN_ROUND>, Cfg::LDS_BYTES, lds_ok[!round]);
    if (e != hipSuccess) return e;
    int cus = 0;
    e = device_cus(&cus);
    if (e != hipSuccess) return e;
    if (opt & QM_OPT_PREPARE) return hipSuccess;
    const int blocks = (p.N + Cfg::BN - 1) / Cfg::BN;
    const int resident = cus * (160 * 1024 / Cfg::LDS_BYTES);  // workgroups the device holds at once (the LDS decides)
    const int grid = blocks < resident ? blocks : resident;
    static_assert(kernarg_bytes(&gemm_skinny_stream_dma_kernel<Cfg, false>) <= 64, "see pack_rows_out");
    return enqueue(kernel, dim3(grid), dim3(Cfg::THREADS), Cfg::LDS_BYTES, stream,
        p.A, p.B, p.C, p.out | (p.M << 2) | (grid << 8), p.N, p.K, p.ldc, p.row_scale, p.col_scale, p.bias);
}
#define QM_SKINNYP(FM, FN, NW, D, R) \
    hipError_t QM_SKINNYP_FN(FM, FN, NW, D, R)(const GemmArgs &p, hipStream_t s, int gm) { return launch_skinny_stream_dma<SkinnyStreamCfg<FM, FN, NW, D, R>>(p, s, gm); }
#define QM_SKINNYD(FM, FN, NW, D) \
    hipError_t QM_SKINNYD_FN(FM, FN, NW, D)(const GemmArgs &p, hipStream_t s, int gm) { return launch_skinny_dma<SkinnyDmaCfg<FM, FN, NW, D>>(p, s, gm); }
#include "qm_configs.inc"

}  // namespace qm

#include "qm_select.hpp"

namespace qm {

static thread_local int g_last_hip_error = 0;

static int ptr_alignment(const void *a, const void *b)
{
    const uintptr_t x = (uintptr_t)a | (uintptr_t)b;
    if (x == 0) return 4096;
    const uintptr_t low = x & (~x + 1);
    return low > 4096 ? 4096 : (int)low;
}

static int check_gemm_args(const void *A, const void *B, void *C, int m, int n, int k)
{
    if (m < 0 || n < 0 || k < 0 || (k & 1)) return QM_ERR_SHAPE;
    if (m == 0 || n == 0) return QM_OK;
    if (!C) return QM_ERR_NULL;
    if ((uintptr_t)C & 3) return QM_ERR_ALIGN;
    if (k > 0 && (!A || !B)) return QM_ERR_NULL;
    return QM_OK;
}

static int fail_launch(hipError_t e)
{
    g_last_hip_error = (int)e;
    return QM_ERR_LAUNCH;
}

// The splits of K that have work (with kps K-steps per split only ceil(kt / kps) have any)
// and the workspace they fill: one padded tile of int32 per (split, tile).
static int effective_ksplit(const ConfigDesc &d, int k, int ksplit)
{
    if (d.kind != KIND_TILE16 || ksplit <= 1) return 1;
    return normalised_ksplit(k, ksplit);
}

static size_t split_workspace_bytes(const ConfigDesc &d, int m, int n, int ksplit)
{
    const size_t tiles = (size_t)((m + d.bm - 1) / d.bm) * (size_t)((n + d.bn - 1) / d.bn);
    return tiles * (size_t)ksplit * (size_t)d.bm * (size_t)d.bn * sizeof(int32_t);
}

static bool workspace_fits(const ConfigDesc &d, int m, int n, int ksplit, const void *ws, size_t ws_bytes)
{
    return ws != nullptr && ((uintptr_t)ws & 15) == 0 && ws_bytes >= split_workspace_bytes(d, m, n, ksplit);
}

// The automatic choice where none of the aligned kernels takes the operands (the "generic"
// configuration: K % 32 != 0, or A or B not 16-byte aligned): the matrix-core kernel of
// qm_ragged.hpp if K and the operands' sizes are within what it addresses -- else, as for an
// explicit "generic", one thread per element.
static bool ragged_fits(int m, int n, int k)
{
    const long long kb = k / 2;
    return k >= 32 && k <= QM_MAX_K_X16 && (long long)m * kb < 0x7fffffffLL && (long long)n * kb < 0x7fffffffLL && (m + 15) / 16 <= 65535;
}

// Blocks of 16 fm rows and 16 fn columns of C, nw waves over K with u chunks in flight each: the largest block that
// leaves more than half of the 256 CUs a workgroup of their own.  It reads (rows + columns) x K / 2
// bytes per rows x columns of C, but a workgroup's time is its K loop and an idle CU helps nobody.
// us, on blocks of 2x1, 2x2, 4x2 and 4x4 times 16: 17 x 3307 x 4100 10.0, 13.2, 15.4, 21.8; 64 x 3307 x 4100 23.0, 16.1,
// 23.5, 30.1; 200 x 3307 x 4100 59, 43, 44, 31; 100 x 1001 x 1002 3.5, 4.2, 5.3, 6.7; 64 x 9000 x 9000 64, 45, 53, 34.  Up
// to 16 rows, 1x1 and 1x2: 16 x 3307 x 4100 8.9, 12.1; 16 x 5001 x 2050 9.5, 7.8.  One thread per element, which
// these calls used to run on: 1 x 9000 x 9000 264 us (here 14.5), 16 x 700 x 8998 195 (12.6), 64 x 1001 x 1002 19 (3.4).
struct RaggedBlock {
    int fm, fn, nw, u;
    long long count(int m, int n) const { return (long long)((n + 16 * fn - 1) / (16 * fn)) * ((m + 16 * fm - 1) / (16 * fm)); }
};
static RaggedBlock ragged_block(int m, int n)
{
    const auto crowded = [&](const RaggedBlock &b) { return b.count(m, n) > 128; };
    if (m <= 16) return crowded({1, 2, 8, 2}) ? RaggedBlock{1, 2, 8, 2} : RaggedBlock{1, 1, 16, 2};
    if (m > 32 && crowded({4, 4, 8, 1})) return {4, 4, 8, 1};
    if (m > 32 && crowded({4, 2, 8, 2})) return {4, 2, 8, 2};
    return crowded({2, 2, 8, 2}) ? RaggedBlock{2, 2, 8, 2} : RaggedBlock{2, 1, 16, 2};
}

// With a workspace a large product can also run on zero-padded copies of A and B on the aligned kernels.
// The faster of the two by what each costs (us), fitted to 3800 products of 1 to 1500 rows, timed both ways with B from HBM
// and from the caches (rms of the fits 11 % here, 8 and 13 % on the copies), and for rows off the multiples of four to 21587, with B from HBM,
// since those are loaded as shifted dwords (7 and 10 %):
//   - here it is the loads: every wave's 16 bytes per lane of the rows of a block go through the L1 of its CU, 0.66 clocks
//     a lane where rows lie on multiples of four bytes and 1.18 where they do not (a dword more each); up to 0.07 x 5.5
//     more where they lie within five bytes of a multiple of 128 from row to row, so that the rows of a block
//     meet in the same banks.  Rows of a block beyond m are copies of the last one and cost next to nothing.  Workgroups
//     beyond one per CU count whole rounds;
//   - on copies, two launches, the rows of both operands read, written and read again, and the GEMM.
// One or two rows never take the copies, which are as large as the weights and at most a fifth faster there.  Above
// 512 rows only small products are left here (809 x 708 x 1096 5.2 / 8.6, 939 x 1094 x 1596 17.7 / 12.7), to 1500 rows off the multiples of four, where the
// rule was measured.  What the loads as they were before, at 1.94 and 0.35 clocks, left to the copies has to be a twentieth below them, an eighth where
// the fits are furthest off: few blocks on a long K, whose GEMM on the copies is one short round (93 x 799 x 6400 at an odd address 10.3 / 7.9), and several rounds of a few
// chunks (76 x 16590 x 448 11.2 / 9.7).  On 5578 others, time against that choice of before: 0.778 in the mean where it is another, 10 of those more than 2 % slower (2 more than 10: 127 x
// 40507 x 5898 79.0 -> 94.7).
static bool ragged_before_copies(int m, int n, int k, int ptr_align)
{
    if (m <= 2) return true;
    const bool dwords = k / 2 % 4 == 0 && ptr_align >= 4;
    const RaggedBlock b = ragged_block(m, n);
    const int kb = k / 2, off = std::min(kb % 128, 128 - kb % 128), kp = (k + 127) / 128 * 128;
    const double chunks = (kb + 63) / 64, out = 4e-6 * m * n, rounds = (double)((b.count(m, n) + 255) / 256);
    const double rows16 = std::min(m / 16.0, (double)b.fm) + b.fn, near_line = std::max(0.0, 5.5 - off);
    const auto here = [&](double l1_clocks) {
        return 1.56 + 0.33 * (double)(((kb + 63) / 64 + b.nw * b.u - 1) / (b.nw * b.u)) + 0.06e-6 * n * kb + 0.62 * out
               + rounds * chunks * (64 * rows16 * l1_clocks + 6 * b.fm * b.fn) / 2400;
    };
    const double moved = 1e-6 * ((double)m + n) * (kp / 2), mfma = 2.0 * m * n * kp / 4.5e9, steps = kp / 128;
    const double copies = m <= 64 ? 5.35 + 0.425 * moved + 0.025 * steps + 0.54 * out + 1.9 * mfma : 6.7 + 0.52 * moved + 0.034 * steps + 0.18 * out + 1.66 * mfma;
    const bool small = m <= 512 || (long long)m * n * k < (1LL << 29);
    if (small && here(dwords ? 0.66 : 1.94 + 0.35 * near_line) < copies) return true;
    if (dwords || m > 1500) return false;
    const double shifted_copies = m <= 64 ? 5.06 + 0.45 * moved + 0.0242 * steps + 0.656 * out + 1.553 * mfma : 5.41 + 0.4224 * moved + 0.0325 * steps + 0.279 * out + 2.546 * mfma;
    const bool few_long = (long long)((m + 31) / 32) * ((n + 31) / 32) <= 128 && k > 5000, many_short = k <= 640 && rounds >= 2;
    return here(1.18 + 0.072 * near_line) < (few_long || many_short ? 0.87 : 0.95) * shifted_copies;
}

// Automatic choice only: K padded to a multiple of 128 (operands copied into the workspace) so
// that the pipelined kernel can run instead of the generic one.  Worth it when the shape is
// large -- the copy is (M + N) K / 2 bytes twice over -- and the kernel for operands at any
// address is not the faster one.  `direct` is the choice without padding.  The size of the
// workspace (qm_gemm_workspace_bytes) and the launch (run_gemm) both come from this plan: a
// call is never asked for memory that it then leaves alone.
struct PadPlan {
    bool on = false;
    int kp = 0;
    Choice ch{};
    size_t a_bytes = 0, b_bytes = 0;
    size_t bytes() const { return a_bytes + b_bytes; }
};

static PadPlan plan_padded_k(int m, int n, int k, int ptr_align, const Choice &direct)
{
    PadPlan pl;
    const int kind = g_configs[direct.cfg].kind;
    if (kind == KIND_TILE16 || kind == KIND_SKINNY) return pl;
    const int kp = (k + 127) / 128 * 128;
    const long long outs = (long long)m * n;
    // (kp: a K below one K-step counts as the step it is padded to.  Before the costs, which are worked out
    // twice a call, 30 to 50 ns each time: small products are bound by the host)
    if (outs * kp < (1LL << 27)) return pl;
    if (ragged_fits(m, n, k) && ragged_before_copies(m, n, k, ptr_align)) return pl;
    if (kp > QM_MAX_K_X16 || !fast_path_ok(m, n, kp, 256)) return pl;
    Choice ch = heuristic(m, n, kp, 256, false);
    if (g_configs[ch.cfg].kind == KIND_GENERIC) return pl;
    ch.ksplit = 1;
    pl.on = true;
    pl.kp = kp;
    pl.ch = ch;
    pl.a_bytes = ((size_t)m * (kp / 2) + 255) / 256 * 256;
    pl.b_bytes = ((size_t)n * (kp / 2) + 255) / 256 * 256;
    return pl;
}

// Rows on multiples of four: they are loaded as they are, others as shifted dwords (Shifted16).
static bool rows_on_dwords(const GemmArgs &p) { return (((uintptr_t)p.A | (uintptr_t)p.B | (uintptr_t)(p.K >> 1)) & 3) == 0; }

// The padded copies of A and B in the workspace, and the arguments of the GEMM on them.
static hipError_t launch_padded(GemmArgs &p, const PadPlan &pl, void *ws, hipStream_t s)
{
    uint8_t *a_p = static_cast<uint8_t *>(ws), *b_p = a_p + pl.a_bytes;
    const PadRowsArgs q{p.A, p.B, reinterpret_cast<v4i *>(a_p), reinterpret_cast<v4i *>(b_p), p.M, p.N, p.K / 2, pl.kp / 32};
    const long long pieces = ((long long)p.M + p.N) * q.ppr;
    const hipError_t e = enqueue(&pad_rows_kernel, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, s, q);
    if (e != hipSuccess) return e;
    p.A = a_p;
    p.B = b_p;
    p.K = pl.kp;
    return hipSuccess;
}

// The same product on the tile kernel for 6-bit floats (qm_tile6.hpp), A re-coded in the workspace ahead of it.
static bool fp6_fits(int m, int n, int k, int ptr_align)
{
    if (k < 256 || k > QM_MAX_K_FP6 || !fast_path_ok(m, n, k, ptr_align)) return false;
    return n >= 256 && n < (1 << 21) && fp6_layout(m, k).code_bytes <= QM_FP6_MAX_BYTES;
}

// What the GEMM takes (us), in the terms of modelled_us: fitted to 272 products of 200 to 8192 rows (rms of the fits 7.5 and 6.3 %), before A's codes
// were read in whole 16-byte pieces, which is 1.5 to 4 % less; the terms of fp6_route for the codes are from before that too (up to 2 us less now).  Per K-step
// and round 0.82 us on tiles of 256 x 256 (int8: 1.19) and 0.53 on 256 x 128 (0.72), per round 13.8 and 5.8.
static double fp6_tile_us(int m, int n, int k, bool narrow)
{
    const double kt = (k + 127) / 128, share = (double)((m + 255) / 256) * (double)((n + (narrow ? 127 : 255)) / (narrow ? 128 : 256)) / 256;
    const double rounds = 0.75 * std::ceil(share) + 0.25 * std::max(1.0, share), fill = std::min(1.0, share);
    if (narrow) return kt * (rounds * (k & 255 ? 0.4774 : 0.4506) + fill * 0.0829) + rounds * 5.82 + 1.04;
    return kt * (rounds * (k & 255 ? 0.5784 : 0.5042) + fill * 0.3183) + rounds * 13.83 - 2.94;
}

// Automatic choice: where the better of the two tiles, with what its operands cost more than those of the int8 configuration
// `direct`, is 5 % below what the model says of that.  A K split of the int8 tiles counts with what it costs.  What A's codes cost, by
// where they come from (us; fitted to the same calls timed both ways):
//   FP6_FROM_PACKED  a launch of its own: 4.7 and 0.17 per million elements of A;
//   FP6_FROM_COPY    the launch that would copy both operands re-codes A instead: 0.5 and 0.3 per thousand rows more;
//   FP6_FROM_X       the layer's quantisation writes codes instead of packed rows: 0.15 per million elements more.
// The model's term for an N that is no multiple of four is left out: the int8 tiles have since come to lose a few percent on
// such a C, the term says twenty.  One round of 256 x 128 that is more than half full has to be 10 % below: with most CUs at
// work it loses more than the model says.  Below a K of 512, or of 1280 from packed rows, it gains nothing.
// Measured against the int8 choice, B from HBM: from packed rows, 2450 products, taken on 2190 and 0.83 of the time in the mean,
// six more than 2 % slower (5 %; 2816 x 2635 x 2112, once taken, 22.3 / 26.5 us); copied, 1260, 0.81 on 1105, three (4 %; 5386 x
// 938 x 1066, once taken, 19.0 / 23.7); layers, 460, 0.82 on 425, one (2 %; 4381 x 951 x 15232, once taken, 99 / 117).  A wider
// margin loses gains of 8 % on average on ten times the calls it saves from a loss.  us, int8 / here: 8192 x 8192 x 8192
// 356 / 297, 1280 x 8192 x 14336 124 / 91, 512 x 28672 x 4096 45.8 / 41.9.
// (The bound on the product comes first: calls that the host bounds do not get as far as the model.)
enum Fp6Route { FP6_NO = 0, FP6_WIDE, FP6_NARROW };
enum Fp6Source { FP6_FROM_PACKED, FP6_FROM_COPY, FP6_FROM_X };
static Fp6Route fp6_route(int m, int n, int k, int ptr_align, const Choice &direct, Fp6Source source)
{
    if ((double)m * n * k < 4e9 || m < 200 || k < (source == FP6_FROM_PACKED ? 1280 : 512) || !fp6_fits(m, n, k, ptr_align)) return FP6_NO;
    const CostFit *f = fit_of(direct.cfg);
    if (f == nullptr) return FP6_NO;  // (the choices for up to 64 rows and the any-address ones have none: neither gets here)
    const double wide = fp6_tile_us(m, n, k, false), narrow = fp6_tile_us(m, n, k, true);
    const double codes = source == FP6_FROM_PACKED ? 4.68 + 0.1685e-6 * m * k : source == FP6_FROM_COPY ? 0.5 + 0.3e-3 * m : 0.15e-6 * m * k;
    const long long tiles = (long long)((m + 255) / 256) * ((n + 127) / 128);
    const double margin = narrow < wide && tiles > 128 && tiles <= 256 ? 0.90 : 0.95;
    if (std::min(wide, narrow) + codes >= margin * modelled_us(*f, g_configs[direct.cfg], m, (n + 3) & ~3, k, direct.ksplit)) return FP6_NO;
    return narrow < wide ? FP6_NARROW : FP6_WIDE;
}
static Fp6Route fp6_asked_for(int cfg) { return cfg == QM_CFG_RECODE ? FP6_WIDE : cfg == QM_CFG_RECODE_NARROW ? FP6_NARROW : FP6_NO; }

static auto tile6_launcher(int out) { return out == OUT_I32 ? &launch_tile6_i32 : out == OUT_F16 ? &launch_tile6_f16 : &launch_tile6_bf16; }

static hipError_t launch_tile6(const GemmArgs &p, const Fp6Operand &a, Fp6Route route, hipStream_t s)
{
    return tile6_launcher(p.out)(p, a, s, route == FP6_NARROW ? QM_OPT_NARROW : 0);
}

static hipError_t launch_fp6(const GemmArgs &p, Fp6Route route, void *ws, hipStream_t s)
{
    const Fp6Operand a = fp6_operand(p.M, p.K, ws);
    const Fp6Layout &l = a.layout;
    const Expand6Args q{p.A, a.codes, a.sums, p.M, p.K, l.kt, l.groups, l.parts};
    const int rows = expand_rows(p.M, p.K);
    const auto kernel = rows == 16 ? &expand_a6_kernel<false, false, 16> : &expand_a6_kernel<false, false, 8>;
    const hipError_t e = enqueue(kernel, dim3(l.groups * (32 / rows) * l.parts), dim3(EXPAND6_THREADS), 0, s, q);
    return e == hipSuccess ? launch_tile6(p, a, route, s) : e;
}

// The same where the operands would be copied (plan_padded_k): A's codes as of rows padded to kp, and the copy of B, in one launch.
static size_t fp6_padded_bytes(int m, int kp, const PadPlan &pl) { return (fp6_layout(m, kp).bytes + 255) / 256 * 256 + pl.b_bytes; }
static hipError_t launch_fp6_padded(GemmArgs p, const PadPlan &pl, Fp6Route route, void *ws, hipStream_t s)
{
    const Fp6Operand a = fp6_operand(p.M, pl.kp, ws);
    uint8_t *b_copy = static_cast<uint8_t *>(ws) + fp6_padded_bytes(p.M, pl.kp, pl) - pl.b_bytes;
    const Fp6Layout &l = a.layout;
    const Expand6Args q{p.A, a.codes, a.sums, p.M, p.K, l.kt, l.groups, l.parts, p.B, reinterpret_cast<v4i *>(b_copy), p.N, pl.kp};
    const long long pieces = (long long)p.N * (pl.kp / 32);
    const int rows = expand_rows(p.M, pl.kp);
    const auto kernel = rows_on_dwords(p) ? (rows == 16 ? &expand_a6_kernel<true, false, 16> : &expand_a6_kernel<true, false, 8>)
                                          : (rows == 16 ? &expand_a6_kernel<true, true, 16> : &expand_a6_kernel<true, true, 8>);
    const hipError_t e = enqueue(kernel, dim3(l.groups * (32 / rows) * l.parts + (unsigned)((pieces + EXPAND6_THREADS - 1) / EXPAND6_THREADS)), dim3(EXPAND6_THREADS), 0, s, q);
    if (e != hipSuccess) return e;
    p.B = b_copy;
    p.K = pl.kp;
    return launch_tile6(p, a, route, s);
}

template <class Cfg>
static hipError_t launch_ragged(const GemmArgs &p, hipStream_t s)
{
    const dim3 grid((p.N + Cfg::BN - 1) / Cfg::BN, (p.M + Cfg::MAX_M - 1) / Cfg::MAX_M);
    const auto kernel = rows_on_dwords(p) ? &gemm_ragged_kernel<Cfg, false> : &gemm_ragged_kernel<Cfg, true>;
    return enqueue(kernel, grid, dim3(Cfg::THREADS), 0, s, p.A, p.B, p.C, p.M, p.N, p.K, p.ldc, p.out, p.row_scale, p.col_scale, p.bias);
}

static hipError_t launch_ragged(const GemmArgs &p, hipStream_t s)
{
    const RaggedBlock b = ragged_block(p.M, p.N);
    if (b.fm == 1) return b.fn == 2 ? launch_ragged<RaggedCfg<1, 2, 8, 2>>(p, s) : launch_ragged<RaggedCfg<1, 1, 16, 2>>(p, s);
    if (b.fm == 4) return b.fn == 4 ? launch_ragged<RaggedCfg<4, 4, 8, 1>>(p, s) : launch_ragged<RaggedCfg<4, 2, 8, 2>>(p, s);
    return b.fn == 2 ? launch_ragged<RaggedCfg<2, 2, 8, 2>>(p, s) : launch_ragged<RaggedCfg<2, 1, 16, 2>>(p, s);
}

static Choice choice_from_code(int cfg)
{
    Choice ch;
    ch.cfg = cfg & 0xFFFF;
    ch.group_m = (cfg >> 16) & 0xFF;
    ch.ksplit = (cfg >> 24) & 0x3F;
    ch.spread = (cfg >> 30) & 1;
    if (ch.group_m == 0) ch.group_m = 4;
    if (ch.ksplit == 0) ch.ksplit = 1;
    return ch;
}

// GEMM with K split into ch.ksplit (> 1, normalised) through the workspace, then the sum of
// the splits into C in the output form p.out.
static hipError_t launch_split_with_workspace(GemmArgs p, const Choice &ch, void *ws, hipStream_t s)
{
    const ConfigDesc &d = g_configs[ch.cfg];
    SplitReduceArgs q;
    q.ws = static_cast<const v4i *>(ws);
    q.C = p.C;
    q.M = p.M;
    q.N = p.N;
    q.tiles_m = (p.M + d.bm - 1) / d.bm;
    q.tiles_n = (p.N + d.bn - 1) / d.bn;
    q.group_m = ch.group_m < 1 ? 1 : (ch.group_m > q.tiles_m ? q.tiles_m : ch.group_m);  // as the launcher clamps it
    q.ksplit = ch.ksplit;
    q.BM = d.bm;
    q.BN = d.bn;
    q.WGN = d.wgn;
    q.FM = d.bm / d.wgm / 16;
    q.FN = d.bn / d.wgn / 16;
    q.waves = d.waves;
    q.row_scale = p.row_scale;
    q.col_scale = p.col_scale;
    q.bias = p.bias;
    q.out = p.out;
    p.out = OUT_I32;
    p.row_scale = p.col_scale = nullptr;
    p.bias = nullptr;
    p.ws = static_cast<int32_t *>(ws);
    hipError_t e = d.launch(p, s, ch.group_m | (ch.ksplit << 8) | (ch.spread << 16));
    if (e != hipSuccess) return e;
    const size_t pieces = (size_t)q.tiles_m * q.tiles_n * (size_t)(d.bm * d.bn / 4);
    if (pieces > 0x7fffff00ULL) return hipErrorInvalidValue;
    return enqueue(&splitk_reduce_kernel, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, s, q);
}

// Operands of this many bytes or more are cut into blocks (below).  2^31 - 1 in production: what
// the kernels' 32-bit row offsets reach.  qm_debug_set_operand_limit lowers it so that tests
// can drive the block paths -- C written through a row stride, blocks of rows then of columns --
// on small shapes.
static std::atomic<long long> g_operand_limit{0x7fffffffLL};

// An A of 2 GiB or more is beyond the 32-bit row offsets of the fast kernels; its row blocks
// are independent (block r0.. of A gives rows r0.. of C), so the call is cut into blocks
// of rows that fit, one after the other on the stream (they share the workspace).  Returns
// the rows per block, 0 when the call needs no cutting or cutting does not help (B too large
// as well, or a shape the fast kernels do not take anyway).
static int row_block_for_large_a(int m, int n, int k, int ptr_align)
{
    (void)n;
    if (k < 32 || k % 32 != 0 || k > QM_MAX_K_X16 || ptr_align < 16) return 0;
    const long long kb = k / 2, limit = g_operand_limit.load(std::memory_order_relaxed);
    if ((long long)m * kb < limit) return 0;
    const long long rows = ((limit - 1) / kb) & ~255LL;
    return rows >= 256 ? (int)rows : 0;
}

// The same for a B of 2 GiB or more (and an A that fits, or a row block of one): blocks of
// rows of B are blocks of columns of C, which the kernels write through a row stride.
static int col_block_for_large_b(int m, int n, int k, int ptr_align)
{
    if (k < 32 || k % 32 != 0 || k > QM_MAX_K_X16 || ptr_align < 16) return 0;
    const long long kb = k / 2, limit = g_operand_limit.load(std::memory_order_relaxed);
    if ((long long)n * kb < limit || (long long)m * kb >= limit) return 0;
    const long long cols = ((limit - 1) / kb) & ~255LL;
    return cols >= 256 ? (int)cols : 0;
}

// One GEMM call, arguments already checked (m, n >= 1, k even).  `out` is OUT_I32 with C in
// `dst`, or OUT_F16 / OUT_BF16 with the scaled and rounded D there.  The two differ in one
// place: a K split whose partial sums have no workspace to meet in falls back to atomic adds
// into a zero-filled C for int32, and is not taken at all for a rounded output.
static int run_gemm(const void *A, const void *B, void *dst, int m, int n, int k, const float *row_scale,
                    const float *col_scale, int out, hipStream_t s, int cfg, void *workspace, size_t workspace_bytes, int ldc = 0,
                    const uint16_t *bias = nullptr)
{
    const bool scaled = out != OUT_I32;
    const size_t cnt = (size_t)m * (size_t)n;
    const int row_stride = ldc != 0 ? ldc : n;   // of the output, in elements
    const bool strided = row_stride != n;        // a block of columns of a wider output
    if (k == 0) {
        const dim3 grid(flat_grid(cnt, 256)), block(256);
        const hipError_t e = scaled && bias ? enqueue(&fill_bias16_kernel, grid, block, 0, s, static_cast<uint16_t *>(dst), bias, n, row_stride, cnt, out)
                             : scaled       ? enqueue(&fill_zero16_kernel, grid, block, 0, s, static_cast<uint16_t *>(dst), cnt)
                                            : enqueue(&fill_zero_kernel, grid, block, 0, s, static_cast<int32_t *>(dst), cnt);
        return e == hipSuccess ? QM_OK : fail_launch(e);
    }
    const int align = ptr_alignment(A, B);
    if (const int rb = cfg == QM_CFG_AUTO ? row_block_for_large_a(m, n, k, align) : 0) {
        for (int r0 = 0; r0 < m; r0 += rb) {
            const int st = run_gemm(static_cast<const uint8_t *>(A) + (size_t)r0 * (size_t)(k / 2), B,
                                    static_cast<uint8_t *>(dst) + (size_t)r0 * (size_t)row_stride * (scaled ? 2 : 4), m - r0 < rb ? m - r0 : rb,
                                    n, k, row_scale ? row_scale + r0 : nullptr, col_scale, out, s, cfg, workspace, workspace_bytes, ldc, bias);
            if (st != QM_OK) return st;
        }
        return QM_OK;
    }
    if (const int cb = cfg == QM_CFG_AUTO ? col_block_for_large_b(m, n, k, align) : 0) {
        for (int c0 = 0; c0 < n; c0 += cb) {
            const int st = run_gemm(A, static_cast<const uint8_t *>(B) + (size_t)c0 * (size_t)(k / 2),
                                    static_cast<uint8_t *>(dst) + (size_t)c0 * (scaled ? 2 : 4), m, n - c0 < cb ? n - c0 : cb, k, row_scale,
                                    col_scale ? col_scale + c0 : nullptr, out, s, cfg, workspace, workspace_bytes, row_stride,
                                    bias ? bias + c0 : nullptr);
            if (st != QM_OK) return st;
        }
        return QM_OK;
    }
    const bool has_ws = workspace != nullptr && workspace_bytes > 0;
    GemmArgs p{static_cast<const uint8_t *>(A), static_cast<const uint8_t *>(B), static_cast<int32_t *>(dst), m, n, k};
    p.row_scale = row_scale;
    p.col_scale = col_scale;
    p.bias = bias;
    p.out = out;
    p.ldc = strided ? row_stride : 0;
    if (strided && cfg != QM_CFG_AUTO) return QM_ERR_CONFIG;
    if (const Fp6Route route = fp6_asked_for(cfg)) {
        if (!fp6_fits(m, n, k, align) || workspace == nullptr || ((uintptr_t)workspace & 15) || workspace_bytes < fp6_layout(m, k).bytes) return QM_ERR_CONFIG;
        const hipError_t e = launch_fp6(p, route, workspace, s);
        return e == hipSuccess ? QM_OK : fail_launch(e);
    }
    const auto launcher = [&](int id) { return scaled ? scaled_launcher(id) : g_configs[id].launch; };
    Choice ch;
    if (strided) {
        // one launch straight into the wider output: no K split (its partial sums are added up
        // into a contiguous C) and no padded copies
        ch = scaled ? select_scaled(m, n, k, align, false) : select_config(m, n, k, align, false);
        ch.ksplit = 1;
        const LaunchFn launch = launcher(ch.cfg);
        if (!launch) return QM_ERR_CONFIG;
        const hipError_t e = launch(p, s, ch.group_m | (1 << 8) | (ch.spread << 16));
        return e == hipSuccess ? QM_OK : fail_launch(e);
    }
    if (cfg == QM_CFG_AUTO) {
        ch = scaled ? select_scaled(m, n, k, align, has_ws) : select_config(m, n, k, align, has_ws);
    } else {
        ch = choice_from_code(cfg);
        if (!config_supports(ch.cfg, m, n, k, align)) return QM_ERR_CONFIG;
        if (ch.ksplit > 1 && g_configs[ch.cfg].kind != KIND_TILE16) return QM_ERR_CONFIG;
    }
    ch.ksplit = effective_ksplit(g_configs[ch.cfg], k, ch.ksplit);
    const bool auto_ws = cfg == QM_CFG_AUTO && has_ws && ((uintptr_t)workspace & 15) == 0;
    if (auto_ws) {
        const Fp6Route route = fp6_route(m, n, k, align, ch, FP6_FROM_PACKED);
        if (route && workspace_bytes >= fp6_layout(m, k).bytes) {
            const hipError_t e = launch_fp6(p, route, workspace, s);
            return e == hipSuccess ? QM_OK : fail_launch(e);
        }
    }
    if (ch.ksplit > 1 && workspace_fits(g_configs[ch.cfg], m, n, ch.ksplit, workspace, workspace_bytes)) {
        const hipError_t e = launch_split_with_workspace(p, ch, workspace, s);
        return e == hipSuccess ? QM_OK : fail_launch(e);
    }
    if (ch.ksplit > 1 && scaled) {
        // partial sums cannot meet in a rounded output: without the workspace, no split
        if (cfg != QM_CFG_AUTO) return QM_ERR_CONFIG;
        ch = select_scaled(m, n, k, align, false);
        ch.ksplit = 1;
    }
    if (cfg == QM_CFG_AUTO && has_ws) {
        PadPlan pl = plan_padded_k(m, n, k, align, ch);
        if (pl.on && auto_ws) {
            const Fp6Route route = fp6_route(m, n, pl.kp, 256, pl.ch, FP6_FROM_COPY);
            if (route && workspace_bytes >= fp6_padded_bytes(m, pl.kp, pl)) {
                const hipError_t e = launch_fp6_padded(p, pl, route, workspace, s);
                return e == hipSuccess ? QM_OK : fail_launch(e);
            }
        }
        if (pl.on && !launcher(pl.ch.cfg)) {
            // a pipelined configuration that has the scaled output, if the shape is one for those
            const int id = find_config("q256x256_w2x2_s9o1");
            if (id >= 0 && launcher(id)) pl.ch.cfg = id; else pl.on = false;
        }
        if (pl.on && ((uintptr_t)workspace & 15) == 0 && workspace_bytes >= pl.bytes()) {
            hipError_t e = launch_padded(p, pl, workspace, s);
            if (e == hipSuccess) e = launcher(pl.ch.cfg)(p, s, pl.ch.group_m | (1 << 8) | (pl.ch.spread << 16));
            return e == hipSuccess ? QM_OK : fail_launch(e);
        }
    }
    if (cfg == QM_CFG_AUTO && g_configs[ch.cfg].kind == KIND_GENERIC && ragged_fits(m, n, k)) {
        const hipError_t e = launch_ragged(p, s);
        return e == hipSuccess ? QM_OK : fail_launch(e);
    }
    if (ch.ksplit > 1) {
        // int32, no workspace: the partial sums meet in C by integer atomic adds, C starts from zero
        const hipError_t ez = enqueue(&fill_zero_kernel, dim3(flat_grid(cnt, 256)), dim3(256), 0, s, static_cast<int32_t *>(dst), cnt);
        if (ez != hipSuccess) return fail_launch(ez);
    }
    const LaunchFn launch = launcher(ch.cfg);
    if (!launch) return QM_ERR_CONFIG;
    const hipError_t e = launch(p, s, ch.group_m | (ch.ksplit << 8) | (ch.spread << 16));
    return e == hipSuccess ? QM_OK : fail_launch(e);
}

}  // namespace qm

using namespace qm;

QM_EXPORT int qm_gemm_i4_ws(const void *A, const void *B, void *C, int m, int n, int k, void *stream, int cfg,
                            void *workspace, size_t workspace_bytes)
{
    const int st = check_gemm_args(A, B, C, m, n, k);
    if (st != QM_OK) return st;
    if (m == 0 || n == 0) return QM_OK;
    return run_gemm(A, B, C, m, n, k, nullptr, nullptr, OUT_I32, reinterpret_cast<hipStream_t>(stream), cfg, workspace, workspace_bytes);
}

// Every one-off set-up a first launch on the current device would otherwise do.
QM_EXPORT int qm_init(void)
{
    GemmArgs p{nullptr, nullptr, nullptr, 256, 256, 256};
    const uint16_t no_bias = 0;
    for (int id = 0; id < g_num_configs; ++id) {
        if (g_configs[id].kind == KIND_GENERIC) continue;
        for (const int k : {256, 256 + 32}) {   // the kernel for whole K-steps and the one with a short last step
            p.K = k;
            for (const int out : {(int)OUT_I32, (int)OUT_F16, (int)OUT_BF16}) {
                const LaunchFn fn = out == OUT_I32 ? g_configs[id].launch : scaled_launcher(id);
                if (!fn || (out != OUT_I32 && g_configs[id].kind != KIND_TILE16)) continue;
                p.out = out;
                for (const uint16_t *bias : {(const uint16_t *)nullptr, &no_bias}) {   // (nothing is launched, nor read)
                    p.bias = out == OUT_I32 ? nullptr : bias;
                    const hipError_t e = fn(p, nullptr, QM_OPT_PREPARE);
                    if (e != hipSuccess) return fail_launch(e);
                }
            }
        }
    }
    for (const int out : {(int)OUT_I32, (int)OUT_F16, (int)OUT_BF16})
        for (const uint16_t *bias : {(const uint16_t *)nullptr, &no_bias}) {
            p.bias = out == OUT_I32 ? nullptr : bias;
            for (const int tile : {0, QM_OPT_NARROW}) {
                const hipError_t e = tile6_launcher(out)(p, Fp6Operand{}, nullptr, QM_OPT_PREPARE | tile);
                if (e != hipSuccess) return fail_launch(e);
            }
        }
    hipError_t e = ready_skinny_linear<QM_IN_F16>();
    if (e == hipSuccess) e = ready_skinny_linear<QM_IN_BF16>();
    if (e != hipSuccess) return fail_launch(e);
    void *ws = nullptr;
    e = static_scratch(&ws);
    return e == hipSuccess ? QM_OK : fail_launch(e);
}

QM_EXPORT int qm_gemm_i4_static(const void *A, const void *B, void *C, int m, int n, int k, void *stream)
{
    const int st = check_gemm_args(A, B, C, m, n, k);
    if (st != QM_OK) return st;
    if (m == 0 || n == 0) return QM_OK;
    const size_t need = qm_gemm_workspace_bytes(m, n, k, ptr_alignment(A, B), QM_CFG_AUTO, 0);
    if (need > (size_t)QM_STATIC_SCRATCH_BYTES) return QM_ERR_SCRATCH;
    void *ws = nullptr;
    if (need > 0) {
        const hipError_t e = static_scratch(&ws);
        if (e != hipSuccess) return fail_launch(e);
    }
    return run_gemm(A, B, C, m, n, k, nullptr, nullptr, OUT_I32, reinterpret_cast<hipStream_t>(stream), QM_CFG_AUTO, ws, ws ? need : 0);
}

QM_EXPORT int qm_gemm_i4_cfg(const void *A, const void *B, void *C, int m, int n, int k, void *stream, int cfg)
{
    return qm_gemm_i4_ws(A, B, C, m, n, k, stream, cfg, nullptr, 0);
}

QM_EXPORT int qm_gemm_i4_scaled_bias_ws(const void *A, const void *B, void *D, int m, int n, int k, const float *row_scale,
                                        const float *col_scale, const void *bias, int out_dtype, void *stream, int cfg,
                                        void *workspace, size_t workspace_bytes)
{
    if (out_dtype != QM_OUT_F16 && out_dtype != QM_OUT_BF16) return QM_ERR_DTYPE;
    if (m < 0 || n < 0 || k < 0 || (k & 1)) return QM_ERR_SHAPE;
    if (m == 0 || n == 0) return QM_OK;
    if (!D) return QM_ERR_NULL;
    if (((uintptr_t)D & 1) || ((uintptr_t)bias & 1)) return QM_ERR_ALIGN;
    if (k > 0 && (!A || !B)) return QM_ERR_NULL;
    return run_gemm(A, B, D, m, n, k, row_scale, col_scale, out_dtype == QM_OUT_F16 ? OUT_F16 : OUT_BF16,
                    reinterpret_cast<hipStream_t>(stream), cfg, workspace, workspace_bytes, 0, static_cast<const uint16_t *>(bias));
}

QM_EXPORT int qm_gemm_i4_scaled_ws(const void *A, const void *B, void *D, int m, int n, int k, const float *row_scale,
                                   const float *col_scale, int out_dtype, void *stream, int cfg, void *workspace,
                                   size_t workspace_bytes)
{
    return qm_gemm_i4_scaled_bias_ws(A, B, D, m, n, k, row_scale, col_scale, nullptr, out_dtype, stream, cfg, workspace, workspace_bytes);
}

QM_EXPORT int qm_gemm_i4_scaled_cfg(const void *A, const void *B, void *D, int m, int n, int k, const float *row_scale,
                                    const float *col_scale, int out_dtype, void *stream, int cfg)
{
    return qm_gemm_i4_scaled_ws(A, B, D, m, n, k, row_scale, col_scale, out_dtype, stream, cfg, nullptr, 0);
}

QM_EXPORT int qm_gemm_i4_scaled(const void *A, const void *B, void *D, int m, int n, int k, const float *row_scale,
                                const float *col_scale, int out_dtype, void *stream)
{
    return qm_gemm_i4_scaled_ws(A, B, D, m, n, k, row_scale, col_scale, out_dtype, stream, QM_CFG_AUTO, nullptr, 0);
}

QM_EXPORT size_t qm_gemm_workspace_bytes(int m, int n, int k, int ptr_align, int cfg, int scaled)
{
    if (m < 1 || n < 1 || k < 2 || (k & 1)) return 0;
    if (const int rb = cfg == QM_CFG_AUTO ? row_block_for_large_a(m, n, k, ptr_align) : 0) {
        // the blocks run one after the other: the largest need of the two block sizes
        const size_t whole = qm_gemm_workspace_bytes(rb, n, k, ptr_align, cfg, scaled);
        const size_t rest = m % rb ? qm_gemm_workspace_bytes(m % rb, n, k, ptr_align, cfg, scaled) : 0;
        return whole > rest ? whole : rest;
    }
    if (cfg == QM_CFG_AUTO && col_block_for_large_b(m, n, k, ptr_align)) return 0;  // blocks of columns: one launch each, no workspace
    if (fp6_asked_for(cfg)) return fp6_fits(m, n, k, ptr_align) ? fp6_layout(m, k).bytes : 0;
    Choice ch;
    if (cfg == QM_CFG_AUTO) {
        ch = scaled ? select_scaled(m, n, k, ptr_align, true) : select_config(m, n, k, ptr_align, true);
    } else {
        ch = choice_from_code(cfg);
        if (!config_supports(ch.cfg, m, n, k, ptr_align)) return 0;
    }
    const int ks = effective_ksplit(g_configs[ch.cfg], k, ch.ksplit);
    if (ks > 1) return split_workspace_bytes(g_configs[ch.cfg], m, n, ks);
    if (cfg == QM_CFG_AUTO) {
        const PadPlan pl = plan_padded_k(m, n, k, ptr_align, ch);
        if (pl.on) return pl.bytes();
    }
    return 0;
}

// The tiles that a call with enough workspace runs on as 6-bit floats (or none), and that workspace.
static Fp6Route recode_route(int m, int n, int k, int ptr_align, int scaled, size_t *bytes)
{
    *bytes = 0;
    if (m < 1 || n < 1 || (double)m * n * k < 3.5e9 || (k & 1)) return FP6_NO;   // (padded to 128, a K that counts here is a sixth longer at most)
    if (row_block_for_large_a(m, n, k, ptr_align) || col_block_for_large_b(m, n, k, ptr_align)) return FP6_NO;
    Choice ch = scaled ? select_scaled(m, n, k, ptr_align, true) : select_config(m, n, k, ptr_align, true);
    ch.ksplit = effective_ksplit(g_configs[ch.cfg], k, ch.ksplit);
    if (const Fp6Route route = fp6_route(m, n, k, ptr_align, ch, FP6_FROM_PACKED)) {
        *bytes = fp6_layout(m, k).bytes;
        return route;
    }
    const PadPlan pl = plan_padded_k(m, n, k, ptr_align, ch);
    const Fp6Route route = pl.on ? fp6_route(m, n, pl.kp, 256, pl.ch, FP6_FROM_COPY) : FP6_NO;
    if (route) *bytes = fp6_padded_bytes(m, pl.kp, pl);
    return route;
}

QM_EXPORT size_t qm_gemm_recode_bytes(int m, int n, int k, int ptr_align, int scaled)
{
    size_t bytes;
    recode_route(m, n, k, ptr_align, scaled, &bytes);
    return bytes;
}

QM_EXPORT int qm_recode_config(int m, int n, int k, int ptr_align, int scaled)
{
    size_t bytes;
    const Fp6Route route = recode_route(m, n, k, ptr_align, scaled, &bytes);
    return route == FP6_WIDE ? QM_CFG_RECODE : route == FP6_NARROW ? QM_CFG_RECODE_NARROW : QM_CFG_AUTO;
}

QM_EXPORT int qm_config_has_scaled(int cfg)
{
    cfg &= 0xFFFF;
    return (cfg >= 0 && cfg < g_num_configs && scaled_launcher(cfg)) ? 1 : 0;
}

QM_EXPORT int qm_gemm_i4(const void *A, const void *B, void *C, int m, int n, int k, void *stream)
{
    return qm_gemm_i4_cfg(A, B, C, m, n, k, stream, QM_CFG_AUTO);
}

QM_EXPORT int qm_select_config(int m, int n, int k, int ptr_align)
{
    if (m < 1 || n < 1 || k < 2 || (k & 1)) return QM_ERR_SHAPE;
    const Choice ch = select_config(m, n, k, ptr_align, true);
    return ch.cfg | (ch.group_m << 16) | (ch.ksplit << 24) | (ch.spread << 30);
}

QM_EXPORT int qm_select_config_ex(int m, int n, int k, int ptr_align, int has_workspace, int scaled)
{
    if (m < 1 || n < 1 || k < 2 || (k & 1)) return QM_ERR_SHAPE;
    Choice ch = scaled ? select_scaled(m, n, k, ptr_align, has_workspace != 0) : select_config(m, n, k, ptr_align, has_workspace != 0);
    if (scaled && ch.ksplit > 1 && !has_workspace) {
        // as run_gemm: partial sums cannot meet in a rounded output
        ch = select_scaled(m, n, k, ptr_align, false);
        ch.ksplit = 1;
    }
    return ch.cfg | (ch.group_m << 16) | (ch.ksplit << 24) | (ch.spread << 30);
}

QM_EXPORT int qm_num_configs(void) { return g_num_configs; }

QM_EXPORT const char *qm_config_name(int cfg)
{
    cfg &= 0xFFFF;
    return (cfg >= 0 && cfg < g_num_configs) ? g_configs[cfg].name : nullptr;
}

QM_EXPORT int qm_config_supports(int cfg, int m, int n, int k, int ptr_align)
{
    return config_supports(cfg & 0xFFFF, m, n, k, ptr_align) ? 1 : 0;
}

QM_EXPORT int qm_pack_i4(const void *src_i8, void *dst_packed, int rows, int k, void *stream)
{
    if (rows < 0 || k < 0 || (k & 1)) return QM_ERR_SHAPE;
    const size_t nbytes = (size_t)rows * (size_t)(k / 2);
    if (nbytes == 0) return QM_OK;
    if (!src_i8 || !dst_packed) return QM_ERR_NULL;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    hipError_t e;
    if (nbytes >= 8) {
        const unsigned grid = flat_grid(nbytes, 8 * PACK_PIECES * PACK_THREADS, 1u << 22);
        e = enqueue(&pack_i4_vec_kernel, dim3((grid + PACK_APART - 1) / PACK_APART * PACK_APART), dim3(PACK_THREADS), 0, s,
            static_cast<const uint8_t *>(src_i8), static_cast<uint8_t *>(dst_packed), nbytes);
    } else {
        e = enqueue(&pack_i4_byte_kernel, dim3(flat_grid(nbytes, 256)), dim3(256), 0, s, static_cast<const uint8_t *>(src_i8), static_cast<uint8_t *>(dst_packed), nbytes);
    }
    return e == hipSuccess ? QM_OK : fail_launch(e);
}

QM_EXPORT int qm_quantize_pack_i4(const void *x, int in_dtype, void *dst_packed, float *scales, int rows, int k, void *stream)
{
    if (in_dtype != QM_IN_F16 && in_dtype != QM_IN_BF16 && in_dtype != QM_IN_F32) return QM_ERR_DTYPE;
    if (rows < 0 || k < 0 || (k & 1)) return QM_ERR_SHAPE;
    if (rows == 0) return QM_OK;
    if (!scales || (k > 0 && (!x || !dst_packed))) return QM_ERR_NULL;
    if (((uintptr_t)x & (in_dtype == QM_IN_F32 ? 3 : 1)) || ((uintptr_t)scales & 3)) return QM_ERR_ALIGN;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    hipError_t e;
    if (in_dtype == QM_IN_F16) e = launch_quantize_pack<QM_IN_F16>(x, dst_packed, scales, rows, k, s);
    else if (in_dtype == QM_IN_BF16) e = launch_quantize_pack<QM_IN_BF16>(x, dst_packed, scales, rows, k, s);
    else e = launch_quantize_pack<QM_IN_F32>(x, dst_packed, scales, rows, k, s);
    return e == hipSuccess ? QM_OK : fail_launch(e);
}

QM_EXPORT int qm_unpack_i4(const void *src_packed, void *dst_i8, int rows, int k, void *stream)
{
    if (rows < 0 || k < 0 || (k & 1)) return QM_ERR_SHAPE;
    const size_t nbytes = (size_t)rows * (size_t)(k / 2);
    if (nbytes == 0) return QM_OK;
    if (!src_packed || !dst_i8) return QM_ERR_NULL;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    hipError_t e;
    if (nbytes >= 8)
        e = enqueue(&unpack_i4_vec_kernel, dim3(flat_grid(nbytes, 8 * PACK_THREADS, 1u << 22)), dim3(PACK_THREADS), 0, s, static_cast<const uint8_t *>(src_packed), static_cast<uint8_t *>(dst_i8), nbytes);
    else
        e = enqueue(&unpack_i4_byte_kernel, dim3(flat_grid(nbytes, 256)), dim3(256), 0, s, static_cast<const uint8_t *>(src_packed), static_cast<int8_t *>(dst_i8), nbytes);
    return e == hipSuccess ? QM_OK : fail_launch(e);
}

// The linear layer's two steps and what they keep in the workspace: the scales of the rows of x, then either the codes
// for the 6-bit tile kernel, or the packed rows and the GEMM's own workspace.
namespace {
struct LinearPlan {
    bool one_launch;
    Fp6Route coded;
    int align;
    size_t scale_bytes, row_bytes, gemm_bytes;
    size_t bytes() const { return scale_bytes + row_bytes + gemm_bytes; }
};
// `apart`: D does not overlap x.  In one launch some workgroups write D while others still read x; in two x is read before.
LinearPlan linear_plan(int m, int n, int k, int in_dtype, int weight_align, bool apart = true)
{
    const auto up = [](size_t v) { return (v + 255) / 256 * 256; };
    LinearPlan pl{};
    if (apart && m <= 16 && fast_path_ok(m, n, k, weight_align) && n < (1 << 24) && (m <= 2 ? dot_linear_pays(m, n, k, in_dtype) : skinny_linear_fits(m, k, in_dtype) && skinny_linear_pays(m, n, k, in_dtype))) {
        pl.one_launch = true;
        return pl;
    }
    pl.align = weight_align < 256 ? weight_align : 256;
    pl.scale_bytes = up((size_t)m * sizeof(float));
    if ((double)m * n * k >= 4e9 && quant6_fits(k, in_dtype) && row_block_for_large_a(m, n, k, pl.align) == 0 && col_block_for_large_b(m, n, k, pl.align) == 0) {
        Choice ch = select_scaled(m, n, k, pl.align, true);
        ch.ksplit = effective_ksplit(g_configs[ch.cfg], k, ch.ksplit);
        pl.coded = fp6_route(m, n, k, pl.align, ch, FP6_FROM_X);
    }
    if (pl.coded) {
        pl.row_bytes = fp6_layout(m, k).bytes;
    } else {
        pl.row_bytes = up((size_t)m * (k / 2));
        pl.gemm_bytes = std::max(qm_gemm_workspace_bytes(m, n, k, pl.align, QM_CFG_AUTO, 1), qm_gemm_recode_bytes(m, n, k, pl.align, 1));
    }
    return pl;
}
}  // namespace

QM_EXPORT size_t qm_linear_workspace_bytes(int m, int n, int k, int in_dtype, int weight_align)
{
    if (m < 1 || n < 1 || k < 2 || (k & 1)) return 0;
    return linear_plan(m, n, k, in_dtype, weight_align).bytes();
}

QM_EXPORT int qm_linear_i4(const void *x, int in_dtype, const void *B, void *D, int m, int n, int k, const float *col_scale, const void *bias,
                           int out_dtype, void *stream, void *workspace, size_t workspace_bytes)
{
    if (in_dtype != QM_IN_F16 && in_dtype != QM_IN_BF16 && in_dtype != QM_IN_F32) return QM_ERR_DTYPE;
    if (out_dtype != QM_OUT_F16 && out_dtype != QM_OUT_BF16) return QM_ERR_DTYPE;
    if (m < 0 || n < 0 || k < 0 || (k & 1)) return QM_ERR_SHAPE;
    if (m == 0 || n == 0) return QM_OK;
    if (!D || (k > 0 && (!x || !B))) return QM_ERR_NULL;
    if (((uintptr_t)D & 1) || ((uintptr_t)bias & 1) || ((uintptr_t)x & (in_dtype == QM_IN_F32 ? 3 : 1))) return QM_ERR_ALIGN;
    const int out = out_dtype == QM_OUT_F16 ? OUT_F16 : OUT_BF16;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (k == 0) return run_gemm(nullptr, nullptr, D, m, n, 0, nullptr, col_scale, out, s, QM_CFG_AUTO, nullptr, 0, 0, static_cast<const uint16_t *>(bias));
    const uintptr_t x0 = (uintptr_t)x, x1 = x0 + (uintptr_t)m * k * (in_dtype == QM_IN_F32 ? 4 : 2), d0 = (uintptr_t)D, d1 = d0 + (uintptr_t)m * n * 2;
    const LinearPlan pl = linear_plan(m, n, k, in_dtype, ptr_alignment(B, nullptr), x1 <= d0 || d1 <= x0);
    if (pl.one_launch) {
        const uint16_t *b16 = static_cast<const uint16_t *>(bias);
        const auto launch = [&](auto in) {
            constexpr int IN = decltype(in)::value;
            if constexpr (IN != QM_IN_F32)
                if (m > 2) return launch_skinny_linear<IN>(x, B, D, m, n, k, col_scale, b16, out, s);
            return launch_dot_linear<IN>(x, B, D, m, n, k, col_scale, b16, out, s);
        };
        const hipError_t e = in_dtype == QM_IN_F16 ? launch(std::integral_constant<int, QM_IN_F16>{})
                             : in_dtype == QM_IN_BF16 ? launch(std::integral_constant<int, QM_IN_BF16>{}) : launch(std::integral_constant<int, QM_IN_F32>{});
        return e == hipSuccess ? QM_OK : fail_launch(e);
    }
    if (workspace == nullptr || ((uintptr_t)workspace & 255) || workspace_bytes < pl.bytes()) return QM_ERR_SCRATCH;
    float *scales = static_cast<float *>(workspace);
    uint8_t *rows = static_cast<uint8_t *>(workspace) + pl.scale_bytes;
    if (pl.coded) {
        Fp6Operand a = fp6_operand(m, k, rows);
        a.layout.parts = 1;
        const Quant6Args q{static_cast<const uint8_t *>(x), a.codes, a.sums, scales, m, k, a.layout.kt, a.layout.groups};
        hipError_t e = in_dtype == QM_IN_F16 ? launch_quantize_a6<QM_IN_F16>(q, s)
                       : in_dtype == QM_IN_BF16 ? launch_quantize_a6<QM_IN_BF16>(q, s) : launch_quantize_a6<QM_IN_F32>(q, s);
        if (e != hipSuccess) return fail_launch(e);
        GemmArgs p{nullptr, static_cast<const uint8_t *>(B), static_cast<int32_t *>(D), m, n, k};
        p.row_scale = scales;
        p.col_scale = col_scale;
        p.bias = static_cast<const uint16_t *>(bias);
        p.out = out;
        e = launch_tile6(p, a, pl.coded, s);
        return e == hipSuccess ? QM_OK : fail_launch(e);
    }
    const int st = qm_quantize_pack_i4(x, in_dtype, rows, scales, m, k, stream);
    if (st != QM_OK) return st;
    return run_gemm(rows, B, D, m, n, k, scales, col_scale, out, s, QM_CFG_AUTO, pl.gemm_bytes ? rows + pl.row_bytes : nullptr, pl.gemm_bytes, 0,
                    static_cast<const uint16_t *>(bias));
}

QM_EXPORT const char *qm_status_string(int status)
{
    switch (status) {
    case QM_OK: return "ok";
    case QM_ERR_NULL: return "null pointer";
    case QM_ERR_SHAPE: return "bad shape (m, n, k must be >= 0 and k even)";
    case QM_ERR_CONFIG: return "unknown kernel configuration, or it cannot run this shape";
    case QM_ERR_LAUNCH: return "HIP launch failed";
    case QM_ERR_ALIGN: return "C must be 4-byte aligned (a 16-bit output 2-byte aligned)";
    case QM_ERR_DTYPE: return "unknown output type";
    case QM_ERR_SCRATCH: return "the call needs more scratch memory than the library's static array (QM_STATIC_SCRATCH_BYTES) holds";
    default: return "unknown status";
    }
}

QM_EXPORT int qm_last_hip_error(void) { return g_last_hip_error; }

QM_EXPORT long long qm_debug_set_operand_limit(long long bytes)
{
    const long long full = 0x7fffffffLL;
    return g_operand_limit.exchange(bytes <= 0 || bytes > full ? full : bytes, std::memory_order_relaxed);
}

#ifndef QM_COMPILER_VERSION
#define QM_COMPILER_VERSION "unknown compiler"
#endif
QM_EXPORT const char *qm_version(void) { return "quadmul-amd 0.3 (gfx950; built with " QM_COMPILER_VERSION ")"; }

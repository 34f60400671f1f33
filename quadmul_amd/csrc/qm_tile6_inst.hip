// Instantiates the tile kernel on 6-bit floats for one output form (QM_TILE6_OUT: an OutKind); compiled once per form so the build runs in parallel.
#include "qm_launch.hpp"
#include "qm_tile6.hpp"

#ifndef QM_TILE6_OUT
#error "compile with -DQM_TILE6_OUT=<0, 1 or 2>"
#endif

namespace qm {

using Tile6 = Tile6Cfg<256, 256, 2, 4>;
using Tile6Narrow = Tile6Cfg<256, 128, 4, 2>;

template <class Cfg, int OUT, bool BIAS, class Kernel>
static hipError_t launch_tile6_kernel(Kernel kernel, const GemmArgs &p, const Fp6Operand &a, hipStream_t s, int opt)
{
    static std::atomic<bool> lds_ok[QM_MAX_DEVICES] = {};
    hipError_t e = ensure_dynamic_lds(kernel, Cfg::LDS_BYTES, lds_ok);
    if (e != hipSuccess) return e;
    int cus = 0;
    e = device_cus(&cus);
    if (e != hipSuccess) return e;
    if (opt & QM_OPT_PREPARE) return hipSuccess;
    const int tiles_m = (p.M + Cfg::BM - 1) / Cfg::BM, tiles_n = (p.N + Cfg::BN - 1) / Cfg::BN;
    const long long items = (long long)tiles_m * tiles_n;
    if (items > 0x7FFFFFFF) return hipErrorInvalidValue;
    // the LDS of a workgroup is all that a CU has: one each, a multiple of 8 so that an item's number modulo 8 names
    // the XCD it runs on
    const int held = cus / 8 * 8 < 8 ? 8 : cus / 8 * 8;
    const int grid = items < held ? (int)items : held;
    // Tiles are numbered in columns of four tile rows: of the 32 that an XCD works on at a time, 4 x 8 share the fewest
    // bytes (4 x 24 KiB of A and 8 x 16 of B per K-step, of B 8 on the narrow tiles)
    const int group_m = tiles_m < 4 ? tiles_m : 4;
    return enqueue(kernel, dim3(grid), dim3(Cfg::THREADS), Cfg::LDS_BYTES, s, p, a.codes, a.sums, a.layout.parts, a.layout.kt, tiles_m, tiles_n, group_m);
}

template <int OUT, bool BIAS>
static hipError_t launch_tile6(const GemmArgs &p, const Fp6Operand &a, hipStream_t s, int opt)
{
    if (opt & QM_OPT_NARROW) return launch_tile6_kernel<Tile6Narrow, OUT, BIAS>(&gemm_tile6_kernel<Tile6Narrow, OUT, BIAS>, p, a, s, opt);
    return launch_tile6_kernel<Tile6, OUT, BIAS>(&gemm_tile6_kernel<Tile6, OUT, BIAS>, p, a, s, opt);
}

#if QM_TILE6_OUT == 0
hipError_t launch_tile6_i32(const GemmArgs &p, const Fp6Operand &a, hipStream_t s, int opt) { return launch_tile6<OUT_I32, false>(p, a, s, opt); }
#elif QM_TILE6_OUT == 1
hipError_t launch_tile6_f16(const GemmArgs &p, const Fp6Operand &a, hipStream_t s, int opt)
{
    return p.bias != nullptr ? launch_tile6<OUT_F16, true>(p, a, s, opt) : launch_tile6<OUT_F16, false>(p, a, s, opt);
}
#else
hipError_t launch_tile6_bf16(const GemmArgs &p, const Fp6Operand &a, hipStream_t s, int opt)
{
    return p.bias != nullptr ? launch_tile6<OUT_BF16, true>(p, a, s, opt) : launch_tile6<OUT_BF16, false>(p, a, s, opt);
}
#endif

}  // namespace qm

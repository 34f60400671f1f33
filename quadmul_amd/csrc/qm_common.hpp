// Shared device helpers for the gfx950 packed-int4 GEMM kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

namespace qm {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
// The same at the alignment of one element: what a row of C has when N % 4 != 0 (or C itself
// is not 16-byte aligned).  A store through these is still one global_store_dwordx4 / x2 --
// the device takes them at any alignment -- where four element-wise stores per lane, 16 bytes
// apart from the next lane's, ran at a third of the speed (1444 x 31702 x 128: 104 us).
typedef v4i v4i_elem_aligned __attribute__((aligned(4)));
typedef v2i v2i_half_aligned __attribute__((aligned(2)));
typedef v4i v4i_half_aligned __attribute__((aligned(2)));
// ... and at any byte address.
typedef v4i v4i_any_aligned __attribute__((aligned(1)));
typedef v2i v2i_any_aligned __attribute__((aligned(1)));
typedef uint32_t u32_any_aligned __attribute__((aligned(1)));

// Output forms: the exact int32 product, or the product scaled per row and per column in
// fp32 and rounded to a 16-bit float (the "dequantise on the way out" use the reference's
// README.md:7 has in mind; no code of the reference does it).
enum OutKind { OUT_I32 = 0, OUT_F16 = 1, OUT_BF16 = 2 };

// kernel<<<grid, block, lds, s>>>(args...) without the detour through the configuration that the compiler's host stub pushes and pops: 0.2 us of the
// host less per launch, which is most of what a small call costs there (1 x 512 x 512 through the C interface 2.53 -> 2.33 us).
template <class T>
struct exactly { using type = T; };
template <class... P>
inline hipError_t enqueue(void (*const kernel)(P...), const dim3 grid, const dim3 block, const size_t lds, hipStream_t s, typename exactly<P>::type... args)
{
    void *at[] = {const_cast<void *>(static_cast<const void *>(&args))...};
    const hipError_t e = hipLaunchKernel(reinterpret_cast<const void *>(kernel), grid, block, at, lds, s);
    if (e != hipSuccess) (void)hipGetLastError();  // (the caller reports it)
    return e;
}

struct GemmArgs {
    const uint8_t *A;  // [M, K/2] packed s4
    const uint8_t *B;  // [N, K/2] packed s4
    int32_t *C;        // [M, N] int32; or [M, N] 16-bit floats when `out` says so
    int M, N, K;
    // scaled output only: D[m][n] = round16(((float)C[m][n] * row_scale[m]) * col_scale[n]),
    // a null pointer standing for all ones
    const float *row_scale = nullptr;  // [M]
    const float *col_scale = nullptr;  // [N]
    // scaled output only: added per column to the rounded value, in the output's type, and rounded
    // again (what a separate in-place addition of a bias to D gives); null: nothing is added
    const uint16_t *bias = nullptr;  // [N]
    int out = OUT_I32;
    // K split over several work items per tile (pipelined kernel): where the partial sums go.
    // Null: they meet in C by atomic adds (C zero-filled beforehand).  Otherwise item i of the
    // launch stores its tile here, 16 bytes per lane in the order the MFMA leaves them, and a
    // second kernel adds the splits up.
    int32_t *ws = nullptr;
    // Row stride of C in elements, 0 standing for N: set when the call computes a block of
    // columns of a wider C (a B beyond the kernels' 32-bit offsets is cut along N).
    int ldc = 0;
};

// The output form above a number of rows below 2^24, one kernel argument for both: with the bias as a
// tenth scalar argument the kernels for a few rows would take more than the 16 dwords that are
// preloaded into SGPRs, and more than the 64 bytes that the runtime writes to the argument buffer
// as one line.  With 72 bytes a call takes longer on the host: 1 x 4096 x 4096 out of an eager loop
// 3.84 to 4.33 us, with 64 bytes 3.56.
constexpr int QM_ROWS_BITS = 24;
inline int pack_rows_out(int rows, int out) { return rows | (out << QM_ROWS_BITS); }
__device__ __forceinline__ int packed_rows(int rows_out) { return rows_out & ((1 << QM_ROWS_BITS) - 1); }
__device__ __forceinline__ int packed_out(int rows_out) { return rows_out >> QM_ROWS_BITS; }

__device__ __forceinline__ int c_stride(const GemmArgs &p) { return p.ldc != 0 ? p.ldc : p.N; }

__device__ __forceinline__ float scale_at(const float *s, int i, int n) { return (s != nullptr && i < n) ? s[i] : 1.0f; }

// fp32 -> 16-bit float, round to nearest even (NaN stays NaN).  Contraction is switched
// off in these helpers: fused, the compiler turns "multiply, then round to fp16" into one
// instruction with a single rounding, which is not the value defined above.
template <int OUT>
__device__ __forceinline__ uint16_t round16(float x)
{
#pragma clang fp contract(off)
    if constexpr (OUT == OUT_F16) {
        // (the empty asm hides where x came from: instruction selection otherwise merges a
        // preceding fp32 multiply and this conversion into v_fma_mixlo_f16, which rounds the
        // exact product once, straight to fp16 -- not the twice-rounded value defined above)
        asm("" : "+v"(x));
        const _Float16 h = (_Float16)x;
        return __builtin_bit_cast(uint16_t, h);
    } else {
        // (both candidates computed and one selected: no per-lane branch in the callers' code)
        const uint32_t u = __builtin_bit_cast(uint32_t, x);
        const uint32_t rounded = (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16, quiet = (u >> 16) | 0x0040u;
        return (uint16_t)(((u & 0x7FFFFFFFu) > 0x7F800000u) ? quiet : rounded);
    }
}
__device__ __forceinline__ uint16_t round16(float x, int out) { return out == OUT_F16 ? round16<OUT_F16>(x) : round16<OUT_BF16>(x); }

// The sum of two 16-bit floats, rounded to nearest even: two bf16 (or fp16) values add up in
// fp32 with enough digits to spare that rounding the fp32 sum is rounding the exact one.
__device__ __forceinline__ uint16_t add16(uint16_t h, uint16_t b, int out)
{
    if (out == OUT_F16) return __builtin_bit_cast(uint16_t, (_Float16)(__builtin_bit_cast(_Float16, h) + __builtin_bit_cast(_Float16, b)));
    return round16<OUT_BF16>(__builtin_bit_cast(float, (uint32_t)h << 16) + __builtin_bit_cast(float, (uint32_t)b << 16));
}

// the scaled value of one element, in the one order of operations everything here uses
__device__ __forceinline__ float scaled(int c, float rs, float cs)
{
#pragma clang fp contract(off)
    const float t = (float)c * rs;
    return t * cs;
}

// Two values at once, the first in the low half.  bf16: one v_cvt_pk_bf16_f32, which gives what
// round16 gives for every one of the 2^32 inputs, NaNs included (tests/test_scaled_gpu.py).
template <int OUT>
__device__ __forceinline__ uint32_t round16_pair(float x, float y)
{
    if constexpr (OUT == OUT_BF16) {
        typedef float f2 __attribute__((ext_vector_type(2)));
        typedef __bf16 h2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{x, y}), h2));
    } else {
        return (uint32_t)round16<OUT_F16>(x) | ((uint32_t)round16<OUT_F16>(y) << 16);
    }
}
template <int OUT>
__device__ __forceinline__ uint32_t add16_pair(uint32_t h, uint32_t b)
{
    if constexpr (OUT == OUT_BF16) {
        return round16_pair<OUT_BF16>(__builtin_bit_cast(float, h << 16) + __builtin_bit_cast(float, b << 16),
                                      __builtin_bit_cast(float, h & 0xFFFF0000u) + __builtin_bit_cast(float, b & 0xFFFF0000u));
    } else {
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, (h2)(__builtin_bit_cast(h2, h) + __builtin_bit_cast(h2, b)));
    }
}
// The bias of columns n .. n+3 as two packed pairs; -0 (which adds nothing to any value, to a
// zero of either sign included) past the last column and without a bias.
__device__ __forceinline__ v2i bias4_at(const GemmArgs &p, int n)
{
    uint32_t b[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) b[e] = (p.bias != nullptr && n + e < p.N) ? p.bias[n + e] : 0x8000u;
    return v2i{(int)(b[0] | (b[1] << 16)), (int)(b[2] | (b[3] << 16))};
}

// the element (.., n) of a 16-bit output: scaled, rounded, the bias (if any) added
__device__ __forceinline__ uint16_t finish16(const GemmArgs &p, int c, float rs, int n)
{
    const uint16_t h = round16(scaled(c, rs, scale_at(p.col_scale, n, p.N)), p.out);
    return p.bias != nullptr && n < p.N ? add16(h, p.bias[n], p.out) : h;
}

// The elements (.., n .. n+3), n < N.  The scales and the biases of all four are fetched before the first
// is used: with one element after the other, each behind its own conditions, every load is waited
// for by itself -- four round trips to the L2 for a block, and four more for the bias.
__device__ __forceinline__ void finish16x4(const GemmArgs &p, const v4i c, float rs, int n, uint16_t (&h)[4])
{
    float cs[4] = {1.0f, 1.0f, 1.0f, 1.0f};
    uint16_t b[4] = {0, 0, 0, 0};
    if (p.col_scale != nullptr) {
#pragma unroll
        for (int e = 0; e < 4; ++e) cs[e] = p.col_scale[min(n + e, p.N - 1)];
    }
    if (p.bias != nullptr) {
#pragma unroll
        for (int e = 0; e < 4; ++e) b[e] = p.bias[min(n + e, p.N - 1)];
    }
    const auto finish = [&](auto out_) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int ce = c[e];
            h[e] = round16<decltype(out_)::value>(scaled(ce, rs, cs[e]));
        }
        if (p.bias != nullptr) {
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = add16(h[e], b[e], decltype(out_)::value);
        }
    };
    if (p.out == OUT_F16) finish(std::integral_constant<int, OUT_F16>{});
    else finish(std::integral_constant<int, OUT_BF16>{});
}

// gfx950 has no int4 MFMA, so nibbles are widened to int8 -- but scaled by 16,
// which needs no per-byte sign fix-up.  For a dword w holding nibbles k0..k7
// (k0 in bits 0..3), read as four int8 lanes:
//     (w << 4) & 0xF0F0F0F0  ==  16 * s4(k0), 16 * s4(k2), 16 * s4(k4), 16 * s4(k6)
//      w       & 0xF0F0F0F0  ==  16 * s4(k1), 16 * s4(k3), 16 * s4(k5), 16 * s4(k7)
// because a nibble n placed in the high half of a byte is the int8 value 16*s4(n).
// Both operands get the same treatment, so every int8 product carries a factor
// 256 and the int32 accumulator holds exactly 256 * C; the epilogue shifts it out.
// |C| <= 64 K, hence exact while 256 * 64 * K < 2^31, i.e. K <= QM_MAX_K_X16.
// The even/odd split permutes K inside a dword; the contraction runs over K and
// A and B are permuted identically, so the sum is unchanged.
constexpr int QM_MAX_K_X16 = 131071;

__device__ __forceinline__ int x16_even(int w) { return (int)(((uint32_t)w << 4) & 0xF0F0F0F0u); }
__device__ __forceinline__ int x16_odd(int w) { return (int)((uint32_t)w & 0xF0F0F0F0u); }

__device__ __forceinline__ void x16_expand(const v4i q, v4i &even, v4i &odd)
{
    even.x = x16_even(q.x); even.y = x16_even(q.y); even.z = x16_even(q.z); even.w = x16_even(q.w);
    odd.x = x16_odd(q.x);   odd.y = x16_odd(q.y);   odd.z = x16_odd(q.z);   odd.w = x16_odd(q.w);
}

// The same in 10 instructions instead of 12: one 64-bit shift per pair of dwords (the nibble
// that crosses into the upper dword lands in a low nibble and is masked away with the rest).
__device__ __forceinline__ void x16_expand_pairs(const v4i q, v4i &even, v4i &odd)
{
    const v2i lo = {q.x, q.y}, hi = {q.z, q.w};
    v2i slo, shi;
    asm("v_lshlrev_b64 %0, 4, %1" : "=v"(slo) : "v"(lo));
    asm("v_lshlrev_b64 %0, 4, %1" : "=v"(shi) : "v"(hi));
    even.x = (int)((uint32_t)slo.x & 0xF0F0F0F0u); even.y = (int)((uint32_t)slo.y & 0xF0F0F0F0u);
    even.z = (int)((uint32_t)shi.x & 0xF0F0F0F0u); even.w = (int)((uint32_t)shi.y & 0xF0F0F0F0u);
    odd.x = x16_odd(q.x); odd.y = x16_odd(q.y); odd.z = x16_odd(q.z); odd.w = x16_odd(q.w);
}

// D(16x16) += S0(16x64) * S1(64x16), int8 in, int32 out.  Lane l supplies row
// l%16 of S0 / column l%16 of S1 for the 16 k-values of group l/16, and owns
// D[4*(l/16) + r][l%16] in register r.
__device__ __forceinline__ v4i mfma16(const v4i s0, const v4i s1, const v4i acc)
{
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(s0, s1, acc, 0, 0, 0);
}

// Byte offset of row `row` of a packed operand with Kb bytes per row, for the skinny
// kernels: both factors are below 2^24 there (the host side sees to it), so the full-rate
// 24-bit multiply does (the 32-bit one issues at a quarter of the rate, and these products
// sit in front of a wave's first load).
__device__ __forceinline__ uint32_t row_bytes24(int row, int Kb) { return __umul24((uint32_t)row, (uint32_t)Kb); }

// 16 bytes at any byte address, as five aligned dwords shifted into place.  The memory pipeline takes 16 bytes per lane at any
// multiple of four in one access and at other addresses in four, so four dwords from the
// multiple of four below and a fifth are less than half the work.  No dword is read that lies partly outside the `bytes`
// from `base` on: where the 16 bytes begin or end too close to them, they are loaded as they are.
// Addresses are 32-bit offsets from `base` rounded down to a multiple of four, which `low` to `high` are inside (dword_span).
struct DwordSpan {
    const uint8_t *base;
    uint32_t lead, low, count;  // bytes from `base` to the operand; offsets low .. low + count - 1 are far enough from both ends
};
__device__ __forceinline__ DwordSpan dword_span(const uint8_t *operand, const uint32_t bytes)
{
    const uint32_t lead = (uint32_t)(uintptr_t)operand & 3u, low = lead != 0 ? 4u : 0u, end = lead + bytes;
    return {operand - lead, lead, low, end >= low + 19u ? end - 18u - low : 0u};
}
struct Shifted16 {
    v4i w;
    int next;
    uint32_t by;
    __device__ __forceinline__ void load(const DwordSpan &s, const uint32_t at)  // `at` bytes into the operand
    {
        const uint32_t off = at + s.lead;
        const bool near = off - s.low >= s.count;
        by = near ? 0u : off & 3u;
        w = *reinterpret_cast<const v4i_any_aligned *>(s.base + (off - by));
        next = *reinterpret_cast<const int *>(s.base + ((near ? off + 3u : off + 15u) & ~3u));
    }
    __device__ __forceinline__ v4i value() const
    {
        return v4i{(int)__builtin_amdgcn_alignbyte((uint32_t)w.y, (uint32_t)w.x, by), (int)__builtin_amdgcn_alignbyte((uint32_t)w.z, (uint32_t)w.y, by),
                   (int)__builtin_amdgcn_alignbyte((uint32_t)w.w, (uint32_t)w.z, by), (int)__builtin_amdgcn_alignbyte((uint32_t)next, (uint32_t)w.w, by)};
    }
};

// Workgroups are dealt round-robin to the 8 XCDs (id % 8), each with a private
// L2.  Renumber so that every XCD owns one contiguous range of tile ids.
__device__ __forceinline__ int xcd_contiguous_id(int bid, int nblocks)
{
    constexpr int XCDS = 8;
    const int xcd = bid % XCDS, local = bid / XCDS;
    const int per = (nblocks + XCDS - 1) / XCDS;  // size of the larger shares
    const int tall = nblocks % XCDS;              // how many XCDs get a larger share (0: all equal)
    if (tall == 0 || xcd < tall) return xcd * per + local;
    return tall * per + (xcd - tall) * (per - 1) + local;
}

// Which of its `cnt` runs of K a wave of the wave-level kernels begins with.  Rows of 4096 bytes or multiples of them have the same columns in the same channels of the
// L2 and of the memory, and workgroups that begin together want the same columns of all their rows: a
// kilobyte of eight waves comes from a quarter of the channels.  There the workgroups of an XCD (every eighth) begin at different
// runs and go round.  us, before -> now, B from HBM: 48 x 8192 x 8192 9.63 -> 8.50, 16 x 4096 x 8192 5.38 -> 4.88, 33 x 8192 x 16384 16.0 -> 13.5, 17 x
// 6144 x 32768 23.9 -> 17.9; over 7463 sizes to 256 rows on a K of 8192 to 57344 0.956 in the geometric mean, 0.959 with B in the caches as far as it fits,
// 9 and 39 of them more than 2 % slower (6 and 7).  Not taken: rows of other lengths, which
// their length spreads (1 % slower in the mean, 16 x 4096 x 11008 3.6), odd multiples of 2048 bytes among them (1.004 over 24 sizes); few columns, whose workgroups share A while it is there
// (592 columns 3.5 % slower); many rows, where B's second reader comes too late, the fewer the longer K (233 x 7945 x 32768 75 -> 92, with B in the caches
// 64 -> 96; 216 x 2117 x 24576 23.2 -> 25.9; 33 to 64 rows on many columns above 32768 1.04 in the mean with B in the caches, 0.99 from HBM); blocks of 48 columns in one
// round on a K of 32768 (50 x 12039 39.2 -> 40.9).  (A form of the kernels of its own: the few instructions before the first load are 0.8 % of 37 x 11008 x 4096.)
constexpr bool goes_round(const int m, const int n, const int k)
{
    const int rows = k <= 8192 ? 256 : k <= 16384 ? 160 : k <= 32768 ? 96 : n <= 4096 ? 64 : 32;
    return k % 8192 == 0 && n >= 2048 && m <= rows && !(k == 32768 && m > 16 && n > 8192 && n <= 12288);
}
__device__ __forceinline__ int first_of_runs(const int cnt, const int waves)
{
    const int turn = blockIdx.x >> 3;
    // (one wave's runs are short and many: with sixteen places 32 x 57344 x 8192 39.5 -> 44.7 us, with four 38.8)
    return waves == 1 ? (turn & 3) * cnt >> 2 : (turn * 5 & 15) * cnt >> 4;
}

}  // namespace qm

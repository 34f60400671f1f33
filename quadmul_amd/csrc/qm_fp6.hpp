// int4 as 6-bit floats (E2M3, upper exponent bit clear: sign and a four-bit magnitude in units of 1/8).
#pragma once
#include "qm_common.hpp"

namespace qm {

typedef int v6i __attribute__((ext_vector_type(6)));

// 16 nibbles in two dwords -> the low four bits of 16 six-bit fields in three.  Fields 6 bits apart and
// nibbles 4 apart coincide modulo 4 up to a shift by two, so one 64-bit shift serves all of them;
// which nibble goes to which field does not matter as long as A and B agree.
constexpr uint32_t FP6_PICK[3] = {0x0F00F00Fu, 0xF00F00F0u, 0x00F00F00u};   // from the dword as it is; the others from the shifted pair
constexpr uint32_t FP6_KEEP[3] = {0xCF3CF3CFu, 0xF3CF3CF3u, 0x3CF3CF3Cu};   // the low four bits of every field
constexpr uint32_t FP6_TOP[3] = {0x08208208u, 0x82082082u, 0x20820820u};    // bit 3 of every field

constexpr int FP6_STEP_BYTES = 96;       // 128 codes of one row
constexpr int FP6_GROUP_BYTES = 32 * 96; // one K-step of 32 rows: their order in memory and in the LDS
constexpr uint32_t FP6_START = 0x48400000u;  // 1.5 * 2^17
constexpr int QM_MAX_K_FP6 = 65535;
constexpr size_t QM_FP6_MAX_BYTES = 256u << 20;  // of codes: what a call may ask of its caller's memory, and within 32-bit offsets

__device__ __forceinline__ void fp6_place(const uint32_t w0, const uint32_t w1, uint32_t (&f)[3])
{
    const uint64_t sh = (((uint64_t)w1 << 32) | w0) << 2;
    const uint32_t lo = (uint32_t)sh, hi = (uint32_t)(sh >> 32);
    f[0] = ((w0 & FP6_PICK[0]) | (lo & ~FP6_PICK[0])) & FP6_KEEP[0];
    f[1] = ((w1 & FP6_PICK[1]) | (hi & ~FP6_PICK[1])) & FP6_KEEP[1];
    f[2] = ((w0 & FP6_PICK[2]) | (hi & ~FP6_PICK[2])) & FP6_KEEP[2];
}

// 16 signed nibbles -> 16 sign-and-magnitude codes
__device__ __forceinline__ void fp6_signed(const uint32_t w0, const uint32_t w1, uint32_t (&f)[3])
{
    const uint32_t s0 = w0 & 0x88888888u, s1 = w1 & 0x88888888u;
    // |v| of a negative nibble is (7 - its low three bits) + 1
    const uint32_t m0 = ((w0 ^ (s0 - (s0 >> 3))) & 0x77777777u) + (s0 >> 3), m1 = ((w1 ^ (s1 - (s1 >> 3))) & 0x77777777u) + (s1 >> 3);
    uint32_t s[3];
    fp6_place(m0, m1, f);
    fp6_place(s0, s1, s);
    f[0] |= s[0] << 2;
    f[1] |= (s[1] << 2) | (s[0] >> 30);
    f[2] |= (s[2] << 2) | (s[1] >> 30);
}

// a lane's 32 nibbles of a fragment -> its six dwords
__device__ __forceinline__ void fp6_fragment(const v4i w, uint32_t (&f)[6])
{
    uint32_t lo[3], hi[3];
    fp6_signed((uint32_t)w.x, (uint32_t)w.y, lo);
    fp6_signed((uint32_t)w.z, (uint32_t)w.w, hi);
#pragma unroll
    for (int e = 0; e < 3; ++e) {
        f[e] = lo[e];
        f[3 + e] = hi[e];
    }
}

// ---- A re-coded, in a workspace ----
// codes  [groups][kt][FP6_GROUP_BYTES]   groups of 32 rows, kt K-steps (an even number); within a group of one step 48 bytes for
//                                        each lane of the fragments that it is, first the one of rows 0..15, then the
//                                        one of rows 16..31, in three pieces of 16 bytes per lane, 1 KiB each
// sums   [parts][32 groups]              per row, over FP6_PART_STEPS K-steps each (a workgroup's share of the re-coding)
constexpr int FP6_PART_STEPS = 32;
struct Fp6Layout {
    int groups, kt, parts;
    size_t code_bytes, bytes;
};
inline Fp6Layout fp6_layout(int m, int k)
{
    Fp6Layout l;
    l.groups = (m + 31) / 32;
    l.kt = ((k + 127) / 128 + 1) / 2 * 2;
    l.parts = (l.kt + FP6_PART_STEPS - 1) / FP6_PART_STEPS;
    l.code_bytes = (size_t)l.groups * l.kt * FP6_GROUP_BYTES;
    l.bytes = l.code_bytes + (size_t)l.parts * l.groups * 32 * sizeof(int);
    return l;
}
struct Fp6Operand {
    Fp6Layout layout;
    uint8_t *codes;
    int *sums;
};
inline Fp6Operand fp6_operand(int m, int k, void *ws)
{
    const Fp6Layout l = fp6_layout(m, k);
    return {l, static_cast<uint8_t *>(ws), reinterpret_cast<int *>(static_cast<uint8_t *>(ws) + l.code_bytes)};
}

}  // namespace qm

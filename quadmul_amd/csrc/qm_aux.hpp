// Kernels beside the MFMA ones, and their launchers: the generic GEMM (any even K, any
// alignment), zero fill, zero-padded operand copies, the kernel that adds up a K split out
// of a workspace, pack / unpack (reference: test.py:6-15, kernel.cu:387-408) and the fused
// quantise + pack.  Included by qm_dispatch.hip only.
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/qm_abi.h"
#include "qm_common.hpp"

namespace qm {

// --------------------------------------------------------------------------
// Fallback kernel: any M, N, even K, any alignment, no limit on K.  One thread
// per element of C over LDS-staged 16x16x(128 nibble) tiles, plain byte loads.
// --------------------------------------------------------------------------
__device__ __forceinline__ int s4_lo(uint32_t b) { return (int)(int8_t)(b << 4) >> 4; }
__device__ __forceinline__ int s4_hi(uint32_t b) { return (int)(int8_t)b >> 4; }

__global__ void __launch_bounds__(256) gemm_generic_kernel(const GemmArgs p, const int tiles_n)
{
    __shared__ uint8_t As[16][64 + 4];
    __shared__ uint8_t Bs[16][64 + 4];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int m0 = (blockIdx.x / tiles_n) * 16, n0 = (blockIdx.x % tiles_n) * 16;
    const size_t Kb = (size_t)(p.K >> 1);
    int32_t sum = 0;
    for (size_t k0 = 0; k0 < Kb; k0 += 64) {
        // 16 rows x 64 bytes per operand = 1024 bytes each, 4 bytes per thread
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int idx = threadIdx.x + t * 256, row = idx >> 6, col = idx & 63;
            const bool kin = k0 + col < Kb;
            As[row][col] = (kin && m0 + row < p.M) ? p.A[(size_t)(m0 + row) * Kb + k0 + col] : (uint8_t)0;
            Bs[row][col] = (kin && n0 + row < p.N) ? p.B[(size_t)(n0 + row) * Kb + k0 + col] : (uint8_t)0;
        }
        __syncthreads();
#pragma unroll 16
        for (int j = 0; j < 64; ++j) {
            const uint32_t a = As[ty][j], b = Bs[tx][j];
            sum += s4_lo(a) * s4_lo(b) + s4_hi(a) * s4_hi(b);
        }
        __syncthreads();
    }
    const int m = m0 + ty, n = n0 + tx;
    if (m < p.M && n < p.N) {
        const size_t at = (size_t)m * c_stride(p) + n;
        if (p.out == OUT_I32) p.C[at] = sum;
        else reinterpret_cast<uint16_t *>(p.C)[at] = finish16(p, sum, scale_at(p.row_scale, m, p.M), n);
    }
}

static hipError_t launch_generic(const GemmArgs &p, hipStream_t stream, int)
{
    const long long tiles_m = (p.M + 15) / 16, tiles_n = (p.N + 15) / 16;
    if (tiles_m * tiles_n > 0x7fffffffLL) return hipErrorInvalidValue;
    return enqueue(&gemm_generic_kernel, dim3((unsigned)(tiles_m * tiles_n)), dim3(256), 0, stream, p, (int)tiles_n);
}

// --------------------------------------------------------------------------
// Zero fill (k == 0) and pack / unpack, flat over the whole array: K is even so
// a byte never straddles two rows.
// --------------------------------------------------------------------------
__global__ void fill_zero16_kernel(uint16_t *dst, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) dst[i] = 0;
}

// k == 0 with a bias: zero plus the bias (which turns a bias of -0 into +0)
__global__ void fill_bias16_kernel(uint16_t *dst, const uint16_t *bias, int ncols, int ldc, size_t n, int out)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        dst[i / ncols * ldc + i % ncols] = add16(0, bias[i % ncols], out);
}

__global__ void fill_zero_kernel(int32_t *dst, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) dst[i] = 0;
}

// --------------------------------------------------------------------------
// Operand copies with every row padded with zeros to a whole number of 128-nibble K-steps
// (zero nibbles add nothing to a product): what lets the pipelined kernel run shapes whose
// K is not a multiple of 32, or whose operands are not 16-byte aligned, out of a
// caller-provided workspace.  Both operands in one launch (a second dependent launch costs
// more than the copy of a small operand): rows 0 .. rows_a-1 are A's, the rest B's.
// Source rows may start at any byte: one 16-byte piece of the copy per thread, loaded at whatever address
// it has.  Where the row ends inside a piece, the load runs on into the next row and those bytes are
// zeroed; a piece that would run past the end of the operand is read byte by byte.  No byte outside
// the operands is read.
// kb: bytes per source row; ppr: 16-byte pieces per row of the copy.
// Bound: HBM on large operands (4096 x 11008 x 4094 13.6 us, 4.6 TB/s of bytes read and written), the
// launch on small ones.  With one wave per row and 4 bytes per lane and turn, put together from
// two aligned words, these took (us, before -> now): 33 x 3307 x 4100 5.5 -> 3.6, 1531 x 3307 x 4100
// 6.3 -> 5.3, 100 x 9000 x 9000 29.1 -> 14.5, 4096 x 11008 x 4094 16.6 -> 13.6.  Non-temporal loads are
// slower (6.2, 1531 x 3307 x 4100), non-temporal stores 0.3 us faster there and 1 us slower on 100 x 9000 x 9000.
// --------------------------------------------------------------------------
struct PadRowsArgs {
    const uint8_t *src_a, *src_b;
    v4i *dst_a, *dst_b;
    int rows_a, rows_b, kb, ppr;
};

__global__ void __launch_bounds__(256) pad_rows_kernel(const PadRowsArgs q)
{
    const uint32_t piece = blockIdx.x * 256u + threadIdx.x;  // (below 2^28: either copy is below 2 GiB)
    const uint32_t r = piece / (uint32_t)q.ppr;
    if (r >= (uint32_t)(q.rows_a + q.rows_b)) return;
    const int at = 16 * (int)(piece - r * (uint32_t)q.ppr);
    const bool is_a = r < (uint32_t)q.rows_a;
    const int row = is_a ? (int)r : (int)r - q.rows_a, rows = is_a ? q.rows_a : q.rows_b;
    const uint8_t *src = (is_a ? q.src_a : q.src_b) + (size_t)row * q.kb + at;
    v4i *out = (is_a ? q.dst_a : q.dst_b) + (size_t)row * q.ppr + (at >> 4);
    const int keep = q.kb - at;  // bytes of the row from this piece on
    v4i v{0, 0, 0, 0};
    if (keep > 0) {
        if ((long long)(rows - row) * q.kb - at >= 16) {
            v = *reinterpret_cast<const v4i_any_aligned *>(src);
        } else {
            uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 15; ++e)  // (fewer than 16 are left)
                if (e < keep) w[e >> 2] |= (uint32_t)src[e] << (8 * (e & 3));
            v = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
        }
        if (keep < 16) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int b = min(max(keep - 4 * e, 0), 4);
                v[e] = b >= 4 ? v[e] : (int)((uint32_t)v[e] & ((1u << (8 * b)) - 1u));
            }
        }
    }
    *out = v;
}

// --------------------------------------------------------------------------
// K split with a workspace (pipelined kernel): item (split s, tile t) of the GEMM launch
// left its BM x BN partial sums in slot s * ntiles + t, wave by wave, block by block, 16
// bytes per lane in the order the MFMA leaves a block (lane l: row l % 16, columns
// 4 * (l / 16) .. + 3).  One thread here adds up the splits of one such 16-byte piece and
// stores the four sums -- as int32, or scaled and rounded to a 16-bit float -- with the
// guards of the matrix edge.  Tiles are numbered as the GEMM kernel numbers them (columns of
// group_m tiles).
// --------------------------------------------------------------------------
struct SplitReduceArgs {
    const v4i *ws;
    void *C;
    int M, N;
    int tiles_m, tiles_n, group_m, ksplit;
    int BM, BN, WGN, FM, FN, waves;
    const float *row_scale, *col_scale;
    const uint16_t *bias;
    int out;
};

__global__ __launch_bounds__(256) void splitk_reduce_kernel(const SplitReduceArgs q)
{
    const int blocks = q.FM * q.FN;
    const size_t per_tile = (size_t)q.waves * blocks * 64;  // 16-byte pieces per slot
    const size_t ntiles = (size_t)q.tiles_m * q.tiles_n;
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;  // (the launcher keeps the count below 2^31)
    if (t >= ntiles * per_tile) return;
    const v4i *src = q.ws + t;
    const size_t stride = ntiles * per_tile;
    v4i sum = {0, 0, 0, 0};
    // four splits at a time, so that their loads are in flight together (splits past the
    // last re-read it and count for nothing)
    for (int s = 0; s < q.ksplit; s += 4) {
        v4i v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = __builtin_nontemporal_load(src + (size_t)min(s + i, q.ksplit - 1) * stride);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int on = s + i < q.ksplit ? -1 : 0;
            sum.x += v[i].x & on; sum.y += v[i].y & on; sum.z += v[i].z & on; sum.w += v[i].w & on;
        }
    }
    const int lane = (int)(t & 63);
    uint32_t u = t >> 6;
    const int blk = (int)(u % (uint32_t)blocks);
    u /= (uint32_t)blocks;
    const int wave = (int)(u % (uint32_t)q.waves);
    const int pid = (int)(u / (uint32_t)q.waves);
    const int width = q.group_m * q.tiles_n;
    const int first_m = (pid / width) * q.group_m;
    const int gsz = min(q.tiles_m - first_m, q.group_m);
    const int tm = first_m + (pid % width) % gsz, tn = (pid % width) / gsz;
    const int m = tm * q.BM + (wave / q.WGN) * q.FM * 16 + (blk / q.FN) * 16 + (lane & 15);
    const int n = tn * q.BN + (wave % q.WGN) * q.FN * 16 + (blk % q.FN) * 16 + (lane >> 4) * 4;
    if (m >= q.M || n >= q.N) return;
    if (q.out == OUT_I32) {
        int32_t *crow = static_cast<int32_t *>(q.C) + (size_t)m * q.N;
        if ((q.N & 3) == 0 && ((uintptr_t)q.C & 15) == 0) {
            *reinterpret_cast<v4i *>(crow + n) = sum;  // n % 4 == 0 and N % 4 == 0: all four inside
        } else if (n + 3 < q.N) {
            *reinterpret_cast<v4i_elem_aligned *>(crow + n) = sum;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + e < q.N) crow[n + e] = sum[e];
        }
    } else {
        uint16_t *drow = static_cast<uint16_t *>(q.C) + (size_t)m * q.N;
        const float rs = scale_at(q.row_scale, m, q.M);
        GemmArgs f{};
        f.N = q.N;
        f.col_scale = q.col_scale;
        f.bias = q.bias;
        f.out = q.out;
        uint16_t h[4];
        finish16x4(f, sum, rs, n, h);
        if ((q.N & 3) == 0 && ((uintptr_t)q.C & 7) == 0) {
            *reinterpret_cast<v2i *>(drow + n) = v2i{(int)(h[0] | ((uint32_t)h[1] << 16)), (int)(h[2] | ((uint32_t)h[3] << 16))};
        } else if (n + 3 < q.N) {
            *reinterpret_cast<v2i_half_aligned *>(drow + n) = v2i{(int)(h[0] | ((uint32_t)h[1] << 16)), (int)(h[2] | ((uint32_t)h[3] << 16))};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + e < q.N) drow[n + e] = h[e];
        }
    }
}

// 16 int8 in -> 8 packed bytes out per thread when aligned, else one byte per thread.
__device__ __forceinline__ uint32_t pack4(uint32_t w)  // 4 int8 -> 2 packed bytes in bits 0..15
{
    uint32_t t = w & 0x0F0F0F0Fu;
    t |= t >> 4;  // byte0 = n0 | n1<<4, byte2 = n2 | n3<<4
    return (t & 0xFFu) | ((t >> 8) & 0xFF00u);
}

// At least 8 packed bytes at any address; the last piece is the last 8 bytes, those that the one before
// has written among them.  Two pieces per thread in flight, 32 KB of values apart: workgroup b takes the
// 4 KB of values number 16 (b / 8) + b % 8 and those eight further on, so that
//   - both are on the XCD of the workgroup that wrote them, if an elementwise kernel with 4 KB to a workgroup did, and
//     are found in its L2 up to about 24 MB; unpack_i4_vec_kernel finds the packed bytes, 2 KB to a workgroup, in the same way;
//   - eight workgroups read 64 KB in a row, which is what HBM wants.
// Loads are non-temporal: they leave the caches to the packed bytes.  us, this way / 8 KB in a row to a workgroup,
// non-temporal / the two pieces a grid apart, plain loads: an elementwise kernel and the packing behind it, same buffer,
// 16 MB 8.9 / 13.7 / 8.9; packing and unpacking, same buffer, 16 MB 8.0 / 11.5 / 7.6, 32 MB 14.1 / 21.3 / 16.8, 48 MB
// 21.5 / 26.7 / 23.8; packing from HBM 16 MB 5.7 / 5.7 / 6.6, 32 MB 9.5 / 9.4 / 11.4, 64 MB 16.8 / 17.1 / 20.3, 160 MB 38.6
// (6.5 TB/s) / 38.4 / 45.5.  Sizes and addresses that are not multiples of 8 once took one byte per thread: 8191 x 8190 42.6 us.
constexpr int PACK_PIECES = 2, PACK_THREADS = 256, PACK_APART = 8;  // (workgroups: one per XCD)
__global__ void __launch_bounds__(PACK_THREADS) pack_i4_vec_kernel(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, size_t nbytes)
{
    static_assert(PACK_PIECES == 2, "the pieces of a group of PACK_APART workgroups");
    // (the grid is a multiple of PACK_APART workgroups)
    const size_t piece = (size_t)(blockIdx.x / PACK_APART) * (PACK_PIECES * PACK_APART) + blockIdx.x % PACK_APART;
    for (size_t i0 = piece * PACK_THREADS + threadIdx.x; 8 * i0 < nbytes; i0 += (size_t)gridDim.x * (PACK_THREADS * PACK_PIECES)) {
        const size_t at[PACK_PIECES] = {min(8 * i0, nbytes - 8), min(8 * (i0 + PACK_APART * PACK_THREADS), nbytes - 8)};
        v4i v[PACK_PIECES];
#pragma unroll
        for (int u = 0; u < PACK_PIECES; ++u) v[u] = __builtin_nontemporal_load(reinterpret_cast<const v4i_any_aligned *>(src + 2 * at[u]));
#pragma unroll
        for (int u = 0; u < PACK_PIECES; ++u) {
            v2i o;
            o.x = (int)(pack4((uint32_t)v[u].x) | (pack4((uint32_t)v[u].y) << 16));
            o.y = (int)(pack4((uint32_t)v[u].z) | (pack4((uint32_t)v[u].w) << 16));
            *reinterpret_cast<v2i_any_aligned *>(dst + at[u]) = o;
        }
    }
}

__global__ void pack_i4_byte_kernel(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, size_t nbytes)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < nbytes; i += (size_t)gridDim.x * blockDim.x)
        dst[i] = (uint8_t)((src[2 * i] & 0x0Fu) | ((src[2 * i + 1] & 0x0Fu) << 4));
}

// 4 packed bytes -> 8 int8: widen nibbles to bytes, sign-extend (bit 3 set => OR 0xF0),
// interleave even/odd elements back into K order.
__device__ __forceinline__ uint32_t sext_nibbles(uint32_t x)  // x = 0x0n0n0n0n
{
    const uint32_t t = x & 0x08080808u;
    return x | ((t << 5) - (t << 1));  // 0x08 -> 0xF0 in each byte (the top byte wraps mod 2^32)
}

__device__ __forceinline__ v2i unpack8(uint32_t w)
{
    const uint32_t ev = sext_nibbles(w & 0x0F0F0F0Fu), od = sext_nibbles((w >> 4) & 0x0F0F0F0Fu);
    // bytes: ev0 od0 ev1 od1 | ev2 od2 ev3 od3
    return v2i{(int)__builtin_amdgcn_perm(od, ev, 0x05010400u), (int)__builtin_amdgcn_perm(od, ev, 0x07030602u)};
}

// At least 8 packed bytes at any address, the last piece as in pack_i4_vec_kernel.  Bound: the stores, two
// thirds of the traffic: 16 bytes per lane, non-temporal (us, 8 bytes per lane and plain stores / 16
// and plain / 16 and non-temporal: 8192 x 8192 22.5 / 20.3 / 16.1 = 6.3 TB/s, 16384 x 14336 74 / 63 / 52.5; 8 MB
// of values 4.2 / 3.8 / 3.4).  A kernel that reads the values next finds fewer of them in the caches: this kernel
// and such a reader together 8 MB 8.2 / 7.7 / 7.9, 24 MB 19.4 / 18.2 / 20.0, 64 MB 43.1 / 40.5 / 43.4, 192 MB 126 / 121 / 116.
__global__ void __launch_bounds__(PACK_THREADS) unpack_i4_vec_kernel(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, size_t nbytes)
{
    for (size_t i = (size_t)blockIdx.x * PACK_THREADS + threadIdx.x; 8 * i < nbytes; i += (size_t)gridDim.x * PACK_THREADS) {
        const size_t at = min(8 * i, nbytes - 8);
        const v2i w = *reinterpret_cast<const v2i_any_aligned *>(src + at);
        const v2i lo = unpack8((uint32_t)w.x), hi = unpack8((uint32_t)w.y);
        __builtin_nontemporal_store(v4i{lo.x, lo.y, hi.x, hi.y}, reinterpret_cast<v4i_any_aligned *>(dst + 2 * at));
    }
}

__global__ void unpack_i4_byte_kernel(const uint8_t *__restrict__ src, int8_t *__restrict__ dst, size_t nbytes)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < nbytes; i += (size_t)gridDim.x * blockDim.x) {
        const uint32_t b = src[i];
        dst[2 * i] = (int8_t)s4_lo(b);
        dst[2 * i + 1] = (int8_t)s4_hi(b);
    }
}

// --------------------------------------------------------------------------
// Per-row symmetric quantisation to int4 fused with the packing, the row held in registers
// between the two passes over it (maximum, then quantise), so HBM is read once.  x is fp16,
// bf16 or fp32; 8 elements (4 packed bytes) per lane and chunk.
//
// Any even k from 8 up and any address: rows are loaded and stored at whatever alignment they
// have (the memory pipeline splits at cache lines), and the last chunk of a row is its last 8
// elements -- those that the chunk before has too are quantised twice to the same bytes.
// Lanes without a chunk load that last one as well and store nothing, so all loads of a
// lane are in flight together (behind a branch per chunk each waited for the one before).
// --------------------------------------------------------------------------
template <int IN> struct QuantIn;
template <> struct QuantIn<QM_IN_F16> {
    static constexpr int BYTES = 2, WORDS = 4;  // of an element, and 32-bit words per chunk
    static __device__ __forceinline__ float widen(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }
};
template <> struct QuantIn<QM_IN_BF16> {
    static constexpr int BYTES = 2, WORDS = 4;
    static __device__ __forceinline__ float widen(uint16_t h) { return __builtin_bit_cast(float, (uint32_t)h << 16); }
};
template <> struct QuantIn<QM_IN_F32> {
    static constexpr int BYTES = 4, WORDS = 8;
};

template <int IN>
struct Chunk8 {
    v4i w[QuantIn<IN>::WORDS / 4];
    __device__ __forceinline__ void load(const uint8_t *src)
    {
#pragma unroll
        for (int i = 0; i < QuantIn<IN>::WORDS / 4; ++i) {
            if constexpr (IN == QM_IN_F32) w[i] = *reinterpret_cast<const v4i_elem_aligned *>(src + 16 * i);
            else w[i] = *reinterpret_cast<const v4i_half_aligned *>(src + 16 * i);
        }
    }
    __device__ __forceinline__ float at(int e) const
    {
        if constexpr (IN == QM_IN_F32) {
            const int d = w[e >> 2][e & 3];
            return __builtin_bit_cast(float, d);
        } else {
            const uint32_t d = (uint32_t)w[0][e >> 1];
            return QuantIn<IN>::widen((uint16_t)((e & 1) ? d >> 16 : d & 0xFFFFu));
        }
    }
    __device__ __forceinline__ float amax(float m) const
    {
#pragma unroll
        for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(at(e)));
        return m;
    }
};

// 8 elements -> 8 nibbles, element e in nibble e (low nibble = even k, test.py:8,14).  The clamp is
// one v_med3_f32, which takes a NaN to -7 as fmin(fmax()) does.  The rounded values are
// small integers, put together in fp32 four at a time without any rounding:
// 2^23 + sum((n_e + 8) 16^e) < 2^24, whose low 16 bits are the nibbles with their sign bits inverted.
__device__ __forceinline__ uint32_t quant4(float r0, float r1, float r2, float r3)
{
    float t = __builtin_fmaf(r3, 16.0f, r2);
    t = __builtin_fmaf(t, 16.0f, r1);
    t = __builtin_fmaf(t, 16.0f, r0 + (8388608.0f + 34952.0f));
    return __builtin_bit_cast(uint32_t, t);
}

template <int IN>
__device__ __forceinline__ uint32_t quant8(const Chunk8<IN> &c, float inv)
{
#pragma clang fp contract(off)
    float r[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = __builtin_amdgcn_fmed3f(__builtin_rintf(c.at(e) * inv), -7.0f, 7.0f);  // (round half to even)
    const uint32_t lo = quant4(r[0], r[1], r[2], r[3]), hi = quant4(r[4], r[5], r[6], r[7]);
    return __builtin_amdgcn_perm(hi, lo, 0x05040100u) ^ 0x88888888u;
}

// The same for fp16 in fewer instructions, where no clamp is needed: no NaN among the elements, the row's maximum and inv finite (|c inv|
// <= 7 and a rounding).  The product is rounded as above, then to an integer, half to even, by the addition of 1.5 * 2^23 + 8, whose
// last bits then count n + 8; the bits of eight such sums are added up sixteen-fold, and what the constant leaves in them is taken
// away.  With the maximum on bit patterns (chunks_amax) 4.1 vector instructions per element where one
// element after the other takes 8: in a graph, us, before -> now, 2048 x 4096 5.76 -> 5.46, 2048 x 8192 8.94 -> 8.56, 8192 x 1024 5.77 ->
// 5.41 (few rows and short ones lose: quantise_many).  bf16, which needs an instruction more to widen and had one less, was no faster (2048 x 8192 8.66 / 8.67).
__device__ __forceinline__ uint32_t quant8_plain(const Chunk8<QM_IN_F16> &c, const float inv)
{
    constexpr float round_to = 12582912.0f + 8.0f;
    constexpr uint32_t left = 0x4B400000u + (0x4B400000u << 4) + (0x4B400000u << 8);  // (further up it has no bits)
    uint32_t sum = 0;
#pragma unroll
    for (int e = 7; e >= 0; --e) {
        // (the widening and the product in one; + 0 only makes a zero positive)
        float t;
        if (e & 1) asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(t) : "v"(c.w[0][e >> 1]), "v"(inv));
        else asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[1,0,0]" : "=v"(t) : "v"(c.w[0][e >> 1]), "v"(inv));
        sum = (sum << 4) + __builtin_bit_cast(uint32_t, t + round_to);
    }
    return (sum - left) ^ 0x88888888u;
}

// The largest magnitude among a lane's chunks, NaNs left out.  fp16: on the bit patterns, two at a time; `plain` comes back false where
// the wave has a NaN, and for the other types.
template <int IN, int NC>
__device__ __forceinline__ float chunks_amax(const Chunk8<IN> (&v)[NC], bool &plain)
{
    plain = false;
    if constexpr (IN == QM_IN_F16) {
        typedef uint16_t v2u __attribute__((ext_vector_type(2)));
        v2u m = {0, 0};
#pragma unroll
        for (int i = 0; i < NC; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int w = v[i].w[0][e] & 0x7FFF7FFF;
                m = __builtin_elementwise_max(m, __builtin_bit_cast(v2u, w));
            }
        const uint16_t most = m.x > m.y ? m.x : m.y;
        plain = !__any(most > 0x7C00);
        if (plain) return QuantIn<IN>::widen(most);
    }
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < NC; ++i) amax = v[i].amax(amax);
    return amax;
}
// put(quant) with the quantisation of a chunk that does for these, the same for the whole wave
template <int IN, class Put>
__device__ __forceinline__ void quantise_chunks(const bool plain, const float amax, const float inv, Put &&put)
{
    if constexpr (IN == QM_IN_F16) {
        if (plain && fmaxf(amax, inv) < __builtin_inff()) {
            put([&](const Chunk8<IN> &c) __attribute__((always_inline)) { return quant8_plain(c, inv); });
            return;
        }
    }
    put([&](const Chunk8<IN> &c) __attribute__((always_inline)) { return quant8(c, inv); });
}

// maximum over the NW waves that share a row (one row per workgroup unless NW == 1)
template <int NW>
__device__ __forceinline__ float row_max(float x, float *lds)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) x = fmaxf(x, __shfl_xor(x, off));
    if constexpr (NW > 1) {
        if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = x;
        __syncthreads();
        x = lds[0];
#pragma unroll
        for (int w = 1; w < NW; ++w) x = fmaxf(x, lds[w]);
    }
    return x;
}

// NW waves per row (4 rows per workgroup if one), NC chunks of 8 elements per lane: k <= 512 * NW * NC.
// NC == 0: any k, the row read twice (the second time out of the L2).
// MANY: fp16 by quant8_plain, which has fewer instructions and a longer chain of them (see quantise_many).
template <int IN, int NW, int NC, bool MANY>
__global__ void __launch_bounds__(NW == 1 ? 256 : 64 * NW) quantize_pack_kernel(const uint8_t *__restrict__ x, uint8_t *__restrict__ dst, float *__restrict__ scales, int rows, int k)
{
    __shared__ float red[NW];
    const int row = NW == 1 ? blockIdx.x * 4 + (threadIdx.x >> 6) : blockIdx.x;
    const int lane = NW == 1 ? threadIdx.x & 63 : threadIdx.x;  // within the row
    if (NW == 1 && row >= rows) return;
    const int nchunks = (k + 7) >> 3;
    const uint8_t *xr = x + (size_t)row * k * QuantIn<IN>::BYTES;
    uint8_t *out = dst + (size_t)row * (k >> 1);
    const auto first = [&](int c) { return min(8 * c, k - 8); };
    float amax = 0.0f;
    if constexpr (NC > 0) {
        Chunk8<IN> v[NC];
#pragma unroll
        for (int i = 0; i < NC; ++i) v[i].load(xr + first(lane + i * 64 * NW) * QuantIn<IN>::BYTES);
        bool plain = false;
        if constexpr (MANY) {
            amax = chunks_amax(v, plain);
        } else {
#pragma unroll
            for (int i = 0; i < NC; ++i) amax = v[i].amax(amax);
        }
        amax = row_max<NW>(amax, red);
        const float inv = amax > 0.0f ? 7.0f / amax : 0.0f;
        if (lane == 0) scales[row] = amax / 7.0f;
        if constexpr (MANY) {
            quantise_chunks<IN>(plain, amax, inv, [&](auto quant) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < NC; ++i) {
                    const int c = lane + i * 64 * NW;
                    const uint32_t q = quant(v[i]);
                    if (c < nchunks) *reinterpret_cast<u32_any_aligned *>(out + (first(c) >> 1)) = q;
                }
            });
        } else {
            // (not through the same function: bf16 and fp32 lost 1 to 2 % on three and four chunks to the order that the compiler gave the loads)
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                const int c = lane + i * 64 * NW;
                const uint32_t q = quant8(v[i], inv);
                if (c < nchunks) *reinterpret_cast<u32_any_aligned *>(out + (first(c) >> 1)) = q;
            }
        }
    } else {
        Chunk8<IN> v;
        for (int c = lane; c < nchunks; c += 64 * NW) {
            v.load(xr + (size_t)first(c) * QuantIn<IN>::BYTES);
            amax = v.amax(amax);
        }
        amax = row_max<NW>(amax, red);
        const float inv = amax > 0.0f ? 7.0f / amax : 0.0f;
        if (lane == 0) scales[row] = amax / 7.0f;
        for (int c = lane; c < nchunks; c += 64 * NW) {
            v.load(xr + (size_t)first(c) * QuantIn<IN>::BYTES);
            *reinterpret_cast<u32_any_aligned *>(out + (first(c) >> 1)) = quant8(v, inv);
        }
    }
}

// k < 8: one pair of elements per thread and pass
template <int IN>
__global__ void __launch_bounds__(256) quantize_pack_scalar_kernel(const uint8_t *__restrict__ x, uint8_t *__restrict__ dst, float *__restrict__ scales, int k)
{
#pragma clang fp contract(off)
    __shared__ float red[4];
    const int row = blockIdx.x, tid = threadIdx.x;
    auto at = [&](int j) -> float {
        if constexpr (IN == QM_IN_F32) {
            return reinterpret_cast<const float *>(x)[(size_t)row * k + j];
        } else {
            return QuantIn<IN>::widen(reinterpret_cast<const uint16_t *>(x)[(size_t)row * k + j]);
        }
    };
    float amax = 0.0f;
    for (int j = tid; j < k; j += 256) amax = fmaxf(amax, fabsf(at(j)));
    amax = row_max<4>(amax, red);
    const float inv = amax > 0.0f ? 7.0f / amax : 0.0f;
    if (tid == 0) scales[row] = amax / 7.0f;
    for (int j = 2 * tid; j < k; j += 512) {
        const float r0 = fminf(fmaxf(__builtin_rintf(at(j) * inv), -7.0f), 7.0f), r1 = fminf(fmaxf(__builtin_rintf(at(j + 1) * inv), -7.0f), 7.0f);
        dst[(size_t)row * (k >> 1) + (j >> 1)] = (uint8_t)(((int)r0 & 0xF) | (((int)r1 & 0xF) << 4));
    }
}

// Where the arithmetic of fp16 rows, and not the launch and the way there and back, is what they take.  quant8_plain over quant8, in a graph, over
// 7000 sizes: to a K of 2048 1.03 on 16 to 512 rows, 1.01 on 513 to 1024, 0.95 beyond; to 4096 1.01, 0.99 from 257 rows on, 0.92 from 1025 on; above 1.00 to
// 0.94 on few rows, 0.96 to 0.87 on more.
inline bool quantise_many(int rows, int k) { return k > 4096 || rows > (k > 2048 ? 256 : 1024); }

template <int IN, int NW, int NC>
static hipError_t launch_quantize_rows(const uint8_t *x, uint8_t *dst, float *scales, int rows, int k, hipStream_t s)
{
    const auto kernel = IN == QM_IN_F16 && NC > 0 && quantise_many(rows, k) ? &quantize_pack_kernel<IN, NW, NC, IN == QM_IN_F16 && NC != 0> : &quantize_pack_kernel<IN, NW, NC, false>;
    constexpr int threads = NW == 1 ? 256 : 64 * NW, rows_per_block = NW == 1 ? 4 : 1;
    constexpr int most = (1 << 21) * rows_per_block;  // a grid has less than 2^32 threads
    for (int r0 = 0; r0 < rows; r0 += most) {
        const int n = rows - r0 < most ? rows - r0 : most;
        const hipError_t e = enqueue(kernel, dim3((unsigned)(n + rows_per_block - 1) / rows_per_block), dim3(threads), 0, s,
            x + (size_t)r0 * k * QuantIn<IN>::BYTES, dst + (size_t)r0 * (k / 2), scales + r0, n, k);
        if (e != hipSuccess || r0 > 0x7fffffff - most) return e;
    }
    return hipSuccess;
}

// Four waves per row: as many chunks per lane as the row takes, none of them empty.  A workgroup per row is
// as much dispatch as work on thousands of rows below 1536 elements, where each wave has
// a row of its own (us, wave / workgroup per row: 8191 x 1030 bf16 6.3 / 8.7, 2048 x 1024 2.85 / 3.2, but
// 2048 x 4096 6.0 / 5.5, 256 x 4096 3.1 / 2.6); beyond 12288 sixteen waves hold a row in two chunks per lane
// (sixteen / four: 8192 x 14336 f32 94.5 / 103.5, 64 x 14336 3.0 / 3.2, but 2048 x 8192 11.1 / 9.0).
// Against one chunk after the other, and one element per thread where k % 8 != 0: 2048 x 8192 bf16
// 12.1 -> 9.0 us (4.6 TB/s), 8 x 11008 3.5 -> 2.65, 2048 x 8194 24.8 -> 9.4, 8191 x 1030 18.5 -> 6.3.
template <int IN>
static hipError_t launch_quantize_pack(const void *x, void *dst, float *scales, int rows, int k, hipStream_t s)
{
    const uint8_t *xb = static_cast<const uint8_t *>(x);
    uint8_t *db = static_cast<uint8_t *>(dst);
    if (k < 8) return enqueue(&quantize_pack_scalar_kernel<IN>, dim3(rows), dim3(256), 0, s, xb, db, scales, k);
    if (k > 16384) return launch_quantize_rows<IN, 16, 0>(xb, db, scales, rows, k, s);
    if (k > 12288) return launch_quantize_rows<IN, 16, 2>(xb, db, scales, rows, k, s);
    if (rows > 1024 && k <= 512) return launch_quantize_rows<IN, 1, 1>(xb, db, scales, rows, k, s);
    if (rows > 1024 && k <= 1024) return launch_quantize_rows<IN, 1, 2>(xb, db, scales, rows, k, s);
    if (rows > 1024 && k <= 1536) return launch_quantize_rows<IN, 1, 3>(xb, db, scales, rows, k, s);
    if (k <= 2048) return launch_quantize_rows<IN, 4, 1>(xb, db, scales, rows, k, s);
    if (k <= 4096) return launch_quantize_rows<IN, 4, 2>(xb, db, scales, rows, k, s);
    if (k <= 6144) return launch_quantize_rows<IN, 4, 3>(xb, db, scales, rows, k, s);
    if (k <= 8192) return launch_quantize_rows<IN, 4, 4>(xb, db, scales, rows, k, s);
    if (k <= 10240) return launch_quantize_rows<IN, 4, 5>(xb, db, scales, rows, k, s);
    return launch_quantize_rows<IN, 4, 6>(xb, db, scales, rows, k, s);
}

static unsigned flat_grid(size_t items, unsigned block, size_t most = 256u * 32u)
{
    size_t g = (items + block - 1) / block;
    if (g < 1) g = 1;
    if (g > most) g = most;
    return (unsigned)g;
}

}  // namespace qm

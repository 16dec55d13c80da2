// Q4_K and MXFP4 matmul for many activation rows on f16 and FP6 matrix instructions.
//
// Per 256-element super-block of weight row n and activation row m (reference arithmetic w = d sc q - dmin m,
// src/kquant_dot.rs:440-465), with the codes taken about their middle,
//
//   sum_k x_k w_k = d s sum_k x'_k p_k + sum_j X_j W_j,    p = sc (q - 8),  W_j = 8 d sc_j - dmin m_j,  X_j = sum of x over sub-block j
//
// where x' = x / s, s the power of two that takes the super-block's largest magnitude to 2^14 .. 2^15.  p is an integer of magnitude up
// to 504, so exact in f16.  x' = h + l, h = f16(x'), and
//
//   x' p = h p + l p:   h p on v_mfma_f32_16x16x32_f16, exact products;   l p, 2^-12 of it, on v_mfma_scale_f32_16x16x128_f8f6f4 with
//                       both factors rounded to E2M3, 1/4 of the cycles.  p's codes stand on a scale of their own sub-block, the power of
//                       two in sc / 32, so that they use E2M3's range whatever sc is (one scale for all, that of sc = 32..63, left
//                       nothing of l p where sc is 1: 2.0e-4 off).  l's stand on the super-block's: at most 8, clamped at 7.5.
//
// into one f32 sum; the second term is one v_mfma_f32_16x16x32_bf16 a super-block with X and W in two bf16 parts each, added to
// the result unscaled.  Off 64 bits (relative 2-norm, 160 x 1024 x 2048; in front of each the int8 GEMM's 16-bit fixed point,
// kernels_mfma_q4k_gemm_i8.hpp): normal activations 2.7e-5 / 0.9e-5 against quantized normal weights, 2.7e-5 / 0.5e-5 against random
// blocks, 2.7e-5 / 0.8e-5 .. 0.6e-5 against blocks with scales up to 63 .. 1 whose weights lie about zero; cubes of normal numbers
// 7.1e-5 / 1.3e-5; one activation in 256 a hundred times the others 1.4e-4 / 2.0e-5.  Only rows that fixed point happens to hold
// exactly, one non-zero activation a super-block (1e-7 / 0.8e-5) or all of them equal (1e-6 / 3.9e-5), are further off here.
// Taking q about 8 is worth a factor of 2.5: the codes' common part, which the min term would take away again, stays out of l p.
//
// Why: the int8 GEMM needs 16 instructions of 16 cycles for 16 x 16 x 256 of the product and seven vector instructions for every
// output and super-block to join its three integer sums; here it is 11 and two (the factor d s, the addition).
//
// Workgroup: NW waves, tile 32 NW activation rows x 16 NG weight rows; a wave owns 32 activation rows against all 16 NG weight
// rows.  Wave w unpacks the 16 weight rows of group w, a sub-block a lane, one half of a super-block (128 k) ahead of the
// multiplication, into one of two LDS buffers of operand-ordered halves (one barrier a half); the activations come prepared in
// operand order (kq_gemm_h6_prep) straight from global memory, four f16 steps ahead.  k runs outside the groups of weight rows,
// so that these loads spread over the whole iteration: with the groups outside and a super-block's operands kept in registers
// all 200 KB were asked for in the last seventh of an iteration, 7 % slower at 512 x 14336 x 4096.
//
// Groups: seven make 256 workgroups of 512 x 14336, eight of 2048 x 4096 (calls: 156 -> 110 us, with rows of 12288 400 -> 317, against
// the better of six groups' 344 workgroups and small tiles) and, with k in four parts, of 512 x 4096 (51 -> 44); nothing fits more.
//
// 512 x 14336 x 4096: 90 us of kernel where the int8 GEMM takes 112 (kernel trace, calls back to back), of the calls' 91 and 112
// among others, 95 and 116 back to back.  Of 151 500 clocks that the chip is busy the matrix cores work 78 800 and the LDS moves
// operands for 60 400 (counters): neither is full, and two waves a SIMD have a barrier every half super-block.  Waves of 64
// activation rows (four a workgroup, half the LDS reads) take 131 us: one wave a SIMD has nothing to hide its vector instructions
// behind.  E2M1 codes of p, a third less to read, would be 2.6e-5 off 64 bits.  The codes' scales cost 1.3 us of a call.
// MXFP4 has no mins and no codes to make: behind the super-block's largest scale a weight is exact in f16, made by one conversion for
// two, and E2M1, what the second instruction multiplies, is its code as it stands in memory, on the block's own scale.  512 x 14336 x
// 4096: 112 -> 87 us a call, 333 x 4096 x 12288 109 -> 79, 2048 x 4096 x 12288 427 -> 277; 2.7e-5 -> 0.57e-5 off 64 bits.  Q6_K and Q8_0, whose
// weights take 12 and 18 bits, were built here too, the weights' own remainders as E2M1 against the activations as E2M3: no faster
// than the int8 GEMM (512 x 14336 x 4096 148 and 143 us against 128 and 130; unpacking twice Q4_K's instructions, and registers for six groups).
#pragma once
#include "kernels_graph.hpp"

#include <utility>

namespace jq {

// f(0), .., f(N - 1) with the index as a constant
template <class F, int... I>
__device__ __forceinline__ void h6_each(std::integer_sequence<int, I...>, F f) { (f(std::integral_constant<int, I>{}), ...); }

typedef _Float16 h6_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h6_h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h6_h32 __attribute__((ext_vector_type(32)));
typedef __bf16 h6_b8 __attribute__((ext_vector_type(8)));
typedef uint32_t h6_u4 __attribute__((ext_vector_type(4)));
typedef uint32_t h6_u2 __attribute__((ext_vector_type(2)));
typedef uint32_t h6_u6 __attribute__((ext_vector_type(6)));
typedef int h6_i8 __attribute__((ext_vector_type(8)));
typedef float h6_f4 __attribute__((ext_vector_type(4)));

// Prepared activations, per (group of 16 activation rows, super-block).  Lane (i = lane % 16, g = lane / 16) of half h
// holds sub-block 4 h + g (32 elements) of row i:
//   2 halves x 4 steps x 64 lanes x 16 bytes: f16(x'), elements 8 s + H6_ORDER of step s
//   2 halves x (64 lanes x 16 bytes, then 64 lanes x 8): the 32 remainders x' - f16(x') as E2M3 in the same order
//   64 lanes x 16 bytes: the operand of the min term
//   the 16 scales
// (MXFP4: no operand of a min term)
constexpr int H6_HI = 8192, H6_LO_HALF = 1536, H6_MIN = H6_HI + 2 * H6_LO_HALF, H6_SCALE = H6_MIN + 1024, H6_REC = H6_SCALE + 64;
template <bool MINS>
constexpr int h6_rec() { return MINS ? H6_REC : H6_MIN + 64; }

// Whether the kernel's offsets hold rows of that many super-blocks: a record's from the start of its row group in 31 bits, a weight
// block's from the first of 16 rows in 32.
constexpr bool h6_offsets_hold(size_t nb, size_t row_bytes) { return nb <= 0x7FFFFFFFu / H6_REC && row_bytes <= (size_t)1 << 27; }

__device__ __forceinline__ uint32_t h6_bf16_bits(float x) {
    return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)x);
}
__device__ __forceinline__ float h6_bf16_value(uint32_t b) { return __builtin_bit_cast(float, b << 16); }

// grid (k / 256 super-blocks, groups of 16 activation rows), 128 threads, one sub-block each.  Rows from m_rows on are
// zero operands.  With PAIRS the activations are silu(gate) * up over rows of 2 k floats in which gate_j and up_j alternate.
//
// Memory bounds it.  A lane's own sub-block is 128 bytes, so its loads touch a line a lane.  That costs nothing while the
// caches hold the rest of the line (8.0 us at 512 x 14336, either way), but the pairs' 256 bytes a lane do not survive there: 2048 x
// 12288 pairs took 86 us so and take 50 with whole rows of memory turned by the LDS, of 54 that 276 MB take in a large copy.  For
// plain rows the detour costs 1 us.  rows_sh's padding: 16 lanes that read 16 rows at one column take 16 different groups of banks.
// NIBBLES: positions 2 j and 2 j + 1 of a sub-block hold elements j and j + 16 (MXFP4's bytes), else H6_ORDER's.
template <bool PAIRS, bool MINS, bool NIBBLES>
static __global__ __launch_bounds__(128) void kq_gemm_h6_prep(const float *__restrict__ X, int m_rows, int k, uint8_t *__restrict__ out) {
    __shared__ float amax_sh[2][16], xs_sh[16][8];
    const int tid = threadIdx.x, lane = tid & 63, h = tid >> 6, i = lane & 15, g = lane >> 4;
    const int b = blockIdx.x, row = 16 * (int)blockIdx.y + i;
    uint8_t *rec = out + ((size_t)blockIdx.y * gridDim.x + b) * h6_rec<MINS>();
    float v[32];
    if constexpr (PAIRS) {
        __shared__ __align__(16) float rows_sh[16][260];
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const int r = 8 * h + q, at = 16 * (int)blockIdx.y + r;
            float4 a = {0.0f, 0.0f, 0.0f, 0.0f};
            if (at < m_rows) {
                const float4 *src = (const float4 *)(X + 2 * ((size_t)at * k + 256 * b + 4 * lane));
                const float4 u = src[0], w = src[1];
                a = {silu(u.x) * u.y, silu(u.z) * u.w, silu(w.x) * w.y, silu(w.z) * w.w};
            }
            *(float4 *)&rows_sh[r][4 * lane] = a;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const float4 a = *(const float4 *)&rows_sh[i][32 * (4 * h + g) + 4 * q];
            v[4 * q] = a.x, v[4 * q + 1] = a.y, v[4 * q + 2] = a.z, v[4 * q + 3] = a.w;
        }
    } else if (row < m_rows) {
        const float4 *src = (const float4 *)(X + (size_t)row * k + 256 * b + 32 * (4 * h + g));
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const float4 a = src[q];
            v[4 * q] = a.x, v[4 * q + 1] = a.y, v[4 * q + 2] = a.z, v[4 * q + 3] = a.w;
        }
    } else {
#pragma unroll
        for (int e = 0; e < 32; e++) v[e] = 0.0f;
    }
    float amax = 0.0f;
#pragma unroll
    for (int e = 0; e < 32; e++) amax = fmaxf(amax, mag_or_inf(v[e]));
    amax = max_xor32(max_xor16(amax));
    if (g == 0) amax_sh[h][i] = amax;
    __syncthreads();
    amax = fmaxf(amax_sh[0][i], amax_sh[1][i]);
    // the power of two that takes the largest magnitude to 2^14 .. 2^15; exact unless the result is below f32's normal range
    const uint32_t e = min(max(__builtin_bit_cast(uint32_t, amax) >> 23, 15u), 254u);
    const bool live = amax < INFINITY;
    float inv = live ? __builtin_bit_cast(float, (268u - e) << 23) : 0.0f;
    float s = !live ? NAN : amax > 0.0f ? __builtin_bit_cast(float, (e - 14u) << 23) : 0.0f;
    if constexpr (!MINS) {
        // What takes the largest to 2^15 itself suits f16 and E2M3 better: magnitudes that are all alike, or few binary fractions of the largest,
        // come out whole (6e-6 off behind the power of two), normal ones 5.7e-6 off for 6.1e-6.  But not where f16 holds every element
        // behind the power of two, as it does those of bf16 activations.
        __shared__ bool whole_sh[2][16];
        bool whole = true;
#pragma unroll
        for (int q = 0; q < 32; q++) whole &= (float)(_Float16)(v[q] * inv) == v[q] * inv;
        const uint64_t all = __ballot(whole), row_lanes = 0x0001000100010001ull << i;
        if (g == 0) whole_sh[h][i] = (all & row_lanes) == row_lanes;
        __syncthreads();
        if (live && amax >= 0x1p-100f && !(whole_sh[0][i] && whole_sh[1][i])) inv = 32768.0f / amax, s = amax * 0x1p-15f;
    }
    float sum = 0.0f;
    h6_h32 hi, lo;
#pragma unroll
    for (int q = 0; q < 32; q++) {
        // position 8 s + p holds element 8 s + {0, 2, 1, 3, 4, 6, 5, 7}[p]: the order in which two of a word's nibbles
        // fall into one register (H6Q4K::piece)
        const int at = NIBBLES ? (q >> 1) + 16 * (q & 1) : (q & ~3) | ((q & 1) << 1) | ((q >> 1) & 1);
        const float x = live ? v[at] * inv : 0.0f;
        hi[q] = (_Float16)x;
        const float r = x - (float)hi[q];
        lo[q] = (_Float16)fminf(fmaxf(r, -7.5f), 7.5f);
    }
    if constexpr (MINS) {
        if (live) {
#pragma unroll
            for (int q = 0; q < 32; q++) sum += v[q] * 0.03125f;
        }
        xs_sh[i][4 * h + g] = sum;
    }
#pragma unroll
    for (int st = 0; st < 4; st++) {
        h6_h8 p;
#pragma unroll
        for (int q = 0; q < 8; q++) p[q] = hi[8 * st + q];
        *(h6_h8 *)(rec + ((4 * h + st) * 64 + lane) * 16) = p;
    }
    const h6_u6 six = __builtin_amdgcn_cvt_scalef32_pk32_fp6_f16(lo, 1.0f);
    *(h6_u4 *)(rec + H6_HI + h * H6_LO_HALF + lane * 16) = h6_u4{six[0], six[1], six[2], six[3]};
    *(h6_u2 *)(rec + H6_HI + h * H6_LO_HALF + 1024 + lane * 8) = h6_u2{six[4], six[5]};
    if constexpr (MINS) __syncthreads();
    if (MINS && h == 0) {  // lane groups 0 and 2: bf16 of the eight means, 1 and 3: what is left of them
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            uint32_t pair = 0;
#pragma unroll
            for (int z = 0; z < 2; z++) {
                const float x = xs_sh[i][2 * j + z];
                const uint32_t first = h6_bf16_bits(x);
                const uint32_t bits = (g & 1) ? h6_bf16_bits(x - h6_bf16_value(first)) : first;
                pair |= bits << (16 * z);
            }
            w[j] = pair;
        }
        *(h6_u4 *)(rec + H6_MIN + lane * 16) = h6_u4{w[0], w[1], w[2], w[3]};
    }
    if (tid < 16) ((float *)(rec + h6_rec<MINS>() - 64))[tid] = s;
}

// LDS: for either half of a super-block and every 16 weight rows 4 steps x 64 lanes x 16 bytes of f16 operands, then
// their E2M3 codes (64 lanes x 16 bytes and x 8); behind the halves, twice (by the super-block's parity), for every 16 rows
// the min operand's two parts (16 rows x 16 bytes each) and the 16 factors d; behind those, for either half, the exponents of
// the codes' scales, 64 lanes x 8 groups of 16 rows: one read gives a lane those of all groups.
// (MXFP4's codes: E2M1, 64 lanes x 16 bytes, no min operand.)
constexpr int H6_T_LO = 4096, H6_HALF = H6_T_LO + 1536, H6_META = 512 + 64, H6_EXPS = 512;
template <int NG>
constexpr int h6_lds_bytes() { return 2 * NG * (H6_HALF + H6_META) + 2 * H6_EXPS; }

// Memory behind an address that is the same in all lanes of a wave, read at a scalar and a lane's own offset: neither costs a
// vector instruction or a register pair, as the lanes' 64-bit addresses would.
struct H6Memory {
    __amdgpu_buffer_rsrc_t at;
    __device__ __forceinline__ explicit H6Memory(const uint8_t *base)
        : at(__builtin_amdgcn_make_buffer_rsrc((void *)base, 0, 0xFFFFFFFFu, 0x00027000)) {}
    __device__ __forceinline__ h6_u4 load16(uint32_t scalar, uint32_t lane) const {
        return __builtin_amdgcn_raw_buffer_load_b128(at, (int)lane, (int)scalar, 0);
    }
    __device__ __forceinline__ h6_u2 load8(uint32_t scalar, uint32_t lane) const {
        return __builtin_amdgcn_raw_buffer_load_b64(at, (int)lane, (int)scalar, 0);
    }
    __device__ __forceinline__ uint32_t load4(uint32_t scalar, uint32_t lane) const {
        return __builtin_amdgcn_raw_buffer_load_b32(at, (int)lane, (int)scalar, 0);
    }
};

// A format's side.  Lane (row i = lane % 16, g = lane / 16) of the wave that unpacks 16 weight rows takes the 32 elements of
// sub-block 4 h + g of its row for half h.
struct H6Q4K {  // w = d sc (q - 8) + (8 d sc - dmin m), 6-bit sc and m, q in 0..15
    static constexpr int BLOCK = 144, ALIGN = 16, LOW = 2;  // LOW: the codes' format, 2: E2M3, 4: E2M1
    static constexpr bool MINS = true, NIBBLES = false;
    static constexpr float D_UNIT = 128.0f;  // the operand is p / 2^7, p = sc (q - 8)
    struct Raw {
        h6_u4 hdr, q0, q1;
        h6_h2 sc, off;  // 2^10 sc and -sc / 16
        float unit;     // the codes' scale, a power of two: sc / 32 with its mantissa cleared
        h6_h32 p;
    };
    __device__ __forceinline__ static void fetch_header(const H6Memory &mem, uint32_t blk, uint32_t row_at, int, int, Raw &raw) {
        raw.hdr = mem.load16(blk, row_at);
    }
    __device__ __forceinline__ static void fetch(const H6Memory &mem, uint32_t blk, uint32_t row_at, int g, int h, Raw &raw) {
        raw.q0 = mem.load16(blk + 16 + 64 * h, row_at + 32 * (uint32_t)(g >> 1));
        raw.q1 = mem.load16(blk + 32 + 64 * h, row_at + 32 * (uint32_t)(g >> 1));
    }
    // The sub-block's scale and its codes'; its part of the row's min operand, and d.
    __device__ __forceinline__ static void header(Raw &raw, int g, int i, int h, uint8_t *meta, uint8_t *exponent) {
        const h6_u4 hdr = raw.hdr;
        const uint32_t s4 = h == 0 ? hdr.y & 0x3F3F3F3Fu : (hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u);
        const uint32_t m4 = h == 0 ? hdr.z & 0x3F3F3F3Fu : ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u);
        const float sc = (float)((s4 >> (8 * g)) & 0xFFu), mn = (float)((m4 >> (8 * g)) & 0xFFu);
        const _Float16 sc16 = (_Float16)(1024.0f * sc), off16 = (_Float16)(-0.0625f * sc);
        raw.sc = h6_h2{sc16, sc16}, raw.off = h6_h2{off16, off16};
        const uint32_t unit = __builtin_bit_cast(uint32_t, 0.03125f * fmaxf(sc, 1.0f)) & 0x7F800000u;
        raw.unit = __builtin_bit_cast(float, unit), *exponent = (uint8_t)(unit >> 23);
        const float d = f16_bits(hdr.x), dmin = f16_bits(hdr.x >> 16);
        const float w = fmaf(256.0f * d, sc, -(32.0f * dmin) * mn);
        const uint32_t first = h6_bf16_bits(w);
        *(uint16_t *)(meta + i * 16 + 2 * (4 * h + g)) = (uint16_t)first;
        *(uint16_t *)(meta + 256 + i * 16 + 2 * (4 * h + g)) = (uint16_t)h6_bf16_bits(w - h6_bf16_value(first));
        if (h == 0) *(float *)(meta + 512 + 4 * i) = D_UNIT * d;  // the same from all four
    }
    // The u-th of 16 pairs of elements; every fourth ends a run of eight, which is stored.
    template <int U>
    __device__ __forceinline__ static void pair(Raw &raw, int g, int lane, uint8_t *tile) {
        constexpr int st = U / 4, half = U / 2 % 2, odd = U % 2;
        const h6_u4 qv = st < 2 ? raw.q0 : raw.q1;
        const uint32_t word = (st & 1) ? (half ? qv.w : qv.z) : (half ? qv.y : qv.x);
        // two nibbles, bits 0.. or 4.. of every other byte, as the f16 numbers 2^-17 q (bits 7..10: below 2^-13 f16 is a fixed-point
        // number, no exponent to be put in), times 2^10 sc
        const uint32_t two = (odd ? word >> (1 + 4 * (g & 1)) : word << (7 - 4 * (g & 1))) & 0x07800780u;
        const h6_h2 v = __builtin_elementwise_fma(__builtin_bit_cast(h6_h2, two), raw.sc, raw.off);
        raw.p[2 * U] = v[0], raw.p[2 * U + 1] = v[1];
        if constexpr (U % 4 == 3)
            *(h6_h8 *)(tile + (st * 64 + lane) * 16) = h6_h8{raw.p[8 * st], raw.p[8 * st + 1], raw.p[8 * st + 2], raw.p[8 * st + 3],
                                                             raw.p[8 * st + 4], raw.p[8 * st + 5], raw.p[8 * st + 6], raw.p[8 * st + 7]};
    }
    __device__ __forceinline__ static void codes(Raw &raw, int lane, uint8_t *tile) {
        const h6_u6 six = __builtin_amdgcn_cvt_scalef32_pk32_fp6_f16(raw.p, raw.unit);
        *(h6_u4 *)(tile + H6_T_LO + lane * 16) = h6_u4{six[0], six[1], six[2], six[3]};
        *(h6_u2 *)(tile + H6_T_LO + 1024 + lane * 8) = h6_u2{six[4], six[5]};
    }
};

// Blocks of 17 bytes start anywhere: what a lane needs comes in whole words that hold a byte of it, and is shifted.
struct H6MXFP4 {  // w = 2^(e - 127) E2M1: exact as f16 against the super-block's largest scale, and the codes are E2M1 themselves
    static constexpr int BLOCK = 136, ALIGN = 4, LOW = 4;
    static constexpr bool MINS = false, NIBBLES = true;
    struct Raw {
        h6_u4 q0;
        uint32_t q1, e0, e1, at, at_e;
        float scale;
        h6_u4 word;
        h6_h32 p;
    };
    __device__ __forceinline__ static void fetch_header(const H6Memory &mem, uint32_t blk, uint32_t row_at, int g, int, Raw &raw) {
        const uint32_t o = row_at + blk + 17 * (uint32_t)g;
        raw.e0 = mem.load4(0, o & ~3u), raw.e1 = mem.load4(68, o & ~3u), raw.at_e = o & 3u;
    }
    __device__ __forceinline__ static void fetch(const H6Memory &mem, uint32_t blk, uint32_t row_at, int g, int h, Raw &raw) {
        const uint32_t o = row_at + blk + 17 * (uint32_t)g + 1, a = o & ~3u;
        raw.at = o & 3u;
        raw.q0 = mem.load16(68 * h, a), raw.q1 = mem.load4(68 * h + 12, raw.at ? a + 4 : a);  // (the fifth word where it is needed)
    }
    __device__ __forceinline__ static void header(Raw &raw, int, int i, int h, uint8_t *meta, uint8_t *exponent) {
        const uint32_t e0 = (raw.e0 >> (8 * raw.at_e)) & 0xFFu, e1 = (raw.e1 >> (8 * raw.at_e)) & 0xFFu, e = h == 0 ? e0 : e1;
        const int most = (int)max_xor32(max_xor16(fmaxf(e0 == 0xFFu ? 0.0f : (float)e0, e1 == 0xFFu ? 0.0f : (float)e1)));
        const bool none = e == 0xFFu || (int)e < most - 60;  // 0xFF: a block of zeros
        const uint32_t by = none ? 0u : (uint32_t)(140 + (int)e - most);  // the largest scale takes codes to 6 x 2^13
        raw.scale = __builtin_bit_cast(float, by << 23), *exponent = (uint8_t)by;
        const uint32_t w[5] = {raw.q0.x, raw.q0.y, raw.q0.z, raw.q0.w, raw.q1};
#pragma unroll
        for (int j = 0; j < 4; j++) raw.word[j] = none ? 0u : __builtin_amdgcn_alignbyte(w[j + 1], w[j], raw.at);
        if (h == 0) *(float *)(meta + 512 + 4 * i) = ldexpf(1.0f, most - 140);
    }
    template <int U>
    __device__ __forceinline__ static void pair(Raw &raw, int, int lane, uint8_t *tile) {
        const h6_h2 v = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(raw.word[U / 4], raw.scale, U % 4);
        raw.p[2 * U] = v[0], raw.p[2 * U + 1] = v[1];
        if constexpr (U % 4 == 3) {
            constexpr int st = U / 4;
            *(h6_h8 *)(tile + (st * 64 + lane) * 16) = h6_h8{raw.p[8 * st], raw.p[8 * st + 1], raw.p[8 * st + 2], raw.p[8 * st + 3],
                                                             raw.p[8 * st + 4], raw.p[8 * st + 5], raw.p[8 * st + 6], raw.p[8 * st + 7]};
        }
    }
    __device__ __forceinline__ static void codes(Raw &raw, int lane, uint8_t *tile) { *(h6_u4 *)(tile + H6_T_LO + lane * 16) = raw.word; }
};

__device__ __forceinline__ h6_i8 h6_operand6(h6_u6 v) {
    return h6_i8{(int)v[0], (int)v[1], (int)v[2], (int)v[3], (int)v[4], (int)v[5], 0, 0};
}

// SWIGLU: the weight rows are gate_j and up_j in turn, and Y gets n / 2 values silu(gate_j) up_j a row: two lanes beside each other hold
// a pair's two products of four rows, and each finishes two of them.  (The 201 MB of 2048 x 24576 products were stored and read again by
// the next product's preparation; times at gemm_h6_swiglu's declaration.)
// (Four waves: two workgroups a compute unit.  Not told so, the compiler keeps the sums in accumulation registers and copies them out:
// 128 to 512 rows x 4096 to 14336 x 4096 to 12288 on this shape, Q4_K 0.96 to 1.00 of the time, MXFP4 0.98 to 1.04, on the picked one 0.96 to 1.01.)
template <class F, int NW, int NG, bool SWIGLU = false>
static __global__ __launch_bounds__(64 * NW, NW == 4 ? 2 : 1) void kq_gemm_h6(const uint8_t *__restrict__ W, size_t row_bytes,
                                                      const uint8_t *__restrict__ acts, float *__restrict__ Y, int m_rows, int n,
                                                      int nb, int groups, int tx, int ty, int nb_total, float *__restrict__ parts) {
    static_assert(NG <= NW && NG <= 8, "one group of 16 weight rows a wave unpacks, a byte each of a lane's eight exponents");
    constexpr int NT = 16 * NG, MT = 32 * NW, REC = h6_rec<F::MINS>();
    extern __shared__ __attribute__((aligned(16))) uint8_t h6_lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, g = lane >> 4;
    int bx, by;
    if (8 % ty == 0) {
        const int xcd = (int)blockIdx.x & 7, slot = (int)blockIdx.x >> 3;
        by = xcd % ty, bx = slot * (8 / ty) + xcd / ty;
    } else {
        by = (int)blockIdx.x / tx, bx = (int)blockIdx.x % tx;
    }
    if (bx >= tx || by >= ty) return;
    const int n0 = bx * NT, m0 = by * MT, b_first = (int)blockIdx.y * nb;
    if (blockIdx.y > 0) Y = parts + (size_t)(blockIdx.y - 1) * m_rows * n;  // k in parts: the first one's sums in place, splitk_add

    // everything is read behind an address that is the same in all lanes of a wave
    const int wv = __builtin_amdgcn_readfirstlane(wave), wu = min(wv, NG - 1);  // (waves past the last group unpack it too)
    auto record_of = [&](int mg) __attribute__((always_inline)) {
        return acts + ((size_t)min(m0 / 16 + 2 * wv + mg, groups - 1) * nb_total + b_first) * REC;
    };
    const H6Memory arec[2] = {H6Memory(record_of(0)), H6Memory(record_of(1))};
    const int first_row = min(n0 + 16 * wu, n - 1);
    const uint8_t *const wfirst = W + (size_t)first_row * row_bytes + (size_t)b_first * F::BLOCK;
    const H6Memory wsrc(wfirst);
    const uint32_t wlane = (uint32_t)min(r, n - 1 - first_row) * (uint32_t)row_bytes;
    uint8_t *const own = h6_lds + wu * H6_HALF, *const meta_lds = h6_lds + 2 * NG * H6_HALF;
    uint8_t *const exps = meta_lds + 2 * NG * H6_META + lane * 8;
    const uint32_t l16 = lane * 16;

    h6_h8 A[2][4];    // f16 operands of four steps, the fifth's in place of the first's
    h6_u6 L[2];       // the remainders of a half
    h6_b8 minA[2];
    h6_f4 sx[2];
    auto load_hi = [&](int mg, int b, int st) __attribute__((always_inline)) {
        A[mg][st & 3] = __builtin_bit_cast(h6_h8, arec[mg].load16(b * REC + st * 1024, l16));
    };
    auto load_lo = [&](int mg, int b, int h) __attribute__((always_inline)) {
        const uint32_t at = b * REC + H6_HI + h * H6_LO_HALF;
        const h6_u4 x = arec[mg].load16(at, l16);
        const h6_u2 y = arec[mg].load8(at + 1024, l16 >> 1);
        L[mg] = h6_u6{x[0], x[1], x[2], x[3], y[0], y[1]};
    };
    auto load_min = [&](int mg, int b) __attribute__((always_inline)) {
        minA[mg] = __builtin_bit_cast(h6_b8, arec[mg].load16(b * REC + H6_MIN, l16));
    };
    auto load_scale = [&](int mg, int b) __attribute__((always_inline)) {
        sx[mg] = __builtin_bit_cast(h6_f4, arec[mg].load16(b * REC + REC - 64, 16u * (uint32_t)g));
    };
    typename F::Raw raw;
    F::fetch_header(wsrc, 0, wlane, g, 0, raw);
    F::fetch(wsrc, 0, wlane, g, 0, raw);
#pragma unroll
    for (int mg = 0; mg < 2; mg++) {
#pragma unroll
        for (int st = 0; st < 4; st++) load_hi(mg, 0, st);
        load_lo(mg, 0, 0);
    }
    F::header(raw, g, r, 0, meta_lds + wu * H6_META, exps + wu);
    h6_each(std::make_integer_sequence<int, 16>{}, [&](auto uc) __attribute__((always_inline)) { F::template pair<decltype(uc)::value>(raw, g, lane, own); });
    F::codes(raw, lane, own);
    F::fetch(wsrc, 0, wlane, g, 1, raw);
    h6_f4 acc[2][NG], sb[2][NG];
    const h6_f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int mg = 0; mg < 2; mg++)
#pragma unroll
        for (int cg = 0; cg < NG; cg++) acc[mg][cg] = zero;
    __syncthreads();

    // The steps of a half: (group of weight rows, kind), kind 0..3: an f16 step of 32 k, 4: the half's remainders, 5: the
    // min term.  The second half takes its last three kinds group by group, so that the
    // groups' sums are complete one after the other and their scaling spreads among the matrix instructions that follow.
    struct Step {
        int cg, kind;
    };
    constexpr int LEAD = F::MINS ? 3 : 2;  // kinds in front of those three
    constexpr auto step_of = [](int h, int t) constexpr {
        if (h == 0) return Step{t % NG, t / NG};
        if (t < LEAD * NG) return Step{t % NG, LEAD == 2 ? t / NG : t < NG ? 5 : t / NG - 1};
        return Step{(t - LEAD * NG) / 3, 2 + (t - LEAD * NG) % 3};
    };
    constexpr int AHEAD = NG == 8 ? 2 : 4;  // operand reads; with eight groups the registers are just enough for two (no difference in time)
    for (int b = 0; b < nb; b++) {
        const int b1 = min(b + 1, nb - 1);
        const uint8_t *meta = meta_lds + (b & 1) * (NG * H6_META);
        h6_each(std::make_integer_sequence<int, 2>{}, [&](auto hc) __attribute__((always_inline)) {
            constexpr int h = decltype(hc)::value, STEPS = (h == 0 ? 5 : LEAD + 3) * NG;
            static_assert(STEPS >= 20, "a step for every pair of elements to be unpacked");
            const uint8_t *buf = h6_lds + h * (NG * H6_HALF);
            // the half that is unpacked meanwhile: the second of this super-block, then the first of the next
            uint8_t *const next = own + (h ^ 1) * (NG * H6_HALF);
            uint8_t *const next_meta = meta_lds + ((b + h) & 1) * (NG * H6_META) + wu * H6_META;
            const h6_u2 units = *(const h6_u2 *)(exps + h * H6_EXPS);
            const uint32_t src_next = (uint32_t)b1 * F::BLOCK;
            auto operand = [&](auto tc) __attribute__((always_inline)) {
                constexpr Step st = step_of(h, decltype(tc)::value);
                const uint8_t *tile = buf + st.cg * H6_HALF;
                if constexpr (st.kind == 5) return *(const h6_u4 *)(meta + st.cg * H6_META + (g >> 1) * 256 + r * 16);
                else return *(const h6_u4 *)(tile + (st.kind * 64 + lane) * 16);
            };
            auto operand_tail = [&](auto tc) __attribute__((always_inline)) {
                return *(const h6_u2 *)(buf + step_of(h, decltype(tc)::value).cg * H6_HALF + H6_T_LO + 1024 + lane * 8);
            };
            constexpr auto has_tail = [](Step st) constexpr { return F::LOW == 2 && st.kind == 4; };
            h6_u4 B[AHEAD];
            h6_u2 B2[AHEAD];
            h6_each(std::make_integer_sequence<int, AHEAD>{}, [&](auto tc) __attribute__((always_inline)) {
                B[decltype(tc)::value] = operand(tc);
                if constexpr (has_tail(step_of(h, decltype(tc)::value))) B2[decltype(tc)::value] = operand_tail(tc);
            });
            float d[2];
            auto finish = [&](int cg, int o) __attribute__((always_inline)) {  // one of the eight results a lane holds of group cg
                const int mg = o >> 2, i = o & 3;
                acc[mg][cg][i] = fmaf(d[cg & 1] * sx[mg][i], sb[mg][cg][i], acc[mg][cg][i]);
            };
            h6_each(std::make_integer_sequence<int, STEPS>{}, [&](auto tc) __attribute__((always_inline)) {
                constexpr int t = decltype(tc)::value;
                constexpr Step st = step_of(h, t);
                const h6_u4 w = B[t % AHEAD];
                const h6_u2 w2 = B2[t % AHEAD];
                if constexpr (t + AHEAD < STEPS) {
                    B[t % AHEAD] = operand(std::integral_constant<int, t + AHEAD>{});
                    if constexpr (has_tail(step_of(h, t + AHEAD))) B2[t % AHEAD] = operand_tail(std::integral_constant<int, t + AHEAD>{});
                }
                if constexpr (h == 1 && st.kind == 2) d[st.cg & 1] = *(const float *)(meta + st.cg * H6_META + 512 + 4 * r);
                // the next half's weights become operands among the matrix instructions; then the half after that is asked for
                if constexpr (t == 1) F::header(raw, g, r, h ^ 1, next_meta, exps + (h ^ 1) * H6_EXPS + wu);
                if constexpr (t >= 2 && t < 18) F::template pair<t - 2>(raw, g, lane, next);
                if constexpr (t == 18) F::codes(raw, lane, next);
                if constexpr (t == 19) F::fetch(wsrc, src_next, wlane, g, h, raw), F::fetch_header(wsrc, src_next, wlane, g, h, raw);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int mg = 0; mg < 2; mg++) {
                    if constexpr (st.kind == 5)
                        acc[mg][st.cg] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(minA[mg], __builtin_bit_cast(h6_b8, w), acc[mg][st.cg], 0, 0, 0);
                    else if constexpr (st.kind == 4) {
                        const h6_i8 low = F::LOW == 2 ? h6_operand6(h6_u6{w[0], w[1], w[2], w[3], w2[0], w2[1]})
                                                      : h6_i8{(int)w[0], (int)w[1], (int)w[2], (int)w[3], 0, 0, 0, 0};
                        sb[mg][st.cg] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(h6_operand6(L[mg]), low, sb[mg][st.cg], 2, F::LOW, 0, 0x7F7F7F7F,
                                                                                          st.cg & 3, (int)units[st.cg >> 2]);
                    }
                    else
                        sb[mg][st.cg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[mg][st.kind], __builtin_bit_cast(h6_h8, w),
                                                                               h == 0 && st.kind == 0 ? zero : sb[mg][st.cg], 0, 0, 0);
                }
                if constexpr (h == 1 && t >= LEAD * NG && st.cg > 0) {  // behind the matrix instructions of the group before
                    constexpr int o = 3 * (st.kind - 2);
                    finish(st.cg - 1, o), finish(st.cg - 1, o + 1);
                    if constexpr (o < 6) finish(st.cg - 1, o + 2);
                }
                if constexpr (st.cg == NG - 1) {  // this operand has done its work: a later one takes its place
#pragma unroll
                    for (int mg = 0; mg < 2; mg++) {
                        if constexpr (st.kind == 5) load_scale(mg, b);
                        else if constexpr (st.kind == 4) load_lo(mg, h == 0 ? b : b1, h ^ 1);
                        else load_hi(mg, h == 0 ? b : b1, 4 * (h ^ 1) + st.kind);
                        if constexpr (F::MINS && h == 0 && st.kind == 1) load_min(mg, b);
                        if constexpr (!F::MINS && h == 1 && st.kind == 0) load_scale(mg, b);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (h == 1) {
#pragma unroll
                for (int o = 0; o < 8; o++) finish(NG - 1, o);
            }
            __syncthreads();
        });
    }
    if constexpr (SWIGLU) {
        const bool odd = r & 1;
#pragma unroll
        for (int mg = 0; mg < 2; mg++)
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
                const int row = m0 + 16 * (2 * wave + mg) + 4 * g + i + (odd ? 1 : 0);
#pragma unroll
                for (int cg = 0; cg < NG; cg++) {
                    const float other = dpp_f<0xB1>(odd ? acc[mg][cg][i] : acc[mg][cg][i + 1]);  // quad_perm: of the lane beside this one
                    const float gate = odd ? other : acc[mg][cg][i], up = odd ? acc[mg][cg][i + 1] : other;
                    const int col = n0 + 16 * cg + r;
                    if (row < m_rows && col < n) Y[(size_t)row * (n / 2) + col / 2] = silu(gate) * up;
                }
            }
        return;
    }
#pragma unroll
    for (int mg = 0; mg < 2; mg++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int row = m0 + 16 * (2 * wave + mg) + 4 * g + i;
            if (row >= m_rows) continue;
#pragma unroll
            for (int cg = 0; cg < NG; cg++) {
                const int col = n0 + 16 * cg + r;
                if (col < n) Y[(size_t)row * n + col] = acc[mg][cg][i];
            }
        }
}

// Y[i] += P[0][i], then P[1][i], .. P[parts - 1][i], four elements a thread.
static __global__ __launch_bounds__(256) void splitk_add(const float *__restrict__ P, float *__restrict__ Y, size_t count, int parts) {
    const size_t i = 4 * ((size_t)blockIdx.x * 256 + threadIdx.x);
    if (i >= count) return;
    if ((count & 3) == 0) {
        float4 a = *(const float4 *)(Y + i);
        for (int p = 0; p < parts; p++) {
            const float4 b = *(const float4 *)(P + (size_t)p * count + i);
            a.x += b.x, a.y += b.y, a.z += b.z, a.w += b.w;
        }
        *(float4 *)(Y + i) = a;
    } else {
        for (size_t j = i; j < count && j < i + 4; j++) {
            float a = Y[j];
            for (int p = 0; p < parts; p++) a += P[(size_t)p * count + j];
            Y[j] = a;
        }
    }
}

}  // namespace jq

// f32 factors as two f16 numbers, hi = f16(x) and lo = f16(x - hi), behind a power of two that fits f16's range: what the
// kernels on split f16 operands share.
#pragma once
#include "kernels_graph.hpp"

namespace jq {

typedef _Float16 s16_h8 __attribute__((ext_vector_type(8)));
typedef _Float16 s16_h2 __attribute__((ext_vector_type(2)));
typedef float s16_f2 __attribute__((ext_vector_type(2)));
typedef float s16_f4 __attribute__((ext_vector_type(4)));
typedef float s16_f16 __attribute__((ext_vector_type(16)));

constexpr int S16_FRAG = 1024;  // bytes of a fragment: 64 lanes x 8 elements

typedef uint32_t s16_u4 __attribute__((ext_vector_type(4), aligned(4)));  // 16 bytes at any word

// Asynchronous global -> LDS copy of 16 bytes a lane, the wave's landing one behind the other at lds_base (wave-uniform); awaited
// by hand with s_waitcnt vmcnt.
__device__ __forceinline__ uint32_t s16_lds_offset(const void *p) {
    return (uint32_t)(uintptr_t)((__attribute__((address_space(3))) const void *)p);
}
__device__ __forceinline__ void s16_copy16(const void *gptr, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(gptr), "s"(__builtin_amdgcn_readfirstlane(lds_base)) : "memory");
}

__device__ __forceinline__ void s16_split(const float (&x)[8], s16_h8 &hi, s16_h8 &lo) {
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        const s16_h2 h = __builtin_convertvector(s16_f2{x[i], x[i + 1]}, s16_h2);
        const s16_h2 l = __builtin_convertvector(s16_f2{x[i] - (float)h[0], x[i + 1] - (float)h[1]}, s16_h2);
        hi[i] = h[0], hi[i + 1] = h[1], lo[i] = l[0], lo[i + 1] = l[1];
    }
}

// The exponent s that puts magnitudes up to `amax` (as float bits, sign cleared) at 2^13 .. 2^14, for every finite one of 2^-113 or more.
// Below, s stays at 126, from where a magnitude of 2^-126 is still 1; zero, infinite and NaN maxima take the nearest s.  2^s and 2^-s are
// normal numbers throughout (a product or quotient of two of them may over- or underflow).
__device__ __forceinline__ int s16_exponent(uint32_t amax_bits) {
    const int e = min(max((int)(amax_bits >> 23), 14), 254);
    return 13 - (e - 127);
}
__device__ __forceinline__ float s16_pow2(int s) { return __builtin_bit_cast(float, (uint32_t)(127 + s) << 23); }
__device__ __forceinline__ uint32_t s16_abs(float x) { return __builtin_bit_cast(uint32_t, x) & 0x7FFFFFFFu; }

// Zeros in place of infinities and NaNs; whether there were none.
template <int N>
__device__ __forceinline__ bool s16_make_finite(float (&x)[N]) {
    bool all = true;
#pragma unroll
    for (int i = 0; i < N; i++) {
        const bool is = s16_abs(x[i]) < 0x7F800000u;
        all &= is, x[i] = is ? x[i] : 0.0f;
    }
    return all;
}

// An address that is the same in all lanes, where the compiler does not see that.
__device__ __forceinline__ const uint8_t *s16_uniform(const uint8_t *p) {
    const uint64_t v = (uint64_t)p;
    return (const uint8_t *)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)v) |
                             (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32);
}

// Of pairs sorted into groups (offsets [groups + 1]), cut into tiles of `rows` pairs that never mix two groups: which group
// tile `mt` belongs to and its first pair there.  False past the last tile.  For whole waves; the results are uniform.
__device__ __forceinline__ bool s16_find_tile(const int *__restrict__ offsets, int groups, int rows, int mt, int &grp, int &at) {
    // lane l counts the tiles of a run of groups
    const int lane = threadIdx.x & 63, per = (groups + 63) / 64;
    int local = 0;
    for (int i = 0; i < per; i++) {
        const int e = lane * per + i;
        if (e < groups) local += (offsets[e + 1] - offsets[e] + rows - 1) / rows;
    }
    int incl = local;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int v = __shfl_up(incl, off, 64);
        if (lane >= off) incl += v;
    }
    if (mt >= __builtin_amdgcn_readlane(incl, 63)) return false;
    int found = -1, first = incl - local;
    if (mt >= first && mt < incl) {
        for (int i = 0; i < per; i++) {
            const int e = lane * per + i, t = e < groups ? (offsets[e + 1] - offsets[e] + rows - 1) / rows : 0;
            if (found < 0 && mt < first + t) found = e;
            else if (found < 0) first += t;
        }
    }
    const int owner = __builtin_ctzll(__ballot(found >= 0));
    grp = __builtin_amdgcn_readlane(found, owner);
    at = (mt - __builtin_amdgcn_readlane(first, owner)) * rows;
    return true;
}

}  // namespace jq

// Products of up to 16 activation rows with packed weights on the f16 matrix cores, without loss of precision: one launch, no
// scratch memory.
//
// Of a super-block of 256 elements a weight is d p, p of at most 13 bits behind one factor d, and an activation s (hi + lo): two f16
// numbers behind the power of two that takes the super-block's largest magnitude to 2^13 .. 2^14 (22 bits).  p is exact in one f16
// number (Q4_K: sc q; MXFP4) or in two, the second what rounding the first left (Q6_K: sc (q - 32); Q8_0: q d').  So a 16 x 16
// tile's sums over 32 elements are two v_mfma_f32_16x16x32_f16, or three (the remainders with each other are below 2^-22): exact
// products, f32 sums.  Up to eight rows need half of the instructions' 16 rows: there the others take the second numbers.
//
// Off 64 bits, relative 2-norm, rows of 2048 to 12288: 0.75e-7 to 0.9e-7 (MXFP4), 1.1e-7 to 1.3e-7 (the f32 row kernels 1.2e-7 to 2.6e-7, the
// int8 GEMM 2.7e-5, 3.7e-5 for Q8_0).
// Bound: the issue of vector instructions (a super-block of 16 weight rows takes 190 (Q4_K), 280 (Q6_K), 210 (Q8_0) or 90 (MXFP4),
// its activations 300 a workgroup) and, at the smallest sizes, one trip to memory.  us, 16 rows, before / now:
//   14336 x 4096   Q6_K 42 / 22     Q8_0 43 / 20     MXFP4 41 / 14
//   6000 x 5120    Q4_K 34 / 13     Q6_K 28 / 16     Q8_0 27 / 15
//   11008 x 3840   Q4_K 122 / 15    14336 x 11264   Q4_K 134 / 36   Q8_0 105 / 47   MXFP4 96 / 35
// A byte of weights is read once: 14336 x 4096 of MXFP4 with 8 rows, 12 us, is 2.7 TB/s, of Q8_0, 19 us, 3.3.
#pragma once
#include "split16_parts.hpp"

namespace jq {

// N words from any even address in LDS: whole words and a shift.
template <int N>
__device__ __forceinline__ void fr_words(const uint8_t *p, uint32_t (&out)[N]) {
    const uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint8_t *)p & 3u;
    const uint32_t *q = (const uint32_t *)(p - at);
    uint32_t x[N + 1];
#pragma unroll
    for (int i = 0; i <= N; i++) x[i] = q[i];
#pragma unroll
    for (int i = 0; i < N; i++) out[i] = __builtin_amdgcn_alignbyte(x[i + 1], x[i], at);
}

// Where a block of 32 has a scale of its own, those of a super-block may lie further apart than what normal f16 numbers hold exactly,
// 2^RANGE (of products with subnormal ones a matrix instruction keeps fewer bits: 1.4e-6 off at 2^36).  Then the super-block is
// multiplied once more for each such range that its scales span: of the blocks whose exponents e0 and e1 (-1: a block of zeros) lie under
// `below`, put(in0, in1, most) takes the ones within RANGE of the largest, and `below` moves under those.  True where some are left.
template <int RANGE, class F>
__device__ __forceinline__ bool fr_level(int e0, int e1, int &below, F put) {
    e0 = e0 < below ? e0 : -1, e1 = e1 < below ? e1 : -1;
    const int most = (int)max_xor32(max_xor16((float)max(e0, e1))), least = max(most - RANGE, 0);
    put(e0 >= least, e1 >= least, most);
    below = least;
    return (e0 >= 0 && e0 < least) || (e1 >= 0 && e1 < least);
}

// A format's side.  Lane (r = lane % 16, g = lane / 16) holds 64 elements of weight row r's super-block, eight for each of its eight
// k-steps.  QUAD(g, q): the first element of the q-th four that the lane reads of an activation row; AT(s, p): which of those 64 stands
// at position p of step s.
// Q4_K's mins, and what taking its codes about their middle leaves: w = d sc (q - 8) + (8 d sc - dmin m), the second factor one of a sub-block,
// in two f16 numbers h + l behind a power of two, against the activations' mean there in three.  (With the codes as they are the two
// sums cancel: 3.9e-7 off 64 bits instead of 1.6e-7.)
struct FrQ4K {  // sub-blocks 2 g (low nibbles) and 2 g + 1 (high) of 32 elements
    static constexpr int BLOCK = 144, ALIGN = 16, REAL = 9, PIECES = 9, PLANES = 1, CHAINS = 1;
    static constexpr bool MINS = true, LEVELS = false, UP = false;
    __device__ static int quad(int g, int q) { return 64 * g + 4 * q; }
    static constexpr int at(int s, int p) { return 8 * s + (p & 4) + ((p & 1) << 1 | (p >> 1 & 1)); }
    struct Raw {
        uint4 hdr, q[2];
        __device__ __forceinline__ void load(const uint8_t *b, int g) {
            hdr = *(const uint4 *)b;
            q[0] = *(const uint4 *)(b + 16 + 32 * g), q[1] = *(const uint4 *)(b + 32 + 32 * g);
        }
    };
    s16_h2 sc[2], off[2];
    s16_h8 mins;
    float d, dm;
    __device__ __forceinline__ bool begin(const Raw &r, int g, int &) {
        const uint32_t s4 = (g < 2 ? r.hdr.y & 0x3F3F3F3Fu : (r.hdr.w & 0x0F0F0F0Fu) | ((r.hdr.y >> 2) & 0x30303030u)) >> (16 * (g & 1));
        const uint32_t m4 = (g < 2 ? r.hdr.z & 0x3F3F3F3Fu : ((r.hdr.w >> 4) & 0x0F0F0F0Fu) | ((r.hdr.z >> 2) & 0x30303030u)) >> (16 * (g & 1));
        d = f16_bits(r.hdr.x);
        const float dmin = f16_bits(r.hdr.x >> 16);
        const uint32_t be = min(max(s16_abs(d), s16_abs(dmin)) >> 23, 254u);
        const float f = __builtin_bit_cast(float, (254u - be) << 23);
        float w[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const float s = (float)((s4 >> (8 * i)) & 0xFFu), m = (float)((m4 >> (8 * i)) & 0xFFu);
            const _Float16 h = (_Float16)(s * (i ? 64.0f : 1024.0f)), o = (_Float16)(s * -0x1p-11f);
            sc[i] = s16_h2{h, h}, off[i] = s16_h2{o, o};  // the operand is 2^-14 sc (q - 8)
            w[i] = fmaf(8.0f * d, s, -dmin * m) * f;
        }
        const s16_h2 h = __builtin_convertvector(s16_f2{w[0], w[1]}, s16_h2), l = __builtin_convertvector(s16_f2{w[0] - (float)h[0], w[1] - (float)h[1]}, s16_h2);
        mins = s16_h8{h[0], h[1], h[0], h[1], l[0], l[1], h[0], h[1]};
        dm = 32.0f * __builtin_bit_cast(float, be << 23), d *= 16384.0f;
        return false;
    }
    template <int S>
    __device__ __forceinline__ void step(const Raw &r, s16_h8 (&p)[1]) const {
        constexpr int nib = S >> 2;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint4 &q = r.q[(S & 3) >> 1];
            const uint32_t w = S & 1 ? (i ? q.w : q.z) : (i ? q.y : q.x);
            // a nibble as it stands is an f16 number below the normal ones, q 2^-24 or 2^-20
            const uint32_t mask = nib ? 0x00F000F0u : 0x000F000Fu;
            const s16_h2 e = __builtin_elementwise_fma(__builtin_bit_cast(s16_h2, w & mask), sc[nib], off[nib]);
            const s16_h2 o = __builtin_elementwise_fma(__builtin_bit_cast(s16_h2, (w >> 8) & mask), sc[nib], off[nib]);
            p[0][4 * i] = e[0], p[0][4 * i + 1] = e[1], p[0][4 * i + 2] = o[0], p[0][4 * i + 3] = o[1];
        }
    }
};

struct FrQ6K {  // w = d sc (q - 32), an int8 sc for 16 elements: element 128 (g / 2) + 16 (g % 2) + 32 t + i, t = s / 2
    static constexpr int BLOCK = 210, ALIGN = 2, REAL = 14, PIECES = 15, PLANES = 2, CHAINS = 1;
    static constexpr bool MINS = false, LEVELS = false, UP = false;
    __device__ static int quad(int g, int q) { return 128 * (g >> 1) + 16 * (g & 1) + 32 * (q >> 2) + 4 * (q & 3); }
    static constexpr int at(int s, int p) { return FrQ4K::at(s, p); }
    struct Raw {
        uint32_t a[4], b[4], h[4], s8[2], dd;
        __device__ __forceinline__ void load(const uint8_t *blk, int g) {
            const uint8_t *q = blk + 64 * (g >> 1) + 16 * (g & 1);
            fr_words(q, a), fr_words(q + 32, b);
            fr_words(blk + 128 + 32 * (g >> 1) + 16 * (g & 1), h);
            fr_words(blk + 192 + 8 * (g >> 1), s8);
            dd = *(const uint16_t *)(blk + 208);
        }
    };
    s16_h2 sc[4];
    float d;
    static constexpr float dm = 0.0f;
    __device__ __forceinline__ bool begin(const Raw &r, int g, int &) {
        const uint32_t by = 8 * (uint32_t)(g & 1);
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int v = (int8_t)(r.s8[t >> 1] >> (by + 16 * (t & 1)));
            const _Float16 f = (_Float16)(float)v;
            sc[t] = s16_h2{f, f};
        }
        d = f16_bits(r.dd);
        return false;
    }
    template <int S>
    __device__ __forceinline__ void step(const Raw &r, s16_h8 (&p)[2]) const {
        constexpr int t = S >> 1, shift = 4 * (t >> 1);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t w = (t & 1 ? r.b : r.a)[2 * (S & 1) + i], x = r.h[2 * (S & 1) + i];
#pragma unroll
            for (int odd = 0; odd < 2; odd++) {
                // 1024 + q: four bits of the nibble, two of the field t
                const uint32_t low = ((w >> (shift + 8 * odd)) & 0x000F000Fu) | 0x64006400u;
                constexpr int up = 4 - 2 * t;  // where the field goes
                const int by = 8 * odd - up;
                const uint32_t u = ((by >= 0 ? x >> by : x << -by) & 0x00300030u) | low;
                const s16_h2 v = __builtin_bit_cast(s16_h2, u) - (_Float16)1056.0f;
                const s16_h2 big = v * sc[t], rest = __builtin_elementwise_fma(v, sc[t], -big);
                p[0][4 * i + 2 * odd] = big[0], p[0][4 * i + 2 * odd + 1] = big[1];
                p[1][4 * i + 2 * odd] = rest[0], p[1][4 * i + 2 * odd + 1] = rest[1];
            }
        }
    }
};

struct FrQ8_0 {  // w = d q, an f16 d for 32 elements: blocks 2 g and 2 g + 1, 68 bytes.  d' = d 2^e, 2^7 <= the super-block's largest < 2^8
    static constexpr int BLOCK = 272, ALIGN = 16, REAL = 17, PIECES = 17, PLANES = 2;
    static constexpr int CHAINS = 2;  // of four matrix instructions each in few_rows, not one of eight: 1.28e-7 -> 1.10e-7, see fr_wave_sums
    static constexpr bool MINS = false, LEVELS = true, UP = false;
    __device__ static int quad(int g, int q) { return 64 * g + 4 * q; }
    static constexpr int at(int s, int p) { return FrQ4K::at(s, p); }
    struct Raw {
        s16_u4 w[4];
        uint32_t last;
        __device__ __forceinline__ void load(const uint8_t *b, int g) {
#pragma unroll
            for (int i = 0; i < 4; i++) w[i] = *(const s16_u4 *)(b + 68 * g + 16 * i);
            last = *(const uint32_t *)(b + 68 * g + 64);
        }
        __device__ __forceinline__ void load_far(const uint8_t *b, int g) { load(b, g); }  // from memory
        __device__ __forceinline__ uint32_t word(int i) const { return i == 16 ? last : w[i >> 2][i & 3]; }
    };
    s16_h2 sc[2];
    float d;
    static constexpr float dm = 0.0f;
    __device__ __forceinline__ bool begin(const Raw &r, int, int &below) {
        const float d0 = f16_bits(r.word(0)), d1 = f16_bits(r.word(8) >> 16);
        const int e0 = s16_abs(d0) ? (int)(s16_abs(d0) >> 23) : -1, e1 = s16_abs(d1) ? (int)(s16_abs(d1) >> 23) : -1;
        return fr_level<21>(e0, e1, below, [&](bool in0, bool in1, int most) __attribute__((always_inline)) {
            const int e = 134 - max(most, 100);  // (an f16 scale is 2^-24 or more)
            const float f = s16_pow2(e);
            const _Float16 h0 = (_Float16)(in0 ? d0 * f : 0.0f), h1 = (_Float16)(in1 ? d1 * f : 0.0f);
            sc[0] = s16_h2{h0, h0}, sc[1] = s16_h2{h1, h1};
            d = s16_pow2(-e);
        });
    }
    template <int S>
    __device__ __forceinline__ void step(const Raw &r, s16_h8 (&p)[2]) const {
        constexpr int b = S >> 2;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int at = 2 * (S & 3) + i;  // block 0's codes start at byte 2, block 1's at a word
            const uint32_t w = (b ? r.word(9 + at) : __builtin_amdgcn_alignbyte(r.word(at + 1), r.word(at), 2)) ^ 0x80808080u;
#pragma unroll
            for (int odd = 0; odd < 2; odd++) {
                const s16_h2 v = __builtin_bit_cast(s16_h2, __builtin_amdgcn_perm(0x64646464u, w, odd ? 0x04030401u : 0x04020400u)) - (_Float16)1152.0f;
                const s16_h2 big = v * sc[b], rest = __builtin_elementwise_fma(v, sc[b], -big);
                p[0][4 * i + 2 * odd] = big[0], p[0][4 * i + 2 * odd + 1] = big[1];
                p[1][4 * i + 2 * odd] = rest[0], p[1][4 * i + 2 * odd + 1] = rest[1];
            }
        }
    }
};

struct FrMXFP4 {  // w = 2^(e - 127) E2M1: blocks 2 g and 2 g + 1, 34 bytes; a byte holds elements j (low nibble) and j + 16 of its block
    static constexpr int BLOCK = 136, ALIGN = 8, REAL = 9, PIECES = 9, PLANES = 1, CHAINS = 1;
    static constexpr bool MINS = false, LEVELS = true, UP = true;
    __device__ static int quad(int g, int q) { return 64 * g + 4 * q; }
    static constexpr int at(int s, int p) { return 32 * (s >> 2) + 4 * (s & 3) + (p >> 1) + 16 * (p & 1); }
    struct Raw {
        uint32_t w[9];
        __device__ __forceinline__ void load(const uint8_t *b, int g) {  // 34 bytes: the ninth word's upper half is not used
            uint32_t first[8];
            fr_words(b + 34 * g, first);
#pragma unroll
            for (int i = 0; i < 8; i++) w[i] = first[i];
            w[8] = *(const uint16_t *)(b + 34 * g + 32);
        }
        __device__ __forceinline__ void load_far(const uint8_t *b, int g) {  // from memory
            const uint16_t *h = (const uint16_t *)(b + 34 * g);
#pragma unroll
            for (int i = 0; i < 8; i++) w[i] = h[2 * i] | (uint32_t)h[2 * i + 1] << 16;
            w[8] = h[16];
        }
        __device__ __forceinline__ uint32_t word(int i) const { return w[i]; }
    };
    float sc[2], d, up;  // (d at most 1, up at least 1: the products behind the activations' unit do not overflow before their sum does)
    static constexpr float dm = 0.0f;
    __device__ __forceinline__ bool begin(const Raw &r, int, int &below) {
        // the scales stand against the super-block's largest, which takes codes to 6 x 2^13; 0xFF: a block of zeros
        const int e0 = (int)(r.word(0) & 0xFFu), e1 = (int)((r.word(4) >> 8) & 0xFFu);
        return fr_level<26>(e0 == 0xFF ? -1 : e0, e1 == 0xFF ? -1 : e1, below, [&](bool in0, bool in1, int most) __attribute__((always_inline)) {
            sc[0] = in0 ? s16_pow2(e0 - most + 13) : 0.0f, sc[1] = in1 ? s16_pow2(e1 - most + 13) : 0.0f;
            d = ldexpf(1.0f, min(most - 140, 0)), up = ldexpf(1.0f, max(most - 140, 0));
        });
    }
    template <int S>
    __device__ __forceinline__ void step(const Raw &r, s16_h8 (&p)[1]) const {
        constexpr int b = S >> 2, first = 1 + 17 * b + 4 * (S & 3);
        const float f = sc[b];
        auto two = [&](auto jc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value;
            const s16_h2 v = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(r.word((first + j) >> 2), f, (first + j) & 3);
            p[0][2 * j] = v[0], p[0][2 * j + 1] = v[1];
        };
        two(std::integral_constant<int, 0>{}), two(std::integral_constant<int, 1>{});
        two(std::integral_constant<int, 2>{}), two(std::integral_constant<int, 3>{});
    }
};

constexpr int FR_ROW = 1040;  // bytes of an activation row's super-block in LDS: 16 rows read at one column meet all banks once
template <class F>
constexpr int few_rows_wave_lds(int tiles, int rows) { return rows * FR_ROW + 256 * tiles * F::PIECES; }
template <class F>
constexpr int few_rows_lds(int waves, int tiles, int rows) {
    const int stage = waves * few_rows_wave_lds<F>(tiles, rows), sums = waves * tiles * 1024;
    return stage > sums ? stage : sums;
}

// x f_hi as an f16 number, and what is left of x f beside it as another, one instruction a number.  The instructions write half a register; the
// hardware wants another one between such a write and the next use of the register, which the order here and the s_nop see to.
__device__ __forceinline__ void fr_split(const float (&x)[8], float f_hi, float f, s16_h8 &hi, s16_h8 &lo) {
    uint32_t h[4], l[4];
    asm("v_fma_mixlo_f16 %0, %8, %16, 0\n\tv_fma_mixlo_f16 %1, %10, %16, 0\n\tv_fma_mixlo_f16 %2, %12, %16, 0\n\tv_fma_mixlo_f16 %3, %14, %16, 0\n\t"
        "v_fma_mixhi_f16 %0, %9, %16, 0\n\tv_fma_mixhi_f16 %1, %11, %16, 0\n\tv_fma_mixhi_f16 %2, %13, %16, 0\n\tv_fma_mixhi_f16 %3, %15, %16, 0\n\t"
        "v_fma_mixlo_f16 %4, %8, %17, -%0 op_sel_hi:[0,0,1]\n\tv_fma_mixlo_f16 %5, %10, %17, -%1 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %6, %12, %17, -%2 op_sel_hi:[0,0,1]\n\tv_fma_mixlo_f16 %7, %14, %17, -%3 op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %4, %9, %17, -%0 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\tv_fma_mixhi_f16 %5, %11, %17, -%1 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %6, %13, %17, -%2 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\tv_fma_mixhi_f16 %7, %15, %17, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "s_nop 1"
        : "=&v"(h[0]), "=&v"(h[1]), "=&v"(h[2]), "=&v"(h[3]), "=&v"(l[0]), "=&v"(l[1]), "=&v"(l[2]), "=&v"(l[3])
        : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(x[4]), "v"(x[5]), "v"(x[6]), "v"(x[7]), "v"(f_hi), "v"(f));
    hi = __builtin_bit_cast(s16_h8, uint4{h[0], h[1], h[2], h[3]}), lo = __builtin_bit_cast(s16_h8, uint4{l[0], l[1], l[2], l[3]});
}

template <int N>
__device__ __forceinline__ void fr_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

extern __shared__ __attribute__((aligned(16))) uint8_t fr_lds[];

// The i-th of the `stride` sums that each wave of a workgroup left in LDS, of up to eight waves, in pairs: three roundings of a sum's size, not
// fifteen (Q8_0, five rows of 2048: 1.40e-7 -> 1.28e-7 off 64 bits; the f32 row kernel 1.22e-7).
__device__ __forceinline__ s16_f4 fr_wave_sums(int i, int stride, int waves) {
    const s16_f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    s16_f4 s[8];
#pragma unroll
    for (int w = 0; w < 8; w++) {
        const s16_f4 v = *(const s16_f4 *)(fr_lds + (min(w, waves - 1) * stride + i) * 16);
        s[w] = w < waves ? v : zero;
    }
    return ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
}

// A workgroup takes 16 NT weight rows; its waves take the super-blocks of a row in turn, each for itself, and add up
// at the end in pairs.  A wave brings its super-block of the activation rows (ROWS of them, the last one again past the m-th)
// and of its tiles of 16 weight rows to LDS by asynchronous loads of contiguous pieces: a lane that reads its own share of a row from memory
// looks up a cache line of its own at every load, two clocks a lane.  A place in LDS is free once its words are in registers, and
// what the next super-block puts there is asked for at once, so up to a whole super-block of all tiles travels while one is multiplied.
// Pieces are whole aligned 16 bytes: of a block that starts between them, all that hold a byte of it.
template <class F, int NT, int ROWS>
static __global__ __launch_bounds__(512, 2) void few_rows(const uint8_t *__restrict__ W, uint32_t row_bytes, const float *__restrict__ X,
                                                          float *__restrict__ Y, int m, int n, int nb) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
    const int waves = blockDim.x >> 6, n0 = blockIdx.x * 16 * NT, k = 256 * nb;
    constexpr bool EVEN = F::ALIGN == 16;  // blocks start at pieces
    constexpr int TILE = 256 * F::PIECES, COPIES = (F::PIECES + 3) / 4;
    const uint8_t *const first = W + (size_t)n0 * row_bytes;
    const uint32_t mis = EVEN ? 0u : (uint32_t)(uintptr_t)first & 15u;
    const uint8_t *const base = s16_uniform(first - mis);
    uint32_t at[NT][COPIES];  // row's offset, piece: of copy 64 j + lane
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int j = 0; j < COPIES; j++) {
            const int id = min(64 * j + lane, 16 * F::PIECES - 1), row = 16 * t + id / F::PIECES, piece = min(id % F::PIECES, F::REAL - 1);
            const uint32_t off = (uint32_t)min(row, n - 1 - n0) * row_bytes;
            at[t][j] = EVEN ? off + 16u * piece : (off + mis) << 4 | (uint32_t)piece;
        }
    uint8_t *const own = fr_lds + wave * few_rows_wave_lds<F>(NT, ROWS);
    const uint32_t own_at = s16_lds_offset(own), own_w = own_at + ROWS * FR_ROW;
    const float *const mine = (const float *)(own + (r & (ROWS - 1)) * FR_ROW);
    // up to eight rows: both planes in one operand, rows 0 .. 7 of the matrix instruction the first numbers, 8 .. 15 the second
    constexpr bool BOTH = ROWS <= 8;
    const uint8_t *const my_w = own + ROWS * FR_ROW + 16 * F::PIECES * r;
    auto fetch_w = [&](int sb, int t) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < COPIES; j++) {
            const uint32_t dst = __builtin_amdgcn_readfirstlane(own_w + t * TILE + 1024 * j), shift = (uint32_t)sb * F::BLOCK;
            const uint32_t off = EVEN ? at[t][j] + shift : (((at[t][j] >> 4) + shift) & ~15u) + ((at[t][j] & 15u) << 4);
            if (F::PIECES % 4 == 0 || j + 1 < COPIES || lane < 16 * (F::PIECES % 4))
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(dst) : "memory");
        }
    };
    auto fetch_x = [&](int sb) __attribute__((always_inline)) {
        const uint8_t *x = s16_uniform((const uint8_t *)(X + 256 * (size_t)sb));
#pragma unroll
        for (int i = 0; i < ROWS; i++) {
            const uint32_t dst = __builtin_amdgcn_readfirstlane(own_at + i * FR_ROW);
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(16 * lane), "s"(x + (size_t)min(i, m - 1) * k * 4), "s"(dst) : "memory");
        }
    };
    const s16_f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    s16_f4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) acc[t] = zero;
    if (wave < nb) {
        fetch_x(wave);
#pragma unroll
        for (int t = 0; t < NT; t++) fetch_w(wave, t);
    }
    for (int sb = wave; sb < nb; sb += waves) {
        const bool more = sb + waves < nb;
        typename F::Raw raw;
        auto read = [&](int t) __attribute__((always_inline)) {
            uint32_t skip = 0;
            if constexpr (!EVEN) skip = (mis + (uint32_t)min(16 * t + r, n - 1 - n0) * row_bytes + (uint32_t)sb * F::BLOCK) & 15u;
            raw.load(my_w + t * TILE + skip, g);
        };
        fr_wait<(NT - 1) * COPIES>();
        float x[64];
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const float4 v = *(const float4 *)(mine + F::quad(g, q));
            x[4 * q] = v.x, x[4 * q + 1] = v.y, x[4 * q + 2] = v.z, x[4 * q + 3] = v.w;
        }
        read(0);
        float amax = 0.0f;  // (a NaN is passed over here and stays one below)
#pragma unroll
        for (int i = 0; i < 64; i += 2) asm volatile("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(amax) : "v"(x[i]), "v"(x[i + 1]));
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (more) fetch_x(sb + waves), fetch_w(sb + waves, 0);
        amax = max_xor32(max_xor16(amax));
        const bool finite = amax < INFINITY;
        const int e = s16_exponent(__builtin_bit_cast(uint32_t, amax));
        const float f = finite ? s16_pow2(e) : 0.0f, unit = finite ? s16_pow2(-e) : __builtin_nanf("");
        s16_h8 hi[8], lo[BOTH ? 1 : 8], xs;
        const float f_first = BOTH && r < 8 ? 0.0f : f;  // (the first numbers are what nothing, taken away, leaves)
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const float v[8] = {x[F::at(s, 0)], x[F::at(s, 1)], x[F::at(s, 2)], x[F::at(s, 3)], x[F::at(s, 4)], x[F::at(s, 5)], x[F::at(s, 6)], x[F::at(s, 7)]};
            s16_h8 h, l;
            fr_split(v, f_first, f, h, l);
            if constexpr (BOTH) hi[s] = l;
            else hi[s] = h, lo[s] = l;
        }
        if constexpr (F::MINS) {  // means of the lane's two sub-blocks
            float sum[2] = {0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < 64; i++) sum[i >> 5] = fmaf(x[i], f, sum[i >> 5]);  // (32 of them as they are may exceed f32)
            const s16_f2 v = {sum[0] * 0.03125f, sum[1] * 0.03125f};
            const s16_h2 h = __builtin_convertvector(v, s16_h2);
            const s16_f2 left = {v[0] - (float)h[0], v[1] - (float)h[1]};
            const s16_h2 l = __builtin_convertvector(left, s16_h2);
            const s16_h2 j = __builtin_convertvector(s16_f2{left[0] - (float)l[0], left[1] - (float)l[1]}, s16_h2);
            const _Float16 z = (_Float16)0.0f;
            if constexpr (BOTH) xs = r < 8 ? s16_h8{h[0], h[1], z, z, h[0], h[1], z, z} : s16_h8{l[0], l[1], j[0], j[1], z, z, z, z};
            else xs = s16_h8{h[0], h[1], l[0], l[1], h[0], h[1], j[0], j[1]};
        }
        __builtin_amdgcn_sched_barrier(0);
        s16_f4 sx;
#pragma unroll
        for (int i = 0; i < 4; i++) sx[i] = __shfl(unit, (BOTH ? 4 * (g & 1) : 4 * g) + i, 64);
#pragma unroll
        for (int t = 0; t < NT; t++) {
            if (t > 0) {
                if (more) fr_wait<(NT - 1) * COPIES + ROWS>();
                else if (t == 1) fr_wait<(NT > 1 ? NT - 2 : 0) * COPIES>();
                else if (t == 2) fr_wait<(NT > 2 ? NT - 3 : 0) * COPIES>();
                else fr_wait<0>();
                read(t);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                if (more) fetch_w(sb + waves, t);
            }
            __builtin_amdgcn_sched_barrier(0);
            F w;
            int below = 256;
            for (bool left = true; left;) {
                left = F::LEVELS ? __any(w.begin(raw, g, below)) : w.begin(raw, g, below);
                s16_f4 big[2] = {zero, zero}, low = zero;
                auto step = [&](auto sc) __attribute__((always_inline)) {
                    constexpr int S = decltype(sc)::value;
                    s16_h8 p[F::PLANES];
                    w.template step<S>(raw, p);
                    constexpr int c = F::CHAINS == 2 ? S & 1 : 0;
                    big[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[S], p[0], big[c], 0, 0, 0);
                    if constexpr (!BOTH) low = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[S], p[0], low, 0, 0, 0);
                    if constexpr (F::PLANES == 2) low = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[S], p[1], low, 0, 0, 0);
                };
                step(std::integral_constant<int, 0>{}), step(std::integral_constant<int, 1>{}), step(std::integral_constant<int, 2>{});
                step(std::integral_constant<int, 3>{}), step(std::integral_constant<int, 4>{}), step(std::integral_constant<int, 5>{});
                step(std::integral_constant<int, 6>{}), step(std::integral_constant<int, 7>{});
                s16_f4 i2 = zero;
                if constexpr (F::MINS) i2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(xs, w.mins, zero, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float sum = w.d * ((F::CHAINS == 2 ? big[0][i] + big[1][i] : big[0][i]) + low[i]);
                    if constexpr (F::UP) acc[t][i] = fmaf(sx[i] * sum, w.up, acc[t][i]);
                    else acc[t][i] = fmaf(sx[i], F::MINS ? fmaf(w.dm, i2[i], sum) : sum, acc[t][i]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; t++) *(s16_f4 *)(fr_lds + ((wave * NT + t) * 64 + lane) * 16) = acc[t];
    __syncthreads();
    for (int i = tid; i < NT * 64; i += 64 * waves) {
        if (BOTH && (i & 32)) continue;  // (the second planes' sums, added below)
        const s16_f4 v = fr_wave_sums(i, NT * 64, waves) + (BOTH ? fr_wave_sums(i + 32, NT * 64, waves) : zero);
        const int col = n0 + 16 * (i >> 6) + (i & 15), row = 4 * ((i >> 4) & 3);
        if (col < n) {
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (row + j < m) Y[(size_t)(row + j) * n + col] = v[j];
        }
    }
}

// ---- more than 16 rows -------------------------------------------------------------------------------------------------------

// Prepared activations, for every 16 rows and super-block: 8 k-steps of two fragments (first numbers, second numbers), the operand
// of the mins, the 16 rows' units.
constexpr int FR_MIN = 16 * S16_FRAG, FR_UNIT = FR_MIN + S16_FRAG, FR_REC = FR_UNIT + 64;

// A lane's 64 elements of a row -> its share of the fragments, and the row's unit.
template <class F>
__device__ __forceinline__ void fr_operands(const float (&x)[64], s16_h8 (&hi)[8], s16_h8 (&lo)[8], s16_h8 &xs, float &unit) {
    float amax = 0.0f;  // (a NaN is passed over here and stays one below)
#pragma unroll
    for (int i = 0; i < 64; i += 2) asm volatile("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(amax) : "v"(x[i]), "v"(x[i + 1]));
    amax = max_xor32(max_xor16(amax));
    const bool finite = amax < INFINITY;
    const int e = s16_exponent(__builtin_bit_cast(uint32_t, amax));
    const float f = finite ? s16_pow2(e) : 0.0f;
    unit = finite ? s16_pow2(-e) : __builtin_nanf("");
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const float v[8] = {x[F::at(s, 0)], x[F::at(s, 1)], x[F::at(s, 2)], x[F::at(s, 3)], x[F::at(s, 4)], x[F::at(s, 5)], x[F::at(s, 6)], x[F::at(s, 7)]};
        fr_split(v, f, f, hi[s], lo[s]);
    }
    if constexpr (F::MINS) {
        float sum[2] = {0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 64; i++) sum[i >> 5] = fmaf(x[i], f, sum[i >> 5]);  // (32 of them as they are may exceed f32)
        const s16_f2 v = {sum[0] * 0.03125f, sum[1] * 0.03125f};
        const s16_h2 h = __builtin_convertvector(v, s16_h2);
        const s16_f2 left = {v[0] - (float)h[0], v[1] - (float)h[1]};
        const s16_h2 l = __builtin_convertvector(left, s16_h2);
        const s16_h2 j = __builtin_convertvector(s16_f2{left[0] - (float)l[0], left[1] - (float)l[1]}, s16_h2);
        xs = s16_h8{h[0], h[1], l[0], l[1], h[0], h[1], j[0], j[1]};
    }
}

// grid (super-blocks, groups of 16 rows), a wave each
template <class F>
static __global__ __launch_bounds__(64) void few_rows_prep(const float *__restrict__ X, int m, int nb, uint8_t *__restrict__ out) {
    const int lane = threadIdx.x, r = lane & 15, g = lane >> 4, row = 16 * (int)blockIdx.y + r;
    uint8_t *rec = out + ((size_t)blockIdx.y * nb + blockIdx.x) * FR_REC;
    const float *src = X + (size_t)min(row, m - 1) * nb * 256 + 256 * blockIdx.x;
    float x[64], unit;
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const float4 v = *(const float4 *)(src + F::quad(g, q));
        x[4 * q] = v.x, x[4 * q + 1] = v.y, x[4 * q + 2] = v.z, x[4 * q + 3] = v.w;
    }
    s16_h8 hi[8], lo[8], xs;
    fr_operands<F>(x, hi, lo, xs, unit);
#pragma unroll
    for (int s = 0; s < 8; s++) {
        *(s16_h8 *)(rec + (2 * s * 64 + lane) * 16) = hi[s];
        *(s16_h8 *)(rec + ((2 * s + 1) * 64 + lane) * 16) = lo[s];
    }
    if constexpr (F::MINS) *(s16_h8 *)(rec + FR_MIN + 16 * lane) = xs;
    if (g == 0) *(float *)(rec + FR_UNIT + 4 * r) = unit;
}

template <class F>
constexpr int few_rows_many_lds(int waves, int nt, int mt) {
    const int stage = waves * 256 * nt * F::PIECES, sums = waves * nt * mt * 1024;
    return stage > sums ? stage : sums;
}

// few_rows for 16 MT activation rows a workgroup.  Bound: the prepared activations on their way from the second level cache, some 35 bytes a
// clock and compute unit (32 rows x 12288 x 4096: 25 us, of them 19 for the 1.5 MB that each compute unit reads), with more tiles a
// workgroup the issue of instructions.  32 rows x 14336 x 4096: Q4_K 27 -> 19 us, Q6_K 43 -> 26, MXFP4 42 -> 17.
// The activations' operands come prepared, straight into registers, AHEAD k-steps before they are multiplied; the weights of NT tiles as
// in few_rows.  Workgroups 8 apart (one XCD) hold the row blocks of one column block.
template <class F, int NT, int MT, int AHEAD>
static __global__ __launch_bounds__(512, 2) void few_rows_many(const uint8_t *__restrict__ W, uint32_t row_bytes, const uint8_t *__restrict__ acts,
                                                               float *__restrict__ Y, int m, int n, int nb, int groups, int blocks) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
    const int waves = blockDim.x >> 6, id = blockIdx.x, n0 = (id / 8 / blocks * 8 + id % 8) * 16 * NT, g0 = id / 8 % blocks * MT;
    if (n0 >= n) return;
    constexpr bool EVEN = F::ALIGN == 16;
    constexpr int TILE = 256 * F::PIECES, COPIES = (F::PIECES + 3) / 4;
    const uint8_t *const first = W + (size_t)n0 * row_bytes;
    const uint32_t mis = EVEN ? 0u : (uint32_t)(uintptr_t)first & 15u;
    const uint8_t *const base = s16_uniform(first - mis);
    uint32_t at[NT][COPIES];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int j = 0; j < COPIES; j++) {
            const int piece_id = min(64 * j + lane, 16 * F::PIECES - 1), row = 16 * t + piece_id / F::PIECES, piece = min(piece_id % F::PIECES, F::REAL - 1);
            const uint32_t off = (uint32_t)min(row, n - 1 - n0) * row_bytes;
            at[t][j] = EVEN ? off + 16u * piece : (off + mis) << 4 | (uint32_t)piece;
        }
    uint8_t *const own = fr_lds + wave * NT * TILE;
    const uint32_t own_at = s16_lds_offset(own);
    const uint8_t *const my_w = own + 16 * F::PIECES * r;
    auto fetch_w = [&](int sb) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int j = 0; j < COPIES; j++) {
                const uint32_t dst = __builtin_amdgcn_readfirstlane(own_at + t * TILE + 1024 * j), shift = (uint32_t)sb * F::BLOCK;
                const uint32_t off = EVEN ? at[t][j] + shift : (((at[t][j] >> 4) + shift) & ~15u) + ((at[t][j] & 15u) << 4);
                if (F::PIECES % 4 == 0 || j + 1 < COPIES || lane < 16 * (F::PIECES % 4))
                    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(dst) : "memory");
            }
    };
    uint32_t rec[MT];  // the groups' records; past the last group: the last one again, not stored
#pragma unroll
    for (int j = 0; j < MT; j++) rec[j] = (uint32_t)(min(g0 + j, groups - 1) - g0) * (uint32_t)nb * FR_REC;
    const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc((void *)s16_uniform(acts + (size_t)g0 * nb * FR_REC), 0, 0xFFFFFFFFu, 0x00027000);
    const int l16 = 16 * lane;
    s16_h8 A[AHEAD][MT][2];
    auto load = [&](int sb, int s) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < MT; j++)
#pragma unroll
            for (int p = 0; p < 2; p++)
                A[s % AHEAD][j][p] = __builtin_bit_cast(s16_h8, __builtin_amdgcn_raw_buffer_load_b128(src, l16, (int)(rec[j] + (uint32_t)sb * FR_REC + (2 * s + p) * S16_FRAG), 0));
    };
    const s16_f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    s16_f4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int j = 0; j < MT; j++) acc[t][j] = zero;
    if (wave < nb) {
        fetch_w(wave);
#pragma unroll
        for (int s = 0; s < AHEAD; s++) load(wave, s);
    }
    for (int sb = wave; sb < nb; sb += waves) {
        const int next = sb + waves < nb ? sb + waves : sb;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        typename F::Raw raw[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            uint32_t skip = 0;
            if constexpr (!EVEN) skip = (mis + (uint32_t)min(16 * t + r, n - 1 - n0) * row_bytes + (uint32_t)sb * F::BLOCK) & 15u;
            raw[t].load(my_w + t * TILE + skip, g);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (next != sb) fetch_w(next);
        __builtin_amdgcn_sched_barrier(0);
        F w[NT];
        bool left = false;  // blocks behind scales too far below the others', multiplied further down
#pragma unroll
        for (int t = 0; t < NT; t++) {
            int below = 256;
            left |= w[t].begin(raw[t], g, below);
        }
        constexpr bool APART = NT * MT <= 4;  // the products with the remainders in sums of their own, where registers are left
        s16_f4 sums[NT][MT], low[APART ? NT : 1][APART ? MT : 1];
        s16_h8 xs[MT];
        s16_f4 unit[MT];
        auto step = [&](auto sc) __attribute__((always_inline)) {
            constexpr int S = decltype(sc)::value;
            s16_h8 a[MT][2];
#pragma unroll
            for (int j = 0; j < MT; j++) a[j][0] = A[S % AHEAD][j][0], a[j][1] = A[S % AHEAD][j][1];
#pragma unroll
            for (int t = 0; t < NT; t++) {
                s16_h8 p[F::PLANES];
                w[t].template step<S>(raw[t], p);
#pragma unroll
                for (int j = 0; j < MT; j++) sums[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j][0], p[0], S == 0 ? zero : sums[t][j], 0, 0, 0);
#pragma unroll
                for (int j = 0; j < MT; j++) {
                    s16_f4 &to = APART ? low[APART ? t : 0][APART ? j : 0] : sums[t][j];
                    to = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j][1], p[0], APART && S == 0 ? zero : to, 0, 0, 0);
                }
                if constexpr (F::PLANES == 2) {
#pragma unroll
                    for (int j = 0; j < MT; j++) {
                        s16_f4 &to = APART ? low[APART ? t : 0][APART ? j : 0] : sums[t][j];
                        to = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j][0], p[1], to, 0, 0, 0);
                    }
                }
            }
            if constexpr (S + AHEAD < 8) load(sb, S + AHEAD);
            else load(next, S + AHEAD - 8);
            if constexpr (S == 7 - AHEAD) {
#pragma unroll
                for (int j = 0; j < MT; j++) {
                    const int at_sb = (int)(rec[j] + (uint32_t)sb * FR_REC);
                    if constexpr (F::MINS) xs[j] = __builtin_bit_cast(s16_h8, __builtin_amdgcn_raw_buffer_load_b128(src, l16, at_sb + FR_MIN, 0));
                    unit[j] = __builtin_bit_cast(s16_f4, __builtin_amdgcn_raw_buffer_load_b128(src, 16 * g, at_sb + FR_UNIT, 0));
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        step(std::integral_constant<int, 0>{}), step(std::integral_constant<int, 1>{}), step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{}), step(std::integral_constant<int, 4>{}), step(std::integral_constant<int, 5>{});
        step(std::integral_constant<int, 6>{}), step(std::integral_constant<int, 7>{});
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int j = 0; j < MT; j++) {
                s16_f4 i2 = zero;
                if constexpr (APART) sums[t][j] += low[t][j];
                if constexpr (F::MINS) i2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(xs[j], w[t].mins, zero, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float sum = w[t].d * sums[t][j][i];
                    if constexpr (F::UP) acc[t][j][i] = fmaf(unit[j][i] * sum, w[t].up, acc[t][j][i]);
                    else acc[t][j][i] = fmaf(unit[j][i], F::MINS ? fmaf(w[t].dm, i2[i], sum) : sum, acc[t][j][i]);
                }
            }
        if constexpr (F::LEVELS) {
            if (__any(left)) {  // everything read again, so that nothing is kept for it
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    typename F::Raw far;
                    far.load_far(first + (size_t)min(16 * t + r, n - 1 - n0) * row_bytes + (size_t)sb * F::BLOCK, g);
                    F v;
                    int below = 256;
                    bool more = __any(v.begin(far, g, below));  // (the turn above)
                    while (more) {
                        more = __any(v.begin(far, g, below));
                        s16_f4 again[MT];
                        auto turn = [&](auto sc) __attribute__((always_inline)) {
                            constexpr int S = decltype(sc)::value;
                            s16_h8 p[F::PLANES];
                            v.template step<S>(far, p);
#pragma unroll
                            for (int j = 0; j < MT; j++) {
                                const int at_step = (int)(rec[j] + (uint32_t)sb * FR_REC + 2 * S * S16_FRAG);
                                const s16_h8 hi = __builtin_bit_cast(s16_h8, __builtin_amdgcn_raw_buffer_load_b128(src, l16, at_step, 0));
                                const s16_h8 lo = __builtin_bit_cast(s16_h8, __builtin_amdgcn_raw_buffer_load_b128(src, l16, at_step + S16_FRAG, 0));
                                again[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, p[0], S == 0 ? zero : again[j], 0, 0, 0);
                                again[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo, p[0], again[j], 0, 0, 0);
                                if constexpr (F::PLANES == 2) again[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, p[1], again[j], 0, 0, 0);
                            }
                            __builtin_amdgcn_sched_barrier(0);
                        };
                        turn(std::integral_constant<int, 0>{}), turn(std::integral_constant<int, 1>{}), turn(std::integral_constant<int, 2>{});
                        turn(std::integral_constant<int, 3>{}), turn(std::integral_constant<int, 4>{}), turn(std::integral_constant<int, 5>{});
                        turn(std::integral_constant<int, 6>{}), turn(std::integral_constant<int, 7>{});
#pragma unroll
                        for (int j = 0; j < MT; j++)
#pragma unroll
                            for (int i = 0; i < 4; i++) {
                                if constexpr (F::UP) acc[t][j][i] = fmaf(unit[j][i] * (v.d * again[j][i]), v.up, acc[t][j][i]);
                                else acc[t][j][i] = fmaf(unit[j][i], v.d * again[j][i], acc[t][j][i]);
                            }
                    }
                }
#pragma unroll
                for (int s = 0; s < AHEAD; s++) load(next, s);
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int j = 0; j < MT; j++) *(s16_f4 *)(fr_lds + ((wave * NT * MT + t * MT + j) * 64 + lane) * 16) = acc[t][j];
    __syncthreads();
    for (int i = tid; i < NT * MT * 64; i += 64 * waves) {
        const s16_f4 v = fr_wave_sums(i, NT * MT * 64, waves);
        const int t = (i >> 6) / MT, j = (i >> 6) % MT, col = n0 + 16 * t + (i & 15), row = 16 * (g0 + j) + 4 * ((i >> 4) & 3);
        if (col < n) {
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (row + q < m) Y[(size_t)(row + q) * n + col] = v[q];
        }
    }
}

}  // namespace jq

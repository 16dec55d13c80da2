// Grouped products of Q4_K experts with some tens of rows each, on the f16 matrix cores without loss of precision.
//
// A Q4_K weight is d p - dmin m with p = sc q an integer of at most 945: exact in f16.  An activation, scaled by a power of two
// that puts its super-block's largest magnitude at 2^13 .. 2^14, is the sum of two f16 numbers hi + lo (22 bits).  So per
// super-block and output
//     I1 = sum p (hi + lo)     two v_mfma_f32_16x16x32_f16 a sub-block, products exact, f32 sums
//     I2 = sum_j m_j XS_j      one more a super-block (XS_j: the sub-block's sum / 32, again hi + lo; the mins exact)
//     y += s (d I1 - 32 dmin I2)
// The packed nibbles become the second operand in registers: (w & 0xF) | 0x6400 is 1024 + q as f16, one
// v_pk_fma_f16 with sc and -1024 sc makes two products (the high nibbles: 0x5400, 64 + q): 1.1 vector instructions a
// weight, and the unpacking of 64 rows serves every activation row of the tile.  (The int8 GEMM's two byte
// planes of the same product cost four instructions a weight and pass through LDS, and its sums seven an output.)
//
// Element order.  Lane (n = lane % 16, g = lane / 16) holds weight row n and, of half a super-block (four sub-blocks, 64
// bytes), bytes 16 g .. + 15: sub-blocks 2 (g / 2) and 2 (g / 2) + 1, elements 16 (g % 2) .. + 15 of each.  They make four
// k-steps t = 2 (low / high nibble) + (first / second 8 bytes), in the order 0 2 1 3 4 6 5 7 of a step's eight.  The activation
// planes are stored in that order, [row][super-block][half][t][plane][g] of 16 bytes, so a fragment is 16 rows' runs of
// 64 bytes, gathered through the pair list by asynchronous loads into LDS.
#pragma once
#include "split16_parts.hpp"

namespace jq {

constexpr int MS16_PLANES = 1024, MS16_XS = 32;  // bytes a row and super-block: hi and lo of 256 elements; of 8 sums
constexpr int MS16_RG = 3;                        // row groups of 16 a tile holds at most
constexpr int MS16_ROWS = 16 * MS16_RG;
constexpr int MS16_SLOTS = 2304;                  // a tile's packed bytes in LDS: headers, first half, second half of a super-block
constexpr int MS16_BUF = MS16_RG * 4 * S16_FRAG;  // a quarter's activation planes
constexpr int MS16_ACTS = 3 * MS16_BUF + MS16_RG * 512;  // three quarters, and a super-block's sums
constexpr int MS16_MAX_NB = 32;                   // super-blocks of a row (the scales of a tile wait in LDS)
// weight rows of a workgroup whose waves take WT tiles of 16 each (DUAL: half of them gate rows, half up rows)
constexpr int moe_split16_cols(int WT) { return 64 * WT; }

struct MoeSplit16Acts {
    uint8_t *planes, *xs;
    float *s;
};

// grid (rows, ceil(nb / 4)), four waves, a wave one (row, super-block).  Row r is X[sel ? sel[r] : r].  A super-block that
// holds an inf or a NaN gets the scale NaN (and the row's result is NaN).
static __global__ __launch_bounds__(256) void moe_split16_prep(const float *__restrict__ X, int k, MoeSplit16Acts a) {
    const int lane = threadIdx.x & 63, nb = k / 256, sb = 4 * (int)blockIdx.y + (threadIdx.x >> 6), row = blockIdx.x;
    if (sb >= nb) return;
    const float4 v = *(const float4 *)(X + (size_t)row * k + 256 * sb + 4 * lane);
    const uint32_t big = max(max(s16_abs(v.x), s16_abs(v.y)), max(s16_abs(v.z), s16_abs(v.w)));
    uint32_t m = big;
#pragma unroll
    for (int off = 32; off; off >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, off, 64));
    const bool finite = m < 0x7F800000u;
    const int e = s16_exponent(m);
    const float f = finite ? s16_pow2(e) : 0.0f;
    // (order 0 2 1 3 of the lane's four)
    const float x[4] = {finite ? v.x * f : 0.0f, finite ? v.z * f : 0.0f, finite ? v.y * f : 0.0f, finite ? v.w * f : 0.0f};
    _Float16 hi[4], lo[4];
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        hi[i] = (_Float16)x[i];
        lo[i] = (_Float16)(x[i] - (float)hi[i]);
        sum += x[i];
    }
    const int j = lane >> 3, pos = 4 * (lane & 7);  // sub-block, element in it
    const int hs = j >> 2, g = 2 * ((j >> 1) & 1) + (pos >> 4), t = 2 * (j & 1) + ((pos >> 3) & 1);
    const size_t rec = (size_t)row * nb + sb;
    uint8_t *d = a.planes + rec * MS16_PLANES + 512 * hs + 128 * t + 16 * g + 2 * (pos & 4);
    __builtin_memcpy(__builtin_assume_aligned(d, 8), hi, 8);
    __builtin_memcpy(__builtin_assume_aligned(d + 64, 8), lo, 8);
#pragma unroll
    for (int off = 4; off; off >>= 1) sum += __shfl_xor(sum, off, 64);
    if ((lane & 7) == 0) {
        const float xs = sum * 0.03125f;
        const _Float16 h = (_Float16)xs, l = (_Float16)(xs - (float)h);
        ((_Float16 *)(a.xs + rec * MS16_XS))[j] = h;
        ((_Float16 *)(a.xs + rec * MS16_XS))[8 + j] = l;
    }
    if (lane == 0) a.s[rec] = finite ? s16_pow2(-e) : __builtin_nanf("");
}

struct MoeSplit16 {
    const uint8_t *const *wa, *const *wb;   // expert bases: gate and up, or down
    size_t row_bytes;
    MoeSplit16Acts acts;
    const int *gexp, *offsets, *xsel, *yrow;  // groups' experts, first pairs; a pair's activation row and result row
    float *Y;
    int groups, n, nb, cols;                // cols: column blocks of the grid
    int rows;                               // pairs of a tile, 32 or 48
    MoeClamp clamp;
};

// A workgroup of four waves multiplies a tile of up to 48 pairs of one expert with 64 WT weight rows (DUAL: half gate rows, half
// the up rows of the same columns, the gated unit in the epilogue); a wave owns WT tiles of 16 rows, RG row groups of 16 pairs.
// Bound: no one thing.  128 experts of 768 x 2048 and 512 tokens (32 pairs an expert), gate and up, 120 us: 31 us of matrix and 34 of vector
// instructions, 44 us for the weights at a large copy's rate, 18 us of starts and ends of workgroups; without its copies the loop takes 30 us
// less, without matrix instructions or unpacking 7 to 11.  The packed bytes come through LDS in pieces of a row (a lane that reads its own share
// of one looks up a cache line for itself, two clocks): the layer 247 -> 223 us.  Two halves of them on their way, and the activations in
// quarters, as two workgroups a compute unit leave room for: 100 tokens 139.5 -> 136.5, 150 tokens 151.5 -> 146.5, 512 tokens as before.
// The int8 GEMM took 3 x 102 us for the three products.
template <bool DUAL, int RG, int WT>
__device__ __forceinline__ void moe_split16_tile(const MoeSplit16 &a, int expert, int beg, int cnt, int cb, uint8_t *lds, float *s_lds,
                                                 int *y_lds, uint8_t *slots) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n16 = lane & 15, g = lane >> 4;
    constexpr int WD = DUAL ? WT / 2 : WT;  // tiles, and distinct columns' tiles
    const int nb = a.nb, c0 = (4 * cb + wave) * 16 * WD;
    uint32_t av[RG];          // this lane's share of a fragment: row n16 of each row group, 16-byte run g
#pragma unroll
    for (int r = 0; r < RG; r++) {
        const uint32_t rec = (uint32_t)a.xsel[beg + min(16 * r + n16, cnt - 1)] * (uint32_t)nb;
        av[r] = rec * MS16_PLANES + 16u * g;
    }
    // the sums: 32 RG pieces of 16 bytes, the same number for every wave
    constexpr int XP = 8 * RG;
    const uint32_t xv = (uint32_t)a.xsel[beg + min((XP * wave + lane) >> 1, cnt - 1)] * (uint32_t)nb * MS16_XS + 16u * (lane & 1);
    // A half's packed bytes of a tile are 64 pieces of 16, a lane's each: row lane / 4, piece lane % 4 turned by the row's quarter, so that 16
    // rows read at one place meet all banks once.  The headers are 16 pieces.
    const uint8_t *wp[WT];
    uint32_t wv[WT], wh[WT];
    const int turned = (lane & 3) ^ ((lane >> 4) & 3);
#pragma unroll
    for (int w = 0; w < WT; w++) {
        const int row = min(c0 + 16 * (w % WD), a.n - 1);
        wp[w] = s16_uniform((w >= WD ? a.wb : a.wa)[expert] + (size_t)row * a.row_bytes);
        wv[w] = (uint32_t)min(lane >> 2, a.n - 1 - row) * (uint32_t)a.row_bytes + 16u * (uint32_t)turned + 16u;
        wh[w] = (uint32_t)min(n16, a.n - 1 - row) * (uint32_t)a.row_bytes;
    }
    uint8_t *const own = slots + wave * WT * MS16_SLOTS;
    const uint32_t own_at = s16_lds_offset(own), lds0 = s16_lds_offset(lds);
    const uint8_t *const my_q = own + 256 + 64 * n16 + 16 * (g ^ (n16 >> 2)), *const my_hdr = own + 16 * n16;
#define JQ_COPY(v, base, dst) asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(v), "s"(base), "s"(__builtin_amdgcn_readfirstlane(dst)) : "memory")
    auto issue_w = [&](int sb, int hs) __attribute__((always_inline)) {
#pragma unroll
        for (int w = 0; w < WT; w++) {
            const uint8_t *base = wp[w] + (size_t)sb * 144;
            if (hs == 0 && lane < 16) JQ_COPY(wh[w], base, own_at + w * MS16_SLOTS);
            JQ_COPY(wv[w], base + 64 * hs, own_at + w * MS16_SLOTS + 256 + 1024 * hs);
        }
    };
    // A quarter is one nibble of a half: two k-steps of two planes, a wave's each; with the last one the sums.
    auto issue = [&](int sb, int qt, int buf) __attribute__((always_inline)) {
        const uint8_t *base = a.acts.planes + (size_t)sb * MS16_PLANES + 256 * qt + 64 * wave;
#pragma unroll
        for (int r = 0; r < RG; r++) JQ_COPY(av[r], base, lds0 + buf * MS16_BUF + (4 * r + wave) * S16_FRAG);
        if (qt == 3 && lane < XP) JQ_COPY(xv, a.acts.xs + (size_t)sb * MS16_XS, lds0 + 3 * MS16_BUF + 16 * XP * wave);
    };
#undef JQ_COPY
    uint4 hdr[WT], q[WT];
    auto read_w = [&](int hs) __attribute__((always_inline)) {
#pragma unroll
        for (int w = 0; w < WT; w++) {
            if (hs == 0) hdr[w] = *(const uint4 *)(my_hdr + w * MS16_SLOTS);
            q[w] = *(const uint4 *)(my_q + w * MS16_SLOTS + 1024 * hs);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // in registers: their places are free
#pragma unroll
        for (int w = 0; w < WT; w++) asm volatile("" : "+v"(q[w].x), "+v"(q[w].y), "+v"(q[w].z), "+v"(q[w].w));
    };
    // The products with the low plane in sums of their own, where registers are left: eight matrix instructions instead of 16 then
    // round a sum of the super-block's size.  128 experts of 2048 x 768, 6 to 16 pairs each: the layer's error against 64 bits
    // 7.3e-7 -> 5.9e-7 (the f32 products of the ring kernel 6.3e-7), its time, with tiles of 32 pairs there, 150 tokens 160.7 -> 162.5 us,
    // 250 tokens 183.8 -> 187.1.  Three row groups keep one chain.
    constexpr bool APART = RG <= 2;
    s16_f4 acc[WT][RG], i1[WT][RG], low[APART ? WT : 1][APART ? RG : 1];
    const s16_f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < WT; w++)
#pragma unroll
        for (int r = 0; r < RG; r++) acc[w][r] = zero;
    // (masks and magic numbers in registers: v_and_or_b32 takes one scalar operand and no two literals)
    uint32_t m_lo = 0x000F000Fu, m_hi = 0x00F000F0u, o_lo = 0x64006400u, o_hi = 0x54005400u;
    asm("" : "+s"(m_lo), "+s"(m_hi), "+v"(o_lo), "+v"(o_hi));
    // byte selectors: scale 2 (g / 2) + nibble of the half's four into both f16 of a register, each under 0x64
    const uint32_t sel0 = 0x04000400u + 0x00010001u * (uint32_t)(2 * (g >> 1)), sel1 = sel0 + 0x00010001u;
    auto multiply = [&](int nib, bool first, const uint32_t (&sc4)[WT], const uint8_t *l) __attribute__((always_inline)) {
        {
            s16_h8 b[2][WT];
#pragma unroll
            for (int w = 0; w < WT; w++) {
                const s16_h2 k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
                const s16_h2 sc = __builtin_bit_cast(s16_h2, __builtin_amdgcn_perm(0x64646464u, sc4[w], nib ? sel1 : sel0)) - k1024;
                const s16_h2 off = sc * (nib ? (_Float16)-64.0f : (_Float16)-1024.0f);
                const uint32_t words[4] = {q[w].x, q[w].y, q[w].z, q[w].w};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t even = words[i], odd = words[i] >> 8;
                    const uint32_t e = nib ? (even & m_hi) | o_hi : (even & m_lo) | o_lo;
                    const uint32_t o = nib ? (odd & m_hi) | o_hi : (odd & m_lo) | o_lo;
                    const s16_h2 pe = __builtin_elementwise_fma(__builtin_bit_cast(s16_h2, e), sc, off);
                    const s16_h2 po = __builtin_elementwise_fma(__builtin_bit_cast(s16_h2, o), sc, off);
                    b[i >> 1][w][4 * (i & 1)] = pe[0], b[i >> 1][w][4 * (i & 1) + 1] = pe[1];
                    b[i >> 1][w][4 * (i & 1) + 2] = po[0], b[i >> 1][w][4 * (i & 1) + 3] = po[1];
                }
            }
#pragma unroll
            for (int s8 = 0; s8 < 2; s8++)
#pragma unroll
                for (int p = 0; p < 2; p++)
#pragma unroll
                    for (int r = 0; r < RG; r++) {
                        const s16_h8 x = *(const s16_h8 *)(l + ((r * 2 + s8) * 2 + p) * S16_FRAG);
#pragma unroll
                        for (int w = 0; w < WT; w++) {
                            s16_f4 &to = APART && p ? low[APART ? w : 0][APART ? r : 0] : i1[w][r];
                            to = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, b[s8][w], first && s8 == 0 && (APART || p == 0) ? zero : to, 0, 0, 0);
                        }
                    }
        }
    };
    // Two halves of the weights are on their way while one is multiplied, and two quarters of the activations.
    issue_w(0, 0);
    issue(0, 0, 0);
    issue_w(0, 1);
    issue(0, 1, 1);
    if (tid < MS16_ROWS) y_lds[tid] = a.yrow[beg + min(tid, cnt - 1)];
    // the scales of the tile's rows, [super-block][row]
    for (int i = tid; i < 16 * RG * nb; i += 256) {
        const int row = i % (16 * RG), sb = i / (16 * RG);
        s_lds[i] = a.acts.s[(size_t)a.xsel[beg + min(row, cnt - 1)] * nb + sb];
    }
    const uint32_t live = g < 2 ? 0xFFFFFFFFu : 0u;
    int buf = 0;
    auto next = [](int b, int by) { return b + by >= 3 ? b + by - 3 : b + by; };
    // a quarter has landed once no more than what was asked for behind it is on its way; the buffer of the one before is free then
#define JQ_LANDED(behind) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(behind) : "memory")
    for (int sb = 0; sb < nb; sb++) {
        const bool more = sb + 1 < nb;
        uint32_t sc4[WT];
        JQ_LANDED(WT + RG);
        __builtin_amdgcn_s_barrier();
        issue(sb, 2, next(buf, 2));
        read_w(0);
        if (more) issue_w(sb + 1, 0);
#pragma unroll
        for (int w = 0; w < WT; w++) sc4[w] = hdr[w].y & 0x3F3F3F3Fu;
        multiply(0, true, sc4, lds + buf * MS16_BUF + 16 * lane);
        buf = next(buf, 1);
        if (more) JQ_LANDED(RG + 2 * WT);
        else JQ_LANDED(RG);
        __builtin_amdgcn_s_barrier();
        issue(sb, 3, next(buf, 2));
        multiply(1, false, sc4, lds + buf * MS16_BUF + 16 * lane);
        buf = next(buf, 1);
        if (more) JQ_LANDED(RG + 1 + 2 * WT);
        else JQ_LANDED(RG + 1);
        __builtin_amdgcn_s_barrier();
        if (more) issue(sb + 1, 0, next(buf, 2));
        read_w(1);
        if (more) issue_w(sb + 1, 1);
#pragma unroll
        for (int w = 0; w < WT; w++) sc4[w] = (hdr[w].w & 0x0F0F0F0Fu) | ((hdr[w].y >> 2) & 0x30303030u);
        multiply(0, false, sc4, lds + buf * MS16_BUF + 16 * lane);
        buf = next(buf, 1);
        if (more) JQ_LANDED(RG + WT);
        else JQ_LANDED(0);
        __builtin_amdgcn_s_barrier();
        if (more) issue(sb + 1, 1, next(buf, 2));
        multiply(1, false, sc4, lds + buf * MS16_BUF + 16 * lane);
        buf = next(buf, 1);
        s16_h8 xs[RG];  // (lane groups 2 and 3 meet zero mins)
#pragma unroll
        for (int r = 0; r < RG; r++) xs[r] = *(const s16_h8 *)(lds + 3 * MS16_BUF + (16 * r + n16) * MS16_XS + 16 * (g & 1));
        // the min term, and the super-block's sums onto the results
        s16_f4 s[RG];
#pragma unroll
        for (int r = 0; r < RG; r++) s[r] = *(const s16_f4 *)(s_lds + sb * 16 * RG + 16 * r + 4 * g);
#pragma unroll
        for (int w = 0; w < WT; w++) {
            const uint32_t mn[2] = {hdr[w].z & 0x3F3F3F3Fu, ((hdr[w].w >> 4) & 0x0F0F0F0Fu) | ((hdr[w].z >> 2) & 0x30303030u)};
            s16_h8 mins;
#pragma unroll
            for (int j = 0; j < 8; j += 2) {
                const s16_h2 k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
                const uint32_t pair = __builtin_amdgcn_perm(0x64646464u, mn[j >> 2], j & 2 ? 0x04030402u : 0x04010400u);
                const s16_h2 m = __builtin_bit_cast(s16_h2, __builtin_bit_cast(uint32_t, __builtin_bit_cast(s16_h2, pair) - k1024) & live);
                mins[j] = m[0], mins[j + 1] = m[1];
            }
            const float d = f16_bits(hdr[w].x), dm = -32.0f * f16_bits(hdr[w].x >> 16);
#pragma unroll
            for (int r = 0; r < RG; r++) {
                const s16_f4 i2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(xs[r], mins, zero, 0, 0, 0);
                if constexpr (APART) i1[w][r] += low[w][r];
#pragma unroll
                for (int i = 0; i < 4; i++) acc[w][r][i] = fmaf(s[r][i], fmaf(dm, i2[i], d * i1[w][r][i]), acc[w][r][i]);
            }
        }
    }
#undef JQ_LANDED
    // every result first, then the stores one behind the other: a load or a branch between them would wait for each
    const float limit = DUAL ? (expert >= a.clamp.n_routed ? a.clamp.shared : a.clamp.routed) : 0.0f;
    const float top = limit > 0.0f ? limit : INFINITY;
#pragma unroll
    for (int r = 0; r < RG; r++)
#pragma unroll
        for (int i = 0; i < 4; i++)
            if constexpr (DUAL) {
#pragma unroll
                for (int w = 0; w < WD; w++) {
                    float gt = acc[w][r][i], up = acc[(w + WD) % WT][r][i];
                    gt = gt > top ? top : gt;
                    up = up > top ? top : (up < -top ? -top : up);  // (comparisons: a NaN stays a NaN)
                    acc[w][r][i] = silu(gt) * up;
                }
            }
    int yr[RG][4];
#pragma unroll
    for (int r = 0; r < RG; r++)
#pragma unroll
        for (int i = 0; i < 4; i++) yr[r][i] = y_lds[16 * r + 4 * g + i];
#pragma unroll
    for (int r = 0; r < RG; r++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float *y = a.Y + (size_t)yr[r][i] * a.n + c0 + n16;
#pragma unroll
            for (int w = 0; w < WD; w++)
                if (16 * r + 4 * g + i < cnt && c0 + 16 * w + n16 < a.n) y[16 * w] = acc[w][r][i];
        }
}

// grid: cols x tiles (a multiple of 8; an upper bound, the rest leaves at once), ids 8 apart (one XCD) holding the column
// blocks of one tile, which read the same activation planes.
inline int moe_split16_lds(int nb, int WT) { return MS16_ACTS + 4 * MS16_ROWS * (nb + 1) + 4 * WT * MS16_SLOTS; }

template <bool DUAL, int WT>
static __global__ __launch_bounds__(256, 2) void moe_split16(MoeSplit16 a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];  // the activations, the scales, the result rows, the weights
    float *s_lds = (float *)(lds + MS16_ACTS);
    int *y_lds = (int *)(s_lds + MS16_ROWS * a.nb);
    uint8_t *slots = (uint8_t *)(y_lds + MS16_ROWS);
    const int id = blockIdx.x, mt = id / (8 * a.cols) * 8 + id % 8, cb = id / 8 % a.cols;
    int grp, at;
    if (!s16_find_tile(a.offsets, a.groups, a.rows, mt, grp, at)) return;  // past the last tile: the whole workgroup
    const int beg = a.offsets[grp] + at, cnt = min(a.offsets[grp + 1] - beg, a.rows), expert = a.gexp[grp];
    if (cnt <= 16) moe_split16_tile<DUAL, 1, WT>(a, expert, beg, cnt, cb, lds, s_lds, y_lds, slots);
    else if (cnt <= 32) moe_split16_tile<DUAL, 2, WT>(a, expert, beg, cnt, cb, lds, s_lds, y_lds, slots);
    else moe_split16_tile<DUAL, 3, WT>(a, expert, beg, cnt, cb, lds, s_lds, y_lds, slots);
}

}  // namespace jq

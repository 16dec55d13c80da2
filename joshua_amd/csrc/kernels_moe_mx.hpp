// Grouped products of MXFP4 experts on the matrix cores' own FP4: v_mfma_scale_f32_16x16x128_f8f6f4 takes 32 E2M1 codes a lane and
// the E8M0 byte of their block as they stand in memory, so a weight costs no vector instruction at all.
//
// An activation is 20-bit fixed point with a power of two a block of 32 (the scale that puts the block's largest magnitude below
// 2^19), written in four signed digits of five bits, X = 32768 d0 + 1024 d1 + 32 d2 + d3, -16 <= d <= 16: every digit is exact in
// FP8 (E4M3), and a digit's weight goes into its block scale.  Digits are columns of the second operand: a 16 x 16 tile
// multiplies 16 weight rows with four activation rows, and the four columns of a row are added at the end.  Products are
// exact, sums f32; the int8 planes of the kernels beside this one hold 16 bits a block.
//
// Element order.  Of a row, lane (n = lane % 16, g = lane / 16) holds weight row n and, of every 512 elements, four blocks in sequence:
// 68 bytes from byte 272 c + 68 g of the row, block st = 0 .. 3 at byte 17 st of them: 17 words, and with v_alignbyte
// (block 3 needs none) the four k-steps' operands; the scale bytes are picked out of the words by the instruction itself.
// In k-step st the inner index of block (c, g, st) is that of lane group g of the FP4 operand: code byte b holds elements b (low nibble) and b + 16.  The FP8 operand holds the same inner index as: lane group g, first
// 16 bytes: half g % 2 of the block of FP4 group g / 2; last 16 bytes: of FP4 group 2 + g / 2.
#pragma once
#include "split16_parts.hpp"

namespace jq {

typedef int mx_i8v __attribute__((ext_vector_type(8)));

constexpr int MX_CHUNK = 512;                    // elements of a row a step of the loop takes: 16 blocks, 272 bytes of weights
constexpr int MX_CHUNK_ACTS = 2048;              // bytes of their digits a row: [st 4][half 2][g 4][plane 4][16]
constexpr int MX_TILE = 16 * 272;                // bytes of a chunk of 16 weight rows

struct MoeMxActs {
    uint8_t *digits;                             // [row][chunk][2048]
    uint32_t *scales;                            // [row][chunk][g 4][plane 4]: the E8M0 bytes of st 0 .. 3
};

// grid (rows, chunks / 4), four waves, a wave a chunk of a row; lane = 4 block + quarter of eight elements.  A block
// that holds an inf or a NaN gets the scale NaN.
static __global__ __launch_bounds__(256) void moe_mx_prep(const float *__restrict__ X, int k, MoeMxActs a) {
    const int lane = threadIdx.x & 63, nc = k / MX_CHUNK, c = 4 * (int)blockIdx.y + (threadIdx.x >> 6), row = blockIdx.x;
    if (c >= nc) return;
    const float *src = X + (size_t)row * k + MX_CHUNK * c + 8 * lane;
    const float4 v0 = *(const float4 *)src, v1 = *(const float4 *)(src + 4);
    const float x[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) m = max(m, s16_abs(x[i]));
    m = max(m, (uint32_t)__shfl_xor((int)m, 1, 64));
    m = max(m, (uint32_t)__shfl_xor((int)m, 2, 64));
    const bool finite = m < 0x7F800000u;
    const int ex = max((int)(m >> 23) - 127, -100);   // largest magnitude below 2^(ex + 1)
    const float f = ldexpf(1.0f, 18 - ex);
    uint32_t d[4][2];                                 // [plane][four elements]
#pragma unroll
    for (int w = 0; w < 2; w++) {
        float dig[4][4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            int X4 = finite ? (int)rintf(x[4 * w + i] * f) : 0;
#pragma unroll
            for (int p = 3; p > 0; p--) {
                const int low = ((X4 + 16) & 31) - 16;
                dig[p][i] = (float)low;
                X4 = (X4 - low) >> 5;
            }
            dig[0][i] = (float)X4;
        }
#pragma unroll
        for (int p = 0; p < 4; p++) {
            int word = __builtin_amdgcn_cvt_pk_fp8_f32(dig[p][0], dig[p][1], 0, false);
            d[p][w] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(dig[p][2], dig[p][3], word, true);
        }
    }
    // Quarters q and q ^ 2 hold elements b and b + 16 of half q & 1 and are interleaved byte by byte; quarters 0 and 1 write planes 0
    // and 1 of their half, quarters 2 and 3 planes 2 and 3.
    const int q = lane & 3, blk = lane >> 2, st = blk & 3, ga = blk >> 2, half = q & 1;
    uint32_t o[4][2];
#pragma unroll
    for (int p = 0; p < 4; p++)
#pragma unroll
        for (int w = 0; w < 2; w++) o[p][w] = (uint32_t)__shfl_xor((int)d[p][w], 2, 64);
    const size_t rec = (size_t)row * nc + c;
    uint8_t *out = a.digits + rec * MX_CHUNK_ACTS + ((st * 2 + (ga >> 1)) * 4 + 2 * (ga & 1) + half) * 64;
#pragma unroll
    for (int pp = 0; pp < 2; pp++) {
        const bool upper = q >= 2;
        uint32_t lo[2], hi[2];
#pragma unroll
        for (int w = 0; w < 2; w++) {
            lo[w] = upper ? o[2 + pp][w] : d[pp][w];      // elements b
            hi[w] = upper ? d[2 + pp][w] : o[pp][w];      // elements b + 16
        }
        const uint4 v{__builtin_amdgcn_perm(hi[0], lo[0], 0x05010400u), __builtin_amdgcn_perm(hi[0], lo[0], 0x07030602u),
                      __builtin_amdgcn_perm(hi[1], lo[1], 0x05010400u), __builtin_amdgcn_perm(hi[1], lo[1], 0x07030602u)};
        *(uint4 *)(out + 16 * (upper ? 2 + pp : pp)) = v;
    }
    // (a block's four lanes: lane q writes plane q's byte)
    ((uint8_t *)(a.scales + rec * 16 + 4 * ga + q))[st] = finite ? (uint8_t)(124 + ex - 5 * q) : 0xFF;
}

struct MoeMx {
    const uint8_t *const *wa, *const *wb;
    size_t row_bytes;
    MoeMxActs acts;
    const int *gexp, *offsets, *xsel, *yrow;
    float *Y;
    int groups, n, nc, cols, span;               // cols: runs of `span` column blocks
    MoeClamp clamp;
};

// A workgroup of WAVES waves multiplies a tile of up to 4 MAXNG pairs of one expert with `span` column blocks, one after the
// other, of 32 WAVES weight rows (DUAL: half gate rows, half the up rows of the same columns); a wave takes 2 x 16 of them.
// The chunks of all blocks are one stream: asynchronous loads bring a chunk of the wave's rows (contiguous 16-byte pieces; read
// straight into operands, each lane touches a cache line of its own, five lookups for its 68 bytes: 1330 us the layer below)
// into a slot in LDS that is free again as soon as its words are in registers, and the digits of the pairs, gathered, into two buffers.
// Bound: memory.  DeepSeek-V3's size, 64 tokens (222 of 256 experts and the shared one, 5.24 GB): the layer 1058 us, 4.9 TB/s of
// weights over the whole call where a large copy moves 5.1 (on the int8 kernels 2016).  At 512 tokens 1.9 ms (3.9): the digits
// cost four columns a pair, and tiles of 16 pairs are read again from the second level cache.
template <bool DUAL, int WAVES, int NG, int MAXNG>
__device__ __forceinline__ void moe_mx_tile(const MoeMx &a, int expert, int beg, int cnt, int cb0, uint8_t *lds, int *y_lds) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n16 = lane & 15, g = lane >> 4;
    constexpr int BUF = NG * 8 * S16_FRAG, ROWS = (DUAL ? 16 : 32) * WAVES, SLOTS = 2 * MAXNG * 8 * S16_FRAG;
    const int nc = a.nc, blocks = min(a.span, (a.n + ROWS - 1) / ROWS - cb0), total = nc * blocks;
    if (tid < 4 * MAXNG) y_lds[tid] = a.yrow[beg + min(tid, cnt - 1)];
    uint32_t av[NG];               // this lane's share of a digit fragment: pair 4 q + n / 4, plane n % 4, run g
    const uint32_t *sp[NG];
#pragma unroll
    for (int q = 0; q < NG; q++) {
        const uint32_t rec = (uint32_t)a.xsel[beg + min(4 * q + (n16 >> 2), cnt - 1)] * (uint32_t)nc;
        av[q] = rec * MX_CHUNK_ACTS + 64u * g + 16u * (n16 & 3);
        sp[q] = a.acts.scales + (size_t)rec * 16 + 4 * g + (n16 & 3);
    }
    uint32_t wv_off[5];            // 16-byte piece 64 j + lane of a tile: row by row, 17 a row
#pragma unroll
    for (int j = 0; j < 5; j++) {
        const int piece = min(64 * j + lane, 271);
        wv_off[j] = (uint32_t)(piece / 17) * (uint32_t)a.row_bytes + 16u * (uint32_t)(piece % 17);
    }
    const uint8_t *wa = a.wa[expert], *wb = DUAL ? a.wb[expert] : nullptr;
    const uint32_t lds0 = s16_lds_offset(lds), slot0 = lds0 + SLOTS + 2 * MX_TILE * wave;
    const uint8_t *slot = lds + SLOTS + 2 * MX_TILE * wave + 272 * n16 + 68 * g;
    auto column = [&](int cb) __attribute__((always_inline)) { return DUAL ? ROWS * cb + 16 * wave : ROWS * cb + 32 * wave; };
    uint32_t s_next[NG];
    auto issue = [&](int c, int cb, int buf) __attribute__((always_inline)) {
        const int c0 = column(cb);
#pragma unroll
        for (int w = 0; w < 2; w++) {  // (rows past the matrix: its last ones, whose results are not stored)
            const uint8_t *base = s16_uniform((DUAL && w ? wb : wa) + (size_t)min(DUAL ? c0 : c0 + 16 * w, a.n - 16) * a.row_bytes + (size_t)c * 272);
#pragma unroll
            for (int j = 0; j < 5; j++) {
                const uint32_t dst = __builtin_amdgcn_readfirstlane(slot0 + w * MX_TILE + 1024 * j);
                if (j < 4 || lane < 16)
                    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(wv_off[j]), "s"(base), "s"(dst) : "memory");
            }
        }
        // digits: the 8 fragments of a group of pairs go round the waves
        const uint8_t *base = s16_uniform(a.acts.digits + (size_t)c * MX_CHUNK_ACTS);
#pragma unroll
        for (int f = 0; f < 8; f++) {
            if (f % WAVES != wave) continue;
#pragma unroll
            for (int q = 0; q < NG; q++) {
                const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + buf * BUF + (q * 8 + f) * S16_FRAG);
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(av[q]), "s"(base + 256 * f), "s"(dst) : "memory");
            }
        }
#pragma unroll
        for (int q = 0; q < NG; q++) s_next[q] = sp[q][(size_t)c * 16];
        __builtin_amdgcn_sched_barrier(0);  // (else these loads sink to where they are read, a step later)
    };
    s16_f4 acc[2][NG];
#pragma unroll
    for (int w = 0; w < 2; w++)
#pragma unroll
        for (int q = 0; q < NG; q++) acc[w][q] = s16_f4{0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t x[2][17], xs[NG];
    auto multiply = [&](const uint8_t *l) __attribute__((always_inline)) {
#define JQ_MX_STEP(ST)                                                                                                                          \
    {                                                                                                                                           \
        mx_i8v wv[2];                                                                                                                           \
        _Pragma("unroll") for (int w = 0; w < 2; w++)                                                                                           \
            _Pragma("unroll") for (int i = 0; i < 4; i++) {                                                                                     \
                wv[w][i] = (int)(ST == 3 ? x[w][4 * ST + 1 + i] : __builtin_amdgcn_alignbyte(x[w][4 * ST + 1 + i], x[w][4 * ST + i], (ST + 1) & 3)); \
                wv[w][4 + i] = 0;                                                                                                               \
            }                                                                                                                                   \
        _Pragma("unroll") for (int q = 0; q < NG; q++) {                                                                                        \
            const uint4 d0 = *(const uint4 *)(l + (q * 8 + 2 * ST) * S16_FRAG), d1 = *(const uint4 *)(l + (q * 8 + 2 * ST + 1) * S16_FRAG);       \
            const mx_i8v dv = {(int)d0.x, (int)d0.y, (int)d0.z, (int)d0.w, (int)d1.x, (int)d1.y, (int)d1.z, (int)d1.w};                         \
            _Pragma("unroll") for (int w = 0; w < 2; w++) acc[w][q] =                                                                           \
                __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wv[w], dv, acc[w][q], 4, 0, ST, (int)x[w][4 * ST], ST, (int)xs[q]);             \
        }                                                                                                                                       \
    }
        JQ_MX_STEP(0)
        JQ_MX_STEP(1)
        JQ_MX_STEP(2)
        JQ_MX_STEP(3)
#undef JQ_MX_STEP
    };
    const float limit = DUAL ? (expert >= a.clamp.n_routed ? a.clamp.shared : a.clamp.routed) : 0.0f;
    const float top = limit > 0.0f ? limit : INFINITY;
    issue(0, cb0, 0);
    int c = 0, cb = cb0;
    for (int t = 0; t < total; t++) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int q = 0; q < NG; q++) {  // (the compiler's own waits: here, and not behind the loads issued next)
            asm volatile("" : "+v"(s_next[q]));
            xs[q] = s_next[q];
        }
        __syncthreads();  // the chunk has landed, and the other digit buffer's readers are done
#pragma unroll
        for (int w = 0; w < 2; w++) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const s16_u4 v = *(const s16_u4 *)(slot + w * MX_TILE + 16 * i);
                x[w][4 * i] = v[0], x[w][4 * i + 1] = v[1], x[w][4 * i + 2] = v[2], x[w][4 * i + 3] = v[3];
            }
            x[w][16] = *(const uint32_t *)(slot + w * MX_TILE + 64);
        }
#pragma unroll
        for (int w = 0; w < 2; w++)
#pragma unroll
            for (int i = 0; i < 17; i++) asm volatile("" : "+v"(x[w][i]));
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the words are in registers: the slot is free
        const int c_now = c, cb_now = cb;
        if (++c == nc) c = 0, cb++;
        if (t + 1 < total) issue(c, cb, (t + 1) & 1);
        // a block whose scale is 0xFF stands for zeros
        bool odd = false;
#pragma unroll
        for (int w = 0; w < 2; w++)
#pragma unroll
            for (int st = 0; st < 4; st++) odd |= ((x[w][4 * st] >> (8 * st)) & 0xFFu) == 0xFFu;
        if (__builtin_expect(__any(odd), 0)) {
            asm volatile("" ::: "memory");  // (a branch: no selects on the common path)
#pragma unroll
            for (int w = 0; w < 2; w++)
#pragma unroll
                for (int st = 0; st < 4; st++) {
                    if (((x[w][4 * st] >> (8 * st)) & 0xFFu) != 0xFFu) continue;
                    x[w][4 * st] &= (1u << (8 * st)) - 1u;
                    x[w][4 * st + 1] = x[w][4 * st + 2] = x[w][4 * st + 3] = 0;
                    x[w][4 * st + 4] &= st == 3 ? 0u : ~((1u << (8 * ((st + 1) & 3))) - 1u);
                }
        }
        multiply(lds + (t & 1) * BUF + 16 * lane);
        if (c_now + 1 < nc) continue;
        // the four digit columns of a pair; lane n % 4 then keeps row n % 4 of its four
        const int p = n16 & 3, row = column(cb_now) + 4 * g + p;
#pragma unroll
        for (int q = 0; q < NG; q++) {
            float y[2];
#pragma unroll
            for (int w = 0; w < 2; w++) {
                float r[4];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float v = acc[w][q][i] + dpp_f<0xB1>(acc[w][q][i]);  // quad_perm [1,0,3,2]
                    r[i] = v + dpp_f<0x4E>(v);                                 // quad_perm [2,3,0,1]
                    acc[w][q][i] = 0.0f;
                }
                y[w] = p == 0 ? r[0] : p == 1 ? r[1] : p == 2 ? r[2] : r[3];
            }
            const int pair = 4 * q + (n16 >> 2);
            float *dst = a.Y + (size_t)y_lds[pair] * a.n + row;
            if constexpr (DUAL) {
                float gt = y[0], up = y[1];
                gt = gt > top ? top : gt;
                up = up > top ? top : (up < -top ? -top : up);  // (comparisons: a NaN stays a NaN)
                if (pair < cnt && row < a.n) *dst = silu(gt) * up;
            } else {
                if (pair < cnt && row < a.n) dst[0] = y[0];
                if (pair < cnt && row + 16 < a.n) dst[16] = y[1];
            }
        }
    }
}

constexpr int moe_mx_lds(int waves, int maxng) { return 2 * maxng * 8 * S16_FRAG + 2 * MX_TILE * waves; }

// grid: cols x tiles, as moe_split16's.
template <bool DUAL, int WAVES, int MAXNG>
static __global__ __launch_bounds__(64 * WAVES, 2) void moe_mx(MoeMx a) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[moe_mx_lds(WAVES, MAXNG)];
    __shared__ int y_lds[4 * MAXNG];
    const int id = blockIdx.x, mt = id / (8 * a.cols) * 8 + id % 8, cb0 = id / 8 % a.cols * a.span;
    int grp, at;
    if (!s16_find_tile(a.offsets, a.groups, 4 * MAXNG, mt, grp, at)) return;  // past the last tile: the whole workgroup
    const int beg = a.offsets[grp] + at, cnt = min(a.offsets[grp + 1] - beg, 4 * MAXNG), expert = a.gexp[grp];
    if (cnt <= 4) moe_mx_tile<DUAL, WAVES, 1, MAXNG>(a, expert, beg, cnt, cb0, lds, y_lds);
    else if (MAXNG == 2 || cnt <= 8) moe_mx_tile<DUAL, WAVES, 2, MAXNG>(a, expert, beg, cnt, cb0, lds, y_lds);
    else if constexpr (MAXNG == 4) moe_mx_tile<DUAL, WAVES, 4, MAXNG>(a, expert, beg, cnt, cb0, lds, y_lds);
}

}  // namespace jq

// Attention of many tokens on the f16 matrix cores at f32 precision.  A factor x is held as the sum of two f16 numbers,
// hi = f16(x) and lo = f16(x - hi): 22 to 23 bits of it.  A product takes three v_mfma_f32_32x32x16_f16, hi hi + hi lo +
// lo hi, with f32 sums; what is left out, lo lo, is at most 2^-22 of it and 2^-25 on average.  Three f16 products run
// at 833 TFLOP/s where the f32 matrix cores have 157.  f16 reaches from 2^-24 to 2^16, so every operand is first scaled by
// a power of two (exact) that puts the largest magnitude of its row, tile or matrix at 2^13 .. 2^14; elements down to 2^-14
// of that one keep all their bits.
//
// The roundings of the f32 sums are what is left of the error: an instruction adds 16 products to a sum where the f32 cores'
// adds four, but three instructions stand in one chain.  Error of the attention alone against 64 bits as a share of the f32
// kernels' (2-norm and largest; mean over 3 draws of 4 or 5 shapes up to 3000 keys; normal operands, channels 20 times
// the others, a first token of 30 times the others, log-normal sizes): the decoder's 0.90 0.79 0.88 0.81 and 0.82 0.76 0.80 0.76;
// latent attention, whose chains are longer and broken up for it, 0.68 0.85 0.84 0.79 and 0.79 0.86 0.80 0.92.
//
// Operands lie in memory as the matrix cores take them: a fragment is 32 rows x 16 of the inner index, lane l holding row
// l % 32 and eight inner elements as 16 bytes, 1 KB in all, and travels global -> LDS -> registers without a shuffle.
// Scores are made transposed, S^T = K Q^T, so that a lane ends with one query's scores of 16 keys (rows 8 (r / 4) +
// 4 (l / 32) + r % 4 of register r): running maximum, sum and the output's rescaling stay in the lane, and the
// weights are the second operand of O^T += V^T P^T as they stand, the keys of V's fragments in that same order.
//
// Bound: the matrix cores (by counters 50 % of the compute units' busy cycles in the decoder's attention and in the expansion, 54 in
// latent attention; no bank conflicts), then the LDS reads of a tile by each of the four waves.  Measured against the f32 matrix
// cores' kernels: the decoder's attention of 2048 tokens, 32 / 8 heads of 128, 606 -> 129 us a layer (796 TFLOP/s of f16
// products) and 10 of preparation; latent attention of DeepSeek-V3's size, 512 tokens behind 0 .. 3584 (on average): 3060 us of
// attention on the absorbed queries, 645 of value projection, 208 of absorption, 122 of merging -> 249 us of expanding, 273 of
// attention and 10 of preparation.  Against 64-bit results the errors of both are the same (1.0e-4 and 1.5e-4 of the norm, the 16-bit
// activations of the products around them).
#pragma once
#include "split16_parts.hpp"

namespace jq {

constexpr int S16_TILE = 32;                         // keys (or tokens) of a tile
constexpr int S16_KV_TILE = 2 * 8 * 2 * S16_FRAG;    // a head's K (128) and V (128) of a tile: 8 fragments each, two planes
constexpr int S16_ROPE_TILE = 4 * 2 * S16_FRAG;      // the shared rope keys (64) of a tile

// What the attention knows of a tile: the powers of two that undo its scales (k: of the keys, or of the rope keys; v: of the
// values), and a bit per key that holds an infinity or a NaN.  Such an element counts as zero in the tile: 0, the weight of a
// key that a query does not see, times it would reach that query's sums, and a scale that follows it would take the other
// keys' bits.  The queries that see the key are NaN.
struct __attribute__((aligned(16))) S16Tile {
    float k, v;
    uint32_t bad, unused;
};

__device__ __forceinline__ uint32_t s16_block_max(uint32_t v, uint32_t *red) {  // 256 threads
#pragma unroll
    for (int off = 32; off; off >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, off, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return max(max(red[0], red[1]), max(red[2], red[3]));
}

__device__ __forceinline__ s16_f16 s16_mma(const s16_h8 &a, const s16_h8 &b, const s16_f16 &c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// ---- keys and values of a cache [kv_head][n_ctx][128] f32 as fragments -----------------------------------------------------
// grid (tiles, kv heads), 256 threads.  Rows at and past n_keys are zero.  Bound: memory (twice the cache's bytes).
__global__ __launch_bounds__(256) void s16_kv_tiles(const float *__restrict__ kc, const float *__restrict__ vc, int n_ctx, int n_keys,
                                                    uint8_t *__restrict__ ws, S16Tile *__restrict__ info) {
    constexpr int D = 128, PAD = 4;
    __shared__ __attribute__((aligned(16))) float vt[S16_TILE][D + PAD];
    __shared__ uint32_t red[4], bad;
    const int tile = blockIdx.x, kvh = blockIdx.y, tid = threadIdx.x;
    if (tid == 0) bad = 0;
    __syncthreads();
    const float *kb = kc + ((size_t)kvh * n_ctx + (size_t)tile * S16_TILE) * D, *vb = vc + ((size_t)kvh * n_ctx + (size_t)tile * S16_TILE) * D;
    uint8_t *out = ws + ((size_t)kvh * gridDim.x + tile) * S16_KV_TILE;
    // K: chunk (k-step s, lane) = row lane % 32, columns 16 s + 8 (lane / 32) ..; two chunks a thread
    float kx[2][8];
    uint32_t km = 0, vm = 0;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int c = tid + 256 * u, row = (c & 31), col = 16 * (c >> 6) + 8 * ((c >> 5) & 1);
        const bool live = tile * S16_TILE + row < n_keys;
#pragma unroll
        for (int i = 0; i < 8; i += 4) {
            const float4 v = live ? *(const float4 *)(kb + (size_t)row * D + col + i) : float4{0.f, 0.f, 0.f, 0.f};
            kx[u][i] = v.x, kx[u][i + 1] = v.y, kx[u][i + 2] = v.z, kx[u][i + 3] = v.w;
        }
        if (!s16_make_finite(kx[u])) atomicOr(&bad, 1u << row);
#pragma unroll
        for (int i = 0; i < 8; i++) km = max(km, s16_abs(kx[u][i]));
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int c = tid + 256 * u, row = c >> 5, col = 4 * (c & 31);
        const float4 v = tile * S16_TILE + row < n_keys ? *(const float4 *)(vb + (size_t)row * D + col) : float4{0.f, 0.f, 0.f, 0.f};
        float x[4] = {v.x, v.y, v.z, v.w};
        if (!s16_make_finite(x)) atomicOr(&bad, 1u << row);
        *(float4 *)&vt[row][col] = float4{x[0], x[1], x[2], x[3]};
#pragma unroll
        for (int i = 0; i < 4; i++) vm = max(vm, s16_abs(x[i]));
    }
    const int ke = s16_exponent(s16_block_max(km, red)), ve = s16_exponent(s16_block_max(vm, red));  // (their barriers publish vt)
    const float kf = s16_pow2(ke), vf = s16_pow2(ve);
    if (tid == 0) info[(size_t)kvh * gridDim.x + tile] = S16Tile{s16_pow2(-ke), s16_pow2(-ve), bad, 0u};
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int c = tid + 256 * u, s = c >> 6, lane = c & 63;
        s16_h8 hi, lo;
#pragma unroll
        for (int i = 0; i < 8; i++) kx[u][i] *= kf;
        s16_split(kx[u], hi, lo);
        *(s16_h8 *)(out + (2 * s) * S16_FRAG + 16 * lane) = hi;
        *(s16_h8 *)(out + (2 * s + 1) * S16_FRAG + 16 * lane) = lo;
    }
    // V^T: chunk (tile of 32 columns mt, 16 keys ks, lane) = column 32 mt + lane % 32, keys 16 ks + 8 (i / 4) + 4 (lane / 32) + i % 4
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int c = tid + 256 * u, f = c >> 6, lane = c & 63, col = 32 * (f >> 1) + (lane & 31);
        float x[8];
#pragma unroll
        for (int i = 0; i < 8; i++) x[i] = vt[16 * (f & 1) + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3)][col] * vf;
        s16_h8 hi, lo;
        s16_split(x, hi, lo);
        *(s16_h8 *)(out + S16_KV_TILE / 2 + (2 * f) * S16_FRAG + 16 * lane) = hi;
        *(s16_h8 *)(out + S16_KV_TILE / 2 + (2 * f + 1) * S16_FRAG + 16 * lane) = lo;
    }
}

// ---- latent attention: the up-projection, the cached latents, the keys and values they stand for -----------------------------
constexpr int S16_LKV = 512, S16_ROPE = 64, S16_HEAD = 128;  // latent, rope part, a head's keys and values

// Once per object.  grid (2, heads), 256 threads: part 0 the rows of W_k[h], part 1 those of W_v[h], [128][512] f32 each, as
// fragments [head][part][k-step 32][row tile 4][plane].  fac[h][part] = {power of two on a product of these fragments and
// those of s16_latent_tiles that keeps it below 2^15, the power of two that undoes the result's scale}: |W_j . c| is
// bounded by |W_j| cmax, cmax the largest 2-norm a normed latent can have (ec: the exponent of its scale).
__global__ __launch_bounds__(256) void s16_up_projection(const float *__restrict__ wkv, uint8_t *__restrict__ frags, float2 *__restrict__ fac,
                                                         float cmax, int ec) {
    __shared__ uint32_t red[4];
    const int part = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const float *W = wkv + ((size_t)h * 2 + part) * S16_HEAD * S16_LKV;
    uint32_t amax = 0, nmax = 0;
    for (int j = wave; j < S16_HEAD; j += 4) {
        float ss = 0.0f;
        for (int c = lane; c < S16_LKV; c += 64) {
            const float v = W[(size_t)j * S16_LKV + c];
            amax = max(amax, s16_abs(v)), ss = fmaf(v, v, ss);
        }
        nmax = max(nmax, s16_abs(sqrtf(wave_sum(ss)) * cmax));
    }
    const int ew = s16_exponent(s16_block_max(amax, red)), er = s16_exponent(s16_block_max(nmax, red));
    const float f = s16_pow2(ew);
    if (tid == 0) fac[2 * h + part] = float2{ldexpf(1.0f, er - ec - ew), s16_pow2(-er)};
    uint8_t *out = frags + ((size_t)h * 2 + part) * (S16_LKV / 16) * 8 * S16_FRAG;
    for (int c = tid; c < (S16_LKV / 16) * 4 * 64; c += 256) {
        const int l = c & 63, rt = (c >> 6) & 3, s = c >> 8;
        const float *src = W + (size_t)(32 * rt + (l & 31)) * S16_LKV + 16 * s + 8 * (l >> 5);
        float x[8];
#pragma unroll
        for (int i = 0; i < 8; i++) x[i] = src[i] * f;
        s16_h8 hi, lo;
        s16_split(x, hi, lo);
        uint8_t *d = out + ((size_t)(s * 4 + rt) * 2) * S16_FRAG + 16 * l;
        *(s16_h8 *)d = hi;
        *(s16_h8 *)(d + S16_FRAG) = lo;
    }
}

// grid tiles (from tile0 on), 256 threads: the normed latents of 32 tokens as fragments [tile][k-step 32][plane] (times 2^ec), their rope keys
// as [tile][k-step 4][plane] with a scale a tile, info[tile].k the power of two that undoes it.
__global__ __launch_bounds__(256) void s16_latent_tiles(const float *__restrict__ lat, const float *__restrict__ kpe, int tile0, int n_keys, float cscale,
                                                        uint8_t *__restrict__ cf, uint8_t *__restrict__ rf, S16Tile *__restrict__ info) {
    __shared__ uint32_t red[4], bad;
    const int tile = tile0 + (int)blockIdx.x, tid = threadIdx.x, lane = tid & 63, row = lane & 31, key = tile * S16_TILE + row;
    const bool live = key < n_keys;
    float x[8];
    bool whole = true;
    auto fetch = [&](const float *src) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; i += 4) {
            const float4 v = live ? *(const float4 *)(src + i) : float4{0.f, 0.f, 0.f, 0.f};
            x[i] = v.x, x[i + 1] = v.y, x[i + 2] = v.z, x[i + 3] = v.w;
        }
        whole &= s16_make_finite(x);
    };
    s16_h8 hi, lo;
    if (tid == 0) bad = 0;
    __syncthreads();
    uint8_t *out = cf + (size_t)tile * (S16_LKV / 16) * 2 * S16_FRAG + 16 * lane;
#pragma unroll 4
    for (int s = tid >> 6; s < S16_LKV / 16; s += 4) {
        fetch(lat + (size_t)key * S16_LKV + 16 * s + 8 * (lane >> 5));
#pragma unroll
        for (int i = 0; i < 8; i++) x[i] *= cscale;
        s16_split(x, hi, lo);
        *(s16_h8 *)(out + (2 * s) * S16_FRAG) = hi;
        *(s16_h8 *)(out + (2 * s + 1) * S16_FRAG) = lo;
    }
    const int s = tid >> 6;
    fetch(kpe + (size_t)key * S16_ROPE + 16 * s + 8 * (lane >> 5));
    if (!whole) atomicOr(&bad, 1u << row);
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) m = max(m, s16_abs(x[i]));
    const int e = s16_exponent(s16_block_max(m, red));
    const float f = s16_pow2(e);
    if (tid == 0) info[tile] = S16Tile{s16_pow2(-e), 1.0f, bad, 0u};
#pragma unroll
    for (int i = 0; i < 8; i++) x[i] *= f;
    s16_split(x, hi, lo);
    out = rf + (size_t)tile * S16_ROPE_TILE + 16 * lane;
    *(s16_h8 *)(out + (2 * s) * S16_FRAG) = hi;
    *(s16_h8 *)(out + (2 * s + 1) * S16_FRAG) = lo;
}

// Keys (part 0) and values (part 1) of `heads` heads from head h0 on, for the n_tiles tiles of cached tokens from tile0 on, written
// as the fragments the attention below reads: [head - h0][tile of `stride`]{K, V}.  grid (token blocks x 2 heads) of four waves; a workgroup multiplies 128
// rows of the up-projection with 128 latents, k in stages of 32 through two LDS buffers.  The accumulators leave as whole
// fragments: of K the product is made with the projection's rows first (a lane holds eight columns of one key), of V with the
// latents first (eight keys of one column).
template <bool V>
__device__ __forceinline__ void s16_expand_workgroup(const uint8_t *__restrict__ wf, const uint8_t *__restrict__ cf, float f, int n_tiles, int tb,
                                                     uint8_t *__restrict__ out, uint8_t *lds) {
    constexpr int STAGE = 2 * 8 * 2 * S16_FRAG, N_STAGES = S16_LKV / 32;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wave & 1, wc = wave >> 1;
    const uint32_t lds0 = s16_lds_offset(lds);
    // a stage: 16 KB of the projection, contiguous; 4 KB of each of four latent tiles (past the last tile: that one again)
    const int ct = min(4 * tb + wave, n_tiles - 1);
    const uint8_t *wsrc = wf + 4096 * wave + 16 * lane, *csrc = cf + (size_t)ct * (S16_LKV / 16) * 2 * S16_FRAG + 16 * lane;
    auto issue = [&](int st, int buf) __attribute__((always_inline)) {
        const uint32_t base = lds0 + buf * STAGE + 4096 * wave;
#pragma unroll
        for (int i = 0; i < 4; i++) s16_copy16(wsrc + (size_t)st * 16384 + 1024 * i, base + 1024 * i);
#pragma unroll
        for (int i = 0; i < 4; i++) s16_copy16(csrc + (size_t)st * 4096 + 1024 * i, base + 16384 + 1024 * i);
    };
    // Sums apart, for their roundings: the products with a low plane, and the others in runs of 128 columns (in one chain of 96
    // matrix instructions the whole attention's error is 1.3 times as large, 1.2 of the f32 kernels' on rows with outliers)
    s16_f16 acc[2][2], low[2][2], run[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[a][b][r] = low[a][b][r] = run[a][b][r] = 0.0f;
    issue(0, 0);
    for (int st = 0; st < N_STAGES; st++) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (st + 1 < N_STAGES) issue(st + 1, (st + 1) & 1);
        const uint8_t *l = lds + (st & 1) * STAGE + 16 * lane;
#pragma unroll
        for (int s = 0; s < 2; s++) {
            s16_h8 w[2][2], c[2][2];  // [tile][plane]
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int p = 0; p < 2; p++) {
                    w[t][p] = *(const s16_h8 *)(l + ((s * 4 + 2 * wr + t) * 2 + p) * S16_FRAG);
                    c[t][p] = *(const s16_h8 *)(l + 16384 + 4096 * (2 * wc + t) + (s * 2 + p) * S16_FRAG);
                }
#pragma unroll
            for (int q = 0; q < 3; q++)  // hi hi, hi lo, lo hi
#pragma unroll
                for (int a = 0; a < 2; a++)
#pragma unroll
                    for (int b = 0; b < 2; b++) {
                        const s16_h8 &x = w[a][q == 2], &y = c[b][q == 1];
                        s16_f16 &to = q ? low[a][b] : run[a][b];
                        to = V ? s16_mma(y, x, to) : s16_mma(x, y, to);
                    }
        }
        if (st % 4 == 3) {
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int b = 0; b < 2; b++)
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[a][b][r] += run[a][b][r], run[a][b][r] = 0.0f;
        }
    }
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[a][b][r] += low[a][b][r];
#pragma unroll
    for (int b = 0; b < 2; b++) {
        const int tile = 4 * tb + 2 * wc + b;
        if (tile >= n_tiles) break;
#pragma unroll
        for (int a = 0; a < 2; a++) {
            uint8_t *d = out + (size_t)tile * S16_KV_TILE + (V ? S16_KV_TILE / 2 : 0) + (2 * wr + a) * 4 * S16_FRAG + 16 * lane;
#pragma unroll
            for (int half = 0; half < 2; half++) {
                float x[8];
#pragma unroll
                for (int i = 0; i < 8; i++) x[i] = acc[a][b][8 * half + i] * f;
                s16_h8 hi, lo;
                s16_split(x, hi, lo);
                *(s16_h8 *)(d + (2 * half) * S16_FRAG) = hi;
                *(s16_h8 *)(d + (2 * half + 1) * S16_FRAG) = lo;
            }
        }
    }
}

__global__ __launch_bounds__(256, 2) void s16_expand(const uint8_t *__restrict__ wfrags, const float2 *__restrict__ fac, const uint8_t *__restrict__ cf,
                                                     int h0, int heads, int tile0, int n_tiles, int stride, uint8_t *__restrict__ ws) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * 2 * 8 * 2 * S16_FRAG];
    // a head stays on one XCD (ids 8 apart), whose L2 then holds its rows while the token blocks go by
    const int hp = (int)blockIdx.x % (2 * heads), tb = (int)blockIdx.x / (2 * heads), h = hp % heads, part = hp / heads;
    const uint8_t *wf = wfrags + ((size_t)(h0 + h) * 2 + part) * (S16_LKV / 16) * 8 * S16_FRAG;
    uint8_t *out = ws + ((size_t)h * stride + tile0) * S16_KV_TILE;
    cf += (size_t)tile0 * (S16_LKV / 16) * 2 * S16_FRAG;
    const float f = fac[2 * (h0 + h) + part].x;
    if (part) s16_expand_workgroup<true>(wf, cf, f, n_tiles, tb, out, lds);
    else s16_expand_workgroup<false>(wf, cf, f, n_tiles, tb, out, lds);
}

// ---- attention ----------------------------------------------------------------------------------------------------------------
struct S16Attention {
    const float *q;            // token t's head h at q + t * q_stride + h * q_head: 128 elements (latent: and 64 rotated ones)
    int q_stride, q_head;
    const uint8_t *kv;         // [kv head][tile]{K, V}
    const S16Tile *info;       // latent: [tile], of the rope keys; else [kv head][tile]
    const float2 *fac;         // latent: of this call's first head, [head][2]
    const uint8_t *rope;       // latent: [tile]
    float *out;                // [t][out_stride], head h at h * 128
    int out_stride;
    int T, pos0, n_tiles;      // tokens of the step at positions pos0 .., tiles that a head's lie apart
    int heads, group;          // query heads of this call; how many of them share a KV head (latent: 1)
    int blocks;                // token blocks
    float scale_log2e;         // the softmax scale times log2(e)
};

// Four waves; a wave owns 32 tokens of one query head, whose scaled queries stay in registers.  LATENT: 128 tokens of one
// head a workgroup; else WH = 1, 2 or 4 heads of a KV head x 4 / WH runs of 32 tokens.  Key tiles pass through two LDS
// buffers (80 KB or 64 KB: two workgroups a compute unit).
template <bool LATENT, int WH>
__global__ __launch_bounds__(256, 2) void s16_attention(S16Attention a) {
    constexpr int STAGE = S16_KV_TILE + (LATENT ? S16_ROPE_TILE : 0), KN = 8, KR = LATENT ? 4 : 0, TB = 32 * (4 / WH);
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * STAGE];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 31, hf = lane >> 5;
    // Workgroup ids 8 apart share an XCD: the token blocks of a KV head (8 or a multiple of 8 of them) read its tiles into
    // one L2.  Of the blocks, the first half of the grid takes the long ones downwards and the second half the short ones
    // upwards, so that the two workgroups a compute unit holds walk about the same number of tiles together.
    const int sets = LATENT ? a.heads : a.heads / WH, set = (int)blockIdx.x % sets, bi = (int)blockIdx.x / sets;
    const int half = (a.blocks + 1) / 2, block = bi < half ? a.blocks - 1 - bi : bi - half;
    const int head = LATENT ? set : set * WH + wave % WH, kvh = LATENT ? set : set * WH / a.group;
    const int t0 = block * TB, tw = t0 + 32 * (wave / WH);               // first token of the workgroup and of the wave
    const int last = a.pos0 + min(t0 + TB, a.T) - 1, n_tiles = last / S16_TILE + 1;
    const int mine = a.pos0 + min(tw + 31, a.T - 1), my_key = a.pos0 + tw + n;  // the wave's and the lane's last key
    const bool idle = tw >= a.T;

    const uint8_t *kv = a.kv + (size_t)kvh * a.n_tiles * S16_KV_TILE + 1024 * wave + 16 * lane, *rope = a.rope + 1024 * wave + 16 * lane;
    const uint32_t lds0 = s16_lds_offset(lds) + 1024 * wave;
    auto issue = [&](int tile, int buf) __attribute__((always_inline)) {
        const uint32_t base = lds0 + buf * STAGE;
#pragma unroll
        for (int i = 0; i < S16_KV_TILE / 4096; i++) s16_copy16(kv + (size_t)tile * S16_KV_TILE + 4096 * i, base + 4096 * i);
        if constexpr (LATENT) {
#pragma unroll
            for (int i = 0; i < S16_ROPE_TILE / 4096; i++)
                s16_copy16(rope + (size_t)tile * S16_ROPE_TILE + 4096 * i, base + S16_KV_TILE + 4096 * i);
        }
    };
    // this lane's query (row tw + n; past the step: its last token) as second operands; the order of the inner index is the
    // keys': of a latent head's 128, element (hf, i) of k-step s is 16 s + 8 (i / 4) + 4 hf + i % 4, else 16 s + 8 hf + i
    s16_h8 qh[KN + KR], ql[KN + KR];
    float qinv, rinv = 0.0f;
    {
        const float *qp = a.q + (size_t)min(tw + n, a.T - 1) * a.q_stride + (size_t)head * a.q_head;
        auto part = [&](auto at, int first, int steps) __attribute__((always_inline)) {
            uint32_t m = 0;
            float x[8][8];
#pragma unroll
            for (int s = 0; s < 8; s++) {
                if (s >= steps) break;
#pragma unroll
                for (int i = 0; i < 8; i += 4) {
                    const float4 v = *(const float4 *)(qp + at(s, i));
                    x[s][i] = v.x, x[s][i + 1] = v.y, x[s][i + 2] = v.z, x[s][i + 3] = v.w;
                }
#pragma unroll
                for (int i = 0; i < 8; i++) m = max(m, s16_abs(x[s][i]));
            }
            m = max(m, (uint32_t)__shfl_xor((int)m, 32, 64));
            const int e = s16_exponent(m);
            const float f = s16_pow2(e);
#pragma unroll
            for (int s = 0; s < 8; s++) {
                if (s >= steps) break;
#pragma unroll
                for (int i = 0; i < 8; i++) x[s][i] *= f;
                s16_split(x[s], qh[first + s], ql[first + s]);
            }
            return s16_pow2(-e);
        };
        if constexpr (LATENT) {
            qinv = part([&](int s, int i) { return 16 * s + 2 * i + 4 * hf; }, KR, KN);
            rinv = part([&](int s, int i) { return 128 + 16 * s + 8 * hf + i; }, 0, 4);
        } else {
            qinv = part([&](int s, int i) { return 16 * s + 8 * hf + i; }, 0, KN);
        }
    }
    s16_f16 o[4];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[t][r] = 0.0f;
    bool spoilt = false;                    // the query sees a key that is not finite
    float m_run = -INFINITY, l_run = 0.0f;  // of the lane's query; the sum over this lane's keys only
    float vref = LATENT ? a.fac[2 * head + 1].y : s16_pow2(-126);  // the scale the outputs are held in: the largest inv.y so far
    const float khead = LATENT ? a.fac[2 * head].y : 1.0f;

    // what is known of the tile, asked for with the tile
    float kinv = 0.0f, vinv = vref;
    uint32_t bad = 0;
    auto scales = [&](int tile) __attribute__((always_inline)) {
        const S16Tile v = a.info[(LATENT ? 0 : (size_t)kvh * a.n_tiles) + tile];
        kinv = v.k, vinv = v.v, bad = v.bad;
    };
    issue(0, 0);
    scales(0);
    for (int tile = 0; tile < n_tiles; tile++) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        // (the compiler waits for the scales where they are first read: here, and not behind the loads issued next)
        asm volatile("" : "+v"(kinv), "+v"(vinv), "+v"(bad));
        const float k_now = kinv, v_now = vinv;
        const uint32_t bad_now = (uint32_t)__builtin_amdgcn_readfirstlane((int)bad);
        __syncthreads();  // the tile has landed, and the other buffer's readers are done
        if (tile + 1 < n_tiles) issue(tile + 1, (tile + 1) & 1), scales(tile + 1);
        if (idle || tile * S16_TILE > mine) continue;  // (the whole wave; the barrier above is met all the same)
        const uint8_t *l = lds + (tile & 1) * STAGE + 16 * lane;
        // scores in units of log2(e): the products of the rope part (latent) and of the head's 128 elements each behind a factor of
        // their own, since that of one side has no bound in units of the other's (a head without keys, a query of zeros)
        auto products = [&](const uint8_t *keys, int first, int steps, s16_f16 &sc) __attribute__((always_inline)) {
            // (latent: the products with a low plane in a sum of their own, for the roundings)
            s16_f16 low;
#pragma unroll
            for (int r = 0; r < 16; r++) sc[r] = low[r] = 0.0f;
            // Zeros that the compiler does not see as such: into a matrix instruction with a constant third operand it puts a
            // 16-register result over the first operand's registers, which the instruction still reads.
            if constexpr (LATENT) asm volatile("" : "+v"(low));
#pragma unroll
            for (int s = 0; s < KN; s++) {
                if (s >= steps) break;
                const s16_h8 kh = *(const s16_h8 *)(keys + (2 * s) * S16_FRAG), kl = *(const s16_h8 *)(keys + (2 * s + 1) * S16_FRAG);
                sc = s16_mma(kh, qh[first + s], sc);
                s16_f16 &to = LATENT ? low : sc;
                to = s16_mma(kh, ql[first + s], to);
                to = s16_mma(kl, qh[first + s], to);
            }
            if constexpr (LATENT) {
#pragma unroll
                for (int r = 0; r < 16; r++) sc[r] += low[r];
            }
        };
        s16_f16 sc;
        if constexpr (LATENT) {
            s16_f16 sr;
            products(l + S16_KV_TILE, 0, KR, sr);
            const float fr = rinv * k_now * a.scale_log2e;
#pragma unroll
            for (int r = 0; r < 16; r++) sr[r] *= fr;
            products(l, KR, KN, sc);
            const float f = qinv * khead * a.scale_log2e;
#pragma unroll
            for (int r = 0; r < 16; r++) sc[r] = fmaf(sc[r], f, sr[r]);
        } else {
            products(l, 0, KN, sc);
            const float f = qinv * k_now * a.scale_log2e;
#pragma unroll
            for (int r = 0; r < 16; r++) sc[r] *= f;
        }
        if (bad_now) {
            const int seen = my_key - tile * S16_TILE;  // the tile's last key that the lane's query sees
            spoilt |= (bad_now & (seen < 0 ? 0u : 0xFFFFFFFFu >> (31 - min(seen, 31)))) != 0;
        }
        const bool edge = tile * S16_TILE + 31 > a.pos0 + tw;  // some query of the wave does not see the whole tile
        float tmax = -INFINITY;
        if (edge) {
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (tile * S16_TILE + 8 * (r >> 2) + 4 * hf + (r & 3) > my_key) sc[r] = -INFINITY;
        }
#pragma unroll
        for (int r = 0; r < 16; r++) tmax = fmaxf(tmax, sc[r]);
        tmax = max_xor32(tmax);
        const float mnew = fmaxf(m_run, tmax);  // finite from tile 0 on, whose first key every query sees
        const float vnew = LATENT ? vref : fmaxf(vref, v_now);
        float keep = __builtin_amdgcn_exp2f(m_run - mnew);
        l_run *= keep;
        keep *= vref / vnew;
        if (__any(keep != 1.0f)) {
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[t][r] *= keep;
        }
        m_run = mnew, vref = vnew;
        // weights times 2^10 (and the tile's share of vref, both powers of two): the small ones keep their bits in f16
        const float up = LATENT ? 1.0f : v_now / vnew;
        s16_h8 ph[2], pl[2];
        float psum = 0.0f;
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            float p[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                p[i] = __builtin_amdgcn_exp2f(sc[8 * ks + i] + (10.0f - mnew));  // (a masked key: 0)
                psum += p[i];
                if constexpr (!LATENT) p[i] *= up;
            }
            s16_split(p, ph[ks], pl[ks]);
        }
        l_run += psum;
        const uint8_t *lv = l + S16_KV_TILE / 2;
#pragma unroll
        for (int ks = 0; ks < 2; ks++)
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const s16_h8 vh = *(const s16_h8 *)(lv + (4 * t + 2 * ks) * S16_FRAG), vl = *(const s16_h8 *)(lv + (4 * t + 2 * ks + 1) * S16_FRAG);
                o[t] = s16_mma(vh, ph[ks], o[t]);
                o[t] = s16_mma(vh, pl[ks], o[t]);
                o[t] = s16_mma(vl, ph[ks], o[t]);
            }
    }
    if (tw + n >= a.T) return;
    const float inv = spoilt ? __builtin_nanf("") : vref / sum_xor32(l_run);
    float *op = a.out + (size_t)(tw + n) * a.out_stride + (size_t)head * 128;
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int b = 0; b < 4; b++)
            *(float4 *)(op + 32 * t + 8 * b + 4 * hf) = float4{o[t][4 * b] * inv, o[t][4 * b + 1] * inv, o[t][4 * b + 2] * inv, o[t][4 * b + 3] * inv};
}

}  // namespace jq

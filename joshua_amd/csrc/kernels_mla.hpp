// Multi-head latent attention (DeepSeek-V2 / V3 / Kimi-K2) in its absorbed form, f32 throughout.
//
// The reference (src/quantized_deepseek2.rs:422-499) expands every new token's latent through the KV
// up-projection into per-head keys and values and caches those: n_head * (qk_nope + qk_rope +
// v_head_dim) floats a token (160 KB at V3 size), all of which a decode step reads back.  The same
// numbers come out of the latent itself: with W_k[h] (qk_nope x kv_lora_rank) and W_v[h] (v_head_dim x
// kv_lora_rank) the rows of the up-projection for head h,
//     q_nope[h] . (W_k[h] c_t)  =  (W_k[h]^T q_nope[h]) . c_t
//     sum_t p_t (W_v[h] c_t)    =  W_v[h] (sum_t p_t c_t)
// so the cache holds, per token, the normed latent c_t (kv_lora_rank) and the rotated shared key k_pe
// (qk_rope): 2.3 KB at V3 size, shared by all heads.  A step is
//   mla_rope_latent   rotate q_pe in place; norm the latent, rotate k_pe, append both to the cache
//   mla_absorb_q      q_abs[h] = W_k[h]^T q_nope[h]
//   mla_attention     scores over the cached latents, running softmax, o_lat[h] = sum p_t c_t, the
//                     context split over workgroups (partial maximum, sum and vector per split)
//   mla_merge         merge the splits into o_lat[h]
//   mla_vproj         ctx[h] = W_v[h] o_lat[h]
// (one token over a Q4_K up-projection: mla_step_q4k, behind a long context mla_absorb_rope_q4k, the attention, mla_merge_vproj_q4k)
// around the quantized projections (q, kv_a, o), which run on the matmul kernels.
#pragma once
#include "kernels_graph.hpp"

namespace jq {

// A wave for (bx <= n_head, token s).  Waves bx < n_head rotate the rope slice of q[s, bx] in place
// (neighbouring pairs (2i, 2i+1), candle's rope_i; cs[p][i] = (cos, sin) of position p, pair i, already
// scaled by the YaRN mscale; reference :302-311).  Wave bx == n_head norms the latent
// comp[s, 0:lkv] (RMSNorm, weight w) into lat[pos0 + s] and rotates comp[s, lkv:] into kpe[pos0 + s]; a token's row of comp
// starts comp_stride floats after the one before.
__device__ __forceinline__ void mla_rope_latent_wave(float *__restrict__ q, const float *__restrict__ comp,
                                                     const float *__restrict__ w, const float2 *__restrict__ cs,
                                                     float *__restrict__ lat, float *__restrict__ kpe, int n_head,
                                                     int nope, int rope, int lkv, int pos0, float eps, int bx, int s,
                                                     int lane, int comp_stride = 0) {
    const int half = rope >> 1;
    const float2 *c = cs + (size_t)(pos0 + s) * half;
    if (bx < n_head) {
        float *v = q + ((size_t)s * n_head + bx) * (nope + rope) + nope;
        for (int i = lane; i < half; i += 64) {
            const float a = v[2 * i], b = v[2 * i + 1];
            v[2 * i] = a * c[i].x - b * c[i].y;
            v[2 * i + 1] = a * c[i].y + b * c[i].x;
        }
        return;
    }
    const float *x = comp + (size_t)s * comp_stride;
    float ss = 0.0f;
    for (int i = lane; i < lkv; i += 64) ss = fmaf(x[i], x[i], ss);
    ss = wave_sum(ss);
    const float inv = 1.0f / sqrtf(ss / (float)lkv + eps);
    float *l = lat + (size_t)(pos0 + s) * lkv, *k = kpe + (size_t)(pos0 + s) * rope;
    for (int i = lane; i < lkv; i += 64) l[i] = x[i] * inv * w[i];
    for (int i = lane; i < half; i += 64) {
        const float a = x[lkv + 2 * i], b = x[lkv + 2 * i + 1];
        k[2 * i] = a * c[i].x - b * c[i].y;
        k[2 * i + 1] = a * c[i].y + b * c[i].x;
    }
}

// The same for S tokens: grid (S, ceil(n_head / MLA_ROPE_HEADS) + 1), 256 threads.  Workgroup (s, y) rotates the heads from
// MLA_ROPE_HEADS y on, a thread their pairs 256 apart; those of the last y take four tokens' latents, a wave each.  (A wave a
// head and token, 66 000 workgroups for 512 tokens of 128 heads, took the launcher 21.7 us; this 11.7.)
constexpr int MLA_ROPE_HEADS = 32;
__global__ __launch_bounds__(256) void mla_rope_latent(float *__restrict__ q, const float *__restrict__ comp,
                                                        const float *__restrict__ w, const float2 *__restrict__ cs,
                                                        float *__restrict__ lat, float *__restrict__ kpe, int n_head,
                                                        int nope, int rope, int lkv, int pos0, float eps, int S, int comp_stride) {
    if (blockIdx.y + 1 == gridDim.y) {
        const int s = 4 * (int)blockIdx.x + (int)(threadIdx.x >> 6);
        if (s < S) mla_rope_latent_wave(q, comp, w, cs, lat, kpe, n_head, nope, rope, lkv, pos0, eps, n_head, s, (int)threadIdx.x & 63, comp_stride);
        return;
    }
    const int s = (int)blockIdx.x, h0 = MLA_ROPE_HEADS * (int)blockIdx.y, half = rope >> 1, pairs = min(MLA_ROPE_HEADS, n_head - h0) * half;
    const float2 *c = cs + (size_t)(pos0 + s) * half;
    float *v = q + ((size_t)s * n_head + h0) * (nope + rope) + nope;
#pragma unroll 4
    for (int e = threadIdx.x; e < pairs; e += 256) {
        const int h = e / half, i = e - h * half;
        float *p = v + (size_t)h * (nope + rope) + 2 * i;
        const float a = p[0], b = p[1];
        const float2 r = c[i];
        p[0] = a * r.x - b * r.y;
        p[1] = a * r.y + b * r.x;
    }
}

// q_abs[s, h, c] = sum_r q[s, h, r] * Wkv[h * (nope + vh) + r, c], r < nope.  grid (n_head, ceil(S / ST)),
// 512 threads: thread (row quarter, column group of CW) walks a quarter of the head's nope rows (the
// rows are read coalesced, once per ST tokens, whose query values wait in LDS); the four quarters sum
// through LDS.  CW = 4 (16-byte loads) needs lkv % 4 == 0 and lkv <= 512; CW = 1 any lkv <= 128.
constexpr int MLA_MAX_NOPE = 256, MLA_MAX_LKV = 512;
template <int ST, int CW>
__device__ __forceinline__ void mla_absorb_q_workgroup(const float *__restrict__ q, const float *__restrict__ Wkv,
                                                       float *__restrict__ qabs, int S, int n_head, int nope, int rope,
                                                       int vh, int lkv, int h, int s0) {
    __shared__ float qs[MLA_MAX_NOPE][ST];
    __shared__ float red[3][ST][128 * CW];
    const int qd = nope + rope;
    for (int e = threadIdx.x; e < nope * ST; e += 512) {
        const int r = e / ST, j = e % ST;
        qs[r][j] = s0 + j < S ? q[((size_t)(s0 + j) * n_head + h) * qd + r] : 0.0f;
    }
    __syncthreads();
    const float *W = Wkv + (size_t)h * (nope + vh) * lkv;
    const int part = threadIdx.x >> 7, c = (threadIdx.x & 127) * CW;
    const int r0 = part * ((nope + 3) >> 2), r1 = min(nope, r0 + ((nope + 3) >> 2));
    float acc[ST][CW];
#pragma unroll
    for (int j = 0; j < ST; j++)
#pragma unroll
        for (int i = 0; i < CW; i++) acc[j][i] = 0.0f;
    if (c < lkv) {
#pragma unroll 8
        for (int r = r0; r < r1; r++) {
            float wv[CW];
            if constexpr (CW == 4) {
                const float4 v = *(const float4 *)(W + (size_t)r * lkv + c);
                wv[0] = v.x, wv[1] = v.y, wv[2] = v.z, wv[3] = v.w;
            } else {
                wv[0] = W[(size_t)r * lkv + c];
            }
#pragma unroll
            for (int j = 0; j < ST; j++)
#pragma unroll
                for (int i = 0; i < CW; i++) acc[j][i] = fmaf(qs[r][j], wv[i], acc[j][i]);
        }
    }
    if (part > 0) {
#pragma unroll
        for (int j = 0; j < ST; j++)
#pragma unroll
            for (int i = 0; i < CW; i++) red[part - 1][j][c + i] = acc[j][i];
    }
    __syncthreads();
    if (part == 0 && c < lkv) {
#pragma unroll
        for (int j = 0; j < ST; j++)
#pragma unroll
            for (int i = 0; i < CW; i++) {
                const float v = acc[j][i] + red[0][j][c + i] + red[1][j][c + i] + red[2][j][c + i];
                if (s0 + j < S) qabs[((size_t)(s0 + j) * n_head + h) * lkv + c + i] = v;
            }
    }
}

template <int ST, int CW>
__global__ __launch_bounds__(512) void mla_absorb_q(const float *__restrict__ q, const float *__restrict__ Wkv,
                                                     float *__restrict__ qabs, int S, int n_head, int nope, int rope,
                                                     int vh, int lkv) {
    mla_absorb_q_workgroup<ST, CW>(q, Wkv, qabs, S, n_head, nope, rope, vh, lkv, (int)blockIdx.x, (int)blockIdx.y * ST);
}

// mla_rope_latent and mla_absorb_q of a single-token step as one launch: grid n_head + 1, 512 threads.  The
// first wave of workgroup x does what wave x of mla_rope_latent_wave does (it touches the rope slice of
// q[x], the absorption reads the other slice); workgroup n_head has nothing else to do.
template <int CW>
__global__ __launch_bounds__(512) void mla_absorb_rope(float *__restrict__ q, const float *__restrict__ Wkv,
                                                        float *__restrict__ qabs, int n_head, int nope, int rope, int vh,
                                                        int lkv, const float *__restrict__ comp, const float *__restrict__ w,
                                                        const float2 *__restrict__ cs, float *__restrict__ lat,
                                                        float *__restrict__ kpe, int pos0, float eps) {
    if (threadIdx.x < 64)
        mla_rope_latent_wave(q, comp, w, cs, lat, kpe, n_head, nope, rope, lkv, pos0, eps, (int)blockIdx.x, 0, (int)threadIdx.x);
    if ((int)blockIdx.x == n_head) return;
    mla_absorb_q_workgroup<1, CW>(q, Wkv, qabs, 1, n_head, nope, rope, vh, lkv, (int)blockIdx.x, 0);
}

// Scores, running softmax and the weighted latent sum for G heads of one query token over one split of
// its context.  grid (n_head / G, n_split, S), four waves; wave w takes tokens t0 + w, t0 + w + 4, ... of
// the split: a lane holds LPL consecutive latent elements (and one rope element) of the token, loaded
// once for the G heads, and the same elements of every head's absorbed query; a score is the wave sum
// of the products.  The four waves' (maximum, sum, vector) merge through LDS into
// part[s, h, split] = {m, l, o[lkv]}, unnormalised.  lkv <= 64 LPL, rope <= 64.  Query token s sees
// cache tokens 0 .. pos0 + s (the causal mask of the reference, :875-889).
constexpr int MLA_SPLIT_MAX = 64;
template <int G, int LPL>
__global__ __launch_bounds__(256) void mla_attention(const float *__restrict__ qabs, const float *__restrict__ q,
                                                      const float *__restrict__ lat, const float *__restrict__ kpe,
                                                      float *__restrict__ part, int n_head, int nope, int rope, int lkv,
                                                      int pos0, int n_split, float scale) {
    __shared__ float wm[4][G], wl[4][G];
    __shared__ float wo[4][G][64 * LPL];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int h0 = blockIdx.x * G, split = blockIdx.y, s = blockIdx.z;
    const int T = pos0 + s + 1, chunk = (T + n_split - 1) / n_split;
    const int t0 = split * chunk, t1 = min(T, t0 + chunk);
    const bool vec = lkv == 64 * LPL && LPL % 4 == 0;  // whole float4 loads
    const int e0 = lane * LPL;

    float qa[G][LPL], qp[G], m[G], l[G], o[G][LPL];
#pragma unroll
    for (int g = 0; g < G; g++) {
        const float *qv = qabs + ((size_t)s * n_head + h0 + g) * lkv;
#pragma unroll
        for (int i = 0; i < LPL; i++) qa[g][i] = e0 + i < lkv ? qv[e0 + i] : 0.0f, o[g][i] = 0.0f;
        qp[g] = lane < rope ? q[((size_t)s * n_head + h0 + g) * (nope + rope) + nope + lane] : 0.0f;
        m[g] = -INFINITY, l[g] = 0.0f;
    }
    for (int t = t0 + wave; t < t1; t += 4) {
        float c[LPL];
        const float *cv = lat + (size_t)t * lkv;
        bool loaded = false;
        if constexpr (LPL % 4 == 0) {
            if (vec) {
#pragma unroll
                for (int i = 0; i < LPL; i += 4) {
                    const float4 v = *(const float4 *)(cv + e0 + i);
                    c[i] = v.x, c[i + 1] = v.y, c[i + 2] = v.z, c[i + 3] = v.w;
                }
                loaded = true;
            }
        }
        if (!loaded) {
#pragma unroll
            for (int i = 0; i < LPL; i++) c[i] = e0 + i < lkv ? cv[e0 + i] : 0.0f;
        }
        const float kp = lane < rope ? kpe[(size_t)t * rope + lane] : 0.0f;
#pragma unroll
        for (int g = 0; g < G; g++) {
            float sc = qp[g] * kp;
#pragma unroll
            for (int i = 0; i < LPL; i++) sc = fmaf(qa[g][i], c[i], sc);
            sc = wave_sum(sc) * scale;
            const float mn = fmaxf(m[g], sc);
            const float a = __expf(m[g] - mn), p = __expf(sc - mn);  // the first token: a = exp(-inf) = 0
            l[g] = fmaf(l[g], a, p);
#pragma unroll
            for (int i = 0; i < LPL; i++) o[g][i] = fmaf(o[g][i], a, p * c[i]);
            m[g] = mn;
        }
    }
#pragma unroll
    for (int g = 0; g < G; g++) {
        if (lane == 0) wm[wave][g] = m[g], wl[wave][g] = l[g];
#pragma unroll
        for (int i = 0; i < LPL; i++) wo[wave][g][e0 + i] = o[g][i];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < G * 64 * LPL; e += 256) {
        const int g = e / (64 * LPL), i = e % (64 * LPL);
        const float M = fmaxf(fmaxf(wm[0][g], wm[1][g]), fmaxf(wm[2][g], wm[3][g]));
        float ov = 0.0f, lv = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const float f = wm[w][g] == -INFINITY ? 0.0f : __expf(wm[w][g] - M);  // a wave without tokens
            ov = fmaf(wo[w][g][i], f, ov);
            lv = fmaf(wl[w][g], f, lv);
        }
        float *p = part + (((size_t)s * n_head + h0 + g) * n_split + split) * (lkv + 2);
        if (i < lkv) p[2 + i] = ov;
        if (i == 0) p[0] = M, p[1] = lv;
    }
}

// The same scores and latent sums on the f32 matrix cores (v_mfma_f32_32x32x2_f32: exact f32 products,
// f32 sums), for the geometry every DeepSeek MLA model has: 512 latent + 64 rope elements, heads in
// groups of 32.  grid (n_head / 32, n_split, S), eight waves.  A tile is 32 heads x 32 tokens; the
// tokens' rows [latent | rope key] (576 floats) wait in LDS.
//   scores  = Q[32 x 576] . C^T[576 x 32]: wave w multiplies columns 72 w .. 72 w + 71 (36 steps of 2;
//             its slice of Q stays in 36 registers), the eight partial tiles sum through LDS;
//   softmax: 16 threads a head, two tokens each, running maximum and sum in registers;
//   o_lat  += P[32 x 32] . C[32 x 512]: wave w owns latent columns 64 w .. 64 w + 63 (two tiles of 32,
//             32 accumulator registers), 16 steps of 2 tokens.
// The next tile's rows are fetched into registers while a tile is worked on.  Output as mla_attention.
constexpr int MLA_M_LKV = 512, MLA_M_ROPE = 64, MLA_M_KT = MLA_M_LKV + MLA_M_ROPE, MLA_M_STRIDE = MLA_M_KT + 4;
typedef float mla_f16v __attribute__((ext_vector_type(16)));

__global__ __launch_bounds__(512) void mla_attention_mfma(const float *__restrict__ qabs, const float *__restrict__ q,
                                                           const float *__restrict__ lat, const float *__restrict__ kpe,
                                                           float *__restrict__ part, int n_head, int nope, int pos0,
                                                           int n_split, float scale) {
    __shared__ __attribute__((aligned(16))) float ct[32][MLA_M_STRIDE];
    __shared__ float sp[8][32][33];
    __shared__ float ps[32][33];
    __shared__ __attribute__((aligned(16))) float al[32];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 31, lk = lane >> 5;
    const int h0 = blockIdx.x * 32, split = blockIdx.y, s = blockIdx.z;
    const int T = pos0 + s + 1, chunk = (T + n_split - 1) / n_split;
    const int t0 = split * chunk, t1 = min(T, t0 + chunk);

    // 32 rows (tokens of a tile, or the heads' queries) x 144 pieces of 16 bytes (128 latent, 16 rope) = 9 a thread
    float4 pre[9];
    auto load_tile = [&](int tb) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 9; u++) {
            const int idx = tid + 512 * u, tok = idx / 144, f = idx % 144, t = tb + tok;
            if (t < t1) pre[u] = f < 128 ? *(const float4 *)(lat + (size_t)t * MLA_M_LKV + 4 * f)
                                         : *(const float4 *)(kpe + (size_t)t * MLA_M_ROPE + 4 * (f - 128));
            else pre[u] = float4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    };
    if (t0 < t1) load_tile(t0);
    // this wave's slice of the 32 heads' queries, element 72 wave + 2 ks + lk of head li, by way of LDS
    // (rows [absorbed query | rotated rope query] read whole, then picked apart)
    float qreg[36];
    {
#pragma unroll
        for (int u = 0; u < 9; u++) {
            const int idx = tid + 512 * u, i = idx / 144, f = idx % 144;
            const size_t row = (size_t)s * n_head + h0 + i;
            *(float4 *)&ct[i][4 * f] = f < 128 ? *(const float4 *)(qabs + row * MLA_M_LKV + 4 * f)
                                               : *(const float4 *)(q + row * (nope + MLA_M_ROPE) + nope + 4 * (f - 128));
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < 36; ks++) qreg[ks] = ct[li][72 * wave + 2 * ks + lk];
        __syncthreads();
    }
    mla_f16v o[2];
#pragma unroll
    for (int nt = 0; nt < 2; nt++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[nt][r] = 0.0f;
    float m_run = -INFINITY, l_run = 0.0f;  // of head tid / 16, the same in its 16 threads

    for (int tb = t0; tb < t1; tb += 32) {
        if (tb > t0) __syncthreads();  // every wave is done with the rows of the tile before
#pragma unroll
        for (int u = 0; u < 9; u++) {
            const int idx = tid + 512 * u, tok = idx / 144, f = idx % 144;
            *(float4 *)&ct[tok][4 * f] = pre[u];
        }
        __syncthreads();
        if (tb + 32 < t1) load_tile(tb + 32);

        mla_f16v sc;
#pragma unroll
        for (int r = 0; r < 16; r++) sc[r] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < 36; ks++)
            sc = __builtin_amdgcn_mfma_f32_32x32x2f32(qreg[ks], ct[li][72 * wave + 2 * ks + lk], sc, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; r++) sp[wave][8 * (r >> 2) + 4 * lk + (r & 3)][li] = sc[r];  // row = head, column = token
        __syncthreads();
        {
            const int i = tid >> 4, j = 2 * (tid & 15);
            float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
            for (int w = 0; w < 8; w++) s0 += sp[w][i][j], s1 += sp[w][i][j + 1];
            s0 = tb + j < t1 ? s0 * scale : -INFINITY;
            s1 = tb + j + 1 < t1 ? s1 * scale : -INFINITY;
            const float mn = fmaxf(m_run, max_row16(fmaxf(s0, s1)));  // finite: token tb is inside the split
            const float p0 = __expf(s0 - mn), p1 = __expf(s1 - mn), a = __expf(m_run - mn);
            l_run = fmaf(l_run, a, sum_row16(p0 + p1));
            m_run = mn;
            ps[i][j] = p0, ps[i][j + 1] = p1;
            if ((tid & 15) == 0) al[i] = a;
        }
        __syncthreads();
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const float4 a = *(const float4 *)&al[8 * b + 4 * lk];
#pragma unroll
            for (int nt = 0; nt < 2; nt++) o[nt][4 * b] *= a.x, o[nt][4 * b + 1] *= a.y, o[nt][4 * b + 2] *= a.z, o[nt][4 * b + 3] *= a.w;
        }
#pragma unroll
        for (int kk = 0; kk < 16; kk++) {
            const float pa = ps[li][2 * kk + lk];
#pragma unroll
            for (int nt = 0; nt < 2; nt++)
                o[nt] = __builtin_amdgcn_mfma_f32_32x32x2f32(pa, ct[2 * kk + lk][64 * wave + 32 * nt + li], o[nt], 0, 0, 0);
        }
    }
#pragma unroll
    for (int nt = 0; nt < 2; nt++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int i = 8 * (r >> 2) + 4 * lk + (r & 3);
            part[(((size_t)s * n_head + h0 + i) * n_split + split) * (MLA_M_LKV + 2) + 2 + 64 * wave + 32 * nt + li] = o[nt][r];
        }
    if ((tid & 15) == 0) {
        float *p = part + (((size_t)s * n_head + h0 + (tid >> 4)) * n_split + split) * (MLA_M_LKV + 2);
        p[0] = m_run, p[1] = l_run;
    }
}

// One token over a short context, 512 latent + 64 rope elements: a wave takes two heads and 16 cached tokens, whose rows it holds
// in registers (a lane 8 latent elements and one rope element of each), so nothing waits for LDS or another wave; grid (n_head / 8,
// n_split = ceil(context / 16)), four waves.  f32 throughout, output as mla_attention.  Bound: one trip to memory and the
// launch: a layer's step of 128 heads behind 100 tokens 46.5 us where the matrix-core kernel, with its rows and sums going through
// LDS between barriers on 16 compute units, makes it 52.3.
constexpr int MLA_SHORT_TOKENS = 16;
__global__ __launch_bounds__(256) void mla_attention_short(const float *__restrict__ qabs, const float *__restrict__ q,
                                                            const float *__restrict__ lat, const float *__restrict__ kpe,
                                                            float *__restrict__ part, int nope, int T, int n_split, float scale) {
    constexpr int H = 2, N = MLA_SHORT_TOKENS;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, h0 = ((int)blockIdx.x * 4 + wave) * H, split = blockIdx.y;
    const int t0 = split * N, cnt = min(N, T - t0);
    float4 qa[H][2], c[N][2];
    float qp[H], kp[N];
#pragma unroll
    for (int h = 0; h < H; h++) {
        const float4 *src = (const float4 *)(qabs + (size_t)(h0 + h) * MLA_M_LKV + 8 * lane);
        qa[h][0] = src[0], qa[h][1] = src[1];
        qp[h] = q[(size_t)(h0 + h) * (nope + MLA_M_ROPE) + nope + lane];
    }
#pragma unroll
    for (int t = 0; t < N; t++) {
        const size_t at = (size_t)min(t0 + t, T - 1);
        const float4 *src = (const float4 *)(lat + at * MLA_M_LKV + 8 * lane);
        c[t][0] = src[0], c[t][1] = src[1];
        kp[t] = kpe[at * MLA_M_ROPE + lane];
    }
#pragma unroll
    for (int h = 0; h < H; h++) {
        float s[N], m = -INFINITY, l = 0.0f;
#pragma unroll
        for (int t = 0; t < N; t++) {
            float v = qp[h] * kp[t];
            v = fmaf(qa[h][0].x, c[t][0].x, fmaf(qa[h][0].y, c[t][0].y, fmaf(qa[h][0].z, c[t][0].z, fmaf(qa[h][0].w, c[t][0].w, v))));
            v = fmaf(qa[h][1].x, c[t][1].x, fmaf(qa[h][1].y, c[t][1].y, fmaf(qa[h][1].z, c[t][1].z, fmaf(qa[h][1].w, c[t][1].w, v))));
            s[t] = wave_sum(v) * scale;
            if (t < cnt) m = fmaxf(m, s[t]);
        }
        float4 o[2] = {float4{0.0f, 0.0f, 0.0f, 0.0f}, float4{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
        for (int t = 0; t < N; t++) {
            const float p = t < cnt ? __expf(s[t] - m) : 0.0f;
            l += p;
#pragma unroll
            for (int i = 0; i < 2; i++) {
                o[i].x = fmaf(p, c[t][i].x, o[i].x), o[i].y = fmaf(p, c[t][i].y, o[i].y);
                o[i].z = fmaf(p, c[t][i].z, o[i].z), o[i].w = fmaf(p, c[t][i].w, o[i].w);
            }
        }
        float *dst = part + ((size_t)(h0 + h) * n_split + split) * (MLA_M_LKV + 2);
        if (lane == 0) dst[0] = m, dst[1] = l;
        const float v[8] = {o[0].x, o[0].y, o[0].z, o[0].w, o[1].x, o[1].y, o[1].z, o[1].w};
#pragma unroll
        for (int i = 0; i < 8; i += 2) *(float2 *)(dst + 2 + 8 * lane + i) = float2{v[i], v[i + 1]};
    }
}

// grid (n_head, S, ceil(lkv / 128)), 128 threads, one latent column each: merges the splits of (s, h)
// into the normalised latent sum olat[s, h, :] = sum_i f_i o_i / sum_i f_i l_i, f_i = exp(m_i - max m).
__global__ __launch_bounds__(128) void mla_merge(const float *__restrict__ part, float *__restrict__ olat, int n_head,
                                                  int lkv, int n_split) {
    __shared__ float f[MLA_SPLIT_MAX];
    __shared__ float Linv;
    const int h = blockIdx.x, s = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const float *p = part + ((size_t)s * n_head + h) * n_split * (lkv + 2);
    if (wave == 0) {  // n_split <= 64
        const float mi = lane < n_split ? p[(size_t)lane * (lkv + 2)] : -INFINITY;
        const float M = wave_max(mi);
        const float fi = mi == -INFINITY ? 0.0f : __expf(mi - M);  // an empty split
        const float L = wave_sum(lane < n_split ? p[(size_t)lane * (lkv + 2) + 1] * fi : 0.0f);
        f[lane] = fi;
        if (lane == 0) Linv = 1.0f / L;
    }
    __syncthreads();
    const int c = blockIdx.z * 128 + threadIdx.x;
    if (c >= lkv) return;
    float v = 0.0f;
#pragma unroll 8
    for (int i = 0; i < n_split; i++) v = fmaf(p[(size_t)i * (lkv + 2) + 2 + c], f[i], v);
    olat[((size_t)s * n_head + h) * lkv + c] = v * Linv;
}

// ctx[s, h * vh + j] = Wkv[h * (nope + vh) + nope + j, :] . olat[s, h, :].  grid (n_head, ceil(vh / 16),
// ceil(S / ST)), four waves: a wave takes four value rows, read coalesced (16-byte loads when VEC:
// lkv % 4 == 0) once for the ST tokens whose latent sums wait in LDS.
template <int ST, bool VEC>
__global__ __launch_bounds__(256) void mla_vproj(const float *__restrict__ olat, const float *__restrict__ Wkv,
                                                  float *__restrict__ ctx, int S, int n_head, int nope, int vh, int lkv) {
    __shared__ __attribute__((aligned(16))) float ol[ST][MLA_MAX_LKV];
    const int h = blockIdx.x, s0 = blockIdx.z * ST, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int e = threadIdx.x; e < ST * lkv; e += 256) {
        const int j = e / lkv, c = e % lkv;
        ol[j][c] = s0 + j < S ? olat[((size_t)(s0 + j) * n_head + h) * lkv + c] : 0.0f;
    }
    __syncthreads();
    const float *W = Wkv + ((size_t)h * (nope + vh) + nope) * lkv;
#pragma unroll
    for (int rr = 0; rr < 4; rr++) {
        const int j = blockIdx.y * 16 + wave * 4 + rr;
        if (j >= vh) break;  // the whole wave
        float acc[ST];
#pragma unroll
        for (int t = 0; t < ST; t++) acc[t] = 0.0f;
        if constexpr (VEC) {
            for (int c = 4 * lane; c < lkv; c += 256) {
                const float4 wv = *(const float4 *)(W + (size_t)j * lkv + c);
#pragma unroll
                for (int t = 0; t < ST; t++) {
                    const float4 o = *(const float4 *)&ol[t][c];
                    acc[t] = fmaf(wv.x, o.x, fmaf(wv.y, o.y, fmaf(wv.z, o.z, fmaf(wv.w, o.w, acc[t]))));
                }
            }
        } else {
            for (int c = lane; c < lkv; c += 64) {
                const float wv = W[(size_t)j * lkv + c];
#pragma unroll
                for (int t = 0; t < ST; t++) acc[t] = fmaf(wv, ol[t][c], acc[t]);
            }
        }
#pragma unroll
        for (int t = 0; t < ST; t++) {
            const float v = wave_sum(acc[t]);
            if (lane == 0 && s0 + t < S) ctx[((size_t)(s0 + t) * n_head + h) * vh + j] = v;
        }
    }
}

// ---- one token over a Q4_K up-projection: its blocks (288 bytes a row of 512) read instead of the 2 KB of f32 a row --------
//
// Lane l of a half-wave holds the same 8 columns of a super-block for every row: the nibbles of word l of its 32, columns
// 64 c + 4 i .. + 3 (low) and 64 c + 32 + 4 i .. + 3 (high) with c = l / 8, i = l % 8; weights as decoded for the f32 copy,
// w = d sc q - dmin m, with the offsets' products summed apart.
struct MlaQ4kWord {
    float lo[4], hi[4];      // q of the eight
    float dl, dh, ml, mh;    // d sc and dmin m of the two sub-blocks
};
__device__ __forceinline__ MlaQ4kWord mla_q4k_word(const uint4 &hdr, uint32_t q, int c) {
    MlaQ4kWord w;
    uint32_t sc, mn;
    q4k_scale_min_pair(hdr.y, hdr.z, hdr.w, c, sc, mn);
    const float d = f16_bits(hdr.x), dmin = f16_bits(hdr.x >> 16);
    w.dl = d * (float)(sc & 0xFFu), w.dh = d * (float)((sc >> 8) & 0xFFu);
    w.ml = dmin * (float)(mn & 0xFFu), w.mh = dmin * (float)((mn >> 8) & 0xFFu);
    const uint32_t lo = q & 0x0F0F0F0Fu, hi = (q >> 4) & 0x0F0F0F0Fu;
#pragma unroll
    for (int b = 0; b < 4; b++) w.lo[b] = (float)((lo >> (8 * b)) & 0xFFu), w.hi[b] = (float)((hi >> (8 * b)) & 0xFFu);
    return w;
}

// mla_absorb_rope over Q4_K blocks: grid (n_head + 1, lkv / 256 super-blocks), 512 threads.  A half-wave takes every 16th of the
// head's nope rows; their 16 sums meet in LDS.  Bound: latency of the rows' loads, all asked for ahead of the arithmetic.
// 128 heads of 128 x 512: 5.4 us (the f32 rows, 33.5 MB: 7.1).
template <int ROWS>  // rows a half-wave, nope / 16
__global__ __launch_bounds__(512) void mla_absorb_rope_q4k(float *__restrict__ q, const uint8_t *__restrict__ Wkv,
                                                            float *__restrict__ qabs, int n_head, int nope, int rope, int vh,
                                                            int lkv, const float *__restrict__ comp, const float *__restrict__ w,
                                                            const float2 *__restrict__ cs, float *__restrict__ lat,
                                                            float *__restrict__ kpe, int pos0, float eps) {
    __shared__ float red[16][256];
    const int h = blockIdx.x, sb = blockIdx.y, tid = threadIdx.x, half = tid >> 5, l = tid & 31, c = l >> 3, nb = lkv / 256;
    if (h == n_head) {
        if (sb == 0 && tid < 64)
            mla_rope_latent_wave(q, comp, w, cs, lat, kpe, n_head, nope, rope, lkv, pos0, eps, h, 0, tid);
        return;
    }
    const uint8_t *src = Wkv + (((size_t)h * (nope + vh) + half) * nb + sb) * 144;
    const size_t step = (size_t)16 * nb * 144;
    uint4 hdr[ROWS];
    uint32_t qs[ROWS];
    float x[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; i++) {
        hdr[i] = *(const uint4 *)(src + i * step);
        qs[i] = *(const uint32_t *)(src + i * step + 16 + 4 * l);
        x[i] = q[(size_t)h * (nope + rope) + half + 16 * i];
    }
    float lo[4] = {0.0f, 0.0f, 0.0f, 0.0f}, hi[4] = {0.0f, 0.0f, 0.0f, 0.0f}, ml = 0.0f, mh = 0.0f;
#pragma unroll
    for (int i = 0; i < ROWS; i++) {
        const MlaQ4kWord v = mla_q4k_word(hdr[i], qs[i], c);
        const float a = x[i] * v.dl, b = x[i] * v.dh;
#pragma unroll
        for (int e = 0; e < 4; e++) lo[e] = fmaf(a, v.lo[e], lo[e]), hi[e] = fmaf(b, v.hi[e], hi[e]);
        ml = fmaf(x[i], v.ml, ml), mh = fmaf(x[i], v.mh, mh);
    }
    const int at = 64 * c + 4 * (l & 7);
    *(float4 *)&red[half][at] = float4{lo[0] - ml, lo[1] - ml, lo[2] - ml, lo[3] - ml};
    *(float4 *)&red[half][at + 32] = float4{hi[0] - mh, hi[1] - mh, hi[2] - mh, hi[3] - mh};
    __syncthreads();
    if (tid < 256) {
        float v = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; i++) v += red[i][tid];
        qabs[(size_t)h * lkv + 256 * sb + tid] = v;
    } else if (sb == 0 && tid < 320) {  // (the rope slice of q[h]: nobody reads it here)
        mla_rope_latent_wave(q, comp, w, cs, lat, kpe, n_head, nope, rope, lkv, pos0, eps, h, 0, tid - 256);
    }
}

// mla_merge and mla_vproj of one token in one launch, over Q4_K blocks of 512 columns: grid (n_head, vh / 64), 512 threads.  A
// workgroup merges the splits of its head (a thread a column), then wave w takes 8 value rows, a lane its 8 columns of either
// super-block.  128 heads of 128 x 512 behind 100 tokens: 6.1 us (merging 4.8 and the f32 rows 8.0).
__global__ __launch_bounds__(512) void mla_merge_vproj_q4k(const float *__restrict__ part, const uint8_t *__restrict__ Wkv,
                                                            float *__restrict__ ctx, int nope, int vh, int n_split) {
    constexpr int LKV = 512, NB = LKV / 256, ROWS = 8;
    __shared__ __attribute__((aligned(16))) float ol[LKV];
    const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, sb = lane >> 5, l = lane & 31, c = l >> 3;
    const int row0 = 64 * (int)blockIdx.y + ROWS * wave;
    const uint8_t *src = Wkv + ((((size_t)h * (nope + vh)) + nope + row0) * NB + sb) * 144;
    uint4 hdr[ROWS];
    uint32_t qs[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; i++) {
        hdr[i] = *(const uint4 *)(src + (size_t)i * NB * 144);
        qs[i] = *(const uint32_t *)(src + (size_t)i * NB * 144 + 16 + 4 * l);
    }
    const float *p = part + (size_t)h * n_split * (LKV + 2);
    const float mi = lane < n_split ? p[(size_t)lane * (LKV + 2)] : -INFINITY;  // n_split <= 64
    const float M = wave_max(mi);
    const float fi = mi == -INFINITY ? 0.0f : __expf(mi - M);  // an empty split
    const float L = wave_sum(lane < n_split ? p[(size_t)lane * (LKV + 2) + 1] * fi : 0.0f);
    float v = 0.0f;
#pragma unroll 8
    for (int i = 0; i < n_split; i++) v = fmaf(p[(size_t)i * (LKV + 2) + 2 + tid], __shfl(fi, i, 64), v);
    ol[tid] = v * (1.0f / L);
    __syncthreads();
    const float4 xl = *(const float4 *)&ol[256 * sb + 64 * c + 4 * (l & 7)], xh = *(const float4 *)&ol[256 * sb + 64 * c + 32 + 4 * (l & 7)];
    const float sl = (xl.x + xl.y) + (xl.z + xl.w), sh = (xh.x + xh.y) + (xh.z + xh.w);
    float mine = 0.0f;
#pragma unroll
    for (int i = 0; i < ROWS; i++) {
        const MlaQ4kWord w = mla_q4k_word(hdr[i], qs[i], c);
        const float a = fmaf(w.lo[0], xl.x, fmaf(w.lo[1], xl.y, fmaf(w.lo[2], xl.z, w.lo[3] * xl.w)));
        const float b = fmaf(w.hi[0], xh.x, fmaf(w.hi[1], xh.y, fmaf(w.hi[2], xh.z, w.hi[3] * xh.w)));
        const float y = wave_sum(fmaf(w.dl, a, fmaf(w.dh, b, -fmaf(w.ml, sl, w.mh * sh))));
        if (lane == i) mine = y;
    }
    if (lane < ROWS && row0 + lane < vh) ctx[(size_t)h * vh + row0 + lane] = mine;
}

// Everything of a step between the query and the output projection in one launch, for one token over a short context and Q4_K blocks
// of 128 key and vh value rows of 512 columns a head.  grid (n_head, vh / 64), 16 waves: a workgroup absorbs its head's query (a
// quarter-wave a row and super-block, a lane two words of it), rotates the query's rope part, norms the new token's latent and rotates
// its key (everybody makes them for himself, the first workgroup appends them to the cache), scores the cached tokens, a wave eight at a
// time with their rows in registers, merges the waves' sums and multiplies with 64 value rows.  f32 throughout.
// Bound: a chain of some 900 vector instructions a wave, four waves a SIMD, and three trips to memory.  128 heads of 128 + 64 elements
// behind 100 tokens: 9.5 to 11.5 us where absorbing, scoring and merging with the value rows, a launch each, take 6.2, 5.1 and 5.0 and
// their boundaries (whole steps: at the dispatch).  All value rows in one workgroup a head, half the compute units idle: 0.5 us a step slower.
__device__ __forceinline__ float mla_sum_half(float v) {  // over the 32 lanes of a half-wave
    v = sum_xor16(v);
    return sum_row16(v);
}
struct MlaQ4kPair {  // two words next to each other: 8 columns of either sub-block
    float lo[8], hi[8], dl, dh, ml, mh;
};
__device__ __forceinline__ MlaQ4kPair mla_q4k_pair(const uint4 &hdr, const uint2 &q, int c) {
    MlaQ4kPair w;
    const MlaQ4kWord a = mla_q4k_word(hdr, q.x, c);
    w.dl = a.dl, w.dh = a.dh, w.ml = a.ml, w.mh = a.mh;
    const uint32_t lo = q.y & 0x0F0F0F0Fu, hi = (q.y >> 4) & 0x0F0F0F0Fu;
#pragma unroll
    for (int b = 0; b < 4; b++) {
        w.lo[b] = a.lo[b], w.hi[b] = a.hi[b];
        w.lo[4 + b] = (float)((lo >> (8 * b)) & 0xFFu), w.hi[4 + b] = (float)((hi >> (8 * b)) & 0xFFu);
    }
    return w;
}
__global__ __launch_bounds__(1024) void mla_step_q4k(const float *__restrict__ q, const uint8_t *__restrict__ Wkv, float *__restrict__ ctx, int vh,
                                                      const float *__restrict__ comp, const float *__restrict__ w,
                                                      const float2 *__restrict__ cs, float *__restrict__ lat, float *__restrict__ kpe,
                                                      int pos, float eps, float scale) {
    constexpr int LKV = MLA_M_LKV, ROPE = MLA_M_ROPE, NOPE = 128, WAVES = 16, RUN = 4, N = 8;  // rows, tokens a wave at a time
    __shared__ __attribute__((aligned(16))) float red[WAVES][LKV], mid[LKV];
    __shared__ float max_sh[WAVES], sum_sh[WAVES];
    const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l = lane & 15, sb = (lane >> 4) & 1, half = lane >> 5, c = l >> 2, col = 256 * sb + 64 * c + 8 * (l & 3);
    const float *qh = q + (size_t)h * (NOPE + ROPE);
    const uint8_t *rows = Wkv + (size_t)h * (NOPE + vh) * (2 * 144) + 144 * sb;
    uint4 hdr[RUN];
    uint2 qs[RUN];
    auto fetch = [&](int first, int n) __attribute__((always_inline)) {  // rows first + 2 (wave + 16 i) + half, i < n
#pragma unroll
        for (int i = 0; i < RUN; i++) {
            if (i >= n) break;
            const uint8_t *src = rows + (size_t)(first + 2 * (wave + WAVES * i) + half) * (2 * 144);
            hdr[i] = *(const uint4 *)src, qs[i] = *(const uint2 *)(src + 16 + 8 * l);
        }
    };
    fetch(0, RUN);
    float x[RUN];
#pragma unroll
    for (int i = 0; i < RUN; i++) x[i] = qh[2 * (wave + WAVES * i) + half];
    const float2 turn = cs[(size_t)pos * (ROPE / 2) + (lane >> 1)];
    const float2 pair = *(const float2 *)(qh + NOPE + (lane & ~1));
    float4 k[N][2];
    float kp[N];
    auto tokens = [&](int t0) __attribute__((always_inline)) {  // t0 + wave + 16 i, those there are
#pragma unroll
        for (int i = 0; i < N; i++) {
            const size_t at = (size_t)min(t0 + wave + WAVES * i, pos - 1);
            const float4 *src = (const float4 *)(lat + at * LKV + 8 * lane);
            k[i][0] = src[0], k[i][1] = src[1];
            kp[i] = kpe[at * ROPE + lane];
        }
    };
    float4 o[2] = {float4{0.0f, 0.0f, 0.0f, 0.0f}, float4{0.0f, 0.0f, 0.0f, 0.0f}};
    float key = 0.0f;
    {
        float lo[8], hi[8], ml = 0.0f, mh = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) lo[e] = hi[e] = 0.0f;
#pragma unroll
        for (int i = 0; i < RUN; i++) {
            const MlaQ4kPair v = mla_q4k_pair(hdr[i], qs[i], c);
            const float a = x[i] * v.dl, b = x[i] * v.dh;
#pragma unroll
            for (int e = 0; e < 8; e++) lo[e] = fmaf(a, v.lo[e], lo[e]), hi[e] = fmaf(b, v.hi[e], hi[e]);
            ml = fmaf(x[i], v.ml, ml), mh = fmaf(x[i], v.mh, mh);
        }
#pragma unroll
        for (int e = 0; e < 8; e++) lo[e] = sum_xor32(lo[e] - ml), hi[e] = sum_xor32(hi[e] - mh);
        if (half == 0) {
            float *to = &red[wave][col];
            *(float4 *)to = float4{lo[0], lo[1], lo[2], lo[3]}, *(float4 *)(to + 4) = float4{lo[4], lo[5], lo[6], lo[7]};
            *(float4 *)(to + 32) = float4{hi[0], hi[1], hi[2], hi[3]}, *(float4 *)(to + 36) = float4{hi[4], hi[5], hi[6], hi[7]};
        }
    }
    if (wave < pos) tokens(0);
    if (wave == pos % WAVES) {  // the new token (of the waves, one of those with the fewest cached tokens)
        float ss = 0.0f;  // (in the order of mla_rope_latent)
#pragma unroll
        for (int i = 0; i < LKV; i += 64) ss = fmaf(comp[i + lane], comp[i + lane], ss);
        const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)LKV + eps);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const float4 v = *(const float4 *)(comp + 8 * lane + 4 * i), g = *(const float4 *)(w + 8 * lane + 4 * i);
            o[i] = float4{v.x * inv * g.x, v.y * inv * g.y, v.z * inv * g.z, v.w * inv * g.w};
        }
        const float2 key2 = *(const float2 *)(comp + LKV + (lane & ~1));
        key = lane & 1 ? key2.x * turn.y + key2.y * turn.x : key2.x * turn.x - key2.y * turn.y;
        if (h == 0 && blockIdx.y == 0) {
            float4 *to = (float4 *)(lat + (size_t)pos * LKV + 8 * lane);
            to[0] = o[0], to[1] = o[1];
            kpe[(size_t)pos * ROPE + lane] = key;
        }
    }
    __syncthreads();
    if (tid < LKV) {
        float v = 0.0f;
#pragma unroll
        for (int i = 0; i < WAVES; i++) v += red[i][tid];
        mid[tid] = v;
    }
    __syncthreads();
    const float4 qa = *(const float4 *)&mid[8 * lane], qb = *(const float4 *)&mid[8 * lane + 4];
    const float qp = lane & 1 ? pair.x * turn.y + pair.y * turn.x : pair.x * turn.x - pair.y * turn.y;
    auto score = [&](const float4 &a, const float4 &b, float key) __attribute__((always_inline)) {
        float v = qp * key;
        v = fmaf(qa.x, a.x, fmaf(qa.y, a.y, fmaf(qa.z, a.z, fmaf(qa.w, a.w, v))));
        v = fmaf(qb.x, b.x, fmaf(qb.y, b.y, fmaf(qb.z, b.z, fmaf(qb.w, b.w, v))));
        return wave_sum(v) * scale;
    };
    float m = -INFINITY, sum = 0.0f;
    if (wave == pos % WAVES) m = score(o[0], o[1], key), sum = 1.0f;
    for (int t0 = 0; t0 + wave < pos; t0 += WAVES * N) {
        if (t0 > 0) tokens(t0);
        float s[N], top = m;
#pragma unroll
        for (int i = 0; i < N; i++) {
            s[i] = score(k[i][0], k[i][1], kp[i]);
            if (t0 + wave + WAVES * i < pos) top = fmaxf(top, s[i]);
        }
        const float keep = m == -INFINITY ? 0.0f : __expf(m - top);
        m = top, sum *= keep;
#pragma unroll
        for (int j = 0; j < 2; j++) o[j].x *= keep, o[j].y *= keep, o[j].z *= keep, o[j].w *= keep;
#pragma unroll
        for (int i = 0; i < N; i++) {
            const float p = t0 + wave + WAVES * i < pos ? __expf(s[i] - m) : 0.0f;
            sum += p;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                o[j].x = fmaf(p, k[i][j].x, o[j].x), o[j].y = fmaf(p, k[i][j].y, o[j].y);
                o[j].z = fmaf(p, k[i][j].z, o[j].z), o[j].w = fmaf(p, k[i][j].w, o[j].w);
            }
        }
    }
    const int first = NOPE + 64 * (int)blockIdx.y;
    fetch(first, 2);
    *(float4 *)&red[wave][8 * lane] = o[0], *(float4 *)&red[wave][8 * lane + 4] = o[1];
    if (lane == 0) max_sh[wave] = m, sum_sh[wave] = sum;
    __syncthreads();
    if (tid < LKV) {
        const float mi = max_sh[lane & 15], M = wave_max(mi);
        const float fi = mi == -INFINITY ? 0.0f : __expf(mi - M);  // a wave without tokens
        const float L = wave_sum(lane < WAVES ? sum_sh[lane & 15] * fi : 0.0f);
        float v = 0.0f;
#pragma unroll
        for (int i = 0; i < WAVES; i++) v = fmaf(red[i][tid], __shfl(fi, i, 64), v);
        mid[tid] = v * (1.0f / L);
    }
    __syncthreads();
    float xl[8], xh[8], sl = 0.0f, sh = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; e++) xl[e] = mid[col + e], xh[e] = mid[col + 32 + e], sl += xl[e], sh += xh[e];
    float mine = 0.0f;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const MlaQ4kPair v = mla_q4k_pair(hdr[i], qs[i], c);
        float a = v.lo[0] * xl[0], b = v.hi[0] * xh[0];
#pragma unroll
        for (int e = 1; e < 8; e++) a = fmaf(v.lo[e], xl[e], a), b = fmaf(v.hi[e], xh[e], b);
        const float y = mla_sum_half(fmaf(v.dl, a, fmaf(v.dh, b, -fmaf(v.ml, sl, v.mh * sh))));
        if (l == i) mine = y;
    }
    if (l < 2 && sb == 0) ctx[(size_t)h * vh + (first - NOPE) + 2 * (wave + WAVES * l) + half] = mine;
}

}  // namespace jq

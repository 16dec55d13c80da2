// The residual stream of decoders that normalise in front of and behind a sublayer: x + mult * norm(y), then the norm
// of the result for the next sublayer, f32 throughout, one workgroup of BT threads a row.
#pragma once
#include "kernels_graph.hpp"

namespace jq {

struct ResidualNorm {
    const float *x;                    // the residual stream
    const float *y;                    // the sublayer's result to add, or null
    const float *post_w, *post_b;      // the norm on y (post_w null: y as it is)
    float mult;
    const float *pre_w, *pre_b;        // the norm that makes h
    float eps;
    int rms;                           // both norms: 1 root mean square, 0 mean and variance (with bias)
    int width;
    size_t ldx;                        // x: from a row to the next (0: width)
    float *x_out;                      // may be x, except where other workgroups read the row
    float *h_out;                      // or null
};

// sum over the workgroup of BT, in every thread; `red` [BT / 64] is not used again before another barrier
template <int BT>
__device__ __forceinline__ float sum_block(float v, float *red) {
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < BT / 64; i++) s += red[i];
    return s;
}

// Element i of a thread's share of a row: four columns side by side, every 4 BT.
template <int BT>
__device__ __forceinline__ int norm_col(int i) { return 4 * (int)threadIdx.x + 4 * BT * (i / 4) + i % 4; }

// The thread's share of a row as it is read: every load is issued whatever the width (past it, from the row's end), so that the
// loads of a row's vectors travel together.
template <int NV, int BT>
__device__ __forceinline__ void ask_row(const float *__restrict__ p, int width, float (&v)[NV]) {
    if ((width & 3) == 0) {
#pragma unroll
        for (int i = 0; i < NV; i += 4) {
            const float4 q = *(const float4 *)(p + min(norm_col<BT>(i), width - 4));
            v[i] = q.x, v[i + 1] = q.y, v[i + 2] = q.z, v[i + 3] = q.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < NV; i++) v[i] = p[min(norm_col<BT>(i), width - 1)];
    }
}
// Zeros past the width.
template <int NV, int BT>
__device__ __forceinline__ void end_row(int width, float (&v)[NV]) {
#pragma unroll
    for (int i = 0; i < NV; i++) v[i] = norm_col<BT>(i) < width ? v[i] : 0.0f;
}

template <int NV, int BT>
__device__ __forceinline__ void store_row(float *__restrict__ p, int width, const float (&v)[NV]) {
    if ((width & 3) == 0) {
#pragma unroll
        for (int i = 0; i < NV; i += 4)
            if (norm_col<BT>(i) < width) *(float4 *)(p + norm_col<BT>(i)) = float4{v[i], v[i + 1], v[i + 2], v[i + 3]};
    } else {
#pragma unroll
        for (int i = 0; i < NV; i++)
            if (norm_col<BT>(i) < width) p[norm_col<BT>(i)] = v[i];
    }
}

// One norm over the row held as v (0 past the width): mean and 1 / deviation.
template <int NV, int BT>
__device__ __forceinline__ void row_stats(const float (&v)[NV], int width, float eps, int rms, float *red, float *mean, float *inv) {
    float mu = 0.0f;
    if (!rms) {
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < NV; i++) s += v[i];
        mu = sum_block<BT>(s, red) / (float)width;
    }
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const float d = norm_col<BT>(i) < width ? v[i] - mu : 0.0f;
        ss = fmaf(d, d, ss);
    }
    *mean = mu;
    *inv = 1.0f / sqrtf(sum_block<BT>(ss, red + BT / 64) / (float)width + eps);
}

// The update of one row by a workgroup; x ends as this thread's share of the normed row.  With `store` the stream goes to
// x_out and the normed row to h_out.  The norms' vectors are asked for together with the row: a single row's time is its
// round trips to memory.  `behind` asks for what the caller wants in flight meanwhile, behind the row: a compute unit's requests are
// served in order.
template <int NV, int BT, class Behind>
__device__ __forceinline__ void residual_norm_row(const ResidualNorm &a, float (&x)[NV], bool store, Behind behind) {
    __shared__ float red[4 * (BT / 64)];  // a part for each of the sums
    const int w = a.width;
    float g[NV], b[NV], mean, inv;
    ask_row<NV, BT>(a.x, w, x);
    if (a.y) {
        float y[NV], pg[NV], pb[NV];
        ask_row<NV, BT>(a.y, w, y);
        if (a.post_w) ask_row<NV, BT>(a.post_w, w, pg);
        if (a.post_w && a.post_b) ask_row<NV, BT>(a.post_b, w, pb);
        ask_row<NV, BT>(a.pre_w, w, g);
        if (a.pre_b) ask_row<NV, BT>(a.pre_b, w, b);
        __builtin_amdgcn_sched_barrier(0);
        behind();
        __builtin_amdgcn_sched_barrier(0);
        end_row<NV, BT>(w, y);
        if (a.post_w) {
            row_stats<NV, BT>(y, w, a.eps, a.rms, red, &mean, &inv);
#pragma unroll
            for (int i = 0; i < NV; i++) y[i] = norm_col<BT>(i) < w ? fmaf((y[i] - mean) * inv, pg[i], a.post_b ? pb[i] : 0.0f) : 0.0f;
        }
        end_row<NV, BT>(w, x);
#pragma unroll
        for (int i = 0; i < NV; i++) x[i] = fmaf(a.mult, y[i], x[i]);
    } else {
        ask_row<NV, BT>(a.pre_w, w, g);
        if (a.pre_b) ask_row<NV, BT>(a.pre_b, w, b);
        __builtin_amdgcn_sched_barrier(0);
        behind();
        __builtin_amdgcn_sched_barrier(0);
        end_row<NV, BT>(w, x);
    }
    if (store && a.x_out) store_row<NV, BT>(a.x_out, w, x);
    row_stats<NV, BT>(x, w, a.eps, a.rms, red + 2 * (BT / 64), &mean, &inv);
    end_row<NV, BT>(w, g);
    if (a.pre_b) end_row<NV, BT>(w, b);
#pragma unroll
    for (int i = 0; i < NV; i++) x[i] = fmaf((x[i] - mean) * inv, g[i], a.pre_b ? b[i] : 0.0f);
    if (store && a.h_out) store_row<NV, BT>(a.h_out, w, x);
}

// The update of many rows, a workgroup a row: x in place, h in f32 (h_out) and / or in the products' element type (he, rows
// `stride` apart, zeros behind the width).  `at`: the rows to take, into the first rows of h (x_out is then left alone), or
// null for rows 0, 1, ..  A thread has columns BT apart.
template <class E, int NV, int BT>
__global__ __launch_bounds__(BT) void residual_norm_rows(ResidualNorm a, typename E::T *__restrict__ he, size_t stride,
                                                         const uint32_t *__restrict__ at) {
    using T = typename E::T;
    constexpr int NW = BT / 64;
    __shared__ float red[4 * NW];
    const int w = a.width, c0 = threadIdx.x;
    const size_t row = at ? at[blockIdx.x] : blockIdx.x;
    const float *xr = a.x + row * (a.ldx ? a.ldx : (size_t)w);
    // Loads past the width repeat the last column, so that none needs a branch, and all of a row's vector are asked for before the first
    // is waited for, and in front of any store: one by one they were 12 of 17.5 us, of one row of 4096 columns or of 512.
    // (128 registers for 70 to 84, so four waves a SIMD for six or seven: rows of 1024 to 16384, 1 to 4096 of them, with and without a norm on y and
    // biases, take 0.62 to 0.98 of the time all the same; 4096 rows of 16384 206 -> 178 us.)
    auto ask = [&](const float *src, float (&v)[NV]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NV; i++) v[i] = src[min(c0 + BT * i, w - 1)];
    };
    auto stats = [&](const float (&v)[NV], float *r, float *mean, float *inv) __attribute__((always_inline)) {
        float mu = 0.0f, ss = 0.0f;
        if (!a.rms) {
            float s = 0.0f;
#pragma unroll
            for (int i = 0; i < NV; i++) s += c0 + BT * i < w ? v[i] : 0.0f;
            mu = sum_block<BT>(s, r) / (float)w;
        }
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const float d = c0 + BT * i < w ? v[i] - mu : 0.0f;
            ss = fmaf(d, d, ss);
        }
        *mean = mu, *inv = 1.0f / sqrtf(sum_block<BT>(ss, r + NW) / (float)w + a.eps);
    };
    float x[NV], g[NV], mean, inv;
    ask(xr, x);
    if (a.y) {
        float y[NV];
        ask(a.y + row * w, y);
        if (a.post_w) {
            ask(a.post_w, g);
            stats(y, red, &mean, &inv);
#pragma unroll
            for (int i = 0; i < NV; i++) y[i] = (y[i] - mean) * inv;
            if (a.post_b) {
                float b[NV];
                ask(a.post_b, b);
#pragma unroll
                for (int i = 0; i < NV; i++) y[i] = fmaf(y[i], g[i], b[i]);
            } else {
#pragma unroll
                for (int i = 0; i < NV; i++) y[i] = fmaf(y[i], g[i], 0.0f);
            }
        }
#pragma unroll
        for (int i = 0; i < NV; i++) x[i] = fmaf(a.mult, y[i], x[i]);
    }
    ask(a.pre_w, g);
    stats(x, red + 2 * NW, &mean, &inv);
    float b[NV];
    if (a.pre_b) {
        ask(a.pre_b, b);
    } else {
#pragma unroll
        for (int i = 0; i < NV; i++) b[i] = 0.0f;
    }
    float *xo = at ? nullptr : a.x_out, *ho = a.h_out ? a.h_out + (size_t)blockIdx.x * w : nullptr;
    T *eo = he ? he + (size_t)blockIdx.x * stride : nullptr;
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int c = c0 + BT * i;
        if (c < w) {
            const float v = fmaf((x[i] - mean) * inv, g[i], b[i]);
            if (xo) xo[row * w + c] = x[i];
            if (ho) ho[c] = v;
            if (eo) eo[c] = (T)v;
        } else if (eo && c < (int)stride) {
            eo[c] = (T)0.0f;
        }
    }
}

}  // namespace jq

// Host side of the GEMM on f16 and FP6 operands.
#include "gemm_h6.hpp"

#include "kernels_mfma_gemm_h6.hpp"

namespace jqh {
namespace {

// Leave to use that much LDS, asked for once a kernel.
template <auto KERN>
hipError_t big_lds_once(int lds) {
    static const hipError_t rc = hipFuncSetAttribute((const void *)KERN, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    return rc;
}

struct Shape {
    int nw, ng;
    // tiles of the activation rows, of the weight rows, workgroups of a launch
    size_t rows(size_t m) const { return (m + 32 * (size_t)nw - 1) / (32 * (size_t)nw); }
    size_t cols(size_t n) const { return (n + 16 * (size_t)ng - 1) / (16 * (size_t)ng); }
    size_t grid(size_t m, size_t n) const {
        const size_t ty = rows(m), tiles = ty * cols(n);
        return 8 % ty == 0 ? (tiles + 7) / 8 * 8 : tiles;
    }
};
constexpr Shape SHAPES[] = {{8, 8}, {8, 7}, {8, 6}, {4, 4}};

// In us, the int8 GEMM's form of estimate (gemm_i8_us) fitted to 714 times of this one's shapes of seven, six and four groups in 1 to 8
// parts (eight groups: 1.09 of seven's super-block, 512 to 2048 rows x 4096 to 24576): the
// preparation, a fixed start, the super-blocks a workgroup walks at a cost that grows with the workgroups at work, the
// starts of further rounds, the sum of the parts.  Over 166 shapes the picks are 0.7 % off the best measured choice on
// average, 5 % at the 95th percentile, 12 % at worst.
double estimate(const Shape &sh, size_t m, size_t nb, size_t n, size_t sp) {
    auto rounds = [](double wgs, double at_once, auto us) {
        const double whole = std::floor(wgs / at_once), rest = wgs - whole * at_once;
        return whole * us(at_once) + (rest > 0.0 ? us(rest) : 0.0);
    };
    const double wgs = (double)(sh.grid(m, n) * sp), nbl = (double)(nb / sp);
    double us = 3.2 + 0.0048 * (double)(nb * ((m + 15) / 16));
    if (sh.nw == 8)
        us += 6.4 + nbl * rounds(wgs, 256.0, [](double w) { return 3.4 + 0.0035 * w; }) * (sh.ng == 8 ? 1.09 : sh.ng == 7 ? 1.0 : 0.92) +
              4.2 * (std::ceil(wgs / 256.0) - 1.0);
    else
        us += 6.6 + nbl * rounds(wgs, 512.0, [](double w) { return w <= 256.0 ? 2.24 + 0.0011 * w : 3.06 + 0.0011 * w; }) +
              2.5 * std::max(0.0, wgs / 512.0 - 1.5);
    if (sp > 1) us += 0.09 * (double)sp + (double)(sp + 1) * (double)(m * n) * 4.0 / 3.4e6;
    return us;
}

// The shape and split over k of the least estimate among those that `may(shape, splits)` admits: the estimate, a negative one if there is none.
template <class May>
double pick(size_t m, size_t nb, size_t n, Shape &best, size_t &splits, May may) {
    double best_us = -1.0;
    for (const Shape &sh : SHAPES)
        for (size_t sp = 1; sp <= 8; sp++) {
            if (nb % sp != 0 || (sp > 1 && nb / sp < 4) || !may(sh, sp)) continue;
            const double us = estimate(sh, m, nb, n, sp);
            if (best_us < 0.0 || us < best_us) best = sh, splits = sp, best_us = us;
        }
    return best_us;
}

// Q4_K and MXFP4 with 128 activation rows or more on f16 and FP6 operands (kq_gemm_h6), us against the int8 GEMM's, whole calls back to back (Q4_K):
// 512 x 14336 x 4096 95 / 116, 2048 x 24576 x 4096 604 / 738, 512 x 4096 x 4096 48 / 50.  166 shapes of 128 to 2048 rows against
// 1000 to 24576 weight rows of 1024 to 16384: 0.77 to 1.08 of its time, 0.91 on average; the 18 that are more than 2 % slower, by
// 0.5 to 2 us, are those against some 1000 weight rows and 333 to 512 rows against 4096.  Below 128 rows the int8 GEMM is as fast
// (64 to 127 rows: 0.90 to 1.07) and keeps them: there unpacking the weights is most of the work in both.  `name` is the one that
// callers of jq_last_kernel know the many-row product by; jq_last_arithmetic says which of the two ran.
// Returns -1 when the shape is outside its reach and where the environment names a shape or a switch of that GEMM.  JQ_GEMM_H6 = 0
// switches this one off, JQ_GEMM_H6_SHAPE and _SPLITS force the choice, _MIN_M moves the fewest rows.
// SWIGLU (the kernel's): declined where k is in parts, whose sums are no products yet.
template <class F, bool SWIGLU = false>
int dispatch(const uint8_t *W, size_t row_bytes, const float *X, float *Y, size_t m, size_t k, size_t n, hipStream_t s, const char *name, const char *name_split, bool swiglu_pairs = false) {
    static const char *mode = getenv("JQ_GEMM_H6"), *i8_mode = getenv("JQ_Q4K_GEMM_I8"), *i8_shape = getenv("JQ_Q4K_GEMM_I8_SHAPE");
    static const char *shape_env = getenv("JQ_GEMM_H6_SHAPE"), *splits_env = getenv("JQ_GEMM_H6_SPLITS");
    static const char *min_m_env = getenv("JQ_GEMM_H6_MIN_M");
    static const size_t min_m = min_m_env ? std::max<size_t>((size_t)atoll(min_m_env), 2) : 128;
    if ((mode && mode[0] == '0') || i8_mode || i8_shape || m < min_m || k % 256 != 0 || k == 0 || row_bytes % F::ALIGN != 0 ||
        !jq::h6_offsets_hold(k / 256, row_bytes) || ((uintptr_t)W & (F::ALIGN - 1)) != 0 || ((uintptr_t)X & 15) != 0 || m > 0x7FFFFFF0ull || n > 0x7FFFFFF0ull)
        return -1;
    const size_t nb = k / 256, groups = (m + 15) / 16;
    const size_t scratch_cap = tl_fixed_scratch ? tl_fixed_scratch->bytes : (size_t)1 << 40;
    // A fixed scratch that holds the int8 GEMM's records of all rows, three quarters of these in size, takes the rows in two turns;
    // what neither GEMM's records fit fails there as it did.  (1024 x 12288: 36 MB in 32.)
    size_t turn = m;
    auto acts_of = [&](size_t rows) { return ((rows + 15) / 16 * nb * (size_t)jq::h6_rec<F::MINS>() + 255) & ~(size_t)255; };
    if (acts_of(m) > scratch_cap) {
        if (groups * nb * INT8_GEMM_REC > scratch_cap) return -1;
        turn = (groups + 1) / 2 * 16;
        if (acts_of(turn) > scratch_cap) return -1;
    }
    const size_t acts_bytes = acts_of(turn);
    if (!min_m_env && SHAPES[3].rows(m) * SHAPES[3].cols(n) * std::max<size_t>(1, std::min<size_t>(nb / 4, 8)) < 64) return -1;
    int want_nw = 0, want_ng = 0;
    const bool forced = shape_env && sscanf(shape_env, "%d,%d", &want_nw, &want_ng) == 2;
    Shape best{};
    size_t splits = 1;
    const double us = pick(m, nb, n, best, splits, [&](const Shape &sh, size_t sp) {
        if (forced && (sh.nw != want_nw || sh.ng != want_ng)) return false;
        if (splits_env && sp != (size_t)atoi(splits_env)) return false;
        return sp == 1 || (m * n <= 0x3FFFFFFFull && acts_bytes + (sp - 1) * turn * n * sizeof(float) <= scratch_cap);
    });
    if (us < 0.0 || best.grid(m, n) > 0x7FFFFFFFull || (SWIGLU && (splits > 1 || n % 2 != 0))) return -1;
    CallScratch scratch;
    uint8_t *acts = nullptr;
    if (scratch.get(acts_bytes + (splits - 1) * turn * n * sizeof(float), s, &acts)) return 1;
    float *parts = (float *)(acts + acts_bytes);  // of all parts of k but the first, which is summed in place
    auto launch = [&](auto kern, int lds, int nw, hipError_t rc) {
        if (rc != hipSuccess) return fail("hipFuncSetAttribute: %s", hipGetErrorString(rc));
        for (size_t m0 = 0; m0 < m; m0 += turn) {
            const size_t rows = std::min(turn, m - m0), row_groups = (rows + 15) / 16, outs = rows * n;
            const float *x = X + m0 * k * (swiglu_pairs ? 2 : 1);
            float *y = Y + m0 * (SWIGLU ? n / 2 : n);
            const dim3 prep((unsigned)nb, (unsigned)row_groups);
            if (swiglu_pairs) hipLaunchKernelGGL((jq::kq_gemm_h6_prep<true, F::MINS, F::NIBBLES>), prep, dim3(128), 0, s, x, (int)rows, (int)k, acts);
            else hipLaunchKernelGGL((jq::kq_gemm_h6_prep<false, F::MINS, F::NIBBLES>), prep, dim3(128), 0, s, x, (int)rows, (int)k, acts);
            hipLaunchKernelGGL(kern, dim3((unsigned)best.grid(rows, n), (unsigned)splits), dim3(64 * nw), lds, s, W, row_bytes,
                               (const uint8_t *)acts, y, (int)rows, (int)n, (int)(nb / splits), (int)row_groups,
                               (int)best.cols(n), (int)best.rows(rows), (int)nb, parts);
            if (splits > 1)
                hipLaunchKernelGGL(jq::splitk_add, dim3((unsigned)((outs + 1023) / 1024)), dim3(256), 0, s, parts, y, outs, (int)splits - 1);
        }
        return 0;
    };
#define JQ_GEMM_H6(NW_, NG_) launch(jq::kq_gemm_h6<F, NW_, NG_, SWIGLU>, jq::h6_lds_bytes<NG_>(), NW_, big_lds_once<&jq::kq_gemm_h6<F, NW_, NG_, SWIGLU>>(jq::h6_lds_bytes<NG_>()))
    const int rc = best.nw == 4 ? JQ_GEMM_H6(4, 4) : best.ng == 8 ? JQ_GEMM_H6(8, 8) : best.ng == 7 ? JQ_GEMM_H6(8, 7) : JQ_GEMM_H6(8, 6);
#undef JQ_GEMM_H6
    if (rc) return rc;
    note_kernel(splits > 1 ? name_split : name, "f16+fp6");
    HIP_TRY(hipGetLastError());
    return 0;
}

}  // namespace

double gemm_h6_us(size_t m, size_t k, size_t n) {
    Shape best;
    size_t splits;
    return pick(m, k / 256, n, best, splits, [](const Shape &, size_t) { return true; });
}

int gemm_h6(uint32_t type, const uint8_t *W, size_t row_bytes, const float *X, float *Y, size_t m, size_t k, size_t n, hipStream_t s,
            const char *name, const char *name_split, bool swiglu_pairs) {
    switch (type) {
    case JQ_TYPE_Q4_K: return dispatch<jq::H6Q4K>(W, row_bytes, X, Y, m, k, n, s, name, name_split, swiglu_pairs);
    case JQ_TYPE_MXFP4: return dispatch<jq::H6MXFP4>(W, row_bytes, X, Y, m, k, n, s, name, name_split, swiglu_pairs);
    default: return -1;
    }
}

int gemm_h6_swiglu(uint32_t type, const uint8_t *W, size_t row_bytes, const float *X, float *Y, size_t m, size_t k, size_t n, hipStream_t s) {
    return type == JQ_TYPE_Q4_K ? dispatch<jq::H6Q4K, true>(W, row_bytes, X, Y, m, k, n, s, "q4k_gemm_i8", nullptr) : -1;
}

}  // namespace jqh

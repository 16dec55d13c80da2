// Host side of the products of a few activation rows.
#include "few_rows.hpp"

#include "kernels_few_rows.hpp"

namespace jqh {
namespace {

constexpr int LDS = 160 * 1024;

// Waves of a workgroup, and the super-blocks that the busiest of a compute unit's four SIMDs takes: as few as can be, then with as many
// waves as fit the LDS.
template <class F>
int waves_of(int tiles, int rows, size_t nb, size_t &most) {
    int best = 1;
    most = nb;
    for (int waves = 2; waves <= 8 && jq::few_rows_lds<F>(waves, tiles, rows) <= LDS; waves++) {
        size_t busiest = 0;
        for (int simd = 0; simd < 4; simd++) {
            size_t mine = 0;
            for (int w = simd; w < waves; w += 4) mine += (nb + waves - 1 - w) / waves;
            busiest = std::max(busiest, mine);
        }
        if (busiest <= most) most = busiest, best = waves;
    }
    return best;
}

template <class F, int NT, int ROWS>
int launch(const uint8_t *W, size_t row_bytes, const float *X, float *Y, size_t m, size_t n, size_t nb, hipStream_t s) {
    static const hipError_t big = hipFuncSetAttribute((const void *)jq::few_rows<F, NT, ROWS>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (big != hipSuccess) return fail("hipFuncSetAttribute: %s", hipGetErrorString(big));
    size_t most;
    const int waves = waves_of<F>(NT, ROWS, nb, most);
    hipLaunchKernelGGL((jq::few_rows<F, NT, ROWS>), dim3((unsigned)((n + 16 * NT - 1) / (16 * NT))), dim3(64 * waves),
                       jq::few_rows_lds<F>(waves, NT, ROWS), s, W, (uint32_t)row_bytes, X, Y, (int)m, (int)n, (int)nb);
    return 0;
}

template <class F>
int dispatch(const uint8_t *W, size_t row_bytes, const float *X, float *Y, size_t m, size_t k, size_t n, hipStream_t s) {
    static const char *tiles_env = getenv("JQ_FEW_ROWS_TILES");
    if (m < 1 || m > 16 || k == 0 || k % 256 != 0 || row_bytes % F::ALIGN != 0 || ((uintptr_t)W & (F::ALIGN - 1)) != 0 || ((uintptr_t)X & 15) != 0 ||
        n > 0x7FFFFF00ull || row_bytes > 0x200000)
        return -1;
    const size_t nb = k / 256;
    const int rows = m <= 4 ? 4 : m <= 8 ? 8 : 16;
    // Tiles of 16 weight rows a workgroup: the fewer, the more compute units at work; the more, the fewer times the activations are split.
    // Splitting takes about four fifths of a tile's time, and a compute unit holds one workgroup.
    int nt = 1;
    double best = 0.0;
    for (int t : {4, 2, 1}) {
        size_t most;
        const int waves = waves_of<F>(t, rows, nb, most);
        const double rounds = std::ceil((double)((n + 16 * t - 1) / (16 * t)) / 256.0);
        const double cost = rounds * (double)most * (0.8 + t) * (waves <= 4 ? 1.1 : 1.0);
        if (best == 0.0 || cost < best) best = cost, nt = t;
    }
    if (tiles_env) nt = atoi(tiles_env);
    int rc = -1;
#define JQ_FEW(NT_, ROWS_) \
    if (nt == NT_ && rows == ROWS_) rc = launch<F, NT_, ROWS_>(W, row_bytes, X, Y, m, n, nb, s);
    JQ_FEW(1, 4) JQ_FEW(1, 8) JQ_FEW(1, 16) JQ_FEW(2, 4) JQ_FEW(2, 8) JQ_FEW(2, 16) JQ_FEW(4, 4) JQ_FEW(4, 8) JQ_FEW(4, 16)
#undef JQ_FEW
    if (rc) return rc;
    note_kernel("few_rows", "f16 pairs");
    HIP_TRY(hipGetLastError());
    return 0;
}

template <class F, int NT, int MT>
int launch_many(const uint8_t *W, size_t row_bytes, const float *X, float *Y, size_t m, size_t n, size_t nb, hipStream_t s) {
    constexpr int AHEAD = 2;  // four: more registers and lines under way than the first level cache holds, 10 to 20 % slower
    auto *const kernel = jq::few_rows_many<F, NT, MT, AHEAD>;
    static const hipError_t big = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (big != hipSuccess) return fail("hipFuncSetAttribute: %s", hipGetErrorString(big));
    const size_t groups = (m + 15) / 16, blocks = (groups + MT - 1) / MT, tiles = (n + 16 * NT - 1) / (16 * NT);
    const size_t bytes = groups * nb * jq::FR_REC, grid = (tiles + 7) / 8 * 8 * blocks;
    if ((tl_fixed_scratch && bytes > tl_fixed_scratch->bytes) || MT * nb * jq::FR_REC > 0x7FFFFFFFull || grid > 0x7FFFFFFFull) return -1;
    int waves = 8;
    while (jq::few_rows_many_lds<F>(waves, NT, MT) > LDS) waves--;
    CallScratch scratch;
    uint8_t *acts = nullptr;
    if (scratch.get(bytes, s, &acts)) return 1;
    hipLaunchKernelGGL(jq::few_rows_prep<F>, dim3((unsigned)nb, (unsigned)groups), dim3(64), 0, s, X, (int)m, (int)nb, acts);
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(64 * waves), jq::few_rows_many_lds<F>(waves, NT, MT), s, W, (uint32_t)row_bytes, acts, Y, (int)m,
                       (int)n, (int)nb, (int)groups, (int)blocks);
    return 0;
}

// Workgroup shapes of few_rows_many: tiles of 16 weight rows, groups of 16 activation rows; us a super-block for a format with one f16 number a
// weight and with two (Q4_K and Q6_K, 32 to 128 rows x 4096 x 4096 and 12288: the slope in k).
struct ManyShape {
    int nt, mt;
    double us[2];
};
constexpr ManyShape MANY_SHAPES[] = {{1, 2, {0.42, 0.41}}, {2, 2, {0.48, 0.53}}, {4, 2, {0.68, 0.92}}, {2, 3, {0.64, 0.68}}, {2, 4, {0.78, 0.85}}};

double many_us(const ManyShape &sh, int planes, size_t m, size_t nb, size_t n) {
    const size_t wgs = ((m + 15) / 16 + sh.mt - 1) / sh.mt * ((n + 16 * sh.nt - 1) / (16 * sh.nt));
    return 5.1 + 0.22 * sh.nt * sh.mt + (double)((wgs + 255) / 256 * nb) * sh.us[planes - 1];
}

const ManyShape &many_shape(int planes, size_t m, size_t nb, size_t n) {
    const ManyShape *best = MANY_SHAPES;
    for (const ManyShape &sh : MANY_SHAPES)
        if (many_us(sh, planes, m, nb, n) < many_us(*best, planes, m, nb, n)) best = &sh;
    return *best;
}

template <class F>
int dispatch_many(const uint8_t *W, size_t row_bytes, const float *X, float *Y, size_t m, size_t k, size_t n, hipStream_t s) {
    static const char *shape_env = getenv("JQ_FEW_ROWS_SHAPE");  // "tiles,groups": one of the shapes
    if (k == 0 || k % 256 != 0 || row_bytes % F::ALIGN != 0 || ((uintptr_t)W & (F::ALIGN - 1)) != 0 || ((uintptr_t)X & 15) != 0 ||
        n > 0x7FFFFF00ull || m > 0x7FFFFF00ull || row_bytes > 0x200000)
        return -1;
    const size_t nb = k / 256;
    const ManyShape &sh = many_shape(F::PLANES, m, nb, n);
    int nt = sh.nt, mt = sh.mt, rc = -1;
    if (shape_env) sscanf(shape_env, "%d,%d", &nt, &mt);
#define JQ_FEW(NT_, MT_) \
    if (nt == NT_ && mt == MT_) rc = launch_many<F, NT_, MT_>(W, row_bytes, X, Y, m, n, nb, s);
    JQ_FEW(1, 2) JQ_FEW(2, 2) JQ_FEW(4, 2) JQ_FEW(2, 3) JQ_FEW(2, 4)
#undef JQ_FEW
    if (rc) return rc;
    note_kernel("few_rows_many", "f16 pairs");
    HIP_TRY(hipGetLastError());
    return 0;
}

}  // namespace

// Whole calls, weights from memory, fitted to 1793 times of 17 to 255 rows (6 % off in root mean square): as many_us, which chooses among the shapes,
// with the preparation and a start for every round.  An XCD takes every eighth tile of weight rows, with all its blocks of activation rows, on 32
// compute units (200 x 576 x 7168 of Q6_K, 252 workgroups: 35 on four of the XCDs, 30 us; 144 x 700 x 9984, 25 on most: 26 us).
double few_rows_many_us(uint32_t type, size_t m, size_t k, size_t n) {
    const int planes = type == JQ_TYPE_Q6_K || type == JQ_TYPE_Q8_0 ? 2 : 1;
    const size_t nb = k / 256, groups = (m + 15) / 16;
    const ManyShape &sh = many_shape(planes, m, nb, n);
    const size_t blocks = (groups + sh.mt - 1) / sh.mt, tiles = (n + 16 * sh.nt - 1) / (16 * sh.nt), rounds = ((tiles + 7) / 8 * blocks + 31) / 32;
    const double work = (double)(rounds * nb) * sh.us[planes - 1], prep = (double)(nb * groups);
    return planes == 1 ? 5.1 + 0.31 * sh.nt * sh.mt + 1.9 * (double)(rounds - 1) + 1.01 * work + 0.0048 * prep
                       : 4.75 + 0.45 * sh.nt * sh.mt + 1.76 * (double)(rounds - 1) + 1.175 * work + 0.0019 * prep;
}

int few_rows_many_matmul(uint32_t type, const uint8_t *W, size_t row_bytes, const float *X, float *Y, size_t m, size_t k, size_t n,
                         hipStream_t s) {
    switch (type) {
    case JQ_TYPE_Q4_K: return dispatch_many<jq::FrQ4K>(W, row_bytes, X, Y, m, k, n, s);
    case JQ_TYPE_Q6_K: return dispatch_many<jq::FrQ6K>(W, row_bytes, X, Y, m, k, n, s);
    case JQ_TYPE_Q8_0: return dispatch_many<jq::FrQ8_0>(W, row_bytes, X, Y, m, k, n, s);
    case JQ_TYPE_MXFP4: return dispatch_many<jq::FrMXFP4>(W, row_bytes, X, Y, m, k, n, s);
    default: return -1;
    }
}

int few_rows_matmul(uint32_t type, const uint8_t *W, size_t row_bytes, const float *X, float *Y, size_t m, size_t k, size_t n,
                    hipStream_t s) {
    switch (type) {
    case JQ_TYPE_Q4_K: return dispatch<jq::FrQ4K>(W, row_bytes, X, Y, m, k, n, s);
    case JQ_TYPE_Q6_K: return dispatch<jq::FrQ6K>(W, row_bytes, X, Y, m, k, n, s);
    case JQ_TYPE_Q8_0: return dispatch<jq::FrQ8_0>(W, row_bytes, X, Y, m, k, n, s);
    case JQ_TYPE_MXFP4: return dispatch<jq::FrMXFP4>(W, row_bytes, X, Y, m, k, n, s);
    default: return -1;
    }
}

}  // namespace jqh

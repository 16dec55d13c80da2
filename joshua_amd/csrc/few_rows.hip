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
int dispatch(const uint8_t *W, size_t row_bytes, const float *X, float *Y, size_t m, size_t k, size_t n, const char *name, hipStream_t s) {
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
    note_kernel(name, "f16 pairs");
    HIP_TRY(hipGetLastError());
    return 0;
}

}  // namespace

int few_rows_matmul(uint32_t type, const uint8_t *W, size_t row_bytes, const float *X, float *Y, size_t m, size_t k, size_t n,
                    const char *name, hipStream_t s) {
    switch (type) {
    case JQ_TYPE_Q4_K: return dispatch<jq::FrQ4K>(W, row_bytes, X, Y, m, k, n, name, s);
    case JQ_TYPE_Q6_K: return dispatch<jq::FrQ6K>(W, row_bytes, X, Y, m, k, n, name, s);
    case JQ_TYPE_Q8_0: return dispatch<jq::FrQ8_0>(W, row_bytes, X, Y, m, k, n, name, s);
    case JQ_TYPE_MXFP4: return dispatch<jq::FrMXFP4>(W, row_bytes, X, Y, m, k, n, name, s);
    default: return -1;
    }
}

}  // namespace jqh

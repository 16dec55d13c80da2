// Host side of the grouped Q4_K products on split f16 activations.
#include "moe_split16.hpp"

#include "kernels_moe_split16.hpp"

namespace jqh {

size_t moe_split16_bytes(size_t rows, size_t k) { return rows * (k / 256) * (jq::MS16_PLANES + jq::MS16_XS + sizeof(float)) + 256; }

bool moe_split16_takes(size_t k, size_t row_bytes, int base_align, size_t rows) {
    const size_t nb = k / 256;
    return k % 256 == 0 && nb >= 1 && nb <= (size_t)jq::MS16_MAX_NB && row_bytes % 16 == 0 && base_align >= 16 &&
           rows * nb * jq::MS16_PLANES <= 0x7FFFFFFFull;
}

int moe_split16(const MoeSplit16Call &c, hipStream_t s) {
    const size_t nb = c.k / 256, recs = c.x_rows * nb;
    jq::MoeSplit16 a{};
    a.acts.planes = c.acts;
    a.acts.xs = a.acts.planes + recs * jq::MS16_PLANES;
    a.acts.s = (float *)(a.acts.xs + recs * jq::MS16_XS);
    a.wa = c.wa, a.wb = c.wb, a.row_bytes = c.row_bytes;
    a.gexp = c.gexp, a.offsets = c.offsets, a.xsel = c.xsel, a.yrow = c.yrow;
    a.Y = c.Y, a.groups = c.groups, a.n = (int)c.n, a.nb = (int)nb, a.clamp = c.clamp;
    // Few pairs an expert: workgroups of half the weight rows, three a compute unit, fill the chip more evenly (an expert of 768
    // rows at 32 pairs each: gate and up 141 us against 151).  More: the tile's activations pass through LDS half as often
    // (the down projection there 68 against 76; 128 pairs an expert, the layer 683 against 728).
    const int wt = c.pairs < (c.wb ? 48 : 16) * (size_t)c.groups ? 2 : 4;
    const size_t per = jq::moe_split16_cols(wt) / (c.wb ? 2 : 1);
    a.cols = (int)((c.n + per - 1) / per);
    const size_t tiles = (c.pairs / jq::MS16_ROWS + (size_t)c.groups + 7) / 8 * 8;
    if (tiles * a.cols > 0x7FFFFFFFull) return -1;
    hipLaunchKernelGGL(jq::moe_split16_prep, dim3((unsigned)((nb + 3) / 4), (unsigned)c.x_rows), dim3(256), 0, s, c.X, (int)c.k, a.acts);
    const int lds = jq::moe_split16_lds((int)nb);
    auto *kernel = c.wb ? (wt == 2 ? jq::moe_split16<true, 2> : jq::moe_split16<true, 4>) : (wt == 2 ? jq::moe_split16<false, 2> : jq::moe_split16<false, 4>);
    hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles * a.cols)), dim3(256), lds, s, a);
    HIP_TRY(hipGetLastError());
    note_kernel("moe_split16");
    return 0;
}

}  // namespace jqh

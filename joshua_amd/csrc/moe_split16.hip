// Host side of the grouped expert products on exact operands: Q4_K on split f16 activations, MXFP4 on FP4 and FP8 digits.
#include "moe_split16.hpp"

#include "kernels_moe_mx.hpp"
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
    // Waves of two tiles only for layers whose rows do not fill workgroups of four (128 experts of 768, the layer, us: 70 tokens 144 with two
    // and 135 with four, 150 tokens 155 / 146, 250 tokens 175 / 173, 512 tokens 235 / 220; 256 experts of 64, whose down projection is of another
    // type, 200 tokens 166 with two and 172 with four, of 128 870 / 878).
    const int wt = c.n <= 128 ? 2 : 4;
    const size_t per = jq::moe_split16_cols(wt) / (c.wb ? 2 : 1);
    a.cols = (int)((c.n + per - 1) / per);
    // Calls of fewer than 16 pairs an expert, which the ring kernel's f32 products would run, take two row groups a tile at most,
    // also of an expert with more pairs: those keep the products with the low plane apart (see moe_split16_tile).
    a.rows = c.few ? 32 : jq::MS16_ROWS;
    const size_t tiles = (c.pairs / (size_t)a.rows + (size_t)c.groups + 7) / 8 * 8;
    if (tiles * a.cols > 0x7FFFFFFFull) return -1;
    hipLaunchKernelGGL(jq::moe_split16_prep, dim3((unsigned)c.x_rows, (unsigned)((nb + 3) / 4)), dim3(256), 0, s, c.X, (int)c.k, a.acts);
    const int lds = jq::moe_split16_lds((int)nb, wt);
    auto *kernel = c.wb ? (wt == 2 ? jq::moe_split16<true, 2> : jq::moe_split16<true, 4>) : (wt == 2 ? jq::moe_split16<false, 2> : jq::moe_split16<false, 4>);
    static const hipError_t big[4] = {
#define JQ_BIG(D, WT) hipFuncSetAttribute((const void *)jq::moe_split16<D, WT>, hipFuncAttributeMaxDynamicSharedMemorySize, jq::moe_split16_lds(jq::MS16_MAX_NB, WT))
        JQ_BIG(true, 2), JQ_BIG(true, 4), JQ_BIG(false, 2), JQ_BIG(false, 4)};
#undef JQ_BIG
    for (const hipError_t e : big)
        if (e != hipSuccess) return fail("hipFuncSetAttribute: %s", hipGetErrorString(e));
    hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles * a.cols)), dim3(256), lds, s, a);
    HIP_TRY(hipGetLastError());
    note_kernel("moe_split16");
    return 0;
}

size_t moe_mx_bytes(size_t rows, size_t k) { return rows * (k / jq::MX_CHUNK) * (jq::MX_CHUNK_ACTS + 64) + 256; }

bool moe_mx_takes(size_t n, size_t k, size_t row_bytes, int base_align, size_t rows) {
    return k % jq::MX_CHUNK == 0 && n % 16 == 0 && row_bytes % 16 == 0 && base_align >= 16 && 16 * row_bytes <= 0x7FFFFFFFull &&
           rows * (k / jq::MX_CHUNK) * jq::MX_CHUNK_ACTS <= 0x7FFFFFFFull;
}

int moe_mx(const MoeSplit16Call &c, hipStream_t s) {
    const size_t nc = c.k / jq::MX_CHUNK, recs = c.x_rows * nc;
    jq::MoeMx a{};
    a.acts.digits = c.acts;
    a.acts.scales = (uint32_t *)(c.acts + recs * jq::MX_CHUNK_ACTS);
    a.wa = c.wa, a.wb = c.wb, a.row_bytes = c.row_bytes;
    a.gexp = c.gexp, a.offsets = c.offsets, a.xsel = c.xsel, a.yrow = c.yrow;
    a.Y = c.Y, a.groups = c.groups, a.n = (int)c.n, a.nc = (int)nc, a.clamp = c.clamp;
    // Tiles of 16 pairs on 8 waves from six pairs an expert on if those workgroups fill the chip twice, else of 8 pairs on 4 waves
    // (7168 x 2048, 256 experts, the layer, us: 64 tokens 1129 / 1056, 512 tokens 1889 / 2384; 1024 x 1024, 32 experts, 16
    // pairs each: 103 / 80).
    const size_t wide = (c.wb ? 16 : 32) * 8;
    const bool many = c.pairs >= 6 * (size_t)c.groups && (c.pairs / 16 + c.groups) * ((c.n + wide - 1) / wide) >= 512;
    const int waves = many ? 8 : 4, rows = many ? 16 : 8;
    const size_t per = (size_t)(c.wb ? 16 : 32) * waves, blocks = (c.n + per - 1) / per;
    // A workgroup's start is some microseconds of dependent loads: about eight chunks each while two fill a compute unit (the
    // layer of 256 experts, 64 tokens: 1068 with two blocks of the down projection, 1098 with one; 64 experts of 512, with
    // eight of them and half a workgroup to a compute unit, 82 against 60 with one).
    const size_t busy = std::min(c.pairs, c.pairs / rows + (size_t)c.groups) * blocks;
    a.span = (int)std::max<size_t>(1, std::min({blocks, 8 / nc, busy / 512}));
    a.cols = (int)((blocks + a.span - 1) / a.span);
    const size_t tiles = (c.pairs / rows + (size_t)c.groups + 7) / 8 * 8;
    if (tiles * a.cols > 0x7FFFFFFFull) return -1;
    hipLaunchKernelGGL(jq::moe_mx_prep, dim3((unsigned)c.x_rows, (unsigned)((nc + 3) / 4)), dim3(256), 0, s, c.X, (int)c.k, a.acts);
    auto *kernel = c.wb ? (many ? jq::moe_mx<true, 8, 4> : jq::moe_mx<true, 4, 2>) : (many ? jq::moe_mx<false, 8, 4> : jq::moe_mx<false, 4, 2>);
    hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles * a.cols)), dim3(64 * waves), 0, s, a);
    HIP_TRY(hipGetLastError());
    note_kernel("moe_mx");
    return 0;
}

}  // namespace jqh

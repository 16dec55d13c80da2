// Grouped products of experts with exact operands: Q4_K on split f16 activations (kernels_moe_split16.hpp), MXFP4 on the matrix
// cores' FP4 (kernels_moe_mx.hpp).
#pragma once
#include "core.hpp"
#include "kernels_valu.hpp"

namespace jqh {

struct MoeSplit16Call {
    const uint8_t *const *wa, *const *wb;   // device tables of expert bases: gate and up, or down and null
    size_t row_bytes;
    const float *X;                         // x_rows rows of k
    size_t x_rows;
    const int *gexp, *offsets, *xsel, *yrow;
    int groups;
    size_t pairs;
    float *Y;                               // rows of n; with wb the gated unit's activations
    size_t k, n;
    jq::MoeClamp clamp;
    uint8_t *acts;                          // moe_split16_bytes(x_rows, k), or moe_mx_bytes
    bool few = false;                       // (moe_split16) fewer than 16 routed pairs an expert
};
size_t moe_split16_bytes(size_t rows, size_t k);
bool moe_split16_takes(size_t k, size_t row_bytes, int base_align, size_t rows);
int moe_split16(const MoeSplit16Call &c, hipStream_t s);
size_t moe_mx_bytes(size_t rows, size_t k);
bool moe_mx_takes(size_t n, size_t k, size_t row_bytes, int base_align, size_t rows);
int moe_mx(const MoeSplit16Call &c, hipStream_t s);

}  // namespace jqh

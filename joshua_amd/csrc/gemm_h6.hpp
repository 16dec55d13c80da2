// Products of many activation rows on f16 and FP6 matrix instructions (kernels_mfma_gemm_h6.hpp).
#pragma once
#include "core.hpp"

namespace jqh {

constexpr size_t INT8_GEMM_REC = 9280;  // bytes of the int8 GEMM's record of 16 rows and a super-block, jq::QI_REC: what that GEMM's scratch is counted in

// Device pointers, shapes validated, k and n > 0.  With `swiglu_pairs` the activations are silu(gate) * up over rows of 2 k floats in which
// gate_j and up_j alternate.  -1: the call is outside its reach.
int gemm_h6(uint32_t type, const uint8_t *W, size_t row_bytes, const float *X, float *Y, size_t m, size_t k, size_t n, hipStream_t s,
            const char *name, const char *name_split, bool swiglu_pairs = false);
// Y, rows of n / 2: silu(gate_j . x) (up_j . x) over weight rows gate_j and up_j in turn.  -1: outside its reach (Q4_K only).  2048 x 24576 x 4096,
// us: the product 570 -> 561, the preparation of the down projection that follows 47 -> 33 (Q4_K) and 66 -> 27 (Q6_K).
int gemm_h6_swiglu(uint32_t type, const uint8_t *W, size_t row_bytes, const float *X, float *Y, size_t m, size_t k, size_t n, hipStream_t s);
double gemm_h6_us(size_t m, size_t k, size_t n);  // its time by estimate, scratch as large as it wants

}  // namespace jqh

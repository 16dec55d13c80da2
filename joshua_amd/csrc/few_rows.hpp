// Products of a few activation rows with packed weights (kernels_few_rows.hpp).
#pragma once
#include "core.hpp"

namespace jqh {

// Device pointers, shapes validated, k and n > 0.  -1: the call is outside their reach.
// Up to 16 rows: one launch, no scratch memory.
int few_rows_matmul(uint32_t type, const uint8_t *W, size_t row_bytes, const float *X, float *Y, size_t m, size_t k, size_t n,
                    hipStream_t s);
// More: the activations prepared first, in the call scratch of the stream.
int few_rows_many_matmul(uint32_t type, const uint8_t *W, size_t row_bytes, const float *X, float *Y, size_t m, size_t k, size_t n,
                         hipStream_t s);
double few_rows_many_us(uint32_t type, size_t m, size_t k, size_t n);  // its time by estimate

}  // namespace jqh

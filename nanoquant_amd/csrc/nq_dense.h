// The dense GEMV of several batch rows on the matrix cores (nq_dense.hip).
#pragma once

#include "nq_common.h"

namespace nq {

struct DenseArgs {
    const uint16_t* w;       // [m][n]
    const uint16_t* x;       // [batch][n]
    const uint16_t* norm_w;  // [n] or nullptr
    void* y;                 // [batch][ldy], float (y_f32) or dtype
    float eps;
    int y_f32, batch, n, m, ldy;
};

// Whether the kernel takes these sizes and is the faster one.
bool dense_mfma_applies(int64_t batch, int64_t n);
void launch_dense_mfma(int dtype, const DenseArgs& a, hipStream_t st);

}  // namespace nq

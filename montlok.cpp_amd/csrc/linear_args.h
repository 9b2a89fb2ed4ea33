// Arguments of the linear kernels (linear.hip, linear_split.hip).
#pragma once

#include <cstdint>

#include "mlk_common.h"

namespace mlk {

struct LinearArgs {
    const float* x;
    int64_t rows, K, x_stride;
    const void* w;
    const float* bias;
    int64_t N;
    float* out;
    int64_t out_stride;
    // Optional residual added to the result (out = residual + (x W^T + b),
    // the add as a separate fp32 rounding), rows res_stride apart.
    const float* residual;
    int64_t res_stride;
    // Optional grouped RMSNorm of x before the product (not in every
    // kernel): weight and eps as the rms_norm operator takes them.
    const float* norm_w;
    double norm_eps;
};

// The fp32-weight linear on the bf16 matrix cores (linear_split.hip), for 16-byte aligned rows of x and W.
// _fits: whether its addressing holds the call. _norm: with the grouped RMSNorm of x (group sizes 8, 16, 32, 64;
// K at most 256). _swiglu: W and bias hold 2 N rows, gate then up; out [rows, N] = silu(gate) * up.
bool linear_split_fits(const LinearArgs& p);
void launch_linear_split(const LinearArgs& p, hipStream_t stream);
void launch_linear_split_norm(const LinearArgs& p, int64_t group_size, hipStream_t stream);
bool linear_swiglu_fits(const LinearArgs& p);
void launch_linear_swiglu(const LinearArgs& p, hipStream_t stream);

}  // namespace mlk

// Launcher of the LayerNorm over partial projection sums (layernorm.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace dflash {

// out = LayerNorm(T(T(sum of `splits` fp32 [rows, hidden] partials + bias) + residual)) for
// fp16 / bf16 rows; hidden a multiple of 4, at most 4096, splits 2, 4 or 8; bias,
// residual, gamma, beta and out 4-element aligned, the partials 16-byte aligned.
int launch_partials_layernorm(const float* part, int splits, const void* bias,
                              const void* residual, const void* gamma, const void* beta,
                              void* out, int rows, int hidden, float eps, int dtype,
                              hipStream_t stream);

}  // namespace dflash

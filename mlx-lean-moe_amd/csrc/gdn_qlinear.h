// Host-side pieces the quantized projections share (gdn_qlinear.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gdn {

// y = the sum, in split order, of `splits` (2, 4, 8 or 16) float32 blocks
// partial[splits][count] (16-byte aligned), plus the residual.
int launch_split_sum(const float* partial, int splits, int64_t count, void* y, int y_dtype, const void* residual,
                     hipStream_t s, const char* who);

}  // namespace gdn

// Host-side pieces the quantized projections share (gdn_qlinear.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gdn {

// y = the sum, in split order, of `splits` (2, 4, 8 or 16) float32 blocks
// partial[splits][count] (16-byte aligned), plus the residual.
int launch_split_sum(const float* partial, int splits, int64_t count, void* y, int y_dtype, const void* residual,
                     hipStream_t s, const char* who);

// The kernel of bf16 rows above the decode sizes (gdn_qlinear_mid.hip): whether
// it takes a shape, the workspace its full K split uses, and its launch (which
// splits K only as far as the workspace goes).
bool mid_kernel_takes(int M, int N, int K, int group_size, int sb_dtype, int64_t ws_bytes);
int64_t mid_workspace_bytes(int M, int N, int K, int group_size, int sb_dtype);
int launch_mid(const void* x, const uint32_t* w, const void* scales, const void* biases, int sb_dtype, void* y,
               int y_dtype, const void* residual, int M, int N, int K, int bits, int group_size, void* workspace,
               int64_t ws_bytes, hipStream_t s);

}  // namespace gdn

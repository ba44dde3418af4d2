// Internal interface of the quantization kernels (quant_ops.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace tfcc_rocm {

// The stream, which is idle, goes away: what is kept for its range reductions is given back.
int quantize_release_stream(hipStream_t stream);

}  // namespace tfcc_rocm

// Internal interface of the one-launch LSTM sequence (lstm_sequence.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace tfcc_rocm {

// The stream, which is idle, goes away: no later launch may order itself behind it.
void lstm_sequence_forget_stream(hipStream_t stream);

}  // namespace tfcc_rocm

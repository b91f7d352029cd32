// Internal launch interface of the sampling-distribution kernels (not part of the C ABI).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mvllm {

// One row's parameters, as mvllm_sampling_row of the C ABI.
struct SamplingRow {
  float temperature;  // 0: greedy
  float top_p;        // >= 1: no limit
  int32_t top_k;      // <= 0 or >= vocab: no limit
};

// Rows of one launch set: their parameters are kernel arguments, so a call copies
// nothing to the device.
constexpr int kSamplingRows = 128;

// probs[r] (fp32, v entries, rows contiguous) = the distribution of logits row r under
// params[r] (host array). `workspace`: sampling_workspace_bytes(rows, v) bytes.
hipError_t launch_sampling_probabilities(float* probs, const void* logits, int64_t rows,
                                         int64_t v, int64_t row_stride, int dtype,
                                         const SamplingRow* params, void* workspace,
                                         hipStream_t stream);
uint64_t sampling_workspace_bytes(int64_t rows, int64_t v);
// Longest row served.
int64_t sampling_max_vocab();

}  // namespace mvllm

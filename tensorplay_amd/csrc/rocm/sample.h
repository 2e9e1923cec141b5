// Launcher of the sort-free draw (sample.hip), called by tpr_sample for k > 1024.
#pragma once

#include <hip/hip_runtime.h>

namespace tpr {

int sample_rows(const float* in, long long rows, long long cols, long long row_stride, long long k, float temperature,
                float top_p, const float* u, long long* ids, hipStream_t st);

}  // namespace tpr

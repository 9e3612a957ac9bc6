// Row moves of the cache's tiers (akv_rows_move).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "akv_hip.h"

namespace akv {

constexpr int kRowsMaxJobs = 20;
struct RowsParams {
    akv_rows_job job[kRowsMaxJobs];
    int unit[kRowsMaxJobs];  // bytes (COPY) or elements of 16 source-side vectors (WIDEN) a thread moves at once
    int tile[kRowsMaxJobs];  // rows of a workgroup
    const int64_t *idx;
    int64_t n_idx;
};

hipError_t rows_move_launch(const akv_rows_job *jobs, int n_jobs, const int64_t *idx, int64_t n_idx, hipStream_t s);

}  // namespace akv

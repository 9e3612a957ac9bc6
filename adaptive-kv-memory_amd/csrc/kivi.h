// Parameter block of the KIVI overflow kernel (akv_kivi_append).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "akv_hip.h"

namespace akv {

struct KiviParams {
    akv_kivi_side side[2];
    int B, H, D, in_dt, group_size, view_dt;
    int64_t n;
};

hipError_t kivi_append_launch(const KiviParams &p, int n_sides, hipStream_t s);

}  // namespace akv

// Weight gradients of wide products, see wgrad_wide.hip.
#pragma once

#include "common.h"

namespace mpa {

// Tiles of 256 x 256 (bfloat16; the jobs are valid ones), where their estimated time is below `other_us`: bytes of workspace, 0 where it
// is not; the launch, kNotWide where it is not.
constexpr int kNotWide = -1;
size_t wgrad_wide_bytes(const mpa_wgrad_job* jobs, int n, int64_t T, float other_us);
int wgrad_wide_run(const mpa_wgrad_job* jobs, int n, int64_t T, float other_us, void* workspace, size_t workspace_bytes, hipStream_t stream);

}  // namespace mpa

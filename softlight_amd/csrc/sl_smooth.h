// sl_smooth.h -- host-side launchers of the kernels in sl_smooth.hip.
#pragma once

#include "sl_device.h"

namespace slg {

// Each launcher runs the boundary pass first (p.bounds: W * H float2;
// p.clippedRows: smooth_rows(W, H) words).
size_t smooth_rows(int W, int H);
hipError_t launch_smooth(const SmoothParams& p, hipStream_t s);
hipError_t launch_smooth_backward(const SmoothParams& p, hipStream_t s);

}  // namespace slg

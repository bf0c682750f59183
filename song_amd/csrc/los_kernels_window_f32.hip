// los_kernels_window_f32.hip — the window organisation (los_window.h) of the
// FP32-compensated form. Its tables are made as the sweep kernels' are (contracted
// in FP64, then rounded) and its sums are theirs, operation by operation.
#include <hip/hip_runtime.h>

#include "los_device.h"
#include "los_window.h"

extern "C" hipError_t los_launch_window_prep_f32(const los_params *P, hipStream_t s)
{
  return launch_window_prep<2>(P, s);
}

extern "C" hipError_t los_launch_window_f32(const los_params *P, int kt, int nl, hipStream_t s)
{
  return launch_window<2>(P, kt, nl, s);
}

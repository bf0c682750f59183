// los_kernels_window_fma.hip — the window organisation (los_window.h) of the FP64
// form with FMA.
#include <hip/hip_runtime.h>

#include "los_device.h"
#include "los_window.h"

extern "C" hipError_t los_launch_window_prep_fma(const los_params *P, hipStream_t s)
{
  return launch_window_prep<1>(P, s);
}

extern "C" hipError_t los_launch_window_fma(const los_params *P, int kt, int nl, hipStream_t s)
{
  return launch_window<1>(P, kt, nl, s);
}

// los_kernels_window_fma.hip — the window organisation (los_window.h) of the FP64
// form with FMA: the plain form's sums over the same tables, contracted.
#include <hip/hip_runtime.h>

#include "los_device.h"
#include "los_window.h"

extern "C" hipError_t los_launch_window_fma(const los_params *P, int kt, int nl, hipStream_t s)
{
  return launch_window<true>(P, kt, nl, s);
}

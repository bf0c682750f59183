// los_kernels_window.hip — the window organisation (los_window.h): its tables and
// the plain FP64 form. Compiled with -ffp-contract=off: per element the
// reference's operations in its order.
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include "los_device.h"
#include "los_window.h"

extern "C" {

hipError_t los_launch_window_prep(const los_params *P, hipStream_t s)
{
  return launch_window_prep<0>(P, s);
}

int los_window_jrows(int NL, int Lmax, int m) { return win_jrows(NL, Lmax, m); }

int los_window_rows_fit(int has_T, int has_P, int LmaxT, int LmaxP)
{
  return window_rows_fit(has_T, has_P, LmaxT, LmaxP) ? 1 : 0;
}

hipError_t los_launch_window_exact(const los_params *P, int kt, int nl, hipStream_t s)
{
  return launch_window<0>(P, kt, nl, s);
}

}  // extern "C"

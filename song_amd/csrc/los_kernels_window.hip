// los_kernels_window.hip — the window organisation (los_window.h) of the plain
// FP64 form. Compiled with -ffp-contract=off: per element the reference's
// operations in its order.
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include "los_device.h"
#include "los_window.h"

extern "C" {

hipError_t los_launch_window_prep(const los_params *P, hipStream_t s)
{
  if (P->F == 0 || P->ntau == 0) return hipSuccess;
  const dim3 grid((unsigned)(P->k_npad / 64), (unsigned)((P->ntau + 63) / 64));
  hipLaunchKernelGGL(los_window_prep, grid, dim3(256), 0, s, *P);
  return hipGetLastError();
}

int los_window_jrows(int NL, int Lmax, int m) { return win_jrows(NL, Lmax, m); }

int los_window_rows_fit(int has_T, int has_P, int LmaxT, int LmaxP)
{
  return window_rows_fit(has_T, has_P, LmaxT, LmaxP) ? 1 : 0;
}

// kt fine k3 and nl (l,m) offsets per wave
hipError_t los_launch_window_exact(const los_params *P, int kt, int nl, hipStream_t s)
{
  switch (kt * 64 + nl) {
    case 64 * 64 + 8: return launch_window_exact<8, 1>(P, s);
    case 32 * 64 + 8: return launch_window_exact<8, 2>(P, s);
    case 16 * 64 + 8: return launch_window_exact<8, 4>(P, s);
    default: return hipErrorInvalidValue;
  }
}

}  // extern "C"

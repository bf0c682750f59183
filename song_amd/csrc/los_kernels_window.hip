// los_kernels_window.hip — the window organisation (los_window.h): its tables and
// the plain FP64 form. Compiled with -ffp-contract=off: per element the
// reference's operations in its order.
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include "los_device.h"
#include "los_window.h"

// The tables of the window kernels. A workgroup makes 64 ranks x 64 time steps:
// it reads the sources along tau (their layout in HBM) and writes along the
// ranks through an LDS transpose.
__global__ void __launch_bounds__(256) los_window_prep(los_params P)
{
  __shared__ double tile[64][65];
  __shared__ long r_off[64];
  __shared__ int r_nc[64];
  __shared__ double r_aw[64], r_bw[64], r_ca[64], r_cb[64], r_h[64];
  const int rb = blockIdx.x, r0 = rb * 64, t0 = blockIdx.y * 64;
  const int tid = threadIdx.x, lane = tid & 63, grp = tid >> 6;
  double kf = 0;
  {
    const int r = min(r0 + lane, P.F - 1);
    const int f = P.korder[r];
    kf = P.kf[f];
    if (tid < 64) {
      const los_pair pr = P.pairs[P.fpair[f]];
      const int br = P.fbr[f];
      const double *kc = P.kc + pr.kc_off;
      const double ks = P.kf[P.fsrc[f]];
      const double h = kc[br + 1] - kc[br];
      const double bw = (ks - kc[br]) / h;
      const double aw = 1 - bw;
      r_off[tid] = pr.src_off + (long)br * P.ntau;
      r_nc[tid] = pr.nc;
      r_h[tid] = h;
      r_aw[tid] = aw;
      r_bw[tid] = bw;
      r_ca[tid] = aw * aw * aw - aw;
      r_cb[tid] = bw * bw * bw - bw;
    }
  }
  for (int i = grp; i < 64; i += 4) {
    const int t = t0 + i;
    if (t >= P.ntau) break;
    const double x = kf * P.t0mt[t];
    const int ix = (int)(x / P.xx_step);
    const long o = ((long)rb * P.ntau + t) * 64 + lane;
    P.wix[o] = ix;
    P.waj[o] = (P.xx[ix + 1] - x) / P.xx_step;
  }
  const int tr = min(t0 + lane, P.ntau - 1);
  __syncthreads();
  for (int set = 0; set < 2; ++set) {
    if (set ? !P.has_T : !(P.has_E || P.has_B)) continue;
    const int Lmax = set ? P.LmaxT : P.LmaxP, nf = set || !P.has_B ? 1 : 2;
    for (int mi = 0; mi < P.m_size; ++mi) {
      const int m = P.m_of_mi[mi], nr = win_jrows(P, set, m), rows = nr * nf;
      double *out = P.wsrc + P.wsrc_off[set][mi] + (long)rb * P.ntau * rows * 64;
      for (int row = 0; row < rows; ++row) {
        const int L = Lmax - nr + 1 + row / nf;
        const bool live = L >= m;
        const int tp = !live ? 0 : set ? P.srcT[L][mi] : row % nf ? P.srcB[L][mi] : P.srcE[L][mi];
#pragma unroll 4
        for (int i = grp; i < 64; i += 4) {
          const double *S = P.src + r_off[i] + (long)tp * r_nc[i] * P.ntau + tr;
          double v;
          if (P.cubic_k3) {
            const double *D = P.dd + (S - P.src);
            v = r_aw[i] * S[0] + r_bw[i] * S[P.ntau] +
                (r_ca[i] * D[0] + r_cb[i] * D[P.ntau]) * r_h[i] * r_h[i] / 6.0;
          } else {
            v = r_aw[i] * S[0] + r_bw[i] * S[P.ntau];
          }
          tile[i][lane] = live ? v : 0.;
        }
        __syncthreads();
        for (int i = grp; i < 64; i += 4)
          if (t0 + i < P.ntau) out[((long)(t0 + i) * rows + row) * 64 + lane] = tile[lane][i];
        __syncthreads();
      }
    }
  }
}

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

hipError_t los_launch_window_exact(const los_params *P, int kt, int nl, hipStream_t s)
{
  return launch_window<false>(P, kt, nl, s);
}

}  // extern "C"

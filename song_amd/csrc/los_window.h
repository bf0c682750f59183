// los_window.h — LOS integral with one fine k3 per lane and the J rows of the
// wave's multipoles staged in LDS, "window" organisation.
//
// A wave (one workgroup) owns a tile of KT = 64/G neighbouring fine k3 (sorted
// work order, one job), one m, one of the two field sets (T, or E and B) and
// a group of consecutive l: lane g*KT + i works on k3 i of the tile and on the l
// numbers j*G + g. At a time step the index_x of neighbouring k3 fall
// within a few x points of each other, so a window of LOS_WIN_W x points of a J
// row serves every lane of the wave for several steps: the wave copies the
// windows of its rows from the k-lane table [jt][L][lm][x] into its own LDS, and
// each lane reads its two nodes there. The list of windows of a tile (first
// step, first x point) depends on the k3 and time grids only and is made when
// the batch is loaded. The reference's skip (index_x < index_xmin_J,
// source/transfer2.c:2232) is tested only in the steps where it can differ
// between the rows and k3 of an l. The next step's sources are in flight while a
// step runs, and no other wave touches the LDS block, so there are no barriers.
//
// Per element the operations are those of the reference, in its order (compile
// without contraction for the plain FP64 form): per time step the integrand of
// each integral is the sum over L of (a_J J_i + (1 - a_J) J_{i+1}) S, the
// integral adds integrand x dtau, E = EE + EB (EB only for m != 0), B = EE -
// EB, then x 1/2, / 4, / (2l+1), / 2 (source/transfer2.c:2259-2329,
// :1861-2098).
//
// What bounds it, and the choices (32 x 32 pairs, T+E+B, 600 steps, 96 l, 41,759
// fine k3: the sweep kernel's best tile took 64.1 ms): 30.0 ms, of which the FP64
// instructions alone are 15.7 ms (9.4e9 of them) and the LDS reads 15 ms (two
// nodes of 8 bytes at 121 B/clk/CU); its L2 misses are 139 GB, 4.5 TB/s, against
// 282 GB of the sweep kernel, mostly sources fetched by every l group of a tile.
// - 32 x points: 0.12 windows a step for 64 k3 (16 points: 0.65, 75 ms). As
//   16-byte pairs the reads are cheaper but half the points fit: 32.0 to 36.2 ms.
// - E and B in one wave (both J types, 4 l): one pass over the sources; two passes
//   (8 l each) drift apart between the l groups, 45 against 44 ms.
// - One wave a workgroup: 6 waves sharing a tile's sources with a barrier a step
//   took 86 ms, without one 58 ms (the slots wait for the longest l).
// - The sources one step ahead in registers: 45 ms against 53 ms without.
// - Tiles of 64, 32 or 16 k3: the sparser the k3, the fewer share a window; the
//   tuner picks (9,404 k3, T only, 48 l: 1.75, 0.89, 0.34 ms against the sweep
//   kernel's 1.11 ms; 14,753 k3 up to 0.2/Mpc: 44.7, 26.6, 27.1 against 53.1 ms).
// The fast forms add a term to the running sums at a time, 32 steps a partial sum.
// 11,178 k3, T+E+B, 96 l, tiles of 64, 32, 16 k3: with FMA 21.1, 15.1, 12.4 ms against
// 22.7 to 29.5 ms of the sweep kernel's tiles; FP32-compensated 15.9, 9.9, 8.2 ms
// against 17.7 to 20.4 ms (half the LDS and table bytes, as many instructions).
//
// Tables, by blocks of 64 sorted ranks (r = 64 rb + lane), so that a wave's
// stream through the time steps is contiguous:
//   wix[rb][t][64], waj[rb][t][64]    index_x and a_J (source/transfer2.c:2195-2202)
//   wsrc: per field set and m (wsrc_off), [rb][t][row][64]: the sources interpolated
//         in k3 (source/transfer2.c:2700-2706), row = (L - L0) of T (or of E without
//         B), 2 (L - L0) of E and 2 (L - L0) + 1 of B; L0: win_jrows
#pragma once

#include <hip/hip_runtime.h>

#include <climits>
#include <type_traits>

#include "los_device.h"
#include "los_policy.h"

typedef double win_d2 __attribute__((ext_vector_type(2)));

// One value of a table of R at a lane's byte offset plus a wave-uniform one.
template <class R>
__device__ __forceinline__ R win_load(__amdgpu_buffer_rsrc_t r, unsigned lane, int off)
{
  if constexpr (sizeof(R) == 8)
    return __builtin_bit_cast(R, __builtin_amdgcn_raw_buffer_load_b64(r, lane, off, 0));
  else
    return __builtin_bit_cast(R, __builtin_amdgcn_raw_buffer_load_b32(r, lane, off, 0));
}

// Forms: 0 plain FP64, 1 FP64 with FMA, 2 FP32-compensated.
template <int FORM>
using win_real = std::conditional_t<FORM == 2, float, double>;

// Running sums of a pass: of the plain form as the reference adds them; of the
// others over 32 time steps, then into the form's sum (of FP32 compensated).
template <int FORM>
struct WinAcc {
  typedef std::conditional_t<FORM == 2, StreamFP32C, StreamFP64> Pol;
  typename Pol::acc_t a;
  win_real<FORM> p;
  __device__ __forceinline__ void fold()
  {
    Pol::fold(a, p);
    p = 0;
  }
  __device__ __forceinline__ double value() const { return Pol::value(a); }
};
template <>
struct WinAcc<0> {
  double s;
  __device__ __forceinline__ void fold() {}
  __device__ __forceinline__ double value() const { return s; }
};

// Raw buffer resource over `bytes` bytes at base (32-bit data, no swizzle): a load
// adds the lane's byte offset and a wave-uniform one.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t win_rsrc(const void *base, unsigned bytes)
{
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes,
                                           0x00020000);
}

// Wave-uniform read of memory that the kernel does not write (a scalar load).
template <class T>
__device__ __forceinline__ T win_uniform(const T *p, long i)
{
  typedef const __attribute__((address_space(4))) T *cptr;
  return ((cptr)(unsigned long long)p)[i];
}

// Orders the wave's LDS writes and reads of one window (one wave: the hardware
// keeps its LDS accesses in order, this keeps the compiler's).
__device__ __forceinline__ void win_fence()
{
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// J rows of the instance that serves a (field set, m): the kernel of NL = largest
// L + 1 has instances for NL, NL - 1 and NL - 2 rows, L = Lmax - rows + 1 .. Lmax;
// rows below m are zero in the J table.
__host__ __device__ static inline int win_jrows(int NL, int Lmax, int m)
{
  const int nr = Lmax - m + 1, least = NL > 2 ? NL - 2 : 1;
  return nr > least ? nr : least;
}
__device__ __forceinline__ int win_jrows(const los_params &P, int set, int m)
{
  return win_jrows(max(P.LmaxT, P.LmaxP) + 1, set ? P.LmaxT : P.LmaxP, m);
}

// The lanes' positions and (l,m) of a wave.
struct WinWave {
  const int *plan;     // windows of the tile: {first step, 2 x first x point + partial}
  double kmin, kmax;   // smallest and largest k3 of the tile
  int rb, rl;          // rank block of the tile and this lane's place in it
  int grp;             // this lane's l group
  const int *lms;      // the wave's (l,m) offsets, -1 padding
  int lm0;             // the first of them
};

// One pass over the time steps: for each l of the wave the rows L = L0 ..
// L0+NR-1 of NT J types (jt[0], jt[1]) against NF source fields; the integral of
// type y and field f goes to acc[j][y*NF + f], without the final 1/2 (SKIP: the
// last of them is not wanted). src: the rank block's sources, NR*NF rows of 64
// per step; field f of J row q is source row q*NF + f.
// The other forms: acc[j][f] is E (f = 0) and B of an l, or its only integral, and
// the sources carry the trapezoid weight. The operations are those of the form's
// sweep kernel in its order, so that both give the same bits from the same tables
// (SKIP: no B sources into E; of one field, a product rounded before it is added).
template <int FORM, int NR, int NF, int NT, bool SKIP, int NLB, int G, int NA,
          class R = win_real<FORM>>
__device__ __forceinline__ void win_pass(const los_params &P, const WinWave &W, R *win, int *xms,
                                         const int (&jt)[NT], int L0, const R *src,
                                         WinAcc<FORM> (&acc)[NLB][NA])
{
  constexpr bool PLAIN = FORM == 0;
  static_assert(NA == (PLAIN ? NT * NF : NF), "integrals of an l");
  // a window is 32 points; 16 lanes (FP64) or 8 stage one with 16 bytes each
  constexpr int LR = 2 * (int)sizeof(R), SR = 64 / LR, RB = 64 * (int)sizeof(R);
  constexpr int NLT = NLB * G, RL = NR * NT, ROWS = RL * NLT, NS = (ROWS + SR - 1) / SR;
  const int lane = threadIdx.x;
#pragma unroll
  for (int j = 0; j < NLB; ++j)
#pragma unroll
    for (int f = 0; f < NA; ++f) acc[j][f] = WinAcc<FORM>{};

  // Steps of each l, lane i searching for l number i of the wave (index_x falls
  // with t): before tsafe every row lives for every k3 of the tile, from tend on
  // none does. Rows with no point in the table are zero there and need no test.
  int tend[NLB], tsafe[NLB], tmax = 0;
  {
    int send = 0, ssafe = INT_MAX;
    const int lmr = lane < NLT ? W.lms[lane] : -1;
    if (lmr >= 0) {
      int xlo = INT_MAX, xhi = -1;
#pragma unroll
      for (int y = 0; y < NT; ++y)
#pragma unroll
        for (int q = 0; q < NR; ++q) {
          const int x = P.xmin[((long)jt[y] * P.L_size + L0 + q) * P.n_lm + lmr];
          xlo = min(xlo, x);
          xhi = x < P.X ? max(xhi, x) : xhi;
        }
      auto search = [&](double k, int x) {
        int lo = 0, hi = P.ntau;
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if ((int)(k * P.t0mt[mid] / P.xx_step) >= x) lo = mid + 1; else hi = mid;
        }
        return lo;
      };
      send = search(W.kmax, xlo);
      ssafe = search(W.kmin, xhi);
    }
#pragma unroll
    for (int j = 0; j < NLB; ++j) {
      tend[j] = 0;
      tsafe[j] = INT_MAX;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        tend[j] = max(tend[j], __builtin_amdgcn_readlane(send, j * G + g));
        tsafe[j] = min(tsafe[j], __builtin_amdgcn_readlane(ssafe, j * G + g));
      }
      tsafe[j] = min(tsafe[j], tend[j]);
      tmax = max(tmax, tend[j]);
    }
  }
  if (tmax == 0) return;

  // staged row s*SR + lane/LR = (l number) * RL + y * NR + q, 16 bytes of x points
  const unsigned rowx = (unsigned)P.X * sizeof(R), typex = (unsigned)P.L_size * P.n_lm * rowx;
  const __amdgpu_buffer_rsrc_t Jr = win_rsrc(P.Jk, P.Jk_bytes);
  unsigned voff[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int ri = min(s * SR + lane / LR, ROWS - 1);
    const int li = ri / RL, yq = ri - li * RL, y = yq / NR, q = yq - y * NR;
    int lmr = W.lms[li];
    lmr = lmr < 0 ? W.lm0 : lmr;
    if (s * SR + lane / LR < ROWS && lane % LR == 0)
      xms[ri] = P.xmin[((long)(NT > 1 && y ? jt[NT - 1] : jt[0]) * P.L_size + L0 + q) * P.n_lm +
                       lmr];
    voff[s] = (unsigned)(NT > 1 && y ? jt[NT - 1] : jt[0]) * typex +
              (unsigned)((L0 + q) * P.n_lm + lmr) * rowx + lane % LR * 16u;
  }
  const long tb = (long)W.rb * P.ntau * 64;
  const __amdgpu_buffer_rsrc_t Ir = win_rsrc(P.wix + tb, (unsigned)P.ntau * 256u),
                               Ar = win_rsrc((const R *)P.waj + tb, (unsigned)P.ntau * RB),
                               Sr = win_rsrc(src, (unsigned)P.ntau * (NR * NF * RB));
  const unsigned rl4 = W.rl * 4u, rlr = W.rl * (unsigned)sizeof(R);
  int ixn = 0;
  R an = 0, svn[NF][NR];
  // index_x, a_J and the sources of step t
  auto load = [&](int t) {
    ixn = (int)__builtin_amdgcn_raw_buffer_load_b32(Ir, rl4, t * 256, 0);
    an = win_load<R>(Ar, rlr, t * RB);
    const int so = t * (NR * NF * RB);
#pragma unroll
    for (int q = 0; q < NR; ++q)
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const int o = (q * NF + f) * RB, hi = o & ~4095;
        svn[f][q] = win_load<R>(Sr, rlr + (o - hi), so + hi);
      }
  };
  auto fold = [&]() {
#pragma unroll
    for (int j = 0; j < NLB; ++j)
#pragma unroll
      for (int f = 0; f < NA; ++f) acc[j][f].fold();
  };

  int i = 0;
  int bt = win_uniform(W.plan, 0), by = win_uniform(W.plan, 1);
  load(0);
  while (bt < tmax) {
    ++i;
    const int nbt = win_uniform(W.plan, 2 * i), nby = win_uniform(W.plan, 2 * i + 1);
    const int x0 = by >> 1;
    const bool partial = by & 1;
    {
      win_d2 w[NS];
#pragma unroll
      for (int s = 0; s < NS; ++s)
        w[s] = __builtin_bit_cast(
            win_d2, __builtin_amdgcn_raw_buffer_load_b128(Jr, voff[s], x0 * (int)sizeof(R), 0));
#pragma unroll
      for (int s = 0; s < NS; ++s)
        if (s * SR + SR - 1 < ROWS || s * SR + lane / LR < ROWS) ((win_d2 *)win)[s * 64 + lane] = w[s];
      __builtin_amdgcn_sched_barrier(0);
    }
    win_fence();
    const int te = min(max(nbt, bt + 1), tmax);
    for (int t = bt; t < te; ++t) {
      const int ix = ixn;
      const R a = an;
      R sv[NF][NR];
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int q = 0; q < NR; ++q) sv[f][q] = svn[f][q];
      const int tn = t + 1 < te ? t + 1 : nbt;
      if (tn < tmax) load(tn);
      const int cell = ix - x0;
      const R *wl = win + W.grp * (RL * LOS_WIN_W) + cell;
      if (!partial || (unsigned)cell < LOS_WIN_W - 1) {
#pragma unroll
        for (int j = 0; j < NLB; ++j) {
          if (t >= tend[j]) continue;
          const bool safe = t < tsafe[j];
          if constexpr (PLAIN) {
            const double ar = 1 - a, dt = win_uniform(P.dtau, t);
#pragma unroll
            for (int y = 0; y < NT; ++y) {
              __builtin_amdgcn_sched_barrier(0);
              const double *wj = wl + (j * G * RL + y * NR) * LOS_WIN_W;
              double v[NF];
              if (safe) {
                // the sum starts with its first term, not with 0 + it: that can only
                // turn a +0 into a -0, which adds the same to acc (never -0 itself)
#pragma unroll
                for (int q = 0; q < NR; ++q) {
                  const double Jv = a * wj[q * LOS_WIN_W] + ar * wj[q * LOS_WIN_W + 1];
#pragma unroll
                  for (int f = 0; f < NF; ++f)
                    if (!(SKIP && y == NT - 1 && f == NF - 1))
                      v[f] = q == 0 ? Jv * sv[f][q] : v[f] + Jv * sv[f][q];
                }
              } else {
                // some row is dead (index_x < index_xmin_J) for some k3: J = 0 there
                const int *xj = xms + W.grp * RL + j * (G * RL) + y * NR;
#pragma unroll
                for (int q = 0; q < NR; ++q) {
                  double Jv = a * wj[q * LOS_WIN_W] + ar * wj[q * LOS_WIN_W + 1];
                  Jv = ix >= xj[q] ? Jv : 0.;
#pragma unroll
                  for (int f = 0; f < NF; ++f)
                    if (!(SKIP && y == NT - 1 && f == NF - 1))
                      v[f] = q == 0 ? Jv * sv[f][q] : v[f] + Jv * sv[f][q];
                }
              }
#pragma unroll
              for (int f = 0; f < NF; ++f)
                if (!(SKIP && y == NT - 1 && f == NF - 1)) acc[j][y * NF + f].s += v[f] * dt;
            }
          } else {
            __builtin_amdgcn_sched_barrier(0);
            const R *wj = wl + j * G * RL * LOS_WIN_W;
            const int *xj = xms + W.grp * RL + j * (G * RL);
            auto fma = [](R x, R y, R z) { return __builtin_elementwise_fma(x, y, z); };
            auto node = [&](int row, bool live) {
              const R j0 = wj[row * LOS_WIN_W], j1 = wj[row * LOS_WIN_W + 1];
              const R v = fma(a, j0 - j1, j1);
              return live || ix >= xj[row] ? v : (R)0;
            };
            auto sum = [&](bool live) {
#pragma clang fp contract(off)
#pragma unroll
              for (int q = 0; q < NR; ++q) {
                const R Je = node(q, live);
                R &pE = acc[j][0].p, &pB = acc[j][NA - 1].p;
                if constexpr (NT == 1) {
                  pE = SKIP ? pE + Je * sv[0][q] : fma(Je, sv[0][q], pE);
                } else {
                  const R Jm = node(NR + q, live), sE = sv[0][q], sB = sv[NF - 1][q];
                  pE += SKIP ? Je * sE : fma(Je, sE, Jm * sB);
                  pB += fma(Je, sB, -(Jm * sE));
                }
              }
            };
            if (safe)
              sum(true);
            else
              sum(false);
          }
        }
      }
      // the same 32 steps a sum as in the sweep kernel, once all windows of the
      // last of them are done
      if (!PLAIN && (t & 31) == 31 && tn != t) fold();
    }
    win_fence();
    bt = nbt;
    by = nby;
  }
  fold();
}

// One wave: the integrals of one field set and its outputs. Set 1: T, NLT l
// numbers; set 0: E and B, half as many with twice the rows (EE: the E and B
// sources into E and B; EB: the E sources into B and, for m != 0, the B sources
// into E).
template <int FORM, int NR, int NLT, int G, class R = win_real<FORM>>
__device__ __forceinline__ void win_item(const los_params &P, const WinWave &W, R *win,
                                         int *xms, const los_tile *tile, int set, int mi)
{
  const int m = P.m_of_mi[mi];
  const int L0 = (set ? P.LmaxT : P.LmaxP) - NR + 1;
  const bool two = !set && P.has_B;
  const R *src =
      (const R *)P.wsrc + P.wsrc_off[set][mi] + (long)W.rb * P.ntau * (NR * (two ? 2 : 1)) * 64;
  auto store = [&](auto &acc) {
    constexpr int NLB = sizeof(acc) / sizeof(acc[0]), N = sizeof(acc[0]) / sizeof(WinAcc<FORM>);
    const int i = threadIdx.x & (64 / G - 1);
    const int pos0 = win_uniform(&tile->pos0, 0), npos = win_uniform(&tile->npos, 0);
    const los_job job = P.jobs[win_uniform(P.pos_job, pos0)];
    const bool valid = i < npos;
    const long ocell = job.obase + P.ocol[pos0 + min(i, npos - 1)];
#pragma unroll
    for (int j = 0; j < NLB; ++j) {
      const int lm = W.lms[j * G + W.grp];
      if (!valid || lm < 0 || lm >= job.n_lm) continue;
      const double den = 2. * P.l_of[lm] + 1;
      double *o = P.out + ocell + (long)lm * job.ostride;
      double *oT = o + (long)job.ttT * job.ostride, *oE = o + (long)job.ttE * job.ostride,
             *oB = o + (long)job.ttB * job.ostride;
      auto scaled = [&](double v) {
        v /= 4.;
        v /= den;
        v /= 2.;
        return v;
      };
      double h[N];
#pragma unroll
      for (int f = 0; f < N; ++f)
        h[f] = acc[j][f].value() * 0.5;
      if (N == 1) {
        *(set ? oT : oE) = scaled(set ? h[0] : h[0] + 0.);
      } else {
        if (P.has_E) *oE = scaled(h[0] + (N == 4 && m != 0 ? h[N - 1] : 0.));
        *oB = scaled(h[1 % N] - (N == 4 ? h[2 % N] : 0.));
      }
    }
  };
  if (two && P.jEB >= 0) {
    WinAcc<FORM> acc[NLT / 2 / G][FORM == 0 ? 4 : 2];
    const int jt[2] = {P.jEE, P.jEB};
    if (m != 0)
      win_pass<FORM, NR, 2, 2, false, NLT / 2 / G, G>(P, W, win, xms, jt, L0, src, acc);
    else
      win_pass<FORM, NR, 2, 2, true, NLT / 2 / G, G>(P, W, win, xms, jt, L0, src, acc);
    store(acc);
  } else {
    WinAcc<FORM> acc[NLT / G][1];
    const int jt[1] = {set ? P.jTT : P.jEE};
    if (FORM == 0 || set)
      win_pass<FORM, NR, 1, 1, false, NLT / G, G>(P, W, win, xms, jt, L0, src, acc);
    else
      win_pass<FORM, NR, 1, 1, FORM != 0, NLT / G, G>(P, W, win, xms, jt, L0, src, acc);
    store(acc);
  }
}

// Workgroup b runs on XCD b % 8; q = b / 8 walks that XCD's items: the field
// sets and m (which share neither sources nor J rows) outermost, then the
// XCD's tiles, costliest first, then the l groups, so that the waves running
// together read the sources of a few neighbouring tiles and the same stretch
// of their J rows through the XCD's L2.
template <int FORM, int NL, int NLT, int G>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
los_window(los_params P)
{
  typedef win_real<FORM> R;
  constexpr int KT = 64 / G;
  __shared__ alignas(16) R win[NL * NLT * LOS_WIN_W];  // windows of the wave's rows
  __shared__ int xms[NL * NLT];                        // and their first live x points
  const int xcd = blockIdx.x & 7;
  int q = blockIdx.x >> 3;
  const int nt = P.xcd_tile[xcd + 1] - P.xcd_tile[xcd];
  int set = P.has_E || P.has_B ? 0 : 1, mi = 0, ng = 0;
  for (;;) {
    ng = P.wgrp_off[set][mi + 1] - P.wgrp_off[set][mi];
    if (q < nt * ng) break;
    q -= nt * ng;
    if (++mi < P.m_size) continue;
    mi = 0;
    if (++set > 1 || !P.has_T) return;
  }
  const int tq = q / ng, g = P.wgrp_off[set][mi] + q - tq * ng;
  const int tile = P.xcd_tile[xcd + 1] - 1 - tq;
  const int pos0 = win_uniform(&P.tiles[tile].pos0, 0), npos = win_uniform(&P.tiles[tile].npos, 0);
  const int lane = threadIdx.x;
  const int r = P.rank_of_f[P.forder[pos0 + min(lane & (KT - 1), npos - 1)]];
  WinWave W;
  W.lms = P.wgrp[set] + (long)g * (set || !P.has_B ? NLT : NLT / 2);
  W.lm0 = win_uniform(W.lms, 0);
  W.grp = lane / KT;
  W.rb = __builtin_amdgcn_readfirstlane(r >> 6);
  W.rl = r & 63;
  W.kmin = win_uniform(P.kf, win_uniform(P.forder, pos0));
  W.kmax = win_uniform(P.kf, win_uniform(P.forder, pos0 + npos - 1));
  W.plan = (const int *)(P.wplan + win_uniform(P.wplan_off, tile));
  const int nr = win_jrows(NL, set ? P.LmaxT : P.LmaxP, P.m_of_mi[mi]);
  if (nr == NL)
    win_item<FORM, NL, NLT, G>(P, W, win, xms, P.tiles + tile, set, mi);
  else if (NL > 1 && nr == NL - 1)
    win_item<FORM, (NL > 1 ? NL - 1 : 1), NLT, G>(P, W, win, xms, P.tiles + tile, set, mi);
  else if (NL > 2)
    win_item<FORM, (NL > 2 ? NL - 2 : 1), NLT, G>(P, W, win, xms, P.tiles + tile, set, mi);
}

// Whether the window kernels cover a batch's multipoles: they have instances
// for NL, NL - 1 and NL - 2 rows, the last also for larger m (rows L < m are
// zero), so a field's rows 0 .. Lmax may be at most two fewer than the other's.
static inline bool window_rows_fit(int has_T, int has_P, int LmaxT, int LmaxP)
{
  const int NL = (LmaxT > LmaxP ? LmaxT : LmaxP) + 1;
  const int least = NL > 2 ? NL - 2 : 1;
  return (!has_T || LmaxT + 1 >= least) && (!has_P || LmaxP + 1 >= least);
}

// P->tiles / P->xcd_tile: tiles of at most 64/G positions; P->wgrp: groups of NLT
// (l,m) offsets, of NLT/2 for E and B with B sources.
template <int FORM, int NLT, int G>
static hipError_t launch_window(const los_params *P, hipStream_t s)
{
  if (P->n_pos == 0 || P->n_lm_max == 0) return hipSuccess;
  long most = 0, groups = 0;
  for (int x = 0; x < 8; ++x) {
    const long n = P->xcd_tile[x + 1] - P->xcd_tile[x];
    most = n > most ? n : most;
  }
  if (P->has_E || P->has_B) groups += P->wgrp_off[0][P->m_size];
  if (P->has_T) groups += P->wgrp_off[1][P->m_size];
  const long grid = 8 * most * groups;
  if (grid == 0) return hipSuccess;
  if (grid > 0x7fffffffL) return hipErrorInvalidValue;
  switch ((P->LmaxT > P->LmaxP ? P->LmaxT : P->LmaxP) + 1) {
#define LOS_WN(n)                                                                              \
  case n:                                                                                      \
    hipLaunchKernelGGL((los_window<FORM, n, NLT, G>), dim3((unsigned)grid), dim3(64), 0, s, *P); \
    break;
    LOS_WN(1) LOS_WN(2) LOS_WN(3) LOS_WN(4) LOS_WN(5) LOS_WN(6) LOS_WN(7) LOS_WN(8)
#undef LOS_WN
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// kt fine k3 and nl (l,m) offsets per wave
template <int FORM>
static hipError_t launch_window(const los_params *P, int kt, int nl, hipStream_t s)
{
  switch (kt * 64 + nl) {
    case 64 * 64 + 8: return launch_window<FORM, 8, 1>(P, s);
    case 32 * 64 + 8: return launch_window<FORM, 8, 2>(P, s);
    case 16 * 64 + 8: return launch_window<FORM, 8, 4>(P, s);
    default: return hipErrorInvalidValue;
  }
}

// The tables of the window kernels. A workgroup makes 64 ranks x 64 time steps:
// it reads the sources along tau (their layout in HBM) and writes along the
// ranks through an LDS transpose. The fast forms' sources carry the
// trapezoid weight.
template <int FORM, class R = win_real<FORM>>
__global__ void __launch_bounds__(256) los_window_prep(los_params P)
{
  __shared__ R tile[64][65];
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
    ((R *)P.waj)[o] = (R)((P.xx[ix + 1] - x) / P.xx_step);
  }
  const int tr = min(t0 + lane, P.ntau - 1);
  const double dt = P.dtau[tr];
  __syncthreads();
  for (int set = 0; set < 2; ++set) {
    if (set ? !P.has_T : !(P.has_E || P.has_B)) continue;
    const int Lmax = set ? P.LmaxT : P.LmaxP, nf = set || !P.has_B ? 1 : 2;
    for (int mi = 0; mi < P.m_size; ++mi) {
      const int m = P.m_of_mi[mi], nr = win_jrows(P, set, m), rows = nr * nf;
      R *out = (R *)P.wsrc + P.wsrc_off[set][mi] + (long)rb * P.ntau * rows * 64;
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
          if (FORM != 0) v = v * dt;
          tile[i][lane] = (R)(live ? v : 0.);
        }
        __syncthreads();
        for (int i = grp; i < 64; i += 4)
          if (t0 + i < P.ntau) out[((long)(t0 + i) * rows + row) * 64 + lane] = tile[lane][i];
        __syncthreads();
      }
    }
  }
}

template <int FORM>
static hipError_t launch_window_prep(const los_params *P, hipStream_t s)
{
  if (P->F == 0 || P->ntau == 0) return hipSuccess;
  const dim3 grid((unsigned)(P->k_npad / 64), (unsigned)((P->ntau + 63) / 64));
  hipLaunchKernelGGL(los_window_prep<FORM>, grid, dim3(256), 0, s, *P);
  return hipGetLastError();
}

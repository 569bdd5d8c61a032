// The z-direction kernels of otbl_zteam.h for a range of row lengths: one
// translation unit per range (otbl_zteam_*.hip), so that the lengths compile
// in parallel.  A workgroup is one wavefront: its teams share nothing, and
// single wavefronts pack a CU's LDS and registers tightest.
#pragma once
#include "otbl_kcommon.h"
#include "otbl_zteam.h"

namespace otbl {

// this lane's team and its row; false for idle lanes and rows past the last
template <int N> struct TeamRow {
  int t, team, row0, row; // row0: the wavefront's first
  __device__ __forceinline__ bool init(int nrows) {
    using Z = ZRow<N>;
    team = threadIdx.x / Z::G;
    t = threadIdx.x - team * Z::G;
    row0 = blockIdx.x * Z::T;
    row = row0 + team;
    return team < Z::T && row < nrows;
  }
};

// maximum over a team, in its lane 0
template <int G, typename R> __device__ __forceinline__ R team_max(R v, int t) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
    if (o < G) {
      const R w = __shfl_down(v, o, 64);
      v = t + o < G ? fmax(v, w) : v;
    }
  return v;
}

// Plane loop 1 of rhsp (rhsp.F90:120-153) for one (j, i) row: r2c(u_x^2) ->
// wki1, r2c(u w_x) -> wki3, r2c(v_x uy) -> wki2 (rows <= ny) and the row's
// maxima of |u|, |w_x|, |v_x|.  The transforms, their pairing and, in FP32,
// the mean flow kept out of them are those of products1_z.
// Bound by the copy rate's latency side: a transform holds E complex values
// and its twiddles, so few wavefronts fit.  FP64 is held to two per SIMD where
// a lane has at most 16 values (a few dozen registers spilled; 459 -> 388 us on
// a 896 x 176 x 224 box, 1.5 GB), the rest is left to the compiler: three per
// SIMD in FP32 (forced to four it spills, 210 -> 288 us).  The LDS kernel took
// 2610 us there, 1567 us in FP32.
template <int N, typename R>
__global__ void __launch_bounds__(64, sizeof(R) == 8 && ZRow<N>::E <= 16 ? 2 : 1)
products1_t(const R *__restrict__ u, R *wki1, R *wki2, R *wki3, const R *__restrict__ uy,
            const typename CT<R>::c *__restrict__ tw, int ny, int nrows, double *rowmax) {
  using C = typename CT<R>::c;
  using Z = ZRow<N>;
  using F = ZRowPhys<N>;
  constexpr int nz1 = 2 * (N / 3);
  constexpr bool SPLIT = sizeof(R) == 4;
  __shared__ C lds_all[Z::T * Z::lds()];
  TeamRow<N> w;
  if (!w.init(nrows)) return;
  const int t = w.t, row = w.row;
  C *lds = lds_all + w.team * Z::lds();
  const int i = row / (ny + 1), j = row - i * (ny + 1); // 0-based plane and row
  const int i0 = w.row0 / (ny + 1), j0 = w.row0 - i0 * (ny + 1);
  // the wavefront's first row of the u-type and v-type fields, and this
  // lane's row from there in complex values
  const size_t bu = (size_t)w.row0 * nz1, bv = ((size_t)i0 * ny + j0) * nz1;
  const unsigned ou = (unsigned)w.team * (nz1 / 2), ov = (unsigned)((i - i0) * ny + j - j0) * (nz1 / 2);
  u += bu;
  uy += bu;
  wki1 += bu;
  wki2 += bv;
  wki3 += bu;
  const bool vrow = j < ny;
  R um = 0, wm = 0, vm = 0;
  C Q[Z::E];
  if (vrow) {
    tload_spectral<N, true>(Q, t, (const R *)wki2, ov, uy, ou);
    const R Uy = SPLIT ? tld<C>(uy, ou).x : R(0);
    if (SPLIT && t == 0) Q[0].y = R(0); // k = 0: lane 0, slot 0
    trun<N, +1, false>(Q, t, tw, lds);
#pragma unroll
    for (int e = 0; e < F::E; ++e) {
      vm = fmax(vm, fabs(Q[e].x));
      Q[e] = mkc<C>(Q[e].x * Q[e].y, R(0));
    }
    trun<N, -1, true>(Q, t, tw, lds);
    tstore_spectral<N, R>(Q, t, lds, wki2, ov, nullptr, 0, SPLIT ? wki2 : nullptr, Uy, Uy);
  }
  R s1[F::E];
  tload_spectral<N, true>(Q, t, u, ou, (const R *)wki3, ou);
  trun<N, +1, false>(Q, t, tw, lds);
#pragma unroll
  for (int e = 0; e < F::E; ++e) {
    um = fmax(um, fabs(Q[e].x));
    wm = fmax(wm, fabs(Q[e].y));
    s1[e] = Q[e].x * Q[e].y;
  }
  tload_spectral<N, false>(Q, t, (const R *)wki1, ou, (const R *)nullptr, 0);
  const R Ux = SPLIT ? tld<C>(wki1, ou).x : R(0);
  if (SPLIT && t == 0) Q[0].x = R(0);
  trun<N, +1, false>(Q, t, tw, lds);
#pragma unroll
  for (int e = 0; e < F::E; ++e) Q[e] = mkc<C>(Q[e].x * Q[e].x, s1[e]);
  trun<N, -1, true>(Q, t, tw, lds);
  tstore_spectral<N, R>(Q, t, lds, wki1, ou, wki3, ou, SPLIT ? wki1 : nullptr, Ux, R(2) * Ux);
  um = team_max<Z::G>(um, t);
  wm = team_max<Z::G>(wm, t);
  vm = team_max<Z::G>(vm, t);
  if (t == 0) {
    rowmax[row] = um;
    rowmax[nrows + row] = wm;
    rowmax[2 * (size_t)nrows + row] = vrow ? (double)vm : 0.0;
  }
}

// Plane loop 2 of rhsp (rhsp.F90:367-415) for one (j, i) row, j <= ny, planes
// 2..nx-1: r2c(v w_v) -> ya, r2c(v_u^2) -> yb, r2c(w^2) -> yc, as products2_z.
// At the copy rate in FP64 (896 x 176 x 224: 1740 -> 258 us, 5.0 TB/s; FP32
// 1005 -> 158 us, 4.1 TB/s).
template <int N, typename R>
__global__ void __launch_bounds__(64)
products2_t(const R *__restrict__ resv, const R *__restrict__ resw, R *ya, R *yb, R *yc,
            const typename CT<R>::c *__restrict__ tw, int ny, int nrows) {
  using C = typename CT<R>::c;
  using Z = ZRow<N>;
  using F = ZRowPhys<N>;
  constexpr int nz1 = 2 * (N / 3);
  __shared__ C lds_all[Z::T * Z::lds()];
  TeamRow<N> w;
  if (!w.init(nrows)) return;
  const int t = w.t;
  C *lds = lds_all + w.team * Z::lds();
  const int i = w.row / ny + 1, j = w.row - (i - 1) * ny; // 0-based plane (from the second) and row
  const int i0 = w.row0 / ny + 1, j0 = w.row0 - (i0 - 1) * ny;
  const size_t bu = ((size_t)i0 * (ny + 1) + j0) * nz1, bv = ((size_t)i0 * ny + j0) * nz1;
  const unsigned ou = (unsigned)((i - i0) * (ny + 1) + j - j0) * (nz1 / 2), ov = (unsigned)w.team * (nz1 / 2);
  resv += bv;
  resw += bu;
  ya += bu;
  yb += bu;
  yc += bu;
  C Q[Z::E];
  tload_spectral<N, true>(Q, t, (const R *)yb, ou, resw, ou);
  trun<N, +1, false>(Q, t, tw, lds);
#pragma unroll
  for (int e = 0; e < F::E; ++e) Q[e] = mkc<C>(Q[e].x * Q[e].x, Q[e].y * Q[e].y);
  trun<N, -1, true>(Q, t, tw, lds);
  tstore_spectral<N, R>(Q, t, lds, yb, ou, yc, ou);
  tload_spectral<N, true>(Q, t, resv, ov, (const R *)ya, ou);
  trun<N, +1, false>(Q, t, tw, lds);
#pragma unroll
  for (int e = 0; e < F::E; ++e) Q[e] = mkc<C>(Q[e].x * Q[e].y, R(0));
  trun<N, -1, true>(Q, t, tw, lds);
  tstore_spectral<N, R>(Q, t, lds, ya, ou, nullptr, 0);
}

// fourxz (ffts.f90:27-67) on independent rows: iopt >= 0 c2r, < 0 r2c
template <int N>
__global__ void __launch_bounds__(64)
fourxz_t(double *fou, double *phys, int iopt, const double2 *__restrict__ tw, int nrows) {
  using Z = ZRow<N>;
  using F = ZRowPhys<N>;
  __shared__ double2 lds_all[Z::T * Z::lds()];
  TeamRow<N> w;
  if (!w.init(nrows)) return;
  const int t = w.t;
  double2 *lds = lds_all + w.team * Z::lds();
  double *X = fou + (size_t)w.row0 * (2 * (N / 3)), *Ph = phys + (size_t)w.row * N;
  const unsigned ox = (unsigned)w.team * (N / 3);
  double2 Q[Z::E];
  if (iopt >= 0) {
    tload_spectral<N, false>(Q, t, (const double *)X, ox, (const double *)nullptr, 0);
    trun<N, +1, false>(Q, t, tw, lds);
#pragma unroll
    for (int m = 0; m < F::MB; ++m)
      if (town<F::NB, Z::G>(t, m)) {
#pragma unroll
        for (int q = 0; q < F::R; ++q) Ph[t + Z::G * m + q * F::NB] = Q[m * F::R + q].x;
      }
  } else {
#pragma unroll
    for (int m = 0; m < F::MB; ++m) {
      const bool own = town<F::NB, Z::G>(t, m);
#pragma unroll
      for (int q = 0; q < F::R; ++q)
        Q[m * F::R + q] = make_double2(own ? Ph[t + Z::G * m + q * F::NB] : 0.0, 0.0);
    }
    trun<N, -1, true>(Q, t, tw, lds);
    tstore_spectral<N, double>(Q, t, lds, X, ox, nullptr, 0);
  }
}

template <int N> static void team_fns(ZTeamFns &f) {
  f.nz = N;
  f.lanes = ZRow<N>::G;
  f.rows = ZRow<N>::T;
  f.p1d = &products1_t<N, double>;
  f.p1f = &products1_t<N, float>;
  f.p2d = &products2_t<N, double>;
  f.p2f = &products2_t<N, float>;
  f.fx = &fourxz_t<N>;
}

// the kernels of length n if it is one of LO, LO + 2, .. HI
template <int LO, int HI> static bool team_find(int n, ZTeamFns &f) {
  if constexpr (LO > HI) return false;
  else {
    if constexpr (zteam_length(LO)) {
      if (n == LO) {
        team_fns<LO>(f);
        return true;
      }
    }
    return team_find<LO + 2, HI>(n, f);
  }
}

} // namespace otbl

// The z-direction kernels of otbl_zteam.h for a range of row lengths: one
// translation unit per range (otbl_zteam_*.hip), so that the lengths compile
// in parallel.  A workgroup is one wavefront: its teams share nothing, and
// single wavefronts pack a CU's LDS and registers tightest.
#pragma once
#include "otbl_kcommon.h"
#include "otbl_stats_row.h"
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
// maxima of |u|, |w_x|, |v_x|.  The transforms and their pairing are those of
// products1_z.  In FP32 the mean flow of u_x, of uy and of u stays out of them:
// u w_x = U w_x + u' w_x with the U term added in spectral space.  With U in the
// transform that it shares with w_x, the error of w's right-hand side at 54 points
// was twice as large.
// Bound by the copy rate's latency side: a transform holds E complex values
// and its twiddles, so few wavefronts fit.  FP64 is held to two per SIMD where
// a lane has at most 16 values (a few dozen registers spilled; 459 -> 388 us on
// a 896 x 176 x 224 box, 1.5 GB), the rest is left to the compiler: three per
// SIMD in FP32 (222 us; forced to four it spills, +37%).  The LDS kernel took
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
  const R U = SPLIT ? tld<C>(u, ou).x : R(0);
  if (SPLIT && t == 0) Q[0].x = R(0);
  trun<N, +1, false>(Q, t, tw, lds);
#pragma unroll
  for (int e = 0; e < F::E; ++e) {
    um = fmax(um, fabs(SPLIT ? Q[e].x + U : Q[e].x));
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
  tstore_spectral<N, R>(Q, t, lds, wki1, ou, wki3, ou, SPLIT ? wki1 : nullptr, Ux, R(2) * Ux, SPLIT ? wki3 : nullptr,
                        U);
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
// 2..nx-1: r2c(v w_v) -> ya, r2c(v_u^2) -> yb, r2c(w^2) -> yc, as products2_z.  In
// FP32 an inverse transform's round-off in one product scales with the other, and
// d/dz multiplies that of w^2 by kz, so the rows keep the pairs of the kernel that
// ran them before: (v_u^2, w^2) and v w_v alone at the engine's lengths, else
// (v w_v, v_u^2) and w^2 alone (ALONE) as on the LDS kernel (with the other pairs
// the error of w's right-hand side was up to 4.9 times, at 980 points).  They keep
// the engine's order of radices, too, the larger at the spectral end (REV): 4 x 16 x
// 16 left 1.26 times the engine's round-off in the highest modes of v's right-hand
// side at 1024 points, 16 x 16 x 4 leaves 1.03 times (plane loop 1 gains nothing from
// it and loses 27% of its time).
// At the copy rate in FP64 (896 x 176 x 224: 1740 -> 258 us, 5.0 TB/s; FP32
// 1005 -> 159 us, 4.1 TB/s).
template <int N, typename R>
__global__ void __launch_bounds__(64)
products2_t(const R *__restrict__ resv, const R *__restrict__ resw, R *ya, R *yb, R *yc,
            const typename CT<R>::c *__restrict__ tw, int ny, int nrows) {
  using C = typename CT<R>::c;
  using Z = ZRow<N>;
  constexpr int nz1 = 2 * (N / 3);
  constexpr bool ENGINE = N == 256 || N == 512 || N == 1024, ALONE = sizeof(R) == 4 && !ENGINE;
  constexpr bool REV = ENGINE && Z::rad(0) < Z::rad(Z::NP - 1);
  using F = ZRowPhys<N, REV>;
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
  tload_spectral<N, true, REV>(Q, t, (const R *)yb, ou, resw, ou);
  trun<N, +1, REV>(Q, t, tw, lds);
  R s1[ALONE ? F::E : 1]; // v_u^2
#pragma unroll
  for (int e = 0; e < F::E; ++e) {
    if constexpr (ALONE) {
      s1[e] = Q[e].x * Q[e].x;
      Q[e] = mkc<C>(Q[e].y * Q[e].y, R(0));
    } else {
      Q[e] = mkc<C>(Q[e].x * Q[e].x, Q[e].y * Q[e].y);
    }
  }
  trun<N, -1, !REV>(Q, t, tw, lds);
  if constexpr (ALONE) tstore_spectral<N, R, REV>(Q, t, lds, yc, ou, nullptr, 0);
  else tstore_spectral<N, R, REV>(Q, t, lds, yb, ou, yc, ou);
  tload_spectral<N, true, REV>(Q, t, resv, ov, (const R *)ya, ou);
  trun<N, +1, REV>(Q, t, tw, lds);
#pragma unroll
  for (int e = 0; e < F::E; ++e) Q[e] = mkc<C>(Q[e].x * Q[e].y, ALONE ? s1[ALONE ? e : 0] : R(0));
  trun<N, -1, !REV>(Q, t, tw, lds);
  if constexpr (ALONE) tstore_spectral<N, R, REV>(Q, t, lds, ya, ou, yb, ou);
  else tstore_spectral<N, R, REV>(Q, t, lds, ya, ou, nullptr, 0);
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

// sum over a team, in its lane 0
template <int G> __device__ __forceinline__ double team_sum(double v, int t) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
    if (o < G) {
      const double w = __shfl_down(v, o, 64);
      v = t + o < G ? v + w : v;
    }
  return v;
}

// Row sums of the statistics (stotf.F90:148-283) for one (j, i) row: three
// packed c2r transforms, the physical products and every sum in FP64, whatever
// the fields hold (R).  FP32 transforms would carry the round-off of the mean
// flow, O(1), into the enstrophy and the triple products: 4 to 12 times the
// error of the former and up to 1e3 times that of u^3 on a mixed box.  Bound by
// FP64 arithmetic and the registers of its transforms.  us per sample of 256 x 96
// rows, one row per workgroup (the LDS kernel) -> here: mixed rows of 64 points
// 3254 -> 57, 96 3408 -> 86, 224 3658 -> 198; FP64 224 3722 -> 210.
template <int N, typename R>
__global__ void __launch_bounds__(64)
stats_t(StatsZ a, const double2 *__restrict__ tw, int nx, int ny, int nrows) {
  using C = double2;
  using Z = ZRow<N>;
  using F = ZRowPhys<N>;
  constexpr int nz1 = 2 * (N / 3), nz2 = N / 3 - 1;
  __shared__ C lds_all[Z::T * Z::lds()];
  TeamRow<N> w;
  if (!w.init(nrows)) return;
  const int t = w.t, row = w.row;
  C *lds = lds_all + w.team * Z::lds();
  const int i = row / ny, j = row - i * ny; // 0-based plane and row
  const size_t ov = (size_t)w.row0 * nz1;
  const unsigned o = (unsigned)w.team * (nz1 / 2);
  const R *Bq[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) Bq[q] = (const R *)a.B[q] + ov;
  const R *V = (const R *)a.v + ov, *DV = (const R *)a.dvdx + ov;
  const size_t om = (size_t)j * nx + i; // (i, j) of the [ny][nx] mean-flow rows
  auto at = [&](const R *p, unsigned k) {
    const typename CT<R>::c b = tld<typename CT<R>::c>(p, o + k);
    return make_double2((double)b.x, (double)b.y);
  };
  // B1 (u_x at the v rows), B4, B6 with the FP64 mean flow of a mixed box (m)
  auto mean_at = [&](const R *p, const double *m, unsigned k) {
    double2 b = at(p, k);
    if (m && k == 0) b.x = m[om];
    return b;
  };
  double sum[NSUM];
#pragma unroll
  for (int q = 0; q < NSUM; ++q) sum[q] = 0.0;
  double s2[F::E], U[F::E];
  C v[Z::E];
  // omega_x + i omega_y
  tload_modes<N, true, C>(v, t, [&](unsigned k, C &x, C &y) {
    const double kz = a.kaz[k];
    const C b7 = at(Bq[6], k), vv = at(V, k), b1 = mean_at(Bq[0], a.m1, k), b3 = at(Bq[2], k);
    x = mkc<C>(b7.x + kz * vv.y, b7.y - kz * vv.x);
    y = mkc<C>(-kz * b1.y - b3.x, kz * b1.x - b3.y);
  });
  trun<N, +1, false>(v, t, tw, lds);
#pragma unroll
  for (int e = 0; e < F::E; ++e) s2[e] = v[e].x * v[e].x + v[e].y * v[e].y;
  // omega_z + i u
  tload_modes<N, true, C>(v, t, [&](unsigned k, C &x, C &y) {
    const C dv = at(DV, k), b6 = mean_at(Bq[5], a.m6, k);
    x = mkc<C>(dv.x - b6.x, dv.y - b6.y);
    y = mean_at(Bq[0], a.m1, k);
  });
  trun<N, +1, false>(v, t, tw, lds);
  float *ens = a.ens + (size_t)row * N;
#pragma unroll
  for (int m = 0; m < F::MB; ++m) {
    const bool own = town<F::NB, Z::G>(t, m);
#pragma unroll
    for (int q = 0; q < F::R; ++q) {
      const int e = m * F::R + q;
      if (own) ens[t + Z::G * m + q * F::NB] = (float)sqrt(s2[e] + v[e].x * v[e].x);
      U[e] = v[e].y;
    }
  }
  // v + i w (a lane without a butterfly holds zeros: nothing in the sums)
  tload_modes<N, true, C>(v, t, [&](unsigned k, C &x, C &y) {
    x = at(V, k);
    y = at(Bq[1], k);
  });
  trun<N, +1, false>(v, t, tw, lds);
#pragma unroll
  for (int e = 0; e < F::E; ++e) {
    const double u = U[e], vv = v[e].x, ww = v[e].y;
    sum[21] += u * u * u;    // u3
    sum[22] += u * ww * ww;  // w2u
    sum[23] += vv * vv * vv; // v3
    sum[24] += vv * ww * ww; // w2v
    sum[25] += u * vv * vv;  // v2u
    sum[26] += vv * u * u;   // u2v
  }
#pragma unroll 1
  for (int k = t; k <= nz2; k += Z::G)
    stats_mode(sum, k == 0 ? 1.0 : 2.0, a.kaz[k], mean_at(Bq[0], a.m1, k), at(Bq[1], k), at(Bq[2], k),
               mean_at(Bq[3], a.m4, k), at(Bq[4], k), mean_at(Bq[5], a.m6, k), at(Bq[6], k), at(Bq[7], k), at(V, k),
               at(DV, k));
#pragma unroll
  for (int q = 0; q < NSUM; ++q) sum[q] = team_sum<Z::G>(sum[q], t);
  if (t != 0) return;
  const size_t S = (size_t)nx * (ny + 1);
  double *acc = a.acc + (size_t)i * (ny + 1) + j;
  stats_add_sums(acc, S, sum);
  stats_add_means(acc, S, mean_at(Bq[0], a.m1, 0).x, at(Bq[1], 0).x, at(Bq[2], 0).x, mean_at(Bq[3], a.m4, 0).x,
                  at(Bq[4], 0).x, mean_at(Bq[5], a.m6, 0).x, at(Bq[6], 0).x, at(Bq[7], 0).x, at(V, 0).x, at(DV, 0).x);
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
  f.std_ = &stats_t<N, double>;
  if constexpr (N != 512 && N != 1024) f.stf = &stats_t<N, float>; // those: stats_zr
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

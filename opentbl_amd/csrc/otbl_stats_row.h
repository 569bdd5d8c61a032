// Row sums of the statistics (stotf.F90:51-291) shared by the z kernels:
// accumulator ids, kernel arguments, the sums of one mode and the row's
// additions to the accumulators.
#pragma once
#include "otbl_kcommon.h"
#include "otbl_fft.h"

namespace otbl {

// accumulator ids (the order of the reference's statistics files:
// escru.F90:318-341 then 490-516)
enum {
  S_US, S_VS, S_WS, S_UV, S_UA, S_VA, S_WA, S_PP, S_PM, S_VORTX, S_VORTY, S_VORTZ, S_VORTXA, S_VORTYA,
  S_VORTZA, S_UW, S_VW, S_DISPU, S_DISPV, S_DISPW, S_DISPUV, S_PUP, S_PVP, S_PDUDX, S_PDVDY, S_PDUDY,
  S_PDVDX, S_PDWDZ, S_V3, S_U2V, S_V2U, S_W2V, S_DUDX0, S_DUDY0, S_DVDX0, S_DVDY0, S_DWDX0, S_DWDY0, S_U3,
  S_W2U, S_COUNT
};
static_assert(S_COUNT == OTBL_NSTAT, "statistic count");

// the sums over modes and over z of one row
constexpr int NSUM = 21 + 6;

struct StatsZ {
  const void *B[8], *v, *dvdx;
  // mixed box: the real part of mode 0 of B1, B4, B6 from the FP64 mean
  // flow, [ny][nx] (null: from the fields)
  const double *m1, *m4, *m6;
  const double *kaz;
  double *acc; // [S_COUNT][nx][ny+1]
  float *ens;  // [nx][ny][nz]
};

template <typename C> struct CPair {
  C x, y;
};

// the 21 mode sums (stotf.F90:156-218) of one mode, weighted cte: the y lines'
// eight fields b1..b8 and v, dv/dx at wavenumber kz
__device__ __forceinline__ void stats_mode(double (&sum)[NSUM], double cte, double kz, double2 b1, double2 b2,
                                           double2 b3, double2 b4, double2 b5, double2 b6, double2 b7, double2 b8,
                                           double2 v, double2 dv) {
  auto re = [](double2 x, double2 y) { return x.x * y.x + x.y * y.y; }; // Re(x conj(y))
  // z derivatives: x kaz = (-kz x.y, kz x.x)
  const double2 uz = make_double2(-kz * b1.y, kz * b1.x), vz = make_double2(-kz * v.y, kz * v.x);
  const double2 wz = make_double2(-kz * b2.y, kz * b2.x);
  const double2 ox = make_double2(b7.x - vz.x, b7.y - vz.y), oy = make_double2(uz.x - b3.x, uz.y - b3.y);
  const double2 oz = make_double2(dv.x - b6.x, dv.y - b6.y);
  sum[0] += cte * re(b1, b1);  // us
  sum[1] += cte * re(v, v);    // vs
  sum[2] += cte * re(b2, b2);  // ws
  sum[3] += cte * re(b1, v);   // uv
  sum[4] += cte * re(b5, b5);  // pp
  sum[5] += cte * re(ox, ox);  // vortx
  sum[6] += cte * re(oy, oy);  // vorty
  sum[7] += cte * re(oz, oz);  // vortz
  sum[8] += cte * re(b1, b2);  // uw
  sum[9] += cte * re(v, b2);   // vw
  sum[10] += cte * (re(b4, b4) + re(uz, uz) + re(b6, b6)); // dispu
  sum[11] += cte * (re(dv, dv) + re(vz, vz) + re(b8, b8)); // dispv
  sum[12] += cte * (re(wz, wz) + re(b3, b3) + re(b7, b7)); // dispw
  sum[13] += cte * (re(uz, vz) + re(b4, dv) + re(b6, b8)); // dispuv
  sum[14] += cte * re(b5, b1); // pup
  sum[15] += cte * re(b5, v);  // pvp
  sum[16] += cte * re(b5, b4); // pdudx
  sum[17] += cte * re(b5, b8); // pdvdy
  sum[18] += cte * re(b5, b6); // pdudy
  sum[19] += cte * re(b5, dv); // pdvdx
  sum[20] += cte * re(b5, wz); // pdwdz
}

// the row's sums added to the accumulators of (j, i) (acc: its address in the
// first one, S: an accumulator's size)
__device__ __forceinline__ void stats_add_sums(double *acc, size_t S, const double (&sum)[NSUM]) {
  constexpr int ID[NSUM] = {S_US,   S_VS,    S_WS,    S_UV,    S_PP,    S_VORTX, S_VORTY, S_VORTZ, S_UW,
                            S_VW,   S_DISPU, S_DISPV, S_DISPW, S_DISPUV, S_PUP,  S_PVP,   S_PDUDX, S_PDVDY,
                            S_PDUDY, S_PDVDX, S_PDWDZ, S_U3,   S_W2U,   S_V3,    S_W2V,   S_V2U,   S_U2V};
#pragma unroll
  for (int q = 0; q < NSUM; ++q) acc[ID[q] * S] += sum[q];
}
// the k = 0 means (stotf.F90:128-144): real parts of mode 0
__device__ __forceinline__ void stats_add_means(double *acc, size_t S, double b1, double b2, double b3, double b4,
                                                double b5, double b6, double b7, double b8, double v0, double dv0) {
  acc[S_UA * S] += b1;
  acc[S_WA * S] += b2;
  acc[S_VA * S] += v0;
  acc[S_PM * S] += b5;
  acc[S_DUDX0 * S] += b4;
  acc[S_DVDX0 * S] += dv0;
  acc[S_DWDX0 * S] += b3;
  acc[S_DUDY0 * S] += b6;
  acc[S_DVDY0 * S] += b8;
  acc[S_DWDY0 * S] += b7;
  acc[S_VORTYA * S] -= b3;
  acc[S_VORTXA * S] += b7;
  acc[S_VORTZA * S] += dv0 - b6;
}

} // namespace otbl

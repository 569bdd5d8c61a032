// The y Poisson solve of one mode by one marching thread.
#pragma once
#include "otbl_kcommon.h"

namespace otbl {

// per-mode y tridiagonal on pencils (pois.f90:102-117, soltriy
// pois.f90:211-239): thread t of one per (kr, kx-mode x), line (j-1, kr) at
// P + ((j-1) nz1 + kr) ld, so rows at stride nz1 ld.
__device__ __forceinline__ void poisson_y_march(size_t t, double *__restrict__ P, double *__restrict__ S,
                                                const DevCoef &c, int nx, int ny, int nz1, int kr_end, int ld) {
  constexpr int RB = 8; // rows whose loads are issued together
  const int N = nx - 1;
  if (t >= (size_t)kr_end * N) return; // columns kr < kr_end
  const int x = (int)(t % N), kr = (int)(t / N), i = x + 2;
  const size_t rs = (size_t)nz1 * ld;
  double *col = P + (size_t)kr * ld + x;
  double *d2 = S + (size_t)kr * ld + x;
  const int ny1 = ny - 1;
  if (kr == 1) { // the zero mode is real (pois.f90:102)
    for (int j = 0; j < ny1; ++j) col[(size_t)j * rs] = 0.0;
    return;
  }
  const double kz2 = c.kaz2[kr / 2], km = c.kmod[i - 1];
  const bool pin = (i == 2 && kr == 0); // its last row: phi = 0 with a doubled diagonal
  double a2prev = C3(c.ayp, 2, 1) - kz2 - km;
  double a3prev = C3(c.ayp, 3, 1);
  double y = (pin && ny1 == 1) ? 0.0 : col[0];
  if (pin && ny1 == 1) col[0] = 0.0;
  // forward elimination as soltriy, rows 2..ny-1
  auto fwd = [&](int j, double b) {
    if (pin && j == ny1) b = 0.0;
    const double d = 1.0 / a2prev;
    d2[(size_t)(j - 2) * rs] = d;
    const double a1 = -C3(c.ayp, 1, j) * d;
    double a2 = (pin && j == ny1) ? 2.0 * C3(c.ayp, 2, j) : C3(c.ayp, 2, j) - kz2 - km;
    a2 = a2 + a1 * a3prev;
    y = b + a1 * y;
    col[(size_t)(j - 1) * rs] = y;
    a2prev = a2;
    a3prev = C3(c.ayp, 3, j);
  };
  int j = 2;
  for (; j + RB - 1 <= ny1; j += RB) {
    double bv[RB];
#pragma unroll
    for (int q = 0; q < RB; ++q) bv[q] = col[(size_t)(j + q - 1) * rs];
#pragma unroll
    for (int q = 0; q < RB; ++q) fwd(j + q, bv[q]);
  }
  for (; j <= ny1; ++j) fwd(j, col[(size_t)(j - 1) * rs]);
  double x_ = y * (1.0 / a2prev);
  col[(size_t)(ny1 - 1) * rs] = x_;
  // back substitution, rows ny-2..1
  auto bwd = [&](int j, double yv, double d) {
    x_ = (yv - C3(c.ayp, 3, j) * x_) * d;
    col[(size_t)(j - 1) * rs] = x_;
  };
  j = ny1 - 1;
  for (; j - RB + 1 >= 1; j -= RB) {
    double yv[RB], dv[RB];
#pragma unroll
    for (int q = 0; q < RB; ++q) {
      yv[q] = col[(size_t)(j - q - 1) * rs];
      dv[q] = d2[(size_t)(j - q - 1) * rs];
    }
#pragma unroll
    for (int q = 0; q < RB; ++q) bwd(j - q, yv[q], dv[q]);
  }
  for (; j >= 1; --j) bwd(j, col[(size_t)(j - 1) * rs], d2[(size_t)(j - 1) * rs]);
}

} // namespace otbl

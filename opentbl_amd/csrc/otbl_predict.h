// The pressure-gradient predictor (rhsp.F90:291-339) of one column, formed
// where its rows are used.
//
// A pass of its own reads u, v, w and p and writes the predicted u, v, w, which
// the final update then reads: seven passes over a field for values that the
// update, which reads the saved velocities anyway, forms from one read of p per
// component (u takes the planes i and i+1, the second of which the next plane's
// workgroup reads as its own).  Measured, ms per substep, predictor pass + final
// update -> final update (HBM-bound): 1536 x 315 x 1024 mixed 1.94 + 4.26 -> 4.77,
// 1024 x 192 x 512 FP64 0.71 + 3.12 -> 3.21; per step: 98.5 -> 94.0 and 37.1 ->
// 35.1, 640 x 144 x 160 mixed 4.39 -> 4.14, 256 x 96 x 64 FP64 1.13 -> 1.11.
#pragma once
#include "otbl_kcommon.h"

namespace otbl {

template <typename T> struct Predictor {
  const T *p; // [nx][ny][nz1]
  double idxx;
  int nx, ny, nz1;
};

template <typename T> inline Predictor<T> predictor(const Box &b) {
  return {reinterpret_cast<const T *>(b.f[OTBL_P]), b.hc.idxx, b.nx, b.ny, b.nz1};
}

// Component K (1 v, 2 w, 3 u) at column kr of the 0-based plane ip.  Rows are
// 0-based; I is the offset type (unsigned for FP32 fields below 2^30 values:
// one register per row address from the uniform base).  The real part of mode 0
// of an FP32 v is predicted by the FP64 mean pressure instead and already in the
// new field (mean: taken from there); that of u takes the FP32 gradient here,
// its FP64 mean flow replaces the field's values after the update.
template <int K, typename T, typename I = size_t> struct PredCol {
  const T *p, *idyy;
  I o, s, d; // offset of (ip, row 0) in p, row stride, plane stride
  T var1, f;
  int top, hi; // last row of p, last predicted row (the first is row 1)
  bool on, mean = false;

  __device__ __forceinline__ PredCol(const Predictor<T> &P, const DevCoefT<T> &c, const DevScalars *ds, int kr,
                                     size_t ip)
      : p(P.p), idyy(c.idyy), s((I)P.nz1), d((I)P.nz1 * (I)P.ny), var1((T)ds->var1), f(var1), top(P.ny - 1),
        hi(K == 1 ? P.ny - 2 : P.ny - 1), on(ip > 0) {
    if constexpr (K == 3) {
      f = var1 * (T)P.idxx;
      on = on && ip + 2 <= (size_t)P.nx;
      if (!on) ip = 0; // a plane without one after it reads the first two
    }
    if constexpr (K == 2) {
      // w -= var1 (i kz p): Re gets -(-kz Im p), Im gets -(kz Re p)
      const T kz = c.kaz[kr / 2];
      f = (kr & 1) ? kz : -kz;
      kr ^= 1;
    }
    if constexpr (K == 1 && sizeof(T) == 4) {
      mean = kr == 0 && on;
      on = on && !mean;
    }
    o = (I)ip * d + (I)kr;
  }
  __device__ __forceinline__ T ld(I e) const {
    if constexpr (sizeof(I) == 4)
      return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + (size_t)(e * I(sizeof(T))));
    else
      return p[e];
  }
  __device__ __forceinline__ int row(int j) const { return j < 0 ? 0 : (j > top ? top : j); }
  // p at row j of the plane, and of the one after it (u)
  __device__ __forceinline__ T at(int j) const { return ld(o + (I)row(j) * s); }
  __device__ __forceinline__ T after(int j) const { return ld(o + (I)row(j) * s + d); }
  __device__ __forceinline__ T dyi(int j) const { return K == 1 ? idyy[row(j) + 1] : T(0); }
  // the predicted row j from the saved value and p: a = at(j), b = after(j) for
  // u, at(j + 1) for v (unused for w), cy = dyi(j)
  __device__ __forceinline__ T apply(T x, int j, T a, T b, T cy) const {
    T y;
    if constexpr (K == 3)
      y = fma(-f, b - a, x);
    else if constexpr (K == 1)
      y = fma(-(var1 * cy), b - a, x);
    else
      y = fma(-var1, f * a, x);
    return on && j >= 1 && j <= hi ? y : x;
  }
  __device__ __forceinline__ T pred(T x, int j) const {
    return apply(x, j, at(j), K == 3 ? after(j) : (K == 1 ? at(j + 1) : T(0)), dyi(j));
  }
};

// The RK3 combination u - (var3 rhs + var2 visc + var4 rhs_prev), and boun's u
// and w rows 1 and ny+1 from the column's rows at(j): written out, as the
// kernels that share them are compared bit for bit
template <typename T> __device__ __forceinline__ T rk_sum(T u, T var3, T rh, T var2, T vis, T var4, T rp) {
  return u - fma(var4, rp, fma(var3, rh, var2 * vis));
}
template <typename T, class At> __device__ __forceinline__ T boun_first(const DevCoefT<T> &c, At at) {
  const T i21 = T(-1) / M4(c.inby, 2, 1);
  return i21 * fma(M4(c.inby, 2, 4), at(3), fma(M4(c.inby, 2, 2), at(1), M4(c.inby, 2, 3) * at(2)));
}
template <typename T, class At> __device__ __forceinline__ T boun_last(const DevCoefT<T> &c, int ny, At at) {
  const T c11 = T(-1) / M2(c.ccon, 1, 1);
  return c11 * fma(M2(c.ccon, 1, 4), at(ny - 3), fma(M2(c.ccon, 1, 2), at(ny - 1), M2(c.ccon, 1, 3) * at(ny - 2)));
}

} // namespace otbl

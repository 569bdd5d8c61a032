// x-line compact operators (interpxx, difvisxx) with the line split over the
// wavefronts of a workgroup.
//
// A workgroup takes 64 lines (consecutive (kr, j) elements of a plane) and a
// span of consecutive chunks of L planes, one chunk per wavefront, held in
// registers: every plane row of a chunk is loaded before any is used.  A chunk
// is solved with zero carries (forward y_i = r_i + m_i y_{i-1}, backward
// x_i = a2_i y_i + b_i x_{i+1}); the carries come from the neighbouring chunks
// through LDS and are applied with the chunk's tabulated responses:
//   x = x_local + C g + D s,
// C the y of the plane before the chunk and D the x of the plane after it.
// Both follow from a few neighbours: a carry is damped by the product of m
// (or b) over every chunk it crosses, so recurrences over `depth` chunks are
// exact to round-off (set by the host from the factored systems).
//
// Lines of at most XCH L planes are one span.  Longer ones are cut into spans
// that overlap by `halo` chunks on each side: a span solves its halo chunks too
// and stores only its own, whose carries no longer know where the span began.
// Neighbouring spans run on one XCD, so the halo's second read stays in its L2
// (lines first, spans second: +20% on the derivatives).
//
// A thread per line segment (otbl_xline.hip) marches its planes in dependent
// steps, each waiting for memory, and starts 32 + 24 planes outside its own.
// Measured, us per launch of interpxx and difvisxx, marching -> chunked (copy
// rate 4.9 TB/s): 256 x 96 x 64 FP64 23 / 42 -> 12.6 / 19; 640 x 144 x 160 mixed
// 43 / 74 -> 19.5 / 40, FP64 51 / 90 -> 41 / 74; 896 x 176 x 224 FP64 110 / 196 ->
// 96 / 173; 1024 x 192 x 512 FP64 interpxx 280 -> 245 (4.4 TB/s); 1536 x 315 x 1024
// mixed interpxx 688 -> 646.
// The derivatives of larger boxes stay on the marching kernel, whose two arrays
// in flight fill the memory system there: FP64 from 30000 lines on (128
// registers leave one workgroup per CU, whose load and store phases do not
// overlap: 1024 x 192 x 768, calls of three boxes in flight, 524 against 712
// us; a launch alone is faster in chunks, 643 against 705), FP32 where it needs at most three segments per line (1536 x 315 x 1024:
// 1033 against 1061 us).
#include "otbl_chunk.h"

namespace otbl {

// an operator's arrays: lines in, velocity (derivatives), lines out, table(s),
// closure rows, mode, values per plane; and up to three of a launch
template <typename T> struct XOp {
  const T *in, *vel;
  T *out;
  const T *tab, *tabv;
  int c1, c2, mode;
  size_t P;
};
template <typename T> struct XOps {
  XOp<T> op[3];
};

// Table of one system of n planes in nc chunks of L (NL = nc L planes), by
// phase, so that a phase reads one stream of scalars:
//   forward   [NL][4]: stencil E1, E2, E3, multiplier M
//   backward  [NL][2]: inverse pivot A2, B = -c A2
//   responses [NL][2]: G, S to unit carries
//   chunk     [nc][4]: PE (product of M), G0, S0 (G, S at the first plane), 0
__global__ void xtab_kernel(double *tabs, DevCoef c, int n, int L, int nc, size_t stride, int first) {
  const int sys = first + blockIdx.y, q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nc) return;
  const double *a = sys == XT_INXU   ? c.inxu
                    : sys == XT_INXV ? c.inxv
                    : sys == XT_DCXU ? c.dcxu
                    : sys == XT_DCXV ? c.dcxv
                    : sys == XT_VIXU ? c.vixu
                                     : c.vixv;
  const size_t NL = (size_t)nc * L;
  double *F = tabs + blockIdx.y * stride, *K = F + 4 * NL, *R = K + 2 * NL, *E = R + 2 * NL;
  double pr = 1.0;
  for (int r = 0; r < L; ++r) {
    const int j = q * L + r, i = j + 1; // i: 1-based plane
    double m = 0.0, a2 = 0.0, b = 0.0, e1 = 0.0, e2 = 0.0, e3 = 0.0;
    if (j < n) {
      m = j == 0 ? 0.0 : C3(a, 1, i);
      a2 = C3(a, 2, i);
      b = j == n - 1 ? 0.0 : -C3(a, 3, i) * a2;
    }
    if (j >= 1 && j <= n - 2) {
      switch (sys) {
      case XT_INXU: e2 = C2(c.cofiux, 1, i), e3 = C2(c.cofiux, 2, i); break;
      case XT_INXV: e2 = C2(c.cofivx, 1, i), e3 = C2(c.cofivx, 2, i); break;
      case XT_DCXU: e1 = C2(c.cofcxu, 1, i), e2 = C2(c.cofcxu, 2, i); break;
      case XT_DCXV: e1 = C2(c.cofcxv, 1, i), e2 = C2(c.cofcxv, 2, i); break;
      case XT_VIXU: e1 = C3(c.cofvxu, 3, i), e2 = C3(c.cofvxu, 2, i), e3 = C3(c.cofvxu, 1, i); break;
      default: e1 = C3(c.cofvxv, 3, i), e2 = C3(c.cofvxv, 2, i), e3 = C3(c.cofvxv, 1, i); break;
      }
    }
    F[4 * j] = e1;
    F[4 * j + 1] = e2;
    F[4 * j + 2] = e3;
    F[4 * j + 3] = m;
    K[2 * j] = a2;
    K[2 * j + 1] = b;
    pr *= m;
    R[2 * j] = pr; // forward response, replaced below
  }
  double g = 0.0, sa = 1.0;
  for (int r = L - 1; r >= 0; --r) {
    const int j = q * L + r;
    g = K[2 * j] * R[2 * j] + K[2 * j + 1] * g;
    sa = K[2 * j + 1] * sa;
    R[2 * j] = g;
    R[2 * j + 1] = sa;
  }
  E[4 * q] = pr;
  E[4 * q + 1] = g;
  E[4 * q + 2] = sa;
  E[4 * q + 3] = 0.0;
}

// the FP64 tables of the interpolations (rows per chunk Li) and derivatives
// (Ld), in the order of the XT_ names
void kxc_tables(Box &b) {
  const XChunk &i = b.xci, &d = b.xcd;
  LAUNCH(b, "xtab", dim3(nblk(i.nc, 64), 2), 64, 0, xtab_kernel, b.xtab, b.dc, b.nx, i.L, i.nc, xtab_size(i), XT_INXU);
  if (d.L)
    LAUNCH(b, "xtab", dim3(nblk(d.nc, 64), 4), 64, 0, xtab_kernel, b.xtab + 2 * xtab_size(i), b.dc, b.nx, d.L, d.nc,
           xtab_size(d), XT_DCXU);
}

// interpxx (lip.f90:248-300): midpoint interpolation along x
template <int L, typename T>
__device__ __forceinline__ void interpxx_b(const T *__restrict__ gen, T *__restrict__ geni, const T *__restrict__ tab,
                                           const T *__restrict__ inbx, int chi, int chi2, int nx, size_t P,
                                           const XChunk &x, T *xch) {
  const XPlace w(x, P);
  const XTabP<T> t(tab, x, L, w.c);
  const int j0 = w.c * L;
  T v[L], y = 0;
  if (w.act) {
#pragma unroll
    for (int r = 0; r < L; ++r) v[r] = (gen + (size_t)min(j0 + r, nx - 1) * P)[w.l];
    const T next = (gen + (size_t)min(j0 + L, nx - 1) * P)[w.l];
    T bot = 0, top = 0;
    if (j0 == 0)
#pragma unroll
      for (int k = 0; k < 4; ++k) bot += M4(inbx, chi2, k + 1) * v[k];
    if (j0 + L >= nx)
#pragma unroll
      for (int k = 0; k < 4; ++k) top += M4(inbx, chi, k + 1) * (gen + (size_t)(nx - 1 - k) * P)[w.l];
    XFENCE();
#pragma unroll
    for (int r = 0; r < L; ++r) {
      if (r % XGRP == 0) XFENCE();
      const int j = j0 + r;
      T rhs = t.E(2, r) * v[r] + t.E(3, r) * (r + 1 < L ? v[r + 1] : next);
      rhs = j == 0 ? bot : rhs;
      rhs = j == nx - 1 ? top : rhs;
      y = rhs + t.M(r) * y;
      v[r] = y;
    }
    XFENCE();
    xback<L>(v, t);
    xch[w.p * 64 + w.lane] = y;
    xch[XCT + w.p * 64 + w.lane] = v[0];
  }
  __syncthreads();
  if (!w.own) return;
  T C, D;
  xcarry(xch, xch + XCT, t, w, x.depth, C, D);
#pragma unroll
  for (int r = 0; r < L; ++r) {
    if (r % XGRP == 0) XFENCE();
    const T o = v[r] + fma(C, t.G(r), D * t.S(r));
    if (w.ok && j0 + r < nx) (geni + (size_t)(j0 + r) * P)[w.l] = o;
  }
}

template <int L, typename T>
__global__ void __launch_bounds__(XCT, sizeof(T) == 4 ? 8 : 1)
interpxx_c(const T *__restrict__ gen, T *__restrict__ geni, const T *__restrict__ tab, const T *__restrict__ inbx,
           int chi, int chi2, int nx, size_t P, XChunk x) {
  __shared__ T xch[2 * XCT];
  interpxx_b<L, T>(gen, geni, tab, inbx, chi, chi2, nx, P, x, xch);
}

// the three components of a substep (blockIdx.y).  For one operator the kernel
// above is faster (its arguments are known not to alias): 4% of the passes over
// 98304 lines of 1024 planes.
template <int L, typename T>
__global__ void __launch_bounds__(XCT, sizeof(T) == 4 ? 8 : 1)
interpxx3_c(XOps<T> a, const T *__restrict__ inbx, int nx, XChunk x) {
  __shared__ T xch[2 * XCT];
  const XOp<T> &o = a.op[blockIdx.y];
  interpxx_b<L, T>(o.in, o.out, o.tab, inbx, o.c1, o.c2, nx, o.P, x, xch);
}

// difvisxx (lip.f90:52-142): convective d/dx of the product plus rex times the
// compact d2/dx2 of the velocity; mode 1 adds to out except on plane nx, which
// gets the outflow derivative U_inf du/dx (lip.f90:105,132).
template <int L, typename T>
__device__ __forceinline__ void difvisxx_b(const T *__restrict__ gp, const T *__restrict__ qv, T *__restrict__ out,
                                           const T *__restrict__ tabc, const T *__restrict__ tabv,
                                           const T *__restrict__ dcbx, const T *__restrict__ cofvbx, int chv, int ic,
                                           int nx, size_t P, double rex_d, double idx_d, int mode, const XChunk &x,
                                           T *xch) {
  const XPlace w(x, P);
  const XTabP<T> tc(tabc, x, L, w.c), tv(tabv, x, L, w.c);
  const int j0 = w.c * L;
  const T rex = (T)rex_d, idx = (T)idx_d;
  T a[L], b[L], flow = 0;
  if (w.act) {
#pragma unroll
    for (int r = 0; r < L; ++r) a[r] = (gp + (size_t)min(j0 + r, nx - 1) * P)[w.l];
#pragma unroll
    for (int r = 0; r < L; ++r) b[r] = (qv + (size_t)min(j0 + r, nx - 1) * P)[w.l];
    T gm = (gp + (size_t)max(j0 - 1, 0) * P)[w.l], qm = (qv + (size_t)max(j0 - 1, 0) * P)[w.l];
    const T qn = (qv + (size_t)min(j0 + L, nx - 1) * P)[w.l];
    T botc = 0, botv = 0, topc = 0, topv = 0;
    if (j0 == 0)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        botc += M5(dcbx, chv, k + 1) * a[k];
        botv += M4(cofvbx, ic, k + 1) * b[k];
      }
    if (j0 + L >= nx) {
      T q[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        q[k] = (qv + (size_t)(nx - 1 - k) * P)[w.l];
        topc += M5(dcbx, chv + 2, k + 1) * (gp + (size_t)(nx - 1 - k) * P)[w.l];
        topv += M4(cofvbx, ic + 1, k + 1) * q[k];
      }
      flow = T(1) * (q[0] - q[1]) * idx + rex * T(0); // outflow row
    }
    XFENCE();
    T y = 0, z = 0;
#pragma unroll
    for (int r = 0; r < L; ++r) {
      if (r % XGRP == 0) XFENCE();
      const int j = j0 + r;
      const T g0 = a[r], q0 = b[r], q1 = r + 1 < L ? b[r + 1] : qn;
      T rc = tc.E(1, r) * gm + tc.E(2, r) * g0;
      T rv = tv.E(3, r) * q1 + tv.E(2, r) * q0 + tv.E(1, r) * qm;
      rc = j == 0 ? botc : rc;
      rv = j == 0 ? botv : rv;
      rc = j == nx - 1 ? topc : rc;
      rv = j == nx - 1 ? topv : rv;
      y = rc + tc.M(r) * y;
      z = rv + tv.M(r) * z;
      a[r] = y;
      b[r] = z;
      gm = g0;
      qm = q0;
    }
    XFENCE();
    xback<L>(a, tc);
    xback<L>(b, tv);
    xch[w.p * 64 + w.lane] = y;
    xch[XCT + w.p * 64 + w.lane] = a[0];
    xch[2 * XCT + w.p * 64 + w.lane] = z;
    xch[3 * XCT + w.p * 64 + w.lane] = b[0];
  }
  __syncthreads();
  if (!w.own) return;
  T C, D, Cv, Dv;
  xcarry(xch, xch + XCT, tc, w, x.depth, C, D);
  xcarry(xch + 2 * XCT, xch + 3 * XCT, tv, w, x.depth, Cv, Dv);
#pragma unroll
  for (int r0 = 0; r0 < L; r0 += XGRP) {
    XFENCE();
    T prev[XGRP];
#pragma unroll
    for (int r = 0; r < XGRP; ++r) prev[r] = mode == 1 ? (out + (size_t)min(j0 + r0 + r, nx - 1) * P)[w.l] : T(0);
#pragma unroll
    for (int k = 0; k < XGRP; ++k) {
      const int r = r0 + k, j = j0 + r;
      const T xc = a[r] + fma(C, tc.G(r), D * tc.S(r)), xv = b[r] + fma(Cv, tv.G(r), Dv * tv.S(r));
      const T o = j == nx - 1 ? flow : prev[k] + (xc + rex * xv);
      if (w.ok && j < nx) (out + (size_t)j * P)[w.l] = o;
    }
  }
}

template <int L, typename T>
__global__ void __launch_bounds__(XCT, sizeof(T) == 4 ? 8 : 4)
difvisxx_c(const T *__restrict__ gp, const T *__restrict__ qv, T *__restrict__ out, const T *__restrict__ tabc,
           const T *__restrict__ tabv, const T *__restrict__ dcbx, const T *__restrict__ cofvbx, int chv, int ic,
           int nx, size_t P, double rex, double idx, int mode, XChunk x) {
  __shared__ T xch[4 * XCT];
  difvisxx_b<L, T>(gp, qv, out, tabc, tabv, dcbx, cofvbx, chv, ic, nx, P, rex, idx, mode, x, xch);
}

template <int L, typename T>
__global__ void __launch_bounds__(XCT, sizeof(T) == 4 ? 8 : 4)
difvisxx3_c(XOps<T> a, const T *__restrict__ dcbx, const T *__restrict__ cofvbx, int nx, double rex, double idx,
           XChunk x) {
  __shared__ T xch[4 * XCT];
  const XOp<T> &o = a.op[blockIdx.y];
  difvisxx_b<L, T>(o.in, o.vel, o.out, o.tab, o.tabv, dcbx, cofvbx, o.c1, o.c2, nx, o.P, rex, idx, o.mode, x, xch);
}

#define XDISPATCH(x, ...)                                                    \
  switch ((x).L) {                                                             \
  case 4: { constexpr int L = 4; __VA_ARGS__; } break;                         \
  case 8: { constexpr int L = 8; __VA_ARGS__; } break;                         \
  case 12: { constexpr int L = 12; __VA_ARGS__; } break;                       \
  case 16: { constexpr int L = 16; __VA_ARGS__; } break;                       \
  case 20: { constexpr int L = 20; __VA_ARGS__; } break;                       \
  case 24: { constexpr int L = 24; __VA_ARGS__; } break;                       \
  default: throw std::invalid_argument("x chunk length not instantiated");     \
  }

template <typename T> static const T *xtab_of(const Box &b, int sys) {
  const size_t at = sys < XT_DCXU ? sys * xtab_size(b.xci) : 2 * xtab_size(b.xci) + (sys - XT_DCXU) * xtab_size(b.xcd);
  if constexpr (sizeof(T) == 8) return b.xtab + at;
  else return b.xtab_f + at;
}

template <typename T>
static XOp<T> x_interp_op(Box &b, const T *gen, T *geni, int which_u, int chi, int chi2, size_t P) {
  return {gen, nullptr, geni, xtab_of<T>(b, which_u ? XT_INXU : XT_INXV), nullptr, chi, chi2, 0, P};
}
template <typename T>
static XOp<T> x_difvis_op(Box &b, const T *prod, const T *vel, T *out, int which_u, int chv, int ic, size_t P,
                          int mode) {
  return {prod, vel, out, xtab_of<T>(b, which_u ? XT_DCXU : XT_DCXV), xtab_of<T>(b, which_u ? XT_VIXU : XT_VIXV), chv,
          ic, mode, P};
}
template <typename T> void kxc_interpxx(Box &b, const T *gen, T *geni, int which_u, int chi, int chi2, size_t P) {
  const unsigned grid = nblk(P, 64) * (unsigned)b.xci.ns;
  XDISPATCH(b.xci, auto kf = &interpxx_c<L, T>;
            LAUNCH(b, "interpxx", grid, XCT, 0, kf, gen, geni, xtab_of<T>(b, which_u ? XT_INXU : XT_INXV),
                   coefs<T>(b).inbx, chi, chi2, b.nx, P, b.xci));
}

template <typename T>
void kxc_difvisxx(Box &b, const T *prod, const T *vel, T *out, int which_u, int chv, int ic, size_t P, int mode) {
  const unsigned grid = nblk(P, 64) * (unsigned)b.xcd.ns;
  XDISPATCH(b.xcd, auto kf = &difvisxx_c<L, T>;
            LAUNCH(b, "difvisxx", grid, XCT, 0, kf, prod, vel, out, xtab_of<T>(b, which_u ? XT_DCXU : XT_DCXV),
                   xtab_of<T>(b, which_u ? XT_VIXU : XT_VIXV), coefs<T>(b).dcbx, coefs<T>(b).cofvbx, chv, ic, b.nx, P,
                   b.hc.rex, b.hc.idx, mode, b.xcd));
}

// three operators in one launch; a shorter plane's last workgroups repeat its
// last line without storing
template <typename T> static void x_interp_launch(Box &b, const XOps<T> &a) {
  const dim3 grid(nblk(a.op[0].P, 64) * (unsigned)b.xci.ns, 3);
  XDISPATCH(b.xci, auto kf = &interpxx3_c<L, T>; LAUNCH(b, "interpxx", grid, XCT, 0, kf, a, coefs<T>(b).inbx, b.nx, b.xci));
}
template <typename T> static void x_difvis_launch(Box &b, const XOps<T> &a) {
  const dim3 grid(nblk(a.op[0].P, 64) * (unsigned)b.xcd.ns, 3);
  XDISPATCH(b.xcd, auto kf = &difvisxx3_c<L, T>;
            LAUNCH(b, "difvisxx", grid, XCT, 0, kf, a, coefs<T>(b).dcbx, coefs<T>(b).cofvbx, b.nx, b.hc.rex, b.hc.idx,
                   b.xcd));
}

// The three interpolations, or derivatives, of a substep (u, v, w) in one launch:
// apart, each leaves part of the chip idle in small boxes and drains it in larger
// ones.  us per substep, three launches -> one, interpxx / difvisxx: 32 x 40 x 24
// FP64 20 / 24 -> 7 / 8, 256 x 96 x 64 FP64 38 / 59 -> 18 / 27, 387 x 113 x 98
// mixed 35 / 54 -> 26 / 40, 896 x 176 x 224 FP64 287 / 568 -> 266 / 541, 1536 x 315
// x 1024 mixed interpxx 1992 -> 1968.
template <typename T> bool kxc_interpxx3(Box &b, const T *const *gen, T *const *geni) {
  if (!b.xchunk) return false;
  x_interp_launch<T>(b,
                     {{x_interp_op<T>(b, gen[0], geni[0], 1, 2, 3, b.pu), x_interp_op<T>(b, gen[1], geni[1], 0, 1, 4, b.pv),
                       x_interp_op<T>(b, gen[2], geni[2], 0, 1, 4, b.pu)}});
  return true;
}
template <typename T> bool kxc_difvisxx3(Box &b, const T *const *prod, const T *const *vel, T *const *out) {
  if (!b.xchunk || !b.xcd.L) return false;
  x_difvis_launch<T>(b,
                     {{x_difvis_op<T>(b, prod[0], vel[0], out[0], 1, 1, 3, b.pu, 1),
                       x_difvis_op<T>(b, prod[1], vel[1], out[1], 0, 2, 1, b.pv, 0),
                       x_difvis_op<T>(b, prod[2], vel[2], out[2], 0, 2, 1, b.pu, 0)}});
  return true;
}

#define XINST(T)                                                                                  \
  template void kxc_interpxx<T>(Box &, const T *, T *, int, int, int, size_t);                    \
  template void kxc_difvisxx<T>(Box &, const T *, const T *, T *, int, int, int, size_t, int);    \
  template bool kxc_interpxx3<T>(Box &, const T *const *, T *const *);                            \
  template bool kxc_difvisxx3<T>(Box &, const T *const *, const T *const *, T *const *);
XINST(double)
XINST(float)

} // namespace otbl

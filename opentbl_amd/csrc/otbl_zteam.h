// FFTs along z with several rows per wavefront, for every even length
// 2^a 3^b 5^c 7^d from 12 to 1024; the engine of otbl_zfft.h (one row per
// wavefront or more) keeps FP32 plane loop 1 at 512 and 1024 and the lengths
// above.
//
// A row of N points belongs to a team of G lanes; a wavefront carries
// T = 64 / G teams (lanes past T G idle).  A transform is two or three
// self-sorting Stockham passes with radices up to 16: in pass p (radix R, Ns
// = product of the earlier radices) lane t owns the butterflies j = t + G m,
// j < N / R; its registers hold the inputs x[j + r N / R] and, after the pass,
// the outputs y[(j / Ns) Ns R + (j mod Ns) + q Ns].  The last pass of a
// transform leaves the outputs j + q N / R, the set that the first pass of a
// transform with the radices reversed reads, so products in physical space
// are formed in registers between a forward and an inverse transform.
//
// One row per workgroup in LDS with run-time radices (otbl_fft.h) spends its
// time on index divisions, on two-level twiddles that every workgroup builds
// and on a workgroup barrier per pass: plane loop 1 of a 896 x 176 x 224 FP64
// box took 2610 us for 1.5 GB.  Here the plan is compiled in, a two-pass row
// goes through LDS once per transform, and a team never leaves its wavefront,
// so no pass needs a workgroup barrier (388 us).
#pragma once
#include "otbl_fft.h"

namespace otbl {

// ---------------------------------------------------------------------------
// radix plans
// ---------------------------------------------------------------------------
struct TeamPlan {
  int np = 0;             // passes (0: no plan)
  int r[3] = {1, 1, 1};   // radices of the forward transform
  int g = 0;              // lanes per row
  int e = 0;              // complex values per lane
};

constexpr int kTeamRadix[] = {2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 14, 15, 16};
// real operations of a radix-R butterfly with its twiddles, and of one LDS
// round trip of a value in the same unit
constexpr int team_ops(int r) {
  return r == 2    ? 10
         : r == 3  ? 28
         : r == 4  ? 36
         : r == 5  ? 70
         : r == 6  ? 78
         : r == 7  ? 130
         : r == 8  ? 110
         : r == 9  ? 160
         : r == 10 ? 170
         : r == 12 ? 180
         : r == 14 ? 290
         : r == 15 ? 300
                   : 270;
}
constexpr int kTeamLds = 14;

// The cheapest plan by lane time per row: every pass takes ceil(N / R / G)
// butterflies of a wavefront that 64 / G rows share.  At most emax values
// per lane.
constexpr TeamPlan team_plan_e(int n, int emax) {
  TeamPlan best;
  long cost = -1;
  auto take = [&](int np, int a, int b, int c) {
    const int r[3] = {a, b, c};
    for (int g = 4; g <= 64; ++g) {
      long s = 0;
      int e = 0;
      for (int p = 0; p < np; ++p) {
        const int mb = (n / r[p] + g - 1) / g;
        s += (long)mb * (team_ops(r[p]) + kTeamLds * r[p]);
        e = mb * r[p] > e ? mb * r[p] : e;
      }
      if (e > emax) continue;
      s = s * (64 + e) / (64 / g); // few registers leave more wavefronts in flight
      if (cost < 0 || s < cost) {
        cost = s;
        best.np = np;
        for (int p = 0; p < 3; ++p) best.r[p] = r[p];
        best.g = g;
        best.e = e;
      }
    }
  };
  for (int a : kTeamRadix) {
    if (n % a) continue;
    for (int b : kTeamRadix) {
      if ((n / a) % b) continue;
      const int c = n / a / b;
      if (c == 1) take(2, a, b, 1);
      for (int d : kTeamRadix)
        if (c == d) take(3, a, b, d);
    }
  }
  return best;
}
constexpr TeamPlan team_plan(int n) {
  const TeamPlan p = team_plan_e(n, 16);
  return p.np ? p : team_plan_e(n, 28);
}

template <int N> struct ZRow {
  static constexpr TeamPlan P = team_plan(N);
  static_assert(P.np > 0, "no team plan for this length");
  static constexpr int NP = P.np, G = P.g, E = P.e, T = 64 / P.g;
  static constexpr int rad(int p) { return P.r[p]; }
  // block size and pitch of the exchange after a pass of radix R, Ns: blocks
  // of Ns R outputs, padded so that the strided writes of neighbouring
  // lanes spread over the banks (Ns = 1: an odd pitch; else the next block
  // starts Ns values further modulo 16)
  static constexpr int pitch(int ns, int r) { return ns == 1 ? (r | 1) : ns * r + ((ns - ns * r) % 16 + 16) % 16; }
  // LDS values of a row: the largest exchange, or the N outputs in order
  static constexpr int lds() {
    int most = N;
    for (int inv = 0; inv < 2; ++inv) {
      int ns = 1;
      for (int p = 0; p + 1 < NP; ++p) {
        const int r = rad(inv ? NP - 1 - p : p), v = N / (ns * r) * pitch(ns, r);
        most = v > most ? v : most;
        ns *= r;
      }
    }
    return most | 1;
  }
};

// ---------------------------------------------------------------------------
// butterflies X_q = sum_r v_r exp(S 2 pi i r q / R)
// ---------------------------------------------------------------------------
// odd prime R from the sums and differences of the pairs v_r, v_{R-r}
template <int R, int S, typename C> __device__ __forceinline__ void tbfly_odd(C *v) {
  using T = decltype(v[0].x);
  constexpr int H = R / 2;
  C t[H], d[H];
  C s0 = v[0];
#pragma unroll
  for (int r = 1; r <= H; ++r) {
    t[r - 1] = cadd(v[r], v[R - r]);
    d[r - 1] = csub(v[r], v[R - r]);
    s0 = cadd(s0, t[r - 1]);
  }
#pragma unroll
  for (int q = 1; q <= H; ++q) {
    C a = v[0];
    T bx = 0, by = 0;
#pragma unroll
    for (int r = 1; r <= H; ++r) {
      const int k = (r * q) % R;
      const T cr = (T)odd_cos<R>(k), sr = (T)(S * odd_sin<R>(k));
      a.x += cr * t[r - 1].x;
      a.y += cr * t[r - 1].y;
      // i sr d
      bx -= sr * d[r - 1].y;
      by += sr * d[r - 1].x;
    }
    // v[q], v[R-q] are read by no later q: t, d hold every pair
    const C b = mkc<C>(bx, by);
    v[q] = cadd(a, b);
    v[R - q] = csub(a, b);
  }
  v[0] = s0;
}

template <int R, int S, typename C> __device__ __forceinline__ void tbfly(C *v);

// R = A B, A and B coprime: with inputs n = (B a + A b) mod R,
// n k / R = a k / A + b k / B, so X_k is the two-dimensional transform at
// (k mod A, k mod B): no twiddles
template <int A, int B, int S, typename C> __device__ __forceinline__ void tbfly_pfa(C *v) {
  constexpr int R = A * B;
  C y[A][B];
#pragma unroll
  for (int a = 0; a < A; ++a) {
    C t[B];
#pragma unroll
    for (int b = 0; b < B; ++b) t[b] = v[(B * a + A * b) % R];
    tbfly<B, S>(t);
#pragma unroll
    for (int b = 0; b < B; ++b) y[a][b] = t[b];
  }
#pragma unroll
  for (int b = 0; b < B; ++b) {
    C t[A];
#pragma unroll
    for (int a = 0; a < A; ++a) t[a] = y[a][b];
    tbfly<A, S>(t);
#pragma unroll
    for (int k = 0; k < R; ++k)
      if (k % B == b) v[k] = t[k % A];
  }
}

// R = A B with the twiddles W_R^{b q} between inner transforms of length A
// over the stride-B inputs and outer ones of length B: X[q + A p]
template <int A, int B, int S, typename C> __device__ __forceinline__ void tbfly_ct(C *v) {
  using T = decltype(v[0].x);
  constexpr int R = A * B;
  static_assert(R == 9 || R == 16, "twiddles of 9 and 16 only");
  // cos, sin of 2 pi k / R for the products k = b q of 3 x 3 and 4 x 4
  constexpr double c9[5] = {1.0, 0.76604444311897803520, 0.17364817766693034885, -0.5, -0.93969262078590838405};
  constexpr double s9[5] = {0.0, 0.64278760968653932632, 0.98480775301220805937, 0.86602540378443864676,
                            0.34202014332566873304};
  constexpr double c16[10] = {1.0, 0.92387953251128675613, 0.70710678118654752440, 0.38268343236508977173, 0.0,
                              0.0, -0.70710678118654752440, 0.0, 0.0, -0.92387953251128675613};
  constexpr double s16[10] = {0.0, 0.38268343236508977173, 0.70710678118654752440, 0.92387953251128675613, 1.0,
                              0.0, 0.70710678118654752440, 0.0, 0.0, -0.38268343236508977173};
  C y[B][A];
#pragma unroll
  for (int b = 0; b < B; ++b) {
    C t[A];
#pragma unroll
    for (int a = 0; a < A; ++a) t[a] = v[b + B * a];
    tbfly<A, S>(t);
#pragma unroll
    for (int q = 0; q < A; ++q) {
      const int k = b * q;
      if (k == 0) y[b][q] = t[q];
      else if (R == 16 && k == 4) y[b][q] = mul_si<S>(t[q]);
      else y[b][q] = cmulc(t[q], mkc<C>((T)(R == 9 ? c9[k] : c16[k]), (T)(S * (R == 9 ? s9[k] : s16[k]))));
    }
  }
#pragma unroll
  for (int q = 0; q < A; ++q) {
    C t[B];
#pragma unroll
    for (int b = 0; b < B; ++b) t[b] = y[b][q];
    tbfly<B, S>(t);
#pragma unroll
    for (int p = 0; p < B; ++p) v[q + A * p] = t[p];
  }
}

template <int R, int S, typename C> __device__ __forceinline__ void tbfly(C *v) {
  if constexpr (R == 5 || R == 7) tbfly_odd<R, S>(v);
  else if constexpr (R == 6) tbfly_pfa<2, 3, S>(v);
  else if constexpr (R == 10) tbfly_pfa<2, 5, S>(v);
  else if constexpr (R == 12) tbfly_pfa<4, 3, S>(v);
  else if constexpr (R == 14) tbfly_pfa<2, 7, S>(v);
  else if constexpr (R == 15) tbfly_pfa<3, 5, S>(v);
  else if constexpr (R == 9) tbfly_ct<3, 3, S>(v);
  else if constexpr (R == 16) tbfly_ct<4, 4, S>(v);
  else bfly<R, S>(v);
}

// ---------------------------------------------------------------------------
// passes
// ---------------------------------------------------------------------------
// orders the LDS accesses of a wavefront's lanes
__device__ __forceinline__ void tsync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// whether lane t owns butterfly m of a pass with NB of them (known at compile
// time except for the last, partly filled m)
template <int NB, int G> __device__ __forceinline__ bool town(int t, int m) {
  return G * (m + 1) <= NB || t + G * m < NB;
}

// twiddles of a pass: the powers 1, 2, 4, 8 of W^k, k = j mod Ns, per
// butterfly, from the table exp(2 pi i m / N)
template <int N, int R, int Ns, typename C>
__device__ __forceinline__ void tpass_twload(C (*base)[4], int t, const C *__restrict__ tw) {
  constexpr int G = ZRow<N>::G, NB = N / R, MB = (NB + G - 1) / G, st = N / (Ns * R);
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int k = (t + G * m) % Ns;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if ((1 << q) < R) base[m][q] = tw[k * (1 << q) * st];
  }
}

template <int N, int R, int Ns, int S, typename C>
__device__ __forceinline__ void tpass_compute(C *v, const C (*tb)[4]) {
  constexpr int G = ZRow<N>::G, NB = N / R, MB = (NB + G - 1) / G;
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    C *b = v + m * R;
    if constexpr (Ns > 1) {
      C base[4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if ((1 << q) < R) {
          base[q] = tb[m][q];
          if (S < 0) base[q].y = -base[q].y;
        }
      // W^r, r = lo + 4 hi, as W^lo W^(4 hi): few powers stay live
      C w[4];
#pragma unroll
      for (int lo = 1; lo < 4 && lo < R; ++lo) w[lo] = lo == 3 ? cmulc(base[0], base[1]) : base[lo - 1];
#pragma unroll
      for (int hi = 0; 4 * hi < R; ++hi) {
        const C wh = hi == 3 ? cmulc(base[2], base[3]) : base[hi == 2 ? 3 : 2];
#pragma unroll
        for (int lo = 0; lo < 4; ++lo) {
          const int r = 4 * hi + lo;
          if (r == 0 || r >= R) continue;
          b[r] = cmulc(b[r], hi == 0 ? w[lo] : (lo == 0 ? wh : cmulc(w[lo], wh)));
        }
      }
    }
    tbfly<R, S>(b);
  }
}

// outputs of a pass (R, Ns) to LDS
template <int N, int R, int Ns, typename C> __device__ __forceinline__ void tpass_store(const C *v, int t, C *lds) {
  constexpr int G = ZRow<N>::G, NB = N / R, MB = (NB + G - 1) / G, PB = ZRow<N>::pitch(Ns, R);
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int j = t + G * m, at = (j / Ns) * PB + j % Ns;
    if (town<NB, G>(t, m)) {
#pragma unroll
      for (int q = 0; q < R; ++q) lds[at + q * Ns] = v[m * R + q];
    }
  }
}

// inputs of a pass of radix R from LDS, left there by a pass with blocks of
// BS outputs at pitch PB; a butterfly past the last holds zeros
template <int N, int R, int BS, int PB, typename C> __device__ __forceinline__ void tpass_load(C *v, int t, const C *lds) {
  constexpr int G = ZRow<N>::G, NB = N / R, MB = (NB + G - 1) / G;
  static_assert(NB % BS == 0, "a butterfly's inputs lie whole blocks apart");
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int j = t + G * m, at = (j / BS) * PB + j % BS;
    const bool own = town<NB, G>(t, m);
#pragma unroll
    for (int r = 0; r < R; ++r) v[m * R + r] = mkc<C>(0.0, 0.0);
    if (own) {
#pragma unroll
      for (int r = 0; r < R; ++r) v[m * R + r] = lds[at + r * (NB / BS) * PB];
    }
  }
}

// passes P.. of a transform (Inv: the radices reversed), sign S; v holds the
// inputs of pass P, then the outputs of the last pass
template <int N, int S, bool Inv, int P, int Ns, typename C>
__device__ __forceinline__ void trun_from(C *v, int t, const C *__restrict__ tw, C *lds, const C (*tb)[4]) {
  using Z = ZRow<N>;
  constexpr int R = Z::rad(Inv ? Z::NP - 1 - P : P);
  tpass_compute<N, R, Ns, S>(v, tb);
  if constexpr (P + 1 < Z::NP) {
    constexpr int R2 = Z::rad(Inv ? Z::NP - 2 - P : P + 1);
    C tb2[(N / R2 + Z::G - 1) / Z::G][4];
    tpass_twload<N, R2, Ns * R>(tb2, t, tw);
    tpass_store<N, R, Ns>(v, t, lds);
    tsync();
    tpass_load<N, R2, Ns * R, Z::pitch(Ns, R)>(v, t, lds);
    tsync();
    trun_from<N, S, Inv, P + 1, Ns * R>(v, t, tw, lds, tb2);
  }
}
template <int N, int S, bool Inv, typename C>
__device__ __forceinline__ void trun(C *v, int t, const C *__restrict__ tw, C *lds) {
  trun_from<N, S, Inv, 0, 1>(v, t, tw, lds, (const C(*)[4]) nullptr);
}

// radix and butterflies per lane of the physical side (the forward
// transform's last pass): slot m R + q of lane t is point t + G m + q N / R.
// REV, here and below: the forward transform takes the radices reversed (and the
// inverse as they are)
template <int N, bool REV = false> struct ZRowPhys {
  static constexpr int R = ZRow<N>::rad(REV ? 0 : ZRow<N>::NP - 1), NB = N / R, MB = (NB + ZRow<N>::G - 1) / ZRow<N>::G;
  static constexpr int E = MB * R;
};

// ---------------------------------------------------------------------------
// spectral rows
// ---------------------------------------------------------------------------
// Rows are addressed as a pointer that is the same for the whole wavefront and
// the lane's row as an offset of values (complex): a scalar base and one
// 32-bit register per address.  The rows of a wavefront follow each other, so
// the offsets are small.  (A 16-byte access needs 4-byte alignment.)
template <typename C, typename R> __device__ __forceinline__ C tld(const R *base, unsigned at) {
  return *(const C *)((const char *)base + at * (unsigned)sizeof(C));
}
template <typename C, typename R> __device__ __forceinline__ void tst(R *base, unsigned at, C v) {
  *(C *)((char *)base + at * (unsigned)sizeof(C)) = v;
}

// The first pass's inputs from the spectra of two real signals x, y (modes
// 0..nz2 = N/3 - 1): the Hermitian-extended spectrum of x + i y, where get(k, x, y)
// gives both signals' mode k (PAIR false: y is absent).  Slots that lie in the
// zero band nz2 < k < N - nz2 for every lane load nothing, slots wholly on one
// side of it need no select.
template <int N, bool PAIR, typename C, bool REV = false, class Get>
__device__ __forceinline__ void tload_modes(C *v, int t, Get get) {
  using R = decltype(v[0].x);
  constexpr int G = ZRow<N>::G, RD = ZRow<N>::rad(REV ? ZRow<N>::NP - 1 : 0), NB = N / RD, MB = (NB + G - 1) / G, nz2 = N / 3 - 1;
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int r = 0; r < RD; ++r) {
      constexpr int last = NB; // butterflies
      const int lo = G * m + r * NB, hi = (G * (m + 1) < last ? G * (m + 1) : last) - 1 + r * NB; // first, last index
      const bool full = G * (m + 1) <= NB;
      const int k = t + lo;
      C z = mkc<C>(0.0, 0.0);
      if (lo <= nz2 || hi >= N - nz2) {
        // a lane without a butterfly here, or in the zero band, reads mode 0
        // and drops it
        const bool own = town<NB, G>(t, m);
        const bool low = hi <= nz2 || (lo < N - nz2 && k <= nz2), high = lo >= N - nz2 || (hi > nz2 && k >= N - nz2);
        const bool use = own && (low || high);
        unsigned kk = low ? k : N - k;
        if (!(full && (hi <= nz2 || lo >= N - nz2))) kk = use ? kk : 0u;
        C x, y = mkc<C>(0.0, 0.0);
        get(kk, x, y);
        const R s = low ? R(-1) : R(1);
        z = PAIR ? mkc<C>(x.x + s * y.y, -s * x.y + y.x) : mkc<C>(x.x, -s * x.y);
        if (lo == 0) z = k == 0 ? mkc<C>(x.x, y.x) : z; // Im of mode 0 does not enter
        if (!(full && (hi <= nz2 || lo >= N - nz2)) && !use) z = mkc<C>(0.0, 0.0);
      }
      v[m * RD + r] = z;
    }
}

// the same from the signals' spectral rows
template <int N, bool PAIR, bool REV = false, typename R>
__device__ __forceinline__ void tload_spectral(typename CT<R>::c *v, int t, const R *X, unsigned ox, const R *Y,
                                               unsigned oy) {
  using C = typename CT<R>::c;
  tload_modes<N, PAIR, C, REV>(v, t, [&](unsigned k, C &x, C &y) {
    x = tld<C>(X, ox + k);
    if (PAIR) y = tld<C>(Y, oy + k);
  });
}

// After the last inverse pass (outputs j + q N / R in order): the spectra of
// a and b of the transform of a + i b, modes 0..nz2, scaled by 1 / N (a null
// B is not written), plus mean-flow terms A_0 += c0a XA_0, A_k += cka XA_k and
// B_k += cb XB_k (XA at A's offset, read before A is written: it may be A; XB, B
// likewise).
template <int N, typename R, bool REV = false>
__device__ __forceinline__ void tstore_spectral(const typename CT<R>::c *v, int t, typename CT<R>::c *lds, R *A,
                                                unsigned oa, R *B, unsigned ob, const R *XA = nullptr, R c0a = R(0),
                                                R cka = R(0), const R *XB = nullptr, R cb = R(0)) {
  using C = typename CT<R>::c;
  constexpr int G = ZRow<N>::G, RD = ZRow<N>::rad(REV ? ZRow<N>::NP - 1 : 0), NB = N / RD, MB = (NB + G - 1) / G, nz2 = N / 3 - 1;
  constexpr int NI = (nz2 + G) / G; // trips over the nz2 + 1 modes
#pragma unroll
  for (int m = 0; m < MB; ++m)
    if (town<NB, G>(t, m)) {
#pragma unroll
      for (int q = 0; q < RD; ++q) {
        const int lo = G * m + q * NB, hi = (G * (m + 1) < NB ? G * (m + 1) : NB) - 1 + q * NB;
        if (!(lo > nz2 && hi < N - nz2)) lds[t + lo] = v[m * RD + q];
      }
    }
  C xa[NI], xb[NI];
#pragma unroll
  for (int it = 0; it < NI; ++it) {
    const int k = t + G * it < nz2 ? t + G * it : nz2;
    xa[it] = XA ? tld<C>(XA, oa + k) : mkc<C>(0.0, 0.0);
    xb[it] = XB ? tld<C>(XB, ob + k) : mkc<C>(0.0, 0.0);
  }
  tsync();
  const R sc = R(1.0 / N);
#pragma unroll
  for (int it = 0; it < NI; ++it) {
    const int k = t + G * it;
    if (k <= nz2) {
      const C z = lds[k], w = lds[k ? N - k : 0];
      R ar = R(0.5) * (z.x + w.x) * sc, ai = (k == 0) ? R(0) : R(0.5) * (z.y - w.y) * sc;
      if (XA) {
        ar += (k == 0 ? c0a : cka) * xa[it].x;
        ai += (k == 0) ? R(0) : cka * xa[it].y;
      }
      tst(A, oa + k, mkc<C>(ar, ai));
      if (B) {
        R br = R(0.5) * (z.y + w.y) * sc, bi = (k == 0) ? R(0) : R(-0.5) * (z.x - w.x) * sc;
        if (XB) {
          br += cb * xb[it].x;
          bi += (k == 0) ? R(0) : cb * xb[it].y;
        }
        tst(B, ob + k, mkc<C>(br, bi));
      }
    }
  }
  tsync();
}

} // namespace otbl

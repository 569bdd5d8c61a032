// Lines split into chunks over the wavefronts of a workgroup: the table of one
// factored tridiagonal system, a wavefront's place in a line, the backward
// sweep of a chunk and its carries (see otbl_xchunk.hip for the method).
#pragma once
#include "otbl_kcommon.h"

namespace otbl {

static constexpr int XCT = 64 * XCH; // threads per workgroup

// one system's table at a chunk (wave-uniform: scalar loads): per plane FS
// forward values (the explicit stencil, then the multiplier M), A2, B; G, S;
// then per chunk PE, G0, S0, 0
template <typename T, int FS = 4> struct XTabP {
  const T *f, *k, *g, *e; // this chunk's rows; e: every chunk's values
  __device__ __forceinline__ XTabP(const T *tab, const XChunk &x, int L, int chunk) {
    const size_t NL = (size_t)x.nc * L, j0 = (size_t)chunk * L;
    f = tab + FS * j0;
    k = tab + FS * NL + 2 * j0;
    g = tab + (FS + 2) * NL + 2 * j0;
    e = tab + (FS + 4) * NL;
  }
  __device__ __forceinline__ T M(int r) const { return f[FS * r + FS - 1]; }
  __device__ __forceinline__ T E(int q, int r) const { return f[FS * r + q - 1]; }
  __device__ __forceinline__ T A2(int r) const { return k[2 * r]; }
  __device__ __forceinline__ T B(int r) const { return k[2 * r + 1]; }
  __device__ __forceinline__ T G(int r) const { return g[2 * r]; }
  __device__ __forceinline__ T S(int r) const { return g[2 * r + 1]; }
  __device__ __forceinline__ T PE(int q) const { return e[4 * q]; }
  __device__ __forceinline__ T G0(int q) const { return e[4 * q + 1]; }
  __device__ __forceinline__ T S0(int q) const { return e[4 * q + 2]; }
};

// a wavefront's chunk c = c0 + p of the nact its workgroup holds
struct ChunkAt {
  int p, lane, c0, nact, c;
};

// a wavefront's place in an x line, and whether it stores
struct XPlace : ChunkAt {
  unsigned l;
  bool act, own, ok;
  __device__ __forceinline__ XPlace(const XChunk &x, size_t P) {
    lane = threadIdx.x & 63;
    p = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned bk = xcd_block(); // neighbouring spans and lines on one XCD
    const unsigned grp = bk / (unsigned)x.ns, sp = bk - grp * x.ns;
    const size_t lg = (size_t)grp * 64 + lane;
    ok = lg < P;
    l = (unsigned)(ok ? lg : P - 1); // a dead lane repeats the last line
    const int u0 = (int)((long)sp * x.nc / x.ns), u1 = (int)((long)(sp + 1) * x.nc / x.ns);
    c0 = max(0, u0 - x.halo);
    nact = min(x.nc, u1 + x.halo) - c0;
    act = p < nact;
    c = c0 + min(p, nact - 1);
    own = act && c >= u0 && c < u1;
  }
};

#define XFENCE() __builtin_amdgcn_sched_barrier(0)
static constexpr int XGRP = 4; // rows per scheduling group of the sweeps

// backward local sweep of a chunk from its forward one (v holds y); the product
// that is rounded on its own is the smaller one, as in the correction v + (C g + D s)
// (the other way: 15% more error than one sweep over the whole line)
template <int L, typename T, int FS> __device__ __forceinline__ void xback(T (&v)[L], const XTabP<T, FS> &t) {
  v[L - 1] = t.A2(L - 1) * v[L - 1];
#pragma unroll
  for (int r = L - 2; r >= 0; --r) {
    if (r % XGRP == 0) XFENCE();
    v[r] = fma(t.A2(r), v[r], t.B(r) * v[r + 1]);
  }
  XFENCE();
}

// carries of chunk p from the chunks' ends in LDS (ye: y at the last plane,
// xs: x_local at the first)
template <typename T, int FS>
__device__ __forceinline__ void xcarry(const T *ye, const T *xs, const XTabP<T, FS> &t, const ChunkAt &w, int depth,
                                       T &C, T &D) {
  C = 0;
  for (int q = max(0, w.p - depth); q < w.p; ++q) C = ye[q * 64 + w.lane] + t.PE(w.c0 + q) * C;
  T Cq = C, prod = 1;
  D = 0;
  const int q1 = min(w.nact - 1, w.p + depth);
  for (int q = w.p + 1; q <= q1; ++q) {
    Cq = ye[(q - 1) * 64 + w.lane] + t.PE(w.c0 + q - 1) * Cq;
    D += prod * (xs[q * 64 + w.lane] + t.G0(w.c0 + q) * Cq);
    prod *= t.S0(w.c0 + q);
  }
}

} // namespace otbl

// Device side of the matrix-free sigma-coordinate Poisson operator and its
// geometric multigrid preconditioner (see nhw_mg.hip for the method), shared
// by the single-scenario solver and the batched one.
#pragma once
#include <type_traits>

#include "nhw_krylov_dev.h"
#include "nhw_impl.h"

namespace nhw {

constexpr int kBSm = 256;

// calls f(std::integral_constant<int, KM>) with the smallest row bucket KM in
// {4, 6, 8, 10, 12, 16} up to KMX that holds K rows: the column kernels keep a
// column's rows in registers and unroll over the bucket, so a bucket that
// fits saves the work on rows that are not there (K = 10 in 12 rows: 10 % of
// k_mg_down and k_mg_up).  K is uniform per workgroup.
template <int KMX, class F>
__host__ __device__ __forceinline__ void by_rows(int K, F &&f) {
  if constexpr (KMX > 4) {
    constexpr int below = KMX == 16 ? 12 : KMX - 2;
    if (K <= below) {
      by_rows<below>(K, f);
      return;
    }
  }
  f(std::integral_constant<int, KMX>());
}

// per-sigma-level constants of one multigrid level, in the vector type: a
// small device table read with scalar loads where a row needs them (kernel
// arguments would hold all of them in scalar registers at once)
template <class V>
struct LvlK {
  V sig, r6, r13, rx, ry;
};
// per-level constants, in the vector type
template <class V>
struct LvlC {
  int M, N, K;
  long MN;
  V cxy, idx2, idy2;
  const LvlK<V> *kc;  // [K]
};

template <class V>
struct G2 {
  const V *ax, *bx, *ay, *by, *rd;
  int ld;  // (M+2): halo layout, interior (i,j) at (i+1) + ld*(j+1)
  __device__ long at(int i, int j) const { return (long)(i + 1) + (long)ld * (j + 1); }
};

template <class V>
struct ColGeo {
  V axc, bxc, ayc, byc, rd, axm, bxm, axp, bxp, aym, bym, ayp, byp;
  bool w, e, s, n;
};

// element idx of an array at a uniform base, addressed through a 32-bit
// byte offset so the load takes the scalar-base + vector-offset form (one
// VGPR per address, not two).  Every sigma plane and every 2-D field stays
// below 4 GiB.
template <class V>
__device__ __forceinline__ V ldo(const V *__restrict__ base, unsigned idx) {
  return *(const V *)((const char *)base + (unsigned)(idx * (unsigned)sizeof(V)));
}
template <class V>
__device__ __forceinline__ void sto(V *__restrict__ base, unsigned idx, V v) {
  *(V *)((char *)base + (unsigned)(idx * (unsigned)sizeof(V))) = v;
}

template <class V>
__device__ __forceinline__ ColGeo<V> load_col(const G2<V> &G, const LvlC<V> &L, int i, int j) {
  ColGeo<V> g;
  const unsigned c = (unsigned)(i + 1) + (unsigned)G.ld * (unsigned)(j + 1), ld = (unsigned)G.ld;
  g.axc = ldo(G.ax, c); g.bxc = ldo(G.bx, c); g.ayc = ldo(G.ay, c); g.byc = ldo(G.by, c); g.rd = ldo(G.rd, c);
  g.axm = ldo(G.ax, c - 1); g.bxm = ldo(G.bx, c - 1); g.axp = ldo(G.ax, c + 1); g.bxp = ldo(G.bx, c + 1);
  g.aym = ldo(G.ay, c - ld); g.bym = ldo(G.by, c - ld); g.ayp = ldo(G.ay, c + ld); g.byp = ldo(G.by, c + ld);
  g.w = i == 0; g.e = i == L.M - 1; g.s = j == 0; g.n = j == L.N - 1;
  return g;
}

// the 15 coefficients of row (i,j,k) in JCoef order (c[0] = centre), folds
// applied in the reference's order (west, east, south, north, bottom, top),
// src/pressure.F:540-555, 649-814
template <class V>
__device__ __forceinline__ void coefs(const LvlC<V> &L, const ColGeo<V> &g, int k, V c[15]) {
  const LvlK<V> kk = L.kc[k];
  const V sg = kk.sig;
  const V dxs = g.axc - sg * g.bxc, dxm = g.axm - sg * g.bxm, dxp = g.axp - sg * g.bxp;
  const V dys = g.ayc - sg * g.byc, dym = g.aym - sg * g.bym, dyp = g.ayp - sg * g.byp;
  const V A1 = dxs * dxs + dys * dys + g.rd * g.rd;
  const V z = V(0);
  c[0] = L.cxy + A1 * (kk.r6 + kk.r13);
  c[1] = -L.idx2; c[8] = -L.idx2;
  c[2] = -L.idy2; c[9] = -L.idy2;
  c[3] = (dym + dys) * kk.ry; c[14] = -c[3];
  c[4] = (dxm + dxs) * kk.rx; c[13] = -c[4];
  c[5] = -A1 * kk.r6; c[12] = -A1 * kk.r13;
  c[6] = -(dxp + dxs) * kk.rx; c[11] = -c[6];
  c[7] = -(dyp + dys) * kk.ry; c[10] = -c[7];
  if (g.w) { c[0] += c[8]; c[5] += c[4]; c[12] += c[13]; c[8] = z; c[4] = z; c[13] = z; }
  if (g.e) { c[0] += c[1]; c[5] += c[6]; c[12] += c[11]; c[1] = z; c[6] = z; c[11] = z; }
  if (g.s) { c[0] += c[9]; c[5] += c[3]; c[12] += c[14]; c[9] = z; c[3] = z; c[14] = z; }
  if (g.n) { c[0] += c[2]; c[5] += c[7]; c[12] += c[10]; c[2] = z; c[7] = z; c[10] = z; }
  if (k == 0) {
    c[5] += c[12]; c[6] += c[11]; c[7] += c[10]; c[4] += c[13]; c[3] += c[14];
    c[12] = z; c[11] = z; c[10] = z; c[13] = z; c[14] = z;
  }
  if (k == L.K - 1) { c[3] = z; c[4] = z; c[5] = z; c[6] = z; c[7] = z; }
}

// plane offsets (zebra layout) of a column and of its four x-y neighbours,
// clamped so every read is in bounds (a clamped neighbour always carries a
// folded, zero coefficient)
struct Nb {
  unsigned c, xm, xp, ym, yp;
};
template <class V>
__device__ __forceinline__ Nb nbrs(const LvlC<V> &L, int i, int j) {
  Nb o;
  o.c = (unsigned)zcol(i, j, L.M);
  o.xm = i > 0 ? (unsigned)zcol(i - 1, j, L.M) : o.c;
  o.xp = i < L.M - 1 ? (unsigned)zcol(i + 1, j, L.M) : o.c;
  o.ym = j > 0 ? (unsigned)zcol(i, j - 1, L.M) : o.c;
  o.yp = j < L.N - 1 ? (unsigned)zcol(i, j + 1, L.M) : o.c;
  return o;
}

// sigma plane k of a level vector (a uniform pointer)
template <class V, class P>
__device__ __forceinline__ P *plane(P *x, const LvlC<V> &L, int k) {
  return x + (long)k * L.MN;
}

// the five values of one sigma plane a row's stencil reads: the column and
// its four x-y neighbours (clamped offsets)
template <class V>
struct Pl {
  V c, xm, xp, ym, yp;
};
template <class V>
__device__ __forceinline__ Pl<V> load_pl(const V *__restrict__ xk, const Nb &o) {
  return Pl<V>{ldo(xk, o.c), ldo(xk, o.xm), ldo(xk, o.xp), ldo(xk, o.ym), ldo(xk, o.yp)};
}
// (A x) at a row from the planes below (pv), at (cu) and above (nx) it; at
// the bottom and top rows the missing plane carries zero coefficients
template <class V>
__device__ __forceinline__ V arow3(const V c[15], const Pl<V> &pv, const Pl<V> &cu, const Pl<V> &nx) {
  return c[0] * cu.c + c[5] * nx.c + c[12] * pv.c + c[1] * cu.xp + c[2] * cu.yp + c[8] * cu.xm + c[9] * cu.ym +
         c[3] * nx.ym + c[4] * nx.xm + c[6] * nx.xp + c[7] * nx.yp + c[10] * pv.yp + c[11] * pv.xp +
         c[13] * pv.xm + c[14] * pv.ym;
}

// Per-column constants of the smoother's and the restriction's rows: the
// operator of coefs(), re-associated for fewer operations (neighbour sums
// formed once per column, the x/y folds of the reference turned into
// per-column terms, fused multiply-adds).  Rounding differs from coefs() in
// the last bits, which the multigrid preconditioner tolerates; the Krylov
// operator itself (mf_col) keeps coefs().
template <class V>
struct ColC {
  V axc, bxc, ayc, byc, rd2, c0b;
  V Axm, Bxm, Axp, Bxp, Aym, Bym, Ayp, Byp;  // neighbour + column sums, 0 on a folded side
  V FAx, FBx, FAy, FBy;                      // the folded sides' sums, moved onto the column
  V hxm, hxp, hym, hyp;                      // same-plane couplings, 0 on a folded side
};
template <class V>
__device__ __forceinline__ ColC<V> col_consts(const G2<V> &G, const LvlC<V> &L, int i, int j) {
  const ColGeo<V> g = load_col(G, L, i, j);
  ColC<V> q;
  q.axc = g.axc; q.bxc = g.bxc; q.ayc = g.ayc; q.byc = g.byc; q.rd2 = g.rd * g.rd;
  const V o = V(1), z = V(0);
  const V kxm = g.w ? z : o, kxp = g.e ? z : o, kym = g.s ? z : o, kyp = g.n ? z : o;
  const V Axm = g.axm + g.axc, Bxm = g.bxm + g.bxc, Axp = g.axp + g.axc, Bxp = g.bxp + g.bxc;
  const V Aym = g.aym + g.ayc, Bym = g.bym + g.byc, Ayp = g.ayp + g.ayc, Byp = g.byp + g.byc;
  q.Axm = kxm * Axm; q.Bxm = kxm * Bxm; q.Axp = kxp * Axp; q.Bxp = kxp * Bxp;
  q.Aym = kym * Aym; q.Bym = kym * Bym; q.Ayp = kyp * Ayp; q.Byp = kyp * Byp;
  // west / east fold c4 / c6 onto c5 (and their negatives onto c12), south /
  // north fold c3 / c7; c4 = (Axm - sg Bxm) rx, c6 = -(Axp - sg Bxp) rx,
  // c3 = (Aym - sg Bym) ry, c7 = -(Ayp - sg Byp) ry
  q.FAx = (o - kxm) * Axm - (o - kxp) * Axp; q.FBx = (o - kxm) * Bxm - (o - kxp) * Bxp;
  q.FAy = (o - kym) * Aym - (o - kyp) * Ayp; q.FBy = (o - kym) * Bym - (o - kyp) * Byp;
  q.c0b = L.cxy - ((o - kxm) + (o - kxp)) * L.idx2 - ((o - kym) + (o - kyp)) * L.idy2;
  q.hxm = -kxm * L.idx2; q.hxp = -kxp * L.idx2; q.hym = -kym * L.idy2; q.hyp = -kyp * L.idy2;
  return q;
}

// the constants of a column whose other columns are taken as zero: its own
// fields and the folded sides' sums, whose neighbour is a zero halo entry
template <class V>
__device__ __forceinline__ ColC<V> col_consts_centre(const G2<V> &G, const LvlC<V> &L, int i, int j) {
  const unsigned c = (unsigned)(i + 1) + (unsigned)G.ld * (unsigned)(j + 1);
  ColC<V> q{};
  q.axc = ldo(G.ax, c); q.bxc = ldo(G.bx, c); q.ayc = ldo(G.ay, c); q.byc = ldo(G.by, c);
  const V rd = ldo(G.rd, c);
  q.rd2 = rd * rd;
  const V w = V(i == 0), e = V(i == L.M - 1), s = V(j == 0), n = V(j == L.N - 1);
  q.FAx = (w - e) * q.axc; q.FBx = (w - e) * q.bxc;
  q.FAy = (s - n) * q.ayc; q.FBy = (s - n) * q.byc;
  q.c0b = L.cxy - (w + e) * L.idx2 - (s + n) * L.idy2;
  return q;
}

// row k from per-column constants: centre c0, couplings to the rows above
// (c5) and below (c12) in the column, and (OFF) the sum s of the couplings
// to the other columns from the planes below / at / above the row
template <class V>
struct ZRow {
  V c0, c5, c12, s;
};
template <class V, bool OFF>
__device__ __forceinline__ ZRow<V> zrow(const LvlC<V> &L, const ColC<V> &q, int k, const Pl<V> &pv,
                                        const Pl<V> &cu, const Pl<V> &nx) {
  const LvlK<V> e = L.kc[k];
  const V sg = e.sig, rxk = e.rx, ryk = e.ry, r6 = e.r6, r13 = e.r13;
  const V dxs = fma(-sg, q.bxc, q.axc), dys = fma(-sg, q.byc, q.ayc);
  const V A1 = fma(dxs, dxs, fma(dys, dys, q.rd2));
  const V F = fma(rxk, fma(-sg, q.FBx, q.FAx), ryk * fma(-sg, q.FBy, q.FAy));
  const bool top = k == L.K - 1;
  ZRow<V> z;
  z.c0 = fma(A1, r6 + r13, q.c0b);
  V c5 = fma(-A1, r6, F), c12 = fma(-A1, r13, -F);
  if (k == 0) {  // bottom: the ghost row below mirrors the row above
    c5 += c12;
    c12 = V(0);
  }
  z.c5 = top ? V(0) : c5;  // top: zero pressure above
  z.c12 = c12;
  z.s = V(0);
  if (OFF) {
    V s = fma(q.hxp, cu.xp, fma(q.hxm, cu.xm, fma(q.hyp, cu.yp, q.hym * cu.ym)));
    if (k > 0) {  // the diagonal couplings cancel on the bottom row
      const V tm = top ? V(0) : V(1);
      const V c4 = rxk * fma(-sg, q.Bxm, q.Axm), c6 = -rxk * fma(-sg, q.Bxp, q.Axp);
      const V c3 = ryk * fma(-sg, q.Bym, q.Aym), c7 = -ryk * fma(-sg, q.Byp, q.Ayp);
      s = fma(c4, fma(tm, nx.xm, -pv.xm), s);
      s = fma(c6, fma(tm, nx.xp, -pv.xp), s);
      s = fma(c3, fma(tm, nx.ym, -pv.ym), s);
      s = fma(c7, fma(tm, nx.yp, -pv.yp), s);
    }
    z.s = s;
  }
  return z;
}

// (A x) at a row from its zrow and planes
template <class V>
__device__ __forceinline__ V zrow_apply(const ZRow<V> &z, const Pl<V> &pv, const Pl<V> &cu, const Pl<V> &nx) {
  return fma(z.c0, cu.c, fma(z.c5, nx.c, fma(z.c12, pv.c, z.s)));
}

// reciprocal for the Thomas pivots: the hardware estimate refined by Newton
// steps (to about an ulp; the pivots are positive and far from the range
// ends)
__device__ __forceinline__ double rcp_nr(double d) {
  double r = __builtin_amdgcn_rcp(d);
  double e = fma(-d, r, 1.0);
  r = fma(r, e, r);
  e = fma(-d, r, 1.0);
  return fma(r, e, r);
}
__device__ __forceinline__ float rcp_nr(float d) {
  float r = __builtin_amdgcn_rcpf(d);
  return fmaf(r, fmaf(-d, r, 1.0f), r);
}

// deterministic fixed-shape block sum of two values into part[3*block + m]
__device__ __forceinline__ void block_sum2(const double (&acc)[2], double *part) {
  __shared__ double sm[2][kBSm];
  sm[0][threadIdx.x] = acc[0];
  sm[1][threadIdx.x] = acc[1];
  __syncthreads();
  for (int s = kBSm / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      sm[0][threadIdx.x] += sm[0][threadIdx.x + s];
      sm[1][threadIdx.x] += sm[1][threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[3 * blockIdx.x] = sm[0][0];
    part[3 * blockIdx.x + 1] = sm[1][0];
  }
}

// ---------------------------------------------------------------------------
// geometry set-up (always from the FP64 state)
// ---------------------------------------------------------------------------
template <class V>
__global__ void k_geom0(Geo g, Dev d, V *ax, V *bx, V *ay, V *by, V *rd, int ld) {
  long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)g.M * g.N) return;
  const int i = (int)(t % g.M), j = (int)(t / g.M);
  const long c = g.c2(g.Ibeg + i, g.Jbeg + j);
  const long h = (long)(i + 1) + (long)ld * (j + 1);
  const double r = 1.0 / d.D[c];
  ax[h] = (V)(d.DelxH[c] * r);
  bx[h] = (V)((d.DelxH[c] + d.DelxEta[c]) * r);
  ay[h] = (V)(d.DelyH[c] * r);
  by[h] = (V)((d.DelyH[c] + d.DelyEta[c]) * r);
  rd[h] = (V)r;
}

// block average of the five column fields onto the next level
template <class V>
__global__ void k_geom_coarsen(int Mf, int Nf, int ldf, int Mc, int Nc, int ldc, int fx, int fy, const V *axf,
                               const V *bxf, const V *ayf, const V *byf, const V *rdf, V *axc, V *bxc, V *ayc,
                               V *byc, V *rdc) {
  long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)Mc * Nc) return;
  const int I = (int)(t % Mc), J = (int)(t / Mc);
  double s[5] = {0, 0, 0, 0, 0};
  int cnt = 0;
  for (int b = 0; b < fy; ++b)
    for (int a = 0; a < fx; ++a) {
      const int i = I * fx + a, j = J * fy + b;
      if (i >= Mf || j >= Nf) continue;
      const long h = (long)(i + 1) + (long)ldf * (j + 1);
      s[0] += axf[h]; s[1] += bxf[h]; s[2] += ayf[h]; s[3] += byf[h]; s[4] += rdf[h];
      ++cnt;
    }
  const double w = 1.0 / cnt;
  const long h = (long)(I + 1) + (long)ldc * (J + 1);
  axc[h] = (V)(s[0] * w); bxc[h] = (V)(s[1] * w); ayc[h] = (V)(s[2] * w); byc[h] = (V)(s[3] * w);
  rdc[h] = (V)(s[4] * w);
}

// ---------------------------------------------------------------------------
// operator kernels (one thread per column, k loop inside)
// ---------------------------------------------------------------------------

// rows of y = A x for one column (runtime row loop), with the dot partials
template <class V, int NDOT>
__device__ __forceinline__ void mf_col(const LvlC<V> &L, const ColGeo<V> &g, const Nb &o, const V *__restrict__ x,
                                       V *__restrict__ y, const V *__restrict__ d1, double (&acc)[2]) {
  Pl<V> cu = load_pl(x, o);
  Pl<V> nx = L.K > 1 ? load_pl(plane(x, L, 1), o) : cu;
  Pl<V> pv = cu;
#pragma unroll 1
  for (int k = 0; k < L.K; ++k) {
    V c[15];
    coefs(L, g, k, c);
    const V v = arow3(c, pv, cu, nx);
    sto(plane(y, L, k), o.c, v);
    if (NDOT >= 1) acc[0] += (double)v * (double)ldo(plane(d1, L, k), o.c);
    if (NDOT >= 2) acc[1] += (double)v * (double)v;
    pv = cu;
    cu = nx;
    if (k + 2 < L.K) nx = load_pl(plane(x, L, k + 2), o);
  }
}

// y = A x; optional dot partials (y, d1) [and (y, y)], accumulated in FP64.
// One thread walks one column bottom to top, keeping the three sigma planes
// its rows read in registers (each x value is loaded once per column pass).
// A runtime row loop: few registers, so many waves hide the latency.
template <class V, int NDOT>
__global__ __launch_bounds__(kBSm) void k_mf_apply(LvlC<V> L, G2<V> G, const V *__restrict__ x, V *__restrict__ y,
                                                   const V *__restrict__ d1, double *part, const int *stop) {
  if (stop[0]) return;
  double acc[2] = {0.0, 0.0};
  for (long col = (long)xcd_block() * kBSm + threadIdx.x; col < L.MN; col += (long)gridDim.x * kBSm) {
    const int i = (int)(col % L.M), j = (int)(col / L.M);
    const ColGeo<V> g = load_col(G, L, i, j);
    const Nb o = nbrs(L, i, j);
    mf_col<V, NDOT>(L, g, o, x, y, d1, acc);
  }
  if (NDOT > 0) block_sum2(acc, part);
}

// start of a (sub)solve, in the FP64 operator: res = b - A x with x and b
// FP64, into rh in the Krylov type R; partials (res,res), (b,b)
template <class R>
__global__ __launch_bounds__(kBSm) void k_mf_init(LvlC<double> L, G2<double> G, const double *__restrict__ x,
                                                  const double *__restrict__ b, R *__restrict__ rh,
                                                  double *part) {
  double acc[2] = {0.0, 0.0};
  for (long col = (long)xcd_block() * kBSm + threadIdx.x; col < L.MN; col += (long)gridDim.x * kBSm) {
    const int i = (int)(col % L.M), j = (int)(col / L.M);
    const ColGeo<double> g = load_col(G, L, i, j);
    const Nb o = nbrs(L, i, j);
    Pl<double> cu = load_pl(x, o);
    Pl<double> nx = L.K > 1 ? load_pl(plane(x, L, 1), o) : cu;
    Pl<double> pv = cu;
    for (int k = 0; k < L.K; ++k) {
      double c[15];
      coefs(L, g, k, c);
      const long q = (long)k * L.MN + o.c;
      const double bv = b[q];
      const double rv = bv - arow3(c, pv, cu, nx);
      rh[q] = (R)rv;
      acc[0] += rv * rv;
      acc[1] += bv * bv;
      pv = cu;
      cu = nx;
      if (k + 2 < L.K) nx = load_pl(plane(x, L, k + 2), o);
    }
  }
  block_sum2(acc, part);
}

// |b - A x|^2 partials for the solve report (FP64 operator)
static __global__ __launch_bounds__(kBSm) void k_mf_true(LvlC<double> L, G2<double> G, const double *__restrict__ x,
                                                  const double *__restrict__ b, double *part) {
  double acc[2] = {0.0, 0.0};
  for (long col = (long)xcd_block() * kBSm + threadIdx.x; col < L.MN; col += (long)gridDim.x * kBSm) {
    const int i = (int)(col % L.M), j = (int)(col / L.M);
    const ColGeo<double> g = load_col(G, L, i, j);
    const Nb o = nbrs(L, i, j);
    Pl<double> cu = load_pl(x, o);
    Pl<double> nx = L.K > 1 ? load_pl(plane(x, L, 1), o) : cu;
    Pl<double> pv = cu;
    for (int k = 0; k < L.K; ++k) {
      double c[15];
      coefs(L, g, k, c);
      const double rv = ldo(plane(b, L, k), o.c) - arow3(c, pv, cu, nx);
      acc[0] += rv * rv;
      pv = cu;
      cu = nx;
      if (k + 2 < L.K) nx = load_pl(plane(x, L, k + 2), o);
    }
  }
  block_sum2(acc, part);
}

// rows 0..KM-1 of a column, bottom to top: f(k, z, pv, cu, nx) gets row k
// (zrow) and the planes below / at / above it.  Plane reads go
// through offsets clamped to the top row, so every load is in bounds and
// none sits behind a branch (the loads of later rows issue while earlier
// rows compute); rows k >= K re-read the top plane and callers discard them.
template <class V, int KM, class F>
__device__ __forceinline__ void walk_col(const LvlC<V> &L, const ColC<V> &q, const Nb &o,
                                         const V *__restrict__ x, F &&f) {
  const int K1 = L.K - 1;
  Pl<V> pv = load_pl(x, o);
  Pl<V> cu = pv;
  Pl<V> nx = load_pl(plane(x, L, min(1, K1)), o);
#pragma unroll
  for (int k = 0; k < KM; ++k) {
    const Pl<V> nn = load_pl(plane(x, L, min(k + 2, K1)), o);
    f(k, zrow<V, true>(L, q, k, pv, cu, nx), pv, cu, nx);
    pv = cu;
    cu = nx;
    nx = nn;
    // keep the loads of later planes in later iterations: two planes ahead
    // cover the latency, and hoisting all of them costs the occupancy
    __builtin_amdgcn_sched_barrier(0);
  }
}

// rows 0..KM-1 of a column vector at byte offset off (clamped like walk_col)
template <class V, int KM>
__device__ __forceinline__ void load_rows(const V *__restrict__ v, unsigned off, const LvlC<V> &L, V (&out)[KM]) {
  const int K1 = L.K - 1;
#pragma unroll
  for (int k = 0; k < KM; ++k) out[k] = ldo(plane(v, L, min(k, K1)), off);
}

// one step of the Thomas forward elimination of a column's tridiagonal
// (sub c12, diagonal c0, super c5; c12 is zero on the bottom row)
template <class V>
__device__ __forceinline__ void thomas_fwd(const ZRow<V> &z, V r, V &cp, V &dp) {
  const V inv = rcp_nr(fma(-z.c12, cp, z.c0));
  cp = z.c5 * inv;
  dp = fma(-z.c12, dp, r) * inv;
}

// back substitution of a column's eliminated tridiagonal, in registers: r
// holds the eliminated right side on entry and the solution on return
// (entries k >= K are not meaningful)
template <class V, int KM>
__device__ __forceinline__ void col_back(const LvlC<V> &L, const V (&cp)[KM], V (&r)[KM]) {
  const int K1 = L.K - 1;
  V xn = V(0);
#pragma unroll
  for (int k = KM - 1; k >= 0; --k) {
    xn = k >= K1 ? r[k] : fma(-cp[k], xn, r[k]);
    r[k] = xn;
  }
}

// a column's rows into x at plane offset off
template <class V, int KM>
__device__ __forceinline__ void store_rows(const LvlC<V> &L, const V (&r)[KM], V *__restrict__ x, unsigned off) {
#pragma unroll
  for (int k = 0; k < KM; ++k)
    if (k < L.K) sto(plane(x, L, k), off, r[k]);
}

// z-line Gauss-Seidel update of a column, in registers: line_rows solves its
// vertical tridiagonal with the couplings to its neighbours' values in x
// moved to the right side r, zero_rows takes the other columns as zero.
// Forward elimination runs as the rows are formed (only the modified
// super-diagonal and right side are kept); r is overwritten by the solution.
template <class V, int KM>
__device__ __forceinline__ void zero_rows(const LvlC<V> &L, const ColC<V> &q, V (&r)[KM]) {
  V cp[KM];
  V cprev = V(0), dprev = V(0);
  const Pl<V> none{};
#pragma unroll
  for (int k = 0; k < KM; ++k) {
    thomas_fwd(zrow<V, false>(L, q, k, none, none, none), r[k], cprev, dprev);
    cp[k] = cprev;
    r[k] = dprev;
  }
  col_back<V, KM>(L, cp, r);
}

// plane stride of the neighbour values is Lx.MN (Lx differs from L only
// there, for values staged in LDS)
template <class V, int KM>
__device__ __forceinline__ void line_rows(const LvlC<V> &Lx, const ColC<V> &q, const Nb &o, V (&r)[KM],
                                          const V *__restrict__ x) {
  V cp[KM];
  V cprev = V(0), dprev = V(0);
  // the column's own values are the unknowns: only its neighbours are read
  walk_col<V, KM>(Lx, q, o, x, [&](int k, const ZRow<V> &z, const Pl<V> &, const Pl<V> &, const Pl<V> &) {
    thomas_fwd(z, r[k] - z.s, cprev, dprev);
    cp[k] = cprev;
    r[k] = dprev;
  });
  col_back<V, KM>(Lx, cp, r);
}

// The coarsest level (at most kMgCoarseCols columns) solved approximately
// inside one workgroup: `sweeps` zebra pairs from a zero guess with x kept in
// LDS between half sweeps, so the whole solve is one launch.
// Each thread owns at most one column of each colour, whose offsets,
// constants and right side it forms once, before the sweeps.
constexpr int kCoarseBS = 512;
template <class V, int KM>
__device__ __forceinline__ void coarse_solve(const LvlC<V> &L, const G2<V> &G, const V *__restrict__ b,
                                             V *__restrict__ x, int sweeps, V *xs /* LDS, KM * kMgCoarseCols */) {
  const int n = (int)L.MN * L.K;
  // clamped neighbours read the column's own (not yet written) value with a
  // zero coefficient: start from zeros so that product is zero
  for (int q = threadIdx.x; q < n; q += kCoarseBS) xs[q] = V(0);
  // thread t takes the t-th column of each colour (at most kCoarseBS of
  // each, as the level has at most 2 kCoarseBS columns): a pair of rows
  // holds M columns of each colour
  bool on[2];
  Nb o[2];
  ColC<V> q[2];
  V rb[2][KM];
  const int t = threadIdx.x;
#pragma unroll
  for (int colour = 0; colour < 2; ++colour) {
    const int P = t / L.M, rem = t - P * L.M;
    const int h0 = (L.M + 1) >> 1, h = colour == 0 ? h0 : L.M - h0;  // in row 2P
    int j = rem < h ? 2 * P : 2 * P + 1, p = rem < h ? rem : rem - h;
    int i = 2 * p + ((j + colour) & 1);
    on[colour] = t < (int)(L.MN + 1) / 2 && j < L.N && i < L.M;
    if (!on[colour]) i = j = 0;  // formed but never used
    o[colour] = nbrs(L, i, j);
    q[colour] = col_consts(G, L, i, j);
    load_rows<V, KM>(b, o[colour].c, L, rb[colour]);
  }
  __syncthreads();
  for (int sw = 0; sw < sweeps; ++sw) {
#pragma unroll
    for (int colour = 0; colour < 2; ++colour) {
      if (on[colour]) {
        V r[KM];
#pragma unroll
        for (int k = 0; k < KM; ++k) r[k] = rb[colour][k];
        if (sw == 0 && colour == 0) zero_rows<V, KM>(L, q[colour], r);
        else line_rows<V, KM>(L, q[colour], o[colour], r, xs);
        store_rows<V, KM>(L, r, xs, o[colour].c);
      }
      __syncthreads();
    }
  }
  for (int r = threadIdx.x; r < n; r += kCoarseBS) x[r] = xs[r];
}

template <class V, int KM>
__global__ __launch_bounds__(kCoarseBS) void k_coarse(LvlC<V> L, G2<V> G, const V *__restrict__ b,
                                                     V *__restrict__ x, int sweeps, const int *stop) {
  if (stop[0]) return;
  __shared__ V xs[KM * kMgCoarseCols];
  coarse_solve<V, KM>(L, G, b, x, sweeps, xs);
}

// bilinear (cell-centred) prolongation weights and coarse plane offsets
// (zebra layout) of fine column (i,j)
template <class V>
struct Pro {
  unsigned c00, c10, c01, c11;
  V wx0, wx1, wy0, wy1;
};
template <class V>
__device__ __forceinline__ Pro<V> pro_at(int Mc, int Nc, int fx, int fy, int i, int j) {
  Pro<V> w;
  int I0 = fx == 2 ? i >> 1 : i, I1 = I0;
  w.wx0 = V(1); w.wx1 = V(0);
  if (fx == 2) {
    I1 = (i & 1) ? I0 + 1 : I0 - 1;
    if (I1 < 0 || I1 >= Mc) I1 = I0;
    w.wx0 = V(0.75); w.wx1 = V(0.25);
  }
  int J0 = fy == 2 ? j >> 1 : j, J1 = J0;
  w.wy0 = V(1); w.wy1 = V(0);
  if (fy == 2) {
    J1 = (j & 1) ? J0 + 1 : J0 - 1;
    if (J1 < 0 || J1 >= Nc) J1 = J0;
    w.wy0 = V(0.75); w.wy1 = V(0.25);
  }
  w.c00 = (unsigned)zcol(I0, J0, Mc); w.c10 = (unsigned)zcol(I1, J0, Mc);
  w.c01 = (unsigned)zcol(I0, J1, Mc); w.c11 = (unsigned)zcol(I1, J1, Mc);
  return w;
}

// ---------------------------------------------------------------------------
// the two halves of a V-cycle on one level, a tile of columns per workgroup
// ---------------------------------------------------------------------------
// A zebra half sweep reads one colour and writes the other, so a V(1,1)
// cycle done sweep by sweep streams the level's vectors through HBM six
// times.  Here each workgroup takes a tile of TX x TY columns and recomputes
// the halo its half sweeps need, so nothing but the level's right side b, the
// coarse vectors and the final x moves:
//
//  k_mg_down: even columns from a zero guess (halo 2), odd columns against
//    them (halo 1), then the residual of the tile's even columns averaged
//    onto the coarse right side (the odd columns' residual is zero: they were
//    just solved exactly).
//  k_mg_up: the even columns' zero-guess solution formed again (cheaper than
//    a store and a load of half a vector) plus the interpolated coarse
//    correction (halo 2), odd columns against them (halo 1), even columns
//    again.  The odd columns of the pre-smoothing are never read after the
//    restriction (a half sweep solves for them from even values only), so
//    they are not kept, and the result needs no copy of x.
//
// Each colour's values pass between the half sweeps through LDS.
//
// Bound on large levels by waits that the three waves a SIMD left by 150 VGPRs
// do not cover (1024 x 1024 x 10: 3.6 and 2.9 TB/s up and down, the VALU 40 to
// 52 % busy), on small ones by the elimination's chain of dependent operations.
// Measured, FP64, a level's whole cycle: 1024 x 1024 x 10 162 us (sweep by sweep
// 195), 512 x 512 54 (68), 64 x 64 22 in two launches (34 in six); a V-cycle of
// the 1024 x 1024 x 10 hierarchy 304 us (385).
template <int TX, int TY>
struct MgTile {
  static_assert(TX % 2 == 0 && TY % 2 == 0, "tiles start on even columns and whole coarse cells");
  static constexpr int HW = TX / 2 + 2;       // slots of one colour in a row, halo 2
  static constexpr int SL = HW * (TY + 4);    // slots of one colour
  static constexpr int OW = HW - 1;           // odd columns of a row within halo 1
  static constexpr int ODD = OW * (TY + 2);
  static constexpr int EV = TX / 2 * TY;      // the tile's own columns of one colour
  static constexpr int NT = (SL + 63) / 64 * 64;  // threads: one even column each
  // LDS of both colours' values for K rows
  static constexpr size_t lds(int K, size_t esize) { return 2 * (size_t)SL * K * esize; }
};

// column of a tile slot: row r (0 .. TY+3 from y0-2), position p in the row
struct TCol {
  int i, j, r, p;
  bool in;  // inside the level
};
template <class V>
__device__ __forceinline__ TCol tile_col(const LvlC<V> &L, int x0, int y0, int r, int p, int colour) {
  TCol c;
  c.r = r;
  c.p = p;
  c.i = x0 - 2 + 2 * p + ((r + colour) & 1);
  c.j = y0 - 2 + r;
  c.in = c.i >= 0 && c.i < L.M && c.j >= 0 && c.j < L.N;
  return c;
}
// LDS slots of a slot's four neighbours, which are of the other colour
template <int HW>
__device__ __forceinline__ Nb tile_nbrs(int r, int p, int colour) {
  Nb o;
  const int s = r * HW + p, m = s - 1 + ((r + colour) & 1);
  o.c = s;
  o.xm = m;
  o.xp = m + 1;
  o.ym = s - HW;
  o.yp = s + HW;
  return o;
}

// The right side of a level's cycle.  On the fine level the iteration's
// vectors are formed where the cycle reads them: MG_S, s = r - alpha v; MG_P,
// p = r + beta (p - omega v).  MG_B: a vector.
enum { MG_B = 0, MG_S, MG_P };
template <class V, int KIND>
struct TileRhs {
  const V *__restrict__ b, *__restrict__ p, *__restrict__ v;
  V *out;
  V f, w;
  // a column's rows of the vectors, and what they make
  template <int KM>
  struct Raw {
    V b[KM], v[KIND == MG_B ? 1 : KM], p[KIND == MG_P ? KM : 1];
  };
  template <int KM>
  __device__ __forceinline__ void ask(unsigned zc, const LvlC<V> &L, Raw<KM> &q) const {
    load_rows<V, KM>(b, zc, L, q.b);
    if constexpr (KIND != MG_B) load_rows<V, KM>(v, zc, L, q.v);
    if constexpr (KIND == MG_P) load_rows<V, KM>(p, zc, L, q.p);
  }
  template <int KM>
  __device__ __forceinline__ void form(const Raw<KM> &q, V (&r)[KM]) const {
#pragma unroll
    for (int k = 0; k < KM; ++k) {
      r[k] = q.b[k];
      if constexpr (KIND == MG_S) r[k] = q.b[k] - f * q.v[k];
      if constexpr (KIND == MG_P) r[k] = q.b[k] + f * (q.p[k] - w * q.v[k]);
    }
  }
  template <int KM>
  __device__ __forceinline__ void load(unsigned zc, const LvlC<V> &L, V (&r)[KM]) const {
    Raw<KM> q;
    ask(zc, L, q);
    form(q, r);
  }
  // the vector formed, where the column is the tile's own
  template <int KM>
  __device__ __forceinline__ void keep(bool own, unsigned zc, const LvlC<V> &L, const V (&r)[KM]) const {
    if (KIND != MG_B && own) store_rows<V, KM>(L, r, out, zc);
  }
};
// host side of it: fin > 0, the scalar step before the launch is its own,
// from `fin` partials (kFuseParts)
template <class V>
struct MgRhs {
  const V *b, *p, *v;
  V *out;
  KScal sc;
  const double *part;
  int fin;
};
template <class V, int KIND>
__device__ __forceinline__ TileRhs<V, KIND> tile_vecs(const MgRhs<V> &in) {
  return TileRhs<V, KIND>{in.b, in.p, in.v, in.out, V(0), V(0)};
}
// the scalars; asked() asks for what else the launch waits for, between the
// partials and their sum.  false: the iteration has stopped.
template <class V, int KIND, class F>
__device__ __forceinline__ bool tile_scalars(const MgRhs<V> &in, TileRhs<V, KIND> &R, F asked) {
  const bool write = blockIdx.x == 0 && threadIdx.x == 0;
  if constexpr (KIND == MG_S) {
    double alpha = in.sc.sc[S_ALPHA];
    const WaveSum rhv(in.part, 0, in.fin);
    asked();
    if (in.fin && !fin1_logic(in.sc, rhv.sum(), alpha, write)) return false;
    R.f = (V)alpha;
  } else if constexpr (KIND == MG_P) {
    double beta = in.sc.sc[S_BETA];
    R.w = (V)in.sc.sc[S_OMEGA];
    const WaveSum rhr(in.part, 0, in.fin), rr(in.part, 1, in.fin);
    asked();
    if (in.fin && !fin3_logic(in.sc, rhr.sum(), rr.sum(), beta, write)) return false;
    R.f = (V)beta;
  } else {
    asked();
  }
  return true;
}

// right-side rows of a tile column, zeros outside the level
template <class V, int KM, int KIND>
__device__ __forceinline__ void tile_rows(const TileRhs<V, KIND> &b, const LvlC<V> &L, const TCol &c, V (&r)[KM]) {
#pragma unroll
  for (int k = 0; k < KM; ++k) r[k] = V(0);
  if (c.in) b.load((unsigned)zcol(c.i, c.j, L.M), L, r);
}
template <class V, int KM, int SL>
__device__ __forceinline__ void tile_put(const LvlC<V> &L, const V (&r)[KM], V *xs, int slot) {
#pragma unroll
  for (int k = 0; k < KM; ++k)
    if (k < L.K) xs[k * SL + slot] = r[k];
}

// zero-guess solve of an even column of the tile from its right side in r
template <class V, int KM>
__device__ __forceinline__ void tile_even_zero(const LvlC<V> &L, const G2<V> &G, const TCol &c, V (&r)[KM]) {
  if (c.in) zero_rows<V, KM>(L, col_consts_centre(G, L, c.i, c.j), r);
}

// odd columns of the tile against the even ones in xe, into xo; solved()
// sees the solution in r
template <class V, int KM, int TX, int TY, class F>
__device__ __forceinline__ void tile_odd(const LvlC<V> &L, const LvlC<V> &Ls, const G2<V> &G, const TCol &c,
                                         bool live, V (&r)[KM], const V *xe, V *xo, F &&solved) {
  using T = MgTile<TX, TY>;
  __syncthreads();
  if (live && c.in) {
    line_rows<V, KM>(Ls, col_consts(G, L, c.i, c.j), tile_nbrs<T::HW>(c.r, c.p, 1), r, xe);
    solved();
  }
  if (live) tile_put<V, KM, T::SL>(L, r, xo, c.r * T::HW + c.p);
  __syncthreads();
}

// residual b - A x of a tile column from its own values xc and its
// neighbours' xn, added to s
template <class V, int KM, int HW, int KIND>
__device__ __forceinline__ void tile_resid(const LvlC<V> &L, const LvlC<V> &Ls, const G2<V> &G,
                                           const TileRhs<V, KIND> &b, int i, int j, int x0, int y0, int colour,
                                           const V *xc, const V *xn, V (&s)[KM]) {
  const int r = j - y0 + 2, p = (i - x0 + 2 - ((r + colour) & 1)) >> 1;
  const Nb o = tile_nbrs<HW>(r, p, colour);
  V bv[KM];
  b.load((unsigned)zcol(i, j, L.M), L, bv);
  const int K1 = L.K - 1, SL = (int)Ls.MN;
  V below = xc[o.c], at = below, above = xc[min(1, K1) * SL + o.c];
  walk_col<V, KM>(Ls, col_consts(G, L, i, j), o, xn,
                  [&](int k, const ZRow<V> &z, const Pl<V> &, const Pl<V> &, const Pl<V> &) {
    s[k] += bv[k] - fma(z.c0, at, fma(z.c5, above, fma(z.c12, below, z.s)));
    below = at;
    at = above;
    above = xc[min(k + 2, K1) * SL + o.c];
  });
}

// scalars(b, asked) completes b (tile_scalars); false ends the launch
template <class V, int KM, int TX, int TY, int KIND, class F>
__device__ __forceinline__ void mg_down_body(const LvlC<V> &L, const G2<V> &G, TileRhs<V, KIND> b, int Mc, int Nc,
                                             int fx, int fy, V *__restrict__ bc, long tile, V *xs, F scalars) {
  using T = MgTile<TX, TY>;
  const int ntx = (L.M + TX - 1) / TX;
  const int ty = (int)(tile / ntx), x0 = (int)(tile - (long)ty * ntx) * TX, y0 = ty * TY;
  const int t = threadIdx.x;
  LvlC<V> Ls = L;
  Ls.MN = T::SL;
  V *xe = xs, *xo = xs + (long)T::SL * L.K;
  // the odd column's right side is requested before the even columns' work
  const bool olive = t < T::ODD;
  const int orow = olive ? 1 + t / T::OW : 1;
  const TCol oc = tile_col(L, x0, y0, orow, (olive ? t % T::OW : 0) + (orow & 1), 1);
  V ro[KM];
  {
    V re[KM];
    const TCol ec = tile_col(L, x0, y0, t / T::HW, t % T::HW, 0);
    auto own = [&](const TCol &q) {
      return q.in && q.i >= x0 && q.i < x0 + TX && q.j >= y0 && q.j < y0 + TY;
    };
    const unsigned ez = (unsigned)zcol(ec.i, ec.j, L.M);
    typename TileRhs<V, KIND>::template Raw<KM> raw;
    if (!scalars(b, [&] {
          if (ec.in) b.ask(ez, L, raw);
        }))
      return;
#pragma unroll
    for (int k = 0; k < KM; ++k) re[k] = V(0);
    if (ec.in) b.form(raw, re);
    b.keep(t < T::SL && own(ec), ez, L, re);
    tile_even_zero<V, KM>(L, G, ec, re);
    tile_rows<V, KM>(b, L, oc, ro);
    b.keep(olive && own(oc), (unsigned)zcol(oc.i, oc.j, L.M), L, ro);
    if (t < T::SL) tile_put<V, KM, T::SL>(L, re, xe, t);
  }
  tile_odd<V, KM, TX, TY>(L, Ls, G, oc, olive, ro, xe, xo, [] {});
  // 2x2 coarse cells: their two even columns on neighbouring lanes, whose
  // residuals meet through a shuffle.  Cells of a level coarsened along one
  // axis: both columns on one lane.
  const bool two = fx == 2 && fy == 2;
  const int c = two ? t >> 1 : t, e = two ? t & 1 : 0;
  const int cw = TX / fx, cx = c % cw, cy = c / cw;
  const int I = x0 / fx + cx, J = y0 / fy + cy, i0 = I * fx, j0 = J * fy;
  const bool cell = t < T::EV && i0 < L.M && j0 < L.N;
  V s[KM];
#pragma unroll
  for (int k = 0; k < KM; ++k) s[k] = V(0);
  for (int a = 0; a < (two ? 1 : 2); ++a) {
    const int i = two ? i0 + e : fx == 2 ? i0 + a : i0, j = two ? j0 + e : fy == 2 ? j0 + a : j0;
    const int odd = (i + j) & 1;
    if (cell && i < L.M && j < L.N)
      tile_resid<V, KM, T::HW>(L, Ls, G, b, i, j, x0, y0, odd, odd ? xo : xe, odd ? xe : xo, s);
  }
  const int cnt = (min(i0 + fx, L.M) - i0) * (min(j0 + fy, L.N) - j0);  // fine cells of the block
  const V w = V(1) / (V)cnt;
  if (two)
#pragma unroll
    for (int k = 0; k < KM; ++k) s[k] += __shfl_xor(s[k], 1, 64);
  if (!cell || e != 0) return;
  const long MNc = (long)Mc * Nc;
  const unsigned zc = (unsigned)zcol(I, J, Mc);
#pragma unroll
  for (int k = 0; k < KM; ++k)
    if (k < L.K) sto(bc + (long)k * MNc, zc, s[k] * w);
}

template <class V, int KM, int TX, int TY>
__device__ __forceinline__ void mg_up_body(const LvlC<V> &L, const G2<V> &G, const V *__restrict__ b, int Mc, int Nc,
                                           int fx, int fy, const V *__restrict__ xc, V *__restrict__ x, long tile,
                                           V *xs) {
  using T = MgTile<TX, TY>;
  const int ntx = (L.M + TX - 1) / TX;
  const int ty = (int)(tile / ntx), x0 = (int)(tile - (long)ty * ntx) * TX, y0 = ty * TY;
  const int t = threadIdx.x;
  LvlC<V> Ls = L;
  Ls.MN = T::SL;
  V *xe = xs, *xo = xs + (long)T::SL * L.K;
  const bool olive = t < T::ODD;
  const int orow = olive ? 1 + t / T::OW : 1;
  const TCol oc = tile_col(L, x0, y0, orow, (olive ? t % T::OW : 0) + (orow & 1), 1);
  V ro[KM];
  {
    V re[KM];
    const TCol ec = tile_col(L, x0, y0, t / T::HW, t % T::HW, 0);
    const TileRhs<V, MG_B> rhs{b};
    tile_rows<V, KM>(rhs, L, ec, re);
    tile_even_zero<V, KM>(L, G, ec, re);
    if (ec.in) {
      const Pro<V> w = pro_at<V>(Mc, Nc, fx, fy, ec.i, ec.j);
      const long MNc = (long)Mc * Nc;
      const int K1 = L.K - 1;
#pragma unroll
      for (int k = 0; k < KM; ++k) {
        const V *xk = xc + MNc * min(k, K1);
        re[k] += w.wy0 * (w.wx0 * ldo(xk, w.c00) + w.wx1 * ldo(xk, w.c10)) +
                 w.wy1 * (w.wx0 * ldo(xk, w.c01) + w.wx1 * ldo(xk, w.c11));
      }
    }
    tile_rows<V, KM>(rhs, L, oc, ro);
    if (t < T::SL) tile_put<V, KM, T::SL>(L, re, xe, t);
  }
  // the tile's own columns of either colour are stored; the halo's are
  // their own tile's to store
  tile_odd<V, KM, TX, TY>(L, Ls, G, oc, olive, ro, xe, xo, [&] {
    if (oc.i >= x0 && oc.i < x0 + TX && oc.j >= y0 && oc.j < y0 + TY)
      store_rows<V, KM>(L, ro, x, (unsigned)zcol(oc.i, oc.j, L.M));
  });
  if (t >= T::EV) return;
  const TCol c = tile_col(L, x0, y0, 2 + t / (TX / 2), 1 + t % (TX / 2), 0);
  if (!c.in) return;
  const unsigned zc = (unsigned)zcol(c.i, c.j, L.M);
  V r[KM];
  load_rows<V, KM>(b, zc, L, r);
  line_rows<V, KM>(Ls, col_consts(G, L, c.i, c.j), tile_nbrs<T::HW>(c.r, c.p, 0), r, (const V *)xo);
  store_rows<V, KM>(L, r, x, zc);
}

// the workgroup's dynamic LDS
template <class V>
__device__ __forceinline__ V *tile_lds() {
  extern __shared__ __align__(16) unsigned char mg_tile_lds[];
  return (V *)mg_tile_lds;
}

template <class V, int KM, int TX, int TY, int KIND>
__global__ __launch_bounds__((MgTile<TX, TY>::NT)) void k_mg_down(LvlC<V> L, G2<V> G, MgRhs<V> in, int Mc, int Nc,
                                                                int fx, int fy, V *__restrict__ bc,
                                                                const int *stop) {
  if (stop[0]) return;
  V *xs = tile_lds<V>();
  mg_down_body<V, KM, TX, TY>(L, G, tile_vecs<V, KIND>(in), Mc, Nc, fx, fy, bc, (long)xcd_block(), xs,
                              [&](TileRhs<V, KIND> &b, auto asked) { return tile_scalars<V, KIND>(in, b, asked); });
}

template <class V, int KM, int TX, int TY>
__global__ __launch_bounds__((MgTile<TX, TY>::NT)) void k_mg_up(LvlC<V> L, G2<V> G, const V *__restrict__ b, int Mc,
                                                              int Nc, int fx, int fy, const V *__restrict__ xc,
                                                              V *__restrict__ x, const int *stop) {
  if (stop[0]) return;
  V *xs = tile_lds<V>();
  mg_up_body<V, KM, TX, TY>(L, G, b, Mc, Nc, fx, fy, xc, x, (long)xcd_block(), xs);
}

// ---------------------------------------------------------------------------
// the rest of a cycle in one workgroup
// ---------------------------------------------------------------------------
template <class V>
struct TailLevel {
  LvlC<V> L;
  G2<V> G;
  V *b, *x;    // of the first level: the caller's
  int fx, fy;  // to the next level
};
template <class V>
struct Tail {
  int n;  // levels, the last of them the hierarchy's coarsest
  TailLevel<V> l[kTailLevels];
};

// thread t's column of a colour (the t-th, as in coarse_solve)
template <class V>
__device__ __forceinline__ bool colour_col(const LvlC<V> &L, int t, int colour, int &i, int &j) {
  const int P = t / L.M, rem = t - P * L.M;
  const int h0 = (L.M + 1) >> 1, h = colour == 0 ? h0 : L.M - h0;
  j = rem < h ? 2 * P : 2 * P + 1;
  i = 2 * (rem < h ? rem : rem - h) + ((j + colour) & 1);
  return t < (int)(L.MN + 1) / 2 && j < L.N && i < L.M;
}

// The V(1,1) cycle of k_mg_down and k_mg_up, every half sweep over the whole
// level with a barrier after it: the same operations on the same values, so
// the same result.  x in LDS; b and the coarse solutions go through memory
// (one CU's: the barrier is enough).
template <class V, int KM, int KIND>
__global__ __launch_bounds__(kCoarseBS) void k_mg_tail(Tail<V> A, MgRhs<V> in, int sweeps, const int *stop) {
  if (stop[0]) return;
  __shared__ V xs[KM * kTailCols];
  const int t = threadIdx.x, K = A.l[0].L.K;
  if constexpr (KIND != MG_B) {  // the first level's right side
    TileRhs<V, KIND> R = tile_vecs<V, KIND>(in);
    if (!tile_scalars<V, KIND>(in, R, [] {})) return;
    const int n = (int)A.l[0].L.MN * K;
    for (int q = t; q < n; q += kCoarseBS) {
      V r = R.b[q];
      if constexpr (KIND == MG_S) r = r - R.f * R.v[q];
      if constexpr (KIND == MG_P) r = r + R.f * (R.p[q] - R.w * R.v[q]);
      R.out[q] = r;
    }
  }
  // a neighbour past the edge is the column itself with a zero coefficient:
  // what it reads has to be finite
  for (int q = t; q < KM * kTailCols; q += kCoarseBS) xs[q] = V(0);
  __syncthreads();
  // even columns from a zero guess, corrected by the coarse solution on the
  // way up; odd columns against them
  auto even_odd = [&](const TailLevel<V> &l, const TailLevel<V> *q) {
    int i, j;
    V r[KM];
    if (colour_col(l.L, t, 0, i, j)) {
      const unsigned zc = (unsigned)zcol(i, j, l.L.M);
      load_rows<V, KM>((const V *)l.b, zc, l.L, r);
      zero_rows<V, KM>(l.L, col_consts_centre(l.G, l.L, i, j), r);
      if (q) {
        const Pro<V> w = pro_at<V>(q->L.M, q->L.N, l.fx, l.fy, i, j);
#pragma unroll
        for (int k = 0; k < KM; ++k) {
          const V *xk = q->x + q->L.MN * min(k, K - 1);
          r[k] += w.wy0 * (w.wx0 * ldo(xk, w.c00) + w.wx1 * ldo(xk, w.c10)) +
                  w.wy1 * (w.wx0 * ldo(xk, w.c01) + w.wx1 * ldo(xk, w.c11));
        }
      }
      store_rows<V, KM>(l.L, r, xs, zc);
    }
    __syncthreads();
    if (colour_col(l.L, t, 1, i, j)) {
      const Nb o = nbrs(l.L, i, j);
      load_rows<V, KM>((const V *)l.b, o.c, l.L, r);
      line_rows<V, KM>(l.L, col_consts(l.G, l.L, i, j), o, r, xs);
      store_rows<V, KM>(l.L, r, xs, o.c);
      if (q) store_rows<V, KM>(l.L, r, l.x, o.c);
    }
    __syncthreads();
  };
  const int last = A.n - 1;
  for (int a = 0; a < last; ++a) {
    const TailLevel<V> &l = A.l[a], &q = A.l[a + 1];
    even_odd(l, nullptr);
    // the residual onto the coarse right side, as in mg_down_body.  Levels so
    // narrow halve along one axis: both columns of a cell on one lane.
    const int I = t % q.L.M, J = t / q.L.M, i0 = I * l.fx, j0 = J * l.fy;
    if (J < q.L.N) {
      V s[KM];
#pragma unroll
      for (int k = 0; k < KM; ++k) s[k] = V(0);
      for (int h = 0; h < 2; ++h) {
        const int i = l.fx == 2 ? i0 + h : i0, j = l.fx == 2 ? j0 : j0 + h;
        if (i >= l.L.M || j >= l.L.N) continue;
        const Nb o = nbrs(l.L, i, j);
        V bv[KM];
        load_rows<V, KM>((const V *)l.b, o.c, l.L, bv);
        const int MN = (int)l.L.MN;
        V below = xs[o.c], at = below, above = xs[min(1, K - 1) * MN + o.c];
        walk_col<V, KM>(l.L, col_consts(l.G, l.L, i, j), o, (const V *)xs,
                        [&](int k, const ZRow<V> &z, const Pl<V> &, const Pl<V> &, const Pl<V> &) {
          s[k] += bv[k] - fma(z.c0, at, fma(z.c5, above, fma(z.c12, below, z.s)));
          below = at;
          at = above;
          above = xs[min(k + 2, K - 1) * MN + o.c];
        });
      }
      const int cnt = (min(i0 + l.fx, l.L.M) - i0) * (min(j0 + l.fy, l.L.N) - j0);
      const V w = V(1) / (V)cnt;
#pragma unroll
      for (int k = 0; k < KM; ++k) s[k] = s[k] * w;
      store_rows<V, KM>(q.L, s, q.b, (unsigned)zcol(I, J, q.L.M));
    }
    __syncthreads();
  }
  coarse_solve<V, KM>(A.l[last].L, A.l[last].G, (const V *)A.l[last].b, A.l[last].x, sweeps, xs);
  __syncthreads();
  for (int a = last - 1; a >= 0; --a) {
    const TailLevel<V> &l = A.l[a];
    even_odd(l, &A.l[a + 1]);
    int i, j;
    if (colour_col(l.L, t, 0, i, j)) {
      const Nb o = nbrs(l.L, i, j);
      V r[KM];
      load_rows<V, KM>((const V *)l.b, o.c, l.L, r);
      line_rows<V, KM>(l.L, col_consts(l.G, l.L, i, j), o, r, (const V *)xs);
      store_rows<V, KM>(l.L, r, l.x, o.c);
    }
    __syncthreads();
  }
}

}  // namespace nhw

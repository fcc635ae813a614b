// Matrix-free sigma-coordinate Poisson operator and a geometric multigrid
// preconditioner for it, templated on the vector type V (double for the FP64
// solve, float for the inner solve of the mixed form).
//
// The operator is the one generate_coef_rhs assembles (src/pressure.F:475-840):
// per row, 15 coefficients built from A1 = DelxS^2 + DelyS^2 + DelzS^2 and the
// face slopes DelxS/DelyS, with Neumann folds on the lateral and bottom
// boundaries and the Dirichlet surface.  Instead of streaming 15 stored
// diagonals (120 B/row) it recomputes them from five 2-D fields per column
// (ax = DelxH/D, bx = (DelxH+DelxEta)/D, ay, by, rD = 1/D, so that
// DelxS = ax - sig_k*bx) and per-level constants: the operator pass then moves
// about three vectors per row.  The coefficients agree with the assembled ones
// to rounding (products by precomputed reciprocals instead of quotients).
//
// Multigrid: cell-centred x-y coarsening by 2 (K kept), coarse operators by
// rediscretisation on block-averaged column fields, zebra z-line Gauss-Seidel
// smoothing (columns coloured by (i+j) parity; each column's vertical
// tridiagonal -- c13, c1, c6 -- solved exactly, which absorbs the strong
// vertical coupling of shallow and dry columns), block-average restriction
// and bilinear prolongation.  One V(1,1)-cycle from a zero guess is a fixed
// linear operator, used as the right preconditioner of BiCGStab.  The
// 15-point stencil has no (+-1,+-1) x-y couplings, so columns of one colour
// are independent and update in parallel.
#include <algorithm>
#include <vector>

#include "nhw_mg_dev.h"

namespace nhw {

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static inline unsigned nb(long n) { return (unsigned)((n + kBSm - 1) / kBSm); }

template <class V>
static LvlC<V> make_lvl(const nhw_ctx *c, const MGLevel &lv) {
  LvlC<V> L{};
  const double dx = lv.dx, dy = lv.dy;
  L.M = lv.M; L.N = lv.N; L.K = c->g.K; L.MN = (long)lv.M * lv.N;
  L.cxy = (V)(2. / (dx * dx) + 2. / (dy * dy));
  L.idx2 = (V)(1. / (dx * dx));
  L.idy2 = (V)(1. / (dy * dy));
  L.kc = (const LvlK<V> *)lv.kc;
  return L;
}

// the sigma-level constants of one level (the rows' coefficients,
// src/pressure.F:540-555), kMgKMax entries (unused ones zero)
template <class V>
static std::vector<LvlK<V>> level_table(const nhw_ctx *c, const MGLevel &lv) {
  std::vector<LvlK<V>> t(kMgKMax, LvlK<V>{V(0), V(0), V(0), V(0), V(0)});
  const std::vector<double> &dsig = c->mg.dsig_h, &sig = c->mg.sig_h;  // 1-based
  for (int kk = 0; kk < c->g.K; ++kk) {
    const int k = c->g.Kbeg + kk;
    const double s = dsig[k] + dsig[k - 1];
    t[kk].sig = (V)sig[k];
    t[kk].r6 = (V)(1. / (0.5 * s * dsig[k]));
    t[kk].r13 = (V)(1. / (0.5 * s * dsig[k - 1]));
    t[kk].rx = (V)(1. / (2. * lv.dx * s));
    t[kk].ry = (V)(1. / (2. * lv.dy * s));
  }
  return t;
}

// uploads every level's table (after the vertical grid is set)
int mg_upload_consts(nhw_ctx *c) {
  for (int h = 0; h < 2; ++h) {
    std::vector<MGLevel> &lvs = h == 0 ? c->mg.lv : c->mg.lvf;
    const bool f32 = h == 1;
    for (const MGLevel &lv : lvs) {
      if (!lv.kc) continue;
      hipError_t e;
      if (f32) {
        const std::vector<LvlK<float>> t = level_table<float>(c, lv);
        e = hipMemcpy(lv.kc, t.data(), sizeof(LvlK<float>) * t.size(), hipMemcpyHostToDevice);
      } else {
        const std::vector<LvlK<double>> t = level_table<double>(c, lv);
        e = hipMemcpy(lv.kc, t.data(), sizeof(LvlK<double>) * t.size(), hipMemcpyHostToDevice);
      }
      if (hip_check(e, "multigrid level constants")) return NHW_EHIP;
    }
  }
  return 0;
}

template <class V>
LvlC<V> mg_level_consts(const nhw_ctx *c, const MGLevel &lv) {
  return make_lvl<V>(c, lv);
}
template LvlC<double> mg_level_consts<double>(const nhw_ctx *, const MGLevel &);
template LvlC<float> mg_level_consts<float>(const nhw_ctx *, const MGLevel &);

template <class V>
static G2<V> g2(const MGLevel &lv) {
  return G2<V>{(const V *)lv.ax, (const V *)lv.bx, (const V *)lv.ay, (const V *)lv.by, (const V *)lv.rd, lv.M + 2};
}

// Levels of one hierarchy; elements are `esize` bytes (8: FP64, 4: FP32).
// maxlev = 1 keeps only the fine-level geometry (the FP64 operator of the
// mixed form's outer residual).
int mg_alloc(nhw_ctx *c, std::vector<MGLevel> &lvs, int esize, int maxlev) {
  const Geo &g = c->g;
  if (g.K > kMgKMax) {
    set_error("mg_alloc: Kglob above the multigrid limit");
    return NHW_EINVAL;
  }
  int M = g.M, N = g.N;
  double dx = g.dx, dy = g.dy;
  while (true) {
    MGLevel lv;
    lv.M = M; lv.N = N; lv.dx = dx; lv.dy = dy;
    const long n = (long)M * N * g.K, n2h = (long)(M + 2) * (N + 2);
    const bool fine = lvs.empty();
    bool ok = true;
    for (double **p : {&lv.ax, &lv.bx, &lv.ay, &lv.by, &lv.rd})
      ok = ok && hipMalloc(p, esize * n2h) == hipSuccess && hipMemset(*p, 0, esize * n2h) == hipSuccess;
    const size_t kcb = (size_t)5 * esize * kMgKMax;
    ok = ok && hipMalloc(&lv.kc, kcb) == hipSuccess && hipMemset(lv.kc, 0, kcb) == hipSuccess;
    if (maxlev > 1 && !fine)  // level 0 solves into the caller's vectors
      for (double **p : {&lv.x, &lv.b})
        ok = ok && hipMalloc(p, esize * n) == hipSuccess && hipMemset(*p, 0, esize * n) == hipSuccess;
    lvs.push_back(lv);
    if (!ok) {
      set_error("mg_alloc: hipMalloc failed");
      return NHW_ENOMEM;
    }
    if ((int)lvs.size() >= maxlev || !mg_coarsens(M, N)) break;
    const int fx = M >= 4 ? 2 : 1, fy = N >= 4 ? 2 : 1;
    lvs.back().fx = fx;
    lvs.back().fy = fy;
    M = (M + fx - 1) / fx;
    N = (N + fy - 1) / fy;
    dx *= fx;
    dy *= fy;
  }
  return 0;
}

void mg_free(std::vector<MGLevel> &lvs) {
  for (MGLevel &lv : lvs) {
    for (double *p : {lv.ax, lv.bx, lv.ay, lv.by, lv.rd, lv.x, lv.b, lv.r})
      if (p) (void)hipFree(p);
    if (lv.kc) (void)hipFree(lv.kc);
  }
  lvs.clear();
}

// column fields of every level from the current D, DelxH/Eta, DelyH/Eta
template <class V>
int mg_setup(nhw_ctx *c, std::vector<MGLevel> &lvs) {
  const Geo &g = c->g;
  hipStream_t st = c->stream;
  if (c->mg.dsig_h.size() != (size_t)g.Kloc + 1) {
    set_error("poisson_solver: vertical grid not set (nhw_set_grid)");
    return NHW_EINVAL;
  }
  MGLevel &l0 = lvs[0];
  {
    Timed t(c, KID_MG_SETUP, 8.0 * 5 * g.M * g.N + sizeof(V) * 5.0 * g.M * g.N);
    hipLaunchKernelGGL(k_geom0<V>, dim3(nb((long)g.M * g.N)), dim3(kBSm), 0, st, g, c->d, (V *)l0.ax, (V *)l0.bx,
                       (V *)l0.ay, (V *)l0.by, (V *)l0.rd, l0.M + 2);
  }
  for (size_t l = 0; l + 1 < lvs.size(); ++l) {
    const MGLevel &f = lvs[l];
    MGLevel &q = lvs[l + 1];
    Timed t(c, KID_MG_SETUP, sizeof(V) * 5.0 * ((double)f.M * f.N + (double)q.M * q.N));
    hipLaunchKernelGGL(k_geom_coarsen<V>, dim3(nb((long)q.M * q.N)), dim3(kBSm), 0, st, f.M, f.N, f.M + 2, q.M,
                       q.N, q.M + 2, f.fx, f.fy, (const V *)f.ax, (const V *)f.bx, (const V *)f.ay,
                       (const V *)f.by, (const V *)f.rd, (V *)q.ax, (V *)q.bx, (V *)q.ay, (V *)q.by, (V *)q.rd);
  }
  return hip_check(hipGetLastError(), "mg_setup");
}
template int mg_setup<double>(nhw_ctx *, std::vector<MGLevel> &);
template int mg_setup<float>(nhw_ctx *, std::vector<MGLevel> &);

// the coarsest level: coarse_sweeps zebra pairs in one single-workgroup
// launch; algorithmic bytes: b read and x written per half sweep pair
template <class V>
static void coarse(nhw_ctx *c, const LvlC<V> &L, const G2<V> &G, const V *b, V *x, const int *stop) {
  const int sw = c->mg.coarse_sweeps;
  Timed t(c, KID_MG_COARSE, sizeof(V) * (2.0 * L.MN * L.K + 5.0 * L.MN));
  by_rows<kMgKMax>(L.K, [&](auto km) {
    hipLaunchKernelGGL((k_coarse<V, decltype(km)::value>), dim3(1), dim3(kCoarseBS), 0, c->stream, L, G, b, x, sw,
                       stop);
  });
}

// algorithmic bytes of the two halves of a level's cycle: b, the five column
// fields and the coarse right side; b, the fields, the coarse solution and x
template <class V, int KM, int TX, int TY, int KIND>
static void down_t(nhw_ctx *c, const LvlC<V> &L, const MGLevel &lv, const MGLevel &q, const MgRhs<V> &b,
                   const int *stop) {
  using T = MgTile<TX, TY>;
  constexpr double rows = KIND == MG_B ? 1.0 : KIND == MG_S ? 3.0 : 4.0;
  Timed t(c, KID_MG_DOWN, sizeof(V) * (rows * L.MN * L.K + (double)q.M * q.N * L.K + 5.0 * L.MN));
  hipLaunchKernelGGL((k_mg_down<V, KM, TX, TY, KIND>), dim3(mg_tiles<TX, TY>(lv)), dim3(T::NT), T::lds(L.K, sizeof(V)), c->stream, L, g2<V>(lv),
                     b, q.M, q.N, lv.fx, lv.fy, (V *)q.b, stop);
}
template <class V, int KM, int TX, int TY>
static void up_t(nhw_ctx *c, const LvlC<V> &L, const MGLevel &lv, const MGLevel &q, const V *b, V *x,
                 const int *stop) {
  using T = MgTile<TX, TY>;
  Timed t(c, KID_MG_UP, sizeof(V) * (2.0 * L.MN * L.K + (double)q.M * q.N * L.K + 5.0 * L.MN));
  hipLaunchKernelGGL((k_mg_up<V, KM, TX, TY>), dim3(mg_tiles<TX, TY>(lv)), dim3(T::NT), T::lds(L.K, sizeof(V)), c->stream, L, g2<V>(lv), b,
                     q.M, q.N, lv.fx, lv.fy, (const V *)q.x, x, stop);
}
// level l and all below it
template <class V, int KIND>
static void tail(nhw_ctx *c, const std::vector<MGLevel> &lvs, size_t l, const MgRhs<V> &in, const V *b, V *x,
                 const int *stop) {
  Tail<V> A{};
  A.n = (int)(lvs.size() - l);
  double bytes = 0.0;
  for (int a = 0; a < A.n; ++a) {
    const MGLevel &lv = lvs[l + a];
    A.l[a] = TailLevel<V>{make_lvl<V>(c, lv), g2<V>(lv), a ? (V *)lv.b : (V *)b, a ? (V *)lv.x : x, lv.fx, lv.fy};
    bytes += sizeof(V) * (3.0 * A.l[a].L.MN * A.l[a].L.K + 10.0 * A.l[a].L.MN);
  }
  Timed t(c, KID_MG_TAIL, bytes);
  by_rows<kMgKMax>(A.l[0].L.K, [&](auto km) {
    hipLaunchKernelGGL((k_mg_tail<V, decltype(km)::value, KIND>), dim3(1), dim3(kCoarseBS), 0, c->stream, A, in,
                       c->mg.coarse_sweeps, stop);
  });
}

// x = V(b): one V(1,1) cycle from a zero guess on level l; the coarsest
// level (at most kMgCoarseCols columns) gets coarse_sweeps zebra sweeps
template <class V, int KIND>
static void vcycle(nhw_ctx *c, const std::vector<MGLevel> &lvs, size_t l, const MgRhs<V> &in, V *x, const int *stop) {
  const MGLevel &lv = lvs[l];
  const LvlC<V> L = make_lvl<V>(c, lv);
  const V *b = KIND == MG_B ? in.b : in.out;
  if (l + 1 == lvs.size()) {
    coarse(c, L, g2<V>(lv), b, x, stop);
    return;
  }
  if (mg_tail((long)lv.M * lv.N, lvs.size() - l)) {
    tail<V, KIND>(c, lvs, l, in, b, x, stop);
    return;
  }
  const MGLevel &q = lvs[l + 1];
  const bool big = mg_big_tiles((long)lv.M * lv.N);
  by_rows<kMgKMax>(L.K, [&](auto km) {
    constexpr int KM = decltype(km)::value;
    // where the cycle forms the vectors, only columns of few rows make up a
    // large level (mg_forms_vectors)
    if constexpr (KIND == MG_B || KM * kMgBigCols <= (long)kFuseParts * kBS)
      if (big) return down_t<V, KM, kTileX, kTileY, KIND>(c, L, lv, q, in, stop);
    down_t<V, KM, kTileSX, kTileSY, KIND>(c, L, lv, q, in, stop);
  });
  vcycle<V, MG_B>(c, lvs, l + 1, MgRhs<V>{(const V *)q.b}, (V *)q.x, stop);
  by_rows<kMgKMax>(L.K, [&](auto km) {
    constexpr int KM = decltype(km)::value;
    if (big) up_t<V, KM, kTileX, kTileY>(c, L, lv, q, b, x, stop);
    else up_t<V, KM, kTileSX, kTileSY>(c, L, lv, q, b, x, stop);
  });
}

template <class V>
void mg_apply(nhw_ctx *c, const std::vector<MGLevel> &lvs, int kind, const MgRhs<V> &b, V *x, const int *stop) {
  if (kind == MG_B) vcycle<V, MG_B>(c, lvs, 0, b, x, stop);
  else if (kind == MG_S) vcycle<V, MG_S>(c, lvs, 0, b, x, stop);
  else vcycle<V, MG_P>(c, lvs, 0, b, x, stop);
}
template void mg_apply<double>(nhw_ctx *, const std::vector<MGLevel> &, int, const MgRhs<double> &, double *,
                               const int *);
template void mg_apply<float>(nhw_ctx *, const std::vector<MGLevel> &, int, const MgRhs<float> &, float *,
                              const int *);

// y = A x on the fine level, with ndot dot partials (y,d1) [and (y,y)]
template <class V>
void mf_apply(nhw_ctx *c, const std::vector<MGLevel> &lvs, const V *x, V *y, const V *d1, int ndot, double *part,
              const int *stop, int nblk, int kid) {
  const MGLevel &l0 = lvs[0];
  const LvlC<V> L = make_lvl<V>(c, l0);
  const G2<V> G = g2<V>(l0);
  const double n = (double)L.MN * L.K;
  Timed t(c, kid, sizeof(V) * 3.0 * n + sizeof(V) * 5.0 * L.MN);
  if (ndot == 0)
    hipLaunchKernelGGL((k_mf_apply<V, 0>), dim3(nblk), dim3(kBSm), 0, c->stream, L, G, x, y, d1, part, stop);
  else if (ndot == 1)
    hipLaunchKernelGGL((k_mf_apply<V, 1>), dim3(nblk), dim3(kBSm), 0, c->stream, L, G, x, y, d1, part, stop);
  else
    hipLaunchKernelGGL((k_mf_apply<V, 2>), dim3(nblk), dim3(kBSm), 0, c->stream, L, G, x, y, d1, part, stop);
}

template void mf_apply<double>(nhw_ctx *, const std::vector<MGLevel> &, const double *, double *, const double *,
                               int, double *, const int *, int, int);
template void mf_apply<float>(nhw_ctx *, const std::vector<MGLevel> &, const float *, float *, const float *, int,
                              double *, const int *, int, int);

// FP64 residual of x against b into the Krylov vectors of type R (see
// k_mf_init); geometry from the FP64 level 0 of `lvs`
template <class R>
void mf_init(nhw_ctx *c, const std::vector<MGLevel> &lvs, const double *x, const double *b, R *rh, double *part,
             int nblk) {
  const MGLevel &l0 = lvs[0];
  const LvlC<double> L = make_lvl<double>(c, l0);
  const double n = (double)L.MN * L.K;
  Timed t(c, KID_MF_RESID, (16.0 + sizeof(R)) * n + 40.0 * L.MN);
  hipLaunchKernelGGL(k_mf_init<R>, dim3(nblk), dim3(kBSm), 0, c->stream, L, g2<double>(l0), x, b, rh, part);
}
template void mf_init<double>(nhw_ctx *, const std::vector<MGLevel> &, const double *, const double *, double *,
                              double *, int);
template void mf_init<float>(nhw_ctx *, const std::vector<MGLevel> &, const double *, const double *, float *,
                             double *, int);

void mf_true_resid(nhw_ctx *c, const std::vector<MGLevel> &lvs, const double *x, const double *b, double *part,
                   int nblk) {
  const MGLevel &l0 = lvs[0];
  const LvlC<double> L = make_lvl<double>(c, l0);
  Timed t(c, KID_MF_RESID, 16.0 * L.MN * L.K + 40.0 * L.MN);
  hipLaunchKernelGGL(k_mf_true, dim3(nblk), dim3(kBSm), 0, c->stream, L, g2<double>(l0), x, b, part);
}

}  // namespace nhw

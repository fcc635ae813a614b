// Device side of the BiCGStab iteration shared by the single-scenario and
// batched Poisson solves: scalar slots, deterministic reductions and the
// per-iteration scalar logic (what the single-thread "fin" steps decide).
#pragma once
#include "nhw_impl.h"

namespace nhw {

constexpr double kInnerTol = 1e-4;  // relative residual reduction of one FP32 inner solve
constexpr int kMaxRefine = 20;      // refinement rounds of the mixed form

enum { S_RHO = 0, S_ALPHA, S_OMEGA, S_BETA, S_BB, S_RR, S_RHV, S_TS, S_TT, S_TRUE, S_REF, S_ITOL, S_RHOP, S_N };

// scalars and flags of one solve.  flag[0]: 0 running, 1 converged,
// 2 breakdown, 3 ITMAX reached, 4 zero right-hand side; flag[1]: iterations;
// flag[2]: breakdown code.  `inner` marks the mixed form's FP32 inner solve,
// which stops on |r| <= itol*|r0| instead of |r| <= tol*|b|.
struct KScal {
  double *sc;
  int *flag;
  int itmax;
  double tol2, itol2;
  int inner;
};

// deterministic block reduction of up to 3 values into part[3*blockIdx+m]
template <int NV>
__device__ __forceinline__ void block_reduce(double (&v)[NV], double *part) {
  __shared__ double sm[NV][kBS];
#pragma unroll
  for (int m = 0; m < NV; ++m) sm[m][threadIdx.x] = v[m];
  __syncthreads();
  for (int s = kBS / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s)
#pragma unroll
      for (int m = 0; m < NV; ++m) sm[m][threadIdx.x] += sm[m][threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0)
#pragma unroll
    for (int m = 0; m < NV; ++m) part[3 * blockIdx.x + m] = sm[m][0];
}

// sums of the first NV partials of blocks b0 .. b1-1 (fixed order:
// deterministic).  One workgroup: eight partials a thread are under way at
// once, and the sums share the barriers (8192 blocks, two sums: 17.6 us one
// after the other, now 7.6).
template <int NV>
__device__ __forceinline__ void final_sums(const double *part, long b0, long b1, double (&out)[NV]) {
  constexpr int U = 8;
  __shared__ double sm[NV][kBS];
  double a[NV];
#pragma unroll
  for (int m = 0; m < NV; ++m) a[m] = 0.0;
  for (long b = b0 + threadIdx.x; b < b1; b += U * kBS) {
    double v[U][NV];
#pragma unroll
    for (int q = 0; q < U; ++q)
#pragma unroll
      for (int m = 0; m < NV; ++m) v[q][m] = b + q * kBS < b1 ? part[3 * (b + q * kBS) + m] : 0.0;
#pragma unroll
    for (int q = 0; q < U; ++q)
#pragma unroll
      for (int m = 0; m < NV; ++m) a[m] += v[q][m];
  }
#pragma unroll
  for (int m = 0; m < NV; ++m) sm[m][threadIdx.x] = a[m];
  __syncthreads();
  for (int s = kBS / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s)
#pragma unroll
      for (int m = 0; m < NV; ++m) sm[m][threadIdx.x] += sm[m][threadIdx.x + s];
    __syncthreads();
  }
#pragma unroll
  for (int m = 0; m < NV; ++m) out[m] = sm[m][0];
}

// final_sums of at most kFuseParts partials, the same additions in the same
// order, by every wavefront on its own: no barrier, and the sum in all of its
// lanes.  A kernel that needs a scalar of the iteration forms it like this in
// each of its wavefronts, where a launch of one workgroup had done it.  The
// constructor only asks for the partials; other loads may follow before sum().
struct WaveSum {
  double v[2][4];
  __device__ __forceinline__ WaveSum(const double *part, int m, int nblk) {
#pragma unroll
    for (int i = 0; i < kFuseParts / kBS; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int b = (int)(threadIdx.x & 63) + 64 * q + kBS * i;
        v[i][q] = b < nblk ? part[3 * b + m] : 0.0;
      }
  }
  __device__ __forceinline__ double sum() const {
    double a[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) a[q] = (0.0 + v[0][q]) + v[1][q];
    double s = (a[0] + a[2]) + (a[1] + a[3]);
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) s += __shfl_down(s, d, 64);
    return __shfl(s, 0, 64);
  }
};

// start of a solve: rr = |r0|^2, bb = |b|^2
__device__ __forceinline__ void fin0_logic(const KScal &k, double rr, double bb) {
  k.sc[S_RR] = rr; k.sc[S_BB] = bb; k.sc[S_RHO] = rr; k.sc[S_TRUE] = rr;
  k.sc[S_REF] = k.inner ? rr : bb;
  // an inner solve reduces its residual by kInnerTol, or only as far as the
  // outer test needs (|r| to TOL|b|, with a factor 2 margin), whichever is
  // less work
  k.sc[S_ITOL] = fmax(k.itol2, 0.25 * k.tol2 * bb / rr);
  k.sc[S_ALPHA] = 1.0; k.sc[S_OMEGA] = 1.0; k.sc[S_BETA] = 0.0;
  k.flag[1] = 0; k.flag[2] = 0;
  if (bb == 0.0) k.flag[0] = 4;                       // zero right-hand side: x = 0
  else if (!(rr == rr)) { k.flag[0] = 2; k.flag[2] = 1; }
  else if (rr <= k.tol2 * bb) k.flag[0] = 1;          // already converged
  else k.flag[0] = 0;
}

// The logic after the dots of an iteration.  Each returns the scalar that the
// kernels after it use and whether they run.  Where it is formed by every
// wavefront of a launch, all come to the same answer and one thread (`write`)
// records it; it writes nothing the others read but flag[0], which may make a
// wavefront that starts late leave early: after a stop nothing the launch
// writes is used, or the launch leaves by the returned `go`.

// alpha = rho / (rh, v)
__device__ __forceinline__ bool fin1_logic(const KScal &k, double rhv, double &alpha, bool write = true) {
  if (write) k.sc[S_RHV] = rhv;
  if (rhv == 0.0 || !(rhv == rhv)) {
    if (write) { k.flag[0] = 2; k.flag[2] = 2; }
    return false;
  }
  alpha = k.sc[S_RHO] / rhv;
  if (write) k.sc[S_ALPHA] = alpha;
  return true;
}

// omega = (t, s) / (t, t); keeps rho for fin3_logic, which replaces it
__device__ __forceinline__ bool fin2_logic(const KScal &k, double ts, double tt, double &omega, bool write = true) {
  // tt == 0 means s == 0: the half step already solves the system
  omega = tt == 0.0 ? 0.0 : ts / tt;
  const bool go = tt == tt;
  if (write) {
    k.sc[S_TS] = ts; k.sc[S_TT] = tt;
    k.sc[S_OMEGA] = omega;
    k.sc[S_RHOP] = k.sc[S_RHO];
    if (!go) { k.flag[0] = 2; k.flag[2] = 3; }
  }
  return go;
}

// convergence test and beta after the update; rhr = (rh, r), rr = |r|^2
__device__ __forceinline__ bool fin3_logic(const KScal &k, double rhr, double rr, double &beta, bool write = true) {
  const double omega = k.sc[S_OMEGA];
  const bool nan = !(rr == rr), done = rr <= (k.inner ? k.sc[S_ITOL] : k.tol2) * k.sc[S_REF];
  const bool broke = rhr == 0.0 || omega == 0.0;
  if (write) {
    const int it = k.flag[1] + 1;
    k.flag[1] = it;
    k.sc[S_RR] = rr;
    if (nan) { k.flag[0] = 2; k.flag[2] = 4; }
    else if (done) k.flag[0] = 1;
    else if (it >= k.itmax) k.flag[0] = 3;
    else if (broke) { k.flag[0] = 2; k.flag[2] = 5; }
  }
  if (nan || done || broke) return false;
  beta = (rhr / k.sc[S_RHOP]) * (k.sc[S_ALPHA] / omega);
  if (write) { k.sc[S_BETA] = beta; k.sc[S_RHO] = rhr; }
  return true;
}

}  // namespace nhw

// Dense (non-diagonal) strategies for many small systems at once.
//
// With a full lin_op the reference's coefficients are matrices
// (etd35.py:602-670 and the other dense update_coeffs): per fraction f of
// z = h L the exponential exp(f z) (scipy's expm) and
//   h psi_r(f z) = h (1/N) sum_m r_m psi_r(r_m) (r_m I - f z)^-1
// over the contour r_m = R exp(2 pi i (m + 1/2) / N); each coefficient is a
// combination of those (the method tableau's recipes); stages are
// matrix-vector products (etd35.py:671-720).  Here every step runs on the
// device for a batch of systems (one lin_op and h each, one workgroup per
// system per launch):
//   * exponentials: scaling and squaring with the degree-13 Pade approximant
//     (Higham, "The scaling and squaring method for the matrix exponential
//     revisited", SIAM J. Matrix Anal. Appl. 26 (2005)), the linear system
//     (V - U) X = V + U by Gauss-Jordan elimination with partial pivoting;
//   * contour: one Gauss-Jordan inverse per (system, fraction, node), then a
//     fixed-order weighted sum over the nodes;
//   * recipes: elementwise combinations into the coefficient matrices;
//   * stages: batched sums of matrix-vector products (rks_dense_combine).
// Matrices are row-major n x n complex128; work matrices live in a device
// workspace (L2-resident at these sizes), each workgroup on its own.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "rkstiff_amd.h"
#include "rks_math.h"
#include "rks_types.h"

void rks_set_last_error(const std::string& msg);  // rks_host.hip
int rks_build_tableau(int method, rks_tableau* out);  // rks_tableau.cpp

namespace {

constexpr int DT = 256;          // threads per system
constexpr int DMAX = 256;        // largest n
constexpr int NPADE = 14;        // degree-13 Pade coefficients b_0..b_13
// coefficients b_0..b_13 of the degree-13 Pade approximant
static constexpr __device__ double PADE[NPADE] = {64764752532480000.0, 32382376266240000.0, 7771770303897600.0, 1187353796428800.0,
                                                129060195264000.0,   10559470521600.0,    670442572800.0,     33522128640.0,
                                                1323241920.0,        40840800.0,          960960.0,           16380.0,
                                                182.0,               1.0};
constexpr double THETA13 = 5.371920351148152;  // 1-norm bound of the degree-13 approximant (Higham 2005)

int dfail(int code, const std::string& msg) {
  rks_set_last_error(msg);
  return code;
}

__device__ __forceinline__ z64 zadd(z64 a, z64 b) { return mkc(a.re + b.re, a.im + b.im); }
__device__ __forceinline__ z64 zsub(z64 a, z64 b) { return mkc(a.re - b.re, a.im - b.im); }
__device__ __forceinline__ z64 zscale(double s, z64 a) { return mkc(s * a.re, s * a.im); }
__device__ __forceinline__ z64 zmul(z64 a, z64 b) {
  return mkc(fma(a.re, b.re, -(a.im * b.im)), fma(a.re, b.im, a.im * b.re));
}
// Smith's division
__device__ __forceinline__ z64 zdiv(z64 a, z64 b) {
  if (fabs(b.re) >= fabs(b.im)) {
    const double r = b.im / b.re, d = b.re + b.im * r;
    return mkc((a.re + a.im * r) / d, (a.im - a.re * r) / d);
  }
  const double r = b.re / b.im, d = b.im + b.re * r;
  return mkc((a.re * r + a.im) / d, (a.im * r - a.re) / d);
}

// C = A B (n x n), every thread of the workgroup; ends on a barrier
__device__ void gemm(int n, const z64* __restrict__ A, const z64* __restrict__ B, z64* __restrict__ C) {
  for (int e = threadIdx.x; e < n * n; e += DT) {
    const int i = e / n, j = e - i * n;
    double re = 0.0, im = 0.0;
    for (int k = 0; k < n; ++k) {
      const z64 a = A[i * n + k], b = B[k * n + j];
      re = fma(a.re, b.re, re);
      re = fma(-a.im, b.im, re);
      im = fma(a.re, b.im, im);
      im = fma(a.im, b.re, im);
    }
    C[e] = mkc(re, im);
  }
  __syncthreads();
}

// Gauss-Jordan elimination with partial pivoting on the n x (n + nr) row-major
// augmented matrix [M | R] (stride w = n + nr): R <- M^-1 R.  piv/fac: LDS scratch.
__device__ void gauss_jordan(int n, int nr, z64* __restrict__ Aug, z64* fac, int* piv) {
  const int w = n + nr;
  const int t = threadIdx.x;
  for (int k = 0; k < n; ++k) {
    if (t < 64) {
      // pivot: largest |re| + |im| in column k at or below row k (first on ties)
      double best = -1.0;
      int bi = k;
      for (int i = k + t; i < n; i += 64) {
        const z64 v = Aug[i * w + k];
        const double a = fabs(v.re) + fabs(v.im);
        if (a > best) {
          best = a;
          bi = i;
        }
      }
      for (int o = 32; o >= 1; o >>= 1) {
        const double ob = __shfl_xor(best, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        if (ob > best || (ob == best && oi < bi)) {
          best = ob;
          bi = oi;
        }
      }
      if (t == 0) *piv = bi;
    }
    __syncthreads();
    const int p = *piv;
    if (p != k)
      for (int j = t; j < w; j += DT) {
        const z64 a = Aug[k * w + j];
        Aug[k * w + j] = Aug[p * w + j];
        Aug[p * w + j] = a;
      }
    __syncthreads();
    const z64 d = Aug[k * w + k];
    __syncthreads();
    for (int j = t; j < w; j += DT) Aug[k * w + j] = zdiv(Aug[k * w + j], d);
    for (int i = t; i < n; i += DT) fac[i] = Aug[i * w + k];
    __syncthreads();
    for (int e = t; e < n * w; e += DT) {
      const int i = e / w, j = e - i * w;
      if (i == k || j < k) continue;
      Aug[e] = zsub(Aug[e], zmul(fac[i], Aug[k * w + j]));
    }
    __syncthreads();
  }
}

struct ExpmJob {
  const z64* L;   // [batch][n][n]
  const double* h;
  int n, nfrac;
  int fnum[RKS_MAX_FRAC], fden[RKS_MAX_FRAC];
  z64* out;       // [batch][nfrac][n][n]: exp(f h L)
  z64* ws;        // [batch][nfrac][9][n][n]: A, A^2, A^4, A^6, U, V, T and the n x 2n system
};

// exp(f h L) of (fraction blockIdx.x, system blockIdx.y)
__global__ __launch_bounds__(DT) void dense_expm(ExpmJob J) {
  __shared__ z64 fac[DMAX];
  __shared__ int piv;
  __shared__ double red[DT / 64];
  __shared__ int s_sq;
  const int f = blockIdx.x, b = blockIdx.y, n = J.n, nn = n * n, t = threadIdx.x;
  const z64* L = J.L + (size_t)b * nn;
  const double h = J.h[b];
  z64* base = J.ws + ((size_t)b * J.nfrac + f) * 9 * nn;
  z64 *A = base, *A2 = base + nn, *A4 = A2 + nn, *A6 = A4 + nn, *U = A6 + nn, *V = U + nn, *T = V + nn;
  z64* Aug = T + nn;  // n x 2n
  const double num = (double)J.fnum[f], den = (double)J.fden[f];
  for (int e = t; e < nn; e += DT) {
    const z64 z = mkc(h * L[e].re, h * L[e].im);
    A[e] = mkc((num * z.re) / den, (num * z.im) / den);
  }
  __syncthreads();
  // 1-norm (largest column sum of |a_ij|) and the scaling 2^-s that brings it under theta_13
  double cmax = 0.0;
  for (int j = t; j < n; j += DT) {
    double s = 0.0;
    for (int i = 0; i < n; ++i) s += hypot(A[i * n + j].re, A[i * n + j].im);
    cmax = s > cmax ? s : cmax;
  }
  for (int o = 32; o >= 1; o >>= 1) {
    const double v = __shfl_xor(cmax, o, 64);
    cmax = v > cmax ? v : cmax;
  }
  if ((t & 63) == 0) red[t >> 6] = cmax;
  __syncthreads();
  if (t == 0) {
    double m = red[0];
    for (int i = 1; i < DT / 64; ++i) m = red[i] > m ? red[i] : m;
    int s = 0;
    if (m > THETA13) s = (int)ceil(log2(m / THETA13));
    s_sq = s < 0 ? 0 : s;
  }
  __syncthreads();
  const int sq = s_sq;
  if (sq > 0) {
    const double sc = ldexp(1.0, -sq);
    for (int e = t; e < nn; e += DT) A[e] = zscale(sc, A[e]);
    __syncthreads();
  }
  gemm(n, A, A, A2);
  gemm(n, A2, A2, A4);
  gemm(n, A4, A2, A6);
  // U = A (A6 (b13 A6 + b11 A4 + b9 A2) + b7 A6 + b5 A4 + b3 A2 + b1 I)
  // V = A6 (b12 A6 + b10 A4 + b8 A2) + b6 A6 + b4 A4 + b2 A2 + b0 I
  for (int e = t; e < nn; e += DT) {
    U[e] = zadd(zadd(zscale(PADE[13], A6[e]), zscale(PADE[11], A4[e])), zscale(PADE[9], A2[e]));
    V[e] = zadd(zadd(zscale(PADE[12], A6[e]), zscale(PADE[10], A4[e])), zscale(PADE[8], A2[e]));
  }
  __syncthreads();
  gemm(n, A6, U, T);
  for (int e = t; e < nn; e += DT) {
    const int i = e / n, j = e - i * n;
    z64 v = zadd(zadd(zadd(T[e], zscale(PADE[7], A6[e])), zscale(PADE[5], A4[e])), zscale(PADE[3], A2[e]));
    if (i == j) v.re += PADE[1];
    U[e] = v;  // inner bracket of U
  }
  __syncthreads();
  gemm(n, A6, V, T);
  for (int e = t; e < nn; e += DT) {
    const int i = e / n, j = e - i * n;
    z64 v = zadd(zadd(zadd(T[e], zscale(PADE[6], A6[e])), zscale(PADE[4], A4[e])), zscale(PADE[2], A2[e]));
    if (i == j) v.re += PADE[0];
    V[e] = v;
  }
  __syncthreads();
  gemm(n, A, U, T);  // T = U
  // (V - U) X = V + U
  for (int e = t; e < nn; e += DT) {
    const int i = e / n, j = e - i * n;
    Aug[i * 2 * n + j] = zsub(V[e], T[e]);
    Aug[i * 2 * n + n + j] = zadd(V[e], T[e]);
  }
  __syncthreads();
  gauss_jordan(n, n, Aug, fac, &piv);
  z64* X = U;
  for (int e = t; e < nn; e += DT) {
    const int i = e / n, j = e - i * n;
    X[e] = Aug[i * 2 * n + n + j];
  }
  __syncthreads();
  // undo the scaling: X <- X^(2^s)
  for (int r = 0; r < sq; ++r) {
    gemm(n, X, X, T);
    z64* tmp = X;
    X = T;
    T = tmp;
  }
  z64* out = J.out + ((size_t)b * J.nfrac + f) * nn;
  for (int e = t; e < nn; e += DT) out[e] = X[e];
}

struct ContourJob {
  const z64* L;
  const double* h;
  int n, npts, nfrac;
  double radius;
  int fnum[RKS_MAX_FRAC], fden[RKS_MAX_FRAC];
  z64* Q;    // [batch][nfrac][npts][n][n]: (r_m I - f h L)^-1
  z64* ws;   // [batch][nfrac][npts][n][2n]
};

// (r_m I - f h L)^-1 of (node blockIdx.x, fraction blockIdx.y, system blockIdx.z)
__global__ __launch_bounds__(DT) void dense_contour_inverse(ContourJob J) {
  __shared__ z64 fac[DMAX];
  __shared__ int piv;
  const int m = blockIdx.x, f = blockIdx.y, b = blockIdx.z, n = J.n, nn = n * n, t = threadIdx.x;
  const size_t job = ((size_t)b * J.nfrac + f) * J.npts + m;
  z64* Aug = J.ws + job * 2 * nn;
  const z64* L = J.L + (size_t)b * nn;
  const double h = J.h[b];
  const double th = (6.283185307179586 * (m + 0.5)) / (double)J.npts;
  const z64 r = mkc(J.radius * cos(th), J.radius * sin(th));
  const double num = (double)J.fnum[f], den = (double)J.fden[f];
  for (int e = t; e < nn; e += DT) {
    const int i = e / n, j = e - i * n;
    const z64 z = mkc(h * L[e].re, h * L[e].im);
    const z64 fz = mkc((num * z.re) / den, (num * z.im) / den);
    Aug[i * 2 * n + j] = (i == j) ? zsub(r, fz) : mkc(-fz.re, -fz.im);
    Aug[i * 2 * n + n + j] = mkc(i == j ? 1.0 : 0.0, 0.0);
  }
  __syncthreads();
  gauss_jordan(n, n, Aug, fac, &piv);
  z64* Q = J.Q + job * nn;
  for (int e = t; e < nn; e += DT) {
    const int i = e / n, j = e - i * n;
    Q[e] = Aug[i * 2 * n + n + j];
  }
}

// ---------------------------------------------------------------------------
// Small systems (n <= DSMALL): the matrices of one exponential or one contour node live in
// LDS.  The global-memory kernels above are bound by latency: per pivot column a
// Gauss-Jordan pass makes five dependent trips to L2, each followed by a barrier.  One
// launch does the nodes and the exponentials of every fraction and system.  The operations
// on each element are those above, in the same order.
// Chebyshev n = 19, ETD35, 64 nodes, one coefficient update: exponentials, inverses and
// recipes took 82 + 61 + 68 us from global memory; whole run (7 updates) 8.0 -> 5.3 ms.
// ---------------------------------------------------------------------------
constexpr int DSMALL = 40;                             // 6 n^2 matrices of 16 bytes: 150 KB
constexpr int DEPT = (DSMALL * DSMALL + DT - 1) / DT;  // elements per thread

// the thread's elements e = t + q DT of an n x n matrix, by row and column
struct Cells {
  int n, row[DEPT], col[DEPT];
  __device__ __forceinline__ explicit Cells(int n_) : n(n_) {
#pragma unroll
    for (int q = 0; q < DEPT; ++q) {
      const int e = (int)threadIdx.x + q * DT;
      row[q] = e / n;
      col[q] = e - row[q] * n;
    }
  }
  template <typename F>
  __device__ __forceinline__ void each(F f) const {
#pragma unroll
    for (int q = 0; q < DEPT; ++q)
      if (row[q] < n) f((int)threadIdx.x + q * DT, row[q], col[q], q);
  }
};

// f(e, i, j, (A B)_e) after every thread has read A and B, so f may overwrite them; ends on a barrier
template <typename F>
__device__ __forceinline__ void lds_gemm(const Cells& c, const z64* A, const z64* B, F f) {
  z64 r[DEPT];
  const int n = c.n;
  c.each([&](int, int i, int j, int q) {
    double re = 0.0, im = 0.0;
#pragma unroll 4
    for (int k = 0; k < n; ++k) {
      const z64 a = A[i * n + k], b = B[k * n + j];
      re = fma(a.re, b.re, re);
      re = fma(-a.im, b.im, re);
      im = fma(a.re, b.im, im);
      im = fma(a.im, b.re, im);
    }
    r[q] = mkc(re, im);
  });
  __syncthreads();
  c.each([&](int e, int i, int j, int q) { f(e, i, j, r[q]); });
  __syncthreads();
}

// gauss_jordan above on an n x 2n system in LDS: R <- M^-1 R
__device__ __forceinline__ void lds_gauss_jordan(int n, z64* Aug, z64* fac, int* piv) {
  const int w = 2 * n, t = threadIdx.x, tx = t & 31, ty = t >> 5;
  for (int k = 0; k < n; ++k) {
    if (t < 64) {
      double best = -1.0;
      int bi = k;
      if (k + t < n) {
        const z64 v = Aug[(k + t) * w + k];
        const double a = fabs(v.re) + fabs(v.im);
        if (a > best) {
          best = a;
          bi = k + t;
        }
      }
      for (int o = 32; o >= 1; o >>= 1) {
        const double ob = __shfl_xor(best, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        if (ob > best || (ob == best && oi < bi)) {
          best = ob;
          bi = oi;
        }
      }
      if (t == 0) *piv = bi;
    }
    __syncthreads();
    const int p = *piv;
    // thread j: the new row k, scaled by the pivot, and the displaced row
    const z64 d = Aug[p * w + k];
    z64 rk = mkc(0.0, 0.0), rp = rk;
    if (t < w) {
      rp = Aug[p * w + t];
      rk = Aug[k * w + t];
    }
    __syncthreads();
    if (t < w) {
      if (p != k) Aug[p * w + t] = rk;
      Aug[k * w + t] = zdiv(rp, d);
    }
    __syncthreads();
    for (int i = t; i < n; i += DT) fac[i] = Aug[i * w + k];
    __syncthreads();
    for (int i = ty; i < n; i += DT / 32) {
      if (i == k) continue;
      const z64 f = fac[i];
      for (int j = k + tx; j < w; j += 32) Aug[i * w + j] = zsub(Aug[i * w + j], zmul(f, Aug[k * w + j]));
    }
    __syncthreads();
  }
}

struct SmallJob {
  const z64* L;     // [batch][n][n]
  const double* h;  // [batch]
  int n, npts, nfrac;
  double radius;
  int fnum[RKS_MAX_FRAC], fden[RKS_MAX_FRAC];
  z64* E;  // [batch][nfrac][n][n]: exp(f h L)
  z64* Q;  // [batch][nfrac][npts][n][n]: (r_m I - f h L)^-1
};

// node blockIdx.x (npts: the exponential) of fraction blockIdx.y, system blockIdx.z
__global__ __launch_bounds__(DT) void dense_small(SmallJob J) {
  extern __shared__ __align__(16) unsigned char dsmem[];
  __shared__ z64 fac[DSMALL];
  __shared__ int piv;
  __shared__ double red[DT / 64];
  __shared__ int s_sq;
  const int m = blockIdx.x, f = blockIdx.y, b = blockIdx.z, n = J.n, nn = n * n, t = threadIdx.x;
  const z64* L = J.L + (size_t)b * nn;
  const double h = J.h[b];
  const double num = (double)J.fnum[f], den = (double)J.fden[f];
  const Cells c(n);
  z64* M = (z64*)dsmem;
  if (m < J.npts) {
    z64* Aug = M;  // n x 2n
    const double th = (6.283185307179586 * (m + 0.5)) / (double)J.npts;
    const z64 r = mkc(J.radius * cos(th), J.radius * sin(th));
    c.each([&](int e, int i, int j, int) {
      const z64 z = mkc(h * L[e].re, h * L[e].im);
      const z64 fz = mkc((num * z.re) / den, (num * z.im) / den);
      Aug[i * 2 * n + j] = (i == j) ? zsub(r, fz) : mkc(-fz.re, -fz.im);
      Aug[i * 2 * n + n + j] = mkc(i == j ? 1.0 : 0.0, 0.0);
    });
    __syncthreads();
    lds_gauss_jordan(n, Aug, fac, &piv);
    z64* Q = J.Q + (((size_t)b * J.nfrac + f) * J.npts + m) * nn;
    c.each([&](int e, int i, int j, int) { Q[e] = Aug[i * 2 * n + n + j]; });
    return;
  }
  // exp(f h L): dense_expm above; A2 and A4 become the n x 2n system
  z64 *A = M, *A2 = M + nn, *A4 = A2 + nn, *A6 = A4 + nn, *U = A6 + nn, *V = U + nn;
  c.each([&](int e, int, int, int) {
    const z64 z = mkc(h * L[e].re, h * L[e].im);
    A[e] = mkc((num * z.re) / den, (num * z.im) / den);
  });
  __syncthreads();
  double cmax = 0.0;
  for (int j = t; j < n; j += DT) {
    double s = 0.0;
    for (int i = 0; i < n; ++i) s += hypot(A[i * n + j].re, A[i * n + j].im);
    cmax = s > cmax ? s : cmax;
  }
  for (int o = 32; o >= 1; o >>= 1) {
    const double v = __shfl_xor(cmax, o, 64);
    cmax = v > cmax ? v : cmax;
  }
  if ((t & 63) == 0) red[t >> 6] = cmax;
  __syncthreads();
  if (t == 0) {
    double mx = red[0];
    for (int i = 1; i < DT / 64; ++i) mx = red[i] > mx ? red[i] : mx;
    int s = 0;
    if (mx > THETA13) s = (int)ceil(log2(mx / THETA13));
    s_sq = s < 0 ? 0 : s;
  }
  __syncthreads();
  const int sq = s_sq;
  if (sq > 0) {
    const double sc = ldexp(1.0, -sq);
    c.each([&](int e, int, int, int) { A[e] = zscale(sc, A[e]); });
    __syncthreads();
  }
  lds_gemm(c, A, A, [&](int e, int, int, z64 r) { A2[e] = r; });
  lds_gemm(c, A2, A2, [&](int e, int, int, z64 r) { A4[e] = r; });
  lds_gemm(c, A4, A2, [&](int e, int, int, z64 r) {
    A6[e] = r;
    U[e] = zadd(zadd(zscale(PADE[13], r), zscale(PADE[11], A4[e])), zscale(PADE[9], A2[e]));
    V[e] = zadd(zadd(zscale(PADE[12], r), zscale(PADE[10], A4[e])), zscale(PADE[8], A2[e]));
  });
  lds_gemm(c, A6, U, [&](int e, int i, int j, z64 r) {
    z64 v = zadd(zadd(zadd(r, zscale(PADE[7], A6[e])), zscale(PADE[5], A4[e])), zscale(PADE[3], A2[e]));
    if (i == j) v.re += PADE[1];
    U[e] = v;
  });
  lds_gemm(c, A6, V, [&](int e, int i, int j, z64 r) {
    z64 v = zadd(zadd(zadd(r, zscale(PADE[6], A6[e])), zscale(PADE[4], A4[e])), zscale(PADE[2], A2[e]));
    if (i == j) v.re += PADE[0];
    V[e] = v;
  });
  z64* Aug = A2;
  lds_gemm(c, A, U, [&](int e, int i, int j, z64 r) {
    Aug[i * 2 * n + j] = zsub(V[e], r);
    Aug[i * 2 * n + n + j] = zadd(V[e], r);
  });
  lds_gauss_jordan(n, Aug, fac, &piv);
  z64* X = U;
  c.each([&](int e, int i, int j, int) { X[e] = Aug[i * 2 * n + n + j]; });
  __syncthreads();
  for (int r = 0; r < sq; ++r) lds_gemm(c, X, X, [&](int e, int, int, z64 v) { X[e] = v; });
  z64* out = J.E + ((size_t)b * J.nfrac + f) * nn;
  c.each([&](int e, int, int, int) { out[e] = X[e]; });
}

struct RecipeJob {
  const z64* E;       // [batch][nfrac][n][n]
  const z64* Q;       // [batch][nfrac][npts][n][n]
  const double* h;
  const z64* w;       // [3][npts]: r_m psi_r(r_m) / N
  int n, npts, nfrac, ncoef;
  z64* C;             // [batch][ncoef][n][n]
  rks_coef coef[RKS_MAX_COEF];  // the method's recipes
};

// coefficient matrix c (blockIdx.x) of system blockIdx.y: its recipe over the
// fraction's exponential and h psi_r (contour sums in node order).  A thread per element:
// the nodes of one element are one serial sum, so the loads of several nodes are issued
// together and the sums of the recipe's psi_r share them.
constexpr int RT = 64;
__global__ __launch_bounds__(RT) void dense_recipes(RecipeJob J) {
  const int c = blockIdx.x, b = blockIdx.y, n = J.n, nn = n * n;
  const rks_coef& cf = J.coef[c];
  const int f = cf.frac;
  const double h = J.h[b];
  const z64* E = J.E + ((size_t)b * J.nfrac + f) * nn;
  const z64* Q = J.Q + ((size_t)b * J.nfrac + f) * J.npts * nn;
  z64* C = J.C + ((size_t)b * J.ncoef + c) * nn;
  bool psi = false;
  for (int k = 0; k < cf.nb; ++k) psi |= cf.kind[k] != RKS_BASIS_EXP;
  for (int e = blockIdx.z * RT + threadIdx.x; e < nn; e += gridDim.z * RT) {
    z64 s[3] = {mkc(0.0, 0.0), mkc(0.0, 0.0), mkc(0.0, 0.0)};
    if (psi) {
      int m = 0;
      constexpr int U = 16;
      for (; m + U <= J.npts; m += U) {
        z64 q[U];
#pragma unroll
        for (int i = 0; i < U; ++i) q[i] = Q[(size_t)(m + i) * nn + e];
#pragma unroll
        for (int i = 0; i < U; ++i)
#pragma unroll
          for (int r = 0; r < 3; ++r) s[r] = zadd(s[r], zmul(J.w[r * J.npts + m + i], q[i]));
      }
      for (; m < J.npts; ++m) {
        const z64 q = Q[(size_t)m * nn + e];
#pragma unroll
        for (int r = 0; r < 3; ++r) s[r] = zadd(s[r], zmul(J.w[r * J.npts + m], q));
      }
    }
    z64 acc = mkc(0.0, 0.0);
    for (int k = 0; k < cf.nb; ++k) {
      const int kind = cf.kind[k];
      const z64 bv = kind == RKS_BASIS_EXP ? E[e] : zscale(h, kind == 1 ? s[0] : (kind == 2 ? s[1] : s[2]));
      const double wk = cf.hmul ? cf.w[k] * h : cf.w[k];
      acc = zadd(acc, zscale(wk, bv));
    }
    if (cf.outer != 1.0) acc = zscale(cf.outer, acc);
    if (cf.den != 1.0) acc = mkc(acc.re / cf.den, acc.im / cf.den);
    C[e] = acc;
  }
}

struct CombineJob {
  rks_dense_term t[RKS_DENSE_MAX_TERMS];
  int nterm, n;
  z64* y;  // [batch][n]
};

// y_b = sum_t alpha_t M_t,b (x_t,b + s2_t x2_t,b) for system blockIdx.x.  A thread per term
// and row: a row's dot product is one serial chain, so the terms' chains run side by side
// (a thread per row walked all of them: 10 us for 6 terms at n = 19), and are then added in
// order.  Dynamic LDS: the vectors and the products, [nterm][n] each.
__global__ __launch_bounds__(DT) void dense_combine(CombineJob J) {
  extern __shared__ __align__(16) unsigned char dsmem[];
  const int b = blockIdx.x, n = J.n, t = threadIdx.x, total = J.nterm * n;
  z64* v = (z64*)dsmem;
  z64* prod = v + total;
  for (int e = t; e < total; e += DT) {
    const int k = e / n, i = e - k * n;
    const rks_dense_term& tm = J.t[k];
    z64 a = ((const z64*)tm.x)[(size_t)b * n + i];
    if (tm.x2) a = zadd(a, zscale(tm.s2, ((const z64*)tm.x2)[(size_t)b * n + i]));
    v[e] = a;
  }
  __syncthreads();
  for (int e = t; e < total; e += DT) {
    const int k = e / n, i = e - k * n;
    const rks_dense_term& tm = J.t[k];
    z64 p = v[e];
    if (tm.mat) {
      const z64* M = (const z64*)tm.mat + (size_t)b * n * n + (size_t)i * n;
      const z64* x = v + k * n;
      double re = 0.0, im = 0.0;
#pragma unroll 8
      for (int j = 0; j < n; ++j) {
        const z64 a = M[j], q = x[j];
        re = fma(a.re, q.re, re);
        re = fma(-a.im, q.im, re);
        im = fma(a.re, q.im, im);
        im = fma(a.im, q.re, im);
      }
      p = mkc(re, im);
    }
    prod[e] = p;
  }
  __syncthreads();
  for (int i = t; i < n; i += DT) {
    z64 acc = mkc(0.0, 0.0);
    for (int k = 0; k < J.nterm; ++k) acc = zadd(acc, zscale(J.t[k].alpha, prod[k * n + i]));
    J.y[(size_t)b * n + i] = acc;
  }
}

// byte offsets of the work memory's parts (the step sizes first)
struct DenseLayout {
  size_t w, E, Q, wsE, wsQ, total;
};

DenseLayout dense_layout(const rks_tableau& tb, int n, int batch, int npts) {
  bool psi = false;
  for (int f = 0; f < tb.nfrac; ++f) psi |= (tb.frac[f].mask & 14) != 0;
  const size_t nn = (size_t)n * n * sizeof(z64), mats = nn * tb.nfrac * batch;
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t o = at;
    at += (bytes + 255) & ~(size_t)255;
    return o;
  };
  DenseLayout d;
  take(sizeof(double) * batch);
  d.w = take(sizeof(z64) * 3 * (size_t)npts);
  d.E = take(mats);
  d.Q = take(psi ? mats * npts : 0);
  d.wsE = take(n > DSMALL ? mats * 9 : 0);
  d.wsQ = take(psi && n > DSMALL ? mats * 2 * npts : 0);
  d.total = at;
  return d;
}

int dense_check(int method, int n, int batch, int contour_points, rks_tableau* tb) {
  if (n < 1 || n > DMAX) return dfail(RKS_ERR_INVALID, "dense systems need 1 <= n <= 256");
  if (batch < 1) return dfail(RKS_ERR_INVALID, "batch must be >= 1");
  if (contour_points < 2) return dfail(RKS_ERR_INVALID, "contour_points must be >= 2 and contour_radius > 0");
  if (rks_build_tableau(method, tb) != RKS_OK) return dfail(RKS_ERR_INVALID, "unknown method");
  return RKS_OK;
}

struct DeviceBuf {
  void* p = nullptr;
  ~DeviceBuf() { (void)hipFree(p); }
};

}  // namespace

extern "C" {

// Work memory of a coefficient update: step sizes, contour weights, exponentials, node
// inverses, and (n > DSMALL) the matrices that the global-memory kernels work on.
int rks_dense_ws_bytes(int method, int n, int batch, int contour_points, size_t* bytes) {
  rks_tableau tb;
  if (!bytes) return dfail(RKS_ERR_INVALID, "null argument");
  const int rc = dense_check(method, n, batch, contour_points, &tb);
  if (rc == RKS_OK) *bytes = dense_layout(tb, n, batch, contour_points).total;
  return rc;
}

int rks_dense_coeffs(int method, int n, int batch, const void* L, const double* h, int contour_points,
                     double contour_radius, void* coeffs, hipStream_t stream) {
  if (!L || !h || !coeffs) return dfail(RKS_ERR_INVALID, "null argument");
  DeviceBuf ws;
  size_t bytes = 0;
  int rc = rks_dense_ws_bytes(method, n, batch, contour_points, &bytes);
  if (rc != RKS_OK) return rc;
  hipError_t e = hipMalloc(&ws.p, bytes);
  if (e != hipSuccess) return dfail(RKS_ERR_HIP, std::string("rks_dense_coeffs: ") + hipGetErrorString(e));
  rc = rks_dense_coeffs_ws(method, n, batch, L, h, contour_points, contour_radius, coeffs, ws.p, bytes, stream);
  if (rc != RKS_OK) return rc;
  // the work buffer is released when the launches are done
  e = hipStreamSynchronize(stream);
  if (e != hipSuccess) return dfail(RKS_ERR_HIP, std::string("rks_dense_coeffs: ") + hipGetErrorString(e));
  return RKS_OK;
}

int rks_dense_coeffs_ws(int method, int n, int batch, const void* L, const double* h, int contour_points,
                        double contour_radius, void* coeffs, void* ws, size_t ws_bytes, hipStream_t stream) {
  if (!L || !h || !coeffs) return dfail(RKS_ERR_INVALID, "null argument");
  rks_tableau tb;
  const int ok = dense_check(method, n, batch, contour_points, &tb);
  if (ok != RKS_OK) return ok;
  if (!(contour_radius > 0.0)) return dfail(RKS_ERR_INVALID, "contour_points must be >= 2 and contour_radius > 0");
  const size_t nn = (size_t)n * n;
  const int nf = tb.nfrac, np = contour_points;
  int need_psi = 0;
  for (int f = 0; f < nf; ++f) need_psi |= (tb.frac[f].mask & 14) != 0;
  // the step sizes and contour weights r_m psi_r(r_m) / N (etd35.py:622-634)
  const DenseLayout at = dense_layout(tb, n, batch, np);
  if (!ws || ws_bytes < at.total) return dfail(RKS_ERR_INVALID, "rks_dense_coeffs_ws: workspace too small");
  std::vector<char> head(at.E);  // step sizes and weights, as they lie in the workspace
  std::copy(h, h + batch, (double*)head.data());
  z64* const w = (z64*)(head.data() + at.w);
  for (int m = 0; m < np; ++m) {
    const double th = (6.283185307179586 * (m + 0.5)) / (double)np;
    const double rr = contour_radius * std::cos(th), ri = contour_radius * std::sin(th);
    // psi_1 = (e^r - 1)/r, psi_2 = 2 (e^r - 1 - r)/r^2, psi_3 = 6 (e^r - 1 - r - r^2/2)/r^3 in
    // std::complex arithmetic on the host (set-up, not a hot path)
    const double er = std::exp(rr);
    const double ec = er * std::cos(ri), es = er * std::sin(ri);
    auto cdiv = [](double ar, double ai, double br, double bi, double* qr, double* qi) {
      const double d = br * br + bi * bi;
      *qr = (ar * br + ai * bi) / d;
      *qi = (ai * br - ar * bi) / d;
    };
    double r2r = rr * rr - ri * ri, r2i = 2 * rr * ri;
    double r3r = r2r * rr - r2i * ri, r3i = r2r * ri + r2i * rr;
    double n1r = ec - 1.0, n1i = es;
    double n2r = n1r - rr, n2i = n1i - ri;
    double n3r = n2r - 0.5 * r2r, n3i = n2i - 0.5 * r2i;
    double p1r, p1i, p2r, p2i, p3r, p3i;
    cdiv(n1r, n1i, rr, ri, &p1r, &p1i);
    cdiv(2 * n2r, 2 * n2i, r2r, r2i, &p2r, &p2i);
    cdiv(6 * n3r, 6 * n3i, r3r, r3i, &p3r, &p3i);
    const double pr[3] = {p1r, p2r, p3r}, pi[3] = {p1i, p2i, p3i};
    for (int r = 0; r < 3; ++r) {
      const double wr = rr * pr[r] - ri * pi[r], wi = rr * pi[r] + ri * pr[r];
      w[(size_t)r * np + m] = z64{wr / np, wi / np};
    }
  }
  char* const base = (char*)ws;
  hipError_t e = hipMemcpyWithStream(base, head.data(), head.size(), hipMemcpyHostToDevice, stream);
  if (e != hipSuccess) return dfail(RKS_ERR_HIP, std::string("rks_dense_coeffs: ") + hipGetErrorString(e));
  z64 *const E = (z64*)(base + at.E), *const Q = (z64*)(base + at.Q);
  auto fill = [&](auto& job) {
    job.L = (const z64*)L;
    job.h = (const double*)base;
    job.n = n;
    job.nfrac = nf;
    for (int f = 0; f < nf; ++f) {
      job.fnum[f] = tb.frac[f].fnum;
      job.fden[f] = tb.frac[f].fden;
    }
  };
  if (n <= DSMALL) {
    SmallJob S{};
    fill(S);
    S.npts = need_psi ? np : 0;
    S.radius = contour_radius;
    S.E = E;
    S.Q = Q;
    const int lds = 6 * (int)(nn * sizeof(z64));
    // the limit of every size: another thread may be between its own call and launch
    e = hipFuncSetAttribute((const void*)dense_small, hipFuncAttributeMaxDynamicSharedMemorySize,
                            6 * DSMALL * DSMALL * (int)sizeof(z64));
    if (e != hipSuccess) return dfail(RKS_ERR_HIP, std::string("rks_dense_coeffs: ") + hipGetErrorString(e));
    hipLaunchKernelGGL(dense_small, dim3(S.npts + 1, nf, batch), dim3(DT), lds, stream, S);
  } else {
    ExpmJob X{};
    fill(X);
    X.out = E;
    X.ws = (z64*)(base + at.wsE);
    hipLaunchKernelGGL(dense_expm, dim3(nf, batch), dim3(DT), 0, stream, X);
    if (need_psi) {
      ContourJob Cj{};
      fill(Cj);
      Cj.npts = np;
      Cj.radius = contour_radius;
      Cj.Q = Q;
      Cj.ws = (z64*)(base + at.wsQ);
      hipLaunchKernelGGL(dense_contour_inverse, dim3(np, nf, batch), dim3(DT), 0, stream, Cj);
    }
  }
  RecipeJob R{};
  R.E = E;
  R.Q = Q;
  R.h = (const double*)base;
  R.w = (const z64*)(base + at.w);
  R.n = n;
  R.npts = np;
  R.nfrac = nf;
  R.ncoef = tb.ncoef;
  R.C = (z64*)coeffs;
  for (int c = 0; c < tb.ncoef; ++c) R.coef[c] = tb.coef[c];
  const int chunks = (int)((nn + RT - 1) / RT);
  hipLaunchKernelGGL(dense_recipes, dim3(tb.ncoef, batch, chunks < 64 ? chunks : 64), dim3(RT), 0, stream, R);
  e = hipGetLastError();
  if (e != hipSuccess) return dfail(RKS_ERR_HIP, std::string("rks_dense_coeffs: ") + hipGetErrorString(e));
  return RKS_OK;
}

int rks_dense_combine(int n, int batch, const rks_dense_term* terms, int nterm, void* y, hipStream_t stream) {
  if (!terms || !y) return dfail(RKS_ERR_INVALID, "null argument");
  if (n < 1 || n > DMAX) return dfail(RKS_ERR_INVALID, "dense systems need 1 <= n <= 256");
  if (batch < 1) return dfail(RKS_ERR_INVALID, "batch must be >= 1");
  if (nterm < 1 || nterm > RKS_DENSE_MAX_TERMS) return dfail(RKS_ERR_INVALID, "1 <= nterm <= 8");
  CombineJob J{};
  for (int k = 0; k < nterm; ++k) {
    if (!terms[k].x) return dfail(RKS_ERR_INVALID, "term without a vector");
    if (terms[k].x == y || terms[k].x2 == y) return dfail(RKS_ERR_INVALID, "y must not alias a term's vector");
    J.t[k] = terms[k];
  }
  J.nterm = nterm;
  J.n = n;
  J.y = (z64*)y;
  const size_t lds = 2 * (size_t)nterm * n * sizeof(z64);  // at most 64 KB
  hipLaunchKernelGGL(dense_combine, dim3(batch), dim3(DT), lds, stream, J);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return dfail(RKS_ERR_HIP, std::string("rks_dense_combine: ") + hipGetErrorString(e));
  return RKS_OK;
}

}  // extern "C"

// Stepping engine for gfx950: one workgroup integrates one trajectory.
//
// A persistent kernel pulls instances from an atomic work queue.  For each
// instance the workgroup runs the reference's whole control flow on the device
// (solveras.py:336-410 step, 556-650 evolve; solvercs.py:163-279):
//   * coefficient arrays are regenerated in FP64 when h changes
//     (exact compare, etd35.py:851-852), stored in engine precision;
//   * every stage is one pass over the modes: k = E u + sum C NL is formed in
//     registers, the nonlinear term takes it from there (inverse FFT, pointwise
//     product, forward FFT, exchanging through LDS) and the new NL array is
//     written once;
//   * the embedded error norm (solveras.py:449-455) is a workgroup reduction
//     accumulated in FP64, and the accept/reject dt controller
//     (solveras.py:457-554) runs in FP64 on the device.
// Nonlinear terms (built in):
//   NLK_ADVECT  coef * rfft(irfft(u) * irfft(i kx u))   (KS, Burgers, KdV)
//   NLK_CUBIC   i gamma fft(|v|^2 v), v = ifft(u)        (cubic NLS)
//   NLK_HANKEL  i gamma S Y (|f|^2 f), f = Y u / S       (radial NLS: the order-zero
//               Hankel transform as a dense nr x nr matrix Y, nr <= 1024 radial points,
//               the modes padded to the size class 2^LOG2N)
// Workspace per instance (engine precision complex, m modes each):
//   nslot NL arrays | 2 candidate buffers | ncoef coefficient arrays.
#pragma once
#include <hip/hip_runtime.h>

#include "rks_fft.h"
#include "rks_math.h"
#include "rks_method.h"
#include "rks_mlp.h"
#include "rks_types.h"

#define NLK_ADVECT 0
#define NLK_CUBIC 1
#define NLK_NONE 2
#define NLK_HANKEL 4

__host__ __device__ constexpr size_t rks_align256(size_t b) { return (b + 255) & ~(size_t)255; }

struct rks_launch {
  const rks_tableau* tab;
  const rks_ctrl* ctl;
  rks_inst* inst;
  const rks_io* io;
  const int* order;
  int count;
  int mode;
  int* queue;      // next item, or null where the grid has a workgroup per trajectory
  const void* tw;  // exp(-2 pi i x / N), x < N, engine precision
  rks_mlp_dev mlp; // learned step-size proposer (mlp.on = 0: the reference's controller only)
};

// threads per workgroup for an N-point problem (N/16 elements... capped at 512,
// at least two elements per thread in every transform)
__host__ __device__ constexpr int rks_threads(int log2n, int nlk) {
  const int N = 1 << log2n;
  if (nlk == NLK_HANKEL) return N < 64 ? 64 : (N > 512 ? 512 : N);
  const int lo = (nlk == NLK_ADVECT) ? (N / 4 < 64 ? N / 4 : 64) : (N / 2 < 64 ? N / 2 : 64);
  const int t = N / 16 > lo ? N / 16 : lo;
  return t > 512 ? 512 : t;
}

// largest in-register radix of the LDS FFT passes
#define RKS_MAXR 16

__device__ __forceinline__ double nanmax(double a, double b) {
  if (a != a) return a;
  if (b != b) return b;
  return a > b ? a : b;
}

template <int T>
__device__ __forceinline__ double wg_max(double v, double* red) {
  constexpr int W = T < 64 ? T : 64;
#pragma unroll
  for (int o = W / 2; o >= 1; o >>= 1) v = nanmax(v, __shfl_xor(v, o, 64));
  if (T <= 64) return v;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) red[wid] = v;
  __syncthreads();
  double r = red[0];
#pragma unroll
  for (int i = 1; i < T / 64; ++i) r = nanmax(r, red[i]);
  __syncthreads();
  return r;
}

template <int T>
__device__ __forceinline__ void wg_sum2(double& a, double& b, double* red) {
  constexpr int W = T < 64 ? T : 64;
#pragma unroll
  for (int o = W / 2; o >= 1; o >>= 1) {
    a += __shfl_xor(a, o, 64);
    b += __shfl_xor(b, o, 64);
  }
  if (T <= 64) return;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) {
    red[2 * wid] = a;
    red[2 * wid + 1] = b;
  }
  __syncthreads();
  a = red[0];
  b = red[1];
#pragma unroll
  for (int i = 1; i < T / 64; ++i) {
    a += red[2 * i];
    b += red[2 * i + 1];
  }
  __syncthreads();
}

// Error ratio s = safety (eps ||u_new|| / ||err||)^(1/q) from the masked sums
// (solveras.py:449-455).  With FP32 NL storage (lowp), stages that agree to
// storage precision -- e.g. a last step of ~1e-15 that lands on tf -- give
// err == 0 exactly: that error is below what the storage resolves, so s is
// DBL_MAX (accept, growth capped at MAX_S), not the FP64 zero-error s = inf
// that the reference rejects.
__device__ __forceinline__ double rks_error_ratio(double su, double se, double eps, double safety, int q,
                                                  bool lowp) {
  if (lowp && se == 0.0 && su > 0.0 && su <= __DBL_MAX__) return __DBL_MAX__;
  return safety * pow(eps * sqrt(su) / sqrt(se), 1.0 / (double)q);
}

// ---------------------------------------------------------------------------
// FP64 coefficients of one mode (etd35.py:169-288 and the other builders)
// ---------------------------------------------------------------------------
__device__ __forceinline__ z64 frac_arg(z64 z, int num, int den, int cplx) {
#pragma clang fp contract(off)
  z64 w = (num == 1) ? z : np_rmul((double)num, z);
  if (den == 1) return w;
  if (cplx) return np_rdiv(w, (double)den);
  return mkc(w.re / (double)den, w.im / (double)den);
}

__device__ __forceinline__ z64 contour_node(int npts, double radius, int j) {
  // R exp(2 pi i (j + 1/2) / N)   (etd35.py:259)
  const double th = (6.283185307179586 * (j + 0.5)) * (1.0 / (double)npts);
  double sn, cs;
  sincos(th, &sn, &cs);
  return mkc(radius * cs, radius * sn);
}

// The coefficient generator runs in a separate (noinline) function, where a
// reference argument is a per-lane generic pointer: every read of the
// tableau would be a vector memory load with full latency inside the
// per-mode recipe loops.  The tableau and controller are uniform and
// read-only during a launch, so the generator reads them through a
// constant-address-space view of the uniform pointer (scalar loads).
#define RKS_AS4 __attribute__((address_space(4)))
typedef RKS_AS4 const rks_tableau rks_ctab;
typedef RKS_AS4 const rks_ctrl rks_cctl;

template <typename P>
__device__ __forceinline__ P* rks_uniform_const(const void* p) {
  const unsigned long long v = (unsigned long long)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
  return (P*)(((unsigned long long)hi << 32) | lo);
}

__device__ __forceinline__ z64 mode_z(const double* __restrict__ L, int L_complex, int m, double h) {
  const z64 Lm = L_complex ? mkc(L[2 * m], L[2 * m + 1]) : mkc(L[m], 0.0);
  return mkc(h * Lm.re, h * Lm.im);
}

// Basis values (exp, h psi1, h psi2, h psi3) of fraction fnum/fden by the closed forms.
__device__ __forceinline__ void frac_direct(int fnum, int fden, int mask, z64 z, double h, int cplx, z64 (&v)[4]) {
#pragma clang fp contract(off)
  const z64 e = np_exp(frac_arg(z, fnum, fden, cplx));
  v[0] = e;
  if (mask & 14) {
    z64 p1, p2, p3 = mkc(0.0, 0.0);
    np_psi123_e(frac_arg(z, fnum, fden, 1), e, mask & 8, &p1, &p2, &p3);
    v[1] = np_rmul(h, p1);
    v[2] = np_rmul(h, p2);
    v[3] = np_rmul(h, p3);
  }
}

// psi_r(f Z) summed into acc[1..3] at one contour point Z.
__device__ __forceinline__ void frac_contour_add(int fnum, int fden, int mask, z64 Z, z64 (&acc)[4]) {
#pragma clang fp contract(off)
  z64 p1, p2, p3 = mkc(0.0, 0.0);
  np_psi123(frac_arg(Z, fnum, fden, 1), mask & 8, &p1, &p2, &p3);
  acc[1] = mkc(acc[1].re + p1.re, acc[1].im + p1.im);
  acc[2] = mkc(acc[2].re + p2.re, acc[2].im + p2.im);
  acc[3] = mkc(acc[3].re + p3.re, acc[3].im + p3.im);
}

// Every coefficient recipe of fraction f: c = (outer * sum_k w_k B_k) / den,
// stored at cbase + coef_off[c]*M in state (RS) or storage (RN) precision.
template <typename RS, typename RN, typename TB>
__device__ __forceinline__ void frac_coefs(TB& tb, int f, const z64 (&v)[4], double h, int cplx,
                                           int m, size_t M, char* __restrict__ cbase) {
#pragma clang fp contract(off)
  for (int c = 0; c < tb.ncoef; ++c) {
    auto& cf = tb.coef[c];
    if (cf.frac != f) continue;
    z64 acc = mkc(0.0, 0.0);
    for (int k = 0; k < cf.nb; ++k) {
      const int kd = cf.kind[k];
      const z64 bv = kd == 0 ? v[0] : (kd == 1 ? v[1] : (kd == 2 ? v[2] : v[3]));
      const double w = cf.hmul ? cf.w[k] * h : cf.w[k];
      const z64 t = (w == 1.0) ? bv : np_rmul(w, bv);
      acc = (k == 0) ? t : mkc(acc.re + t.re, acc.im + t.im);
    }
    if (cf.outer != 1.0) acc = np_rmul(cf.outer, acc);
    if (cf.den != 1.0) {
      if (cplx) acc = np_rdiv(acc, cf.den);
      else acc = mkc(acc.re / cf.den, acc.im / cf.den);
    }
    char* p = cbase + (size_t)tb.coef_off[c] * M;
    const int kind = tb.coef_rs[c];
    if (kind == RKS_CST_RS) ((cx<RS>*)p)[m] = mkc((RS)acc.re, (RS)acc.im);
    else if (kind == RKS_CST_RN) ((cx<RN>*)p)[m] = mkc((RN)acc.re, (RN)acc.im);
    else if (kind == RKS_CST_RS_REAL) ((RS*)p)[m] = (RS)acc.re;
    else ((RN*)p)[m] = (RN)acc.re;
  }
}

// All coefficients of one mode by one thread (generic-path and 2-D
// kernels).  The tableau and controller references must be uniform (one
// object for the launch); they are read through the scalar
// constant-address-space view.
// mL indexes lin_op, mS the coefficient arrays (the 2-D engine keeps them in
// a row-padded layout).
template <typename RS, typename RN>
__device__ void coef_mode_at(const rks_tableau& tb_in, const rks_ctrl& ct_in, const double* __restrict__ L,
                             int L_complex, int mL, int mS, int M, double h, char* __restrict__ cbase) {
#pragma clang fp contract(off)
  rks_ctab& tb = *rks_uniform_const<rks_ctab>(&tb_in);
  rks_cctl& ct = *rks_uniform_const<rks_cctl>(&ct_in);
  const int cplx = L_complex || tb.uses_contour;
  const z64 z = mode_z(L, L_complex, mL, h);
  const bool small = tb.uses_contour && hypot(z.re, z.im) < ct.modecutoff;
  for (int f = 0; f < tb.nfrac; ++f) {
    const int fnum = tb.frac[f].fnum, fden = tb.frac[f].fden, fmask = tb.frac[f].mask;
    z64 v[4];
    v[1] = v[2] = v[3] = mkc(0.0, 0.0);
    frac_direct(fnum, fden, fmask, z, h, cplx, v);
    if (small && (fmask & 14)) {
      z64 acc[4];
      acc[1] = acc[2] = acc[3] = mkc(0.0, 0.0);
      for (int j = 0; j < ct.contour_points; ++j) {
        const z64 nd = contour_node(ct.contour_points, ct.contour_radius, j);
        frac_contour_add(fnum, fden, fmask, mkc(z.re + nd.re, z.im + nd.im), acc);
      }
      for (int r = 1; r <= 3; ++r) {
        const z64 a = r == 1 ? acc[1] : (r == 2 ? acc[2] : acc[3]);
        const z64 b = np_rdiv(np_rmul(h, a), (double)ct.contour_points);
        if (r == 1) v[1] = b;
        else if (r == 2) v[2] = b;
        else v[3] = b;
      }
    }
    frac_coefs<RS, RN>(tb, f, v, h, cplx, mS, (size_t)M, cbase);
  }
}

template <typename RS, typename RN>
__device__ __forceinline__ void coef_mode(const rks_tableau& tb, const rks_ctrl& ct, const double* __restrict__ L,
                                          int L_complex, int m, int M, double h, char* __restrict__ cbase) {
  coef_mode_at<RS, RN>(tb, ct, L, L_complex, m, m, M, h, cbase);
}

// Coefficients of the listed small modes (|z| < modecutoff): groups of up to
// 32 lanes per mode, one lane per contour node, deterministic shuffle sums.
// All T threads of the workgroup call this with the same list.
template <typename RS, typename RN, int T, typename TB, typename CT>
__device__ __forceinline__ void coef_small_group(TB& tb, CT& ct, const double* __restrict__ L, int L_complex,
                                                 int M, double h, char* __restrict__ cbase, const int* list,
                                                 int nsmall) {
#pragma clang fp contract(off)
  const int t = threadIdx.x;
  const int cplx = L_complex || tb.uses_contour;
  if (nsmall > 0) {
    constexpr int GS = T < 32 ? T : 32;
    constexpr int NG = T / GS;
    const int g = t / GS, lane = t % GS;
    for (int base = 0; base < nsmall; base += NG) {
      const int idx = base + g;
      if (idx < nsmall) {
        const int m = list[idx];
        const z64 z = mode_z(L, L_complex, m, h);
        for (int f = 0; f < tb.nfrac; ++f) {
          const int fnum = tb.frac[f].fnum, fden = tb.frac[f].fden, fmask = tb.frac[f].mask;
          z64 v[4];
          v[1] = v[2] = v[3] = mkc(0.0, 0.0);
          if (fmask & 14) {
            z64 acc[4];
            acc[1] = acc[2] = acc[3] = mkc(0.0, 0.0);
            for (int j = lane; j < ct.contour_points; j += GS) {
              const z64 nd = contour_node(ct.contour_points, ct.contour_radius, j);
              frac_contour_add(fnum, fden, fmask, mkc(z.re + nd.re, z.im + nd.im), acc);
            }
#pragma unroll
            for (int o = GS / 2; o >= 1; o >>= 1) {
#pragma unroll
              for (int r = 1; r <= 3; ++r) {
                acc[r].re += __shfl_xor(acc[r].re, o, 64);
                acc[r].im += __shfl_xor(acc[r].im, o, 64);
              }
            }
            v[1] = np_rdiv(np_rmul(h, acc[1]), (double)ct.contour_points);
            v[2] = np_rdiv(np_rmul(h, acc[2]), (double)ct.contour_points);
            v[3] = np_rdiv(np_rmul(h, acc[3]), (double)ct.contour_points);
          }
          if (lane == 0) {
            v[0] = np_exp(frac_arg(z, fnum, fden, cplx));
            frac_coefs<RS, RN>(tb, f, v, h, cplx, m, (size_t)M, cbase);
          }
        }
      }
    }
  }
}

// All coefficients of an instance by one workgroup: closed forms per thread,
// then the small modes' contour means spread over groups of up to 32 lanes
// (one lane per node, deterministic shuffle reduction).  Modes 0..Mg-1 are
// generated into arrays of stride M.  `list` is LDS scratch for up to Mg
// ints; *count is an LDS counter.
template <typename RS, typename RN, int T, int MPT>
__device__ __attribute__((noinline)) void coef_update(const rks_tableau& tb_in, const rks_ctrl& ct_in,
                                                      const double* __restrict__ L, int L_complex, int M, int Mg,
                                                      double h, char* __restrict__ cbase, int* list, int* count) {
#pragma clang fp contract(off)
  rks_ctab& tb = *rks_uniform_const<rks_ctab>(&tb_in);
  rks_cctl& ct = *rks_uniform_const<rks_cctl>(&ct_in);
  const int t = threadIdx.x;
  const int cplx = L_complex || tb.uses_contour;
  if (t == 0) *count = 0;
  __syncthreads();
  for (int i = 0; i < MPT; ++i) {
    const int m = t + i * T;
    if (m >= Mg) break;
    const z64 z = mode_z(L, L_complex, m, h);
    if (tb.uses_contour && hypot(z.re, z.im) < ct.modecutoff) {
      list[atomicAdd(count, 1)] = m;
      continue;
    }
    for (int f = 0; f < tb.nfrac; ++f) {
      z64 v[4];
      v[1] = v[2] = v[3] = mkc(0.0, 0.0);
      frac_direct(tb.frac[f].fnum, tb.frac[f].fden, tb.frac[f].mask, z, h, cplx, v);
      frac_coefs<RS, RN>(tb, f, v, h, cplx, m, (size_t)M, cbase);
    }
  }
  __syncthreads();
  coef_small_group<RS, RN, T>(tb, ct, L, L_complex, M, h, cbase, list, *count);
  __syncthreads();
}

// All fractions of one method's tableau for one mode: recipe constants as literals.
// v: the basis values of fraction F, by get(F, v)
template <typename TT, int F, typename RS, typename RN, typename Get>
__device__ __forceinline__ void method_fracs(Get get, double h, int m, size_t M, char* __restrict__ cbase) {
  if constexpr (F < TT::tab.nfrac) {
    z64 v[4];
    v[1] = v[2] = v[3] = mkc(0.0, 0.0);
    get(TT::tab.frac[F].fnum, TT::tab.frac[F].fden, TT::tab.frac[F].mask, v);
    coef_recipes<TT, F, RS, RN>(v, h, m, M, cbase, std::make_integer_sequence<int, TT::tab.ncoef>{});
    method_fracs<TT, F + 1, RS, RN>(get, h, m, M, cbase);
  }
}

// One small mode's contour means by GS lanes, one node each: summed by a butterfly, or
// (ORDERED) node by node in the order in which one thread sums them.
template <typename TT, int F, typename RS, typename RN, int GS, bool ORDERED, typename CT>
__device__ __forceinline__ void method_small(CT& ct, z64 z, int lane, double h, int m, size_t M,
                                             char* __restrict__ cbase) {
  if constexpr (F < TT::tab.nfrac) {
#pragma clang fp contract(off)
    constexpr int fnum = TT::tab.frac[F].fnum, fden = TT::tab.frac[F].fden, fmask = TT::tab.frac[F].mask;
    z64 v[4];
    v[1] = v[2] = v[3] = mkc(0.0, 0.0);
    if constexpr ((fmask & 14) != 0) {
      z64 acc[4];
      acc[1] = acc[2] = acc[3] = mkc(0.0, 0.0);
      if constexpr (ORDERED) {
        const int np = ct.contour_points;
        for (int j0 = 0; j0 < np; j0 += GS) {
          z64 p[4];
          p[1] = p[2] = p[3] = mkc(0.0, 0.0);
          const z64 nd = contour_node(np, ct.contour_radius, j0 + lane < np ? j0 + lane : 0);
          frac_contour_add(fnum, fden, fmask, mkc(z.re + nd.re, z.im + nd.im), p);
          for (int j = 0; j < GS && j0 + j < np; ++j) {
#pragma unroll
            for (int r = 1; r <= 3; ++r) {
              acc[r].re += __shfl(p[r].re, j, GS);
              acc[r].im += __shfl(p[r].im, j, GS);
            }
          }
        }
      } else {
        for (int j = lane; j < ct.contour_points; j += GS) {
          const z64 nd = contour_node(ct.contour_points, ct.contour_radius, j);
          frac_contour_add(fnum, fden, fmask, mkc(z.re + nd.re, z.im + nd.im), acc);
        }
#pragma unroll
        for (int o = GS / 2; o >= 1; o >>= 1) {
#pragma unroll
          for (int r = 1; r <= 3; ++r) {
            acc[r].re += __shfl_xor(acc[r].re, o, 64);
            acc[r].im += __shfl_xor(acc[r].im, o, 64);
          }
        }
      }
#pragma unroll
      for (int r = 1; r <= 3; ++r) v[r] = np_rdiv(np_rmul(h, acc[r]), (double)ct.contour_points);
    }
    if (lane == 0) {
      v[0] = np_exp(frac_arg(z, fnum, fden, 1));
      coef_recipes<TT, F, RS, RN>(v, h, m, M, cbase, std::make_integer_sequence<int, TT::tab.ncoef>{});
    }
    method_small<TT, F + 1, RS, RN, GS, ORDERED>(ct, z, lane, h, m, M, cbase);
  }
}

// coef_update of one method.  The generator was bound by the tableau it walked: per mode,
// every fraction searched the whole coefficient list and divided by run-time constants.
// Whether L is complex is a literal (LC): the host picks these kernels only for plans whose
// lin_ops are all of that kind.
template <typename TT, typename RS, typename RN, int T, int MPT>
__device__ __attribute__((noinline)) void coef_update_method(const rks_ctrl& ct_in, const double* __restrict__ L,
                                                             int M, int Mg, double h, char* __restrict__ cbase,
                                                             int* list, int* count) {
#pragma clang fp contract(off)
  rks_cctl& ct = *rks_uniform_const<rks_cctl>(&ct_in);
  constexpr int LC = TT::tab.coef_rs[0] == RKS_CST_RS || TT::tab.coef_rs[0] == RKS_CST_RN;
  constexpr int cplx = LC || TT::tab.uses_contour;
  const int t = threadIdx.x;
  if (TT::tab.uses_contour) {
    if (t == 0) *count = 0;
    __syncthreads();
  }
#pragma unroll 1
  for (int i = 0; i < MPT; ++i) {
    const int m = t + i * T;
    if (m >= Mg) break;
    const z64 z = mode_z(L, LC, m, h);
    if (TT::tab.uses_contour && hypot(z.re, z.im) < ct.modecutoff) {
      list[atomicAdd(count, 1)] = m;
      continue;
    }
    method_fracs<TT, 0, RS, RN>(
        [&](int fnum, int fden, int fmask, z64(&v)[4]) { frac_direct(fnum, fden, fmask, z, h, cplx, v); }, h, m,
        (size_t)M, cbase);
  }
  if constexpr (TT::tab.uses_contour != 0) {
    __syncthreads();
    const int nsmall = *count;
    constexpr int GS = T < 32 ? T : 32;
    const int g = t / GS, lane = t % GS;
    for (int idx = g; idx < nsmall; idx += T / GS) {
      const int m = list[idx];
      method_small<TT, 0, RS, RN, GS, false>(ct, mode_z(L, LC, m, h), lane, h, m, (size_t)M, cbase);
    }
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------
// Stage combinations and the error estimate, chunked and term-major: CH modes
// of one thread at once (a ChunkIdx: m0 + i*T), so every term issues CH independent loads.  Arithmetic is in the state precision RS; NL arrays and the non-
// propagator coefficients may be stored in RN (converted on load).
//   term (rks_term grouping):  inner = NL[src] + scale2 * NL[src2]
//     hmode 0: scale * (C * inner)   1: ((h * C) * inner) * scale   2: ((scale*h)/den) * inner
// Every decision that depends on the tableau is uniform and taken once per
// term, and modes past the end load index 0 (always in bounds) instead of
// branching, so a chunk's loads are straight-line code and issue back to
// back; callers discard the lanes with ok[i] false.
//
// Mirror pairs (sym): slots 2j and 2j+1 hold a mode and its mirror (2-D: rows
// q and n - q of one column; q = 0 pairs with n/2), and
// the linear operator is mirror-symmetric, so both have the same
// coefficients.  Coefficients are stored for the modes below `lim` only
// (rows 0..n/2); an odd slot at or past lim reads its even
// slot's coefficient, one below lim (the n/2 partner of q = 0) its own.
// anyq = 0: only slot 1 can hold such a partner.
// ---------------------------------------------------------------------------
template <int CH>
struct ChunkIdx {
  int m[CH];
  bool ok[CH];
  int sym;   // slots are mirror pairs sharing coefficients
  int lim;   // first mode without stored coefficients (sym only)
  int anyq;  // any odd slot may lie below lim (else only slot 1)
  __device__ __forceinline__ ChunkIdx() {}
  __device__ __forceinline__ ChunkIdx(int m0, int T, int mlim) : sym(0), lim(0), anyq(0) {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int x = m0 + i * T;
      ok[i] = x < mlim;
      m[i] = ok[i] ? x : 0;
    }
  }
};

// Mode ownership in the persistent kernel: thread t holds the modes m = t + k T, the
// elements that its first and last transform butterflies hold (rks_fft.h chain_reg), so
// stage values, NL values and the state pass between the stage sums and the transforms
// in registers.  rfft layout: slots k < N / (2T), and slot N / (2T) is the n/2 mode of
// thread 0.  Every M-sized array is read and written through this map, so each element a
// stage pass produces is consumed by the same thread.
template <int N, int M, int T, int NLK>
struct Own {
  static constexpr int MPT = (M + T - 1) / T;
  static constexpr bool RFFT = M == N / 2 + 1;
  int lim;   // modes below it (the Hankel kind's radial points; every mode otherwise)
  int fold;  // mirror-symmetric lin_op: N (coefficients of modes 0..N/2 only), else 0
  int t;     // the thread
  __device__ __forceinline__ int raw(int k) const { return t + k * T; }
  // The same map behind an opaque copy of the thread index: addresses derived from it are
  // formed where they are used.  Otherwise the compiler hoists every slot's offset out of
  // the stage loop and holds them (up to 48 registers) through the transforms.
  __device__ __forceinline__ Own fresh() const {
    Own o = *this;
    asm volatile("" : "+v"(o.t));
    return o;
  }
  __device__ __forceinline__ bool ok(int k) const {
    if (M % T == 0 && NLK != NLK_HANKEL) return true;
    if (RFFT && M == (MPT - 1) * T + 1 && k < MPT - 1) return true;
    return raw(k) < lim;
  }
  // always in bounds: a slot without a mode reads one of the thread's (or mode 0)
  __device__ __forceinline__ int m(int k) const { return ok(k) ? raw(k) : 0; }
  __device__ __forceinline__ int c(int k) const {
    const int x = m(k);
    return (fold && x > N / 2) ? N - x : x;
  }
};

// Modes of the general kernel's stage passes, chunk c.  fft layout: the mirror pairs q = t + jT
// (slot 2j) and N - q (slot 2j + 1; N/2 for q = 0), as in the norm (NormOrder), so a pair shares
// one load of each coefficient of a mirror-symmetric L; by the thread's own modes every mode
// loads its own.  One FP32 evolve, n = 8192, own modes / pairs: ETD34 1.31 / 1.20 ms, ETD5 5.01 /
// 4.35, IF45DP 288 / 245; n = 4096 1.11 / 1.04, 3.63 / 3.28, 205 / 183.  Else the thread's own
// modes.
template <int N, int M, int T, int NLK, int CH>
__device__ __forceinline__ ChunkIdx<CH> pass_chunk(int c, const Own<N, M, T, NLK>& ow) {
  ChunkIdx<CH> ix;
  ix.anyq = 0;
  if constexpr (M == N && NLK != NLK_HANKEL) {
    static_assert(CH % 2 == 0 && N % (2 * T) == 0, "whole mirror pairs per chunk");
    ix.sym = ow.fold != 0;
    ix.lim = N / 2 + 1;
#pragma unroll
    for (int j = 0; j < CH / 2; ++j) {
      const int q = ow.t + (c * (CH / 2) + j) * T;
      ix.m[2 * j] = q;
      ix.m[2 * j + 1] = q == 0 ? N / 2 : N - q;
      ix.ok[2 * j] = ix.ok[2 * j + 1] = true;
    }
  } else {
    ix.sym = 0;
    ix.lim = 0;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int x = ow.t + (c * CH + i) * T;
      ix.ok[i] = x < ow.lim;
      ix.m[i] = ix.ok[i] ? x : 0;
    }
  }
  return ix;
}

// The order of the error norm's sums, mode(k) of slot k: fft layout, thread t adds the mirror
// pairs q = t + jT (slot 2j) and N - q (slot 2j + 1; N/2 for q = 0), else its own modes.  One
// order for all kernels of a size: s in its last bits reaches h, in MIXED a changed h rounds
// the FP32 coefficients anew (~1e-9 of the state), and unresolved runs amplify any change.
// The Hankel kind's sums run over the lanes of NT threads (t + k NT), whatever T is.
template <int N, int M, int T, int NLK>
struct NormOrder {
  static constexpr int NT = NLK == NLK_HANKEL ? (N / 4 < 64 ? 64 : (N / 4 > 256 ? 256 : N / 4)) : T;
  static constexpr int SLOTS = (M + NT - 1) / NT;
  static constexpr bool OWN = !(M == N && (NLK != NLK_HANKEL || NT != T));  // the thread's own modes in order
  static __device__ __forceinline__ int mode(int k) {
    const int t = threadIdx.x;
    if constexpr (M == N && NLK != NLK_HANKEL) {
      const int q = t + (k >> 1) * T;
      return (k & 1) == 0 ? q : (q == 0 ? N / 2 : N - q);
    } else {
      return t + k * NT;
    }
  }
  static __device__ __forceinline__ bool ok(int k, int lim) { return (int)threadIdx.x < NT && mode(k) < lim; }
};

// How a pass reads its arrays.  Through the scalar view of the tableau (rks_ctab: the general
// passes below) the array's base is uniform, kept in scalar registers and indexed by 32 bits;
// with a plain tableau an array is read as the pointer stands.
template <typename TB>
struct ViewOf {
  static constexpr bool SCALAR = false;
};
template <>
struct ViewOf<rks_ctab> {
  static constexpr bool SCALAR = true;
};
template <bool SCALAR, typename P>
__device__ __forceinline__ P* view(P* p) {
  if constexpr (SCALAR) return uni(p);
  else return p;
}
template <bool SCALAR, typename R>
__device__ __forceinline__ cx<R> vload(const cx<R>* p, int i) {
  if constexpr (SCALAR) return gload(p, i);
  else return p[i];
}
template <bool SCALAR, typename R>
__device__ __forceinline__ R vload_real(const R* p, int i) {
  if constexpr (SCALAR) return gload_real(p, i);
  else return p[i];
}

// coefficient array c of the chunk's modes; M is the array stride (modes)
template <typename RS, typename RN, int CH, typename TB>
__device__ __forceinline__ void load_coef(TB& tb, const char* cbase, size_t M, int c,
                                          const ChunkIdx<CH>& ix, cx<RS> (&w)[CH]) {
  constexpr bool SC = ViewOf<TB>::SCALAR;
  const char* q = view<SC>(cbase + (size_t)tb.coef_off[c] * M);
  const int kind = tb.coef_rs[c];
  // Mirror pairs: FP32-state kernels issue one load per pair (plus the n/2
  // partner of q = 0).  The FP64-state kernels have no registers to spare
  // for that second code path, so their odd slot repeats the even slot's
  // address and the caches serve the repeat.
  int ci[CH];
#pragma unroll
  for (int i = 0; i < CH; ++i) ci[i] = ix.m[i];
  if constexpr (CH % 2 == 0 && sizeof(RS) > 4) {
#pragma unroll
    for (int j = 0; j < CH / 2; ++j)
      if (ix.sym) ci[2 * j + 1] = (ix.m[2 * j + 1] < ix.lim) ? ix.m[2 * j + 1] : ix.m[2 * j];
  }
  auto gather = [&](auto ld) {
    if constexpr (CH % 2 == 0 && sizeof(RS) == 4) {
      if (ix.sym) {
#pragma unroll
        for (int j = 0; j < CH / 2; ++j) {
          w[2 * j] = ld(ix.m[2 * j]);
          w[2 * j + 1] = w[2 * j];
        }
        if (ix.anyq) {
#pragma unroll
          for (int j = 0; j < CH / 2; ++j)
            if (ix.m[2 * j + 1] < ix.lim) w[2 * j + 1] = ld(ix.m[2 * j + 1]);
        } else if (ix.m[1] < ix.lim) {
          w[1] = ld(ix.m[1]);
        }
        return;
      }
    }
#pragma unroll
    for (int i = 0; i < CH; ++i) w[i] = ld(ci[i]);
  };
  if (kind == RKS_CST_RS) {
    const cx<RS>* p = (const cx<RS>*)q;
    gather([&](int m) { return vload<SC>(p, m); });
  } else if (kind == RKS_CST_RN) {
    const cx<RN>* p = (const cx<RN>*)q;
    gather([&](int m) { return cvt<RS>(vload<SC>(p, m)); });
  } else if (kind == RKS_CST_RS_REAL) {
    const RS* p = (const RS*)q;
    gather([&](int m) { return mkc(vload_real<SC>(p, m), (RS)0); });
  } else {
    const RN* p = (const RN*)q;
    gather([&](int m) { return mkc((RS)vload_real<SC>(p, m), (RS)0); });
  }
}

// slotp(s): NL array of slot s (const cx<RN>*)
template <typename RS, typename RN, int CH, bool HSUM, typename TB, typename TM, typename SlotF>
__device__ __forceinline__ void add_terms(TB& tb, TM* terms, int nterm, SlotF slotp,
                                          const char* cbase, size_t M, const ChunkIdx<CH>& ix, double h,
                                          cx<RS> (&acc)[CH]) {
  using C = cx<RS>;
  constexpr bool SC = ViewOf<TB>::SCALAR;
  for (int j = 0; j < nterm; ++j) {
    auto& tm = terms[j];
    const cx<RN>* nl = view<SC>(slotp(tm.src));
    C v[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) v[i] = cvt<RS>(vload<SC>(nl, ix.m[i]));
    if (tm.src2 >= 0) {
      const cx<RN>* nl2 = view<SC>(slotp(tm.src2));
      const RS s2 = (RS)tm.scale2;
#pragma unroll
      for (int i = 0; i < CH; ++i) v[i] = v[i] + s2 * cvt<RS>(vload<SC>(nl2, ix.m[i]));
    }
    if (tm.hmode == 2) {
      const RS hs = (RS)((tm.scale * h) / tm.den);
#pragma unroll
      for (int i = 0; i < CH; ++i) v[i] = hs * v[i];
    } else {
      const RS hr = (RS)h;
      if (tm.coef >= 0) {
        C w[CH];
        load_coef<RS, RN, CH>(tb, cbase, M, tm.coef, ix, w);
        if (tm.hmode == 1) {
#pragma unroll
          for (int i = 0; i < CH; ++i) v[i] = (hr * w[i]) * v[i];
        } else {
#pragma unroll
          for (int i = 0; i < CH; ++i) v[i] = w[i] * v[i];
        }
      } else if (tm.hmode == 1) {
#pragma unroll
        for (int i = 0; i < CH; ++i) v[i] = hr * v[i];
      }
      if (tm.scale != 1.0) {
        const RS sc = (RS)tm.scale;
#pragma unroll
        for (int i = 0; i < CH; ++i) v[i] = sc * v[i];
      }
    }
#pragma unroll
    for (int i = 0; i < CH; ++i) acc[i] = (HSUM && j == 0) ? v[i] : acc[i] + v[i];
  }
}

// k = E u + terms, or E u + h * sum(terms) for stages that factor h out (if34.py:126-128);
// lanes past mlim come back zero
template <typename RS, typename RN, int CH, typename TB, typename ST, typename SlotF>
__device__ __forceinline__ void stage_chunk(TB& tb, ST& S, const cx<RS>* __restrict__ u,
                                            SlotF slotp, const char* cbase, size_t M, const ChunkIdx<CH>& ix,
                                            double h, cx<RS> (&acc)[CH]) {
  using C = cx<RS>;
  constexpr bool SC = ViewOf<TB>::SCALAR;
#pragma unroll
  for (int i = 0; i < CH; ++i) acc[i] = vload<SC>(u, ix.m[i]);
  if (S.ecoef >= 0) {
    C e[CH];
    load_coef<RS, RN, CH>(tb, cbase, M, S.ecoef, ix, e);
#pragma unroll
    for (int i = 0; i < CH; ++i) acc[i] = e[i] * acc[i];
  }
  if (S.hsum) {
    C sum[CH];
    add_terms<RS, RN, CH, true>(tb, S.t, S.nterm, slotp, cbase, M, ix, h, sum);
#pragma unroll
    for (int i = 0; i < CH; ++i) acc[i] = acc[i] + (RS)h * sum[i];
  } else {
    add_terms<RS, RN, CH, false>(tb, S.t, S.nterm, slotp, cbase, M, ix, h, acc);
  }
#pragma unroll
  for (int i = 0; i < CH; ++i)
    if (!ix.ok[i]) acc[i] = mkc((RS)0, (RS)0);
}

// modes m0 + i*T below mlim
template <typename RS, typename RN, int CH, typename TB, typename ST, typename SlotF>
__device__ __forceinline__ void stage_chunk(TB& tb, ST& S, const cx<RS>* __restrict__ u,
                                            SlotF slotp, const char* cbase, size_t M, int m0, int T, int mlim,
                                            double h, cx<RS> (&acc)[CH]) {
  stage_chunk<RS, RN, CH>(tb, S, u, slotp, cbase, M, ChunkIdx<CH>(m0, T, mlim), h, acc);
}

// embedded error estimate (etd35.py:344, etd34.py:190, if34.py:130, if45dp.py:170-177)
template <typename RS, typename RN, int CH, typename TB, typename SlotF>
__device__ __forceinline__ void error_chunk(TB& tb, SlotF slotp, const char* cbase, size_t M,
                                            const ChunkIdx<CH>& ix, double h, cx<RS> (&ev)[CH]) {
  add_terms<RS, RN, CH, true>(tb, tb.err, tb.nerr, slotp, cbase, M, ix, h, ev);
  if (tb.err_factored) {
    if (tb.err_hpow) {
#pragma unroll
      for (int i = 0; i < CH; ++i) ev[i] = (RS)h * ev[i];
    }
    if (tb.err_scale != 1.0) {
#pragma unroll
      for (int i = 0; i < CH; ++i) ev[i] = (RS)tb.err_scale * ev[i];
    }
    if (tb.err_coef >= 0) {
      cx<RS> w[CH];
      load_coef<RS, RN, CH>(tb, cbase, M, tb.err_coef, ix, w);
#pragma unroll
      for (int i = 0; i < CH; ++i) ev[i] = w[i] * ev[i];
    }
  }
#pragma unroll
  for (int i = 0; i < CH; ++i)
    if (!ix.ok[i]) ev[i] = mkc((RS)0, (RS)0);
}

template <typename RS, typename RN, int CH, typename TB, typename SlotF>
__device__ __forceinline__ void error_chunk(TB& tb, SlotF slotp, const char* cbase, size_t M, int m0,
                                            int T, int mlim, double h, cx<RS> (&ev)[CH]) {
  error_chunk<RS, RN, CH>(tb, slotp, cbase, M, ChunkIdx<CH>(m0, T, mlim), h, ev);
}

// The last stage and the embedded error read the same NL slots in the same
// order with scalar error weights (ETD35: k = E u + sum c_j NL_j,
// err = a75 (-NL1 + 4 NL3 - 6 NL4 + 4 NL5 - NL6), etd35.py:340-344): one pass
// forms both from a single load of each NL value.  Arithmetic per quantity is
// that of stage_chunk / error_chunk.
__host__ __device__ __forceinline__ bool rks_fused_final(const rks_tableau& tb) {
  if (!tb.adaptive || !tb.err_factored) return false;
  const rks_stage& S = tb.st[tb.nstage - 1];
  if (S.has_nl || S.hsum || S.nterm != tb.nerr) return false;
  for (int j = 0; j < tb.nerr; ++j) {
    const rks_term &a = S.t[j], &e = tb.err[j];
    if (a.src != e.src || a.src2 >= 0 || e.src2 >= 0 || e.coef >= 0 || a.hmode != 0 || e.hmode != 0) return false;
  }
  return true;
}

template <typename RS, typename RN, int CH, typename TB, typename SlotF>
__device__ __forceinline__ void final_chunk(TB& tb, const cx<RS>* __restrict__ u, SlotF slotp,
                                            const char* cbase, size_t M, const ChunkIdx<CH>& ix, double h,
                                            cx<RS> (&acc)[CH], cx<RS> (&ev)[CH]) {
  using C = cx<RS>;
  constexpr bool SC = ViewOf<TB>::SCALAR;
  auto& S = tb.st[tb.nstage - 1];
#pragma unroll
  for (int i = 0; i < CH; ++i) acc[i] = vload<SC>(u, ix.m[i]);
  if (S.ecoef >= 0) {
    C e[CH];
    load_coef<RS, RN, CH>(tb, cbase, M, S.ecoef, ix, e);
#pragma unroll
    for (int i = 0; i < CH; ++i) acc[i] = e[i] * acc[i];
  }
  for (int j = 0; j < S.nterm; ++j) {
    auto& tm = S.t[j];
    const cx<RN>* nl = view<SC>(slotp(tm.src));
    C v[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) v[i] = cvt<RS>(vload<SC>(nl, ix.m[i]));
    {
      C c[CH];
      if (tm.coef >= 0) {
        load_coef<RS, RN, CH>(tb, cbase, M, tm.coef, ix, c);
#pragma unroll
        for (int i = 0; i < CH; ++i) c[i] = c[i] * v[i];
      } else {
#pragma unroll
        for (int i = 0; i < CH; ++i) c[i] = v[i];
      }
      if (tm.scale != 1.0) {
        const RS sc = (RS)tm.scale;
#pragma unroll
        for (int i = 0; i < CH; ++i) c[i] = sc * c[i];
      }
#pragma unroll
      for (int i = 0; i < CH; ++i) acc[i] = acc[i] + c[i];
    }
    const double es = tb.err[j].scale;
    if (es != 1.0) {
      const RS se = (RS)es;
#pragma unroll
      for (int i = 0; i < CH; ++i) v[i] = se * v[i];
    }
#pragma unroll
    for (int i = 0; i < CH; ++i) ev[i] = (j == 0) ? v[i] : ev[i] + v[i];
  }
  if (tb.err_hpow) {
#pragma unroll
    for (int i = 0; i < CH; ++i) ev[i] = (RS)h * ev[i];
  }
  if (tb.err_scale != 1.0) {
#pragma unroll
    for (int i = 0; i < CH; ++i) ev[i] = (RS)tb.err_scale * ev[i];
  }
  if (tb.err_coef >= 0) {
    C w[CH];
    load_coef<RS, RN, CH>(tb, cbase, M, tb.err_coef, ix, w);
#pragma unroll
    for (int i = 0; i < CH; ++i) ev[i] = w[i] * ev[i];
  }
}

// ---------------------------------------------------------------------------
// nonlinear term.  The spectrum is in registers, slot k of thread t holding mode
// t + kT (Own), and the NL values come back in the same slots: the transforms take
// their inputs from and leave their results in registers (fft_reg), and the
// pointwise products are formed between them without a trip through LDS.  A cubic
// n = 8192 evaluation (radix 16, 16, 16, 2) makes 6 exchanges; filling the buffer,
// two LDS-to-LDS transforms and the product between them made 8 and a third more
// barriers.  Called by all threads; the LDS buffers are free at the call and at the
// return.
// ---------------------------------------------------------------------------
// Modes per chunk of the stage passes of the general kernels.  Eight FP64 modes take all the
// registers of general_pass and leave nothing to overlap a chunk's loads with; four are faster
// (eight / four, FP64: ETD34 n = 8192 1.63 / 1.27 ms, ETD5 n = 4096 3.75 / 3.22) except in a
// one-wave workgroup, where a term costs its latency whatever the chunk holds (MIXED n = 1024,
// IF45DP: 157 / 172 ms).
template <int MPT, int ES, int T>
struct Chunk {
  static constexpr int MAX = ES > 8 && MPT >= 8 && T > 64 ? 4 : 8;
  static constexpr int CH = MPT < MAX ? MPT : MAX;
  static constexpr int NCH = (MPT + CH - 1) / CH;
};

// exchange buffers must leave room for the twiddle tables and the reduction scratch (160 KB per CU)
#define RKS_LDS_MAX (148 * 1024)

// Two exchange buffers where they fit beside the register-bound number of waves: a
// workgroup takes at most 512 threads x 16 elements x 8 bytes (padded, 70 KB) per
// buffer then, and a one-wave workgroup has no barriers to save.
template <typename R, int LOG2N, int T, int NLK>
__host__ __device__ constexpr bool rks_two_buffers() {
  return NLK != NLK_HANKEL && T > 64 && ((1 << LOG2N) / T) * (int)sizeof(cx<R>) <= 128 &&
         2 * rksfft::padded_size(1 << LOG2N) * (int)sizeof(cx<R>) <= RKS_LDS_MAX;
}

// LDS elements of the exchange buffers
template <typename R, int LOG2N, int T, int NLK>
__host__ __device__ constexpr int rks_buf_elems() {
  return rksfft::padded_size(1 << LOG2N) * (rks_two_buffers<R, LOG2N, T, NLK>() ? 2 : 1);
}

// LDS bytes of the persistent kernel: exchange buffers + twiddle tables (Hankel:
// the stage values and the |f|^2 f vector)
template <typename R, int LOG2N, int T, int NLK>
__host__ __device__ constexpr int rks_lds_bytes() {
  return (rks_buf_elems<R, LOG2N, T, NLK>() + (NLK == NLK_HANKEL ? (1 << LOG2N) : rksfft::TwSplit<LOG2N>::SIZE)) *
         (int)sizeof(cx<R>);
}

// Hankel kind: yt = Y transposed (nr x nr, engine precision), hs = S.  A thread forms whole
// rows of both products, summing over the columns in order with FMAs.  Column k of Y is a row
// of yt, so a wave reads it as one run of memory (row by row of Y, every lane would touch a
// line of its own), and the vector comes from LDS as broadcasts: the products are bound by
// the 8 nr^2 bytes of yt per product that each trajectory streams from L2 (80 KB at nr = 100,
// beyond the L1), with a thread per row so that all of a row's latency is spent once.  1024
// beams, nr = 100, ETD35 FP64, one evolve: 21.2 ms row by row with n/4 threads, 8.6 ms.
// Values as the batched transform's (rks_hankel.hip): f = (1/S) sum, |f|^2 f, then
// i gamma (S sum).  Batches of 10 columns: 16 (7.6 -> 8.9 ms) and 32 (9.6) were slower, also
// with the next batch prefetched (9.6).
template <typename R, int LOG2N, int T, int MPT>
__device__ __forceinline__ void hankel_rows(cx<R> (&v)[MPT], const cx<R>* x, const R* __restrict__ yt, int nr) {
#pragma unroll
  for (int i = 0; i < MPT; ++i) {
    const int r = (int)threadIdx.x + i * T;
    const R* col = yt;
    const int rr = r < nr ? r : 0;
    R ar = (R)0, ai = (R)0;
    int k = 0;
    constexpr int U = 10;
    for (; k + U <= nr; k += U, col += U * nr) {
      R y[U];
#pragma unroll
      for (int j = 0; j < U; ++j) y[j] = gload_real(col, rr + j * nr);
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const cx<R> q = x[k + j];
        ar = fma(y[j], q.re, ar);
        ai = fma(y[j], q.im, ai);
      }
    }
    for (; k < nr; ++k, col += nr) {
      const R y = gload_real(col, rr);
      const cx<R> q = x[k];
      ar = fma(y, q.re, ar);
      ai = fma(y, q.im, ai);
    }
    v[i] = mkc(ar, ai);
  }
}

template <typename R, int LOG2N, int T, int MPT>
__device__ __forceinline__ void nl_hankel(cx<R> (&v)[MPT], cx<R>* buf, R coef, const R* __restrict__ yt, int nr,
                                          double hs) {
#pragma clang fp contract(off)
  using C = cx<R>;
  const int t = threadIdx.x;
  C* w = buf + rksfft::padded_size(1 << LOG2N);
  const R ci = (R)(1.0 / hs), cs = (R)hs;
#pragma unroll
  for (int i = 0; i < MPT; ++i)
    if (t + i * T < nr) buf[t + i * T] = v[i];
  __syncthreads();
  hankel_rows<R, LOG2N, T, MPT>(v, buf, yt, nr);
#pragma unroll
  for (int i = 0; i < MPT; ++i) {
    const R vr = ci * v[i].re, vi = ci * v[i].im;
    const R m2 = fma(vi, vi, vr * vr);
    if (t + i * T < nr) w[t + i * T] = mkc(vr * m2, vi * m2);
  }
  __syncthreads();
  hankel_rows<R, LOG2N, T, MPT>(v, w, yt, nr);
#pragma unroll
  for (int i = 0; i < MPT; ++i) {
    const R vr = cs * v[i].re, vi = cs * v[i].im;
    v[i] = mkc(-coef * vi, coef * vr);
  }
  // w is next written after the barrier that follows the next fill of buf
}

// Slots whose imaginary parts of U + iV take the product unrounded: those whose products the
// compiler fused in the earlier kernels, which transformed from LDS to LDS.  Nothing in the
// mathematics sets these slots apart; they keep the results of runs that no rounding is small
// for.  On a spectrum that reaches the grid's end k U outweighs U a thousandfold and a run that
// is not resolved amplifies the last bit: with one rule for all slots Burgers (viscosity 5e-4, n =
// 4096 and 8192) moves by 2e-4 to 7e-3 of the state, its distance from 64-bit results 1e-4 to
// 8e-3, and with every product fused an FP32 KS ensemble by 3e-6.  Damped FP64 runs move by
// rounding only, whichever rule.
template <int T>
__device__ __forceinline__ constexpr bool fused_imag(int k) {
  return k >= 1 && k <= (T == 512 ? 6 : T == 256 ? 4 : 0);
}

template <typename R, int LOG2N, int T, int NLK, int MPT>
__device__ __forceinline__ void nl_regs(cx<R> (&v)[MPT], cx<R>* buf, const cx<R>* twl, R coef,
                                        const R* __restrict__ kx, int nr, double hs) {
  using C = cx<R>;
  using rksfft::pad;
  constexpr int N = 1 << LOG2N;
  constexpr bool PP = rks_two_buffers<R, LOG2N, T, NLK>();
  constexpr int PS = rksfft::padded_size(N);
  // An opaque copy of the thread index, as in Own::fresh: the transforms' LDS addresses are
  // formed here, at each call.  Hoisted out of the stage loop they were held (and spilled)
  // through it: 448 bytes of scratch per lane at n = 8192 (advective IF34 FP64), now 128, and
  // a step 122 -> 112 us; 640 -> 80 in FP32, the KS ensemble (2048) 23.8 -> 22.5 ms.
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  const R inv = (R)1 / (R)N;
  if constexpr (NLK == NLK_HANKEL) {
    nl_hankel<R, LOG2N, T, MPT>(v, buf, coef, kx, nr, hs);
  } else if constexpr (NLK == NLK_CUBIC) {
    constexpr int X = rksfft::exchanges<N, T, RKS_MAXR>();
    rksfft::fft_reg<R, N, T, true, LOG2N, RKS_MAXR, PP, 0, true>(v, buf, twl, t, [&](C w) {
      const C v1 = inv * w;
      const R a = v1.re * v1.re + v1.im * v1.im;
      return a * v1;
    });
    rksfft::fft_reg<R, N, T, false, LOG2N, RKS_MAXR, PP, X & 1, false>(
        v, buf, twl, t, [&](C w) { return mkc(-coef * w.im, coef * w.re); });
    if constexpr (PP) __syncthreads();
  } else {
    // inverse transform of the spectrum of u + i u_x: Y[m] = U + iV, Y[N-m] = conj(U) +
    // i conj(V); DC and Nyquist keep only the real parts, as irfft does.  The lower half
    // is the thread's own, the upper half comes from its mirror through LDS.
    constexpr int H = N / 2, E = N / T, EH = E / 2;
    static_assert(MPT == EH + 1 && EH >= 2, "rfft layout");
    // the half-length transform by half of the threads where all of them would have two points
    // each (9 passes of radix 2 at n = 1024, or 5 of radix 4: an evolve with four times the
    // base threads 2.16 -> 2.03 ms)
    constexpr int TH = EH == 2 && T > 64 ? T / 2 : T, EZ = H / TH;
    constexpr int XI = rksfft::exchanges<N, T, RKS_MAXR>(), XF = rksfft::exchanges<H, TH, RKS_MAXR>();
    C y[E];
#pragma unroll
    for (int k = 0; k < MPT; ++k) {
      if (k == EH && t != 0) continue;
      const int m = t + k * T;
      const C U = v[k];
      const R q = gload_real(kx, m);
      const R vr = scaled_re(-q, U.im);  // V = i q U
      C lo = mkc(fma(-q, U.re, U.re), add_re(U.im, vr));
      C up = mkc(fma(q, U.re, U.re), add_re(vr, -U.im));
      if (fused_imag<T>(k)) {
        lo.im = fma(-q, U.im, U.im);
        up.im = fma(-q, U.im, -U.im);
      }
      const C edge = mkc(U.re, vr);
      if (k == EH) {
        buf[0] = edge;
      } else if (k == 0) {
        // m = 0 keeps the real parts and has no mirror
        y[0] = t == 0 ? edge : lo;
        if (t != 0) buf[pad(H - m)] = up;
      } else {
        y[k] = lo;
        buf[pad(H - m)] = up;
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < EH; ++k) y[EH + k] = buf[pad(t + k * T)];
    if constexpr (!PP) __syncthreads();
    rksfft::fft_reg<R, N, T, true, LOG2N, RKS_MAXR, PP, 1, true>(y, buf, twl, t, [](C w) { return w; });
    // u u_x, a real sequence: complex element j of its half-length transform is the pair 2j, 2j+1
    constexpr int B2 = PP ? (1 + XI) & 1 : 0;
    C* const bp = buf + B2 * PS;
#pragma unroll
    for (int k = 0; k < E; ++k) {
      const int x = t + k * T;
      ((R*)(bp + pad(x >> 1)))[x & 1] = (y[k].re * inv) * (y[k].im * inv);
    }
    __syncthreads();
    const bool on = TH == T || t < TH;
    C z[EZ];
    if (on) {
#pragma unroll
      for (int k = 0; k < EZ; ++k) z[k] = bp[pad(t + k * TH)];
    }
    if constexpr (!PP) __syncthreads();
    constexpr int B3 = PP ? (B2 + 1) & 1 : 0;
    rksfft::fft_reg<R, H, TH, false, LOG2N, RKS_MAXR, PP, B3, true>(z, buf, twl, t, [](C w) { return w; }, on);
    constexpr int B4 = PP ? (B3 + XF) & 1 : 0;
    C* const bm = buf + B4 * PS;
    if (on) {
#pragma unroll
      for (int k = 0; k < EZ; ++k) bm[pad(t + k * TH)] = z[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < MPT; ++k) {
      if (k == EH && t != 0) continue;
      const int m = t + k * T;
      C Zk;
      if constexpr (TH == T) Zk = k < EH ? z[k < EH ? k : 0] : z[0];
      else Zk = bm[pad(m & (H - 1))];
      rksfft::leaf(Zk);
      const C Zc = conjc(bm[pad((H - m) & (H - 1))]);
      const C Ev = (R)0.5 * (Zk + Zc);
      const C D = Zk - Zc;
      const C O = mkc((R)0.5 * D.im, (R)-0.5 * D.re);
      const C W = Ev + rksfft::twiddle<R, LOG2N>(twl, m) * O;
      v[k] = coef * W;
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Stage passes of the general kernels, in functions of their own (noinline).  Their term loops
// are bound by the instructions that walk the tableau; inlined beside the transforms, whose
// butterflies take every register, they spilled and read the tableau by vector loads.  Here a
// pass has the registers to itself and reads the tableau by scalar loads, and every array from a
// uniform base.  One evolve, inlined / like this: FP64 n = 8192 ETD34 1.54 / 1.27 ms, ETD5 6.4 /
// 4.8, IF45DP 373 / 262; MIXED n = 4096 x 300 2.04 / 1.69, 7.8 / 5.6, 534 / 344; FP32 n = 8192 x
// 300 3.13 / 2.70, 12.4 / 9.5, 718 / 522.
// ---------------------------------------------------------------------------
#define RKS_AS3 __attribute__((address_space(3)))

// what every pass reads (uniform)
struct PassArgs {
  const void* ws;       // NL slots
  const char* cbase;    // coefficients, arrays of stride Mc
  double h;
  unsigned smap;
  int Mc, lim, fold;    // Own
};

// One stage: its argument (fin: the last stage and the error estimate from one load of each NL
// value, rks_fused_final) into the LDS buffer at `lds` by mode, the last stage's into cand as
// well.  Returns the thread's largest |u_new| (fin) or |u_new|^2.
template <typename R, typename RN, int LOG2N, int T, int NLK>
__device__ __attribute__((noinline)) double general_pass(const rks_tableau* tbp, int s, int fin, const cx<R>* u,
                                                         cx<R>* cand, RKS_AS3 unsigned char* lds, PassArgs A) {
  using C = cx<R>;
  using CN = cx<RN>;
  constexpr int N = 1 << LOG2N;
  constexpr int M = (NLK == NLK_ADVECT) ? N / 2 + 1 : N;
  using OW = Own<N, M, T, NLK>;
  using CK = Chunk<OW::MPT, (int)sizeof(C), T>;
  constexpr int CH = CK::CH;
  rks_ctab& tb = *rks_uniform_const<rks_ctab>(tbp);
  s = uni(s);
  fin = uni(fin);
  u = uni(u);
  cand = uni(cand);
  const unsigned base = (unsigned)uni((int)(unsigned)(unsigned long long)lds);
  const char* cbase = uni(A.cbase);
  const unsigned smap = (unsigned)uni((int)A.smap);
  CN* const slot_base = (CN*)uni((char*)A.ws);
  const size_t Mc = (size_t)uni(A.Mc);
  const double h = uni(A.h);
  OW ow;
  ow.lim = uni(A.lim);
  ow.fold = uni(A.fold);
  ow.t = threadIdx.x;
  auto slot = [&](int k) -> CN* { return slot_base + (size_t)((smap >> (4 * k)) & 15u) * M; };
  auto put = [&](int m, C v) {
    typedef typename GVec<R>::t V;
    V w;
    w.x = v.re;
    w.y = v.im;
    ((RKS_AS3 V*)(unsigned long long)base)[m] = w;
  };
  auto& S = tb.st[s];
  const bool last = s == tb.nstage - 1;
  double mx = 0.0;
#pragma unroll 1
  for (int c = 0; c < CK::NCH; ++c) {
    const ChunkIdx<CH> ix = pass_chunk<N, M, T, NLK, CH>(c, ow.fresh());
    C acc[CH];
    if (fin) {
      C ev[CH];
      final_chunk<R, RN, CH>(tb, u, slot, cbase, Mc, ix, h, acc, ev);
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        if (!ix.ok[i]) continue;
        gstore(cand, ix.m[i], acc[i]);
        const double a = hypot((double)acc[i].re, (double)acc[i].im);
        const double er = (double)ev[i].re, ei = (double)ev[i].im;
        mx = nanmax(mx, a);
        // FP64 keeps |err|^2; an FP32 buffer keeps |err| (|err|^2 would flush to zero
        // below ~1e-19 and turn a real error into an unconditional accept)
        if constexpr (sizeof(R) == sizeof(double)) put(ix.m[i], mkc((R)a, (R)(er * er + ei * ei)));
        else put(ix.m[i], mkc((R)a, (R)hypot(er, ei)));
      }
    } else {
      stage_chunk<R, RN, CH>(tb, S, u, slot, cbase, Mc, ix, h, acc);
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        if (!ix.ok[i]) continue;
        if (last) {
          gstore(cand, ix.m[i], acc[i]);
          if (tb.adaptive)
            mx = nanmax(mx, (double)acc[i].re * (double)acc[i].re + (double)acc[i].im * (double)acc[i].im);
        }
        put(ix.m[i], acc[i]);
      }
    }
  }
  return mx;
}

// The thread's masked sums of the error norm where the last stage has an NL (NormOrder):
// modes with lim < |u_new|^2 <= DBL_MAX.
struct NormSums {
  double su, se;
};
template <typename R, typename RN, int LOG2N, int T, int NLK>
__device__ __attribute__((noinline)) NormSums general_error(const rks_tableau* tbp, const cx<R>* cand, double lim,
                                                            PassArgs A) {
#pragma clang fp contract(off)
  using C = cx<R>;
  using CN = cx<RN>;
  constexpr int N = 1 << LOG2N;
  constexpr int M = (NLK == NLK_ADVECT) ? N / 2 + 1 : N;
  using OW = Own<N, M, T, NLK>;
  constexpr int CH = Chunk<OW::MPT, (int)sizeof(C), T>::CH;
  using NO = NormOrder<N, M, T, NLK>;
  constexpr int NCH = (NO::SLOTS + CH - 1) / CH;
  rks_ctab& tb = *rks_uniform_const<rks_ctab>(tbp);
  cand = uni(cand);
  lim = uni(lim);
  const char* cbase = uni(A.cbase);
  const unsigned smap = (unsigned)uni((int)A.smap);
  CN* const slot_base = (CN*)uni((char*)A.ws);
  const size_t Mc = (size_t)uni(A.Mc);
  const double h = uni(A.h);
  OW ow;
  ow.lim = uni(A.lim);
  ow.fold = uni(A.fold);
  ow.t = threadIdx.x;
  auto slot = [&](int k) -> CN* { return slot_base + (size_t)((smap >> (4 * k)) & 15u) * M; };
  NormSums n = {0.0, 0.0};
#pragma unroll 1
  for (int c = 0; c < NCH; ++c) {
    ChunkIdx<CH> ix = pass_chunk<N, M, T, NLK, CH>(c, ow.fresh());
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      ix.ok[i] = NO::ok(c * CH + i, ow.lim);
      ix.m[i] = ix.ok[i] ? NO::mode(c * CH + i) : 0;
    }
    C ev[CH];
    error_chunk<R, RN, CH>(tb, slot, cbase, Mc, ix, h, ev);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      if (!ix.ok[i]) continue;
      const C kv = gload(cand, ix.m[i]);
      const double kr = (double)kv.re, ki = (double)kv.im, er = (double)ev[i].re, ei = (double)ev[i].im;
      const double a = fma(kr, kr, ki * ki);
      if (a > lim && a <= __DBL_MAX__) {
        n.su += a;
        n.se += fma(er, er, ei * ei);
      }
    }
  }
  return n;
}

// ---------------------------------------------------------------------------
// learned step-size proposer: features of an accepted state, the training
// record, and the proposal that replaces the controller's next step
// ---------------------------------------------------------------------------
// Inputs (raw, before standardization): for b < 64,
//   f_b = 0.5 ln(mean |u_hat|^2 over bin b / n^2 + 1e-30),
// where mode m has wavenumber index w = m (rfft layout) or min(m, n - m)
// (fft layout) and lies in bin (64 w) / (n/2 + 1); f_64 = ln h of the accepted
// step, f_65 = ln min(s, 1e4) of its attempt.  |u_hat| comes from the LDS
// buffer where the fused final stage left it, else from the candidate array.
// Bin b covers the wavenumber indices w_lo(b) <= w < w_lo(b + 1) with
// w_lo(b) = ceil(b (n/2 + 1) / 64); the T/64 lanes of bin b sum fixed pieces
// of it in index order and a fixed butterfly adds the pieces, so the features
// do not depend on thread scheduling.
// A training record is written after every accept when records are on; the
// network runs when run_net is set (every (period 512 / T)-th accept).  Returns the
// next step: with d = y - margin and h_ref = h_suggest (the reference
// controller's proposal),
//   propose (0): h itself when keep_lo <= d < keep_hi (no coefficient
//                regeneration), else h exp(clamp(d, ln min_s, ln max_s));
//   guard (1):   h_ref unless d < ln(h_ref / h) + keep_lo (the network
//                predicts its rejection); then h exp(max(d, ln min_s));
//   grow (2):    as guard, and when d >= ln(h_ref / h) + g (g = keep_hi > 0)
//                h_ref e^(j g) with j = floor((d - ln(h_ref / h)) / g), capped
//                at h max_s: the network lets the step grow ahead of the
//                reference on a geometric grid of ratio e^g.
// Without a proposer, without run_net or with a non-finite y: h_ref.
template <typename R, int LOG2N, int T, int NLK>
__device__ __forceinline__ double learned_after_accept(const rks_launch& P, const rks_ctrl& ct, rks_inst* in,
                                                       const cx<R>* ucand, const cx<R>* buf, bool fused,
                                                       double h_used, double s_acc, double h_suggest, bool run_net,
                                                       float* bins, float* scr) {
  static_assert(T >= RKS_MLP_NBIN && T % 64 == 0, "whole waves, at least one thread per spectral input");
  constexpr int N = 1 << LOG2N;
  constexpr int W = N / 2 + 1;                // wavenumber indices 0..n/2
  constexpr int TPB = T / RKS_MLP_NBIN;       // threads per bin: consecutive lanes of one wave
  const int t = threadIdx.x;
  const int b = t / TPB, part = t % TPB;
  __syncthreads();  // the fused final stage's LDS values are complete
  // bin b covers wavenumber indices [w0, w1); this thread sums the part-th of TPB
  // contiguous pieces, the pieces are combined by a fixed butterfly: the same sum
  // in every run
  const int w0 = (b * W + RKS_MLP_NBIN - 1) / RKS_MLP_NBIN;
  const int w1 = ((b + 1) * W + RKS_MLP_NBIN - 1) / RKS_MLP_NBIN;
  const int q0 = w0 + ((w1 - w0) * part) / TPB, q1 = w0 + ((w1 - w0) * (part + 1)) / TPB;
  double pw = 0.0;
  int cnt = 0;
#pragma unroll 1
  for (int w = q0; w < q1; ++w) {
    // modes of wavenumber index w: m = w, and (fft layout) m = n - w for 0 < w < n/2
    const int nm = (NLK == NLK_ADVECT || w == 0 || w == N / 2) ? 1 : 2;
    for (int k = 0; k < nm; ++k) {
      const int m = k == 0 ? w : N - w;
      if (fused) {
        const double a = (double)buf[m].re;
        pw += a * a;
      } else {
        const cx<R> v = ucand[m];
        pw += (double)v.re * (double)v.re + (double)v.im * (double)v.im;
      }
      ++cnt;
    }
  }
#pragma unroll
  for (int o = 1; o < TPB; o <<= 1) {
    pw += __shfl_xor(pw, o, 64);
    cnt += __shfl_xor(cnt, o, 64);
  }
  const float f = 0.5f * logf((float)(pw / (double)cnt) / ((float)N * (float)N) + 1e-30f);
  __syncthreads();
  if (part == 0) bins[b] = f;
  if (t == 0) {
    bins[RKS_MLP_NBIN] = (float)log(h_used);
    bins[RKS_MLP_NBIN + 1] = (float)log(s_acc < RKS_MLP_S_CAP ? s_acc : RKS_MLP_S_CAP);
  }
  __syncthreads();
  const int rec_count = in->rec_count;
  if (in->rec != nullptr && rec_count < in->rec_cap) {
    float* r = in->rec + (size_t)rec_count * RKS_MLP_REC;
    for (int j = t; j < RKS_MLP_NIN; j += T) r[j] = bins[j];
    __syncthreads();  // every thread has read the counters before they change
    if (t == 0) {
      r[RKS_MLP_NIN] = __builtin_nanf("");
      r[RKS_MLP_NIN + 1] = 0.f;
      in->rec_pending = rec_count;
      in->rec_count = rec_count + 1;
    }
  }
  if (P.mlp.on && run_net) {
    rks_mlp_standardize<T>(P.mlp, bins, scr);
    const float y = rks_mlp_infer<T>(P.mlp, scr, scr + RKS_MLP_K0);
    if (!(isinf(y) || isnan(y))) {
      double yl = (double)y - (double)P.mlp.margin;
      if (P.mlp.policy == 1 || P.mlp.policy == 2) {
        const double lref = log(h_suggest / h_used);
        if (yl < lref + (double)P.mlp.keep_lo) {
          const double lo = log(ct.min_s);
          h_suggest = h_used * exp(yl < lo ? lo : yl);
        } else if (P.mlp.policy == 2 && P.mlp.keep_hi > 0.f) {
          const double g = (double)P.mlp.keep_hi;
          const double j = floor((yl - lref) / g);
          if (j >= 1.0) {
            double ln = lref + j * g;
            const double hi = log(ct.max_s);
            h_suggest = h_used * exp(ln < hi ? ln : hi);
          }
        }
      } else if (yl >= (double)P.mlp.keep_lo && yl < (double)P.mlp.keep_hi) {
        h_suggest = h_used;
      } else {
        const double lo = log(ct.min_s), hi = log(ct.max_s);
        yl = yl < lo ? lo : (yl > hi ? hi : yl);
        h_suggest = h_used * exp(yl);
      }
    }
  }
  return h_suggest;
}

// ---------------------------------------------------------------------------
// one instance: evolve / step / nl
// ---------------------------------------------------------------------------
// Returns nonzero (proposer variant only) when the evolve stopped after an
// accepted step for the proposer: the state is in the instance record, and the
// caller runs learned_between_steps and calls again with reenter set.
template <typename R, typename RN, int LOG2N, int T, int NLK, bool LEARN, int METH>
__device__ int run_instance(const rks_launch& P, int idx, cx<R>* buf, const cx<R>* twl, double* red,
                            int* lds_count, bool reenter) {
  using C = cx<R>;
  using CN = cx<RN>;
  constexpr int N = 1 << LOG2N;
  constexpr int M = (NLK == NLK_ADVECT) ? N / 2 + 1 : N;
  using OW = Own<N, M, T, NLK>;
  constexpr int MPT = OW::MPT;
  constexpr bool METHOD = METH != RKS_METH_ANY;
  using CK = Chunk<MPT, (int)sizeof(C), T>;
  constexpr int CH = CK::CH;
  // the general kernel's tableau entries as uniform values (the Hankel kind: as they stand)
  auto un = [](int x) { return NLK == NLK_HANKEL ? x : uni(x); };
  constexpr bool PAIRED = !METHOD && M == N && NLK != NLK_HANKEL;  // pass_chunk: other modes than the transforms'
  using TT = MethodTab<METHOD ? METH : 0, (int)sizeof(C), (int)sizeof(CN), NLK == NLK_ADVECT>;
  constexpr bool FUSED = TT::tab.st[TT::tab.nstage - 1].has_nl == 0;  // (METHOD) no NL in the last stage
  constexpr int LAST_SLOT = TT::tab.st[FUSED ? TT::tab.nstage - 2 : TT::tab.nstage - 1].nl_slot;
  const rks_tableau* __restrict__ tbp = P.tab;
  const rks_ctrl* __restrict__ ctp = P.ctl;
  const rks_tableau& tb = *tbp;
  const rks_ctrl& ct = *ctp;
  rks_inst* in = uni(P.inst + idx);
  const rks_io io = P.io[idx];
  const int t = threadIdx.x;
  const R* kx = uni((const R*)in->kx);
  const R nlc = (R)uni(in->nl_coef);
  const double* Ld = uni(in->L);
  const int Lc = uni(in->L_complex);
  // workspace: nslot NL arrays (RN) | 2 candidate states (R) | coefficients
  // (each region 256-byte aligned; layout computed by the host, rks_ws_layout)
  char* ws = uni((char*)in->ws);
  const int nslot = METHOD ? TT::tab.nslot : tb.nslot;
  CN* const slot_base = (CN*)ws;
  C* const cand0 = (C*)(ws + rks_align256((size_t)nslot * M * sizeof(CN)));
  C* const cand1 = cand0 + rks_align256((size_t)M * sizeof(C)) / sizeof(C);
  char* cbase = (char*)(cand1 + rks_align256((size_t)M * sizeof(C)) / sizeof(C));
  // mirror-symmetric L (complex state): coefficients of modes 0..N/2 in
  // arrays of stride Mc (a multiple of 64 modes, at most M)
  const int sym = (M == N) && uni(in->coef_sym);
  constexpr int MSYM = ((N / 2 + 1 + 63) / 64) * 64 < M ? ((N / 2 + 1 + 63) / 64) * 64 : M;
  const int Mc = sym ? MSYM : M;
  // modes in use: the Hankel kind's nr radial points (arrays keep the stride M of
  // its size class), every mode otherwise
  const int Mr = NLK == NLK_HANKEL ? uni(in->m) : M;
  const int Mg = sym ? N / 2 + 1 : Mr;
  const double hs = uni(in->nl_scale);
  OW ow;
  ow.lim = Mr;
  ow.fold = sym ? N : 0;
  ow.t = t;
  const C* const uin = uni((const C*)io.u_in);
  // the thread's modes of an array, and back
  auto load_modes = [&](C(&v)[MPT], const C* src) {
    const OW of = ow.fresh();
#pragma unroll
    for (int k = 0; k < MPT; ++k) v[k] = gload(src, of.m(k));
  };
  auto copy_modes = [&](C* dst, const C* src) {
    C v[MPT];
    load_modes(v, src);
#pragma unroll
    for (int k = 0; k < MPT; ++k)
      if (ow.ok(k)) gstore(dst, ow.m(k), v[k]);
  };

  if (P.mode == RKS_MODE_NL) {
    C v[MPT];
    load_modes(v, uin);
    nl_regs<R, LOG2N, T, NLK>(v, buf, twl, nlc, kx, Mr, hs);
    C* out = uni((C*)io.u_out);
#pragma unroll
    for (int k = 0; k < MPT; ++k)
      if (ow.ok(k)) gstore(out, ow.m(k), v[k]);
    return 0;
  }

  // ---- load persistent state (uniform across the workgroup) ----
  double tc = uni(in->tc), tf = uni(in->tf), h = uni(in->h), h_coeff = uni(in->h_coeff), h_next = uni(in->h_next);
  double h_used = uni(in->h_used);
  int started = uni(in->started), accept = uni(in->accept), steps = uni(in->steps), attempts = uni(in->attempts);
  int rejects = uni(in->rejects), status = uni(in->status), ubuf = uni(in->ubuf);
  int log_count = uni(in->log_count), snap_count = uni(in->snap_count);
  int nl_calls = uni(in->nl_calls), coef_updates = uni(in->coef_updates);
  // slot map packed 4 bits per slot (no dynamically indexed register array)
  unsigned smap = 0;
#pragma unroll
  for (int s = 0; s < RKS_MAX_SLOTS; ++s) smap |= (unsigned)(uni(in->slot_map[s]) & 15) << (4 * s);
  const int store_freq = uni(in->store_freq), snap_cap = uni(in->snap_cap), log_cap = uni(in->log_cap);

  if (io.reset && !reenter) {
    started = 0;
    accept = 0;
    h_coeff = __builtin_nan("");
    smap = 0x76543210u;
  }
  const bool adaptive = METHOD ? TT::tab.adaptive != 0 : un(tb.adaptive) != 0;
  const bool evolve = (P.mode == RKS_MODE_EVOLVE);
  if (reenter) {
    // back from the proposer: h_next holds its proposal (solveras.py:638-641)
    status = RKS_ST_RUNNING;
    h = uni((tc + h_next > tf) ? tf - tc : h_next);
  } else if (evolve && !io.resume) {
    tc = uni(io.t0);
    tf = uni(io.tf);
    h = uni(io.h_in);
    steps = attempts = rejects = 0;
    log_count = snap_count = 0;
    nl_calls = coef_updates = 0;
    ubuf = -1;
    status = RKS_ST_RUNNING;
    if (adaptive && tc + h > tf) h = uni(tf - tc);  // solveras.py:620-621
    if (LEARN && in->rec != nullptr) {
      // record counters live in the instance record: the stepping loop does not carry them
      __syncthreads();
      if (t == 0) {
        in->rec_count = 0;
        in->rec_pending = -1;
        in->h_prop = h;
      }
      __syncthreads();
    }
    if (store_freq > 0) {
      copy_modes(uni((C*)in->snap), uin);
      if (t == 0) in->snap_t[0] = tc;
      snap_count = 1;
    }
  } else if (evolve) {
    status = RKS_ST_RUNNING;
  } else {
    h = uni(io.h_in);
    status = RKS_ST_RUNNING;
    attempts = rejects = 0;
  }

  auto slot = [&](int s) -> CN* { return slot_base + (size_t)((smap >> (4 * s)) & 15u) * M; };
  auto pass_args = [&]() { return PassArgs{ws, cbase, h, smap, Mc, ow.lim, ow.fold}; };
  auto cur_u = [&]() -> const C* { return ubuf < 0 ? uin : (const C*)(ubuf == 0 ? cand0 : cand1); };
  const bool fused = METHOD ? FUSED : un((int)rks_fused_final(tb)) != 0;
  const bool recompute = (METHOD ? TT::tab.nl1_policy : un(tb.nl1_policy)) == RKS_NL1_RECOMPUTE;
  const int nstage = METHOD ? TT::tab.nstage : un(tb.nstage);

  bool done = false;
  int pending = 0;      // proposer variant: stopped after an accept for the proposer
  double s_hand = 0.0;  // s of that accept
  while (!done) {
    if (evolve) {
      if (!(tc < tf)) {
        status = RKS_ST_OK;
        break;
      }
      if (store_freq > 0 && snap_count >= snap_cap) {
        status = RKS_ST_PAUSED;
        break;
      }
    }
    const C* u = uni(evolve ? cur_u() : uin);
    C* cand = uni(evolve ? (ubuf == 0 ? cand1 : cand0) : (C*)io.u_out);
    int numloops = 0;
    double h_suggest = h;
    double s_acc;  // s of the accepted attempt (set where the attempt loop accepts)
    // ---------------- attempt loop (solveras.py:384-410) ----------------
    for (;;) {
      if (h != h_coeff) {
        if constexpr (METHOD)
          coef_update_method<TT, R, RN, T, MPT>(ct, Ld, Mc, Mg, h, cbase, (int*)buf, lds_count);
        else
          coef_update<R, RN, T, MPT>(tb, ct, Ld, Lc, Mc, Mg, h, cbase, (int*)buf, lds_count);
        h_coeff = h;
        ++coef_updates;
      }
      bool first_nl = false;  // NL1 = nl(u) before the first stage
      if (!started) {
        first_nl = true;
        started = 1;
      } else if (accept || !adaptive) {
        if (recompute) {
          first_nl = true;
        } else {
          const unsigned f4 = 4u * (unsigned)(METHOD ? TT::tab.fsal_slot : un(tb.fsal_slot));
          const unsigned a = smap & 15u, b = (smap >> f4) & 15u;
          smap = (smap & ~(15u | (15u << f4))) | b | (a << f4);
        }
      }
      double mx = 0.0;    // max |u_new| (fused last stage) or |u_new|^2
      double su = 0.0, se = 0.0;
      CN nv[MPT];         // NL values of the last evaluation
#pragma unroll
      for (int k = 0; k < MPT; ++k) nv[k] = mkc((RN)0, (RN)0);
#pragma unroll 1
      for (int s = un(first_nl ? -1 : 0); s < nstage; ++s) {
        const bool last = s == nstage - 1;
        C v[MPT];
        int ns = 0;  // NL slot this pass writes
        if constexpr (METHOD) {
          if (s < 0) {
            load_modes(v, u);
          } else {
            if (FUSED && last) break;
            stage_switch<TT, 0, true>(s, v, nv, u, ow, slot, cbase, (size_t)Mc, h);
            if (!FUSED && last) {
#pragma unroll
              for (int k = 0; k < MPT; ++k) {
                if (ow.ok(k)) {
                  gstore(cand, ow.m(k), v[k]);
                  if (TT::tab.adaptive)
                    mx = nanmax(mx, (double)v[k].re * (double)v[k].re + (double)v[k].im * (double)v[k].im);
                }
              }
            }
            static_assert(TT::tab.st[0].nl_slot == 1 && LAST_SLOT == TT::tab.nslot - 1, "stage s writes slot s + 1");
            ns = s + 1;
          }
        } else if constexpr (NLK == NLK_HANKEL) {
          // Inlined, tableau and arrays read as they stand: with a mode or two per thread nothing
          // spills, and the code around the products decides how the compiler orders their loads.
          // By general_pass IF34 takes 0.47 ms for 84 MIXED beams of nr = 126 (like this 0.43) and
          // 1.06 for 64 FP32 beams of nr = 500 (0.92).
          if (s < 0) {
            load_modes(v, u);
          } else {
            const rks_stage& S = tb.st[s];
            if (last && fused) {
              // per-mode |u_new| and |err|^2 (FP32 buffer: |err|) wait in the idle LDS buffer
#pragma unroll 1
              for (int c = 0; c < CK::NCH; ++c) {
                const ChunkIdx<CH> ix = pass_chunk<N, M, T, NLK, CH>(c, ow.fresh());
                C acc[CH], ev[CH];
                final_chunk<R, RN, CH>(tb, u, slot, cbase, (size_t)Mc, ix, h, acc, ev);
#pragma unroll
                for (int i = 0; i < CH; ++i) {
                  const int m = ix.m[i];
                  if (ix.ok[i]) {
                    cand[m] = acc[i];
                    const double a = hypot((double)acc[i].re, (double)acc[i].im);
                    const double er = (double)ev[i].re, ei = (double)ev[i].im;
                    mx = nanmax(mx, a);
                    // FP64 keeps |err|^2; an FP32 buffer keeps |err| (|err|^2 would flush to zero
                    // below ~1e-19 and turn a real error into an unconditional accept)
                    if constexpr (sizeof(R) == sizeof(double)) buf[m] = mkc((R)a, (R)(er * er + ei * ei));
                    else buf[m] = mkc((R)a, (R)hypot(er, ei));
                  }
                }
              }
              break;
            }
            // the stage argument through the thread's own places of the LDS buffer: the run-time
            // term loop stays rolled over the chunks
#pragma unroll 1
            for (int c = 0; c < CK::NCH; ++c) {
              const ChunkIdx<CH> ix = pass_chunk<N, M, T, NLK, CH>(c, ow.fresh());
              C acc[CH];
              stage_chunk<R, RN, CH>(tb, S, u, slot, cbase, (size_t)Mc, ix, h, acc);
#pragma unroll
              for (int i = 0; i < CH; ++i) {
                if (!ix.ok[i]) continue;
                if (last) {
                  cand[ix.m[i]] = acc[i];
                  if (adaptive)
                    mx = nanmax(mx, (double)acc[i].re * (double)acc[i].re + (double)acc[i].im * (double)acc[i].im);
                }
                buf[ix.m[i]] = acc[i];
              }
            }
            if (!S.has_nl) continue;
            const OW of = ow.fresh();
#pragma unroll
            for (int k = 0; k < MPT; ++k) v[k] = buf[of.m(k)];
            __syncthreads();
            ns = S.nl_slot;
          }
        } else {
          // the argument through the LDS buffer, u itself too: loaded into v here, it would be
          // held through the call of the other branch
          bool has_nl = true;
          if (s < 0) {
            const OW of = ow.fresh();
#pragma unroll
            for (int k = 0; k < MPT; ++k)
              if (of.ok(k)) buf[of.m(k)] = gload(u, of.m(k));
          } else {
            const bool fin = last && fused;
            const double m = general_pass<R, RN, LOG2N, T, NLK>(tbp, s, fin, u, cand, (RKS_AS3 unsigned char*)buf,
                                                                pass_args());
            if (last) mx = m;
            if (fin) break;
            has_nl = uni(tb.st[s].has_nl) != 0;
            ns = uni(tb.st[s].nl_slot);
          }
          if constexpr (PAIRED) __syncthreads();  // buf, and cand for what copies it
          if (!has_nl) continue;
          const OW of = ow.fresh();
#pragma unroll
          for (int k = 0; k < MPT; ++k) v[k] = buf[of.m(k)];
          __syncthreads();
        }
        nl_regs<R, LOG2N, T, NLK>(v, buf, twl, nlc, kx, Mr, hs);
        ++nl_calls;
        CN* const dst = slot(ns);
        const OW of = ow.fresh();
#pragma unroll
        for (int k = 0; k < MPT; ++k) {
          nv[k] = cvt<RN>(v[k]);
          if (of.ok(k)) gstore(dst, of.m(k), nv[k]);
        }
        if constexpr (PAIRED) __syncthreads();  // the stage passes read them by pairs
      }
      if (!adaptive) {
        h_suggest = h;
        accept = 1;
        break;
      }
      // ---------------- embedded error norm (solveras.py:449-455) ----------------
      // masked sums of |u_new|^2 and |err|^2 (FP64) over |u_new| / max |u_new| > cutoff.  Where
      // the last stage has no NL, |u_new| is kept (mx: its maximum), else its square; the mask
      // compares those instead of dividing.  A square that overflows or vanishes does so in the
      // sums as well, and the attempt is rejected either way.
      const double cut = ct.adapt_cutoff;
      if constexpr (METHOD) {
#pragma clang fp contract(off)
        using NO = NormOrder<N, M, T, NLK>;
        constexpr int NS = NO::OWN ? MPT : NO::SLOTS;
        double a[MPT], e[MPT], an[NS], en[NS];
        final_sum<TT, LAST_SLOT, 0, rks_sum_chunk<R>(), !FUSED>(a, e, cand, nv, u, ow, slot, cbase, (size_t)Mc, h);
        if constexpr (FUSED) {
#pragma unroll
          for (int k = 0; k < MPT; ++k) mx = nanmax(mx, a[k]);
        }
        if constexpr (!NO::OWN) {
          // into NormOrder through the idle buffer, where the proposer finds |u_new|
          double* const db = (double*)buf;
          constexpr bool PAIRS = FUSED || sizeof(R) == sizeof(double);  // both values fit an element
#pragma unroll
          for (int k = 0; k < MPT; ++k) {
            if (!ow.ok(k)) continue;
            if constexpr (PAIRS) buf[ow.raw(k)] = mkc((R)a[k], (R)e[k]);
            else db[ow.raw(k)] = a[k];
          }
          __syncthreads();
#pragma unroll
          for (int k = 0; k < NS; ++k) {
            const bool ok = NO::ok(k, ow.lim);
            const int m = ok ? NO::mode(k) : 0;
            if constexpr (PAIRS) {
              an[k] = ok ? (double)buf[m].re : 0.0;
              en[k] = ok ? (double)buf[m].im : 0.0;
            } else {
              an[k] = ok ? db[m] : 0.0;
            }
          }
          __syncthreads();
          if constexpr (!PAIRS) {
#pragma unroll
            for (int k = 0; k < MPT; ++k)
              if (ow.ok(k)) db[ow.raw(k)] = e[k];
            __syncthreads();
#pragma unroll
            for (int k = 0; k < NS; ++k) en[k] = NO::ok(k, ow.lim) ? db[NO::mode(k)] : 0.0;
            __syncthreads();
          }
        } else {
#pragma unroll
          for (int k = 0; k < NS; ++k) {
            an[k] = a[k];
            en[k] = e[k];
            if constexpr (LEARN && FUSED) {
              if (ow.ok(k)) buf[ow.m(k)].re = (R)a[k];
            }
          }
        }
        mx = wg_max<T>(mx, red);
        const double lim = FUSED ? cut * mx : (cut < 0.0 ? -1.0 : cut * cut * mx);
#pragma unroll
        for (int k = 0; k < NS; ++k) {
          const bool on = an[k] > lim && an[k] <= __DBL_MAX__;
          const double x = on ? an[k] : 0.0, y = on ? en[k] : 0.0;
          su = FUSED ? fma(x, x, su) : su + x;
          se = (FUSED && sizeof(R) < sizeof(double)) ? fma(y, y, se) : se + y;
        }
      } else {
#pragma clang fp contract(off)
        mx = wg_max<T>(mx, red);
        const double lim = fused ? cut * mx : (cut < 0.0 ? -1.0 : cut * cut * mx);
        __syncthreads();  // every thread's last NL values, candidate and buffer values
        using NO = NormOrder<N, M, T, NLK>;
        if constexpr (NLK == NLK_HANKEL) {
          constexpr int NCH = (NO::SLOTS + CH - 1) / CH;
#pragma unroll 1
          for (int c = 0; c < NCH; ++c) {
            ChunkIdx<CH> ix = pass_chunk<N, M, T, NLK, CH>(c, ow.fresh());
#pragma unroll
            for (int i = 0; i < CH; ++i) {
              ix.ok[i] = NO::ok(c * CH + i, ow.lim);
              ix.m[i] = ix.ok[i] ? NO::mode(c * CH + i) : 0;
            }
            C ev[CH];
            if (!fused) error_chunk<R, RN, CH>(tb, slot, cbase, (size_t)Mc, ix, h, ev);
#pragma unroll
            for (int i = 0; i < CH; ++i) {
              if (!ix.ok[i]) continue;
              if (fused) {
                const C q = buf[ix.m[i]];
                const double a = (double)q.re, e = (double)q.im;
                if (a > lim && a <= __DBL_MAX__) {
                  su = fma(a, a, su);
                  se = sizeof(R) < sizeof(double) ? fma(e, e, se) : se + e;
                }
              } else {
                const C kv = cand[ix.m[i]];
                const double kr = (double)kv.re, ki = (double)kv.im, er = (double)ev[i].re, ei = (double)ev[i].im;
                const double a = fma(kr, kr, ki * ki);
                if (a > lim && a <= __DBL_MAX__) {
                  su += a;
                  se += fma(er, er, ei * ei);
                }
              }
            }
          }
        } else if (fused) {
#pragma unroll 1
          for (int k = 0; k < NO::SLOTS; ++k) {
            if (!NO::ok(k, ow.lim)) continue;
            const C q = buf[NO::mode(k)];
            const double a = (double)q.re, e = (double)q.im;
            if (a > lim && a <= __DBL_MAX__) {
              su = fma(a, a, su);
              se = sizeof(R) < sizeof(double) ? fma(e, e, se) : se + e;
            }
          }
        } else {
          const NormSums n = general_error<R, RN, LOG2N, T, NLK>(tbp, cand, lim, pass_args());
          su = n.su;
          se = n.se;
        }
        if (fused) __syncthreads();  // the buffer's values are read
      }
      wg_sum2<T>(su, se, red);
      const int q = METHOD ? TT::tab.q : tb.q;
      const double sv = uni(rks_error_ratio(su, se, ct.epsilon, ct.safety_f, q, sizeof(RN) < sizeof(double)));
      ++attempts;
      if (t == 0 && log_count < log_cap) {
        in->log[2 * log_count] = h;
        in->log[2 * log_count + 1] = sv;
      }
      ++log_count;
      if (LEARN && evolve && in->rec != nullptr) {
        // target of the record left by the last accept: ln(h s / h_accepted)
        const int pend = in->rec_pending;
        __syncthreads();  // every thread has read rec_pending before thread 0 clears it
        if (pend >= 0 && t == 0) {
          float* r = in->rec + (size_t)pend * RKS_MLP_REC;
          const bool ok = (h == in->h_prop) && !(isinf(sv) || isnan(sv)) && sv < 1e300;
          r[RKS_MLP_NIN] = (float)log(h * sv / h_used);
          r[RKS_MLP_NIN + 1] = ok ? 1.f : 0.f;
          in->rec_pending = -1;
        }
      }
      if (isinf(sv) || isnan(sv) || sv < 1.0) {
        // reject (solveras.py:490-506)
        accept = 0;
        ++rejects;
        if (isinf(sv) || isnan(sv)) {
          h = uni(ct.min_s * h);
        } else {
          double sc = sv > ct.min_s ? sv : ct.min_s;
          sc = sc < ct.decr_f ? sc : ct.decr_f;
          h = uni(sc * h);
        }
        ++numloops;
        if (numloops > ct.max_loops) {
          status = RKS_ST_MAXLOOPS;
          done = true;
          break;
        }
        if (h < ct.minh) {
          status = RKS_ST_MINSTEP;
          done = true;
          break;
        }
        continue;
      }
      // accept (solveras.py:543-554)
      accept = 1;
      s_acc = sv;
      const double sc = sv < ct.max_s ? sv : ct.max_s;
      h_suggest = uni((sc > ct.incr_f) ? sc * h : h);
      break;
    }
    if (done) break;
    // ---------------- accepted step ----------------
    h_used = h;
    h_next = h_suggest;
    if (!evolve) {
      status = RKS_ST_OK;
      ++steps;
      break;
    }
    ubuf = (ubuf == 0) ? 1 : 0;
    const double tprev = tc;
    tc = uni(tc + h);
    ++steps;
    if (!(tc > tprev)) {
      // h below the resolution of tc: the reference would loop forever here;
      // stop with the minimum-step status instead of spinning on the device
      status = RKS_ST_MINSTEP;
      break;
    }
    if (store_freq > 0 && (steps % store_freq) == 0) {
      copy_modes(uni((C*)in->snap) + (size_t)snap_count * Mr, cur_u());
      if (t == 0) in->snap_t[snap_count] = tc;
      ++snap_count;
    }
    if constexpr (LEARN && T >= 64) {
      // the network runs after every (period 512 / T)-th accepted step: a batch-1
      // inference streams the same ~300 KB of weights through T / 64 waves, so small
      // workgroups, whose attempts are short, consult it proportionally less often;
      // records (when on) are written after each accepted step.  The proposer runs
      // outside this loop (the caller, learned_between_steps): a call here would keep
      // every loop-carried value live across it and spill inside the stage passes.
      const bool run_net = P.mlp.on && (steps % (P.mlp.period * (512 / T))) == 0;
      if (adaptive && tc < tf && (run_net || in->rec != nullptr)) {
        pending = run_net ? 3 : 1;
        s_hand = s_acc;
        break;
      }
    }
    if (adaptive) h = uni((tc + h_suggest > tf) ? tf - tc : h_suggest);  // solveras.py:638-641
  }
  if (evolve && status != RKS_ST_PAUSED && !pending) copy_modes(uni((C*)io.u_out), cur_u());
  __syncthreads();
  if (t == 0) {
    in->tc = tc;
    in->tf = tf;
    in->h = h;
    in->h_coeff = h_coeff;
    in->h_next = h_next;
    in->h_used = h_used;
    in->started = started;
    in->accept = accept;
    in->steps = steps;
    in->attempts = attempts;
    in->rejects = rejects;
    in->status = status;
    in->ubuf = ubuf;
    in->log_count = log_count;
    in->snap_count = snap_count;
    in->nl_calls = nl_calls;
    in->coef_updates = coef_updates;
#pragma unroll
    for (int s = 0; s < RKS_MAX_SLOTS; ++s) in->slot_map[s] = (int)((smap >> (4 * s)) & 15u);
    if (LEARN) {
      in->s_acc = s_hand;
      in->learn_pending = pending;
    }
  }
  return pending;
}

// The proposer between two steps of an evolve (proposer variant): run_instance
// stopped after an accepted step with its state in the instance record (h_next:
// the reference controller's proposal; s_acc, learn_pending).  Features and
// records from the accepted state (the LDS buffer still holds the fused final
// stage's |u_new|), then the network's proposal replaces h_next.
template <typename R, typename RN, int LOG2N, int T, int NLK>
__device__ __forceinline__ void learned_between_steps(const rks_launch& P, int idx, const cx<R>* buf, float* bins,
                                                      float* scr) {
  constexpr int N = 1 << LOG2N;
  constexpr int M = (NLK == NLK_ADVECT) ? N / 2 + 1 : N;
  __syncthreads();  // thread 0's stores to the record are visible
  rks_inst* in = P.inst + idx;
  const rks_tableau& tb = *P.tab;
  // the accepted state: candidate buffer ubuf of the workspace (rks_ws_layout)
  const char* ws = (const char*)in->ws;
  const cx<R>* cand0 = (const cx<R>*)(ws + rks_align256((size_t)tb.nslot * M * sizeof(cx<RN>)));
  const cx<R>* ucur = in->ubuf == 0 ? cand0 : cand0 + rks_align256((size_t)M * sizeof(cx<R>)) / sizeof(cx<R>);
  const int pend = in->learn_pending;
  const double h_ref = in->h_next;
  const double h_new = learned_after_accept<R, LOG2N, T, NLK>(P, *P.ctl, in, ucur, buf, rks_fused_final(tb), in->h_used,
                                                              in->s_acc, h_ref, (pend & 2) != 0, bins, scr);
  __syncthreads();  // every thread has read the record
  if (threadIdx.x == 0) {
    in->h_next = h_new;
    if (in->rec != nullptr) in->h_prop = h_new;
    in->learn_pending = 0;
  }
  __syncthreads();
}

// waves per SIMD the register allocation must allow: 2 (256 registers) for
// every kernel.  At 168 registers (3 waves) the stage passes spill: the FP32
// buckets ran 6-28% slower (n = 256 .. 4096, KS and NLS families, best tile
// each; KS n = 1024 181 vs 239 ms, NLS n = 4096 1248 vs 1572 ms), the KS
// ensemble 5-19% slower in FP64 and 9-14% in MIXED.
__host__ __device__ constexpr int rks_min_waves(int /*log2n*/, int /*state_bytes*/) { return 2; }

// LEARN: the variant with the learned step-size proposer and its training
// records; the plain variant carries none of that code, so the stepping loop
// keeps its register allocation.
// TILE 1: twice the threads per trajectory (half the modes per thread in the
// stage passes and FFTs), where every transform keeps >= 2 elements per thread.
// METH: one method's stage sums and coefficients as literals (rks_method.h), or
// RKS_METH_ANY.
template <typename R, typename RN, int LOG2N, int NLK, bool LEARN, int TILE, int METH>
__global__ __launch_bounds__(rks_threads(LOG2N, NLK) << TILE, rks_min_waves(LOG2N, (int)sizeof(R))) void rks_kernel(
    rks_launch P) {
  constexpr int T = rks_threads(LOG2N, NLK) << TILE;
  static_assert(T <= 1024 && (NLK == NLK_HANKEL || T <= (NLK == NLK_ADVECT ? (1 << LOG2N) / 4 : (1 << LOG2N) / 2)),
                "tile too wide");
  extern __shared__ __align__(16) unsigned char rks_smem[];
  __shared__ double red[2 * (T / 64 + 1)];
  __shared__ int s_item;
  __shared__ int s_count;
  // proposer scratch: spectrum bins, and input/activation vectors (in the
  // FFT buffer, idle between attempts, when it is large enough)
  constexpr bool kScrInBuf =
      rksfft::padded_size(1 << LOG2N) * sizeof(cx<R>) >= RKS_MLP_LDS_FLOATS * sizeof(float);
  __shared__ float s_bins[LEARN ? 2 * RKS_MLP_NBIN : 1];
  __shared__ float s_scr[(LEARN && !kScrInBuf) ? RKS_MLP_LDS_FLOATS : 1];
  cx<R>* buf = (cx<R>*)rks_smem;
  cx<R>* twl = buf + rks_buf_elems<R, LOG2N, T, NLK>();
  float* scr = kScrInBuf ? (float*)rks_smem : s_scr;
  if constexpr (NLK != NLK_HANKEL) rksfft::load_twiddles<R, LOG2N, T>(twl, (const cx<R>*)P.tw);
  for (bool first = true;; first = false) {
    int item = first ? (int)blockIdx.x : P.count;  // without a queue: a workgroup per trajectory
    if (P.queue != nullptr) {
      if (threadIdx.x == 0) s_item = atomicAdd(P.queue, 1);
      __syncthreads();
      item = uni(s_item);
      __syncthreads();
    }
    if (item >= P.count) break;
    const int idx = uni(P.order[item]);
    if constexpr (LEARN && T >= 64) {
      bool reenter = false;
      while (run_instance<R, RN, LOG2N, T, NLK, LEARN, METH>(P, idx, buf, twl, red, &s_count, reenter)) {
        learned_between_steps<R, RN, LOG2N, T, NLK>(P, idx, buf, s_bins, scr);
        reenter = true;
      }
    } else {
      run_instance<R, RN, LOG2N, T, NLK, LEARN, METH>(P, idx, buf, twl, red, &s_count, false);
    }
    __syncthreads();
  }
}

// What a launch needs of a kernel; the host's table of them is filled by the units that
// instantiate the kernels (rks_k.hip, one per precision x nonlinearity x method).
struct rks_kernel_entry {
  const void* fn;
  int threads;
  int lds;
};

// Stage sums, error estimate and coefficient generator of one method as literals.
//
// The method tableau is a constant (rks_tableau.h), so every term's slots, scales,
// coefficient array and storage kind are compile-time: a stage sum is straight-line code
// whose loads are all independent and issue back to back.  Read from memory instead
// (add_terms, coef_update in rks_kernels.h), each term is a run of uniform branches with
// its own wait, about 90 dependent round trips per n = 8192 ETD35 attempt, and the
// allocator spills around them (1104 bytes of scratch per lane in FP64).  Only the methods
// and storage kinds that the workloads run are compiled this way (method_variant, rks_host.hip).
#pragma once
#include <utility>

#include "rks_math.h"
#include "rks_tableau.h"

// generic kernels: the tableau read from memory, every method and storage kind
#define RKS_METH_ANY (-1)

template <int METH, int ES, int NS, bool REAL>
struct MethodTab {
  static constexpr rks_tableau tab = rks_tab::with_layout(METH, ES, NS, REAL);
};

// Global-memory accesses by 32-bit index from a wave-uniform base pointer.  A pointer
// read from a record is generic, and a generic ("flat") access counts as an LDS access
// too: every wait for an LDS exchange would also wait for the loads in flight.
template <typename R>
struct GVec;
template <>
struct GVec<double> {
  typedef double t __attribute__((ext_vector_type(2), may_alias));
};
template <>
struct GVec<float> {
  typedef float t __attribute__((ext_vector_type(2), may_alias));
};
#define RKS_AS1 __attribute__((address_space(1)))

template <typename R>
__device__ __forceinline__ cx<R> gload(const cx<R>* p, int i) {
  typedef typename GVec<R>::t V;
  const V v = ((RKS_AS1 const V*)(unsigned long long)p)[(unsigned)i];
  return mkc((R)v.x, (R)v.y);
}
template <typename R>
__device__ __forceinline__ R gload_real(const R* p, int i) {
  return ((RKS_AS1 const R*)(unsigned long long)p)[(unsigned)i];
}
template <typename R>
__device__ __forceinline__ void gstore(cx<R>* p, int i, cx<R> v) {
  typedef typename GVec<R>::t V;
  V w;
  w.x = v.re;
  w.y = v.im;
  ((RKS_AS1 V*)(unsigned long long)p)[(unsigned)i] = w;
}

// a wave-uniform value kept in scalar registers
template <typename P>
__device__ __forceinline__ P* uni(P* p) {
  const unsigned long long v = (unsigned long long)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
  return (P*)(((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ double uni(double d) {
  const unsigned long long v = __builtin_bit_cast(unsigned long long, d);
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Coefficient array C of TT at index i (complex, or real where the lin_op is real).
template <typename TT, int C, typename RS, typename RN>
struct CoefOf {
  static constexpr int KIND = TT::tab.coef_rs[C];
  static constexpr int OFF = TT::tab.coef_off[C];
  static constexpr bool REAL = KIND == RKS_CST_RS_REAL || KIND == RKS_CST_RN_REAL;
  static __device__ __forceinline__ auto load(const char* cbase, size_t M, int i) {
    const char* q = cbase + (size_t)OFF * M;
    if constexpr (KIND == RKS_CST_RS) return gload((const cx<RS>*)q, i);
    else if constexpr (KIND == RKS_CST_RN) return cvt<RS>(gload((const cx<RN>*)q, i));
    else if constexpr (KIND == RKS_CST_RS_REAL) return gload_real((const RS*)q, i);
    else return (RS)gload_real((const RN*)q, i);
  }
};

// products rounded on their own (never fused into a following sum)
template <typename R>
__device__ __forceinline__ cx<R> scaled(R s, cx<R> v) {
#pragma clang fp contract(off)
  return mkc(s * v.re, s * v.im);
}
template <typename R>
__device__ __forceinline__ R scaled_re(R s, R w) {
#pragma clang fp contract(off)
  return s * w;
}
template <typename R>
__device__ __forceinline__ R add_re(R a, R b) {
#pragma clang fp contract(off)
  return a + b;
}
template <typename R>
__device__ __forceinline__ cx<R> times(R s, cx<R> v) {
  return scaled(s, v);
}
template <typename R>
__device__ __forceinline__ R times(R s, R w) {
  return scaled_re(s, w);
}
template <typename R>
__device__ __forceinline__ cx<R> times(cx<R> w, cx<R> v) {
#pragma clang fp contract(off)
  if constexpr (sizeof(R) == sizeof(double)) return w * v;
  else return mkc(fma(w.re, v.re, -(w.im * v.im)), fma(w.im, v.re, w.re * v.im));
}

// NL values read by the stage sums: those of slot NEW are still in the registers `nv`
// (the evaluation just before), the others come from memory.
template <typename TT, int SLOT, int NEW, typename RS, typename RN, int MPT, typename SlotF>
__device__ __forceinline__ cx<RS> nl_value(const cx<RN> (&nv)[MPT], SlotF slotp, int k, int m) {
  if constexpr (SLOT == NEW) return cvt<RS>(nv[k]);
  else return cvt<RS>(gload(slotp(SLOT), m));
}

// term J of stage S (S = -1: of the error estimate), in the grouping of rks_term
template <typename TT, int S, int J>
constexpr rks_term term_of() {
  return S < 0 ? TT::tab.err[J] : TT::tab.st[S < 0 ? 0 : S].t[J];
}

// acc[0..CH) (+)= term J at the modes of slots K0 .. K0 + CH - 1
template <typename TT, int S, int J, int NEW, int K0, int CH, bool FIRST, typename RS, typename RN, int MPT, typename OW,
          typename SlotF>
__device__ __forceinline__ void add_term(cx<RS> (&acc)[CH], const cx<RN> (&nv)[MPT], const OW& ow, SlotF slotp,
                                         const char* cbase, size_t Mc, double h) {
  // every product and sum rounded as in the general kernels, whose branches keep the
  // products apart from the sums, so both give the same bits
#pragma clang fp contract(off)
  constexpr rks_term tm = term_of<TT, S, J>();
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int k = K0 + i, m = ow.m(k);
    cx<RS> v = nl_value<TT, tm.src, NEW, RS, RN>(nv, slotp, k, m);
    if constexpr (tm.src2 >= 0) {
      const cx<RS> v2 = nl_value<TT, (tm.src2 >= 0 ? tm.src2 : 0), NEW, RS, RN>(nv, slotp, k, m);
      v = mkc(fma((RS)tm.scale2, v2.re, v.re), fma((RS)tm.scale2, v2.im, v.im));
    }
    if constexpr (tm.hmode == 2) {
      v = scaled((RS)((tm.scale * h) / tm.den), v);
    } else {
      if constexpr (tm.coef >= 0) {
        const auto w = CoefOf<TT, (tm.coef >= 0 ? tm.coef : 0), RS, RN>::load(cbase, Mc, ow.c(k));
        if constexpr (tm.hmode == 1) v = times(times((RS)h, w), v);
        else v = times(w, v);
      } else if constexpr (tm.hmode == 1) {
        v = scaled((RS)h, v);
      }
      if constexpr (tm.scale != 1.0) v = scaled((RS)tm.scale, v);
    }
    acc[i] = FIRST ? v : mkc(acc[i].re + v.re, acc[i].im + v.im);
  }
}

template <typename TT, int S, int NEW, int K0, int CH, bool HSUM, typename RS, typename RN, int MPT, typename OW,
          typename SlotF, int... J>
__device__ __forceinline__ void add_all(cx<RS> (&acc)[CH], const cx<RN> (&nv)[MPT], const OW& ow, SlotF slotp,
                                        const char* cbase, size_t Mc, double h, std::integer_sequence<int, J...>) {
  (add_term<TT, S, J, NEW, K0, CH, HSUM && J == 0>(acc, nv, ow, slotp, cbase, Mc, h), ...);
}

// E u of stage S at slots K0 .. K0 + CH - 1
template <typename TT, int S, int K0, int CH, typename RS, typename RN, typename OW>
__device__ __forceinline__ void load_eu(cx<RS> (&acc)[CH], const cx<RS>* u, const OW& ow, const char* cbase, size_t Mc) {
  constexpr int EC = TT::tab.st[S].ecoef;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    acc[i] = gload(u, ow.m(K0 + i));
    if constexpr (EC >= 0) acc[i] = times(CoefOf<TT, (EC >= 0 ? EC : 0), RS, RN>::load(cbase, Mc, ow.c(K0 + i)), acc[i]);
  }
}

// Argument of stage S into acc (every slot of the thread), CH slots at a time so that one
// chunk's loads, not all of them, are in flight in registers.
template <typename TT, int S, int NEW, int K0, int CHMAX, typename RS, typename RN, int MPT, typename OW, typename SlotF>
__device__ __forceinline__ void stage_sum(cx<RS> (&acc)[MPT], const cx<RN> (&nv)[MPT], const cx<RS>* u, const OW& ow,
                                          SlotF slotp, const char* cbase, size_t Mc, double h) {
  if constexpr (K0 < MPT) {
    constexpr int CH = MPT - K0 <= CHMAX + 1 ? MPT - K0 : CHMAX;
    const OW of = ow.fresh();
    __builtin_amdgcn_sched_barrier(0);
    constexpr int NT = TT::tab.st[S].nterm;
    using JS = std::make_integer_sequence<int, NT>;
    cx<RS> a[CH];
    load_eu<TT, S, K0, CH, RS, RN>(a, u, of, cbase, Mc);
    if constexpr (TT::tab.st[S].hsum != 0) {
      cx<RS> sum[CH];
      add_all<TT, S, NEW, K0, CH, true>(sum, nv, of, slotp, cbase, Mc, h, JS{});
#pragma unroll
      for (int i = 0; i < CH; ++i) a[i] = mkc(fma((RS)h, sum[i].re, a[i].re), fma((RS)h, sum[i].im, a[i].im));
    } else {
      add_all<TT, S, NEW, K0, CH, false>(a, nv, of, slotp, cbase, Mc, h, JS{});
    }
#pragma unroll
    for (int i = 0; i < CH; ++i) acc[K0 + i] = a[i];
    stage_sum<TT, S, NEW, K0 + CH, CHMAX>(acc, nv, u, ow, slotp, cbase, Mc, h);
  }
}

// Modes per chunk of the literal stage sums: what a chunk loads is in flight in registers
// together (up to 12 values per mode), beside the stage value and the last NL value.
template <typename R>
__host__ __device__ constexpr int rks_sum_chunk() {
  return sizeof(R) == 4 ? 8 : 4;
}

// Argument of stage s (uniform), CH modes at a time (0: rks_sum_chunk).  KEEP: the NL values
// of the stage before are in nv.
template <typename TT, int S, bool KEEP, int CH = 0, typename RS, typename RN, int MPT, typename OW, typename SlotF>
__device__ __forceinline__ void stage_switch(int s, cx<RS> (&acc)[MPT], const cx<RN> (&nv)[MPT], const cx<RS>* u,
                                             const OW& ow, SlotF slotp, const char* cbase, size_t Mc, double h) {
  constexpr int LAST = TT::tab.nstage - (TT::tab.st[TT::tab.nstage - 1].has_nl ? 1 : 2);
  constexpr int NEW = (KEEP && S > 0) ? TT::tab.st[S > 0 ? S - 1 : 0].nl_slot : -1;
  if constexpr (S < LAST) {
    if (s != S) {
      stage_switch<TT, S + 1, KEEP, CH>(s, acc, nv, u, ow, slotp, cbase, Mc, h);
      return;
    }
  }
  stage_sum<TT, S, NEW, 0, CH != 0 ? CH : rks_sum_chunk<RS>()>(acc, nv, u, ow, slotp, cbase, Mc, h);
}

// embedded error estimate at slots K0 .. K0 + CH - 1
template <typename TT, int NEW, int K0, int CH, typename RS, typename RN, int MPT, typename OW, typename SlotF>
__device__ __forceinline__ void error_sum(cx<RS> (&ev)[CH], const cx<RN> (&nv)[MPT], const OW& ow, SlotF slotp,
                                          const char* cbase, size_t Mc, double h) {
  add_all<TT, -1, NEW, K0, CH, true>(ev, nv, ow, slotp, cbase, Mc, h,
                                     std::make_integer_sequence<int, TT::tab.nerr>{});
  if constexpr (TT::tab.err_factored != 0) {
    constexpr int EC = TT::tab.err_coef;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      if constexpr (TT::tab.err_hpow != 0) ev[i] = scaled((RS)h, ev[i]);
      if constexpr (TT::tab.err_scale != 1.0) ev[i] = scaled((RS)TT::tab.err_scale, ev[i]);
      if constexpr (EC >= 0) ev[i] = times(CoefOf<TT, (EC >= 0 ? EC : 0), RS, RN>::load(cbase, Mc, ow.c(K0 + i)), ev[i]);
    }
  }
}

// Last stage and error estimate, then the values of the masked norm per mode (FP64): |u_new|
// and |err|^2 where the last stage has no NL (FP32: |u_new| and |err|, rounded to FP32; a
// square would flush to zero below ~1e-19), else |u_new|^2 and |err|^2.  A method whose last
// stage has no NL (ETD35) forms both from the same NL values;
// LAST_NL: the candidate is already stored (it went through the last NL evaluation).
template <typename TT, int NEW, int K0, int CHMAX, bool LAST_NL, typename RS, typename RN, int MPT, typename OW,
          typename SlotF>
__device__ __forceinline__ void final_sum(double (&a2)[MPT], double (&e2)[MPT], cx<RS>* cand, const cx<RN> (&nv)[MPT],
                                          const cx<RS>* u, const OW& ow, SlotF slotp, const char* cbase, size_t Mc,
                                          double h) {
#pragma clang fp contract(off)
  if constexpr (K0 < MPT) {
    constexpr int CH = MPT - K0 <= CHMAX + 1 ? MPT - K0 : CHMAX;
    constexpr int S = TT::tab.nstage - 1;
    const OW of = ow.fresh();
    __builtin_amdgcn_sched_barrier(0);
    cx<RS> a[CH], ev[CH];
    if constexpr (LAST_NL) {
#pragma unroll
      for (int i = 0; i < CH; ++i) a[i] = gload(cand, of.m(K0 + i));
    } else {
      load_eu<TT, S, K0, CH, RS, RN>(a, u, of, cbase, Mc);
      add_all<TT, S, NEW, K0, CH, false>(a, nv, of, slotp, cbase, Mc, h,
                                         std::make_integer_sequence<int, TT::tab.st[S].nterm>{});
    }
    error_sum<TT, NEW, K0, CH>(ev, nv, of, slotp, cbase, Mc, h);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int k = K0 + i;
      const double ar = (double)a[i].re, ai = (double)a[i].im, er = (double)ev[i].re, ei = (double)ev[i].im;
      const bool ok = of.ok(k);
      if constexpr (!LAST_NL) {
        if (ok) gstore(cand, of.m(k), a[i]);
      }
      double x, y = fma(er, er, ei * ei);
      if constexpr (LAST_NL) {
        x = fma(ar, ar, ai * ai);
      } else {
        x = hypot(ar, ai);
        if constexpr (sizeof(RS) < sizeof(double)) {
          x = (double)(float)x;
          y = (double)(float)hypot(er, ei);
        }
      }
      a2[k] = ok ? x : 0.0;
      e2[k] = ok ? y : 0.0;
    }
    final_sum<TT, NEW, K0 + CH, CHMAX, LAST_NL>(a2, e2, cand, nv, u, ow, slotp, cbase, Mc, h);
  }
}

// ---------------------------------------------------------------------------
// coefficient generator: the recipes of coef_update (rks_kernels.h) as literals, the same
// operations in the same order
// ---------------------------------------------------------------------------
template <typename TT, int C, typename RS, typename RN>
__device__ __forceinline__ void coef_recipe(const z64 (&v)[4], double h, int m, size_t M, char* cbase) {
#pragma clang fp contract(off)
  constexpr rks_coef cf = TT::tab.coef[C];
  constexpr int kind = TT::tab.coef_rs[C];
  constexpr bool cplx = TT::tab.uses_contour || kind == RKS_CST_RS || kind == RKS_CST_RN;
  z64 acc = mkc(0.0, 0.0);
#pragma unroll
  for (int k = 0; k < cf.nb; ++k) {
    const double w = cf.hmul ? cf.w[k] * h : cf.w[k];
    const z64 t = (w == 1.0) ? v[cf.kind[k]] : np_rmul(w, v[cf.kind[k]]);
    acc = (k == 0) ? t : mkc(acc.re + t.re, acc.im + t.im);
  }
  if constexpr (cf.outer != 1.0) acc = np_rmul(cf.outer, acc);
  if constexpr (cf.den != 1.0) {
    if constexpr (cplx) acc = np_rdiv(acc, cf.den);
    else acc = mkc(acc.re / cf.den, acc.im / cf.den);
  }
  char* p = cbase + (size_t)TT::tab.coef_off[C] * M;
  if constexpr (kind == RKS_CST_RS) gstore((cx<RS>*)p, m, mkc((RS)acc.re, (RS)acc.im));
  else if constexpr (kind == RKS_CST_RN) gstore((cx<RN>*)p, m, mkc((RN)acc.re, (RN)acc.im));
  else if constexpr (kind == RKS_CST_RS_REAL) ((RS*)p)[m] = (RS)acc.re;
  else ((RN*)p)[m] = (RN)acc.re;
}

template <typename TT, int F, typename RS, typename RN, int... C>
__device__ __forceinline__ void coef_recipes(const z64 (&v)[4], double h, int m, size_t M, char* cbase,
                                             std::integer_sequence<int, C...>) {
  ((TT::tab.coef[C].frac == F ? coef_recipe<TT, C, RS, RN>(v, h, m, M, cbase) : (void)0), ...);
}

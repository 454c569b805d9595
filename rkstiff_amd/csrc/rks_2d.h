// Batched engine for 2-D periodic problems on an N x N rfft2 grid.
//
// Layout: NumPy's rfft2 order, row-major [ky][kx] with kx = 0..N/2, so an
// instance has M = N (N/2 + 1) modes; the reference flattens it to a 1-D
// diagonal lin_op (solver.py:129-135, demos/allen_cahn.ipynb).  Built-in term
// (Allen-Cahn): nl(u) = rfft2(w - c w^3), w = irfft2(u).
//
// One trajectory does not fit one workgroup's LDS (512 x 257 complex), so an
// attempt is a fixed sequence of kernels over all trajectories, each one pass
// over HBM:
//   col   forward column FFTs of the previous stage's transform buffer T
//         -> NL slot; the next stage combination E u + sum C NL; inverse
//         column FFTs -> T, all in registers (CG adjacent columns per
//         workgroup, so every row segment read or written is contiguous)
//   row   per pair of rows: one complex inverse FFT of both rows' half
//         spectra, w - c w^3 on the real and imaginary parts, one forward
//         FFT, split into the two rows' half spectra (in place in T)
//   norm  masked sums of the embedded error norm (solveras.py:449-455),
//         FP64 partials per workgroup
//   ctrl  FP64 accept/reject and dt per trajectory (solveras.py:384-410,
//         457-554; evolve 605-650), and the start of the next attempt
// ctrl/snap keep each trajectory's own controller state, so finished
// or rejected trajectories drop out of (or repeat) work per launch while the
// others advance.  The host captures the sequence once into a hipGraph and
// replays it until no trajectory is running.
#pragma once
#include "rks_2d_host.h"
#include "rks_kernels.h"

#define NLK_AC2D 3

// per-trajectory flags of the current attempt
struct rks2_state {
  int active;     // takes part in this attempt
  int need_nl1;   // NL1 = nl(u) first (start, or RECOMPUTE after an accept)
  int need_coef;  // h changed: regenerate coefficient arrays
  int store;      // copy the current state to snapshot snap_idx
  int snap_idx;
  int pad;
};

struct rks2_launch {
  const rks_tableau* tab;
  const rks_ctrl* ctl;
  rks_inst* inst;
  const rks_io* io;
  rks2_state* st;
  const void* tw;    // exp(-2 pi i x / N), x < N, state precision
  double* pmax;      // [ninst][ncg] partial max |u_new|
  double* psum;      // [ninst][nnb][2] partial masked sums
  int* active_count;
  size_t off_cand0, off_cand1, off_coef, off_T;  // byte offsets in an instance workspace
  int ninst, mode, ncg, nnb;
  int lowp;  // NL arrays stored in FP32
};

template <typename R, int LOG2>
struct Geo2 {
  static constexpr int N = 1 << LOG2;
  static constexpr int NXH = N / 2 + 1;
  static constexpr int M = N * NXH;  // modes (the caller's rfft2 layout, row stride NXH)
  // internal arrays (NL slots, candidates, coefficients): row stride XS
  static constexpr int XS = rks2_istride(N);
  static constexpr int MI = N * XS;
  // row stride of the transform buffer T (elements): whole 128-byte lines, so
  // a column tile's row segments do not straddle cache lines
  static constexpr int TXS = rks2_t_stride(N, (int)sizeof(cx<R>));
  static constexpr int PS = rksfft::padded_size(N);
  // column kernel: consecutive lanes hold the same element of CG columns, then the next
  // element; a buffer stride of 4 modulo 32 (FP64: 2 modulo 16) elements spreads both over
  // the banks
  static constexpr int CBM = sizeof(R) == 4 ? 32 : 16, CBR = sizeof(R) == 4 ? 4 : 2;
  static constexpr int CPS = PS + (CBM + CBR - PS % CBM) % CBM;
  static constexpr int TWS = rksfft::TwSplit<LOG2>::SIZE;
  // column kernel: CG columns of N points, CTG threads per column
  static constexpr int CG = sizeof(R) == 4 ? 16 : 8;
  // At least four points a thread, for fewer passes on short columns: 8 x 64^2 ETD35 FP64 3.4 ms
  // with two (radix 2 throughout), 2.7 with four, 3.1 with eight (too few waves); 128^2 3.37,
  // 3.22, 3.38
  static constexpr int CTG = (N / 4 < 512 / CG) ? N / 4 : 512 / CG;
  static constexpr int CT = CG * CTG;
  static constexpr int CEPT = N / CTG;  // tile elements per thread
  // modes per chunk of the stage combination: 4 in FP64 keeps the column
  // kernel within 128 VGPRs without spills (two workgroups per CU, LDS-bound)
  static constexpr int CCH_MAX = sizeof(R) == 4 ? 8 : 4;
  static constexpr int CCH = CEPT < CCH_MAX ? CEPT : CCH_MAX;
  static constexpr int NCG = (NXH + CG - 1) / CG;
  static constexpr int COL_LDS = (CG * CPS + TWS) * (int)sizeof(cx<R>);
  // row kernel: RG complex transforms (2 RG rows), RTG threads each (N = 512:
  // 64 threads, 8 points each, three radix-8 passes)
  static constexpr int RG = 8;
  static constexpr int RTG = (N / 4 < 512 / RG) ? N / 4 : 512 / RG;
  static constexpr int RT = RG * RTG;
  static constexpr int NRG = N / (2 * RG);
  static constexpr int ROW_LDS = (RG * PS + TWS) * (int)sizeof(cx<R>);
  // norm kernel
  // mirror-symmetric lin_op (L[r][c] == L[n - r][c]): coefficients of rows
  // 0..n/2 in arrays of stride MSYM (a multiple of 64 modes)
  static constexpr int MGEN_SYM = (N / 2 + 1) * NXH;            // caller layout
  static constexpr int MGEN_SYM_I = (N / 2 + 1) * XS;            // internal layout
  static constexpr int MSYM = ((MGEN_SYM_I + 63) / 64) * 64 < MI ? ((MGEN_SYM_I + 63) / 64) * 64 : MI;
  static constexpr int NT = 256, NE = 8;
  static constexpr int NNB = (M + NT * NE - 1) / (NT * NE);
  static_assert(N >= 2 * RG, "grid too small for the row kernel");
  static_assert(CEPT >= 2, "column transform needs two elements per thread");
};

__device__ __forceinline__ unsigned rks2_smap(const rks_inst* in) {
  unsigned smap = 0;
#pragma unroll
  for (int s = 0; s < RKS_MAX_SLOTS; ++s) smap |= (unsigned)(in->slot_map[s] & 15) << (4 * s);
  return smap;
}

// current state and candidate buffer of an instance (internal layout).  An
// evolve or step starts by copying the caller's u0 into cand0 (k2_in); a step
// attempts from cand0 into cand1, which k2_out copies to the caller.  The
// nonlinear-term mode reads the caller's u (its layout) directly.
template <typename R>
__device__ __forceinline__ void rks2_states(const rks2_launch& P, const rks_inst* in, const rks_io& io,
                                            const cx<R>** u, cx<R>** cand) {
  char* ws = (char*)in->ws;
  cx<R>* c0 = (cx<R>*)(ws + P.off_cand0);
  cx<R>* c1 = (cx<R>*)(ws + P.off_cand1);
  if (P.mode == RKS_MODE_EVOLVE) {
    const int ub = in->ubuf;
    *u = ub == 1 ? c1 : c0;
    *cand = ub == 1 ? c0 : c1;
  } else if (P.mode == RKS_MODE_STEP) {
    *u = c0;
    *cand = c1;
  } else {
    *u = (const cx<R>*)io.u_in;
    *cand = nullptr;
  }
}

// ---------------------------------------------------------------------------
// col: [forward column FFTs of T -> NL slot fwd_slot] then [argument of stage
// `arg` (arg == -1: u itself; arg == -2: none) -> candidate (last stage) and/or
// inverse column FFTs -> T].  fwd_need_nl1: the forward part only for
// trajectories that evaluated NL1 in this attempt; prelude: the whole kernel
// only for those.
// ---------------------------------------------------------------------------
// Launch bounds ask for 4 waves per SIMD (<= 128 VGPRs): with ~70 KB of LDS
// per workgroup at N = 512, two workgroups share a CU.
// FUSE (the last stage of a method whose error estimate reads the same NL
// slots, rks_fused_final): the candidate and the embedded error come from one
// load of each NL value; |u_new| and |err|^2 (FP32: |err|) per mode go to T,
// idle at that point, for k2_norm_fused.  A separate instantiation, so the
// other stages keep their register allocation (no spills at 4 waves per SIMD).
// METH: the stage sums of one method as literals (rks_method.h), else the tableau.
// A thread holds rows r0 + i CTG of one column from the load of T to its store: both
// transforms take their first inputs from and leave their results in registers (chain_reg),
// the NL values just formed enter the next stage sum without a trip to memory, and only the
// exchanges between the transforms' passes go through LDS.  What bounds a pass then is HBM:
// 64 x 512^2 ETD35 FP32, 0.5 GB for a middle stage.  Batches, one evolve, tableau read from
// memory / literal sums with transforms from LDS to LDS / in registers:
//   64 x 512^2 FP32, tf = 4    75.2 / 60.7 / 55.8 ms    8 x 128^2 FP64, tf = 4   10.3 / 6.6 / 5.4 ms
//   32 x 512^2 FP64, tf = 2    41.3 / - / 23.5 ms
// The generic kernels (METH = RKS_METH_ANY) form their stage sums over mirror row pairs and
// pass them to the transform's rows through LDS.

// Modes of the literal stage sums: slot k holds row row[k] of a column; coefficients of the
// mirror row where L is mirror-symmetric.
template <int N, int XS, int CH>
struct OwnRows {
  int row[CH];
  int col, sym;
  bool valid;
  __device__ __forceinline__ bool ok(int) const { return valid; }
  __device__ __forceinline__ int m(int k) const { return valid ? row[k] * XS + col : 0; }
  __device__ __forceinline__ int c(int k) const {
    const int r = (sym && row[k] > N / 2) ? N - row[k] : row[k];
    return valid ? r * XS + col : 0;
  }
  __device__ __forceinline__ OwnRows fresh() const { return *this; }
};

template <typename R, typename RN, int LOG2, bool FUSE, int METH>
__global__ __launch_bounds__((Geo2<R, LOG2>::CT), 4) void k2_col(rks2_launch P, int fwd_slot, int fwd_need_nl1,
                                                            int arg, int prelude) {
  using G = Geo2<R, LOG2>;
  using C = cx<R>;
  using CN = cx<RN>;
  using rksfft::pad;
  constexpr int N = G::N, NXH = G::NXH, XS = G::XS, MI = G::MI, CG = G::CG, CT = G::CT, CEPT = G::CEPT;
  // the fused last stage keeps the candidate and the error per mode: half the chunk
  constexpr int CH = (FUSE && G::CCH >= 4) ? G::CCH / 2 : G::CCH, NCH = CEPT / CH, RS = CT / CG, PS = G::CPS;
  extern __shared__ __align__(16) unsigned char rks2_smem[];
  __shared__ double red[2 * (CT / 64 + 1)];
  const int inst = blockIdx.y;
  const rks2_state st = P.st[inst];
  if (!st.active || (prelude && !st.need_nl1)) return;
  C* buf = (C*)rks2_smem;
  C* twl = buf + CG * PS;
  const rks_tableau& tb = *P.tab;
  rks_inst* in = P.inst + inst;
  const rks_io& io = P.io[inst];
  char* ws = uni((char*)in->ws);
  const double h = uni(in->h);
  const unsigned smap = (unsigned)uni((int)rks2_smap(in));
  CN* const slot_base = (CN*)ws;
  auto slot = [&](int s) -> CN* { return slot_base + (size_t)((smap >> (4 * s)) & 15u) * MI; };
  const C* u;
  C* cand;
  rks2_states<R>(P, in, io, &u, &cand);
  u = uni(u);
  cand = uni(cand);
  const int ustride = P.mode == RKS_MODE_NL ? NXH : XS;  // the caller's u in the nonlinear-term mode
  C* Tb = (C*)(ws + P.off_T);
  const char* cbase = ws + P.off_coef;
  rksfft::load_twiddles<R, LOG2, CT>(twl, (const C*)P.tw);
  const int t = threadIdx.x, c = t % CG, r0 = t / CG;
  const int col = blockIdx.x * CG + c;
  const bool valid = col < NXH;
  C* const bc = buf + c * PS;
  const C zero = mkc((R)0, (R)0);
  __syncthreads();
  constexpr bool METHOD = METH != RKS_METH_ANY;
  using TT = MethodTab<METHOD ? METH : 0, (int)sizeof(C), (int)sizeof(CN), true>;
  // the last NL values of a method that recomputes NL1 are only read by this very pass
  constexpr bool KEEP_LAST = !(FUSE && METHOD && TT::tab.nl1_policy == RKS_NL1_RECOMPUTE);
  C w[CEPT];  // rows r0 + i RS: NL values, then the stage argument
#pragma unroll
  for (int i = 0; i < CEPT; ++i) w[i] = zero;
  if (fwd_slot >= 0 && (!fwd_need_nl1 || st.need_nl1)) {
#pragma unroll
    for (int i = 0; i < CEPT; ++i) w[i] = valid ? Tb[(r0 + i * RS) * G::TXS + col] : zero;
    rksfft::chain_reg<R, N, G::CTG, 1, false, LOG2, 1, RKS_MAXR, false, 0, true>(w, bc, twl, r0, [](C z) { return z; });
    if (valid) {
      if (P.mode == RKS_MODE_NL) {
        C* dst = (C*)io.u_out;
#pragma unroll
        for (int i = 0; i < CEPT; ++i) dst[(r0 + i * RS) * NXH + col] = w[i];
      } else if (KEEP_LAST) {
        CN* dst = slot(fwd_slot);
#pragma unroll
        for (int i = 0; i < CEPT; ++i) gstore(dst, (r0 + i * RS) * XS + col, cvt<RN>(w[i]));
      }
    }
  }
  if (arg < -1) return;
  if constexpr (!METHOD) __syncthreads();  // the rows below are other threads'
  const bool has_nl = arg < 0 || tb.st[arg].has_nl;
  const bool last = arg >= 0 && arg == tb.nstage - 1;
  const int sym = in->coef_sym;
  const size_t Mc = sym ? G::MSYM : MI;
  const bool fused = FUSE && last;
  double mx = 0.0;
  if constexpr (METHOD) {
    // the thread's own rows r0 + i RS, whose NL values of the stage before are still in w
    CN nv[CEPT];
#pragma unroll
    for (int i = 0; i < CEPT; ++i) nv[i] = cvt<RN>(w[i]);
    if constexpr (FUSE) {
      constexpr int NEW = TT::tab.st[TT::tab.nstage > 1 ? TT::tab.nstage - 2 : 0].nl_slot;
#pragma unroll
      for (int ch = 0; ch < NCH; ++ch) {
        OwnRows<N, XS, CH> ow;
        CN nc[CH];
#pragma unroll
        for (int i = 0; i < CH; ++i) {
          ow.row[i] = r0 + (ch * CH + i) * RS;
          nc[i] = nv[ch * CH + i];
        }
        ow.col = col;
        ow.sym = sym;
        ow.valid = valid;
        double a[CH], e[CH];
        final_sum<TT, NEW, 0, CH, false>(a, e, cand, nc, u, ow, slot, cbase, Mc, h);
#pragma unroll
        for (int i = 0; i < CH; ++i) {
          if (!valid) continue;
          gstore(Tb, ow.row[i] * G::TXS + col, mkc((R)a[i], (R)e[i]));
          mx = nanmax(mx, a[i]);
        }
      }
    } else if (arg < 0) {
#pragma unroll
      for (int i = 0; i < CEPT; ++i) w[i] = valid ? gload(u, (r0 + i * RS) * ustride + col) : zero;
    } else {
      OwnRows<N, XS, CEPT> ow;
#pragma unroll
      for (int i = 0; i < CEPT; ++i) ow.row[i] = r0 + i * RS;
      ow.col = col;
      ow.sym = sym;
      ow.valid = valid;
      stage_switch<TT, 0, true, G::CCH>(arg, w, nv, u, ow, slot, cbase, Mc, h);
#pragma unroll
      for (int i = 0; i < CEPT; ++i) {
        if (last && valid) {
          gstore(cand, ow.m(i), w[i]);
          mx = nanmax(mx, hypot((double)w[i].re, (double)w[i].im));
        }
        if (!valid) w[i] = zero;
      }
    }
  } else {
    // over mirror row pairs: slot 2j row q = r0 + (ch CH/2 + j) RS, slot 2j + 1 row n - q
    // (n/2 for q = 0), so a mirror-symmetric L shares coefficients
#pragma unroll 1
    for (int ch = 0; ch < NCH; ++ch) {
      ChunkIdx<CH> ix;
      int row[CH];
      ix.sym = sym;
      ix.lim = G::MGEN_SYM_I;
      ix.anyq = 0;
#pragma unroll
      for (int j = 0; j < CH / 2; ++j) {
        const int q = r0 + (ch * (CH / 2) + j) * RS;
        row[2 * j] = q;
        row[2 * j + 1] = q == 0 ? N / 2 : N - q;
        ix.m[2 * j] = valid ? row[2 * j] * XS + col : 0;
        ix.m[2 * j + 1] = valid ? row[2 * j + 1] * XS + col : 0;
        ix.ok[2 * j] = ix.ok[2 * j + 1] = valid;
      }
      C acc[CH];
      if (arg < 0) {
#pragma unroll
        for (int i = 0; i < CH; ++i) acc[i] = valid ? u[row[i] * ustride + col] : zero;
      } else if (fused) {
        if constexpr (FUSE) {
          C ev[CH];
          final_chunk<R, RN, CH>(tb, u, slot, cbase, Mc, ix, h, acc, ev);
#pragma unroll
          for (int i = 0; i < CH; ++i) {
            if (valid) {
              const double a = hypot((double)acc[i].re, (double)acc[i].im);
              const double er = (double)ev[i].re, ei = (double)ev[i].im;
              if constexpr (sizeof(R) == sizeof(double))
                Tb[row[i] * G::TXS + col] = mkc((R)a, (R)(er * er + ei * ei));
              else
                Tb[row[i] * G::TXS + col] = mkc((R)a, (R)hypot(er, ei));
            }
          }
        }
      } else {
        stage_chunk<R, RN, CH>(tb, tb.st[arg], u, slot, cbase, Mc, ix, h, acc);
      }
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        if (last && valid) {
          cand[ix.m[i]] = acc[i];
          mx = nanmax(mx, hypot((double)acc[i].re, (double)acc[i].im));
        }
        if (has_nl) bc[pad(row[i])] = valid ? acc[i] : zero;
      }
    }
    if (has_nl) {
      __syncthreads();
#pragma unroll
      for (int i = 0; i < CEPT; ++i) w[i] = bc[pad(r0 + i * RS)];
      __syncthreads();
    }
  }
  if (last && tb.adaptive) {
    mx = wg_max<CT>(mx, red);
    if (t == 0) P.pmax[inst * P.ncg + blockIdx.x] = mx;
  }
  if (has_nl) {
    rksfft::chain_reg<R, N, G::CTG, 1, true, LOG2, 1, RKS_MAXR, false, 0, true>(w, bc, twl, r0, [](C z) { return z; });
    if (valid) {
#pragma unroll
      for (int i = 0; i < CEPT; ++i) gstore(Tb, (r0 + i * RS) * G::TXS + col, w[i]);
    }
  }
}

// ---------------------------------------------------------------------------
// row: irfft along rows, w - c w^3, rfft along rows; two rows per complex
// transform (z = w1 + i w2).  T holds the column-inverse-transformed spectrum
// and is overwritten in place with the rows' forward spectra.
// ---------------------------------------------------------------------------
template <typename R, int LOG2>
__global__ __launch_bounds__((Geo2<R, LOG2>::RT)) void k2_row(rks2_launch P, int prelude) {
  using G = Geo2<R, LOG2>;
  using C = cx<R>;
  using rksfft::pad;
  constexpr int N = G::N, NXH = G::NXH, RG = G::RG, RT = G::RT, PS = G::PS;
  extern __shared__ __align__(16) unsigned char rks2_smem[];
  const int inst = blockIdx.y;
  const rks2_state st = P.st[inst];
  if (!st.active || (prelude && !st.need_nl1)) return;
  C* buf = (C*)rks2_smem;
  C* twl = buf + RG * PS;
  const rks_inst* in = P.inst + inst;
  C* Tb = (C*)((char*)in->ws + P.off_T);
  const R c3 = (R)in->nl_coef;
  const R inv = (R)(1.0 / ((double)N * (double)N));  // irfft2 normalisation (exact)
  rksfft::load_twiddles<R, LOG2, RT>(twl, (const C*)P.tw);
  const int t = threadIdx.x;
  const int row0 = blockIdx.x * 2 * RG;
  for (int e = t; e < RG * NXH; e += RT) {
    const int g = e / NXH, k = e - g * NXH;
    const C a = Tb[(row0 + 2 * g) * G::TXS + k];
    const C b = Tb[(row0 + 2 * g + 1) * G::TXS + k];
    C* bg = buf + g * PS;
    // full spectrum of w1 + i w2 from the two half spectra; DC and Nyquist keep
    // only their real parts, as irfft does
    if (k == 0 || k == N / 2) {
      bg[pad(k)] = mkc(a.re, b.re);
    } else {
      bg[pad(k)] = mkc(a.re - b.im, a.im + b.re);
      bg[pad(N - k)] = mkc(a.re + b.im, b.re - a.im);
    }
  }
  __syncthreads();
  // both transforms and the pointwise term between them in registers (chain_reg): an exchange
  // through LDS per pass but the last, instead of one per pass and two around the term
  constexpr int RTG = G::RTG, EPT = N / RTG;
  const int q = t % RTG;
  C* const bq = buf + (t / RTG) * PS;
  C v[EPT];
#pragma unroll
  for (int k = 0; k < EPT; ++k) v[k] = bq[pad(q + k * RTG)];
  __syncthreads();
  rksfft::chain_reg<R, N, RTG, 1, true, LOG2, 1, RKS_MAXR, false, 0, true>(v, bq, twl, q, [&](C z) {
    const R w1 = z.re * inv, w2 = z.im * inv;
    return mkc(w1 - c3 * (w1 * w1 * w1), w2 - c3 * (w2 * w2 * w2));
  });
  rksfft::chain_reg<R, N, RTG, 1, false, LOG2, 1, RKS_MAXR, false, 0, true>(v, bq, twl, q, [](C z) { return z; });
#pragma unroll
  for (int k = 0; k < EPT; ++k) bq[pad(q + k * RTG)] = v[k];
  __syncthreads();
  for (int e = t; e < RG * NXH; e += RT) {
    const int g = e / NXH, k = e - g * NXH;
    const C* bg = buf + g * PS;
    const C z = bg[pad(k)];
    const C y = bg[pad((N - k) & (N - 1))];
    // Z = F1 + i F2 with F1, F2 Hermitian: F1 = (Z + conj Y)/2, F2 = (Z - conj Y)/(2i)
    const R hf = (R)0.5;
    Tb[(row0 + 2 * g) * G::TXS + k] = mkc((z.re + y.re) * hf, (z.im - y.im) * hf);
    Tb[(row0 + 2 * g + 1) * G::TXS + k] = mkc((z.im + y.im) * hf, (y.re - z.re) * hf);
  }
}

// ---------------------------------------------------------------------------
// coefficients (FP64 arithmetic) of trajectories whose h changed
// ---------------------------------------------------------------------------
template <typename R, typename RN, int LOG2, int METH>
__global__ __launch_bounds__(256) void k2_coef(rks2_launch P) {
  using G = Geo2<R, LOG2>;
  const int inst = blockIdx.y;
  if (inst == 0 && blockIdx.x == 0 && threadIdx.x == 0) *P.active_count = 0;  // k2_ctrl counts anew
  const rks2_state st = P.st[inst];
  if (!st.active || !st.need_coef) return;
  const rks_inst* in = P.inst + inst;
  char* cbase = uni((char*)in->ws) + P.off_coef;
  // mirror-symmetric L: rows 0..n/2 only (stride MSYM); lin_op in the caller's
  // layout, coefficients in the internal one
  const int Mg = in->coef_sym ? G::MGEN_SYM : G::M;
  const int Mc = in->coef_sym ? G::MSYM : G::MI;
  if constexpr (METH == RKS_METH_ANY) {
    for (int m = blockIdx.x * 256 + threadIdx.x; m < Mg; m += gridDim.x * 256) {
      const int r = m / G::NXH, c = m - r * G::NXH;
      coef_mode_at<R, RN>(*P.tab, *P.ctl, in->L, in->L_complex, m, r * G::XS + c, Mc, in->h, cbase);
    }
  } else {
    // literal recipes; a workgroup's few small modes (|z| < modecutoff), whose contour
    // means are 32 psi evaluations each, wait in a list and are spread over its lanes
    using TT = MethodTab<METH, (int)sizeof(cx<R>), (int)sizeof(cx<RN>), true>;
    __shared__ int list[256];
    __shared__ int count;
    rks_cctl& ct = *rks_uniform_const<rks_cctl>(P.ctl);
    const double* L = uni(in->L);
    const double h = uni(in->h);
    for (int m0 = blockIdx.x * 256; m0 < Mg; m0 += gridDim.x * 256) {
      const int m = m0 + (int)threadIdx.x;
      if constexpr (TT::tab.uses_contour != 0) {
        if (threadIdx.x == 0) count = 0;
        __syncthreads();
      }
      if (m < Mg) {
        const int r = m / G::NXH, c = m - r * G::NXH;
        const z64 z = mode_z(L, 0, m, h);
        if (TT::tab.uses_contour && hypot(z.re, z.im) < ct.modecutoff)
          list[atomicAdd(&count, 1)] = m;
        else
          method_fracs<TT, 0, R, RN>(
              [&](int fnum, int fden, int fmask, z64(&v)[4]) {
                frac_direct(fnum, fden, fmask, z, h, TT::tab.uses_contour, v);
              },
              h, r * G::XS + c, (size_t)Mc, cbase);
      }
      if constexpr (TT::tab.uses_contour != 0) {
        __syncthreads();
        const int nsmall = count;
        for (int idx = threadIdx.x / 32; idx < nsmall; idx += 256 / 32) {
          const int ms = list[idx], r = ms / G::NXH, c = ms - r * G::NXH;
          method_small<TT, 0, R, RN, 32, true>(ct, mode_z(L, 0, ms, h), threadIdx.x % 32, h, r * G::XS + c, (size_t)Mc,
                                               cbase);
        }
        __syncthreads();
      }
    }
  }
}


// Largest of the n partial maxima, the same in every lane: a lane per partial (one load, not
// n in a row).
__device__ __forceinline__ double rks2_max(const double* p, int n) {
  const int lane = threadIdx.x & 63;
  double mx = p[lane < n ? lane : 0];
  for (int j = lane + 64; j < n; j += 64) mx = nanmax(mx, p[j]);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) mx = nanmax(mx, __shfl_xor(mx, o, 64));
  return mx;
}

// ---------------------------------------------------------------------------
// norm: masked sums |u_new|^2, |err|^2 over modes with |u_new|/max > cutoff
// ---------------------------------------------------------------------------
template <typename R, typename RN, int LOG2>
__global__ __launch_bounds__(256) void k2_norm(rks2_launch P) {
  using G = Geo2<R, LOG2>;
  using C = cx<R>;
  using CN = cx<RN>;
  constexpr int MI = G::MI, NT = G::NT, NE = G::NE;
  __shared__ double red[2 * (NT / 64 + 1)];
  const int inst = blockIdx.y;
  const rks2_state st = P.st[inst];
  const rks_tableau& tb = *P.tab;
  if (!st.active || !tb.adaptive) return;
  const rks_inst* in = P.inst + inst;
  const rks_io& io = P.io[inst];
  char* ws = (char*)in->ws;
  const unsigned smap = rks2_smap(in);
  CN* const slot_base = (CN*)ws;
  auto slot = [&](int s) -> CN* { return slot_base + (size_t)((smap >> (4 * s)) & 15u) * MI; };
  const C* u;
  C* cand;
  rks2_states<R>(P, in, io, &u, &cand);
  const double mx = rks2_max(P.pmax + (size_t)inst * P.ncg, P.ncg);
  const int t = threadIdx.x;
  // NE/2 mirror row pairs per thread: pair p = (q, col) holds rows q and n - q (n/2 for q = 0)
  constexpr int N = G::N, NXH = G::NXH, XS = G::XS;
  const int sym = in->coef_sym;
  ChunkIdx<NE> ix;
  ix.sym = sym;
  ix.lim = G::MGEN_SYM_I;
  ix.anyq = 1;
#pragma unroll
  for (int j = 0; j < NE / 2; ++j) {
    const int p = blockIdx.x * NT * (NE / 2) + t + j * NT;
    const bool ok = p < (N / 2) * NXH;
    const int q = ok ? p / NXH : 0, col = ok ? p % NXH : 0;
    ix.m[2 * j] = q * XS + col;
    ix.m[2 * j + 1] = ok ? (q == 0 ? N / 2 : N - q) * XS + col : 0;
    ix.ok[2 * j] = ix.ok[2 * j + 1] = ok;
  }
  C ev[NE];
  error_chunk<R, RN, NE>(tb, slot, ws + P.off_coef, sym ? (size_t)G::MSYM : (size_t)MI, ix, in->h, ev);
  const double cut = P.ctl->adapt_cutoff;
  double su = 0.0, se = 0.0;
#pragma unroll
  for (int i = 0; i < NE; ++i) {
    if (ix.ok[i]) {
      const C kv = cand[ix.m[i]];
      const double kr = (double)kv.re, ki = (double)kv.im;
      if (hypot(kr, ki) / mx > cut) {
        const double er = (double)ev[i].re, ei = (double)ev[i].im;
        su += kr * kr + ki * ki;
        se += er * er + ei * ei;
      }
    }
  }
  wg_sum2<NT>(su, se, red);
  if (t == 0) {
    double* ps = P.psum + 2 * ((size_t)inst * P.nnb + blockIdx.x);
    ps[0] = su;
    ps[1] = se;
  }
}

// masked sums from the per-mode |u_new| and |err|^2 (FP32: |err|) that the
// fused last stage left in T: one read per mode instead of the candidate and
// every NL slot of the error estimate
template <typename R, int LOG2>
__global__ __launch_bounds__(256) void k2_norm_fused(rks2_launch P) {
  using G = Geo2<R, LOG2>;
  using C = cx<R>;
  constexpr int M = G::M, NXH = G::NXH, NT = G::NT, NE = G::NE;
  __shared__ double red[2 * (NT / 64 + 1)];
  const int inst = blockIdx.y;
  const rks2_state st = P.st[inst];
  if (!st.active) return;
  const rks_inst* in = P.inst + inst;
  const C* Tb = (const C*)((const char*)in->ws + P.off_T);
  const double mx = rks2_max(P.pmax + (size_t)inst * P.ncg, P.ncg);
  const double cut = P.ctl->adapt_cutoff;
  const int t = threadIdx.x;
  double su = 0.0, se = 0.0;
#pragma unroll
  for (int j = 0; j < NE; ++j) {
    const int e = blockIdx.x * NT * NE + t + j * NT;
    if (e < M) {
      const int r = e / NXH, c = e - r * NXH;
      const C v = Tb[r * G::TXS + c];
      const double a = (double)v.re;
      if (a / mx > cut) {
        su += a * a;
        if constexpr (sizeof(R) == sizeof(double)) {
          se += (double)v.im;
        } else {
          const double q = (double)v.im;
          se += q * q;
        }
      }
    }
  }
  wg_sum2<NT>(su, se, red);
  if (t == 0) {
    double* ps = P.psum + 2 * ((size_t)inst * P.nnb + blockIdx.x);
    ps[0] = su;
    ps[1] = se;
  }
}

// ---------------------------------------------------------------------------
// per-trajectory control
// ---------------------------------------------------------------------------
// set-up of a launch: evolve / resume / step (run_instance's set-up)
__global__ void k2_init(rks2_launch P) {
  const rks_tableau& tb = *P.tab;
  for (int i = threadIdx.x; i < P.ninst; i += blockDim.x) {
    const rks_io io = P.io[i];
    rks_inst& in = P.inst[i];
    rks2_state& st = P.st[i];
    st.active = st.need_nl1 = st.need_coef = st.store = st.snap_idx = 0;
    if (io.reset) {
      in.started = 0;
      in.accept = 0;
      in.h_coeff = __builtin_nan("");
      for (int s = 0; s < RKS_MAX_SLOTS; ++s) in.slot_map[s] = s;
    }
    if (P.mode == RKS_MODE_EVOLVE && !io.resume) {
      in.tc = io.t0;
      in.tf = io.tf;
      in.h = io.h_in;
      in.steps = in.attempts = in.rejects = 0;
      in.log_count = in.snap_count = 0;
      in.nl_calls = in.coef_updates = 0;
      in.ubuf = 0;  // k2_in copies u0 into cand0
      in.status = RKS_ST_RUNNING;
      if (tb.adaptive && in.tc + in.h > in.tf) in.h = in.tf - in.tc;  // solveras.py:620-621
      if (in.store_freq > 0) {
        st.store = 1;
        st.snap_idx = 0;
        in.snap_t[0] = in.tc;
        in.snap_count = 1;
      }
    } else if (P.mode == RKS_MODE_EVOLVE) {
      in.status = RKS_ST_RUNNING;
    } else if (P.mode == RKS_MODE_STEP) {
      in.h = io.h_in;
      in.status = RKS_ST_RUNNING;
      in.attempts = in.rejects = 0;
    } else {  // RKS_MODE_NL
      st.active = 1;
      st.need_nl1 = 1;
    }
    in.numloops = 0;
  }
  if (threadIdx.x == 0) *P.active_count = 0;
}

// Start of an attempt of trajectory i, by one thread: who runs, coefficient and NL1 needs,
// FSAL slot swap.
__device__ __forceinline__ void rks2_begin(const rks2_launch& P, rks_inst& in, rks2_state& st) {
  const rks_tableau& tb = *P.tab;
  int active = 0;
  if (in.status == RKS_ST_RUNNING) {
    const bool evolve = P.mode == RKS_MODE_EVOLVE;
    if (evolve && !(in.tc < in.tf)) in.status = RKS_ST_OK;
    else if (evolve && in.store_freq > 0 && in.snap_count >= in.snap_cap) in.status = RKS_ST_PAUSED;
    else active = 1;
  }
  st.active = active;
  st.need_nl1 = 0;
  st.need_coef = 0;
  if (!active) return;
  atomicAdd(P.active_count, 1);
  if (in.h != in.h_coeff) {
    st.need_coef = 1;
    in.h_coeff = in.h;
    ++in.coef_updates;
  }
  if (!in.started) {
    st.need_nl1 = 1;
    in.started = 1;
  } else if (in.accept || !tb.adaptive) {
    if (tb.nl1_policy == RKS_NL1_RECOMPUTE) {
      st.need_nl1 = 1;
    } else {
      const int f = tb.fsal_slot, a = in.slot_map[0];
      in.slot_map[0] = in.slot_map[f];
      in.slot_map[f] = a;
    }
  }
  int nl = st.need_nl1;
  for (int s = 0; s < tb.nstage; ++s) nl += tb.st[s].has_nl ? 1 : 0;
  in.nl_calls += nl;
}

// the first attempt's start (the others': k2_ctrl); one block per trajectory, as k2_ctrl
__global__ void k2_begin(rks2_launch P) {
  if (threadIdx.x == 0) rks2_begin(P, P.inst[blockIdx.x], P.st[blockIdx.x]);
}

// End of an attempt of a trajectory, by one thread: error ratio from the sums, accept/reject,
// dt, time, snapshots.
__device__ __forceinline__ void rks2_end(const rks2_launch& P, rks_inst& in, rks2_state& st, int i, double su,
                                         double se) {
  const rks_tableau& tb = *P.tab;
  const rks_ctrl& ct = *P.ctl;
  const double h = in.h;
  double h_suggest = h;
  if (tb.adaptive) {
    const double sv = rks_error_ratio(su, se, ct.epsilon, ct.safety_f, tb.q, P.lowp != 0);
    ++in.attempts;
    if (in.log_count < in.log_cap) {
      in.log[2 * in.log_count] = h;
      in.log[2 * in.log_count + 1] = sv;
    }
    ++in.log_count;
    if (isinf(sv) || isnan(sv) || sv < 1.0) {  // reject (solveras.py:490-506)
      in.accept = 0;
      ++in.rejects;
      double hn;
      if (isinf(sv) || isnan(sv)) {
        hn = ct.min_s * h;
      } else {
        double sc = sv > ct.min_s ? sv : ct.min_s;
        sc = sc < ct.decr_f ? sc : ct.decr_f;
        hn = sc * h;
      }
      in.h = hn;
      ++in.numloops;
      if (in.numloops > ct.max_loops) in.status = RKS_ST_MAXLOOPS;
      else if (hn < ct.minh) in.status = RKS_ST_MINSTEP;
      return;
    }
    in.accept = 1;  // accept (solveras.py:543-554)
    const double sc = sv < ct.max_s ? sv : ct.max_s;
    h_suggest = (sc > ct.incr_f) ? sc * h : h;
  } else {
    in.accept = 1;
  }
  in.numloops = 0;
  in.h_used = h;
  in.h_next = h_suggest;
  if (P.mode != RKS_MODE_EVOLVE) {
    in.status = RKS_ST_OK;
    ++in.steps;
    return;
  }
  in.ubuf = in.ubuf == 0 ? 1 : 0;
  const double tprev = in.tc;
  in.tc += h;
  ++in.steps;
  if (!(in.tc > tprev)) {  // h below the resolution of tc
    in.status = RKS_ST_MINSTEP;
    return;
  }
  if (tb.adaptive) in.h = (in.tc + h_suggest > in.tf) ? in.tf - in.tc : h_suggest;  // solveras.py:638-641
  if (in.store_freq > 0 && (in.steps % in.store_freq) == 0) {
    st.store = 1;
    st.snap_idx = in.snap_count;
    in.snap_t[in.snap_count] = in.tc;
    ++in.snap_count;
  }
}

// Between two attempts: the end of one and the start of the next, a wave per trajectory.  The
// partial sums are loaded a lane each and added in order by one lane from LDS; loaded one after
// the other by a thread per trajectory they took 23 us at n = 512 (65 partials).
__global__ __launch_bounds__(64) void k2_ctrl(rks2_launch P) {
  __shared__ double part[2 * 64];
  const int i = blockIdx.x, t = threadIdx.x;
  rks_inst& in = P.inst[i];
  rks2_state& st = P.st[i];
  double su = 0.0, se = 0.0;
  const bool active = st.active != 0;
  if (active && P.tab->adaptive) {
    const double* ps = P.psum + 2 * (size_t)i * P.nnb;
    for (int b0 = 0; b0 < P.nnb; b0 += 64) {
      const int nb = P.nnb - b0 < 64 ? P.nnb - b0 : 64;
      __syncthreads();
      if (t < nb) {
        part[2 * t] = ps[2 * (b0 + t)];
        part[2 * t + 1] = ps[2 * (b0 + t) + 1];
      }
      __syncthreads();
      if (t == 0)
        for (int b = 0; b < nb; ++b) {
          su += part[2 * b];
          se += part[2 * b + 1];
        }
    }
  }
  if (t != 0) return;
  st.store = 0;
  if (active) rks2_end(P, in, st, i, su, se);
  rks2_begin(P, in, st);
}

// The caller's u0 (rfft2 layout, row stride NXH) into cand0 (row stride XS):
// the start of an evolve (not a resume) or of a step.
template <typename R, int LOG2>
__global__ __launch_bounds__(256) void k2_in(rks2_launch P) {
  using G = Geo2<R, LOG2>;
  const int inst = blockIdx.y;
  const rks_io& io = P.io[inst];
  if (P.mode == RKS_MODE_EVOLVE && io.resume) return;
  const cx<R>* src = (const cx<R>*)io.u_in;
  cx<R>* dst = (cx<R>*)((char*)P.inst[inst].ws + P.off_cand0);
  for (int m = blockIdx.x * 256 + threadIdx.x; m < G::M; m += gridDim.x * 256) {
    const int r = m / G::NXH, c = m - r * G::NXH;
    dst[r * G::XS + c] = src[m];
  }
}

// snapshot copy of the current state (after ctrl / init), into the caller's layout
template <typename R, int LOG2>
__global__ __launch_bounds__(256) void k2_snap(rks2_launch P) {
  using G = Geo2<R, LOG2>;
  const int inst = blockIdx.y;
  const rks2_state st = P.st[inst];
  if (!st.store) return;
  const rks_inst* in = P.inst + inst;
  const rks_io& io = P.io[inst];
  const cx<R>* u;
  cx<R>* cand;
  rks2_states<R>(P, in, io, &u, &cand);
  cx<R>* dst = (cx<R>*)in->snap + (size_t)st.snap_idx * G::M;
  for (int m = blockIdx.x * 256 + threadIdx.x; m < G::M; m += gridDim.x * 256) {
    const int r = m / G::NXH, c = m - r * G::NXH;
    dst[m] = u[r * G::XS + c];
  }
}

// result into the caller's layout: the state at the end of an evolve (not for
// paused trajectories), the accepted candidate of a step
template <typename R, int LOG2>
__global__ __launch_bounds__(256) void k2_out(rks2_launch P) {
  using G = Geo2<R, LOG2>;
  const int inst = blockIdx.y;
  const rks_inst* in = P.inst + inst;
  if (in->status == RKS_ST_PAUSED) return;
  const rks_io& io = P.io[inst];
  const cx<R>* u;
  cx<R>* cand;
  rks2_states<R>(P, in, io, &u, &cand);
  const cx<R>* src = P.mode == RKS_MODE_STEP ? cand : u;
  cx<R>* dst = (cx<R>*)io.u_out;
  for (int m = blockIdx.x * 256 + threadIdx.x; m < G::M; m += gridDim.x * 256) {
    const int r = m / G::NXH, c = m - r * G::NXH;
    dst[m] = src[r * G::XS + c];
  }
}

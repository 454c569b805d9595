// Stockham FFT of P = 2^k complex points by T threads of one workgroup, the elements in
// registers and exchanged through LDS between its passes.  Pass (NS, RAD): a thread
// twiddles and transforms its E / RAD butterflies, then writes them in Stockham autosort
// order, and the next pass's come from there:
//   inputs  element j + r*P/RAD                     (r < RAD, j < P/RAD)
//   twiddle by W_{NS*RAD}^{r*(j mod NS)}
//   outputs element (j/NS)*NS*RAD + (j mod NS) + r*NS
// Layout and twiddles:
//   * element x lives at LDS index pad(x) = x + x/16: one spare element every
//     16 makes the stride-RAD writes of the first pass and all later passes
//     free of bank conflicts for 8- and 16-byte elements;
//   * W_N^x = T1[x >> S] * T2[x & (2^S-1)] from two small LDS tables
//     (sqrt(N) entries each, filled once per workgroup from the correctly
//     rounded global table), so no pass waits on global memory;
//   * radix = largest power of two <= 32 dividing the per-thread element
//     count E = P/T (radix-32 first: 8192 points with E = 32 take 3 passes).
// INV selects exp(+...) (unnormalised).
#pragma once
#include "rks_math.h"

namespace rksfft {

__device__ __forceinline__ constexpr int pad(int x) { return x + (x >> 4); }
// LDS elements needed for a padded P-point buffer
__host__ __device__ constexpr int padded_size(int P) { return P + (P >> 4) + 1; }

// two-level twiddle table geometry for an N-point base table
template <int LOG2N>
struct TwSplit {
  static constexpr int S = (LOG2N + 1) / 2;
  static constexpr int N1 = (1 << LOG2N) >> S;  // T1[i] = W_N^(i << S)
  static constexpr int N2 = 1 << S;              // T2[j] = W_N^j
  static constexpr int SIZE = N1 + N2;
};

// fill the LDS tables from the global table tw[x] = exp(-2 pi i x / N)
template <typename R, int LOG2N, int T>
__device__ __forceinline__ void load_twiddles(cx<R>* twl, const cx<R>* __restrict__ tw) {
  using TS = TwSplit<LOG2N>;
  for (int i = threadIdx.x; i < TS::SIZE; i += T)
    twl[i] = (i < TS::N1) ? tw[i << TS::S] : tw[i - TS::N1];
}

// W_N^x, 0 <= x < N
template <typename R, int LOG2N>
__device__ __forceinline__ cx<R> twiddle(const cx<R>* twl, int x) {
  using TS = TwSplit<LOG2N>;
  const cx<R> a = twl[x >> TS::S];
  const cx<R> b = twl[TS::N1 + (x & (TS::N2 - 1))];
  return a * b;
}

// exp(-2 pi i k / 32), k = 0..15, correctly rounded
__device__ __forceinline__ double c32(int k) {
  const double v[16] = {1.0, 0.9807852804032304491262, 0.9238795325112867561282, 0.8314696123025452370788,
                        0.7071067811865475244008, 0.5555702330196022247428, 0.3826834323650897717285,
                        0.1950903220161282678483, 0.0, -0.1950903220161282678483, -0.3826834323650897717285,
                        -0.5555702330196022247428, -0.7071067811865475244008, -0.8314696123025452370788,
                        -0.9238795325112867561282, -0.9807852804032304491262};
  return v[k];
}
__device__ __forceinline__ double s32(int k) {
  const double v[16] = {0.0, 0.1950903220161282678483, 0.3826834323650897717285, 0.5555702330196022247428,
                        0.7071067811865475244008, 0.8314696123025452370788, 0.9238795325112867561282,
                        0.9807852804032304491262, 1.0, 0.9807852804032304491262, 0.9238795325112867561282,
                        0.8314696123025452370788, 0.7071067811865475244008, 0.5555702330196022247428,
                        0.3826834323650897717285, 0.1950903220161282678483};
  return v[k];
}

// d * W_len^i (forward: exp(-2 pi i i/len); inverse: conjugate)
template <int LEN, bool INV, typename R>
__device__ __forceinline__ cx<R> tw_const(int i, cx<R> d) {
  const int k = i * (32 / LEN);
  if (k == 0) return d;
  if (k == 8) return mul_mi<INV>(d);
  const R c = (R)c32(k);
  const R s = INV ? (R)s32(k) : (R)(-s32(k));
  return mkc(d.re * c - d.im * s, d.re * s + d.im * c);
}

template <int RAD>
__device__ constexpr int bitrev(int i) {
  int r = 0;
  for (int b = 1; b < RAD; b <<= 1) {
    r = (r << 1) | (i & 1);
    i >>= 1;
  }
  return r;
}

// In-register DFT of RAD points (radix-2 decimation in frequency).
template <int RAD, bool INV, typename R>
__device__ __forceinline__ void dft_small(cx<R> (&v)[RAD]) {
#pragma unroll
  for (int len = RAD; len >= 2; len >>= 1) {
    const int half = len / 2;
#pragma unroll
    for (int blk = 0; blk < RAD; blk += len) {
#pragma unroll
      for (int i = 0; i < half; ++i) {
        cx<R> a = v[blk + i], b = v[blk + i + half];
        v[blk + i] = a + b;
        cx<R> d = a - b;
        if (len == 32) v[blk + i + half] = tw_const<32, INV>(i, d);
        else if (len == 16) v[blk + i + half] = tw_const<16, INV>(i, d);
        else if (len == 8) v[blk + i + half] = tw_const<8, INV>(i, d);
        else if (len == 4) v[blk + i + half] = tw_const<4, INV>(i, d);
        else v[blk + i + half] = d;
      }
    }
  }
  cx<R> t[RAD];
#pragma unroll
  for (int i = 0; i < RAD; ++i) t[i] = v[bitrev<RAD>(i)];
#pragma unroll
  for (int i = 0; i < RAD; ++i) v[i] = t[i];
}

template <int E, int MAXR>
struct pick_radix {
  static constexpr int v = (E % 32 == 0 && MAXR >= 32) ? 32
                           : (E % 16 == 0 && MAXR >= 16) ? 16
                           : (E % 8 == 0 && MAXR >= 8) ? 8
                           : (E % 4 == 0 && MAXR >= 4) ? 4 : 2;
};

// v[r] *= W_N^(r step) (conjugate for INV), r = 1..RAD-1.  FP64: powers of
// the one table value w = W_N^step by squaring and products p[r] = p[hb]
// p[r - hb] (hb the highest power of two <= r), at most four multiplications
// deep, so a butterfly reads two table entries instead of 2 (RAD - 1).  FP32
// keeps one table lookup per twiddle (the products' rounding would show).
template <int RAD, bool INV, int LOG2N, typename R>
__device__ __forceinline__ void apply_twiddles(cx<R> (&v)[RAD], const cx<R>* twl, int step) {
  if constexpr (sizeof(R) == sizeof(double)) {
    cx<R> p[RAD];
    p[1] = twiddle<R, LOG2N>(twl, step);
#pragma unroll
    for (int r = 2; r < RAD; ++r) {
      const int hb = (r >= 8) ? 8 : (r >= 4) ? 4 : (r >= 2) ? 2 : 1;
      p[r] = (r == hb) ? p[r / 2] * p[r / 2] : p[hb] * p[r - hb];
    }
#pragma unroll
    for (int r = 1; r < RAD; ++r) v[r] = cmul_tw<INV>(v[r], p[r]);
  } else {
#pragma unroll
    for (int r = 1; r < RAD; ++r) v[r] = cmul_tw<INV>(v[r], twiddle<R, LOG2N>(twl, r * step));
  }
}

// Register-resident transform: v[k] holds element t + k T (k < E = P / T) on entry
// and on exit, for every radix sequence, because both the first pass's inputs
// j + r P / RAD and the last pass's outputs j + r NS (NS = P / RAD) of the
// butterflies j = t + b T are congruent to t mod T.  So the stage values enter the
// first butterfly straight from registers and the results leave the last one in
// registers: a transform of p passes exchanges p - 1 times through LDS, where the
// LDS-to-LDS form exchanges p times and is filled and drained once more.
// PP: two buffers (buf and, padded_size(2^LOG2N) further, the other) used in turn, so an
// exchange takes one barrier instead of two; BUF is the one that the next exchange writes.
// post(x): applied to each output.  on: the thread takes part (every thread calls, for the
// barriers).
//
// Which product of a sum of two the compiler fuses hangs on the order in which it sees the
// operands, and on which loads it finds equal.  leaf() makes the first pass's inputs opaque
// values in the order in which an LDS-to-LDS pass loads them, and FENCE ends each of the last
// pass's butterflies as its stores would, so a transform rounds alike in every kernel that
// inlines it.
template <typename R>
__device__ __forceinline__ void leaf(cx<R>& v) {
  asm volatile("" : "+v"(v.re));
  asm volatile("" : "+v"(v.im));
}

template <typename R, int P, int T, int NS, bool INV, int LOG2N, int TSCALE, int MAXR, bool PP, int BUF, bool FENCE, typename Post>
__device__ __forceinline__ void chain_reg(cx<R> (&v)[P / T], cx<R>* buf, const cx<R>* twl, int t, Post post,
                                          bool on = true) {
  constexpr int E = P / T;
  constexpr int R0 = pick_radix<E, MAXR>::v;
  constexpr int REM = P / NS;
  constexpr int RAD = (R0 <= REM) ? R0 : REM;
  constexpr int NB = E / RAD;
  constexpr bool LAST = NS * RAD == P;
  constexpr int PREV = PP ? 1 - BUF : 0;  // the buffer of the exchange before this pass
  constexpr int BS = padded_size(1 << LOG2N);
  cx<R> w[NB][RAD];
  if (on) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int j = t + b * T;
#pragma unroll
      for (int r = 0; r < RAD; ++r) {
        if constexpr (NS == 1) {
          w[b][r] = v[b + r * NB];
          leaf(w[b][r]);
        } else {
          w[b][r] = buf[PREV * BS + pad(j + r * (P / RAD))];
        }
      }
    }
  }
  if constexpr (NS > 1 && !PP) __syncthreads();
  if (on) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int j = t + b * T;
      const int k = j & (NS - 1);
      if constexpr (NS > 1) apply_twiddles<RAD, INV, LOG2N>(w[b], twl, k * (P / (NS * RAD)) * TSCALE);
      dft_small<RAD, INV>(w[b]);
      const int base = (j - k) * RAD + k;
#pragma unroll
      for (int r = 0; r < RAD; ++r) {
        if constexpr (LAST) v[b + r * NB] = post(w[b][r]);
        else buf[(PP ? BUF : 0) * BS + pad(base + r * NS)] = w[b][r];
      }
      if constexpr (LAST && FENCE && NB > 1) asm volatile("" ::: "memory");
    }
  }
  if constexpr (!LAST) {
    __syncthreads();
    chain_reg<R, P, T, NS * RAD, INV, LOG2N, TSCALE, MAXR, PP, PP ? 1 - BUF : 0, FENCE>(v, buf, twl, t, post, on);
  }
}

// number of LDS exchanges of a register-resident P-point transform
template <int P, int T, int MAXR>
constexpr int exchanges() {
  int n = 0, ns = 1;
  const int r0 = pick_radix<P / T, MAXR>::v;
  while (ns < P) {
    ns *= r0 <= P / ns ? r0 : P / ns;
    ++n;
  }
  return n - 1;
}

// Full P-point register-resident transform (chain_reg) by the threads t.  The buffers are free when it
// is called.  Without PP they are free again when it returns; with PP the buffer of the
// last exchange, (BUF + exchanges - 1) % 2, may still be read by other threads.
template <typename R, int P, int T, bool INV, int LOG2N, int MAXR, bool PP, int BUF, bool FENCE, typename Post>
__device__ __forceinline__ void fft_reg(cx<R> (&v)[P / T], cx<R>* buf, const cx<R>* twl, int t, Post post,
                                        bool on = true) {
  static_assert((P & (P - 1)) == 0, "power of two");
  static_assert(P / T >= 2, "need at least two elements per thread");
  chain_reg<R, P, T, 1, INV, LOG2N, (1 << LOG2N) / P, MAXR, PP, BUF, FENCE>(v, buf, twl, t, post, on);
}

}  // namespace rksfft

// Host side of the 2-D rfft2 engine (kernels in rks_2d.h, launches in rks_2d.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

#include "rks_types.h"

struct rks2_launch;
struct rks2_ctx;

// 1 if kernels exist for this precision and N = 2^log2n
int rks2_supported(int prec, int log2n);
// modes of an N x N rfft2 grid
inline int rks2_modes(int log2n) { return (1 << log2n) * ((1 << log2n) / 2 + 1); }
// row stride (elements) of the transform buffer T: N/2 + 1 columns rounded up
// to whole 128-byte lines of esize-byte elements
__host__ __device__ constexpr int rks2_t_stride(int n, int esize) {
  return ((n / 2 + 1) * esize + 127) / 128 * 128 / esize;
}
// row stride (elements) of the internal state, NL and coefficient arrays: N/2 + 1
// columns rounded up to 32, so rows of 4-, 8- and 16-byte elements all start on
// 128-byte lines and a column tile's row segments do not straddle lines.  The
// caller's arrays (u0, uf, lin_op, snapshots) keep NumPy's rfft2 layout.
__host__ __device__ constexpr int rks2_istride(int n) { return (n / 2 + 1 + 31) / 32 * 32; }
// elements of one internal array
inline int rks2_imodes(int log2n) { return (1 << log2n) * rks2_istride(1 << log2n); }

// Allocates the per-trajectory flags and reduction partials and sets kernel
// attributes.  The workspace of instance i holds (byte offsets)
//   NL slots at 0 | cand0 at off_cand0 | cand1 at off_cand1 | coefficients at
//   off_coef | transform buffer T (N rows of rks2_t_stride state-precision
//   complex values) at off_T;
// NL slots, candidates and coefficient arrays have rks2_imodes elements each
// (rows of rks2_istride).
// variant: the method whose kernels are compiled for it (real lin_op), or RKS_METH_ANY.
int rks2_create(rks2_ctx** out, int prec, int variant, int log2n, int ninst, const rks_tableau* d_tab, const rks_ctrl* d_ctl,
                rks_inst* d_inst, const rks_io* d_io, const void* d_tw, size_t off_cand0, size_t off_cand1,
                size_t off_coef, size_t off_T);
// One launch set: mode RKS_MODE_EVOLVE / RKS_MODE_STEP (attempts until every
// trajectory has finished) or RKS_MODE_NL; store: trajectories keep snapshots.
// Synchronises `stream`.
hipError_t rks2_run(rks2_ctx* c, const rks_tableau& tab, int mode, bool store, hipStream_t stream);
void rks2_destroy(rks2_ctx* c);

/* rkstiff_amd: MI355X (gfx950) stepping engine for rkstiff's diagonal solvers.
 *
 * C ABI of librkstiff_amd.so.  Plain pointers and sizes; state arrays are
 * device pointers (complex interleaved, float64x2 for RKS_F64, float32x2 for
 * RKS_F32); per-instance scalars are host arrays.  Functions return RKS_OK or an
 * error code; rks_last_error() gives the message (thread-local).
 *
 * The reference (rkstiff, pure Python/NumPy) has no FFI: each entry point below
 * replaces one Python-level operation of the reference, cited per function.
 * A plan owns its workspace and device records, is bound to one device and is
 * not thread-safe (like the reference's solver object); distinct plans may run
 * concurrently on distinct streams.
 */
#ifndef RKSTIFF_AMD_H
#define RKSTIFF_AMD_H

#include <hip/hip_runtime_api.h>

#ifdef __cplusplus
extern "C" {
#endif

/* status / error codes */
enum {
  RKS_OK = 0,
  RKS_ERR_INVALID = 1, /* ValueError in the reference's terms */
  RKS_ERR_HIP = 2,     /* runtime failure */
  RKS_MAXLOOPS = 3,    /* BaseSolverAS.MaxLoopsExceeded (solveras.py:399-406) */
  RKS_MINSTEP = 4,     /* BaseSolverAS.MinimumStepReached (solveras.py:407-410) */
  RKS_PAUSED = 5,      /* evolve paused: snapshot buffer full, call rks_resume */
  RKS_RUNNING = 6
};

/* methods: the reference's seven diagonal solver classes */
enum {
  RKS_ETD35 = 0, /* etd35.py:723-889 */
  RKS_ETD34 = 1, /* etd34.py:439-621 */
  RKS_ETD4 = 2,  /* etd4.py:311-422 */
  RKS_ETD5 = 3,  /* etd5.py:485-655 */
  RKS_IF34 = 4,  /* if34.py:260-338 */
  RKS_IF45DP = 5,/* if45dp.py:8-249 */
  RKS_IF4 = 6    /* if4.py:202-275 */
};

/* built-in nonlinear terms (the user nl_func patterns of the reference) */
enum {
  RKS_NL_ADVECT_RFFT = 0, /* c * rfft(irfft(u) * irfft(i kx u)): KS/Burgers (c=-1, README.md:94-97,
                             models.py:189-192), KdV (c=-6, models.py:140-143); n real points */
  RKS_NL_CUBIC_FFT = 1,   /* i g fft(|v|^2 v), v = ifft(u): cubic NLS (demos/nls.ipynb cell 29); n points */
  RKS_NL_NONE = 2,        /* caller evaluates nl (generic path): only coefficients, stage combinations
                             and the error norm run here; n = number of modes */
  RKS_NL_AC2D_RFFT2 = 3,  /* rfft2(w - c w^3), w = irfft2(u): Allen-Cahn reaction term (the cubic of
                             demos/allen_cahn.ipynb cell 4) on an n x n periodic grid, modes flattened
                             row-major as the reference requires of multi-D problems (solver.py:129-135);
                             n a power of two in [32, 512], ny = n, m = n (n/2 + 1) */
  RKS_NL_HANKEL_CUBIC = 4 /* i c S Y (|f|^2 f), f = Y u / S: the radial NLS term of demos/nls.ipynb cell 8
                             with the order-zero Hankel transform ht = S Y, iht = Y / S
                             (transforms.py:172-240); n = nr in [4, 1024] radial points = modes,
                             kx = Y (nr x nr float64, row-major), nl_scale = S, nl_coef = c (gamma) */
};

/* engine precision: state/FFT/propagators + NL and coefficient storage
 *   RKS_F64    all FP64
 *   RKS_F32    all FP32 (coefficients generated in FP64; norm and dt control FP64)
 *   RKS_MIXED  FP64 state, propagators exp(f h L) and FFTs; FP32 NL arrays and other
 *              coefficients.  State pointers are complex128. */
enum { RKS_F64 = 0, RKS_F32 = 1, RKS_MIXED = 2 };

/* SolverConfig (solveras.py:27-169), the class constants MAX_LOOPS/MAX_S/MIN_S
 * (solveras.py:255-257) and ETDConfig (etd.py:46-131), passed by value. */
typedef struct rks_config {
  double epsilon, incr_f, decr_f, safety_f, adapt_cutoff, minh;
  double max_s, min_s;
  int max_loops;
  int contour_points;
  double modecutoff, contour_radius;
} rks_config;

/* One trajectory's operator (solver.py:91-136: lin_op 1-D => diagonal). */
typedef struct rks_instance_desc {
  int n;               /* real-space points (power of two, 16..8192), radial points (Hankel) or modes
                          for RKS_NL_NONE */
  int L_is_complex;    /* lin_op dtype: 0 float64[m], 1 complex128[m] */
  const void* L;       /* lin_op, float64 data, host or device pointer (copied) */
  const double* kx;    /* wavenumbers float64[m] (RKS_NL_ADVECT_RFFT) or the Hankel matrix float64[n n]
                          (RKS_NL_HANKEL_CUBIC), host or device (copied; instances passing the same
                          Hankel matrix pointer share one device copy) */
  double nl_coef;      /* c of the advective term / g of the cubic term / c of the rfft2 term */
  int ny;              /* rows of a 2-D grid (RKS_NL_AC2D_RFFT2, = n); ignored otherwise */
  double nl_scale;     /* S of the Hankel transform (RKS_NL_HANKEL_CUBIC); ignored otherwise */
} rks_instance_desc;

typedef struct rks_stats {
  double tc;           /* current time (evolve) */
  double h_used;       /* last accepted step */
  double h_next;       /* suggested next step (step(): third return value) */
  double h;            /* next step the evolve loop would try */
  int steps, attempts, rejects, status;
  int log_count, snap_count, nl_calls, coef_updates;
} rks_stats;

typedef struct rks_plan rks_plan;

/* Create a plan for `ninst` trajectories of one method / nonlinearity / precision.
 * Replaces the solver constructors (e.g. ETD35.__init__, etd35.py:784-830, and
 * BaseSolverAS.__init__, solveras.py:262-282). */
int rks_plan_create(int method, int nl_kind, int precision, const rks_config* cfg, int ninst,
                    const rks_instance_desc* desc, rks_plan** out);
int rks_plan_destroy(rks_plan* p);
int rks_plan_info(const rks_plan* p, int* ninst, int* nslot, int* ncoef, int* esize);
/* Replace the controller/ETD configuration (the reference reads solver.config and the
 * MAX_LOOPS/MAX_S/MIN_S attributes at every step, solveras.py:384-410). */
int rks_set_config(rks_plan* p, const rks_config* cfg, hipStream_t stream);

/* Snapshot storage (store_data / store_freq of evolve, solveras.py:609-611,643-646)
 * and the per-attempt (h, s) log.  snap_cap snapshots per instance; an evolve
 * pauses with RKS_PAUSED when the buffer is full. */
int rks_set_storage(rks_plan* p, int store_freq, int snap_cap, int log_cap);

/* Integrate every instance from t0[i] to tf[i]: BaseSolverAS.evolve
 * (solveras.py:556-650; h[i] = h_init, clamped to tf-t0 like 620-621) or
 * BaseSolverCS.evolve (solvercs.py:191-279; h[i] = constant step).  u0[i] is
 * read, uf[i] receives u(tf).  1-D plans: asynchronous on `stream` (one persistent
 * launch per size bucket runs every trajectory to tf).  2-D (rfft2) plans: the attempt
 * sequence is replayed in groups of four until no trajectory is active, which the host
 * reads back after each group, so the call returns with `stream` synchronized and the
 * evolve complete. */
int rks_evolve(rks_plan* p, const void* const* u0, void* const* uf, const double* t0, const double* tf,
               const double* h, hipStream_t stream);
/* Continue trajectories paused on a full snapshot buffer (synchronization as rks_evolve). */
int rks_resume(rks_plan* p, hipStream_t stream);

/* One accepted step from u[i] with suggested h[i]: BaseSolverAS.step
 * (solveras.py:336-410) or BaseSolverCS.step (solvercs.py:163-186).  Solver state
 * (FSAL NL1, coefficient cache, accept flag) persists between calls. */
int rks_step(rks_plan* p, const void* const* u, void* const* u_new, const double* h, hipStream_t stream);
/* BaseSolverAS.reset / BaseSolverCS.reset: clear FSAL and coefficient state. */
int rks_reset(rks_plan* p, hipStream_t stream);

/* Evaluate the built-in nonlinear term: nl_func(u) (models.py:140-143, README.md:94-97). */
int rks_nl_eval(rks_plan* p, const void* const* u, void* const* nl_out, hipStream_t stream);

/* Coefficient arrays of instance `inst` at step h (e.g. _Etd35Diagonal.update_coeffs,
 * etd35.py:157-288), computed in FP64 and stored in the plan precision.
 * dst (optional, device) receives ncoef x m complex values (every mode, also where
 * the stepping kernels keep a mirror-symmetric lin_op's modes 0..n/2 only); the
 * stepping kernels regenerate their own coefficient cache after this call. */
int rks_coeffs(rks_plan* p, int inst, double h, void* dst, hipStream_t stream);
/* Generic-nl path: one stage combination k = E u + sum C NL (e.g. etd35.py:320-343),
 * stage = -1 gives the embedded error estimate (etd35.py:344).  slots: nslot device
 * pointers to the NL arrays.  Coefficients come from the last rks_coeffs call. */
int rks_combine(rks_plan* p, int inst, int stage, double h, const void* u, const void* const* slots, void* out,
                hipStream_t stream);
/* Generic-nl path: s of BaseSolverAS._compute_s (solveras.py:412-455) into s_dev (device double). */
int rks_error_s(rks_plan* p, int inst, const void* u_new, const void* err, double* s_dev, hipStream_t stream);

/* Launch shape of the persistent kernels (no counterpart in the reference, which
 * has no launches; set by the autotuner, rkstiff_amd.autotune).  Instances are
 * grouped in size buckets (one kernel launch each, largest n first).
 * rks_plan_buckets: nbucket and, per bucket (up to cap), log2 n, the instance
 * count, the most resident workgroups per CU the kernel allows and the number
 * of FFT tiles available (2 for n = 512 .. 4096: tile 1 runs twice the threads
 * per trajectory, half the modes per thread).
 * rks_plan_set_launch: concurrent != 0 (the default) launches the buckets on
 * private streams forked from and joined back to the caller's stream, so a
 * bucket's tail overlaps the others; 0 launches them in order on the caller's
 * stream.  wg_per_cu[b] (NULL: all 0) caps bucket b's resident workgroups per
 * CU, 0 = as many as fit; tile[b] picks bucket b's FFT tile: 0 the base tile, 1
 * twice its threads (n = 512 .. 4096; without a proposer or records also the cubic
 * n = 8192), 2 four times (n = 1024 and the cubic n = 2048, without a proposer or
 * records; these, attached later, bring the base tile back), -1 (also tile NULL, as
 * before the first call) the library's choice.  That is a wider tile for FP64
 * trajectories of n >= 512, by their own size, method and (advective term) damping at
 * the grid's end, whatever else is in the plan; the base tile in other precisions and
 * while a proposer, records or an attempt log are attached.  Results do not depend on
 * the shape; another tile rounds in another order, so an FP64 run with a log repeats
 * the run without one to rounding, and bit for bit where both set the same tile.
 * rks_plan_tiles: the tile each bucket (up to cap) runs on now (0, 1 or 2; where only
 * some of its trajectories keep the base tile for lack of damping, the others'). */
int rks_plan_buckets(rks_plan* p, int* nbucket, int* log2n, int* count, int* max_wg_per_cu, int* ntile, int cap);
int rks_plan_set_launch(rks_plan* p, int concurrent, const int* wg_per_cu, const int* tile, int nbucket);
int rks_plan_tiles(rks_plan* p, int* tile, int cap);
/* Order in which each size bucket's workgroups take their trajectories:
 * descending cost[i] (host array, one finite value per instance; equal costs
 * keep instance order), so the longest trajectories start first and the
 * bucket's tail is short (longest-processing-time-first).  Results do not
 * depend on it.  Synchronises the device. */
int rks_plan_set_priority(rks_plan* p, const double* cost);

/* Synchronise `stream` and read per-instance counters/status (host array of ninst). */
int rks_get_stats(rks_plan* p, rks_stats* out, hipStream_t stream);
/* Attempt log of instance `inst`: cap (h, s) pairs into host_hs. */
int rks_read_log(rks_plan* p, int inst, double* host_hs, int cap, hipStream_t stream);
/* Copy `count` stored snapshots of `inst` to dst_dev (device, count x m complex) and
 * their times to t_host; marks the buffer consumed. */
int rks_read_snapshots(rks_plan* p, int inst, void* dst_dev, double* t_host, int count, hipStream_t stream);

/* ---------------------------------------------------------------------------
 * Learned step-size proposer.  No counterpart in the reference: its controller
 * keeps h after an accept unless s > incr_f (solveras.py:543-554).  This is an
 * opt-in addition for batched evolves.  A small MLP (66 -> 256 -> 256 -> 256 -> 1,
 * GELU, BF16 weights, FP32 accumulation on the matrix cores) proposes the step
 * after each accepted one.  The embedded error estimate still judges every
 * attempt, a rejection still uses the reference's rule, and a non-finite output
 * falls back to the reference's proposal.
 *
 * Inputs of an accepted state (raw, RKS_PROPOSER_NIN floats):
 *   f_b  = 0.5 ln(mean |u_hat|^2 over bin b / n^2 + 1e-30), b < 64.  Mode m has
 *          wavenumber index w = m (rfft) or min(m, n - m) (fft) and lies in bin
 *          (64 w) / (n/2 + 1).
 *   f_64 = ln h of the accepted step.
 *   f_65 = ln min(s, 1e4) of its attempt.
 * The network sees (f - mu) / sig.  Its output y estimates ln(h' s' / h), where
 * (h', s') is the next attempt.  With d = y - margin, the next step is:
 *   RKS_PROPOSE  h itself when keep_lo <= d < keep_hi (like the reference keeping
 *                h for 1 <= s <= incr_f, this leaves the coefficient cache
 *                valid), else h exp(clamp(d, ln min_s, ln max_s));
 *   RKS_GUARD    the reference controller's proposal h_ref, unless
 *                d < ln(h_ref / h) + keep_lo (its rejection is predicted); then
 *                h exp(max(d, ln min_s)).
 *   RKS_GROW     as RKS_GUARD, and when d >= ln(h_ref / h) + g with g = keep_hi > 0,
 *                h_ref e^(j g), j = floor((d - ln(h_ref / h)) / g), at most
 *                h max_s: the step grows ahead of the reference on a grid of
 *                ratio e^g (few distinct steps, few coefficient regenerations).
 * The network runs after every (period * 512 / T)-th accepted step, T the
 * trajectory's workgroup size (64..512: small grids consult it less often, as
 * their attempts are short next to one inference); after the other accepted
 * steps the reference controller's proposal stands.
 *
 * Parameters: one float32 vector of RKS_PROPOSER_NPARAM values,
 *   W1 [256][96] (columns 66..95 are zero padding), b1 [256], W2 [256][256], b2,
 *   W3 [256][256], b3, w4 [256], b4 [1].
 * A training record (RKS_PROPOSER_REC floats): 66 inputs, the target
 * ln(h' s' / h), and a valid flag.  The flag is 0 when the next attempt was
 * clamped to tf or its error was zero or non-finite.
 * ------------------------------------------------------------------------- */
enum { RKS_PROPOSER_NIN = 66, RKS_PROPOSER_REC = 68, RKS_PROPOSER_NPARAM = 156673 };
enum { RKS_PROPOSE = 0, RKS_GUARD = 1, RKS_GROW = 2 };

typedef struct rks_mlp rks_mlp;

/* Create on the current device from host params / mu / sig (float32). */
int rks_mlp_create(const float* params, const float* mu, const float* sig, rks_mlp** out);
int rks_mlp_destroy(rks_mlp* net);
/* Synchronise and copy the FP32 parameters to the host. */
int rks_mlp_get_params(rks_mlp* net, float* params);
/* nsteps Adam steps (lr, beta 0.9 / 0.999, eps 1e-8) on minibatches of `batch`
 * (a multiple of 64) device records rec[idx[step * batch + j]], j < batch.
 * loss_kind 0: pinball loss rho_tau(y - yhat); 1: 0.5 (yhat - y)^2.  Targets
 * are used as given (clip them beforehand).  loss_dev (optional, device)
 * receives the batch-mean loss of every step. */
int rks_mlp_train(rks_mlp* net, const float* rec, int nrec, const int* idx, int batch, int nsteps, int loss_kind,
                  double tau, double lr, float* loss_dev, hipStream_t stream);
/* Batched forward of nrec device records into yhat (device). */
int rks_mlp_forward(rks_mlp* net, const float* rec, int nrec, float* yhat, hipStream_t stream);
/* Gradient of the mean loss over nrec records (a multiple of 64) without an
 * update: grad (device, RKS_PROPOSER_NPARAM); yhat and loss_dev optional. */
int rks_mlp_gradient(rks_mlp* net, const float* rec, int nrec, int loss_kind, double tau, float* grad, float* yhat,
                     float* loss_dev, hipStream_t stream);
/* Batch-1 forward of each record by one workgroup of `threads` (64..512):
 * the code path the stepping kernels run after an accepted step. */
int rks_mlp_infer_single(rks_mlp* net, const float* rec, int nrec, int threads, float* yhat, hipStream_t stream);
/* Attach (net != NULL) or detach the proposer for the plan's evolves.  The plan
 * must be adaptive, 1-D built-in (n >= 256 rfft, n >= 128 fft).  The net must
 * outlive the plan's use of it. */
int rks_plan_set_proposer(rks_plan* p, const rks_mlp* net, int policy, double margin, double keep_lo,
                          double keep_hi, int period);
/* Record up to rec_cap training records per instance during evolve (0 turns off). */
int rks_set_records(rks_plan* p, int rec_cap);
/* Synchronise; counts[i] (host, optional) = records of instance i; dst_dev
 * (optional, device) receives ninst x rec_cap x RKS_PROPOSER_REC floats. */
int rks_read_records(rks_plan* p, float* dst_dev, int* counts, hipStream_t stream);

/* ---------------------------------------------------------------------------
 * Quasi-discrete Hankel transform of order zero: HankelTransform.ht / .iht
 * (transforms.py:172-240) and the radial cubic NLS term of demos/nls.ipynb
 * cell 8.  Y is the reference's nr x nr matrix 2 J0(j_i j_j / j_{N+1}) /
 * (j_{N+1} J1(j_j)^2) (transforms.py:113-117, row-major float64, host or
 * device, copied); scale is S = rmax^2 / j_{N+1}.  Vectors are rows of nr
 * values (complex128 interleaved when cplx, else float64), device pointers.
 * Calls on one transform object must not overlap (it keeps one scratch).
 * ------------------------------------------------------------------------- */
typedef struct rks_hankel rks_hankel;
int rks_hankel_create(int nr, const double* Y, double scale, rks_hankel** out);
int rks_hankel_destroy(rks_hankel* h);
/* out[b] = S Y in[b] (forward, ht) or Y in[b] / S (inverse, iht), b < batch. */
int rks_hankel_apply(rks_hankel* h, int inverse, const void* in, void* out, int batch, int cplx, hipStream_t stream);
/* out[b] = 1j gamma ht(|f|^2 f), f = iht(in[b]) (complex128 only). */
int rks_hankel_cubic(rks_hankel* h, double gamma, const void* in, void* out, int batch, hipStream_t stream);
/* rks_hankel_cubic without any device allocation.  No counterpart in the
 * reference: for callers that cannot allocate (code under HIP graph capture,
 * serving loops, harnesses that forbid hipMalloc).  The |f|^2 f intermediate
 * lives in a library-owned static device array of 4 MiB per GPU (held until
 * the process ends), so nr * batch must be <= 262144; larger calls return
 * RKS_ERR_INVALID.  Every call on one GPU shares that array: calls that
 * overlap on one GPU (other streams, other threads, other transforms) race. */
int rks_hankel_cubic_noalloc(rks_hankel* h, double gamma, const void* in, void* out, int batch,
                             hipStream_t stream);

/* ---------------------------------------------------------------------------
 * Dense (non-diagonal) strategies for a batch of small systems (n <= 256):
 * the matrix coefficients of the reference's dense update_coeffs
 * (etd35.py:602-670, etd34.py:356-404, etd4.py:235-283, etd5.py:360-434,
 * if34.py:225-234, if4.py:152-169) and the matrix-vector stage combinations
 * of their update_stages (etd35.py:671-720, etd34.py:405-436, etd4.py:284-308,
 * etd5.py:435-482, if34.py:235-254, if4.py:170-199).  Matrices are
 * row-major n x n complex128, vectors n complex128, system b at offset b n n
 * (b n); device pointers.
 * ------------------------------------------------------------------------- */
/* coeffs[b][c] = coefficient matrix c (tableau order) of method `method` at
 * z = h[b] L[b]: exponentials by scaling and squaring with the degree-13 Pade
 * approximant, psi functions by the contour mean over contour_points nodes of
 * radius contour_radius.  h is a host array of `batch` step sizes.  Returns
 * after the work is done (its work buffers are released). */
int rks_dense_coeffs(int method, int n, int batch, const void* L, const double* h, int contour_points,
                     double contour_radius, void* coeffs, hipStream_t stream);
/* The same in the caller's work memory (device, 256-byte aligned, at least
 * the *bytes of rks_dense_ws_bytes): the launches are queued on `stream` and ws
 * must live until they are done. */
int rks_dense_ws_bytes(int method, int n, int batch, int contour_points, size_t* bytes);
int rks_dense_coeffs_ws(int method, int n, int batch, const void* L, const double* h, int contour_points,
                        double contour_radius, void* coeffs, void* ws, size_t ws_bytes, hipStream_t stream);
#define RKS_DENSE_MAX_TERMS 8
/* One term of a stage sum: alpha * mat (x + s2 x2); mat NULL: the identity,
 * x2 NULL: no second vector. */
typedef struct rks_dense_term {
  const void* mat;
  const void* x;
  const void* x2;
  double s2;
  double alpha;
} rks_dense_term;
/* y[b] = sum_k terms[k] for every system b (y must not alias an x). */
int rks_dense_combine(int n, int batch, const rks_dense_term* terms, int nterm, void* y, hipStream_t stream);

/* Method tableau (host-only, no device needed): fills `bytes` >= rks_sizeof(0). */
int rks_get_tableau(int method, void* out, int bytes);
int rks_sizeof(int what);
const char* rks_last_error(void);

#ifdef __cplusplus
}
#endif
#endif /* RKSTIFF_AMD_H */

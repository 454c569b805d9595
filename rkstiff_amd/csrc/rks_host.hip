// Host side of the stepping engine: plans, launches and the C ABI of
// include/rkstiff_amd.h.  Kernel instantiations live in rks_k.hip (compiled once
// per precision x nonlinearity x method, in parallel).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "rks_2d_host.h"
#include "rks_kernels.h"

// ---------------------------------------------------------------------------
// generic-nl path kernels (arbitrary caller-supplied nonlinear term)
// ---------------------------------------------------------------------------
template <typename R>
__global__ void rks_coef_kernel(const rks_tableau* tab, const rks_ctrl* ctl, const double* L, int Lc, int M,
                                double h, char* cbase) {
  for (int m = blockIdx.x * blockDim.x + threadIdx.x; m < M; m += gridDim.x * blockDim.x)
    coef_mode<R, R>(*tab, *ctl, L, Lc, m, M, h, cbase);
}

struct rks_combine_args {
  const rks_tableau* tab;
  const void* u;
  const void* slots[RKS_MAX_SLOTS];
  const char* coefs;
  void* out;
  int stage;
  int is_err;
  int M;
  int pad;
  double h;
};

template <typename R>
__global__ void rks_combine_kernel(rks_combine_args A) {
  using C = cx<R>;
  const C* u = (const C*)A.u;
  C* out = (C*)A.out;
  auto slotp = [&](int s) -> const C* { return (const C*)A.slots[s]; };
  for (int m = blockIdx.x * blockDim.x + threadIdx.x; m < A.M; m += gridDim.x * blockDim.x) {
    C v[1];
    if (A.is_err) error_chunk<R, R, 1>(*A.tab, slotp, A.coefs, (size_t)A.M, m, 1, A.M, A.h, v);
    else stage_chunk<R, R, 1>(*A.tab, A.tab->st[A.stage], u, slotp, A.coefs, (size_t)A.M, m, 1, A.M, A.h, v);
    out[m] = v[0];
  }
}

// real coefficient storage -> complex (the copy-out of rks_coeffs)
template <typename R>
__global__ void rks_real_to_complex(const R* a, cx<R>* b, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    b[i] = mkc(a[i], (R)0);
}

// s = safety * (eps ||u[idx]|| / ||err[idx]||)^(1/q), idx = |u|/max|u| > cutoff; one workgroup
template <typename R>
__global__ __launch_bounds__(1024) void rks_norm_kernel(const cx<R>* u, const cx<R>* err, int M, double eps,
                                                        double safety, double cutoff, int q, double* s_out) {
  __shared__ double red[2 * 17];
  double mx = 0.0;
  bool any = false;
  for (int m = threadIdx.x; m < M; m += 1024) {
    const double a = hypot((double)u[m].re, (double)u[m].im);
    mx = any ? nanmax(mx, a) : a;
    any = true;
  }
  mx = wg_max<1024>(mx, red);
  double su = 0.0, se = 0.0;
  for (int m = threadIdx.x; m < M; m += 1024) {
    const double ur = u[m].re, ui = u[m].im, er = err[m].re, ei = err[m].im;
    if (hypot(ur, ui) / mx > cutoff) {
      su += ur * ur + ui * ui;
      se += er * er + ei * ei;
    }
  }
  wg_sum2<1024>(su, se, red);
  if (threadIdx.x == 0) *s_out = rks_error_ratio(su, se, eps, safety, q, sizeof(R) < sizeof(double));
}

__global__ void rks_zero_int(int* p, int n) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0;
}

template <typename R>
__global__ void rks_twiddle_kernel(cx<R>* tw, int N) {
  for (int x = blockIdx.x * blockDim.x + threadIdx.x; x < N; x += gridDim.x * blockDim.x) {
    double s, c;
    sincospi(-2.0 * (double)x / (double)N, &s, &c);
    tw[x] = mkc((R)c, (R)s);
  }
}

__global__ void rks_f64_to_f32(const double* a, float* b, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) b[i] = (float)a[i];
}

// the Hankel matrix for the stepping kernels: transposed, engine precision
template <typename R>
__global__ void rks_transpose(const double* a, R* b, int n) {
  const int total = n * n;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x)
    b[i] = (R)a[(i % n) * n + i / n];
}

// Whether the last mode is damped at DAMPED times the rate at which a field of unit size is
// advected across it: -Re L >= DAMPED |coef| k.
constexpr double DAMPED = 100.0;
__host__ __device__ inline bool rks_damped(double re, double coef, double k) { return -re >= DAMPED * fabs(coef) * k; }

// Marks the advective trajectories whose last mode is not.
__global__ void rks_mark_undamped(const rks_inst* inst, int ninst, int* undamped) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ninst) return;
  const rks_inst& r = inst[i];
  const int m = r.m - 1;
  undamped[i] = rks_damped(r.L_complex ? r.L[2 * m] : r.L[m], r.nl_coef, ((const double*)r.kx)[m]) ? 0 : 1;
}

// ===========================================================================
// host side: plans and the C ABI
// ===========================================================================
#include "rkstiff_amd.h"

int rks_build_tableau(int method, rks_tableau* out);

// the stepping kernels of each precision (f64, f32, mix) x nonlinearity (advect, cubic,
// hankel) x method (any: the tableau read from memory); rks_k.hip, RKS_TABLE
#define RKS_TABLES(X)                                                                        \
  X(f64_advect_any) X(f64_advect_etd35) X(f64_advect_if34) X(f64_cubic_any) X(f64_cubic_etd35) \
  X(f64_cubic_if34) X(f64_hankel_any) X(f64_hankel_etd35) X(f32_advect_any)                   \
  X(f32_advect_etd35) X(f32_advect_if34) X(f32_cubic_any) X(f32_cubic_etd35) X(f32_cubic_if34) \
  X(f32_hankel_any) X(f32_hankel_etd35) X(mix_advect_any) X(mix_advect_etd35)                 \
  X(mix_advect_if34) X(mix_cubic_any) X(mix_cubic_etd35) X(mix_cubic_if34) X(mix_hankel_any)  \
  X(mix_hankel_etd35)
#define RKS_DECLARE_TABLE(name) bool rks_k_##name(int log2n, bool learn, int tile, rks_kernel_entry* e);
RKS_TABLES(RKS_DECLARE_TABLE)
rks_mlp_dev rks_mlp_device(const rks_mlp* n, int policy, double margin, double keep_lo, double keep_hi, int period);
int rks_mlp_device_of(const rks_mlp* n);

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

}  // namespace

// error channel shared with the proposer unit (rks_mlp.hip)
void rks_set_last_error(const std::string& msg) { g_err = msg; }

namespace {

#define HIPCHK(x)                                                                          \
  do {                                                                                     \
    hipError_t e_ = (x);                                                                   \
    if (e_ != hipSuccess) return fail(RKS_ERR_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

typedef rks_kernel_entry KernelEntry;

// Which stepping kernel runs a plan: the one compiled for its method where that exists, else
// the one that reads the tableau.  ETD35 and IF34 are the methods of the benchmark's workloads;
// their kernels are compiled for lin_ops of one kind (real with the advective and the rfft2
// terms, complex with the cubic ones) and read every L of the plan so.  A complex lin_op with the
// advective term (KdV), a real one with a cubic term, or a plan that holds both kinds takes the
// general kernel, which reads each trajectory's kind.  IF34 with the Hankel term is not compiled
// either: its general kernel takes 1.10 ms for one beam of nr = 100 and 2.95 for 1024, one of its
// own 0.79 and 2.56, and the radial runs use ETD35.
int method_variant(int method, int nlk, int n_complex, int ninst) {
  const bool real = nlk == RKS_NL_ADVECT_RFFT || nlk == RKS_NL_AC2D_RFFT2;
  if (n_complex != (real ? 0 : ninst)) return RKS_METH_ANY;
  if (method == RKS_M_ETD35) return method;
  if (method == RKS_M_IF34 && nlk != RKS_NL_HANKEL_CUBIC) return method;
  return RKS_METH_ANY;
}

// learn: the proposer variant (a proposer or training records are attached);
// tile: 0 the base tile (rks_threads), 1 twice and 2 four times the threads per trajectory
bool lookup(int prec, int nlk, int variant, int log2n, bool learn, KernelEntry* e, int tile = 0) {
#define RKS_PICK(p)                                                                                        \
  do {                                                                                                     \
    if (nlk == RKS_NL_ADVECT_RFFT)                                                                         \
      return variant == RKS_M_ETD35  ? rks_k_##p##_advect_etd35(log2n, learn, tile, e)                     \
             : variant == RKS_M_IF34 ? rks_k_##p##_advect_if34(log2n, learn, tile, e)                      \
                                     : rks_k_##p##_advect_any(log2n, learn, tile, e);                      \
    if (nlk == RKS_NL_CUBIC_FFT)                                                                           \
      return variant == RKS_M_ETD35  ? rks_k_##p##_cubic_etd35(log2n, learn, tile, e)                      \
             : variant == RKS_M_IF34 ? rks_k_##p##_cubic_if34(log2n, learn, tile, e)                       \
                                     : rks_k_##p##_cubic_any(log2n, learn, tile, e);                       \
    if (nlk == RKS_NL_HANKEL_CUBIC)                                                                        \
      return variant == RKS_M_ETD35 ? rks_k_##p##_hankel_etd35(log2n, learn, tile, e)                      \
                                    : rks_k_##p##_hankel_any(log2n, learn, tile, e);                       \
    return false;                                                                                          \
  } while (0)
  if (prec == RKS_F64) RKS_PICK(f64);
  if (prec == RKS_MIXED) RKS_PICK(mix);
  RKS_PICK(f32);
#undef RKS_PICK
}

// Tile of a trajectory whose caller chose none: by its size, method and precision, and not by
// what else is in the plan, so that its FP64 result is the same alone and in a batch.  A
// trajectory is a serial
// chain of butterflies, exchanges and stage sums, so more waves with fewer modes each shorten
// every link of it, until a transform takes more passes or a workgroup's registers and LDS
// keep others off a loaded CU.  Measured per FP64 evolve, base tile / twice / four times
// (MI355X; another interval for x 1000, ETD34 for the methods that read their tableau):
//   cubic ETD35  n = 512   x 1   3.49 / 2.21 ms          x 256   5.7 / 3.8 ms
//                n = 1024  x 1   6.73 / 3.80 / 2.38      x 256  11.5 / 6.7 / 4.0     x 1000  6.0 / 3.7 / 2.8 ms
//                n = 2048  x 1   6.68 / 4.09 / 3.24      x 256  13.2 / 7.8 / 5.3     x 1000  6.3 / 4.9 / 4.4
//                n = 4096  x 1   7.60 / 5.65 / 7.09      x 256  19.1 / 14.5 / 15.3   x 1000  9.7 / 8.1
//                n = 8192  x 1  12.04 / 12.77            x 256  30.2 / 27.0          x 1000 18.6 / 16.3
//         ETD34  n = 512   x 1   1.60 / 0.93             x 256   3.0 / 1.8           x 1000  3.8 / 2.5
//                n = 1024  x 1   1.89 / 1.04 / 0.63      x 256   4.4 / 2.4 / 1.5     x 1000  5.3 / 3.1 / 2.8
//                n = 2048  x 1   1.33 / 0.77 / 0.57      x 256   4.1 / 2.3 / 1.6     x 1000  5.3 / 3.5 / 3.7
//                n = 4096  x 1   1.05 / 0.74             x 256   3.1 / 2.0           x 1000  5.3 / 4.9
//                n = 8192  x 1   1.17 / 1.36             x 256   3.1 / 3.3           x 1000  8.8 / 10.9
//         IF34   n = 512   x 1   0.18 / 0.14             x 256   0.47 / 0.39         x 1000  1.00 / 0.89
//                n = 1024  x 1   0.35 / 0.23 / 0.17                                  x 1000  1.55 / 1.23 / 1.15
//                n = 2048  x 1   0.37 / 0.26 / 0.24                                  x 1000  2.00 / 1.84 / 2.11
//                n = 4096  x 1   0.43 / 0.35             x 256   1.29 / 1.00         x 1000  3.30 / 3.26
//                n = 8192  x 1   0.71 / 0.77                                         x 1000  6.9 / 7.0
//   advect IF34  n = 512   x 1   1.85 / 1.60             x 256   2.8 / 2.5           x 1000  1.03 / 1.00
//                n = 1024  x 1   3.28 / 2.26 / 2.03      x 256   4.0 / 3.0 / 2.8     x 1000  1.54 / 1.24 / 1.21
//                n = 2048  x 1   4.08 / 2.80 / 3.06      x 256   6.1 / 4.0 / 4.1     x 1000  1.88 / 1.64
//                n = 4096  x 1   4.93 / 3.94 / 6.24      x 256   8.2 / 5.8 / 8.9     x 1000  2.70 / 2.73
//                n = 8192  x 1   7.91 / 9.71             x 256  12.7 / 16.7
//         ETD35  n = 1024  x 1   0.62 / 0.38 / 0.29      x 256   1.37 / 0.85 / 0.68  x 1000  2.06 / 1.47 / 1.59
//                n = 4096  x 1   0.64 / 0.52             x 256   1.72 / 1.28         x 1000  4.32 / 3.93
//         ETD34  n = 512   x 1   0.61 / 0.39             x 256   0.95 / 0.62         x 1000  1.46 / 1.19
//                n = 1024  x 1   0.89 / 0.50 / 0.36      x 256   1.29 / 0.78 / 0.64  x 1000  2.10 / 1.45 / 1.60
//                n = 2048  x 1   0.77 / 0.48             x 256   1.25 / 0.85         x 1000  2.16 / 2.01
//                n = 4096  x 1   0.77 / 0.56             x 256   1.37 / 1.03         x 1000  3.09 / 3.31
// FP32 and MIXED runs gain as much, but keep the base tile: a tile has its own order of
// rounding, and in FP32 storage that moves the step sizes and with them the results (MIXED
// soliton ensembles by 4e-9, FP32 KS by 3e-6), so there the caller chooses.  Likewise an
// advective term on a grid whose last modes are not damped (rks_damped): a spectrum
// that reaches the grid's end amplifies rounding (viscosity 5e-4, n = 4096: 2e-3 of the
// state; KS: 1e-13).  The proposer
// counts accepted steps by the workgroup's size, so its kernels keep the base tile; so do
// runs that log their attempts, whose logs compare with the proposer's attempt by attempt.
int default_tile(int prec, int nlk, int variant, int log2n, bool base_only) {
  if (base_only || prec != RKS_F64 || nlk == RKS_NL_HANKEL_CUBIC || log2n < 9 || log2n == 13) return 0;
  if (log2n == 10 || (nlk == RKS_NL_CUBIC_FFT && log2n == 11 && variant != RKS_M_IF34)) return 2;
  return 1;
}

int ilog2(int n) {
  int l = 0;
  while ((1 << l) < n) ++l;
  return (1 << l) == n ? l : -1;
}

// size class of a Hankel grid of n radial points: 2^l >= n, l >= 4
int hankel_log2(int n) {
  int l = 4;
  while ((1 << l) < n) ++l;
  return l;
}

}  // namespace

struct rks_plan {
  int method = 0, nlk = 0, prec = 0, ninst = 0, device = 0, cu = 256;
  int esize = 16;  // state element bytes (complex)
  int coef_real = 0;  // coefficients stored real (RKS_CST_*_REAL)
  int variant = RKS_METH_ANY;  // method_variant
  int nsize = 16;  // NL / coefficient storage element bytes (complex)
  size_t coef_bytes_per_mode = 0;
  rks_tableau tab;
  rks_ctrl ctl;
  std::vector<rks_inst> h_inst;
  std::vector<rks_io> h_io;
  std::vector<int> modes;
  rks_tableau* d_tab = nullptr;
  rks_ctrl* d_ctl = nullptr;
  rks_inst* d_inst = nullptr;
  rks_io* d_io = nullptr;
  void* d_ws = nullptr;
  double* d_L = nullptr;
  void* d_kx = nullptr;
  double* d_log = nullptr;
  void* d_snap = nullptr;
  double* d_snap_t = nullptr;
  int* d_queue = nullptr;
  int* d_order = nullptr;
  void* d_tw[14] = {nullptr};
  std::vector<size_t> ws_off;
  std::vector<size_t> ws_modes;  // elements per workspace array (2-D: padded rows)
  // size buckets: instances grouped by log2(n)
  std::vector<int> bucket_log2, bucket_start, bucket_count;
  std::vector<int> order;
  int snap_cap = 0, store_freq = 0, log_cap = 0;
  // 2-D rfft2 engine (RKS_NL_AC2D_RFFT2): one grid size for the whole plan
  rks2_ctx* c2 = nullptr;
  int log2n2 = 0;
  // learned step-size proposer (attached by rks_plan_set_proposer) and
  // the training-record buffer (rks_set_records)
  rks_mlp_dev mlp{};
  float* d_rec = nullptr;
  int rec_cap = 0;
  // launch shape (rks_plan_set_launch): buckets on private streams, and a
  // cap on resident workgroups per CU per bucket (0: as many as fit)
  int concurrent = 1;
  std::vector<int> wg_per_cu;
  std::vector<int> undamped;        // per trajectory: its rounding at the grid's end need not decay
  std::vector<int> bucket_undamped;  // per bucket: how many are
  std::vector<int> tile;  // per bucket: 0 base tile, 1 twice, 2 four times the threads, -1 by default_tile
  std::vector<hipStream_t> bstream;
  std::vector<hipEvent_t> bdone;
  hipEvent_t fork = nullptr;
};

static void fill_ctrl(rks_ctrl* c, const rks_config* cfg);
static hipError_t upload_order(rks_plan* p);

// L[r][c] == L[(rows - r) mod rows][c] bitwise for every mode of a rows x cols
// lin_op in device memory (1-D: cols = 1): the ETD/IF coefficients of a mode
// depend on h L only, so mirror modes share them.
static bool mirror_symmetric(const double* L, int cplx, int rows, int cols) {
  const int w = cplx ? 2 : 1;
  const size_t rw = (size_t)cols * w;
  std::vector<double> v((size_t)rows * rw);
  if (hipMemcpy(v.data(), L, sizeof(double) * v.size(), hipMemcpyDeviceToHost) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  for (int r = 1; r < rows; ++r)
    if (std::memcmp(&v[(size_t)r * rw], &v[(size_t)(rows - r) * rw], sizeof(double) * rw) != 0) return false;
  return true;
}

extern "C" {

const char* rks_last_error(void) { return g_err.c_str(); }

int rks_get_tableau(int method, void* out, int bytes) {
  if (bytes < (int)sizeof(rks_tableau)) return fail(RKS_ERR_INVALID, "tableau buffer too small");
  rks_tableau t;
  if (rks_build_tableau(method, &t)) return fail(RKS_ERR_INVALID, "unknown method");
  std::memcpy(out, &t, sizeof(t));
  return RKS_OK;
}

int rks_sizeof(int what) {
  switch (what) {
    case 0: return (int)sizeof(rks_tableau);
    case 1: return (int)sizeof(rks_inst);
    case 2: return (int)sizeof(rks_io);
    case 3: return (int)sizeof(rks_ctrl);
    case 4: return (int)sizeof(rks_instance_desc);
    case 5: return (int)sizeof(rks_config);
    case 6: return (int)sizeof(rks_stats);
    default: return -1;
  }
}

int rks_plan_create(int method, int nl_kind, int precision, const rks_config* cfg, int ninst,
                    const rks_instance_desc* desc, rks_plan** out) {
  if (!out || !cfg || !desc || ninst <= 0) return fail(RKS_ERR_INVALID, "null argument or ninst <= 0");
  *out = nullptr;
  if (precision != RKS_F64 && precision != RKS_F32 && precision != RKS_MIXED)
    return fail(RKS_ERR_INVALID, "precision must be RKS_F64, RKS_F32 or RKS_MIXED");
  if (precision == RKS_MIXED && nl_kind == RKS_NL_NONE)
    return fail(RKS_ERR_INVALID, "mixed precision needs a built-in nonlinearity");
  if (nl_kind != RKS_NL_ADVECT_RFFT && nl_kind != RKS_NL_CUBIC_FFT && nl_kind != RKS_NL_NONE &&
      nl_kind != RKS_NL_AC2D_RFFT2 && nl_kind != RKS_NL_HANKEL_CUBIC)
    return fail(RKS_ERR_INVALID, "unknown nonlinear kind");
  const bool is2d = nl_kind == RKS_NL_AC2D_RFFT2;
  const bool hankel = nl_kind == RKS_NL_HANKEL_CUBIC;
  rks_plan* p = new rks_plan();
  if (rks_build_tableau(method, &p->tab)) {
    delete p;
    return fail(RKS_ERR_INVALID, "unknown method");
  }
  p->method = method;
  p->nlk = nl_kind;
  p->prec = precision;
  p->ninst = ninst;
  p->esize = precision == RKS_F32 ? 8 : 16;
  p->nsize = precision == RKS_F64 ? 16 : 8;
  // coefficient layout: index order for uniform precision; propagators (state
  // precision) first, then the rest, for mixed precision.  Plans with a
  // built-in term whose lin_op is real everywhere store every coefficient real
  // at half the bytes: z = h L is real, so are exp and the psi functions, and
  // the reference's complex coefficients have imaginary parts that are exactly
  // zero, or rounding (below 2e-15 of the array's largest value) in the
  // contour means, whose nodes come in conjugate pairs.  The generic path (no built-in term) keeps the
  // reference's complex arrays.
  {
    int n_complex = 0;
    for (int i = 0; i < ninst; ++i) n_complex += desc[i].L_is_complex ? 1 : 0;
    const bool real = nl_kind != RKS_NL_NONE && n_complex == 0;
    p->coef_real = real ? 1 : 0;
    p->coef_bytes_per_mode = (size_t)rks_tab::layout(p->tab, p->esize, p->nsize, real);
    p->variant = method_variant(method, nl_kind, n_complex, ninst);
  }
  fill_ctrl(&p->ctl, cfg);
  if (cfg->contour_points < 2) {
    delete p;
    return fail(RKS_ERR_INVALID, "contour_points must be > 1");
  }
  (void)hipGetDevice(&p->device);
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, p->device) == hipSuccess) p->cu = prop.multiProcessorCount;
  // geometry
  size_t ws_total = 0, L_total = 0, kx_total = 0;
  p->modes.resize(ninst);
  p->ws_off.resize(ninst);
  p->ws_modes.resize(ninst);
  std::vector<size_t> Loff(ninst), kxoff(ninst);
  std::vector<char> kx_copy(ninst, 1);
  std::map<const double*, size_t> y_shared;  // Hankel matrices by source pointer
  for (int i = 0; i < ninst; ++i) {
    const int n = desc[i].n;
    int m;
    if (hankel) {
      if (n < 4 || n > 1024) {
        rks_plan_destroy(p);
        return fail(RKS_ERR_INVALID, "Hankel grids need 4 to 1024 radial points");
      }
      if (!desc[i].kx || !(desc[i].nl_scale > 0.0)) {
        rks_plan_destroy(p);
        return fail(RKS_ERR_INVALID, "the Hankel nonlinearity needs the matrix Y (kx) and S > 0 (nl_scale)");
      }
      m = n;
    } else if (nl_kind == RKS_NL_ADVECT_RFFT) {
      const int l2 = ilog2(n);
      if (l2 < 4 || l2 > 13) {
        rks_plan_destroy(p);
        return fail(RKS_ERR_INVALID, "rfft grid size must be a power of two in [16, 8192]");
      }
      m = n / 2 + 1;
    } else if (is2d) {
      const int l2 = ilog2(n);
      if (desc[i].ny != n || !rks2_supported(precision, l2)) {
        rks_plan_destroy(p);
        return fail(RKS_ERR_INVALID, "rfft2 grids must be square, N x N with N a power of two in [32, 512]");
      }
      if (i > 0 && desc[i].n != desc[0].n) {
        rks_plan_destroy(p);
        return fail(RKS_ERR_INVALID, "all trajectories of an rfft2 plan share one grid size");
      }
      m = rks2_modes(l2);
      p->log2n2 = l2;
    } else if (nl_kind == RKS_NL_CUBIC_FFT) {
      const int l2 = ilog2(n);
      if (l2 < 4 || l2 > 13) {
        rks_plan_destroy(p);
        return fail(RKS_ERR_INVALID, "fft grid size must be a power of two in [16, 8192]");
      }
      m = n;
    } else {
      if (n <= 0) {
        rks_plan_destroy(p);
        return fail(RKS_ERR_INVALID, "number of modes must be positive");
      }
      m = n;
    }
    if (!desc[i].L) {
      rks_plan_destroy(p);
      return fail(RKS_ERR_INVALID, "lin_op pointer is null");
    }
    if (nl_kind == RKS_NL_ADVECT_RFFT && !desc[i].kx) {
      rks_plan_destroy(p);
      return fail(RKS_ERR_INVALID, "advective nonlinearity needs kx");
    }
    p->modes[i] = m;
    p->ws_off[i] = ws_total;
    // elements of each workspace array: the 2-D engine pads rows to whole cache lines,
    // the Hankel kind pads the modes to its size class
    const size_t mw = is2d ? (size_t)rks2_imodes(ilog2(n)) : hankel ? ((size_t)1 << hankel_log2(n)) : (size_t)m;
    p->ws_modes[i] = mw;
    ws_total += rks_align256((size_t)p->tab.nslot * mw * p->nsize) + 2 * rks_align256(mw * p->esize) +
                rks_align256(p->coef_bytes_per_mode * mw);
    if (is2d)  // transform buffer T, rows padded to whole cache lines
      ws_total += rks_align256((size_t)n * rks2_t_stride(n, (int)p->esize) * p->esize);
    Loff[i] = L_total;
    L_total += (size_t)m * (desc[i].L_is_complex ? 2 : 1);
    if (hankel) {
      // one device copy per distinct matrix (every trajectory of a radial grid reads the same Y)
      const auto it = y_shared.find(desc[i].kx);
      if (it != y_shared.end()) {
        kxoff[i] = it->second;
        kx_copy[i] = 0;
      } else {
        kxoff[i] = kx_total;
        y_shared[desc[i].kx] = kx_total;
        kx_total += (size_t)m * m;
      }
    } else {
      kxoff[i] = kx_total;
      kx_total += (size_t)m;
    }
  }
  HIPCHK(hipMalloc(&p->d_tab, sizeof(rks_tableau)));
  HIPCHK(hipMalloc(&p->d_ctl, sizeof(rks_ctrl)));
  HIPCHK(hipMalloc(&p->d_inst, sizeof(rks_inst) * ninst));
  HIPCHK(hipMalloc(&p->d_io, sizeof(rks_io) * ninst));
  HIPCHK(hipMalloc(&p->d_ws, ws_total));
  HIPCHK(hipMalloc(&p->d_L, L_total * sizeof(double)));
  HIPCHK(hipMalloc(&p->d_kx, kx_total * (p->esize / 2)));
  HIPCHK(hipMalloc(&p->d_queue, sizeof(int) * 64));
  HIPCHK(hipMalloc(&p->d_order, sizeof(int) * 2 * ninst));
  HIPCHK(hipMemcpy(p->d_tab, &p->tab, sizeof(rks_tableau), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(p->d_ctl, &p->ctl, sizeof(rks_ctrl), hipMemcpyHostToDevice));
  HIPCHK(hipMemset(p->d_ws, 0, ws_total));
  double* d_kx64 = nullptr;
  if (kx_total) HIPCHK(hipMalloc(&d_kx64, kx_total * sizeof(double)));
  for (int i = 0; i < ninst; ++i) {
    const int m = p->modes[i];
    HIPCHK(hipMemcpy(p->d_L + Loff[i], desc[i].L, sizeof(double) * m * (desc[i].L_is_complex ? 2 : 1),
                     hipMemcpyDefault));
    const size_t nk = hankel ? (size_t)m * m : (size_t)m;
    if (!kx_copy[i]) continue;
    if (desc[i].kx) HIPCHK(hipMemcpy(d_kx64 + kxoff[i], desc[i].kx, sizeof(double) * nk, hipMemcpyDefault));
    else HIPCHK(hipMemset(d_kx64 + kxoff[i], 0, sizeof(double) * nk));
  }
  if (hankel) {
    for (int i = 0; i < ninst; ++i) {
      if (!kx_copy[i]) continue;
      const int m = p->modes[i];
      if (precision != RKS_F32)
        hipLaunchKernelGGL(rks_transpose<double>, dim3(256), dim3(256), 0, 0, d_kx64 + kxoff[i],
                           (double*)p->d_kx + kxoff[i], m);
      else
        hipLaunchKernelGGL(rks_transpose<float>, dim3(256), dim3(256), 0, 0, d_kx64 + kxoff[i],
                           (float*)p->d_kx + kxoff[i], m);
      HIPCHK(hipGetLastError());
    }
  } else if (precision != RKS_F32) {
    HIPCHK(hipMemcpy(p->d_kx, d_kx64, kx_total * sizeof(double), hipMemcpyDeviceToDevice));
  } else if (kx_total) {
    hipLaunchKernelGGL(rks_f64_to_f32, dim3(256), dim3(256), 0, 0, d_kx64, (float*)p->d_kx, (int)kx_total);
    HIPCHK(hipGetLastError());
  }
  HIPCHK(hipDeviceSynchronize());
  if (d_kx64) (void)hipFree(d_kx64);
  // instance records
  p->h_inst.assign(ninst, rks_inst());
  p->h_io.assign(ninst, rks_io());
  for (int i = 0; i < ninst; ++i) {
    rks_inst& r = p->h_inst[i];
    std::memset(&r, 0, sizeof(r));
    r.n = desc[i].n;
    r.m = p->modes[i];
    r.L_complex = desc[i].L_is_complex ? 1 : 0;
    r.L = p->d_L + Loff[i];
    r.kx = (char*)p->d_kx + kxoff[i] * (p->esize / 2);
    r.nl_coef = desc[i].nl_coef;
    r.nl_scale = hankel ? desc[i].nl_scale : 0.0;
    r.ws = (char*)p->d_ws + p->ws_off[i];
    r.h_coeff = std::nan("");
    r.ubuf = -1;
    r.rec_pending = -1;
    for (int s = 0; s < RKS_MAX_SLOTS; ++s) r.slot_map[s] = s;
    if (nl_kind == RKS_NL_CUBIC_FFT) r.coef_sym = mirror_symmetric(r.L, r.L_complex, r.m, 1) ? 1 : 0;
    if (is2d) r.coef_sym = mirror_symmetric(r.L, r.L_complex, r.n, r.m / r.n) ? 1 : 0;
  }
  HIPCHK(hipMemcpy(p->d_inst, p->h_inst.data(), sizeof(rks_inst) * ninst, hipMemcpyHostToDevice));
  if (is2d) {
    const int l = p->log2n2, N = 1 << l, m = p->modes[0];
    HIPCHK(hipMalloc(&p->d_tw[l], (size_t)N * p->esize));
    if (precision != RKS_F32)
      hipLaunchKernelGGL(rks_twiddle_kernel<double>, dim3((N + 255) / 256), dim3(256), 0, 0, (cx<double>*)p->d_tw[l],
                         N);
    else
      hipLaunchKernelGGL(rks_twiddle_kernel<float>, dim3((N + 255) / 256), dim3(256), 0, 0, (cx<float>*)p->d_tw[l],
                         N);
    HIPCHK(hipGetLastError());
    HIPCHK(hipDeviceSynchronize());
    const size_t mw = p->ws_modes[0];
    const size_t off_c0 = rks_align256((size_t)p->tab.nslot * mw * p->nsize);
    const size_t off_c1 = off_c0 + rks_align256(mw * p->esize);
    const size_t off_cf = off_c1 + rks_align256(mw * p->esize);
    const size_t off_T = off_cf + rks_align256(p->coef_bytes_per_mode * mw);
    if (rks2_create(&p->c2, precision, p->variant, l, ninst, p->d_tab, p->d_ctl, p->d_inst, p->d_io, p->d_tw[l], off_c0, off_c1,
                    off_cf, off_T)) {
      rks_plan_destroy(p);
      return fail(RKS_ERR_HIP, "2-D engine set-up failed");
    }
  }
  // buckets by size
  if (nl_kind != RKS_NL_NONE && !is2d) {
    std::vector<std::vector<int>> byl(14);
    for (int i = 0; i < ninst; ++i) byl[hankel ? hankel_log2(desc[i].n) : ilog2(desc[i].n)].push_back(i);
    for (int l = 13; l >= 4; --l) {
      if (byl[l].empty()) continue;
      p->bucket_log2.push_back(l);
      p->bucket_start.push_back((int)p->order.size());
      p->bucket_count.push_back((int)byl[l].size());
      for (int i : byl[l]) p->order.push_back(i);
      KernelEntry e;
      if (!lookup(precision, nl_kind, p->variant, l, false, &e)) {
        rks_plan_destroy(p);
        return fail(RKS_ERR_INVALID, "no kernel for this size");
      }
      HIPCHK(hipFuncSetAttribute(e.fn, hipFuncAttributeMaxDynamicSharedMemorySize, e.lds));
      KernelEntry el;
      if (lookup(precision, nl_kind, p->variant, l, true, &el))
        HIPCHK(hipFuncSetAttribute(el.fn, hipFuncAttributeMaxDynamicSharedMemorySize, el.lds));
      for (int tile = 1; tile <= 2; ++tile)
        if (lookup(precision, nl_kind, p->variant, l, false, &el, tile))
          HIPCHK(hipFuncSetAttribute(el.fn, hipFuncAttributeMaxDynamicSharedMemorySize, el.lds));
      if (hankel) continue;  // no transform tables
      const int N = 1 << l;
      HIPCHK(hipMalloc(&p->d_tw[l], (size_t)N * p->esize));
      if (precision != RKS_F32)
        hipLaunchKernelGGL(rks_twiddle_kernel<double>, dim3((N + 255) / 256), dim3(256), 0, 0,
                           (cx<double>*)p->d_tw[l], N);
      else
        hipLaunchKernelGGL(rks_twiddle_kernel<float>, dim3((N + 255) / 256), dim3(256), 0, 0,
                           (cx<float>*)p->d_tw[l], N);
      HIPCHK(hipGetLastError());
    }
    p->undamped.assign(ninst, 0);
    if (nl_kind == RKS_NL_ADVECT_RFFT && precision == RKS_F64 && ninst <= 4) {
      // a few: from the caller's arrays, without a launch and a read back
      for (int i = 0; i < ninst; ++i) {
        const int m = p->modes[i] - 1;
        double re = 0.0, k = 0.0;
        HIPCHK(hipMemcpy(&re, (const double*)desc[i].L + (desc[i].L_is_complex ? 2 * m : m), sizeof(double), hipMemcpyDefault));
        HIPCHK(hipMemcpy(&k, (const double*)desc[i].kx + m, sizeof(double), hipMemcpyDefault));
        p->undamped[i] = rks_damped(re, desc[i].nl_coef, k) ? 0 : 1;
      }
    } else if (nl_kind == RKS_NL_ADVECT_RFFT && precision == RKS_F64) {
      hipLaunchKernelGGL(rks_mark_undamped, dim3((ninst + 255) / 256), dim3(256), 0, 0, p->d_inst, ninst, p->d_order);
      HIPCHK(hipGetLastError());
      HIPCHK(hipMemcpy(p->undamped.data(), p->d_order, sizeof(int) * ninst, hipMemcpyDeviceToHost));
    }
    for (size_t b = 0; b < p->bucket_start.size(); ++b) {
      int n = 0;
      for (int k = 0; k < p->bucket_count[b]; ++k) n += p->undamped[p->order[p->bucket_start[b] + k]];
      p->bucket_undamped.push_back(n);
    }
    HIPCHK(upload_order(p));
    HIPCHK(hipDeviceSynchronize());
  }
  *out = p;
  return RKS_OK;
}

static void fill_ctrl(rks_ctrl* c, const rks_config* cfg) {
  c->epsilon = cfg->epsilon;
  c->incr_f = cfg->incr_f;
  c->decr_f = cfg->decr_f;
  c->safety_f = cfg->safety_f;
  c->adapt_cutoff = cfg->adapt_cutoff;
  c->minh = cfg->minh;
  c->max_s = cfg->max_s;
  c->min_s = cfg->min_s;
  c->max_loops = cfg->max_loops;
  c->contour_points = cfg->contour_points;
  c->modecutoff = cfg->modecutoff;
  c->contour_radius = cfg->contour_radius;
}

// d_order: every bucket's trajectories in the order in which its workgroups take them, then
// every bucket's once more with those that keep the base tile (undamped) behind the others.
static hipError_t upload_order(rks_plan* p) {
  std::vector<int> o(p->order);
  o.insert(o.end(), p->order.begin(), p->order.end());
  for (size_t b = 0; b < p->bucket_start.size(); ++b) {
    auto first = o.begin() + p->ninst + p->bucket_start[b];
    std::stable_partition(first, first + p->bucket_count[b], [&](int i) { return !p->undamped[i]; });
  }
  return hipMemcpy(p->d_order, o.data(), sizeof(int) * o.size(), hipMemcpyHostToDevice);
}

int rks_set_config(rks_plan* p, const rks_config* cfg, hipStream_t stream) {
  if (!p || !cfg) return fail(RKS_ERR_INVALID, "null argument");
  if (cfg->contour_points < 2) return fail(RKS_ERR_INVALID, "contour_points must be > 1");
  fill_ctrl(&p->ctl, cfg);
  HIPCHK(hipMemcpyAsync(p->d_ctl, &p->ctl, sizeof(rks_ctrl), hipMemcpyHostToDevice, stream));
  HIPCHK(hipStreamSynchronize(stream));
  return RKS_OK;
}

int rks_plan_destroy(rks_plan* p) {
  if (!p) return RKS_OK;
  (void)hipFree(p->d_tab);
  (void)hipFree(p->d_ctl);
  (void)hipFree(p->d_inst);
  (void)hipFree(p->d_io);
  (void)hipFree(p->d_ws);
  (void)hipFree(p->d_L);
  (void)hipFree(p->d_kx);
  (void)hipFree(p->d_log);
  (void)hipFree(p->d_snap);
  (void)hipFree(p->d_snap_t);
  (void)hipFree(p->d_queue);
  (void)hipFree(p->d_order);
  (void)hipFree(p->d_rec);
  for (hipStream_t st : p->bstream) (void)hipStreamDestroy(st);
  for (hipEvent_t ev : p->bdone) (void)hipEventDestroy(ev);
  if (p->fork) (void)hipEventDestroy(p->fork);
  for (int l = 0; l < 14; ++l) (void)hipFree(p->d_tw[l]);
  rks2_destroy(p->c2);
  delete p;
  return RKS_OK;
}

int rks_plan_info(const rks_plan* p, int* ninst, int* nslot, int* ncoef, int* esize) {
  if (!p) return fail(RKS_ERR_INVALID, "null plan");
  if (ninst) *ninst = p->ninst;
  if (nslot) *nslot = p->tab.nslot;
  if (ncoef) *ncoef = p->tab.ncoef;
  if (esize) *esize = p->esize;
  return RKS_OK;
}

int rks_set_storage(rks_plan* p, int store_freq, int snap_cap, int log_cap) {
  if (!p) return fail(RKS_ERR_INVALID, "null plan");
  if (store_freq < 0 || snap_cap < 0 || log_cap < 0) return fail(RKS_ERR_INVALID, "negative storage size");
  if (store_freq > 0 && snap_cap < 2) return fail(RKS_ERR_INVALID, "snapshot capacity must be >= 2");
  if (p->nlk == RKS_NL_NONE) return fail(RKS_ERR_INVALID, "storage needs a built-in nonlinearity");
  HIPCHK(hipDeviceSynchronize());
  (void)hipFree(p->d_snap);
  (void)hipFree(p->d_snap_t);
  (void)hipFree(p->d_log);
  p->d_snap = nullptr;
  p->d_snap_t = nullptr;
  p->d_log = nullptr;
  size_t tot_modes = 0;
  for (int m : p->modes) tot_modes += (size_t)m;
  if (store_freq > 0) {
    HIPCHK(hipMalloc(&p->d_snap, tot_modes * snap_cap * p->esize));
    HIPCHK(hipMalloc(&p->d_snap_t, sizeof(double) * snap_cap * p->ninst));
  }
  if (log_cap > 0) HIPCHK(hipMalloc(&p->d_log, sizeof(double) * 2 * (size_t)log_cap * p->ninst));
  // patch the device records: read back state, set pointers, write back
  HIPCHK(hipMemcpy(p->h_inst.data(), p->d_inst, sizeof(rks_inst) * p->ninst, hipMemcpyDeviceToHost));
  size_t off = 0;
  for (int i = 0; i < p->ninst; ++i) {
    rks_inst& r = p->h_inst[i];
    r.store_freq = store_freq;
    r.snap_cap = store_freq > 0 ? snap_cap : 0;
    r.snap = store_freq > 0 ? (char*)p->d_snap + off * snap_cap * p->esize : nullptr;
    r.snap_t = store_freq > 0 ? p->d_snap_t + (size_t)snap_cap * i : nullptr;
    r.log_cap = log_cap;
    r.log = log_cap > 0 ? p->d_log + 2 * (size_t)log_cap * i : nullptr;
    off += (size_t)p->modes[i];
  }
  HIPCHK(hipMemcpy(p->d_inst, p->h_inst.data(), sizeof(rks_inst) * p->ninst, hipMemcpyHostToDevice));
  p->store_freq = store_freq;
  p->snap_cap = snap_cap;
  p->log_cap = log_cap;
  return RKS_OK;
}

// start of the coefficient region of instance `inst` (mirror of run_instance)
// Invalidate an instance's coefficient cache: rks_coeffs overwrites it with
// all M modes of another step size.
__global__ void rks_coef_invalidate(rks_inst* in) { in->h_coeff = __builtin_nan(""); }

static char* inst_cbase(const rks_plan* p, int inst) {
  const size_t M = p->ws_modes[inst];
  return (char*)p->h_inst[inst].ws + rks_align256((size_t)p->tab.nslot * M * p->nsize) +
         2 * rks_align256(M * p->esize);
}

// the proposer variant runs: a proposer or training records are attached
static bool learns(const rks_plan* p) { return p->mlp.on || p->d_rec != nullptr; }

// the tile of bucket b's trajectories (those with damped, or undamped, last modes): the caller's
// choice (a tile without a proposer variant gives way to the base tile when a proposer or records
// are attached after it), else default_tile
static int bucket_tile(const rks_plan* p, size_t b, bool undamped) {
  if (b < p->tile.size() && p->tile[b] >= 0) {
    KernelEntry e;
    return lookup(p->prec, p->nlk, p->variant, p->bucket_log2[b], learns(p), &e, p->tile[b]) ? p->tile[b] : 0;
  }
  return default_tile(p->prec, p->nlk, p->variant, p->bucket_log2[b], undamped || learns(p) || p->d_log != nullptr);
}

// The launches of a plan: a bucket each, or two where its trajectories run on different tiles.
struct LaunchPart {
  size_t bucket;
  const int* order;
  int count, tile;
};

static std::vector<LaunchPart> launch_parts(const rks_plan* p) {
  std::vector<LaunchPart> v;
  for (size_t b = 0; b < p->bucket_log2.size(); ++b) {
    const int n = p->bucket_count[b], nu = p->bucket_undamped[b], start = p->bucket_start[b];
    const int td = bucket_tile(p, b, false), tu = bucket_tile(p, b, true);
    if (nu == 0 || nu == n || td == tu) {
      v.push_back({b, p->d_order + start, n, nu == n ? tu : td});
    } else {
      v.push_back({b, p->d_order + p->ninst + start, n - nu, td});
      v.push_back({b, p->d_order + p->ninst + start + n - nu, nu, tu});
    }
  }
  return v;
}

static int launch_all(rks_plan* p, int mode, hipStream_t stream) {
  if (p->c2) {
    const hipError_t e = rks2_run(p->c2, p->tab, mode, p->store_freq > 0, stream);
    if (e != hipSuccess) return fail(RKS_ERR_HIP, std::string("2-D engine: ") + hipGetErrorString(e));
    return RKS_OK;
  }
  rks_launch L{};
  L.mlp = p->mlp;
  L.tab = p->d_tab;
  L.ctl = p->d_ctl;
  L.inst = p->d_inst;
  L.io = p->d_io;
  L.mode = mode;
  const std::vector<LaunchPart> parts = launch_parts(p);
  const size_t np = parts.size();
  const bool learn = learns(p);
  std::vector<KernelEntry> kern(np);
  std::vector<int> grid(np);
  bool queued = false;
  for (size_t i = 0; i < np; ++i) {
    KernelEntry& e = kern[i];
    const size_t b = parts[i].bucket;
    if (!lookup(p->prec, p->nlk, p->variant, p->bucket_log2[b], learn, &e, parts[i].tile))
      return fail(RKS_ERR_INVALID, "no kernel for this grid size, variant and tile");
    grid[i] = parts[i].count;
    if (grid[i] <= p->cu) continue;  // a CU holds at least one workgroup
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, e.fn, e.threads, e.lds) != hipSuccess || per_cu < 1)
      per_cu = 1;
    if (b < p->wg_per_cu.size() && p->wg_per_cu[b] > 0 && p->wg_per_cu[b] < per_cu) per_cu = p->wg_per_cu[b];
    if (grid[i] > per_cu * p->cu) {
      grid[i] = per_cu * p->cu;
      queued = true;
    }
  }
  // the queue's counters, where a launch has more trajectories than workgroups: a launch of its
  // own, 3 us of a single step (62 -> 59)
  if (queued) {
    hipLaunchKernelGGL(rks_zero_int, dim3(1), dim3(64), 0, stream, p->d_queue, 64);
    HIPCHK(hipGetLastError());
  }
  const bool conc = p->concurrent && np > 1;
  if (conc) {
    // fork: every launch's stream waits for the caller's stream (queue counters cleared)
    if (p->bstream.size() < np) {
      HIPCHK(hipDeviceSynchronize());
      if (!p->fork) HIPCHK(hipEventCreateWithFlags(&p->fork, hipEventDisableTiming));
      while (p->bstream.size() < np) {
        hipStream_t st;
        hipEvent_t ev;
        HIPCHK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
        p->bstream.push_back(st);
        HIPCHK(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
        p->bdone.push_back(ev);
      }
    }
    HIPCHK(hipEventRecord(p->fork, stream));
  }
  for (size_t i = 0; i < np; ++i) {
    const KernelEntry& e = kern[i];
    L.order = parts[i].order;
    L.count = parts[i].count;
    L.queue = grid[i] < L.count ? p->d_queue + i : nullptr;
    L.tw = p->d_tw[p->bucket_log2[parts[i].bucket]];
    void* args[] = {&L};
    hipStream_t st = stream;
    if (conc) {
      st = p->bstream[i];
      HIPCHK(hipStreamWaitEvent(st, p->fork, 0));
    }
    HIPCHK(hipLaunchKernel(e.fn, dim3(grid[i]), dim3(e.threads), args, (size_t)e.lds, st));
    if (conc) HIPCHK(hipEventRecord(p->bdone[i], st));
  }
  // join after every launch is queued: a wait on the caller's stream is a
  // barrier in the hardware queue that stream maps to, and a bucket stream
  // sharing that queue would otherwise start only when the earlier ones end
  if (conc)
    for (size_t i = 0; i < np; ++i) HIPCHK(hipStreamWaitEvent(stream, p->bdone[i], 0));
  return RKS_OK;
}

static int upload_io(rks_plan* p, const void* const* u_in, void* const* u_out, const double* t0,
                     const double* tf, const double* h, int reset, int resume, hipStream_t stream) {
  for (int i = 0; i < p->ninst; ++i) {
    rks_io& o = p->h_io[i];
    if (!resume) {
      if (!u_in || !u_out || !u_in[i] || !u_out[i]) return fail(RKS_ERR_INVALID, "null state pointer");
      if (u_in[i] == u_out[i]) return fail(RKS_ERR_INVALID, "u_in and u_out must not alias");
      o.u_in = u_in[i];
      o.u_out = u_out[i];
      o.t0 = t0 ? t0[i] : 0.0;
      o.tf = tf ? tf[i] : 0.0;
      o.h_in = h ? h[i] : 0.0;
    }
    o.reset = reset;
    o.resume = resume;
  }
  HIPCHK(hipMemcpyAsync(p->d_io, p->h_io.data(), sizeof(rks_io) * p->ninst, hipMemcpyHostToDevice, stream));
  return RKS_OK;
}

int rks_evolve(rks_plan* p, const void* const* u0, void* const* uf, const double* t0, const double* tf,
               const double* h, hipStream_t stream) {
  if (!p) return fail(RKS_ERR_INVALID, "null plan");
  if (p->nlk == RKS_NL_NONE) return fail(RKS_ERR_INVALID, "evolve needs a built-in nonlinearity");
  for (int i = 0; i < p->ninst; ++i) {
    if (!(h && h[i] >= 0.0)) return fail(RKS_ERR_INVALID, "step size must be >= 0");
    if (!p->tab.adaptive && t0[i] < tf[i] && !(h[i] > 0.0))
      return fail(RKS_ERR_INVALID, "constant-step evolve needs h > 0");
    if (!p->tab.adaptive && (tf[i] - t0[i]) / h[i] > 1e9)
      return fail(RKS_ERR_INVALID, "constant-step evolve would take more than 1e9 steps");
  }
  int rc = upload_io(p, u0, uf, t0, tf, h, 1, 0, stream);
  if (rc) return rc;
  return launch_all(p, RKS_MODE_EVOLVE, stream);
}

int rks_resume(rks_plan* p, hipStream_t stream) {
  if (!p) return fail(RKS_ERR_INVALID, "null plan");
  int rc = upload_io(p, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 1, stream);
  if (rc) return rc;
  return launch_all(p, RKS_MODE_EVOLVE, stream);
}

int rks_step(rks_plan* p, const void* const* u, void* const* u_new, const double* h, hipStream_t stream) {
  if (!p) return fail(RKS_ERR_INVALID, "null plan");
  if (p->nlk == RKS_NL_NONE) return fail(RKS_ERR_INVALID, "step needs a built-in nonlinearity");
  for (int i = 0; i < p->ninst; ++i)
    if (!(h && h[i] >= 0.0)) return fail(RKS_ERR_INVALID, "step size must be >= 0");
  int rc = upload_io(p, u, u_new, nullptr, nullptr, h, 0, 0, stream);
  if (rc) return rc;
  return launch_all(p, RKS_MODE_STEP, stream);
}

int rks_reset(rks_plan* p, hipStream_t stream) {
  if (!p) return fail(RKS_ERR_INVALID, "null plan");
  HIPCHK(hipStreamSynchronize(stream));
  HIPCHK(hipMemcpy(p->h_inst.data(), p->d_inst, sizeof(rks_inst) * p->ninst, hipMemcpyDeviceToHost));
  for (auto& r : p->h_inst) {
    r.started = 0;
    r.accept = 0;
    r.h_coeff = std::nan("");
    r.ubuf = -1;
    r.rec_pending = -1;
    r.status = RKS_ST_OK;
    for (int s = 0; s < RKS_MAX_SLOTS; ++s) r.slot_map[s] = s;
  }
  HIPCHK(hipMemcpy(p->d_inst, p->h_inst.data(), sizeof(rks_inst) * p->ninst, hipMemcpyHostToDevice));
  return RKS_OK;
}

int rks_nl_eval(rks_plan* p, const void* const* u, void* const* nl_out, hipStream_t stream) {
  if (!p) return fail(RKS_ERR_INVALID, "null plan");
  if (p->nlk == RKS_NL_NONE) return fail(RKS_ERR_INVALID, "no built-in nonlinearity");
  int rc = upload_io(p, u, nl_out, nullptr, nullptr, nullptr, 0, 0, stream);
  if (rc) return rc;
  return launch_all(p, RKS_MODE_NL, stream);
}

int rks_coeffs(rks_plan* p, int inst, double h, void* dst, hipStream_t stream) {
  if (!p || inst < 0 || inst >= p->ninst) return fail(RKS_ERR_INVALID, "bad plan or instance");
  if (p->prec == RKS_MIXED && dst) return fail(RKS_ERR_INVALID, "coefficient copy-out needs uniform precision");
  const int M = p->modes[inst];
  const size_t nbytes = (size_t)p->tab.ncoef * M * p->esize;
  const rks_inst& r = p->h_inst[inst];
  char* cbase = inst_cbase(p, inst);
  const int grid = (M + 255) / 256;
  if (p->prec == RKS_F64)
    hipLaunchKernelGGL(rks_coef_kernel<double>, dim3(grid), dim3(256), 0, stream, p->d_tab, p->d_ctl, r.L,
                       r.L_complex, M, h, cbase);
  else if (p->prec == RKS_F32)
    hipLaunchKernelGGL(rks_coef_kernel<float>, dim3(grid), dim3(256), 0, stream, p->d_tab, p->d_ctl, r.L,
                       r.L_complex, M, h, cbase);
  else
    return fail(RKS_ERR_INVALID, "mixed-precision coefficients are generated inside the stepping kernel");
  HIPCHK(hipGetLastError());
  hipLaunchKernelGGL(rks_coef_invalidate, dim3(1), dim3(1), 0, stream, p->d_inst + inst);
  HIPCHK(hipGetLastError());
  if (dst && p->coef_real) {
    // real coefficient storage: ncoef x M reals, returned as complex
    const size_t n = (size_t)p->tab.ncoef * M;
    const dim3 grid((unsigned)((n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096));
    if (p->prec == RKS_F64)
      hipLaunchKernelGGL(rks_real_to_complex<double>, grid, dim3(256), 0, stream, (const double*)cbase,
                         (cx<double>*)dst, n);
    else
      hipLaunchKernelGGL(rks_real_to_complex<float>, grid, dim3(256), 0, stream, (const float*)cbase,
                         (cx<float>*)dst, n);
    HIPCHK(hipGetLastError());
  } else if (dst) {
    HIPCHK(hipMemcpyAsync(dst, cbase, nbytes, hipMemcpyDeviceToDevice, stream));
  }
  return RKS_OK;
}

int rks_combine(rks_plan* p, int inst, int stage, double h, const void* u, const void* const* slots, void* out,
                hipStream_t stream) {
  if (!p || inst < 0 || inst >= p->ninst) return fail(RKS_ERR_INVALID, "bad plan or instance");
  if (p->prec == RKS_MIXED) return fail(RKS_ERR_INVALID, "generic path needs uniform precision");
  const rks_tableau& tb = p->tab;
  const rks_term* terms;
  int nterm;
  const bool is_err = (stage == -1);
  if (stage >= 0 && stage < tb.nstage) {
    terms = tb.st[stage].t;
    nterm = tb.st[stage].nterm;
  } else if (is_err && tb.adaptive) {
    terms = tb.err;
    nterm = tb.nerr;
  } else {
    return fail(RKS_ERR_INVALID, "bad stage index");
  }
  if (!out) return fail(RKS_ERR_INVALID, "null output");
  if (!is_err && !u) return fail(RKS_ERR_INVALID, "null u");
  rks_combine_args A;
  std::memset(&A, 0, sizeof(A));
  for (int s = 0; s < tb.nslot && s < RKS_MAX_SLOTS; ++s) A.slots[s] = slots ? slots[s] : nullptr;
  for (int j = 0; j < nterm; ++j) {
    if (!A.slots[terms[j].src]) return fail(RKS_ERR_INVALID, "missing NL slot for this stage");
    if (terms[j].src2 >= 0 && !A.slots[terms[j].src2]) return fail(RKS_ERR_INVALID, "missing NL slot for this stage");
  }
  const int M = p->modes[inst];
  const rks_inst& r = p->h_inst[inst];
  A.tab = p->d_tab;
  A.u = u;
  A.coefs = inst_cbase(p, inst);
  A.out = out;
  A.stage = stage;
  A.is_err = is_err ? 1 : 0;
  A.M = M;
  A.h = h;
  int grid = (M + 255) / 256;
  if (grid > 4 * p->cu) grid = 4 * p->cu;
  if (p->prec == RKS_F64) hipLaunchKernelGGL(rks_combine_kernel<double>, dim3(grid), dim3(256), 0, stream, A);
  else hipLaunchKernelGGL(rks_combine_kernel<float>, dim3(grid), dim3(256), 0, stream, A);
  HIPCHK(hipGetLastError());
  return RKS_OK;
}

int rks_error_s(rks_plan* p, int inst, const void* u_new, const void* err, double* s_dev, hipStream_t stream) {
  if (!p || inst < 0 || inst >= p->ninst || !u_new || !err || !s_dev)
    return fail(RKS_ERR_INVALID, "bad arguments");
  const int M = p->modes[inst];
  if (p->prec == RKS_F64)
    hipLaunchKernelGGL(rks_norm_kernel<double>, dim3(1), dim3(1024), 0, stream, (const cx<double>*)u_new,
                       (const cx<double>*)err, M, p->ctl.epsilon, p->ctl.safety_f, p->ctl.adapt_cutoff,
                       p->tab.q, s_dev);
  else
    hipLaunchKernelGGL(rks_norm_kernel<float>, dim3(1), dim3(1024), 0, stream, (const cx<float>*)u_new,
                       (const cx<float>*)err, M, p->ctl.epsilon, p->ctl.safety_f, p->ctl.adapt_cutoff,
                       p->tab.q, s_dev);
  HIPCHK(hipGetLastError());
  return RKS_OK;
}

int rks_get_stats(rks_plan* p, rks_stats* out, hipStream_t stream) {
  if (!p || !out) return fail(RKS_ERR_INVALID, "null argument");
  HIPCHK(hipStreamSynchronize(stream));
  HIPCHK(hipMemcpy(p->h_inst.data(), p->d_inst, sizeof(rks_inst) * p->ninst, hipMemcpyDeviceToHost));
  for (int i = 0; i < p->ninst; ++i) {
    const rks_inst& r = p->h_inst[i];
    rks_stats& s = out[i];
    s.tc = r.tc;
    s.h_used = r.h_used;
    s.h_next = r.h_next;
    s.h = r.h;
    s.steps = r.steps;
    s.attempts = r.attempts;
    s.rejects = r.rejects;
    s.status = r.status;
    s.log_count = r.log_count;
    s.snap_count = r.snap_count;
    s.nl_calls = r.nl_calls;
    s.coef_updates = r.coef_updates;
  }
  return RKS_OK;
}

// the proposer and its records need an adaptive 1-D plan whose workgroups
// are whole waves (n >= 256 for rfft grids, n >= 128 for fft grids)
static int learned_supported(const rks_plan* p) {
  if (p->c2 || (p->nlk != RKS_NL_ADVECT_RFFT && p->nlk != RKS_NL_CUBIC_FFT))
    return fail(RKS_ERR_INVALID, "the step-size proposer needs a 1-D built-in nonlinearity");
  if (!p->tab.adaptive) return fail(RKS_ERR_INVALID, "the step-size proposer needs an adaptive method");
  for (int l : p->bucket_log2)
    if (rks_threads(l, p->nlk) < 64)
      return fail(RKS_ERR_INVALID, "the step-size proposer needs n >= 256 (rfft) or n >= 128 (fft)");
  return RKS_OK;
}

int rks_plan_set_proposer(rks_plan* p, const rks_mlp* net, int policy, double margin, double keep_lo,
                          double keep_hi, int period) {
  if (!p) return fail(RKS_ERR_INVALID, "null plan");
  if (!net) {
    p->mlp = rks_mlp_dev{};
    return RKS_OK;
  }
  int rc = learned_supported(p);
  if (rc) return rc;
  if (rks_mlp_device_of(net) != p->device) return fail(RKS_ERR_INVALID, "proposer and plan are on different devices");
  if (!std::isfinite(margin) || !std::isfinite(keep_lo) || !std::isfinite(keep_hi))
    return fail(RKS_ERR_INVALID, "margin and keep band must be finite");
  if (policy != RKS_PROPOSE && policy != RKS_GUARD && policy != RKS_GROW)
    return fail(RKS_ERR_INVALID, "unknown proposer policy");
  if (period < 1) return fail(RKS_ERR_INVALID, "proposer period must be >= 1");
  p->mlp = rks_mlp_device(net, policy, margin, keep_lo, keep_hi, period);
  return RKS_OK;
}

int rks_set_records(rks_plan* p, int rec_cap) {
  if (!p) return fail(RKS_ERR_INVALID, "null plan");
  if (rec_cap < 0) return fail(RKS_ERR_INVALID, "negative record capacity");
  if (rec_cap > 0) {
    int rc = learned_supported(p);
    if (rc) return rc;
  }
  HIPCHK(hipDeviceSynchronize());
  (void)hipFree(p->d_rec);
  p->d_rec = nullptr;
  if (rec_cap > 0)
    HIPCHK(hipMalloc(&p->d_rec, sizeof(float) * RKS_MLP_REC * (size_t)rec_cap * p->ninst));
  HIPCHK(hipMemcpy(p->h_inst.data(), p->d_inst, sizeof(rks_inst) * p->ninst, hipMemcpyDeviceToHost));
  for (int i = 0; i < p->ninst; ++i) {
    rks_inst& r = p->h_inst[i];
    r.rec = rec_cap > 0 ? p->d_rec + (size_t)RKS_MLP_REC * rec_cap * i : nullptr;
    r.rec_cap = rec_cap;
    r.rec_count = 0;
    r.rec_pending = -1;
  }
  HIPCHK(hipMemcpy(p->d_inst, p->h_inst.data(), sizeof(rks_inst) * p->ninst, hipMemcpyHostToDevice));
  p->rec_cap = rec_cap;
  return RKS_OK;
}

int rks_read_records(rks_plan* p, float* dst_dev, int* counts, hipStream_t stream) {
  if (!p) return fail(RKS_ERR_INVALID, "null plan");
  if (!p->d_rec) return fail(RKS_ERR_INVALID, "records not enabled (rks_set_records)");
  HIPCHK(hipStreamSynchronize(stream));
  HIPCHK(hipMemcpy(p->h_inst.data(), p->d_inst, sizeof(rks_inst) * p->ninst, hipMemcpyDeviceToHost));
  if (counts)
    for (int i = 0; i < p->ninst; ++i) counts[i] = p->h_inst[i].rec_count;
  if (dst_dev) {
    HIPCHK(hipMemcpyAsync(dst_dev, p->d_rec, sizeof(float) * RKS_MLP_REC * (size_t)p->rec_cap * p->ninst,
                          hipMemcpyDeviceToDevice, stream));
    HIPCHK(hipStreamSynchronize(stream));
  }
  return RKS_OK;
}

int rks_plan_set_priority(rks_plan* p, const double* cost) {
  if (!p || !cost) return fail(RKS_ERR_INVALID, "null argument");
  if (p->c2) return fail(RKS_ERR_INVALID, "the 2-D engine has a fixed launch sequence");
  for (int i = 0; i < p->ninst; ++i)
    if (!std::isfinite(cost[i])) return fail(RKS_ERR_INVALID, "costs must be finite");
  // longest first within each size bucket (stable: equal costs keep their order)
  for (size_t b = 0; b < p->bucket_start.size(); ++b) {
    auto first = p->order.begin() + p->bucket_start[b];
    std::stable_sort(first, first + p->bucket_count[b], [&](int a, int c) { return cost[a] > cost[c]; });
  }
  HIPCHK(hipDeviceSynchronize());
  HIPCHK(upload_order(p));
  return RKS_OK;
}

int rks_plan_buckets(rks_plan* p, int* nbucket, int* log2n, int* count, int* max_wg_per_cu, int* ntile, int cap) {
  if (!p || !nbucket) return fail(RKS_ERR_INVALID, "null argument");
  *nbucket = (int)p->bucket_log2.size();
  for (int b = 0; b < *nbucket && b < cap; ++b) {
    if (log2n) log2n[b] = p->bucket_log2[b];
    if (count) count[b] = p->bucket_count[b];
    if (ntile) {
      KernelEntry e1;
      ntile[b] = lookup(p->prec, p->nlk, p->variant, p->bucket_log2[b], true, &e1, 1) ? 2 : 1;
    }
    if (max_wg_per_cu) {
      KernelEntry e;
      int per_cu = 0;
      if (!lookup(p->prec, p->nlk, p->variant, p->bucket_log2[b], learns(p), &e) ||
          hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, e.fn, e.threads, e.lds) != hipSuccess || per_cu < 1)
        per_cu = 1;
      max_wg_per_cu[b] = per_cu;
    }
  }
  return RKS_OK;
}

int rks_plan_set_launch(rks_plan* p, int concurrent, const int* wg_per_cu, const int* tile, int nbucket) {
  if (!p) return fail(RKS_ERR_INVALID, "null plan");
  if (p->c2) return fail(RKS_ERR_INVALID, "the 2-D engine has a fixed launch sequence");
  const int nb = (int)p->bucket_log2.size();
  if ((wg_per_cu || tile) && nbucket != nb) return fail(RKS_ERR_INVALID, "one value per size bucket needed");
  std::vector<int> w(nb, 0), ti(nb, -1);
  for (int b = 0; b < nb; ++b) {
    if (wg_per_cu) {
      if (wg_per_cu[b] < 0) return fail(RKS_ERR_INVALID, "wg_per_cu must be >= 0");
      w[b] = wg_per_cu[b];
    }
    if (tile) {
      // -1: default_tile's choice; else a tile that the plan can run on as it is
      KernelEntry e1;
      if (tile[b] < -1 || (tile[b] > 0 && !lookup(p->prec, p->nlk, p->variant, p->bucket_log2[b], learns(p), &e1, tile[b])))
        return fail(RKS_ERR_INVALID, "tile 1 exists for n = 512 .. 4096; without a proposer or records also tile 1 for "
                                     "the cubic n = 8192, tile 2 for n = 1024 and the cubic n = 2048");
      ti[b] = tile[b];
    }
  }
  p->concurrent = concurrent ? 1 : 0;
  p->wg_per_cu = w;
  p->tile = ti;
  return RKS_OK;
}

int rks_plan_tiles(rks_plan* p, int* tile, int cap) {
  if (!p || !tile) return fail(RKS_ERR_INVALID, "null argument");
  for (size_t b = 0; b < p->bucket_log2.size() && (int)b < cap; ++b)
    tile[b] = bucket_tile(p, b, p->bucket_undamped[b] == p->bucket_count[b]);
  return RKS_OK;
}

int rks_read_log(rks_plan* p, int inst, double* host_hs, int cap, hipStream_t stream) {
  if (!p || inst < 0 || inst >= p->ninst || !host_hs) return fail(RKS_ERR_INVALID, "bad arguments");
  if (!p->d_log) return fail(RKS_ERR_INVALID, "attempt log not enabled");
  HIPCHK(hipStreamSynchronize(stream));
  int n = cap < p->log_cap ? cap : p->log_cap;
  HIPCHK(hipMemcpy(host_hs, p->d_log + 2 * (size_t)p->log_cap * inst, sizeof(double) * 2 * n,
                   hipMemcpyDeviceToHost));
  return RKS_OK;
}

int rks_read_snapshots(rks_plan* p, int inst, void* dst_dev, double* t_host, int count, hipStream_t stream) {
  if (!p || inst < 0 || inst >= p->ninst) return fail(RKS_ERR_INVALID, "bad arguments");
  if (!p->d_snap) return fail(RKS_ERR_INVALID, "snapshots not enabled");
  if (count < 0 || count > p->snap_cap) return fail(RKS_ERR_INVALID, "bad snapshot count");
  const rks_inst& r = p->h_inst[inst];
  if (count == 0) return RKS_OK;
  if (dst_dev)
    HIPCHK(hipMemcpyAsync(dst_dev, r.snap, (size_t)count * r.m * p->esize, hipMemcpyDeviceToDevice, stream));
  if (t_host) {
    HIPCHK(hipStreamSynchronize(stream));
    HIPCHK(hipMemcpy(t_host, r.snap_t, sizeof(double) * count, hipMemcpyDeviceToHost));
  }
  // consumed: the next resume starts filling at index 0
  HIPCHK(hipStreamSynchronize(stream));
  HIPCHK(hipMemcpy(p->h_inst.data(), p->d_inst, sizeof(rks_inst) * p->ninst, hipMemcpyDeviceToHost));
  p->h_inst[inst].snap_count = 0;
  HIPCHK(hipMemcpy(p->d_inst + inst, &p->h_inst[inst], sizeof(rks_inst), hipMemcpyHostToDevice));
  return RKS_OK;
}

}  // extern "C"

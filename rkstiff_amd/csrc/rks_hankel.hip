// Quasi-discrete Hankel transform of order zero on the device.
//
// The reference applies an nr x nr matrix Y of J0 values (transforms.py:
// 113-117) as ht(f) = S Y f and iht(g) = Y g / S with S = rmax^2 / j_{N+1}
// (transforms.py:172-240); its radial NLS demo (demos/nls.ipynb cell 8)
// evaluates 1j gamma ht(|f|^2 f), f = iht(g), at every stage.
//
// Here one launch multiplies Y by a batch of vectors: out[b] = c Y in[b], on
// the FP64 matrix cores (hankel_gemm).  The epilogue
// scales, or forms |f|^2 f (after the inverse), or multiplies by i gamma (after
// the forward), so the radial NLS term is two launches.
#include <hip/hip_runtime.h>

#include <mutex>
#include <string>

#include "rkstiff_amd.h"

void rks_set_last_error(const std::string& msg);  // rks_host.hip

// Scratch of the allocation-free cubic term (4 MiB: nr * batch <= 262144 complex values).
constexpr size_t kScratchDoubles = (size_t)1 << 19;
static __device__ __align__(256) double scratch[kScratchDoubles];

namespace {

constexpr int HB_K = 32;   // K chunk
constexpr int HB_B = 16;   // column pairs per tile: 16 complex or 32 real vectors
constexpr int HB_CU = 256; // compute units

enum { EPI_SCALE = 0, EPI_CUBIC = 1, EPI_TIMES_I = 2 };

int hfail(int code, const std::string& msg) {
  rks_set_last_error(msg);
  return code;
}

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));  // two doubles at any double's address

// out[b][i] = epi(c * sum_j Y[i][j] in[b][j]); complex vectors (CPLX) are
// interleaved (re, im), real vectors are plain doubles.  A column pair is one
// complex vector's two parts, or real vectors b and b + 16 of a tile.
//
// V_MFMA_F64_16X16X4: lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and
// D[4 r + l / 16][l % 16], r < 4.  The vectors are A's rows, so a lane's results are one
// row i of 4 vectors and 16 lanes store 16 consecutive i.  The four k of an instruction
// need not be neighbours: lane group l / 16 takes a run of k of its own, read from LDS in
// 16-byte pieces (row strides odd in those: no bank conflicts).  The matrix rate is the
// vector units' FP64 rate, but an instruction of 2048 operations reads two LDS values per
// lane where 32 FMAs of a 4 x 2 register tile read 24; those reads bounded the vector form.
// The next chunk's global loads are in flight during a chunk's products, one barrier each.
// ROWS 64: a wave has 16 rows of its own.  ROWS 16: the four waves share one tile, so four times
// the workgroups; taken while 64-row tiles would leave CUs idle.  There wave w takes the quarter
// w of each chunk's k; with 64 rows a wave keeps the four quarters' sums apart and adds them in
// the same order, so a vector's result does not depend on the batch it is in.  Two waves per
// SIMD (256 registers) keep the sums out of the accumulation registers, to and from which each
// chunk would copy them (12.0 us).
// nr = 251, 1024 complex vectors: 43.5 us by FMAs on a 4 x 2 register tile, now 10.2 (the
// products alone take 3.3 us at 78 TFLOP/s; with one sum per wave 10.4).
template <bool CPLX, int EPI, int ROWS>
__global__ __launch_bounds__(256, 2) void hankel_gemm(const double* __restrict__ Y, int nr,
                                                   const double* __restrict__ in, double* __restrict__ out,
                                                   int batch, double c, double gamma) {
  constexpr bool SPLIT = ROWS == 16;
  constexpr int YS = HB_K + 2, YE = ROWS * HB_K / 256, XE = HB_B * HB_K / 256;
  __shared__ __align__(16) double Ys[2][ROWS][YS];
  __shared__ __align__(16) d2 Xs[2][HB_B][HB_K + 1];
  const int t = threadIdx.x, w = t / 64, l = t % 64, g = l / 16, n = l % 16;
  const int i0 = blockIdx.x * ROWS, b0 = blockIdx.y * (CPLX ? HB_B : 2 * HB_B);
  const int kt = t % HB_K, rt = t / HB_K;  // this thread's column of a chunk; rows rt + 8 e
  double yr[YE];
  d2 xr[XE];
  auto load = [&](int k0) {
    const int k = k0 + kt;
#pragma unroll
    for (int e = 0; e < YE; ++e) {
      const int i = i0 + rt + 8 * e;
      yr[e] = (i < nr && k < nr) ? Y[(size_t)i * nr + k] : 0.0;
    }
#pragma unroll
    for (int e = 0; e < XE; ++e) {
      const int b = b0 + rt + 8 * e;
      d2 v = {0.0, 0.0};
      if (CPLX) {
        if (b < batch && k < nr) v = *(const d2u*)(in + 2 * ((size_t)b * nr + k));
      } else {
        if (b < batch && k < nr) v.x = in[(size_t)b * nr + k];
        if (b + HB_B < batch && k < nr) v.y = in[(size_t)(b + HB_B) * nr + k];
      }
      xr[e] = v;
    }
  };
  constexpr int NP = SPLIT ? 1 : 4;  // quarters of a chunk per wave
  d4 a0[NP], a1[NP];
#pragma unroll
  for (int q = 0; q < NP; ++q) a0[q] = a1[q] = d4{0.0, 0.0, 0.0, 0.0};
  load(0);
  for (int k0 = 0, buf = 0; k0 < nr; k0 += HB_K, buf ^= 1) {
#pragma unroll
    for (int e = 0; e < YE; ++e) Ys[buf][rt + 8 * e][kt] = yr[e];
#pragma unroll
    for (int e = 0; e < XE; ++e) Xs[buf][rt + 8 * e][kt] = xr[e];
    if (k0 + HB_K < nr) load(k0 + HB_K);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const int kb = (SPLIT ? w : q) * (HB_K / 4) + 2 * g;
      const d2 y = *(const d2*)&Ys[buf][SPLIT ? n : w * 16 + n][kb];
      const d2 x0 = Xs[buf][n][kb], x1 = Xs[buf][n][kb + 1];
      a0[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(x0.x, y.x, a0[q], 0, 0, 0);
      a1[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(x0.y, y.x, a1[q], 0, 0, 0);
      a0[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(x1.x, y.y, a0[q], 0, 0, 0);
      a1[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(x1.y, y.y, a1[q], 0, 0, 0);
    }
  }
  const int i = i0 + (SPLIT ? n : w * 16 + n);
  auto store = [&](int v, double vr, double vi) {
    const int b = b0 + v;
    vr *= c;
    vi *= c;
    if (i >= nr) return;
    if (EPI == EPI_CUBIC) {
      const double m2 = fma(vr, vr, vi * vi);
      vr *= m2;
      vi *= m2;
    } else if (EPI == EPI_TIMES_I) {
      const double q = vr;
      vr = -gamma * vi;
      vi = gamma * q;
    }
    if (CPLX) {
      if (b < batch) {
        d2u o = {vr, vi};
        *(d2u*)(out + 2 * ((size_t)b * nr + i)) = o;
      }
    } else {
      if (b < batch) out[(size_t)b * nr + i] = vr;
      if (b + HB_B < batch) out[(size_t)(b + HB_B) * nr + i] = vi;
    }
  };
  // the four partial sums in order
  if constexpr (SPLIT) {
    // wave w finishes the results r = w
    __shared__ d2 part[4][4][64];
#pragma unroll
    for (int r = 0; r < 4; ++r) part[w][r][l] = d2{a0[0][r], a1[0][r]};
    __syncthreads();
    d2 v = part[0][w][l];
#pragma unroll
    for (int q = 1; q < 4; ++q) v += part[q][w][l];
    store(4 * w + g, v.x, v.y);
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      store(4 * r + g, a0[0][r] + a0[1][r] + a0[2][r] + a0[3][r], a1[0][r] + a1[1][r] + a1[2][r] + a1[3][r]);
  }
}

template <bool CPLX, int EPI>
void hankel_launch(const double* Y, int nr, const double* in, double* out, int batch, double c, double gamma,
                   hipStream_t stream) {
  const int nb = (batch + (CPLX ? HB_B : 2 * HB_B) - 1) / (CPLX ? HB_B : 2 * HB_B), ni = (nr + 63) / 64;
  if (ni * nb >= HB_CU)
    hipLaunchKernelGGL((hankel_gemm<CPLX, EPI, 64>), dim3(ni, nb), dim3(256), 0, stream, Y, nr, in, out, batch, c,
                       gamma);
  else
    hipLaunchKernelGGL((hankel_gemm<CPLX, EPI, 16>), dim3((nr + 15) / 16, nb), dim3(256), 0, stream, Y, nr, in, out,
                       batch, c, gamma);
}

// Allocation-free cubic term (rks_hankel_cubic_noalloc): its |f|^2 f intermediate
// lives in this file-scope device array, one copy per GPU, held until the
// process ends.  Host code never passes `scratch` itself (in host code the name
// is a stand-in, not a device address); it uses the address that
// hipGetSymbolAddress returned for the device, kept in scratch_ptr.
constexpr int kMaxDevices = 64;
std::mutex scratch_mu;
double* scratch_ptr[kMaxDevices] = {};

// Once per device, with that device current: the device address of `scratch`.
int scratch_setup(int device) {
  if (device < 0 || device >= kMaxDevices) return hfail(RKS_ERR_INVALID, "device index beyond the scratch table");
  std::lock_guard<std::mutex> lk(scratch_mu);
  if (scratch_ptr[device]) return RKS_OK;
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p)
    return hfail(RKS_ERR_HIP, std::string("scratch address: ") + hipGetErrorString(e));
  scratch_ptr[device] = (double*)p;
  return RKS_OK;
}

double* scratch_for(int device) {
  if (device < 0 || device >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lk(scratch_mu);
  return scratch_ptr[device];
}

}  // namespace

struct rks_hankel {
  int nr = 0, device = 0;
  double scale = 1.0;
  double* d_Y = nullptr;
  double* d_tmp = nullptr;  // |f|^2 f of the cubic term
  int tmp_batch = 0;
};

extern "C" {

int rks_hankel_create(int nr, const double* Y, double scale, rks_hankel** out) {
  if (!out || !Y) return hfail(RKS_ERR_INVALID, "null argument");
  *out = nullptr;
  if (nr < 4) return hfail(RKS_ERR_INVALID, "nr must be >= 4");
  if (!(scale > 0.0)) return hfail(RKS_ERR_INVALID, "scale must be positive");
  rks_hankel* h = new rks_hankel();
  h->nr = nr;
  h->scale = scale;
  hipError_t e = hipGetDevice(&h->device);
  if (e == hipSuccess) e = hipMalloc(&h->d_Y, sizeof(double) * (size_t)nr * nr);
  if (e == hipSuccess) e = hipMemcpy(h->d_Y, Y, sizeof(double) * (size_t)nr * nr, hipMemcpyDefault);
  if (e != hipSuccess) {
    rks_hankel_destroy(h);
    return hfail(RKS_ERR_HIP, std::string("rks_hankel_create: ") + hipGetErrorString(e));
  }
  const int rc = scratch_setup(h->device);  // the transform's device is current here
  if (rc != RKS_OK) {
    rks_hankel_destroy(h);
    return rc;
  }
  *out = h;
  return RKS_OK;
}

int rks_hankel_destroy(rks_hankel* h) {
  if (!h) return RKS_OK;
  (void)hipDeviceSynchronize();
  (void)hipFree(h->d_Y);
  (void)hipFree(h->d_tmp);
  delete h;
  return RKS_OK;
}

int rks_hankel_apply(rks_hankel* h, int inverse, const void* in, void* out, int batch, int cplx,
                     hipStream_t stream) {
  if (!h || !in || !out) return hfail(RKS_ERR_INVALID, "null argument");
  if (batch < 0) return hfail(RKS_ERR_INVALID, "batch must be >= 0");
  if (in == out) return hfail(RKS_ERR_INVALID, "in and out must not alias");
  if (batch == 0) return RKS_OK;
  const double c = inverse ? 1.0 / h->scale : h->scale;
  if (cplx)
    hankel_launch<true, EPI_SCALE>(h->d_Y, h->nr, (const double*)in, (double*)out, batch, c, 0.0, stream);
  else
    hankel_launch<false, EPI_SCALE>(h->d_Y, h->nr, (const double*)in, (double*)out, batch, c, 0.0, stream);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hfail(RKS_ERR_HIP, std::string("rks_hankel_apply: ") + hipGetErrorString(e));
  return RKS_OK;
}

int rks_hankel_cubic(rks_hankel* h, double gamma, const void* in, void* out, int batch, hipStream_t stream) {
  if (!h || !in || !out) return hfail(RKS_ERR_INVALID, "null argument");
  if (batch < 0) return hfail(RKS_ERR_INVALID, "batch must be >= 0");
  if (in == out) return hfail(RKS_ERR_INVALID, "in and out must not alias");
  if (batch == 0) return RKS_OK;
  if (batch > h->tmp_batch) {
    const hipError_t se = hipStreamSynchronize(stream);
    if (se != hipSuccess) return hfail(RKS_ERR_HIP, std::string("rks_hankel_cubic: ") + hipGetErrorString(se));
    (void)hipFree(h->d_tmp);
    h->d_tmp = nullptr;
    h->tmp_batch = 0;
    const hipError_t e = hipMalloc(&h->d_tmp, sizeof(double) * 2 * (size_t)h->nr * batch);
    if (e != hipSuccess) return hfail(RKS_ERR_HIP, std::string("rks_hankel_cubic: ") + hipGetErrorString(e));
    h->tmp_batch = batch;
  }
  hankel_launch<true, EPI_CUBIC>(h->d_Y, h->nr, (const double*)in, h->d_tmp, batch, 1.0 / h->scale, 0.0, stream);
  hankel_launch<true, EPI_TIMES_I>(h->d_Y, h->nr, h->d_tmp, (double*)out, batch, h->scale, gamma, stream);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hfail(RKS_ERR_HIP, std::string("rks_hankel_cubic: ") + hipGetErrorString(e));
  return RKS_OK;
}

int rks_hankel_cubic_noalloc(rks_hankel* h, double gamma, const void* in, void* out, int batch,
                             hipStream_t stream) {
  if (!h || !in || !out) return hfail(RKS_ERR_INVALID, "null argument");
  if (batch < 0) return hfail(RKS_ERR_INVALID, "batch must be >= 0");
  if (in == out) return hfail(RKS_ERR_INVALID, "in and out must not alias");
  if (batch == 0) return RKS_OK;
  const size_t need = 2 * (size_t)h->nr * (size_t)batch;
  if (need > kScratchDoubles)
    return hfail(RKS_ERR_INVALID, "rks_hankel_cubic_noalloc: nr * batch = " + std::to_string(need / 2) +
                                      " exceeds the allocation-free scratch of " +
                                      std::to_string(kScratchDoubles / 2) + " complex values");
  double* scr = scratch_for(h->device);
  if (!scr) return hfail(RKS_ERR_HIP, "rks_hankel_cubic_noalloc: no scratch address for the transform's device");
  hankel_launch<true, EPI_CUBIC>(h->d_Y, h->nr, (const double*)in, scr, batch, 1.0 / h->scale, 0.0, stream);
  hankel_launch<true, EPI_TIMES_I>(h->d_Y, h->nr, scr, (double*)out, batch, h->scale, gamma, stream);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hfail(RKS_ERR_HIP, std::string("rks_hankel_cubic_noalloc: ") + hipGetErrorString(e));
  return RKS_OK;
}

}  // extern "C"

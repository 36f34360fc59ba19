// Krylov drivers above the operator: the role PETSc's KSP plays for ellip
// (src/fs/tests/ellip.c:701-747), on device vectors.
//
//   * PCG with the embedded-Q1 matrix as preconditioner, applied approximately either by a
//     Jacobi-preconditioned Chebyshev iteration of fixed degree (a fixed polynomial in
//     D^{-1} A_q1 times D^{-1}, hence symmetric, so CG stays valid) or by a multigrid V-cycle
//     on the Q1 matrix with Jacobi-Chebyshev smoothing (symmetric as well).
//   * Plain path: everything in FP64.
//   * Mixed path: FP64 outer defect correction x += A32^{-1}(b - A64 x) with the inner PCG in
//     FP32 (FP32 operator and Q1 applies); residuals of the outer loop and every Krylov dot
//     product accumulate in FP64.
//   * FP32-preconditioner path: FP64 PCG whose preconditioner (V-cycle or Chebyshev, learned
//     weights included) runs in FP32.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <vector>

#include "common.h"

using namespace dohp;

extern "C" dErr dohpEllipGetQ1Context_Private(dohpEllip op, dohpFS *fs, dohpEllipParam *prm, const double **kvert,
                                              const double **state, int *q1mode);

namespace {

constexpr int kRedBlocks = 2048;  // blocks of a reduction (one partial sum each): eight per compute unit

template <typename T>
__global__ void dot_partial_kernel(long n, const T *__restrict__ a, const T *__restrict__ b, double *__restrict__ part)
{
  __shared__ double sh[256];
  double s = 0.0;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    s += (double)a[i] * (double)b[i];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

__global__ void dot_final_kernel(int nb, const double *__restrict__ part, double *__restrict__ out)
{
  __shared__ double sh[256];
  double s = 0.0;
  for (int i = threadIdx.x; i < nb; i += blockDim.x) s += part[i];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = sh[0];
}

// y = a*x + b*y
template <typename T>
__global__ void axpby_kernel(long n, T a, const T *__restrict__ x, T b, T *__restrict__ y)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = a * x[i] + b * y[i];
}

// z = s * d * r  (diagonal scaling)
template <typename T>
__global__ void dscale_kernel(long n, T s, const T *__restrict__ dinv, const T *__restrict__ r, T *__restrict__ z)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) z[i] = s * dinv[i] * r[i];
}

__global__ void inv_kernel(long n, const double *__restrict__ d, double *__restrict__ di, float *__restrict__ di32)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    di[i] = 1.0 / d[i];
    di32[i] = (float)di[i];
  }
}

template <typename T>
__global__ void fill_kernel(long n, T v, T *__restrict__ y)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = v;
}

// y32 = s * x64 ; x64 += s * y32
__global__ void demote_kernel(long n, double s, const double *__restrict__ x, float *__restrict__ y)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = (float)(s * x[i]);
}
__global__ void promote_add_kernel(long n, double s, const float *__restrict__ y, double *__restrict__ x)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] += s * (double)y[i];
}

// ---- CG's vector work, fused.  An iteration's scalars stay on the device: a kernel that needs one sums the partial
// sums that the previous kernel left (kRedBlocks of them, in a fixed order, once per workgroup), and only ||r||^2 goes to
// the host, which reads it while the preconditioner already runs.  Per iteration (FP64 CG, FP32 preconditioner) 58 bytes
// a row in four launches and one wait instead of 96 in eleven launches and four waits.
__device__ __forceinline__ double sum_block(double s, double *sh)
{
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  const double r = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  __syncthreads();
  return r;
}
__device__ __forceinline__ double sum_partials(const double *__restrict__ part, double *sh)
{
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < kRedBlocks / 256; i++) s += part[i * 256 + threadIdx.x];
  return sum_block(s, sh);
}

// r = b - q (and its FP32 copy if lr is not null), partial sums of b.b and r.r
template <typename T>
__global__ void __launch_bounds__(256) krylov_init_kernel(long n, const T *__restrict__ b, const T *__restrict__ q,
                                                          T *__restrict__ r, float *__restrict__ lr,
                                                          double *__restrict__ part_bb, double *__restrict__ part_rr)
{
  __shared__ double sh[4];
  double sb = 0.0, sr = 0.0;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += 256L * gridDim.x) {
    const T bi = b[i], ri = bi - q[i];
    r[i] = ri;
    if (lr) lr[i] = (float)ri;
    sb += (double)bi * (double)bi;
    sr += (double)ri * (double)ri;
  }
  const double tb = sum_block(sb, sh), tr = sum_block(sr, sh);
  if (threadIdx.x == 0) {
    part_bb[blockIdx.x] = tb;
    part_rr[blockIdx.x] = tr;
  }
}

// host[j] = sum of the j-th array of partial sums (host: pinned memory, read by the host after the kernel has ended)
__global__ void __launch_bounds__(256) krylov_read_kernel(const double *__restrict__ part, int m,
                                                          double *__restrict__ host)
{
  __shared__ double sh[4];
  for (int j = 0; j < m; j++) {
    const double t = sum_partials(part + (long)j * kRedBlocks, sh);
    if (threadIdx.x == 0) host[j] = t;
  }
}

// alpha = rz / p.q;  x += alpha p;  r -= alpha q (and its FP32 copy), partial sums of r.r
template <typename T>
__global__ void __launch_bounds__(256) krylov_update_kernel(long n, const double *__restrict__ part_pq,
                                                            const double *__restrict__ rz, double *__restrict__ alpha,
                                                            const T *__restrict__ p, const T *__restrict__ q,
                                                            T *__restrict__ x, T *__restrict__ r,
                                                            float *__restrict__ lr, double *__restrict__ part_rr)
{
  __shared__ double sh[4];
  const double al = rz[0] / sum_partials(part_pq, sh);
  const T a = (T)al;
  double s = 0.0;
#pragma unroll 2
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += 256L * gridDim.x) {
    x[i] = a * p[i] + x[i];
    const T ri = -a * q[i] + r[i];
    r[i] = ri;
    if (lr) lr[i] = (float)ri;
    s += (double)ri * (double)ri;
  }
  const double t = sum_block(s, sh);
  if (threadIdx.x == 0) {
    part_rr[blockIdx.x] = t;
    if (blockIdx.x == 0) alpha[0] = al;
  }
}

// partial sums of r.z and, if q is not null, of z.q
template <typename T, typename Z>
__global__ void __launch_bounds__(256) krylov_zdots_kernel(long n, const T *__restrict__ r, const Z *__restrict__ z,
                                                           const T *__restrict__ q, double *__restrict__ part_rz,
                                                           double *__restrict__ part_zq)
{
  __shared__ double sh[4];
  double s0 = 0.0, s1 = 0.0;
#pragma unroll 2
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += 256L * gridDim.x) {
    const double zi = (double)z[i];
    s0 += (double)r[i] * zi;
    if (q) s1 += zi * (double)q[i];
  }
  const double t0 = sum_block(s0, sh), t1 = sum_block(s1, sh);
  if (threadIdx.x == 0) {
    part_rz[blockIdx.x] = t0;
    part_zq[blockIdx.x] = t1;
  }
}

// rz_new = r.z;  p = z + beta p with beta = rz_new / rz (mode KB_STANDARD), -alpha z.q / rz (KB_FLEXIBLE) or 0
// (KB_FIRST: p = z, p is not read);  q = 0 for the operator's scatter
enum { KB_FIRST, KB_STANDARD, KB_FLEXIBLE };
template <typename T, typename Z>
__global__ void __launch_bounds__(256) krylov_direction_kernel(long n, int mode, const double *__restrict__ part_rz,
                                                               const double *__restrict__ part_zq,
                                                               const double *__restrict__ rz,
                                                               double *__restrict__ rz_new,
                                                               const double *__restrict__ alpha,
                                                               const Z *__restrict__ z, T *__restrict__ p,
                                                               T *__restrict__ q)
{
  __shared__ double sh[4];
  const double rzn = sum_partials(part_rz, sh);
  double beta = 0.0;
  if (mode == KB_STANDARD) beta = rzn / rz[0];
  if (mode == KB_FLEXIBLE) beta = -alpha[0] * sum_partials(part_zq, sh) / rz[0];
  const T be = (T)beta;
#pragma unroll 2
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += 256L * gridDim.x) {
    const T zi = (T)z[i];
    p[i] = mode == KB_FIRST ? zi : zi + be * p[i];
    q[i] = T(0);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) rz_new[0] = rzn;
}

inline dim3 grid(long n) { return dim3((n + 255) / 256); }

struct Ctx {
  hipStream_t st;
  long n;
  Pool *pool;  // the operator's: every work vector of a solve comes from it
  PoolBuf<double> part, res;
  double *host = nullptr;  // pinned scalars of the operator, and their device address
  double *host_dev = nullptr;
};

struct Event {
  hipEvent_t e = nullptr;
  ~Event()
  {
    if (e) (void)hipEventDestroy(e);
  }
};

template <typename T>
dErr dot(Ctx &c, const T *a, const T *b, double *out)
{
  hipLaunchKernelGGL(dot_partial_kernel<T>, dim3(kRedBlocks), dim3(256), 0, c.st, c.n, a, b, c.part.ptr);
  hipLaunchKernelGGL(dot_final_kernel, dim3(1), dim3(256), 0, c.st, kRedBlocks, c.part.ptr, c.res.ptr);
  DOHP_HIP(hipMemcpyAsync(out, c.res.ptr, sizeof(double), hipMemcpyDeviceToHost, c.st));
  DOHP_HIP(hipStreamSynchronize(c.st));
  return 0;
}

template <typename T>
dErr axpby(Ctx &c, T a, const T *x, T b, T *y)
{
  hipLaunchKernelGGL(axpby_kernel<T>, grid(c.n), dim3(256), 0, c.st, c.n, a, x, b, y);
  DOHP_HIP(hipGetLastError());
  return 0;
}

// Operators of one precision.
template <typename T>
struct Ops;
template <>
struct Ops<double> {
  static dErr A(dohpEllip op, const double *x, double *y, hipStream_t s) { return dohpEllipMatMult_Private(op, x, y, s); }
  static dErr A_add(dohpEllip op, const double *x, double *y, hipStream_t s)
  {
    return dohpEllipMatMultAdd_Private(op, x, y, s);
  }
  static dErr Q(dohpMat m, const double *x, double *y, hipStream_t s) { return dohpMatMult(m, x, y, s); }
};
template <>
struct Ops<float> {
  static dErr A(dohpEllip op, const float *x, float *y, hipStream_t s) { return dohpEllipMatMult_Private(op, x, y, s); }
  static dErr A_add(dohpEllip op, const float *x, float *y, hipStream_t s)
  {
    return dohpEllipMatMultAdd_Private(op, x, y, s);
  }
  static dErr Q(dohpMat m, const float *x, float *y, hipStream_t s) { return dohpMatMultF32(m, x, y, s); }
};

// Preconditioner: degree-k Chebyshev iteration on A_q1 z = r with Jacobi scaling, z0 = 0.
template <typename T>
struct Cheb {
  dohpMat q1;
  const T *dinv;
  double lmin, lmax;
  int degree;
  PoolBuf<T> res, d, w;
  dErr alloc(Ctx &c)
  {
    DOHP_CALL(res.alloc(*c.pool, c.n));
    DOHP_CALL(d.alloc(*c.pool, c.n));
    return w.alloc(*c.pool, c.n);
  }
  dErr apply(Ctx &c, const T *r, T *z)
  {
    const double theta = 0.5 * (lmax + lmin), delta = 0.5 * (lmax - lmin), sigma = theta / delta;
    double rho = 1.0 / sigma;
    hipLaunchKernelGGL(dscale_kernel<T>, grid(c.n), dim3(256), 0, c.st, c.n, (T)(1.0 / theta), dinv, r, d.ptr);
    DOHP_HIP(hipMemcpyAsync(z, d.ptr, sizeof(T) * c.n, hipMemcpyDeviceToDevice, c.st));
    DOHP_HIP(hipMemcpyAsync(res.ptr, r, sizeof(T) * c.n, hipMemcpyDeviceToDevice, c.st));
    for (int k = 1; k < degree; k++) {
      DOHP_CALL(Ops<T>::Q(q1, d.ptr, w.ptr, c.st));
      DOHP_CALL(axpby<T>(c, T(-1), w.ptr, T(1), res.ptr));  // res = r - A z
      const double rho_new = 1.0 / (2.0 * sigma - rho);
      hipLaunchKernelGGL(dscale_kernel<T>, grid(c.n), dim3(256), 0, c.st, c.n, (T)(2.0 * rho_new / delta), dinv,
                         res.ptr, w.ptr);
      DOHP_CALL(axpby<T>(c, T(1), w.ptr, (T)(rho_new * rho), d.ptr));  // d = rho' rho d + 2 rho'/delta D^-1 res
      DOHP_CALL(axpby<T>(c, T(1), d.ptr, T(1), z));
      rho = rho_new;
    }
    return 0;
  }
};

__global__ void scale2_kernel(long n, const double *__restrict__ s, const void *__restrict__ x, void *__restrict__ y,
                              int f32)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (f32) ((float *)y)[i] = (float)s[i] * ((const float *)x)[i];
  else ((double *)y)[i] = s[i] * ((const double *)x)[i];
}

// Preconditioner of one precision: Jacobi-Chebyshev on the Q1 matrix, or a multigrid V-cycle on
// it, optionally corrected by learned node weights, z = S M(S r).
template <typename T>
struct Prec {
  Cheb<T> *cheb = nullptr;
  dohpMG mg = nullptr;
  dohpMG mg_fb = nullptr;  // plain multigrid taking over from mg (a learned embedded-Q1 matrix's) when learned_on drops
  const double *s = nullptr;  // learned node weights, or null
  T *tmp = nullptr;
  bool learned_on = false;
  dErr apply(Ctx &c, const T *r, T *z);
};
template <typename T>
dErr mg_apply(dohpMG mg, const T *r, T *z, hipStream_t st);
template <>
dErr mg_apply<double>(dohpMG mg, const double *r, double *z, hipStream_t st) { return dohpMGApply(mg, r, z, st); }
template <>
dErr mg_apply<float>(dohpMG mg, const float *r, float *z, hipStream_t st) { return dohpMGApplyF32(mg, r, z, st); }
template <typename T>
dErr Prec<T>::apply(Ctx &c, const T *r, T *z)
{
  if (!mg) return cheb->apply(c, r, z);
  if (mg_fb && !learned_on) return mg_apply<T>(mg_fb, r, z, c.st);
  if (!(s && learned_on)) return mg_apply<T>(mg, r, z, c.st);
  const int f32 = sizeof(T) == 4;
  hipLaunchKernelGGL(scale2_kernel, grid(c.n), dim3(256), 0, c.st, c.n, s, (const void *)r, (void *)tmp, f32);
  DOHP_CALL(mg_apply<T>(mg, tmp, z, c.st));
  hipLaunchKernelGGL(scale2_kernel, grid(c.n), dim3(256), 0, c.st, c.n, s, (const void *)z, (void *)z, f32);
  DOHP_HIP(hipGetLastError());
  return 0;
}

// Iteration budget shared by the sweeps of one solve: after `fallback_its` iterations with the
// learned correction, the plain preconditioner takes over.
struct Budget {
  int used = 0;
  int fallback_its = 0;
  int fell_back = 0;
};

// Largest eigenvalue of D^{-1} A_q1 by power iteration (FP64).
dErr estimate_lmax(Ctx &c, dohpMat q1, const double *dinv, int its, double *lmax)
{
  PoolBuf<double> v, w;
  DOHP_CALL(v.alloc(*c.pool, c.n));
  DOHP_CALL(w.alloc(*c.pool, c.n));
  std::vector<double> h(c.n);
  uint64_t s = 0x9E3779B97F4A7C15ULL;
  for (long i = 0; i < c.n; i++) {
    s ^= s << 13; s ^= s >> 7; s ^= s << 17;
    h[i] = (double)(s >> 11) / 9007199254740992.0 - 0.5;
  }
  DOHP_HIP(hipMemcpy(v.ptr, h.data(), sizeof(double) * c.n, hipMemcpyHostToDevice));
  double lam = 0, nv;
  DOHP_CALL(dot(c, v.ptr, v.ptr, &nv));
  DOHP_CALL(axpby<double>(c, 0.0, v.ptr, 1.0 / std::sqrt(nv), v.ptr));
  for (int k = 0; k < its; k++) {
    DOHP_CALL(dohpMatMult(q1, v.ptr, w.ptr, c.st));
    hipLaunchKernelGGL(dscale_kernel<double>, grid(c.n), dim3(256), 0, c.st, c.n, 1.0, dinv, w.ptr, w.ptr);
    double vw, ww;
    DOHP_CALL(dot(c, v.ptr, w.ptr, &vw));
    DOHP_CALL(dot(c, w.ptr, w.ptr, &ww));
    lam = vw;
    DOHP_CALL(axpby<double>(c, 1.0 / std::sqrt(ww), w.ptr, 0.0, v.ptr));
  }
  *lmax = lam;
  return 0;
}

// PCG on A x = b (x holds the initial guess).  Stops at ||r|| <= rtol ||b|| or max_it.  When the
// budget switches the learned correction off, CG restarts with the plain preconditioner from the
// current iterate.  snap (FP64 only): x after every `every`-th iteration, at most nsnap copies.
// flexible: beta in the Polak-Ribiere form z_{k+1}.(r_{k+1} - r_k) / z_k.r_k = -alpha z_{k+1}.q_k / z_k.r_k (one more
// dot product), equal to the usual z_{k+1}.r_{k+1} / z_k.r_k when the preconditioner is symmetric and exact, and
// robust when it is not: an FP32 V-cycle inside FP64 CG is symmetric only to FP32 rounding, which on the reference
// arithmetic's matrix at 48^3, p = 6 sometimes doubled the iteration count (91 -> 193).
// The preconditioner works on Z vectors: with Z = float inside FP64 CG, r is rounded to FP32 and z used exactly.
// The preconditioner of the next iteration is launched before ||r|| is known while the last known ||r|| is more than
// four times the tolerance (the wait is hidden behind it; were it the last iteration, one application is for nothing).
template <typename T, typename Z>
dErr pcg(Ctx &c, dohpEllip op, Prec<Z> &M, Budget &bud, const T *b, T *x, double rtol, int max_it, int *its,
         double *rnorm, double *bnorm, T *snap = nullptr, int nsnap = 0, int every = 0, int *nsnapped = nullptr,
         bool flexible = false)
{
  constexpr bool LOW = sizeof(Z) < sizeof(T);
  PoolBuf<T> r, p, q;
  PoolBuf<Z> z, lr;
  PoolBuf<double> part, sc;
  DOHP_CALL(r.alloc(*c.pool, c.n));
  DOHP_CALL(p.alloc(*c.pool, c.n));
  DOHP_CALL(q.alloc(*c.pool, c.n));
  DOHP_CALL(z.alloc(*c.pool, c.n));
  if (LOW) DOHP_CALL(lr.alloc(*c.pool, c.n));
  DOHP_CALL(part.alloc(*c.pool, 4 * kRedBlocks));
  DOHP_CALL(sc.alloc(*c.pool, 3));
  double *part_pq = part.ptr, *part_rr = part_pq + kRedBlocks, *part_rz = part_rr + kRedBlocks,
         *part_zq = part_rz + kRedBlocks, *alpha = sc.ptr + 2;
  const dim3 red(kRedBlocks), bs(256);
  float *lrp = LOW ? (float *)lr.ptr : nullptr;
  Event ev;
  DOHP_HIP(hipEventCreateWithFlags(&ev.e, hipEventDisableTiming));
  DOHP_CALL(Ops<T>::A(op, x, q.ptr, c.st));
  hipLaunchKernelGGL(krylov_init_kernel<T>, red, bs, 0, c.st, c.n, b, q.ptr, r.ptr, lrp, part_pq, part_rr);
  hipLaunchKernelGGL(krylov_read_kernel, dim3(1), bs, 0, c.st, part_pq, 2, c.host_dev);
  DOHP_HIP(hipStreamSynchronize(c.st));
  const double bb = c.host[0];
  double rr = c.host[1];
  *bnorm = std::sqrt(bb);
  DOHP_CHECK(std::isfinite(bb) && std::isfinite(rr), dohpERR_NAN, "PCG: non-finite right-hand side or initial residual");
  const double tol = rtol * std::sqrt(bb);
  int k = 0, ns = 0;
  bool restart = false;
  auto switches = [&](int used) { return M.learned_on && bud.fallback_its > 0 && used >= bud.fallback_its; };
  auto fall_back = [&]() {
    if (!switches(bud.used)) return;
    M.learned_on = false;
    bud.fell_back = 1;
    restart = true;
  };
  auto precondition = [&]() -> dErr {
    fall_back();
    if constexpr (LOW) return M.apply(c, lr.ptr, z.ptr);
    else return M.apply(c, r.ptr, z.ptr);
  };
  // p and r.z of the next iteration from z (k counts the slots of r.z, which alternate)
  auto direction = [&](int mode) -> dErr {
    const T *qz = mode == KB_FLEXIBLE ? q.ptr : nullptr;
    hipLaunchKernelGGL((krylov_zdots_kernel<T, Z>), red, bs, 0, c.st, c.n, r.ptr, z.ptr, qz, part_rz, part_zq);
    hipLaunchKernelGGL((krylov_direction_kernel<T, Z>), red, bs, 0, c.st, c.n, mode, part_rz, part_zq,
                       sc.ptr + ((k + 1) & 1), sc.ptr + (k & 1), alpha, z.ptr, p.ptr, q.ptr);
    DOHP_HIP(hipGetLastError());
    return 0;
  };
  if (std::sqrt(rr) > tol && max_it > 0) {
    DOHP_CALL(precondition());
    restart = false;
    DOHP_CALL(direction(KB_FIRST));
  }
  while (std::sqrt(rr) > tol && k < max_it) {
    DOHP_CALL(Ops<T>::A_add(op, p.ptr, q.ptr, c.st));  // (q is zero)
    hipLaunchKernelGGL(dot_partial_kernel<T>, red, bs, 0, c.st, c.n, p.ptr, q.ptr, part_pq);
    hipLaunchKernelGGL(krylov_update_kernel<T>, red, bs, 0, c.st, c.n, part_pq, sc.ptr + (k & 1), alpha, p.ptr, q.ptr, x,
                       r.ptr, lrp, part_rr);
    hipLaunchKernelGGL(krylov_read_kernel, dim3(1), bs, 0, c.st, part_rr, 1, c.host_dev);
    DOHP_HIP(hipGetLastError());
    DOHP_HIP(hipEventRecord(ev.e, c.st));
    const bool ahead = std::sqrt(rr) > 4 * tol && k + 1 < max_it && !switches(bud.used + 1);
    if (ahead) DOHP_CALL(precondition());
    DOHP_HIP(hipEventSynchronize(ev.e));
    rr = c.host[0];
    if (!std::isfinite(rr)) DOHP_HIP(hipStreamSynchronize(c.st));  // (the work vectors go back to the pool)
    DOHP_CHECK(std::isfinite(rr), dohpERR_NAN, "PCG: non-finite residual at iteration " + std::to_string(k + 1));
    k++;
    bud.used++;
    if (snap && every > 0 && k % every == 0 && ns < nsnap) {
      DOHP_HIP(hipMemcpyAsync(snap + (long)ns * c.n, x, sizeof(T) * c.n, hipMemcpyDeviceToDevice, c.st));
      ns++;
    }
    if (std::sqrt(rr) <= tol) break;
    if (k >= max_it) {  // (a budget used up by the last iteration is reported)
      fall_back();
      break;
    }
    if (!ahead) DOHP_CALL(precondition());
    // (a preconditioner that changed starts a new Krylov sequence)
    DOHP_CALL(direction(restart ? KB_FIRST : flexible ? KB_FLEXIBLE : KB_STANDARD));
    restart = false;
  }
  *its = k;
  *rnorm = std::sqrt(rr);
  if (nsnapped) *nsnapped = ns;
  return 0;
}

}  // namespace

namespace {

// Multigrid hierarchy of q1 at smoothing degree `deg` (0 = the default for its arithmetic), kept with the matrix.
dErr hierarchy(dohpMat q1, int deg, hipStream_t st, dohpMG *mg)
{
  deg = deg > 0 ? deg : (q1->corrected || q1->scaled ? 1 : 2);
  if (q1->mg && q1->mg_degree == deg) {
    if (q1->mg_stale) DOHP_CALL(dohpMGRefresh(q1->mg, q1, st));
  } else {
    dohpMGDestroy(&q1->mg);
    DOHP_CALL(dohpMGCreate(q1, deg, 0, &q1->mg, st));
    q1->mg_degree = deg;
  }
  q1->mg_stale = false;
  *mg = q1->mg;
  return 0;
}

dErr solve_impl(dohpEllip op, dohpMat q1, dohpMLP mlp, const double *b, double *x, const dohpSolveOpts *opts,
                dohpSolveStats *stats, double *snap, int nsnap, int every, int *nsnapped, hipStream_t st,
                dohpMat q1fb = nullptr)
{
  DOHP_CHECK(op && q1 && b && x && opts && stats, dohpERR_ARG, "null argument");
  DOHP_CHECK(opts->pc >= 0 && opts->pc <= 1, dohpERR_ARG, "pc must be 0 (Jacobi-Chebyshev) or 1 (multigrid)");
  DOHP_CHECK(!mlp || opts->pc == 1, dohpERR_ARG, "the learned correction applies to the multigrid preconditioner");
  DOHP_CHECK(!q1fb || opts->pc == 1, dohpERR_ARG, "the fallback matrix applies to the multigrid preconditioner");
  const auto t0 = std::chrono::steady_clock::now();
  Ctx c;
  c.st = st;
  long nrows;
  DOHP_CALL(dohpMatGetSizes(q1, &nrows, nullptr));
  c.n = nrows;
  c.pool = dohpEllipPool_Private(op);
  DOHP_CALL(c.part.alloc(*c.pool, kRedBlocks));
  DOHP_CALL(c.res.alloc(*c.pool, 1));
  DOHP_CALL(dohpEllipPinned_Private(op, &c.host, &c.host_dev));
  *stats = dohpSolveStats{};
  // Jacobi scaling and, for the one-level preconditioner, the Chebyshev interval
  // [lmax/ratio, 1.05 lmax] of D^{-1} A_q1
  PoolBuf<double> diag, dinv;
  PoolBuf<float> dinv32;
  if (opts->pc == 0 || mlp) {
    DOHP_CALL(diag.alloc(*c.pool, c.n));
    DOHP_CALL(dinv.alloc(*c.pool, c.n));
    DOHP_CALL(dinv32.alloc(*c.pool, c.n));
    DOHP_CALL(dohpMatGetDiagonal(q1, diag.ptr, c.st));
    hipLaunchKernelGGL(inv_kernel, grid(c.n), dim3(256), 0, c.st, c.n, diag.ptr, dinv.ptr, dinv32.ptr);
  }
  double lmax = 1.0;
  if (opts->pc == 0) {
    DOHP_CALL(estimate_lmax(c, q1, dinv.ptr, opts->eig_its > 0 ? opts->eig_its : 20, &lmax));
    lmax *= 1.05;
  }
  const double lmin = lmax / (opts->cheb_ratio > 1 ? opts->cheb_ratio : 30.0);
  stats->lmax = lmax;
  const int degree = opts->cheb_degree > 0 ? opts->cheb_degree : 4;
  struct {
    dohpMG mg = nullptr, mg_fb = nullptr;
  } mgh;
  if (opts->pc == 1) {  // the hierarchy is kept with the matrix until it is refilled
    // default smoothing degree: 1 on the corrected Q1 matrix and on one with learned sub-cell scales (fastest,
    // measured), 2 on the reference arithmetic's (where degree 1 with the FP32 V-cycle can stall); a fallback
    // matrix gets its own default
    DOHP_CALL(hierarchy(q1, opts->mg_degree, c.st, &mgh.mg));
    if (q1fb) DOHP_CALL(hierarchy(q1fb, opts->mg_degree, c.st, &mgh.mg_fb));
    DOHP_CHECK(opts->mg_coeffs == 0 || opts->mg_coeffs == 1, dohpERR_ARG, "mg_coeffs must be 0 (FP16) or 1 (FP32)");
    DOHP_CALL(dohpMGSetCoefficients(mgh.mg, opts->mg_coeffs == 0));
    if (mgh.mg_fb) DOHP_CALL(dohpMGSetCoefficients(mgh.mg_fb, opts->mg_coeffs == 0));
  }
  Budget bud;
  bud.fallback_its = mlp || q1fb ? opts->fallback_its : 0;
  // learned node weights (computed once: the features do not depend on the residual)
  PoolBuf<double> wts;
  PoolBuf<double> tmp64;
  PoolBuf<float> tmp32;
  if (mlp) {
    dohpFS fs;
    dohpEllipParam prm;
    const double *kv, *stt;
    DOHP_CALL(dohpEllipGetQ1Context_Private(op, &fs, &prm, &kv, &stt, nullptr));
    long np;
    DOHP_CALL(dohpMLPNumPatches(q1, &np));
    PoolBuf<float> X;
    DOHP_CALL(X.alloc(*c.pool, (size_t)(np > 0 ? np : 1) * dohpMLPNumInputs()));
    DOHP_CALL(wts.alloc(*c.pool, c.n));
    DOHP_CALL(dohpMLPFeatures(q1, fs, dinv.ptr, X.ptr, c.st));
    DOHP_CALL(dohpMLPWeights(mlp, q1, X.ptr, wts.ptr, nullptr, c.st));
    DOHP_CALL(tmp64.alloc(*c.pool, c.n));
    DOHP_CALL(tmp32.alloc(*c.pool, c.n));
    DOHP_HIP(hipStreamSynchronize(c.st));
  }
  const auto t_setup = std::chrono::steady_clock::now();
  stats->setup_seconds = std::chrono::duration<double>(t_setup - t0).count();
  if (opts->mixed == 2) {  // FP64 PCG, preconditioner in FP32
    Cheb<float> C32{q1, dinv32.ptr, lmin, lmax, degree};
    if (opts->pc == 0) DOHP_CALL(C32.alloc(c));
    Prec<float> M32;
    M32.cheb = &C32;
    M32.mg = mgh.mg;
    M32.mg_fb = mgh.mg_fb;
    M32.s = wts.ptr;
    M32.tmp = tmp32.ptr;
    M32.learned_on = mlp != nullptr || q1fb != nullptr;
    int its;
    double rn, bn;
    DOHP_CALL((pcg<double, float>(c, op, M32, bud, b, x, opts->rtol, opts->max_it, &its, &rn, &bn, snap, nsnap, every,
                                  nsnapped, true)));
    stats->inner_its = its;
    stats->outer_its = 1;
    stats->rnorm = rn;
    stats->bnorm = bn;
  } else if (!opts->mixed) {
    Cheb<double> C64{q1, dinv.ptr, lmin, lmax, degree};
    if (opts->pc == 0) DOHP_CALL(C64.alloc(c));
    Prec<double> M;
    M.cheb = &C64;
    M.mg = mgh.mg;
    M.mg_fb = mgh.mg_fb;
    M.s = wts.ptr;
    M.tmp = tmp64.ptr;
    M.learned_on = mlp != nullptr || q1fb != nullptr;
    int its;
    double rn, bn;
    DOHP_CALL((pcg<double, double>(c, op, M, bud, b, x, opts->rtol, opts->max_it, &its, &rn, &bn, snap, nsnap, every,
                                   nsnapped)));
    stats->inner_its = its;
    stats->outer_its = 1;
    stats->rnorm = rn;
    stats->bnorm = bn;
  } else {
    Cheb<float> C32{q1, dinv32.ptr, lmin, lmax, degree};
    if (opts->pc == 0) DOHP_CALL(C32.alloc(c));
    Prec<float> M;
    M.cheb = &C32;
    M.mg = mgh.mg;
    M.mg_fb = mgh.mg_fb;
    M.s = wts.ptr;
    M.tmp = tmp32.ptr;
    M.learned_on = mlp != nullptr || q1fb != nullptr;
    PoolBuf<double> r, t;
    PoolBuf<float> r32, e32;
    DOHP_CALL(r.alloc(*c.pool, c.n));
    DOHP_CALL(t.alloc(*c.pool, c.n));
    DOHP_CALL(r32.alloc(*c.pool, c.n));
    DOHP_CALL(e32.alloc(*c.pool, c.n));
    double bb;
    DOHP_CALL(dot(c, b, b, &bb));
    stats->bnorm = std::sqrt(bb);
    int outer = 0, inner_total = 0;
    for (;;) {
      // FP64 defect r = b - A64 x
      DOHP_CALL(dohpEllipMatMult_Private(op, x, t.ptr, c.st));
      DOHP_HIP(hipMemcpyAsync(r.ptr, b, sizeof(double) * c.n, hipMemcpyDeviceToDevice, c.st));
      DOHP_CALL(axpby<double>(c, -1.0, t.ptr, 1.0, r.ptr));
      double rr;
      DOHP_CALL(dot(c, r.ptr, r.ptr, &rr));
      stats->rnorm = std::sqrt(rr);
      DOHP_CHECK(std::isfinite(rr), dohpERR_NAN, "defect correction: non-finite FP64 residual");
      if (stats->rnorm <= opts->rtol * stats->bnorm || outer >= opts->max_outer) break;
      // FP32 correction, normalized so the inner problem is O(1)
      const double s = 1.0 / stats->rnorm;
      hipLaunchKernelGGL(demote_kernel, grid(c.n), dim3(256), 0, c.st, c.n, s, r.ptr, r32.ptr);
      hipLaunchKernelGGL(fill_kernel<float>, grid(c.n), dim3(256), 0, c.st, c.n, 0.0f, e32.ptr);
      int its;
      double rn, bn;
      // the last sweep needs only the reduction that is left to reach rtol ||b||
      const double need = 0.5 * opts->rtol * stats->bnorm / stats->rnorm;
      const double irtol = std::max(opts->inner_rtol, need);
      DOHP_CALL((pcg<float, float>(c, op, M, bud, r32.ptr, e32.ptr, irtol, opts->max_it, &its, &rn, &bn)));
      inner_total += its;
      hipLaunchKernelGGL(promote_add_kernel, grid(c.n), dim3(256), 0, c.st, c.n, stats->rnorm, e32.ptr, x);
      outer++;
    }
    stats->outer_its = outer;
    stats->inner_its = inner_total;
  }
  stats->fallback = bud.fell_back;
  DOHP_HIP(hipStreamSynchronize(c.st));
  stats->seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  return 0;
}

}  // namespace

extern "C" dErr dohpEllipSolve(dohpEllip op, dohpMat q1, const double *b, double *x, const dohpSolveOpts *opts,
                               dohpSolveStats *stats, void *stream)
{
  return solve_impl(op, q1, nullptr, b, x, opts, stats, nullptr, 0, 0, nullptr, (hipStream_t)stream);
}

extern "C" dErr dohpEllipSolveLearned(dohpEllip op, dohpMat q1, dohpMLP mlp, const double *b, double *x,
                                      const dohpSolveOpts *opts, dohpSolveStats *stats, void *stream)
{
  DOHP_CHECK(mlp, dohpERR_ARG, "null network");
  return solve_impl(op, q1, mlp, b, x, opts, stats, nullptr, 0, 0, nullptr, (hipStream_t)stream);
}

extern "C" dErr dohpEllipSolveRecord(dohpEllip op, dohpMat q1, const double *b, double *x, const dohpSolveOpts *opts,
                                     dohpSolveStats *stats, double *snap_dev, int nsnap, int every, int *nsnapped,
                                     void *stream)
{
  DOHP_CHECK(opts && !opts->mixed, dohpERR_ARG, "iterates are recorded by the plain FP64 solve");
  DOHP_CHECK(snap_dev && nsnap > 0 && every > 0 && nsnapped, dohpERR_ARG, "bad snapshot arguments");
  return solve_impl(op, q1, nullptr, b, x, opts, stats, snap_dev, nsnap, every, nsnapped, (hipStream_t)stream);
}

extern "C" dErr dohpEllipSolveFallback(dohpEllip op, dohpMat q1, dohpMat q1_fallback, const double *b, double *x,
                                       const dohpSolveOpts *opts, dohpSolveStats *stats, void *stream)
{
  DOHP_CHECK(q1_fallback, dohpERR_ARG, "null fallback matrix");
  return solve_impl(op, q1, nullptr, b, x, opts, stats, nullptr, 0, 0, nullptr, (hipStream_t)stream, q1_fallback);
}

// Batched dEFSApply for isotropic tensor-product hexahedra (dEFSApply_Tensor_Hex,
// src/jacobi/impls/tensor/efstopo.c:368-423, with TensorMult_Hex_nounroll,
// src/jacobi/impls/tensor/inlinetmulthex.h:19-100, and the geometry mappings of
// efstopo.c:518-623).
#include <algorithm>
#include <mutex>
#include <vector>

#include "common.h"

using namespace dohp;

namespace {

constexpr int kEfsMaxP = 12;
constexpr int kEfsTab = 2 * kEfsMaxP * kEfsMaxP;  // B and D, [out][in] each

// Arguments of one launch, tables included (2.4 KB of kernel arguments, read as scalars: no device copy of the tables, so
// calls need no allocation and do not share anything).  a: length of the contracted lines, b: length of the results.
struct EfsArgs {
  int b, D, dc, nelem, epb, add;
  const double *jinv, *in;
  double *out;
  double tab[kEfsTab];
};
enum { EFS_INTERP, EFS_GRAD, EFS_GRAD_T };

__host__ __device__ constexpr int odd(int n) { return n | 1; }
// LDS of one element with dc components (doubles): region 0, then region 1 (see efs_kernel).
__host__ __device__ constexpr int efs_r0(int mode, int a, int b, int dc)
{
  const int pz = odd(b * dc), pa = odd(a * dc), x = a * a * pa;
  if (mode == EFS_GRAD_T) return 3 * b * a * pa > b * b * b * dc ? 3 * b * a * pa : b * b * b * dc;
  const int y = (mode == EFS_GRAD ? 3 : 1) * a * b * pz;
  return x > y ? x : y;
}
__host__ __device__ constexpr int efs_r1(int mode, int a, int b, int dc)
{
  return mode == EFS_GRAD_T ? 2 * b * b * odd(a * dc) : (mode == EFS_GRAD ? 2 : 1) * a * a * odd(b * dc);
}

// out(q) = sum_m M[q][m] in[m] for a line held in registers; the row of M is uniform over the workgroup.  From five points
// on the two halves are summed from the line's ends inwards and added: half the chain, and fewer roundings in each.  Error
// against 80-bit arithmetic, one chain and halves, in 1e-16: interpolation from 5 points 1.36 and 1.28, from 7 1.59 and
// 1.40, from 12 2.07 and 1.64; the gradient's transpose from 4 points 1.61 and 1.63.  (Every other point in a second chain:
// 1.46 from 7 points, but 1.17 from 2 where one chain has 0.98.)
template <int A>
__device__ __forceinline__ double row_dot(const double *M, int q, const double (&in)[A])
{
  constexpr int H = A > 4 ? (A + 1) / 2 : A;
  double s = 0.0, t = 0.0;
#pragma unroll
  for (int m = 0; m < H; m++) s = fma(M[q * A + m], in[m], s);
  if constexpr (H == A) return s;
#pragma unroll
  for (int m = A - 1; m >= H; m--) t = fma(M[q * A + m], in[m], t);
  return s + t;
}

// A workgroup takes epb elements, dc components at a time.  Values keep the reference's order [i][j][k][d] in LDS; every
// pass contracts one index of one line per thread, the line in registers and the table row as scalar operands, so an
// element's tables are read once per line and no value is read from LDS more than once per pass.  The gradient shares
// its partial products (8 line passes instead of 9 full contractions of three):
//   forward:  along k: B x, D x;  along j: B, D of the first, B of the second;  along i: D, B, B, straight to the output
//   transpose: along i: the mapped fluxes, straight from the input, D^T, B^T, B^T;  along j: B^T + D^T, B^T;  along k.
// Rows of lines along k have an odd pitch (bank conflicts at even lengths).  What bounds it is the bytes: input, inverse
// Jacobians and output once each.  8192 elements, P = Q = 7, D = 1, gradient with inverse Jacobians (292 MB): 221 -> 65 us
// (4.5 TB/s) against three full contractions per component out of LDS with the output updated once per direction; 1500
// elements, P = 4, Q = 5, D = 3, transposed gradient (29 MB): 28.0 -> 9.2 us.
template <int A, int MODE, bool ONE>
__global__ void __launch_bounds__(256) efs_kernel(EfsArgs g)
{
  extern __shared__ double lds[];
  constexpr int AA = A * A, A3 = AA * A;
  const int tid = threadIdx.x, b = g.b, D = ONE ? 1 : g.D, bb = b * b, b3 = bb * b;
  const long e0 = (long)blockIdx.x * g.epb;
  const int ne = (int)min((long)g.epb, g.nelem - e0);
  const double *B = g.tab, *Dm = g.tab + b * A;
  for (int d0 = 0; d0 < D; d0 += g.dc) {
    const int dc = ONE ? 1 : min(g.dc, D - d0), aw = A * dc, bw = b * dc;
    const int pa = odd(aw), pb = odd(bw), s0 = efs_r0(MODE, A, b, dc), s1 = efs_r1(MODE, A, b, dc);
    double *R0 = lds, *R1 = lds + ne * s0;
    if constexpr (MODE != EFS_GRAD_T) {
      constexpr int NZ = MODE == EFS_GRAD ? 2 : 1, NY = MODE == EFS_GRAD ? 3 : 1;
      const int sz = AA * pb, sy = A * b * pb;
      for (int t = tid; t < ne * AA * aw; t += 256) {
        const int l = t / (AA * aw), t2 = t - l * AA * aw, r = t2 / aw, c = t2 - r * aw, k = ONE ? c : c / dc;
        R0[l * s0 + r * pa + c] = g.in[((e0 + l) * A3 + r * A + k) * D + d0 + (c - k * dc)];
      }
      __syncthreads();
      for (int t = tid; t < ne * AA * dc; t += 256) {  // along k
        const int l = t / (AA * dc), t2 = t - l * AA * dc, r = ONE ? t2 : t2 / dc, d = t2 - r * dc;
        double v[A];
#pragma unroll
        for (int m = 0; m < A; m++) v[m] = R0[l * s0 + r * pa + m * dc + d];
        double *o = &R1[l * s1 + r * pb + d];
        for (int q = 0; q < b; q++) {
          o[q * dc] = row_dot<A>(B, q, v);
          if (NZ > 1) o[sz + q * dc] = row_dot<A>(Dm, q, v);
        }
      }
      __syncthreads();
      for (int t = tid; t < ne * A * bw; t += 256) {  // along j
        const int l = t / (A * bw), t2 = t - l * A * bw, i = t2 / bw, c = t2 - i * bw;
        const double *z = &R1[l * s1 + i * A * pb + c];
        double *o = &R0[l * s0 + i * b * pb + c];
        double v[A], w[NZ > 1 ? A : 1];
#pragma unroll
        for (int m = 0; m < A; m++) {
          v[m] = z[m * pb];
          if constexpr (NZ > 1) w[m] = z[sz + m * pb];
        }
        for (int q = 0; q < b; q++) {
          o[q * pb] = row_dot<A>(B, q, v);
          if constexpr (NZ > 1) {
            o[sy + q * pb] = row_dot<A>(Dm, q, v);
            o[2 * sy + q * pb] = row_dot<A>(B, q, w);
          }
        }
      }
      __syncthreads();
      for (int t = tid; t < ne * b * bw; t += 256) {  // along i
        const int l = t / (b * bw), t2 = t - l * b * bw, j = t2 / bw, c = t2 - j * bw, k = ONE ? c : c / dc;
        const double *y = &R0[l * s0 + j * pb + c];
        double v[NY][A];
#pragma unroll
        for (int m = 0; m < A; m++)
#pragma unroll
          for (int n = 0; n < NY; n++) v[n][m] = y[n * sy + m * b * pb];
        const long pt0 = (e0 + l) * b3 + j * b + k;
        const int d = d0 + (c - k * dc);
        for (int q = 0; q < b; q++) {
          const long pt = pt0 + q * bb;
          if constexpr (MODE == EFS_INTERP) {
            const double r = row_dot<A>(B, q, v[0]);
            double *o = &g.out[pt * D + d];
            *o = g.add ? *o + r : r;
          } else {
            const double f0 = row_dot<A>(Dm, q, v[0]), f1 = row_dot<A>(B, q, v[1]), f2 = row_dot<A>(B, q, v[2]);
            double r[3] = {f0, f1, f2};
            if (g.jinv) {
              const double *J = g.jinv + pt * 9;
#pragma unroll
              for (int e = 0; e < 3; e++) r[e] = f0 * J[e] + f1 * J[3 + e] + f2 * J[6 + e];
            }
            double *o = &g.out[(pt * D + d) * 3];
#pragma unroll
            for (int e = 0; e < 3; e++) o[e] = g.add ? o[e] + r[e] : r[e];
          }
        }
      }
    } else {
      const int sx = b * A * pa, sy = bb * pa;
      for (int t = tid; t < ne * A * aw; t += 256) {  // along i
        const int l = t / (A * aw), t2 = t - l * A * aw, j = t2 / aw, c = t2 - j * aw, k = ONE ? c : c / dc;
        const long pt0 = (e0 + l) * A3 + j * A + k;
        const int d = d0 + (c - k * dc);
        double f[3][A];
#pragma unroll
        for (int m = 0; m < A; m++) {
          const long pt = pt0 + m * AA;
          const double *u = &g.in[(pt * D + d) * 3], *J = g.jinv + pt * 9;
          const double u0 = u[0], u1 = u[1], u2 = u[2];
#pragma unroll
          for (int n = 0; n < 3; n++) f[n][m] = u0 * J[n * 3] + u1 * J[n * 3 + 1] + u2 * J[n * 3 + 2];
        }
        double *o = &R0[l * s0 + j * pa + c];
        for (int q = 0; q < b; q++) {
          o[q * A * pa] = row_dot<A>(Dm, q, f[0]);
          o[sx + q * A * pa] = row_dot<A>(B, q, f[1]);
          o[2 * sx + q * A * pa] = row_dot<A>(B, q, f[2]);
        }
      }
      __syncthreads();
      for (int t = tid; t < ne * b * aw; t += 256) {  // along j
        const int l = t / (b * aw), t2 = t - l * b * aw, i = t2 / aw, c = t2 - i * aw;
        const double *x = &R0[l * s0 + i * A * pa + c];
        double v[3][A];
#pragma unroll
        for (int m = 0; m < A; m++)
#pragma unroll
          for (int n = 0; n < 3; n++) v[n][m] = x[n * sx + m * pa];
        double *o = &R1[l * s1 + i * b * pa + c];
        for (int q = 0; q < b; q++) {
          o[q * pa] = row_dot<A>(B, q, v[0]) + row_dot<A>(Dm, q, v[1]);
          o[sy + q * pa] = row_dot<A>(B, q, v[2]);
        }
      }
      __syncthreads();
      for (int t = tid; t < ne * bb * dc; t += 256) {  // along k
        const int l = t / (bb * dc), t2 = t - l * bb * dc, r = ONE ? t2 : t2 / dc, d = t2 - r * dc;
        const double *y = &R1[l * s1 + r * pa + d];
        double v[2][A];
#pragma unroll
        for (int m = 0; m < A; m++)
#pragma unroll
          for (int n = 0; n < 2; n++) v[n][m] = y[n * sy + m * dc];
        double *o = &R0[l * s0 + r * bw + d];
        for (int q = 0; q < b; q++) o[q * dc] = row_dot<A>(B, q, v[0]) + row_dot<A>(Dm, q, v[1]);
      }
      __syncthreads();
      for (int t = tid; t < ne * bb * bw; t += 256) {
        const int l = t / (bb * bw), t2 = t - l * bb * bw, r = ONE ? t2 : t2 / dc;
        double *o = &g.out[((e0 + l) * b3 + r) * D + d0 + (t2 - r * dc)];
        const double v = R0[l * s0 + t2];
        *o = g.add ? *o + v : v;
      }
    }
    if (d0 + g.dc < D) __syncthreads();  // the next components overwrite the regions
  }
}

// 1-D weights of a tensor rule, passed by value.
struct RuleW {
  double w[kMaxN];
};

// dRuleComputePhysical for every point of nelem elements (one thread per point): the cofactor inverse of
// dGeomInvert3 (include/dohpgeom.h:57-75, same operation order), jw = w_i w_j w_k det.  flag[0] is set at a
// negative determinant (jacobi.c:397), flag[1] at a non-finite one (pinned host memory).  The 72-byte matrices go through
// LDS, so that global memory is read and written in order (lane-strided reads of them, nine passes over 4.6 KB per
// wavefront, outgrow the first-level cache); matrices lie nine doubles apart there, without bank conflicts.  2.8 M points
// (427 MB): 120 -> 100 us a call.
__global__ void __launch_bounds__(256) rule_physical_kernel(int Q, RuleW rw, long npts, const double *__restrict__ jac,
                                                            double *__restrict__ jinv, double *__restrict__ jw,
                                                            int *__restrict__ flag)
{
  __shared__ double m[256 * 9];
  const int tid = threadIdx.x;
  const long p0 = (long)blockIdx.x * 256, t = p0 + tid;
  const int nm = (int)min(256L, npts - p0) * 9;
#pragma unroll
  for (int r = 0; r < 9; r++)
    if (r * 256 + tid < nm) m[r * 256 + tid] = jac[p0 * 9 + r * 256 + tid];
  __syncthreads();
  if (t < npts) {
    const int Q3 = Q * Q * Q, q = (int)(t % Q3), i = q / (Q * Q), j = (q / Q) % Q, k = q % Q;
    double a[9];
#pragma unroll
    for (int r = 0; r < 9; r++) a[r] = m[tid * 9 + r];
    const double b0 = (a[1 * 3 + 1] * a[2 * 3 + 2] - a[2 * 3 + 1] * a[1 * 3 + 2]);
    const double b3 = -(a[1 * 3 + 0] * a[2 * 3 + 2] - a[2 * 3 + 0] * a[1 * 3 + 2]);
    const double b6 = (a[1 * 3 + 0] * a[2 * 3 + 1] - a[2 * 3 + 0] * a[1 * 3 + 1]);
    const double det = a[0] * b0 + a[1] * b3 + a[2] * b6;
    const double id = 1.0 / det;
    double *b = &m[tid * 9];
    b[0] = id * b0;
    b[1] = -id * (a[0 * 3 + 1] * a[2 * 3 + 2] - a[2 * 3 + 1] * a[0 * 3 + 2]);
    b[2] = id * (a[0 * 3 + 1] * a[1 * 3 + 2] - a[1 * 3 + 1] * a[0 * 3 + 2]);
    b[3] = id * b3;
    b[4] = id * (a[0 * 3 + 0] * a[2 * 3 + 2] - a[2 * 3 + 0] * a[0 * 3 + 2]);
    b[5] = -id * (a[0 * 3 + 0] * a[1 * 3 + 2] - a[1 * 3 + 0] * a[0 * 3 + 2]);
    b[6] = id * b6;
    b[7] = -id * (a[0 * 3 + 0] * a[2 * 3 + 1] - a[2 * 3 + 0] * a[0 * 3 + 1]);
    b[8] = id * (a[0 * 3 + 0] * a[1 * 3 + 1] - a[1 * 3 + 0] * a[0 * 3 + 1]);
    jw[t] = rw.w[i] * rw.w[j] * rw.w[k] * det;
    if (det < 0.0) flag[0] = 1;
    if (!__builtin_isfinite(det)) flag[1] = 1;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 9; r++)
    if (r * 256 + tid < nm) jinv[p0 * 9 + r * 256 + tid] = m[r * 256 + tid];
}

// Two pinned flags for one call, which a kernel sets and the host reads after its wait.  At most kKept pairs are kept
// for later calls (any thread, any device); the rest, and those at the library's end, are freed.  A device flag that a
// call allocates, clears, copies back and frees took 12 of the 28 us of a call on 2400 points.
class PinnedFlags {
  static constexpr size_t kKept = 8;
  struct Store {
    std::mutex m;
    std::vector<int *> kept;
    ~Store()
    {
      for (int *p : kept) (void)hipHostFree(p);
    }
  };
  static Store &store()
  {
    static Store s;
    return s;
  }
  int *p = nullptr;
  bool idle = false;

public:
  PinnedFlags() = default;
  PinnedFlags(const PinnedFlags &) = delete;
  PinnedFlags &operator=(const PinnedFlags &) = delete;
  dErr acquire()
  {
    {
      Store &s = store();
      std::lock_guard<std::mutex> lock(s.m);
      if (!s.kept.empty()) {
        p = s.kept.back();
        s.kept.pop_back();
      }
    }
    if (!p && hipHostMalloc((void **)&p, 2 * sizeof(int), hipHostMallocPortable) != hipSuccess) {
      p = nullptr;
      (void)hipGetLastError();
      set_error("pinned allocation failed");
      return dohpERR_OOM;
    }
    p[0] = p[1] = 0;
    return 0;
  }
  int *ptr() const { return p; }
  void waited() { idle = true; }
  int read(int i) const { return ((volatile int *)p)[i]; }
  ~PinnedFlags()
  {
    if (!p || !idle) return;  // (a kernel that was not waited for may still write: the pair is given up)
    Store &s = store();
    std::lock_guard<std::mutex> lock(s.m);
    if (s.kept.size() < kKept)
      s.kept.push_back(p);
    else
      (void)hipHostFree(p);
  }
};

}  // namespace

extern "C" dErr dRuleComputePhysicalBatched(int Q, const double *weight, int nelem, const double *jac, double *jinv,
                                            double *jw, void *stream)
{
  DOHP_CHECK(Q >= 1 && Q <= kMaxN, dohpERR_ARG, "dRuleComputePhysicalBatched supports 1 <= Q <= 16");
  DOHP_CHECK(nelem >= 0, dohpERR_ARG, "negative element count");
  DOHP_CHECK(weight && jac && jinv && jw, dohpERR_ARG, "null argument");  // jacobi.c:389-390
  if (nelem == 0) return 0;
  RuleW rw{};
  for (int q = 0; q < Q; q++) rw.w[q] = weight[q];
  hipStream_t st = (hipStream_t)stream;
  PinnedFlags flag;
  DOHP_CALL(flag.acquire());
  const long npts = (long)nelem * Q * Q * Q;
  hipLaunchKernelGGL(rule_physical_kernel, dim3((unsigned)((npts + 255) / 256)), dim3(256), 0, st, Q, rw, npts, jac,
                     jinv, jw, flag.ptr());
  DOHP_HIP(hipGetLastError());
  DOHP_HIP(hipStreamSynchronize(st));
  flag.waited();
  DOHP_CHECK(!flag.read(0), dohpERR_NEGATIVE_JACOBIAN, "Negative Jacobian at a quadrature point");
  DOHP_CHECK(!flag.read(1), dohpERR_NAN, "Non-finite Jacobian determinant at a quadrature point");
  return 0;
}

namespace {

dErr efs_check(int P, int Q, int nelem, const double *rcoord, const double *jinv, int D, const double *in,
               double *out, int amode, int imode)
{
  DOHP_CHECK(P >= 2 && P <= kEfsMaxP && Q >= 1 && Q <= kEfsMaxP, dohpERR_ARG,
             "dEFSApplyHexBatched supports 2<=P<=12, 1<=Q<=12");
  DOHP_CHECK(nelem >= 0, dohpERR_ARG, "negative element count");
  DOHP_CHECK(D >= 1, dohpERR_ARG, "dofs must be positive");  // jacobi.c:495
  DOHP_CHECK(imode == dINSERT_VALUES || imode == dADD_VALUES, dohpERR_ARG, "InsertMode not supported");
  DOHP_CHECK(amode >= dAPPLY_INTERP && amode <= dAPPLY_GRAD_TRANSPOSE, dohpERR_ARG, "invalid dApplyMode");
  DOHP_CHECK(amode != dAPPLY_GRAD_TRANSPOSE || jinv, dohpERR_ARG, "No Jinv, need a mapping");
  DOHP_CHECK(rcoord && in && out, dohpERR_ARG, "null argument");
  return 0;
}

template <int A, int MODE>
dErr efs_launch(const EfsArgs &g, size_t lds, hipStream_t st)
{
  const auto kernel = g.D == 1 ? efs_kernel<A, MODE, true> : efs_kernel<A, MODE, false>;
  if (lds > 65536)
    DOHP_HIP(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(kernel, dim3((unsigned)((g.nelem + g.epb - 1) / g.epb)), dim3(256), lds, st, g);
  DOHP_HIP(hipGetLastError());
  return 0;
}

template <int MODE>
dErr efs_dispatch(int a, const EfsArgs &g, size_t lds, hipStream_t st)
{
  switch (a) {
#define DOHP_CASE(AA) \
  case AA: return efs_launch<AA, MODE>(g, lds, st);
    DOHP_CASE(1)
    DOHP_CASE(2)
    DOHP_CASE(3)
    DOHP_CASE(4)
    DOHP_CASE(5)
    DOHP_CASE(6)
    DOHP_CASE(7)
    DOHP_CASE(8)
    DOHP_CASE(9)
    DOHP_CASE(10)
    DOHP_CASE(11)
    DOHP_CASE(12)
#undef DOHP_CASE
  }
  return dohpERR_ARG;  // (not reached: P and Q are checked)
}

// Lays out one launch.  All components of an element at once while they fit in 64 KB of LDS (the gradients' largest
// element, P = Q = 12, takes 75 KB for one); as many elements as give every thread of the longest pass a line, at most
// 40 KB (four workgroups per compute unit) and leaving at least four workgroups per compute unit.
dErr efs_apply(int P, int Q, const double *rcoord, int nelem, const double *jinv, int D, const double *in, double *out,
               int amode, int imode, hipStream_t st)
{
  const bool tr = amode == dAPPLY_INTERP_TRANSPOSE || amode == dAPPLY_GRAD_TRANSPOSE;
  const int mode = amode == dAPPLY_GRAD ? EFS_GRAD : amode == dAPPLY_GRAD_TRANSPOSE ? EFS_GRAD_T : EFS_INTERP;
  const int a = tr ? Q : P, b = tr ? P : Q, m = std::max(a, b);
  EfsArgs g;
  double t[kEfsTab];
  DOHP_CALL(dohpTensorBasis(P, Q, rcoord, t, t + Q * P, nullptr, nullptr));
  for (int o = 0; o < 2; o++)
    for (int q = 0; q < b; q++)
      for (int i = 0; i < a; i++) g.tab[(o * b + q) * a + i] = t[o * Q * P + (tr ? i * P + q : q * P + i)];
  const auto bytes = [&](int dc) { return sizeof(double) * (efs_r0(mode, a, b, dc) + efs_r1(mode, a, b, dc)); };
  g.b = b;
  g.D = D;
  g.dc = std::min(D, 64);
  while (g.dc > 1 && bytes(g.dc) > 65536) g.dc--;
  const int lines = m * m * g.dc;
  g.epb = std::max(1, std::min({256 / lines, (int)(40960 / bytes(g.dc)), nelem / 1024}));
  g.nelem = nelem;
  g.add = imode == dADD_VALUES;
  g.jinv = jinv;
  g.in = in;
  g.out = out;
  const size_t lds = g.epb * bytes(g.dc);
  if (mode == EFS_INTERP) return efs_dispatch<EFS_INTERP>(a, g, lds, st);
  if (mode == EFS_GRAD) return efs_dispatch<EFS_GRAD>(a, g, lds, st);
  return efs_dispatch<EFS_GRAD_T>(a, g, lds, st);
}

}  // namespace

extern "C" dErr dEFSApplyHexBatched(int P, int Q, const double *rcoord, int nelem, const double *jinv, int D,
                                    const double *in, double *out, int amode, int imode, void *stream)
{
  DOHP_CALL(efs_check(P, Q, nelem, rcoord, jinv, D, in, out, amode, imode));
  if (nelem == 0) return 0;
  hipStream_t st = (hipStream_t)stream;
  DOHP_CALL(efs_apply(P, Q, rcoord, nelem, jinv, D, in, out, amode, imode, st));
  DOHP_HIP(hipStreamSynchronize(st));  // (the results are there when the call returns)
  return 0;
}

extern "C" dErr dEFSApplyHexBatchedNoAlloc(int P, int Q, const double *rcoord, int nelem, const double *jinv, int D,
                                           const double *in, double *out, int amode, int imode, void *stream)
{
  DOHP_CALL(efs_check(P, Q, nelem, rcoord, jinv, D, in, out, amode, imode));
  if (nelem == 0) return 0;
  return efs_apply(P, Q, rcoord, nelem, jinv, D, in, out, amode, imode, (hipStream_t)stream);
}

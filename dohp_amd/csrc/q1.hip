// Embedded-Q1 preconditioning matrix (EllipJacobian, src/fs/tests/ellip.c:474-536) on the GPU,
// and the device CSR matrix it fills.
//
// The element's GLL sub-cells carry Q1 bases; each is integrated on its 2x2x2 Gauss points of the
// SPARSE rule (src/jacobi/quadrature/impls/tensor/tensorquad.c:32-49,73,120-169).  As in the
// reference (src/jacobi/impls/tensor/efstopo.c:660-717):
//   * sub-cell derivatives are +-1 per unit element-reference coordinate (no 1/h factor);
//   * the inverse Jacobian used for sub-cell point (patch, q) is the element-natural one at index
//     patch*8+q, because the iterator passes its element-ordered array
//     (src/fs/interface/fsrulesetit.c:684) to a routine that indexes it in patch order;
//   * u, grad u and the weights are taken at the correct patch points.
// dohpEllipSetQ1Mode(op, 1) assembles the corrected matrix instead (the Q1 finite-element stiffness of
// the GLL sub-mesh): sub-cell derivatives +-1/h and the inverse Jacobian at each patch point.
// The 8x8 sub-cell matrices are added over owned nodes only (Dirichlet rows and columns are dropped,
// src/fs/interface/fsbuild.c:31-34).  One kernel forms the sub-cell matrices of a few layers of elements, one thread per
// sub-cell, and a second adds them up, one thread per row of the 27-point stencil: every sum is taken in a fixed order, so
// the matrix is bitwise reproducible, and every entry is written once.
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <utility>
#include <vector>

#include "common.h"
#include "element.h"

using namespace dohp;


namespace {

constexpr int kMaxP = 10;  // degree limit of the sub-cell kernel (n <= 11)

struct Q1Phys {
  double p, eps2, lambda;
  int has_k, qpow;     // qpow: 4 (p-2)/2 when it is an integer in [-8, 8], else 99 (powe)
  int M1, M2, Ly, Lz;  // block extents: elements, and node lattice (the state is in lattice order)
};

__device__ inline void jac_at(const double (&X)[8][3], double x0, double x1, double x2, double (&J)[3][3])
{
  const double f[3][2] = {{0.5 * (1 - x0), 0.5 * (1 + x0)}, {0.5 * (1 - x1), 0.5 * (1 + x1)},
                          {0.5 * (1 - x2), 0.5 * (1 + x2)}};
  for (int d = 0; d < 3; d++) J[d][0] = J[d][1] = J[d][2] = 0.0;
  for (int t = 0; t < 8; t++) {
    const int a = t >> 2, b = (t >> 1) & 1, c = t & 1;
    const double s0 = (a ? 0.5 : -0.5) * f[1][b] * f[2][c];
    const double s1 = f[0][a] * (b ? 0.5 : -0.5) * f[2][c];
    const double s2 = f[0][a] * f[1][b] * (c ? 0.5 : -0.5);
    for (int d = 0; d < 3; d++) {
      J[d][0] += X[t][d] * s0;
      J[d][1] += X[t][d] * s1;
      J[d][2] += X[t][d] * s2;
    }
  }
}

// Cofactor inverse (dGeomInvert3, include/dohpgeom.h:57-75).
__device__ inline double invert3(const double (&a)[3][3], double (&b)[3][3])
{
  const double b0 = a[1][1] * a[2][2] - a[2][1] * a[1][2];
  const double b3 = -(a[1][0] * a[2][2] - a[2][0] * a[1][2]);
  const double b6 = a[1][0] * a[2][1] - a[2][0] * a[1][1];
  const double det = a[0][0] * b0 + a[0][1] * b3 + a[0][2] * b6;
  const double id = 1.0 / det;
  b[0][0] = id * b0;
  b[0][1] = -id * (a[0][1] * a[2][2] - a[2][1] * a[0][2]);
  b[0][2] = id * (a[0][1] * a[1][2] - a[1][1] * a[0][2]);
  b[1][0] = id * b3;
  b[1][1] = id * (a[0][0] * a[2][2] - a[2][0] * a[0][2]);
  b[1][2] = -id * (a[0][0] * a[1][2] - a[1][0] * a[0][2]);
  b[2][0] = id * b6;
  b[2][1] = -id * (a[0][0] * a[2][1] - a[2][0] * a[0][1]);
  b[2][2] = id * (a[0][0] * a[1][1] - a[1][0] * a[0][1]);
  return det;
}

// position of entry (r, c) of a symmetric 8x8 block in its row-major upper triangle
__host__ __device__ constexpr int sym_index(int r, int c)
{
  return r <= c ? r * 8 - r * (r - 1) / 2 + (c - r) : c * 8 - c * (c - 1) / 2 + (r - c);
}

// row and column of entry t of that triangle
__host__ __device__ constexpr int sym_row(int t)
{
  int r = 0;
  while (t >= sym_index(r, 7) + 1) r++;
  return r;
}
__host__ __device__ constexpr int sym_col(int t) { return sym_row(t) + t - sym_index(sym_row(t), sym_row(t)); }

template <typename F, int... I>
__device__ __forceinline__ void static_for(std::integer_sequence<int, I...>, F f)
{
  (f(std::integral_constant<int, I>()), ...);
}

// exp out of line: its registers do not constrain the allocation of the sub-cell block
__device__ __noinline__ double q1_exp(double x) { return exp(x); }

// LDS (doubles per element: the state contracted along z, then along z and y; the node values share the latter's space)
// and elements per workgroup of the sub-cell kernel: as many as fill two lanes a sub-cell of its 256 threads and fit.  At
// degree 1 with a state 112 instead of 128 leave LDS for a second workgroup on the compute unit: 8 M sub-cells 5.61 ->
// 3.96 ms an assembly (without a state 3.19 with 128, 3.27 with 112).
constexpr int q1_lds_z(int N) { return 2 * N * N * 2 * (N - 1); }
constexpr int q1_lds_y(int N) { return 3 * N * 4 * (N - 1) * (N - 1); }
constexpr int q1_epb(int N, bool has_u)
{
  const int P3 = (N - 1) * (N - 1) * (N - 1), want = P3 >= 216 ? 1 : P3 == 1 ? (has_u ? 112 : 128) : 256 / P3;
  const int fit = 8000 / (q1_lds_z(N) + q1_lds_y(N));
  return want < fit ? want : fit < 1 ? 1 : fit;
}
constexpr int q1_threads(int) { return 256; }

// The value of the other lane of an even-odd pair.
__device__ __forceinline__ double pair_swap(double v)
{
  const long b = __builtin_bit_cast(long, v);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, 0xB1, 0xF, 0xF, true);  // quad_perm [1, 0, 3, 2]
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0xB1, 0xF, 0xF, true);
  return __builtin_bit_cast(double, ((long)hi << 32) | (unsigned)lo);
}

// Trilinear map of an element as polynomials in the reference coordinates: column m of the Jacobian is bilinear in the
// other two coordinates, G[m][0..3] = constant, first, second, product; k is trilinear, Gk[8] (bit 2: x0, 1: x1, 0: x2).
struct Q1Geo {
  double G[3][4][3], Gk[8];
};
__device__ inline void q1_geo(const double *__restrict__ vxyz, const double *__restrict__ kv, const int *ev, int t,
                              Q1Geo &g)
{
  if (t < 9) {  // column m, component d
    const int m = t / 3, d = t % 3, sm = m == 0 ? 4 : m == 1 ? 2 : 1, s1 = m == 0 ? 2 : 4, s2 = m == 2 ? 2 : 1;
    double S[2][2];
    for (int i = 0; i < 2; i++)
      for (int j = 0; j < 2; j++)
        S[i][j] = 0.5 * (vxyz[3 * (long)ev[sm + i * s1 + j * s2] + d] - vxyz[3 * (long)ev[i * s1 + j * s2] + d]);
    g.G[m][0][d] = 0.25 * ((S[0][0] + S[0][1]) + (S[1][0] + S[1][1]));
    g.G[m][1][d] = 0.25 * ((S[1][0] + S[1][1]) - (S[0][0] + S[0][1]));
    g.G[m][2][d] = 0.25 * ((S[0][1] + S[1][1]) - (S[0][0] + S[1][0]));
    g.G[m][3][d] = 0.25 * ((S[1][1] - S[0][1]) - (S[1][0] - S[0][0]));
  } else if (t < 17 && kv) {
    const int c = t - 9;
    double s = 0;
    for (int v = 0; v < 8; v++) s += __builtin_popcount(c & ~v) & 1 ? -kv[ev[v]] : kv[ev[v]];
    g.Gk[c] = 0.125 * s;
  }
}
// Rows J[m] = dX/dx_m of the Jacobian's transpose at (x0, x1, x2); its inverse rows c[m] = grad x_m and determinant.  This
// reciprocal, the powers and the roots below are the operator's (element.h: hardware estimates refined by two Newton steps
// in FP64).  Matrix entries against 80-bit arithmetic, nine cases of p = 1.25 to 2 and degree 1 to 6: 1.8e-16 to 4.9e-16 in
// the Frobenius norm, and the same to 15 % with pow, sqrt and divisions, which take a Newton step at 32^3, p = 6 from 7.67
// to 7.91 ms.
__device__ __forceinline__ double q1_inverse(const Q1Geo &g, double x0, double x1, double x2, double (&c)[3][3])
{
  double J[3][3];
  const double a[3] = {x1, x0, x0}, b[3] = {x2, x2, x1};
#pragma unroll
  for (int m = 0; m < 3; m++)
#pragma unroll
    for (int d = 0; d < 3; d++)
      J[m][d] = (g.G[m][0][d] + a[m] * g.G[m][1][d]) + b[m] * (g.G[m][2][d] + a[m] * g.G[m][3][d]);
  cross3(J[1], J[2], c[0]);
  cross3(J[2], J[0], c[1]);
  cross3(J[0], J[1], c[2]);
  const double det = J[0][0] * c[0][0] + J[0][1] * c[0][1] + J[0][2] * c[0][2], id = recip(det);
#pragma unroll
  for (int m = 0; m < 3; m++)
#pragma unroll
    for (int d = 0; d < 3; d++) c[m][d] *= id;
  return det;
}

// Sub-cell matrices of `nel` elements from element `first` on, two threads per GLL sub-cell, n = N nodes per direction:
// the 36 upper entries K[sym_index] of sub-cell (G0, G1, G2) of the block's sub-cell lattice go to
// KC[entry * ring + ((G0 % slots) * (M1 p) + G1) * (M2 p) + G2], ring = slots * M1 p * M2 p.
//  - The state's values and reference gradient at the (2p)^3 points of an element are formed by contractions along z and
//    y in LDS, shared by its sub-cells, and along x per sub-cell: about 360 multiply-adds per sub-cell at p = 6 where each
//    sub-cell contracted the whole element's state for itself (1,700).
//  - The integrand at a point is g_r . M g_c with the basis gradients g, which are products of one-dimensional factors
//    (-+1 or the two interpolation weights), and one symmetric M, so the sum over the 2 x 2 x 2 points is contracted one
//    direction at a time: 14 sums over the first direction, 31 over the second, then the 36 entries: about 900 operations
//    against 36 x 8 x 8 and the gradients.
//  - A pair of lanes shares a sub-cell, one for each point of the last direction, and exchanges halves of the entries at
//    the end: one thread with the entries and all partial sums live needs 360 registers (one wavefront per SIMD).
//  - Four wavefronts a workgroup in two rounds at 245 registers: two workgroups per compute unit, so one's contractions
//    overlap the other's points (seven wavefronts in one round: 190 us a pass of 663,000 sub-cells against 148).
// Eight coloured launches that added 64 entries per sub-cell into the stencil, and its clearing, took 6.2 ms at 32^3
// elements, p = 6 (7.1 M sub-cells); this and the gather below take 2.3 ms (1.5 and 0.7).
template <int N, bool STATE, bool LAM>
__global__ void __launch_bounds__(q1_threads(N)) __attribute__((amdgpu_waves_per_eu(2))) q1_cell_kernel(
                                                                long first, long nel, int slots,
                                                                const int *__restrict__ everts,
                                                                const double *__restrict__ vxyz,
                                                                const double *__restrict__ kv,
                                                                const double *__restrict__ ustate, int corrected,
                                                                const double *__restrict__ tab, Q1Phys ph,
                                                                const float *__restrict__ cscale,
                                                                double *__restrict__ KC)
{
  constexpr int P = N - 1, NP3 = P * P * P, NQ = 2 * P, NN = N * N, EPB = q1_epb(N, STATE), NT = q1_threads(N);
  constexpr int LZ = q1_lds_z(N), LY = q1_lds_y(N);
  extern __shared__ double lds[];  // [EPB][LZ], [EPB][LY] (with a state)
  __shared__ Q1Geo geo[EPB];
  __shared__ int el[EPB][3];  // the elements' places in the block (their divisions once an element, not a point or sub-cell)
  __shared__ double tb[2 * NQ + P + 2 * NQ * N];  // zq, wq, hsub, B, D
  const double *zq = tb, *wq = tb + NQ, *hsub = tb + 2 * NQ, *Bs = tb + 2 * NQ + P, *Ds = Bs + NQ * N;
  const int tid = threadIdx.x;
  const long e0 = first + (long)blockIdx.x * EPB;
  const int ne = (int)min((long)EPB, first + nel - e0);
  for (int t = tid; t < 2 * NQ + P + 2 * NQ * N; t += NT) tb[t] = tab[t];
  for (int t = tid; t < ne; t += NT) {  // (nelem is an int)
    const int e = (int)e0 + t, col = e / ph.M2, ex = col / ph.M1;
    el[t][0] = ex;
    el[t][1] = col - ex * ph.M1;
    el[t][2] = e - col * ph.M2;
  }
  for (int t = tid; t < ne * 17; t += NT)
    q1_geo(vxyz, ph.has_k ? kv : nullptr, everts + (e0 + t / 17) * 8, t % 17, geo[t / 17]);
  // (a branch on the pointer, not on STATE alone: without it the compiler forms several points' states at once and spills,
  // 4.7 -> 8.0 ms at 40^3 elements, p = 6)
  const bool has_u = STATE && ustate;
  double *Z = lds, *Y = lds + EPB * LZ;
  if (has_u) {
    __syncthreads();
    for (int t = tid; t < ne * NN * N; t += NT) {
      const int l = t / (NN * N), r = t - l * NN * N, a = r / NN, b = (r / N) % N, c = r % N;
      const long I = (long)el[l][0] * P + a;
      const int J = el[l][1] * P + b, K = el[l][2] * P + c;
      Y[l * LY + r] = ustate[(I * ph.Ly + J) * ph.Lz + K];
    }
    __syncthreads();
    for (int t = tid; t < ne * NN * NQ; t += NT) {  // along z: values, derivatives
      const int l = t / (NN * NQ), r = t - l * NN * NQ, ab = r / NQ, q = r - ab * NQ;
      double v = 0, d = 0;
#pragma unroll
      for (int c = 0; c < N; c++) {
        const double u = Y[l * LY + ab * N + c];
        v += Bs[q * N + c] * u;
        d += Ds[q * N + c] * u;
      }
      Z[l * LZ + r] = v;
      Z[l * LZ + NN * NQ + r] = d;
    }
    __syncthreads();
    for (int t = tid; t < ne * N * NQ * NQ; t += NT) {  // along y: (B, B), (D, B), (B, D) in (y, z)
      const int l = t / (N * NQ * NQ), r = t - l * N * NQ * NQ, a = r / (NQ * NQ), q = r - a * NQ * NQ, qj = q / NQ,
                qk = q - qj * NQ;
      const double *z = Z + l * LZ + a * N * NQ + qk;
      double bb = 0, db = 0, bd = 0;
#pragma unroll
      for (int b = 0; b < N; b++) {
        const double v = z[b * NQ], d = z[NN * NQ + b * NQ];
        bb += Bs[qj * N + b] * v;
        db += Ds[qj * N + b] * v;
        bd += Bs[qj * N + b] * d;
      }
      double *y = Y + l * LY + r;
      y[0] = bb;
      y[N * NQ * NQ] = db;
      y[2 * N * NQ * NQ] = bd;
    }
  }
  __syncthreads();
  constexpr double WI[2] = {0.78867513459481287, 0.21132486540518713};  // basis values at a sub-cell's two points
  for (int item = tid; item < 2 * ne * NP3; item += NT) {
    // pairs of lanes walk (a, b, element, c): runs of consecutive sub-cells along z over neighbouring elements
    const int t = item >> 1, kk = item & 1, ab = t / (ne * P), rest = t - ab * ne * P, l = rest / P,
              pc = rest - l * P, pa = ab / P, pb = ab - pa * P;
    const long e = e0 + l;
    const int pidx = ab * P + pc;
    // sub-cell derivative scale per reference direction: 1 (the reference's), 1/h (corrected), times the learned
    // per-sub-cell factors when given
    double sx = corrected ? 1.0 / hsub[pa] : 1.0, sy = corrected ? 1.0 / hsub[pb] : 1.0,
           sz = corrected ? 1.0 / hsub[pc] : 1.0;
    if (cscale) {
      const float *s = cscale + 3 * (e * NP3 + pidx);
      sx *= (double)s[0];
      sy *= (double)s[1];
      sz *= (double)s[2];
    }
    // sums over the first two directions: 00 [r1 c1], 01 [x][y], 02 [x][r1 c1], 11 [r0 c0], 22 [r0 c0][r1 c1],
    // 12 [r0 c0][y], and the Bratu term's [r0 c0][r1 c1]; a pair (0 0), (0 1), (1 1) is indexed 0, 1, 2
    double B00[3] = {0, 0, 0}, B01[2][2] = {{0, 0}, {0, 0}}, B02[2][3] = {{0, 0, 0}, {0, 0, 0}}, B11[3] = {0, 0, 0},
           B22[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, B12[3][2] = {{0, 0}, {0, 0}, {0, 0}},
           BL[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll
    for (int pt = 0; pt < 4; pt++) {
      const int ii = pt & 1, jj = pt >> 1, qi = 2 * pa + ii, qj = 2 * pb + jj, qk = 2 * pc + kk;
      {
        double U = 0, G0 = 0, G1 = 0, G2 = 0;
        if (has_u) {
          const double *y = Y + l * LY + qj * NQ + qk, *bx = Bs + qi * N, *dx = Ds + qi * N;
#pragma unroll
          for (int a = 0; a < N; a++) {
            const double y0 = y[a * NQ * NQ], y1 = y[(N + a) * NQ * NQ], y2 = y[(2 * N + a) * NQ * NQ];
            if (LAM) U += bx[a] * y0;
            G0 += dx[a] * y0;
            G1 += bx[a] * y1;
            G2 += bx[a] * y2;
          }
        }
        int lg = l;  // the element's polynomials are read here, not kept in registers over the loops
        asm volatile("" : "+v"(lg));
        const Q1Geo &g = geo[lg];
        const double x0 = zq[qi], x1 = zq[qj], x2 = zq[qk];
        double Ji[3][3], cj[3][3];
        const double det = q1_inverse(g, x0, x1, x2, Ji);
        const double w = wq[qi] * wq[qj] * wq[qk] * det;
        double kq = 1.0;
        if (ph.has_k)
          kq = ((g.Gk[0] + x2 * g.Gk[1]) + x1 * (g.Gk[2] + x2 * g.Gk[3])) +
               x0 * ((g.Gk[4] + x2 * g.Gk[5]) + x1 * (g.Gk[6] + x2 * g.Gk[7]));
        if (corrected) {  // the inverse Jacobian at the point itself
#pragma unroll
          for (int m = 0; m < 3; m++)
#pragma unroll
            for (int d = 0; d < 3; d++) cj[m][d] = Ji[m][d];
        } else {  // element-natural point pidx*8+q, decoded on the (2p)^3 sparse lattice
          const int qe = pidx * 8 + ii * 4 + jj * 2 + kk;
          q1_inverse(g, zq[qe / (NQ * NQ)], zq[(qe / NQ) % NQ], zq[qe % NQ], cj);
        }
#pragma unroll
        for (int d = 0; d < 3; d++) {
          cj[0][d] *= sx;
          cj[1][d] *= sy;
          cj[2][d] *= sz;
        }
        // EllipPointwiseComputeStore (ellip.c:333-343) with the coefficient factor
        double etaw = w * kq, sm[3] = {0, 0, 0};
        if (has_u) {
          double Du[3];
#pragma unroll
          for (int d = 0; d < 3; d++) Du[d] = G0 * Ji[0][d] + G1 * Ji[1][d] + G2 * Ji[2][d];
          const double espg = ph.eps2 + 0.5 * (Du[0] * Du[0] + Du[1] * Du[1] + Du[2] * Du[2]);
          const double ex = (ph.p - 2) / 2, eta = powe(espg, ex, ph.qpow);
          const double smdc = sqrt_pos(-ex * eta * recip(espg)) * sqrt_pos(kq);
#pragma unroll
          for (int d = 0; d < 3; d++) sm[d] = smdc * Du[d];
          etaw *= eta;
        }
        // EllipPointwiseJacobian (ellip.c:369-377): g_r . M g_c, M_mn = eta w c_m . c_n - w (s . c_m)(s . c_n)
        double tm[3], M[3][3];
#pragma unroll
        for (int m = 0; m < 3; m++) tm[m] = sm[0] * cj[m][0] + sm[1] * cj[m][1] + sm[2] * cj[m][2];
#pragma unroll
        for (int m = 0; m < 3; m++)
#pragma unroll
          for (int n = m; n < 3; n++)
            M[m][n] = etaw * (cj[m][0] * cj[n][0] + cj[m][1] * cj[n][1] + cj[m][2] * cj[n][2]) - w * tm[m] * tm[n];
        const double u[2] = {WI[ii], WI[1 - ii]}, v[2] = {WI[jj], WI[1 - jj]};
        const double f[3] = {u[0] * u[0], u[0] * u[1], u[1] * u[1]}, g2[3] = {v[0] * v[0], v[0] * v[1], v[1] * v[1]};
        double lw = 0;
        if constexpr (LAM) lw = -w * (ph.lambda * q1_exp(U));
#pragma unroll
        for (int c = 0; c < 3; c++) {
          B00[c] += g2[c] * M[0][0];
          B11[c] += f[c] * M[1][1];
#pragma unroll
          for (int d = 0; d < 2; d++) {
            B02[d][c] += (u[d] * g2[c]) * M[0][2];
            B12[c][d] += (f[c] * v[d]) * M[1][2];
          }
#pragma unroll
          for (int d = 0; d < 3; d++) {
            B22[c][d] += (f[c] * g2[d]) * M[2][2];
            if (LAM) BL[c][d] += (f[c] * g2[d]) * lw;
          }
        }
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
          for (int d = 0; d < 2; d++) B01[c][d] += (u[c] * v[d]) * M[0][1];
      }
      __builtin_amdgcn_sched_barrier(0);  // (points one after another: fewer registers)
    }
    const double h[2] = {kk ? WI[1] : WI[0], kk ? WI[0] : WI[1]};
    const auto entry = [&](auto T) {  // this point's share of entry T
      constexpr int r = sym_row(decltype(T)::value), c = sym_col(decltype(T)::value);
      constexpr int r0 = r >> 2, r1 = (r >> 1) & 1, r2 = r & 1, c0 = c >> 2, c1 = (c >> 1) & 1, c2 = c & 1;
      constexpr int x = r0 + c0, y = r1 + c1;  // pair indices
      const auto sg = [](int i, int j) { return i == j ? 1.0 : -1.0; };
      double in = sg(r0, c0) * B00[y] + sg(r1, c1) * B11[x] + (sg(r0, c1) * B01[c0][r1] + sg(r1, c0) * B01[r0][c1]);
      if (LAM) in += BL[x][y];
      return h[r2] * h[c2] * in + sg(r2, c2) * B22[x][y] +
             h[r2] * (sg(r0, c2) * B02[c0][y] + sg(r1, c2) * B12[x][c1]) +
             h[c2] * (sg(r2, c0) * B02[r0][y] + sg(r2, c1) * B12[x][r1]);
    };
    const int ex = el[l][0], ey = el[l][1], ez = el[l][2];
    const long G1 = (long)ph.M1 * P, G2 = (long)ph.M2 * P, ring = slots * G1 * G2;
    double *out = KC + (kk ? 18 * ring : 0) + ((long)((ex * P + pa) % slots) * G1 + ey * P + pb) * G2 + ez * P + pc;
    // lane 0 of the pair stores the first 18 entries, lane 1 the others, each with the other lane's point added
    static_for(std::make_integer_sequence<int, 18>(), [&](auto T) {
      constexpr int i = decltype(T)::value;
      const double k0 = entry(std::integral_constant<int, i>()), k1 = entry(std::integral_constant<int, 18 + i>());
      out[i * ring] = (kk ? k1 : k0) + pair_swap(kk ? k0 : k1);
      __builtin_amdgcn_sched_barrier(0);  // (entries are formed one after another: fewer registers)
    });
  }
}

// Rows of the 27-point stencil st[27][n] on node planes plane0 .. of the lattice, from the sub-cell matrices of the
// sub-cells around them: a thread adds the diagonal and the 13 upper entries of its row (36 values, each sub-cell entry
// read once) and also stores each upper entry as the lower one of that neighbour's row; entries toward nodes that are not
// owned are zero.  I0, J0, K0: first owned node of the lattice; line0: first line of this launch; G: sub-cells per
// direction.
__global__ void __launch_bounds__(256) q1_gather_kernel(int plane0, int line0, int slots, int I0, int J0, int K0, int nx,
                                                        int ny, int nz, int G0, int G1, int G2,
                                                        const double *__restrict__ KC, double *__restrict__ st)
{
  const int K = blockIdx.x * 64 + threadIdx.x, J = line0 + blockIdx.y * 4 + threadIdx.y, I = plane0 + blockIdx.z - I0;
  if (K >= nz || J >= ny || I < 0 || I >= nx) return;
  const long n = (long)nx * ny * nz, i = ((long)I * ny + J) * nz + K, ring = (long)slots * G1 * G2;
  // sub-cell (node - r) for each corner r of it that this node is (clamped: one outside the block adds nothing)
  long cell[8];
  bool has[8];
#pragma unroll
  for (int r = 0; r < 8; r++) {
    const int a = I + I0 - (r >> 2), b = J + J0 - ((r >> 1) & 1), c = K + K0 - (r & 1);
    has[r] = a >= 0 && a < G0 && b >= 0 && b < G1 && c >= 0 && c < G2;
    cell[r] = has[r] ? ((long)(a % slots) * G1 + b) * G2 + c : 0;
  }
#pragma unroll
  for (int s = 0; s < 27; s++) {
    const int di = s / 9 - 1, dj = (s / 3) % 3 - 1, dk = s % 3 - 1;
    const bool in = I + di >= 0 && I + di < nx && J + dj >= 0 && J + dj < ny && K + dk >= 0 && K + dk < nz;
    if (s < 13) {  // written by the lower neighbour's row, or zero
      if (!in) st[s * n + i] = 0.0;
      continue;
    }
    double v = 0.0;
#pragma unroll
    for (int r = 0; r < 8; r++) {
      const int c0 = (r >> 2) + di, c1 = ((r >> 1) & 1) + dj, c2 = (r & 1) + dk;
      if (c0 < 0 || c0 > 1 || c1 < 0 || c1 > 1 || c2 < 0 || c2 > 1) continue;
      const double k = KC[sym_index(r, c0 * 4 + c1 * 2 + c2) * ring + cell[r]];
      v += has[r] ? k : 0.0;
    }
    st[s * n + i] = in ? v : 0.0;
    if (s > 13 && in) st[(26 - s) * n + i + ((long)di * ny + dj) * nz + dk] = v;
  }
}

template <typename T>
__global__ void csr_spmv_kernel(long nrows, const int *__restrict__ rowptr, const int *__restrict__ col,
                                const T *__restrict__ val, const T *__restrict__ x, T *__restrict__ y)
{
  const long r = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nrows) return;
  T s = 0;
  for (int k = rowptr[r]; k < rowptr[r + 1]; k++) s += val[k] * x[col[k]];
  y[r] = s;
}

__global__ void csr_diag_kernel(long nrows, const int *__restrict__ rowptr, const int *__restrict__ col,
                                const double *__restrict__ val, double *__restrict__ d)
{
  const long r = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nrows) return;
  double s = 0;
  for (int k = rowptr[r]; k < rowptr[r + 1]; k++)
    if (col[k] == r) s = val[k];
  d[r] = s;
}

__global__ void copy_f64_kernel(const double *__restrict__ a, double *__restrict__ b, long n)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i];
}

// GLL node a of the element from the sub-interval widths.
__device__ inline double gll_node(const double *hsub, int a)
{
  double z = -1.0;
  for (int i = 0; i < a; i++) z += hsub[i];
  return z;
}

// Features of each GLL sub-cell for the learned derivative scales (kQ1CellInputs values): the log widths of its
// three reference sub-intervals, its centre in element-reference coordinates, the log physical lengths of the three
// reference directions at the centre minus their mean, log det J minus their sum (skew, <= 0), and log k at the
// centre minus the mean log k of the element's vertices (0 without a coefficient).
template <int N>
__global__ void q1_cell_features_kernel(int nelem, const int *__restrict__ everts, const double *__restrict__ vxyz,
                                        const double *__restrict__ kv, const double *__restrict__ tab,
                                        float *__restrict__ X)
{
  constexpr int P = N - 1, NP3 = P * P * P, NQ = 2 * P;
  const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (tid >= (long)nelem * NP3) return;
  const long e = tid / NP3;
  const int pidx = (int)(tid - e * NP3), pa = pidx / (P * P), pb = (pidx / P) % P, pc = pidx % P;
  const double *hsub = tab + 2 * NQ;
  const int *ev = everts + e * 8;
  double Xv[8][3];
  for (int t = 0; t < 8; t++)
    for (int d = 0; d < 3; d++) Xv[t][d] = vxyz[3 * (long)ev[t] + d];
  const double c0 = gll_node(hsub, pa) + 0.5 * hsub[pa], c1 = gll_node(hsub, pb) + 0.5 * hsub[pb],
               c2 = gll_node(hsub, pc) + 0.5 * hsub[pc];
  double J[3][3], Ji[3][3];
  jac_at(Xv, c0, c1, c2, J);
  const double det = invert3(J, Ji);
  double len[3], mean = 0;
  for (int a = 0; a < 3; a++) {
    len[a] = 0.5 * log(J[0][a] * J[0][a] + J[1][a] * J[1][a] + J[2][a] * J[2][a]);
    mean += len[a] / 3;
  }
  double lk = 0;
  if (kv) {
    const double f[3][2] = {{0.5 * (1 - c0), 0.5 * (1 + c0)}, {0.5 * (1 - c1), 0.5 * (1 + c1)},
                            {0.5 * (1 - c2), 0.5 * (1 + c2)}};
    double kc = 0, lmean = 0;
    for (int t = 0; t < 8; t++) {
      kc += kv[ev[t]] * f[0][t >> 2] * f[1][(t >> 1) & 1] * f[2][t & 1];
      lmean += log(kv[ev[t]]) / 8;
    }
    lk = log(kc) - lmean;
  }
  float *x = X + tid * kQ1CellInputs;
  x[0] = (float)log(hsub[pa]);
  x[1] = (float)log(hsub[pb]);
  x[2] = (float)log(hsub[pc]);
  x[3] = (float)c0;
  x[4] = (float)c1;
  x[5] = (float)c2;
  for (int a = 0; a < 3; a++) x[6 + a] = (float)(len[a] - mean);
  x[9] = (float)(log(det) - 3 * mean);
  x[10] = (float)lk;
}

// Gradient of the bilinear form w^T K(sigma) z of the linear operator's embedded-Q1 matrix (ellip p = 2, lambda = 0)
// in the sub-cell derivative scales: the sub-cell block is K = sum_q W_q D_q D_q^T with D_q = sum_a sigma_a U_qa
// (U_qa: the +-1 sub-cell derivative along reference direction a times the inverse Jacobian row a, as assembled), so
// d(w^T K z)/d sigma_a = sum_q W_q [(U_qa^T w) . (D_q^T z) + (D_q^T w) . (U_qa^T z)].  g[cell][a] += coef times it.
// w and z are vectors over the owned nodes (zero on Dirichlet nodes, whose rows and columns are dropped).
template <int N>
__global__ void __launch_bounds__(128) q1_scale_grad_kernel(int nelem, const int *__restrict__ enodes,
                                                           const int *__restrict__ everts,
                                                           const double *__restrict__ vxyz,
                                                           const double *__restrict__ kv, long nowned, int corrected,
                                                           const double *__restrict__ tab,
                                                           const float *__restrict__ cscale,
                                                           const double *__restrict__ wv, const double *__restrict__ zv,
                                                           double coef, float *__restrict__ g)
{
  constexpr int P = N - 1, NP3 = P * P * P, NQ = 2 * P;
  const double *zq = tab, *wq = tab + NQ, *hsub = tab + 2 * NQ;
  const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (tid >= (long)nelem * NP3) return;
  const long e = tid / NP3;
  const int pidx = (int)(tid - e * NP3), pa = pidx / (P * P), pb = (pidx / P) % P, pc = pidx % P;
  const int *ev = everts + e * 8;
  const int *en = &enodes[e * N * N * N];
  double w8[8], z8[8];
  for (int b = 0; b < 8; b++) {
    const int gi = en[((pa + (b >> 2)) * N + pb + ((b >> 1) & 1)) * N + pc + (b & 1)];
    w8[b] = gi < nowned ? wv[gi] : 0.0;
    z8[b] = gi < nowned ? zv[gi] : 0.0;
  }
  const double base[3] = {corrected ? 1.0 / hsub[pa] : 1.0, corrected ? 1.0 / hsub[pb] : 1.0,
                          corrected ? 1.0 / hsub[pc] : 1.0};
  double sig[3] = {1.0, 1.0, 1.0};
  if (cscale)
    for (int a = 0; a < 3; a++) sig[a] = (double)cscale[3 * tid + a];
  double Xv[8][3];
  for (int t = 0; t < 8; t++)
    for (int d = 0; d < 3; d++) Xv[t][d] = vxyz[3 * (long)ev[t] + d];
  const double i1[2][2] = {{0.78867513459481287, 0.21132486540518713}, {0.21132486540518713, 0.78867513459481287}};
  const double d1[2][2] = {{-1., 1.}, {-1., 1.}};
  double acc[3] = {0, 0, 0};
  for (int q = 0; q < 8; q++) {
    const int ii = q >> 2, jj = (q >> 1) & 1, kk = q & 1;
    const int qi = 2 * pa + ii, qj = 2 * pb + jj, qk = 2 * pc + kk;
    double J[3][3], Ji[3][3], cj[3][3];
    jac_at(Xv, zq[qi], zq[qj], zq[qk], J);
    const double det = invert3(J, Ji);
    double kq = 1.0;
    if (kv) {
      const double f0[2] = {0.5 * (1 - zq[qi]), 0.5 * (1 + zq[qi])};
      const double f1[2] = {0.5 * (1 - zq[qj]), 0.5 * (1 + zq[qj])};
      const double f2[2] = {0.5 * (1 - zq[qk]), 0.5 * (1 + zq[qk])};
      kq = 0;
      for (int t = 0; t < 8; t++) kq += kv[ev[t]] * f0[t >> 2] * f1[(t >> 1) & 1] * f2[t & 1];
    }
    if (corrected) {
      for (int r = 0; r < 3; r++)
        for (int d = 0; d < 3; d++) cj[r][d] = Ji[r][d];
    } else {  // element-natural point pidx*8+q, as the assembly
      const int qe = pidx * 8 + q;
      const int ei = qe / (NQ * NQ), ej = (qe / NQ) % NQ, ek = qe % NQ;
      double J2[3][3];
      jac_at(Xv, zq[ei], zq[ej], zq[ek], J2);
      invert3(J2, cj);
    }
    const double W = wq[qi] * wq[qj] * wq[qk] * det * kq;
    // reference derivative sums along each direction: sum_b dd_a[b] v_b
    double rw[3] = {0, 0, 0}, rz[3] = {0, 0, 0};
    for (int b = 0; b < 8; b++) {
      const int a0 = b >> 2, a1 = (b >> 1) & 1, a2 = b & 1;
      const double dd[3] = {d1[ii][a0] * i1[jj][a1] * i1[kk][a2], i1[ii][a0] * d1[jj][a1] * i1[kk][a2],
                            i1[ii][a0] * i1[jj][a1] * d1[kk][a2]};
      for (int a = 0; a < 3; a++) {
        rw[a] += dd[a] * w8[b];
        rz[a] += dd[a] * z8[b];
      }
    }
    double Uw[3][3], Uz[3][3], Dw[3] = {0, 0, 0}, Dz[3] = {0, 0, 0};
    for (int a = 0; a < 3; a++)
      for (int d = 0; d < 3; d++) {
        Uw[a][d] = base[a] * rw[a] * cj[a][d];
        Uz[a][d] = base[a] * rz[a] * cj[a][d];
        Dw[d] += sig[a] * Uw[a][d];
        Dz[d] += sig[a] * Uz[a][d];
      }
    for (int a = 0; a < 3; a++)
      acc[a] += W * (Uw[a][0] * Dz[0] + Uw[a][1] * Dz[1] + Uw[a][2] * Dz[2] + Dw[0] * Uz[a][0] + Dw[1] * Uz[a][1] +
                     Dw[2] * Uz[a][2]);
  }
  for (int a = 0; a < 3; a++) g[3 * tid + a] += (float)(coef * acc[a]);
}

}  // namespace

// Accessors the operator file uses (defined there).
extern "C" dErr dohpEllipGetQ1Context_Private(dohpEllip op, dohpFS *fs, dohpEllipParam *prm, const double **kvert,
                                              const double **state, int *q1mode);
const float *dohpEllipGetQ1CellScales_Private(dohpEllip op);

// CSR pattern of the 27-point stencil on a box of rows in lexicographic order, built on the device: row (i, j, k)
// couples to its box neighbours in increasing index, and its offset has a closed form (the count of entries of the
// rows before it, a product of per-direction counts 1 + [i > 0] + [i < n - 1]).
__device__ __forceinline__ long box_prefix(int i, int n) { return i + (i > 0 ? i - 1 : 0) + (i < n - 1 ? i : n - 1); }

__global__ void box_pattern_kernel(int nx, int ny, int nz, int *__restrict__ rowptr, int *__restrict__ col)
{
  const long n = (long)nx * ny * nz;
  const long r = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  const int k = (int)(r % nz), j = (int)((r / nz) % ny), i = (int)(r / ((long)ny * nz));
  const long cj = 1 + (j > 0) + (j < ny - 1), ck = 1 + (k > 0) + (k < nz - 1), ci = 1 + (i > 0) + (i < nx - 1);
  const long Sy = 3L * ny - 2, Sz = 3L * nz - 2;
  const long off = box_prefix(i, nx) * Sy * Sz + ci * box_prefix(j, ny) * Sz + ci * cj * box_prefix(k, nz);
  rowptr[r] = (int)off;
  if (r == n - 1) rowptr[n] = (int)((3L * nx - 2) * Sy * Sz);
  long m = off;
  for (int di = -1; di <= 1; di++)
    for (int dj = -1; dj <= 1; dj++)
      for (int dk = -1; dk <= 1; dk++) {
        const int a = i + di, b = j + dj, c = k + dk;
        if (a < 0 || b < 0 || c < 0 || a >= nx || b >= ny || c >= nz) continue;
        col[m++] = (int)(((long)a * ny + b) * nz + c);
      }
}

static dErr build_pattern_box(dohpFS fs, _p_dohpMat *A, bool *done)
{
  const long L0 = (long)fs->p * fs->M[0] + 1, L1 = (long)fs->p * fs->M[1] + 1, L2 = (long)fs->p * fs->M[2] + 1;
  const int m = fs->dirichlet_mask;
  const long nx = L0 - ((m & 1) ? 2 : 0), ny = L1 - ((m & 1) ? 2 : 0), nz = L2 - ((m & 2) ? 1 : 0) - ((m & 4) ? 1 : 0);
  *done = false;
  if (nx <= 0 || ny <= 0 || nz <= 0 || nx * ny * nz != fs->nowned) return 0;
  const long nnz = (3 * nx - 2) * (3 * ny - 2) * (3 * nz - 2);
  if (nnz > 2147483647L) return 0;  // 32-bit offsets
  A->nrows = fs->nowned;
  A->nnz = nnz;
  DOHP_CALL(A->rowptr.alloc(A->nrows + 1));
  DOHP_CALL(A->col.alloc(nnz));
  DOHP_CALL(A->val.alloc(nnz));
  DOHP_CALL(A->val32.alloc(nnz));
  hipLaunchKernelGGL(box_pattern_kernel, dim3((unsigned)((A->nrows + 255) / 256)), dim3(256), 0, nullptr, (int)nx,
                     (int)ny, (int)nz, A->rowptr.ptr, A->col.ptr);
  DOHP_HIP(hipGetLastError());
  DOHP_HIP(hipDeviceSynchronize());
  *done = true;
  return 0;
}

// Pattern of the Q1 matrix on the GLL sub-cell lattice: row of every owned node, columns of the
// owned nodes among its 27 lattice neighbours (dFSCreateMatrix preallocates 27 per row,
// src/fs/interface/fs.c:770-813).
static dErr build_pattern(dohpFS fs, _p_dohpMat *A)
{
  bool done = false;
  DOHP_CALL(build_pattern_box(fs, A, &done));
  if (done) return 0;
  const long L0 = (long)fs->p * fs->M[0] + 1, L1 = (long)fs->p * fs->M[1] + 1, L2 = (long)fs->p * fs->M[2] + 1;
  // invert the closure numbering: lattice index of each closure node
  std::vector<long> c2l(fs->nclosure);
  const int n = fs->n, n3 = n * n * n;
  for (int e = 0; e < fs->nelem; e++) {
    const long e0 = e / ((long)fs->M[1] * fs->M[2]), e1 = (e / fs->M[2]) % fs->M[1], e2 = e % fs->M[2];
    for (int a = 0; a < n; a++)
      for (int b = 0; b < n; b++)
        for (int c = 0; c < n; c++)
          c2l[fs->elem_nodes[(long)e * n3 + (a * n + b) * n + c]] =
              ((e0 * fs->p + a) * L1 + e1 * fs->p + b) * L2 + e2 * fs->p + c;
  }
  std::vector<int> l2c(L0 * L1 * L2);
  for (long c = 0; c < fs->nclosure; c++) l2c[c2l[c]] = (int)c;
  A->nrows = fs->nowned;
  A->h_rowptr.assign(fs->nowned + 1, 0);
  std::vector<int> cols;
  cols.reserve(fs->nowned * 27);
  for (long r = 0; r < fs->nowned; r++) {
    const long l = c2l[r], I = l / (L1 * L2), J = (l / L2) % L1, K = l % L2;
    int buf[27], m = 0;
    for (int di = -1; di <= 1; di++)
      for (int dj = -1; dj <= 1; dj++)
        for (int dk = -1; dk <= 1; dk++) {
          const long a = I + di, b = J + dj, c = K + dk;
          if (a < 0 || b < 0 || c < 0 || a >= L0 || b >= L1 || c >= L2) continue;
          const int cc = l2c[(a * L1 + b) * L2 + c];
          if (cc < fs->nowned) buf[m++] = cc;
        }
    std::sort(buf, buf + m);
    cols.insert(cols.end(), buf, buf + m);
    A->h_rowptr[r + 1] = (int)cols.size();
  }
  A->nnz = (long)cols.size();
  DOHP_CALL(A->rowptr.upload(A->h_rowptr.data(), A->h_rowptr.size()));
  DOHP_CALL(A->col.upload(cols.data(), cols.size()));
  DOHP_CALL(A->val.alloc(A->nnz));
  DOHP_CALL(A->val32.alloc(A->nnz));
  return 0;
}

namespace {

// Ring of sub-cell matrices of an assembly: as many layers of elements per pass as keep it in the 256 MB cache, so that
// the gather does not read them from HBM (32^3 elements, p = 6: 96 MB 2.61 ms, 192 MB 2.31, 512 MB 2.64, one pass 3.02).
constexpr size_t kQ1RingBytes = (size_t)192 << 20;
constexpr int kQ1MaxGrid = 65535;  // blocks of a launch along y and z

template <typename F>
dErr q1_dispatch(int n, F f)
{
  switch (n) {
  case 2: f(std::integral_constant<int, 2>()); break;
  case 3: f(std::integral_constant<int, 3>()); break;
  case 4: f(std::integral_constant<int, 4>()); break;
  case 5: f(std::integral_constant<int, 5>()); break;
  case 6: f(std::integral_constant<int, 6>()); break;
  case 7: f(std::integral_constant<int, 7>()); break;
  case 8: f(std::integral_constant<int, 8>()); break;
  case 9: f(std::integral_constant<int, 9>()); break;
  case 10: f(std::integral_constant<int, 10>()); break;
  case 11: f(std::integral_constant<int, 11>()); break;
  default: set_error("embedded-Q1 assembly supports degree 1..10"); return dohpERR_ARG;
  }
  DOHP_HIP(hipGetLastError());
  return 0;
}

// The passes of an assembly: sub-cell matrices of lx layers of elements into the ring of `slots` layers of sub-cells, and
// the node planes that they complete into the matrix's stencil.
dErr q1_passes(dohpFS fs, const dohpEllipParam &prm, const Q1Phys &ph, _p_dohpMat *A, const double *kvert,
               const double *state, int q1mode, const float *cscale, int lx, int slots, double *ring, hipStream_t st)
{
  const int G[3] = {fs->M[0] * fs->p, fs->M[1] * fs->p, fs->M[2] * fs->p};
  const int m = fs->dirichlet_mask, I0 = m & 1, K0 = (m >> 2) & 1;
  for (int x0 = 0; x0 < fs->M[0]; x0 += lx) {
    const int x1 = std::min(fs->M[0], x0 + lx);
    const long first = (long)x0 * fs->M[1] * fs->M[2], nel = (long)(x1 - x0) * fs->M[1] * fs->M[2];
    DOHP_CALL(q1_dispatch(fs->n, [&](auto NN) {
      constexpr int N = decltype(NN)::value;
      const auto go = [&](auto kernel, bool with_state) {
        const int epb = q1_epb(N, with_state);
        const size_t lds = with_state ? sizeof(double) * epb * (q1_lds_z(N) + q1_lds_y(N)) : 0;
        if (lds > 65536)
          (void)hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        hipLaunchKernelGGL(kernel, dim3((unsigned)((nel + epb - 1) / epb)), dim3(q1_threads(N)), lds, st, first, nel, slots,
                           fs->d_elem_verts.ptr, fs->d_vcoords.ptr, kvert, state, q1mode, A->q1tab.ptr, ph, cscale, ring);
      };
      // the state enters a sub-cell only through eta(grad u) and s (p != 2) and lambda e^u: for the linear operator
      // (p = 2, lambda = 0) eta = 1 and s = 0 whatever the state, and its interpolation is left out
      if (prm.lambda != 0.0)
        go(q1_cell_kernel<N, true, true>, true);
      else if (prm.p != 2.0)
        go(q1_cell_kernel<N, true, false>, true);
      else
        go(q1_cell_kernel<N, false, false>, false);
    }));
    // node planes whose sub-cells are all there: up to the pass's last layer of sub-cells, and the block's last plane
    const int p0 = x0 * fs->p, p1 = x1 == fs->M[0] ? G[0] + 1 : x1 * fs->p;
    for (int line0 = 0; line0 < A->box[1]; line0 += 4 * kQ1MaxGrid) {
      const dim3 grid((A->box[2] + 63) / 64, std::min(kQ1MaxGrid, (A->box[1] - line0 + 3) / 4), p1 - p0);
      hipLaunchKernelGGL(q1_gather_kernel, grid, dim3(64, 4), 0, st, p0, line0, slots, I0, I0, K0, A->box[0], A->box[1],
                         A->box[2], G[0], G[1], G[2], ring, A->st64.ptr);
    }
    DOHP_HIP(hipGetLastError());
  }
  return 0;
}

}  // namespace

extern "C" dErr dohpEllipAssembleQ1(dohpEllip op, const double *u, dohpMat *out, void *stream)
{
  DOHP_CHECK(op && out, dohpERR_ARG, "null argument");
  dohpFS fs;
  dohpEllipParam prm;
  const double *kvert, *state;
  int q1mode = 0;
  DOHP_CALL(dohpEllipGetQ1Context_Private(op, &fs, &prm, &kvert, &state, &q1mode));
  DOHP_CHECK(fs->p <= kMaxP, dohpERR_ARG, "Q1 assembly supports degree <= 10");
  DOHP_CHECK(fs->is_block(), dohpERR_ARG, "the embedded-Q1 matrix needs a block space (dFSCreateBlock)");
  const float *cscale = dohpEllipGetQ1CellScales_Private(op);
  hipStream_t st = (hipStream_t)stream;
  // Not in a capture: a replay would change the stencil behind the flags that say which of the matrix's other forms, and of
  // its hierarchy, still have to follow.
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  DOHP_HIP(hipStreamIsCapturing(st, &cap));
  DOHP_CHECK(cap == hipStreamCaptureStatusNone, dohpERR_HIP, "the embedded-Q1 assembly cannot be captured in a graph");
  if (u) {
    DOHP_CALL(dohpEllipFunctionState_Private(op, u, st));
    DOHP_HIP(hipStreamSynchronize(st));  // (u has been read when the call returns; its kernels go on)
  }
  _p_dohpMat *A = *out;
  if (A) A->mg_stale = true;  // new values: the cached hierarchy is recomputed, in its own buffers, when next used
  SharedScratch &ring = *dohpEllipQ1Ring_Private(op);
  const auto with_room = [&](auto alloc) -> dErr {  // (the ring of an earlier assembly makes room for a matrix)
    const dErr err = alloc();
    if (err != dohpERR_OOM || !ring.buf.ptr) return err;
    ring.buf.release();
    return alloc();
  };
  if (!A) {
    A = new _p_dohpMat;
    dErr err = with_room([&]() { return build_pattern(fs, A); });
    if (err) {
      delete A;
      return err;
    }
    *out = A;
  }
  A->corrected = q1mode;
  A->scaled = cscale != nullptr;
  if (A->q1tab_degree != fs->p) {  // 1-D tables of the degree: zq, wq (2p each), hsub (p), Bs, Ds (2p x n each)
    double zg[kMaxN], wg[kMaxN], zq[2 * kMaxP], wq[2 * kMaxP];
    gauss_lobatto(fs->n, zg, wg);
    int nq;
    DOHP_CALL(dohpTensorRule(dQUADRATURE_METHOD_SPARSE, dGAUSS_LEGENDRE, 2 * fs->p, &nq, zq, wq));
    std::vector<double> Bs(nq * fs->n), Ds(nq * fs->n), tab(zq, zq + nq);
    DOHP_CALL(dohpTensorBasis(fs->n, nq, zq, Bs.data(), Ds.data(), nullptr, nullptr));
    tab.insert(tab.end(), wq, wq + nq);
    for (int i = 0; i < fs->p; i++) tab.push_back(zg[i + 1] - zg[i]);
    tab.insert(tab.end(), Bs.begin(), Bs.end());
    tab.insert(tab.end(), Ds.begin(), Ds.end());
    A->q1tab_degree = 0;
    DOHP_CALL(A->q1tab.upload(tab.data(), tab.size()));
    A->q1tab_degree = fs->p;
  }
  const double q4 = 2.0 * (prm.p - 2.0);
  Q1Phys ph{prm.p, prm.epsilon * prm.epsilon, prm.lambda, kvert != nullptr,
            q4 == std::floor(q4) && std::fabs(q4) <= 8.0 ? (int)q4 : 99, fs->M[1], fs->M[2],
            fs->p * fs->M[1] + 1, fs->p * fs->M[2] + 1};
  // On a block space the owned nodes form a box and the matrix is a 27-point stencil (without owned nodes there is
  // nothing to assemble); the CSR values are read back from it on demand.
  bool box = false;
  DOHP_CALL(with_room([&]() { return dohpMatPrepareStencil_Private(A, fs, &box, st); }));
  A->csr_stale = box;
  if (!box) return 0;
  // Layers of elements per pass: the sub-cell matrices of a pass (288 bytes per sub-cell) and of the layer of sub-cells
  // before it are kept in a ring of layers.
  const int G[3] = {fs->M[0] * fs->p, fs->M[1] * fs->p, fs->M[2] * fs->p};
  const size_t layer = (size_t)G[1] * G[2] * 36;
  // (and as many as leave the gather's planes and blocks of lines within a grid's 65536)
  int lx = (int)std::min<size_t>({(size_t)fs->M[0], (size_t)(kQ1MaxGrid / fs->p - 1),
                                  std::max<size_t>(1, kQ1RingBytes / (8 * layer * fs->p))});
  int slots = 0;
  for (;; lx = (lx + 1) / 2) {
    slots = lx * fs->p + 1;
    if (ring.buf.n >= slots * layer) break;
    const dErr err = ring.buf.alloc(slots * layer);
    if (!err) break;
    if (err != dohpERR_OOM || lx == 1) return err;
  }
  DOHP_CALL(ring.begin(st));
  const dErr err = q1_passes(fs, prm, ph, A, kvert, state, q1mode, cscale, lx, slots, ring.buf.ptr, st);
  DOHP_CALL(ring.end(st));  // (also after an error: what was launched still uses the ring)
  return err;
}

extern "C" dErr dohpMatGetSizes(dohpMat A, long *nrows, long *nnz)
{
  DOHP_CHECK(A, dohpERR_ARG, "null matrix");
  if (nrows) *nrows = A->nrows;
  if (nnz) *nnz = A->nnz;
  return 0;
}

dErr dohpMatSyncCSR_Private(_p_dohpMat *A, hipStream_t st)
{
  if (!A->csr_stale) return 0;
  DOHP_CALL(dohpMatStencilToCSR_Private(A, st));
  A->csr_stale = false;
  return 0;
}

extern "C" dErr dohpMatGetCSR(dohpMat A, int *rowptr, int *col, double *val)
{
  DOHP_CHECK(A, dohpERR_ARG, "null matrix");
  DOHP_HIP(hipDeviceSynchronize());
  DOHP_CALL(dohpMatSyncCSR_Private(A, nullptr));
  DOHP_HIP(hipDeviceSynchronize());
  if (rowptr) DOHP_HIP(hipMemcpy(rowptr, A->rowptr.ptr, sizeof(int) * (A->nrows + 1), hipMemcpyDeviceToHost));
  if (col) DOHP_HIP(hipMemcpy(col, A->col.ptr, sizeof(int) * A->nnz, hipMemcpyDeviceToHost));
  if (val) DOHP_HIP(hipMemcpy(val, A->val.ptr, sizeof(double) * A->nnz, hipMemcpyDeviceToHost));
  return 0;
}

extern "C" dErr dohpMatMult(dohpMat A, const double *x, double *y, void *stream)
{
  DOHP_CHECK(A && x && y, dohpERR_ARG, "null argument");
  if (A->st64.ptr) return dohpStencilMult_Private(A, x, y, (hipStream_t)stream);
  hipLaunchKernelGGL(csr_spmv_kernel<double>, dim3((A->nrows + 255) / 256), dim3(256), 0, (hipStream_t)stream, A->nrows,
                     A->rowptr.ptr, A->col.ptr, A->val.ptr, x, y);
  DOHP_HIP(hipGetLastError());
  return 0;
}

extern "C" dErr dohpMatMultF32(dohpMat A, const float *x, float *y, void *stream)
{
  DOHP_CHECK(A && x && y, dohpERR_ARG, "null argument");
  if (A->st32.ptr) {
    DOHP_CALL(dohpMatSyncCSR_Private(A, (hipStream_t)stream));
    return dohpStencilMultF32_Private(A, x, y, (hipStream_t)stream);
  }
  hipLaunchKernelGGL(csr_spmv_kernel<float>, dim3((A->nrows + 255) / 256), dim3(256), 0, (hipStream_t)stream, A->nrows,
                     A->rowptr.ptr, A->col.ptr, A->val32.ptr, x, y);
  DOHP_HIP(hipGetLastError());
  return 0;
}

extern "C" dErr dohpMatGetDiagonal(dohpMat A, double *d, void *stream)
{
  DOHP_CHECK(A && d, dohpERR_ARG, "null argument");
  if (A->st64.ptr)  // the stencil form holds the diagonal as its middle plane (the CSR values are read from it)
    hipLaunchKernelGGL(copy_f64_kernel, dim3((A->nrows + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                       A->st64.ptr + 13 * A->nrows, d, A->nrows);
  else
    hipLaunchKernelGGL(csr_diag_kernel, dim3((A->nrows + 255) / 256), dim3(256), 0, (hipStream_t)stream, A->nrows,
                       A->rowptr.ptr, A->col.ptr, A->val.ptr, d);
  DOHP_HIP(hipGetLastError());
  return 0;
}

extern "C" dErr dohpMatDestroy(dohpMat *A)
{
  if (A && *A) {
    delete *A;
    *A = nullptr;
  }
  return 0;
}

// ------------------------------------------------------ learned sub-cell scales of the embedded-Q1 matrix

extern "C" dErr dohpQ1CellCount(dohpEllip op, long *ncell)
{
  DOHP_CHECK(op && ncell, dohpERR_ARG, "null argument");
  dohpFS fs;
  dohpEllipParam prm;
  const double *kv, *stt;
  DOHP_CALL(dohpEllipGetQ1Context_Private(op, &fs, &prm, &kv, &stt, nullptr));
  *ncell = (long)fs->nelem * fs->p * fs->p * fs->p;
  return 0;
}

extern "C" dErr dohpQ1CellFeatures(dohpEllip op, dohpMat q1, float *X, void *stream)
{
  DOHP_CHECK(op && q1 && X, dohpERR_ARG, "null argument");
  DOHP_CHECK(q1->q1tab.ptr, dohpERR_ARG, "the embedded-Q1 matrix has not been assembled");
  dohpFS fs;
  dohpEllipParam prm;
  const double *kv, *stt;
  DOHP_CALL(dohpEllipGetQ1Context_Private(op, &fs, &prm, &kv, &stt, nullptr));
  const long nt = (long)fs->nelem * fs->p * fs->p * fs->p;
  const dim3 grid((unsigned)((nt + 127) / 128));
  hipStream_t st = (hipStream_t)stream;
  return q1_dispatch(fs->n, [&](auto NN) {
    hipLaunchKernelGGL(q1_cell_features_kernel<decltype(NN)::value>, grid, dim3(128), 0, st, fs->nelem,
                       fs->d_elem_verts.ptr, fs->d_vcoords.ptr, kv, q1->q1tab.ptr, X);
  });
}

extern "C" dErr dohpQ1CellScaleGradient(dohpEllip op, dohpMat q1, const double *w, const double *z, double coef,
                                        float *g, void *stream)
{
  DOHP_CHECK(op && q1 && w && z && g, dohpERR_ARG, "null argument");
  DOHP_CHECK(q1->q1tab.ptr, dohpERR_ARG, "the embedded-Q1 matrix has not been assembled");
  dohpFS fs;
  dohpEllipParam prm;
  const double *kv, *stt;
  DOHP_CALL(dohpEllipGetQ1Context_Private(op, &fs, &prm, &kv, &stt, nullptr));
  DOHP_CHECK(prm.p == 2.0 && prm.lambda == 0.0, dohpERR_ARG,
             "the sub-cell scale gradient is for the linear operator (ellip p = 2, lambda = 0)");
  const float *cscale = dohpEllipGetQ1CellScales_Private(op);
  const long nt = (long)fs->nelem * fs->p * fs->p * fs->p;
  const dim3 grid((unsigned)((nt + 127) / 128));
  hipStream_t st = (hipStream_t)stream;
  return q1_dispatch(fs->n, [&](auto NN) {
    hipLaunchKernelGGL(q1_scale_grad_kernel<decltype(NN)::value>, grid, dim3(128), 0, st, fs->nelem,
                       fs->d_elem_nodes.ptr, fs->d_elem_verts.ptr, fs->d_vcoords.ptr, kv, fs->nowned, q1->corrected,
                       q1->q1tab.ptr, cscale, w, z, coef, g);
  });
}

// Geometric multigrid on the embedded-Q1 matrix of a block space: the multilevel solve that
// ellip's driver obtains from PETSc's preconditioners applied to the Q1 matrix
// (src/fs/tests/ellip.c:594-652,701-747).
//
// The owned nodes of a block space form a box of the GLL node lattice and the Q1 matrix is a
// 27-point stencil on it.  Levels coarsen every box dimension d to floor(d/2): coarse node c
// sits on fine node 2c+1; fine node 2c interpolates its neighbours c-1 and c with weight 1/2
// (missing neighbours are Dirichlet zeros).  Coarse operators are Galerkin products P^T A P
// (again 27-point), smoothing is a Jacobi-preconditioned Chebyshev polynomial on
// [lo * lmax, hi * lmax] of D^{-1} A, the coarsest level (at most a few hundred nodes) is solved
// with its explicit inverse.  The V-cycle works on symmetric half stencils (see
// half_row).  Pre- and post-smoothers are the same polynomial, so the V-cycle is
// a symmetric operator and serves as a CG preconditioner.
#include <algorithm>
#include <cmath>
#include <vector>

#include "common.h"

using namespace dohp;

namespace {

struct Box {
  int nx, ny, nz;
  __host__ __device__ long n() const { return (long)nx * ny * nz; }
};

// Box kernels launch a 3-D grid: x covers the last (contiguous) index K in chunks of 64, y the
// middle index J in chunks of 4 (threadIdx.y), z the first index I; no index division.
constexpr int kBX = 64, kBY = 4;
inline dim3 box_grid(const Box &b)
{
  return dim3((unsigned)((b.nz + kBX - 1) / kBX), (unsigned)((b.ny + kBY - 1) / kBY), (unsigned)b.nx);
}
inline dim3 box_block() { return dim3(kBX, kBY); }
__device__ __forceinline__ bool box_index(const Box &b, int &I, int &J, int &K, long &r)
{
  K = blockIdx.x * kBX + threadIdx.x;
  J = blockIdx.y * kBY + threadIdx.y;
  I = blockIdx.z;
  if (K >= b.nz || J >= b.ny) return false;
  r = ((long)I * b.ny + J) * b.nz + K;
  return true;
}

__device__ __forceinline__ bool inside(const Box &b, int I, int J, int K)
{
  return I >= 0 && I < b.nx && J >= 0 && J < b.ny && K >= 0 && K < b.nz;
}

__device__ __forceinline__ void unrank(const Box &b, long r, int &I, int &J, int &K)
{
  const long yz = (long)b.ny * b.nz;
  I = (int)(r / yz);
  const long rem = r - (long)I * yz;
  J = (int)(rem / b.nz);
  K = (int)(rem - (long)J * b.nz);
}

// stencil -> CSR values (and the FP32 copies of both).  A workgroup takes 256 consecutive rows: it
// converts their stencil planes to FP32 (one row per thread) and walks their CSR entries, which are
// contiguous, one entry per thread (coalesced), finding each entry's row by binary search in the
// rows' offsets staged in LDS.
__global__ void __launch_bounds__(256) stencil_to_csr_kernel(Box b, const int *__restrict__ rowptr,
                                                             const int *__restrict__ col,
                                                             const double *__restrict__ st, double *__restrict__ val,
                                                             float *__restrict__ val32, float *__restrict__ st32)
{
  __shared__ int rp[257];
  const long n = b.n();
  const long r0 = (long)blockIdx.x * 256;
  const int nr = (int)min(256L, n - r0), t = threadIdx.x;
  if (t < nr) {
    const long r = r0 + t;
    for (int s = 0; s < 27; s++) st32[s * n + r] = (float)st[s * n + r];
  }
  for (int j = t; j <= nr; j += 256) rp[j] = rowptr[r0 + j];
  __syncthreads();
  const int kb = rp[0], ke = rp[nr];
  for (int k = kb + t; k < ke; k += 256) {
    int lo = 0, hi = nr - 1;  // last row whose entries start at or before k
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (rp[mid] <= k)
        lo = mid;
      else
        hi = mid - 1;
    }
    const long r = r0 + lo;
    int I, J, K, I2, J2, K2;
    unrank(b, r, I, J, K);
    unrank(b, col[k], I2, J2, K2);
    const int di = I2 - I, dj = J2 - J, dk = K2 - K;
    double v = 0.0;
    if (di >= -1 && di <= 1 && dj >= -1 && dj <= 1 && dk >= -1 && dk <= 1)
      v = st[((di + 1) * 9 + (dj + 1) * 3 + (dk + 1)) * n + r];
    val[k] = v;
    val32[k] = (float)v;
  }
}

// y = A x.  Entries are summed in increasing column order, as the CSR product does.
template <typename T>
__global__ void stencil_mult_kernel(Box b, const T *__restrict__ A, const T *__restrict__ x, T *__restrict__ y)
{
  const long n = b.n();
  int I, J, K;
  long r;
  if (!box_index(b, I, J, K, r)) return;
  const long sy = b.nz, sx = (long)b.ny * b.nz;
  // every load is issued unconditionally (a neighbour outside the box reads the row's own x and is dropped by a
  // select), so the 27 loads of a row are in flight together instead of one branch and wait each
  T acc = 0;
#pragma unroll
  for (int s = 0; s < 27; s++) {
    const int di = s / 9 - 1, dj = (s / 3) % 3 - 1, dk = s % 3 - 1;
    const bool in = inside(b, I + di, J + dj, K + dk);
    const T v = A[s * n + r] * x[in ? r + di * sx + dj * sy + dk : r];
    acc += in ? v : T(0);
  }
  y[r] = acc;
}

// The Q1 matrix and its Galerkin coarse operators are symmetric, so the levels keep only the
// diagonal and the 13 upper neighbours, H[s - 13][r] for s = 13..26; the entry of a lower
// neighbour is the upper entry stored at that neighbour's row.  The product reads 14 coefficient
// streams instead of 27 (the shifted reads of the lower half hit the caches).
//
// Sweeps (products with the half stencil).  A workgroup of 64 x BY threads takes NR planes of 64 x BY rows and stages
// the iterate on their neighbourhood (NR + 2 planes, BY + 2 rows, 66 columns, zero outside the box) in LDS: a row then
// issues its 27 coefficient loads and 2 to 5 staged ones instead of 54.  What bounds the row-per-thread form without
// staging is the vector memory path, not the bytes: at 191^3 rows in FP64 it takes 281 us whatever the shape of the
// block (and the bytes it fetches), 202 us if the iterate is not loaded; staged, 215 us with 64 x 4 rows of one plane,
// 204 us with two planes (2.7 instead of 4.6 staged loads per row) and 200 us with 64 x 8 rows of two planes, 4.7 TB/s
// on the 17 values a row cannot do without (a large copy reaches 4.9).  239^3: 561 -> 438, 416, 410 us.
template <int BY, int NR>
struct SweepTile {
  static constexpr int TX = kBX + 2, TY = BY + 2, N = (NR + 2) * TY * TX, NT = kBX * BY, IT = (N + NT - 1) / NT;
};
// Levels take the 64 x 8 x 2 tile where it leaves at least four workgroups per compute unit (1024: from about 90^3
// rows), the 64 x 4 x 1 tile below (47^3: 144 workgroups against 564).
inline bool sweep_big(const Box &b)
{
  return (long)((b.nz + kBX - 1) / kBX) * ((b.ny + 7) / 8) * ((b.nx + 1) / 2) >= 1024;
}

// Workgroups and the eight L2 caches.  Consecutive workgroups go to the XCDs in turn, so tiles in natural order share
// none of the lines that they have in common: the FP16 sweeps fetched 2.2 times the bytes of a row (1.18 GB at 239^3),
// the Galerkin product 3.7 times, and ran at the rate of that traffic.  A box's lines are therefore split into eight
// parts along J, one per XCD (blockIdx.x & 7), each traversed x, y, z in order, so that a part's last plane is still in
// its L2 (191^3: 36 k entries of 112 bytes a plane over eight caches of 4 MB).  At 239^3 the FP16 sweeps fetch 0.63 GB and
// take 158 to 195 instead of 170 to 221 us, the Galerkin product (with a load a fine node) 1.37 instead of 1.62 ms, the
// half stencils 1.10 instead of 1.44 ms; a power iteration at 191^3 231 instead of 244 us.  Boxes with fewer than two
// tiles of lines per part are not split (47^3, all of it in every L2: no difference), nor are boxes with short lines, whose
// blocks are many and touch little: V-cycles of three steps on 399 x 399 x 15 rows 2580 (FP64), 917 (FP16) and 699 us
// split, 2311, 871 and 626 not, on 359 x 359 x 35 1781, 819, 758 and 1711, 779, 726, but on 59 x 449 x 59 449, 235, 232 and
// 478, 247, 262.
struct Split {
  int lg, lines;  // log2 of the number of parts, lines of a part
  __device__ __forceinline__ int j0(unsigned bx, unsigned by, int BY) const
  {
    return (int)(bx & ((1u << lg) - 1)) * lines + (int)by * BY;
  }
  __device__ __forceinline__ int k0(unsigned bx) const { return (int)(bx >> lg) * kBX; }
  __device__ __forceinline__ int j1(unsigned bx, int ny) const
  {
    return min(ny, ((int)(bx & ((1u << lg) - 1)) + 1) * lines);
  }
};
inline Split split_of(const Box &b, int BY)
{
  const int l = (b.ny + 15) / 16 * 2;  // (even: the coarse tiles start at half the first line)
  return l >= 2 * BY && b.nz >= 48 ? Split{3, l} : Split{0, b.ny};
}
inline dim3 split_grid(const Box &b, const Split &s, int BY, int NR)
{
  return dim3((unsigned)((b.nz + kBX - 1) / kBX) << s.lg, (unsigned)((s.lines + BY - 1) / BY),
              (unsigned)((b.nx + NR - 1) / NR));
}

// Entry `row` (the workgroup's part of the row number) + i (the thread's) of an array: a scalar base and a 32-bit offset,
// so that the streams of a row share one address register.  With 64-bit row numbers per thread and stream the addresses
// of a row were half of the vector instructions of a sweep (285 a row in the FP16 one, now 152).
template <typename T>
__device__ __forceinline__ const T &at(const T *p, long row, unsigned i)
{
  return *(const T *)((const char *)(p + row) + i * (unsigned)sizeof(T));
}
template <typename T>
__device__ __forceinline__ T &at(T *p, long row, unsigned i)
{
  return *(T *)((char *)(p + row) + i * (unsigned)sizeof(T));
}

// Fills the tile of the block at (I0, J0, K0) with load(row, i, gi, gj, gk), row + i the row of the tile entry at
// (gi, gj, gk) (every load unconditional: entries outside the box load a row inside it and are zero).  A wavefront takes
// whole lines of 64 columns, whose line numbers are scalars; the two columns beside them go to the first threads (zero
// without a load where one tile covers the lines).  Ends with a barrier.
template <int BY, int NR, typename T, typename Load>
__device__ __forceinline__ void stage_tile(const Box &bx, int I0, int J0, int K0, int tid, T *tile, Load load)
{
  using S = SweepTile<BY, NR>;
  constexpr int L = (NR + 2) * S::TY, IT = (L + BY - 1) / BY;
  static_assert(2 * L <= S::NT, "one halo entry per thread");
  const long sy = bx.nz, sx = (long)bx.ny * bx.nz;
  const int lane = tid & (kBX - 1), w = __builtin_amdgcn_readfirstlane(tid / kBX);
  const bool ink = K0 + lane < bx.nz;
  const unsigned kl = ink ? lane : 0;
  T v[IT], h = T(0);
#pragma unroll
  for (int u = 0; u < IT; u++) {
    const int l = min(w + u * BY, L - 1), gi = I0 + l / S::TY - 1, gj = J0 + l % S::TY - 1;
    const bool in = gi >= 0 && gi < bx.nx && gj >= 0 && gj < bx.ny;
    const T y = load(in ? gi * sx + gj * sy + K0 : (long)K0, kl, gi, gj, K0 + lane);
    v[u] = in && ink ? y : T(0);
  }
  if (bx.nz > kBX && tid < 2 * L) {
    const int l = tid >> 1, gi = I0 + l / S::TY - 1, gj = J0 + l % S::TY - 1, gk = tid & 1 ? K0 + kBX : K0 - 1;
    const bool in = inside(bx, gi, gj, gk);
    const T y = load(in ? gi * sx + gj * sy + gk : 0L, 0u, gi, gj, gk);
    h = in ? y : T(0);
  }
#pragma unroll
  for (int u = 0; u < IT; u++)
    if (w + u * BY < L) tile[(w + u * BY) * S::TX + 1 + lane] = v[u];
  if (tid < 2 * L) tile[(tid >> 1) * S::TX + (tid & 1 ? kBX + 1 : 0)] = h;
  __syncthreads();
}

// Coarse correction of a block's tile: the coarse nodes that interpolate to the tile's fine ones, staged in LDS (zero
// outside the coarse box).  Fine index f has the coarse parents f/2 - 1 and f/2 with weight 1/2 if it is even and
// (f-1)/2 if it is odd; with I0, J0, K0 the block's first fine row, the parents of I0 - 1 .. I0 + NR start at
// I0/2 - 1.  A prolongation of its own (read and write the iterate, 8 coarse loads per row) took 78 us at 239^3 rows in
// FP32, as much as half a smoothing step.
template <int BY, int NR>
struct CoarseTile {
  static constexpr int X = kBX / 2 + 2, Y = BY / 2 + 2, Z = 3, N = X * Y * Z, NT = kBX * BY, IT = (N + NT - 1) / NT;
  static_assert(NR <= 2 && BY % 2 == 0, "three coarse planes cover the tile");
};
template <int BY, int NR, typename T>
__device__ __forceinline__ void stage_coarse(const Box &cb, const T *__restrict__ xc, int I0, int J0, int K0, int tid,
                                             T *ct)
{
  using C = CoarseTile<BY, NR>;
  T v[C::IT];
#pragma unroll
  for (int u = 0; u < C::IT; u++) {
    const int t = min(tid + u * C::NT, C::N - 1);
    const int p = t / (C::Y * C::X), rem = t - p * (C::Y * C::X), jj = rem / C::X, kk = rem - jj * C::X;
    const int ci = (I0 >> 1) - 1 + p, cj = (J0 >> 1) - 1 + jj, ck = (K0 >> 1) - 1 + kk;
    const bool in = inside(cb, ci, cj, ck);
    const T y = xc[in ? ((long)ci * cb.ny + cj) * cb.nz + ck : 0L];
    v[u] = in ? y : T(0);
  }
#pragma unroll
  for (int u = 0; u < C::IT; u++)
    if (tid + u * C::NT < C::N) ct[tid + u * C::NT] = v[u];
  __syncthreads();
}
// The correction at fine node (gi, gj, gk) of the tile.
template <int BY, int NR, typename T>
__device__ __forceinline__ T coarse_value(const T *ct, int I0, int J0, int K0, int gi, int gj, int gk)
{
  using C = CoarseTile<BY, NR>;
  const int i1 = (gi >> 1) - (I0 >> 1) + 1, j1 = (gj >> 1) - (J0 >> 1) + 1, k1 = (gk >> 1) - (K0 >> 1) + 1;
  const int i0 = i1 - 1 + (gi & 1), j0 = j1 - 1 + (gj & 1), k0 = k1 - 1 + (gk & 1);  // odd: the one parent twice
  const T *a = ct + i0 * C::Y * C::X, *b = ct + i1 * C::Y * C::X;
  const int r0 = j0 * C::X, r1 = j1 * C::X;
  return T(0.125) * (((a[r0 + k0] + a[r0 + k1]) + (a[r1 + k0] + a[r1 + k1])) +
                     ((b[r0 + k0] + b[r0 + k1]) + (b[r1 + k0] + b[r1 + k1])));
}

// Row `row` + i of the product, on plane q of the block's tile; tj, tk its row and column there.  A neighbour outside the
// box is zero in the tile; its lower coefficient is read at whatever entry lies there (the stream of direction s starts
// (s - 13) n entries into H, further than the direction reaches back).
template <int BY, typename T>
__device__ __forceinline__ T half_row(const Box &bx, const T *__restrict__ H, const T *tile, int q, int tj, int tk,
                                      long row, unsigned i)
{
  constexpr int TX = SweepTile<BY, 1>::TX, TY = SweepTile<BY, 1>::TY;
  const long n = bx.n(), sy = bx.nz, sx = (long)bx.ny * bx.nz;
  T acc = at(H, row, i) * tile[((q + 1) * TY + tj) * TX + tk];
#pragma unroll
  for (int s = 14; s < 27; s++) {
    const int di = s / 9 - 1, dj = (s / 3) % 3 - 1, dk = s % 3 - 1;
    const long off = di * sx + dj * sy + dk;
    acc += at(H, (s - 13) * n + row, i) * tile[((q + 1 + di) * TY + tj + dj) * TX + tk + dk];
    acc += at(H, (s - 13) * n + row - off, i) * tile[((q + 1 - di) * TY + tj - dj) * TX + tk - dk];
  }
  return acc;
}

// SW_RESID: out = b - A x (b may be null).  SW_CHEB: one Chebyshev step of the smoother, out of place (Jacobi needs the
// old iterate at the neighbours): dn = a d + c D^-1 (b - A x), out = x + dn; d is read when a != 0 and written when
// keep_d.  The _FIRST forms start from the first step's iterate x1 = c1 D^-1 b, formed in the staging: SW_FIRST_CHEB
// takes the second step from it, SW_FIRST_RESID stores it in x1 and its residual in out.  SW_PRO_CHEB takes its step
// from x + P xc, the iterate with the coarse correction.
enum { SW_RESID, SW_CHEB, SW_FIRST_CHEB, SW_FIRST_RESID, SW_PRO_CHEB };
template <typename T, int MODE, int BY, int NR>
__global__ void __launch_bounds__(kBX *BY, 4) half_sweep_kernel(Box bx, Split sp, const T *__restrict__ H,
                                                             const T *__restrict__ dinv, const T *__restrict__ b,
                                                             const T *__restrict__ x, T *__restrict__ out,
                                                             T *__restrict__ d, T *__restrict__ x1, T a, T c, T c1,
                                                             int keep_d, Box cb, const T *__restrict__ xc)
{
  using S = SweepTile<BY, NR>;
  constexpr bool FIRST = MODE == SW_FIRST_CHEB || MODE == SW_FIRST_RESID, PRO = MODE == SW_PRO_CHEB;
  __shared__ T tile[S::N];
  __shared__ T ct[PRO ? CoarseTile<BY, NR>::N : 1];
  const int I0 = blockIdx.z * NR, J0 = sp.j0(blockIdx.x, blockIdx.y, BY), K0 = sp.k0(blockIdx.x);
  const int J1 = sp.j1(blockIdx.x, bx.ny);
  if (J0 >= J1) return;
  if constexpr (PRO) stage_coarse<BY, NR>(cb, xc, I0, J0, K0, threadIdx.y * kBX + threadIdx.x, ct);
  stage_tile<BY, NR>(bx, I0, J0, K0, threadIdx.y * kBX + threadIdx.x, tile,
                     [&](long g, unsigned i, int gi, int gj, int gk) {
    if constexpr (FIRST) return c1 * at(dinv, g, i) * at(b, g, i);
    else if constexpr (PRO) return at(x, g, i) + coarse_value<BY, NR>(ct, I0, J0, K0, gi, gj, gk);
    else return at(x, g, i);
  });
  const int J = J0 + threadIdx.y, K = K0 + threadIdx.x, tj = threadIdx.y + 1, tk = threadIdx.x + 1;
  if (K >= bx.nz || J >= J1) return;
  const unsigned i = threadIdx.y * (unsigned)bx.nz + threadIdx.x;
#pragma unroll
  for (int q = 0; q < NR; q++) {
    const int I = I0 + q;
    if (NR > 1 && I >= bx.nx) break;
    const long row = ((long)I * bx.ny + J0) * bx.nz + K0;
    const T ax = half_row<BY, T>(bx, H, tile, q, tj, tk, row, i);
    const T r = (MODE != SW_RESID || b ? at(b, row, i) : T(0)) - ax;
    const T xi = tile[((q + 1) * S::TY + tj) * S::TX + tk];
    if constexpr (MODE == SW_RESID) {
      at(out, row, i) = r;
    } else if constexpr (MODE == SW_FIRST_RESID) {
      at(x1, row, i) = xi;
      at(out, row, i) = r;
    } else {
      const T dn = (MODE == SW_FIRST_CHEB ? a * xi : a == T(0) ? T(0) : a * at(d, row, i)) + c * at(dinv, row, i) * r;
      if (keep_d) at(d, row, i) = dn;
      at(out, row, i) = xi + dn;
    }
  }
}

template <typename T, int MODE>
void sweep(const Box &bx, const T *H, const T *dinv, const T *b, const T *x, T *out, T *d, T *x1, T a, T c, T c1,
           int keep_d, hipStream_t st, const Box &cb = Box{}, const T *xc = nullptr)
{
  const auto launch = [&](auto kernel, int BY, int NR) {
    const Split sp = split_of(bx, BY);
    hipLaunchKernelGGL(kernel, split_grid(bx, sp, BY, NR), dim3(kBX, BY), 0, st, bx, sp, H, dinv, b, x, out, d, x1, a,
                       c, c1, keep_d, cb, xc);
  };
  if (sweep_big(bx))
    launch(half_sweep_kernel<T, MODE, 8, 2>, 8, 2);
  else
    launch(half_sweep_kernel<T, MODE, 4, 1>, 4, 1);
}

// r = b - A x (b may be null) on a level.
template <typename T>
void residual(const Box &bx, const T *H, const T *b, const T *x, T *r, hipStream_t st)
{
  sweep<T, SW_RESID>(bx, H, nullptr, b, x, r, nullptr, nullptr, T(0), T(0), T(0), 0, st);
}

// Power iterations for the largest eigenvalue of D^-1 A, on all smoothed levels at once: an iteration is one launch
// over the blocks of every level (the coarse ones ride along with the finest), w = D^-1 A (v / ||v||) with the scaling
// applied in the staging and the sums of squares of w reduced per block; where a norm is wanted, one more sums each
// level's block sums in order.  Against a residual, a scaling, a sum and a normalisation per level and iteration: 191^3
// rows and their coarse levels, 15 iterations, 6.5 -> 3.5 ms (4.7 TB/s on the 17 values a row cannot do without); 2.3 ms
// with the largest levels in pairs (pair_kernel).
constexpr int kMaxLevels = 16, kPowerThreads = kBX * 8;
struct PowerLevel {
  Box bx;
  const double *H, *dinv;
  double *v[2], *part;
  Split sp;
  unsigned first, gx, gy;  // first block of the level (a multiple of eight), its grid along x and y
  int blocks, big;         // number of blocks; 64 x 8 x 2 tiles, else 64 x 8 x 1
};
struct PowerArgs {
  PowerLevel l[kMaxLevels];
  int nl;
};

// Sum over the workgroup in a fixed order (within each wavefront, then over the wavefronts); the result is valid in
// thread 0.  sh: one entry per wavefront.
template <int NT>
__device__ __forceinline__ double block_sum(double s, int t, double *sh)
{
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
  if ((t & 63) == 0) sh[t >> 6] = s;
  __syncthreads();
  double r = 0;
  if (t == 0)
#pragma unroll
    for (int w = 0; w < NT / 64; w++) r += sh[w];
  return r;
}

template <int NR>
__device__ __forceinline__ double power_rows(const PowerLevel &l, unsigned blk, double inv, const double *v, double *w,
                                             double *tile)
{
  using S = SweepTile<8, NR>;
  const Box &bx = l.bx;
  const unsigned tx = blk % l.gx, rest = blk / l.gx, ty = rest % l.gy, tz = rest / l.gy;
  const int I0 = tz * NR, J0 = l.sp.j0(tx, ty, 8), J1 = l.sp.j1(tx, bx.ny), K0 = l.sp.k0(tx);
  const int lx = threadIdx.x & (kBX - 1), ly = threadIdx.x / kBX;
  if (J0 >= J1) return 0.0;
  stage_tile<8, NR>(bx, I0, J0, K0, threadIdx.x, tile, [&](long g, unsigned i, int, int, int) { return inv * at(v, g, i); });
  const int J = J0 + ly, K = K0 + lx;
  const unsigned i = ly * (unsigned)bx.nz + lx;
  double s = 0;
  if (K < bx.nz && J < J1) {
#pragma unroll
    for (int q = 0; q < NR; q++) {
      const int I = I0 + q;
      if (NR > 1 && I >= bx.nx) break;
      const long row = ((long)I * bx.ny + J0) * bx.nz + K0;
      const double y = at(l.dinv, row, i) * half_row<8, double>(bx, l.H, tile, q, ly + 1, lx + 1, row, i);
      at(w, row, i) = y;
      s += y * y;
    }
  }
  return s;
}

__global__ void __launch_bounds__(kPowerThreads) power_step_kernel(PowerArgs g, int from,
                                                                   const double *__restrict__ inv)
{
  __shared__ double tile[SweepTile<8, 2>::N];
  __shared__ double sh[kPowerThreads / 64];
  int k = 0;
  while (k + 1 < g.nl && blockIdx.x >= g.l[k + 1].first) k++;
  const PowerLevel &l = g.l[k];
  const unsigned blk = blockIdx.x - l.first;
  if (blk >= (unsigned)l.blocks) return;  // (the next level starts at a multiple of eight)
  const double s = l.big ? power_rows<2>(l, blk, inv[k], l.v[from], l.v[1 - from], tile)
                         : power_rows<1>(l, blk, inv[k], l.v[from], l.v[1 - from], tile);
  const double t = block_sum<kPowerThreads>(s, threadIdx.x, sh);
  if (threadIdx.x == 0) l.part[blk] = t;
}

// FP16 coefficients of the FP32 V-cycle.  With the row scales s_i = sqrt(a_ii) (FP32), a level keeps the 13 upper
// off-diagonals as h_ij = fp16(a_ij / (s_i s_j)) (|h_ij| <= 1 for a symmetric positive definite matrix) and, in FP32,
// the diagonal d_i = a_ii + sum_j (a_ij - s_i s_j h_ij) over all 26 neighbours: the rounding of the off-diagonals
// moves into the diagonal, so every row sum (and with it the near-null space of constants, on which the
// preconditioner's quality rests) is that of the FP64 matrix.  The V-cycle's sweeps work in the scaled variables
// y = s x, b' = b / s, in which row i reads b'_i - e_i y_i - sum_j h_ij y_j with e_i = d_i / s_i^2: 28 + 4 bytes of
// coefficients (the 13 off-diagonals padded to 7 pairs) instead of 56, and one load per neighbour.
__device__ __forceinline__ _Float16 coeff16(double a, float si, float sj)
{
  return (_Float16)(float)(a / ((double)si * (double)sj));
}

// Row scales and inverse diagonals of a level from its 27-point stencil.
__global__ void diag_kernel(long n, const double *__restrict__ A, double *__restrict__ dinv, float *__restrict__ dinv32,
                            float *__restrict__ sc)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double a = A[13 * n + i], r = 1.0 / a;
  dinv[i] = r;
  dinv32[i] = (float)r;
  if (sc) sc[i] = (float)sqrt(a);
}

// The half stencil of a level in FP64 (H, null where the level's own stencil serves), FP32 and FP16 in one pass over its
// 27-point stencil A: a row's 13 upper entries are read once for all three, the row scales of its neighbours come from
// a staged tile, and its lower neighbours' entries (which those rows round) are read for the diagonal's compensation.
// 112 bytes read and 112 + 56 + 48 written per row and 27 FP64 divisions: 191^3 rows 0.95 -> 0.51 ms against a copy of the
// half stencil and an FP16 pass that took 52 square roots per row.
__global__ void __launch_bounds__(256) half_setup_kernel(Box bx, Split sp, const double *__restrict__ A,
                                                         double *__restrict__ H, float *__restrict__ H32,
                                                         _Float16 *__restrict__ H16,
                                                         float *__restrict__ dg, const float *__restrict__ sc,
                                                         float *__restrict__ eg, float *__restrict__ fg, int scaled_in)
{
  using S = SweepTile<kBY, 1>;
  __shared__ float tile[S::N];
  const int I = blockIdx.z, J0 = sp.j0(blockIdx.x, blockIdx.y, kBY), J1 = sp.j1(blockIdx.x, bx.ny);
  const int K0 = sp.k0(blockIdx.x);
  if (J0 >= J1) return;
  stage_tile<kBY, 1>(bx, I, J0, K0, threadIdx.y * kBX + threadIdx.x, tile,
                     [&](long g, unsigned i, int, int, int) { return at(sc, g, i); });
  const int J = J0 + threadIdx.y, K = K0 + threadIdx.x, tj = threadIdx.y + 1, tk = threadIdx.x + 1;
  if (K >= bx.nz || J >= J1) return;
  const long n = bx.n(), sy = bx.nz, sx = (long)bx.ny * bx.nz, i = ((long)I * bx.ny + J) * bx.nz + K;
  const float si = tile[(S::TY + tj) * S::TX + tk];
  const double aii = A[13 * n + i];
  if (H) H[i] = aii;
  H32[i] = (float)aii;
  double comp = 0;
  unsigned pair = 0;
#pragma unroll
  for (int s = 14; s < 27; s++) {
    const int di = s / 9 - 1, dj = (s / 3) % 3 - 1, dk = s % 3 - 1;
    const long off = di * sx + dj * sy + dk;
    const bool up = inside(bx, I + di, J + dj, K + dk), lo = inside(bx, I - di, J - dj, K - dk);
    const double a = A[s * n + i], al = A[s * n + (lo ? i - off : i)];
    if (H) H[(s - 13) * n + i] = a;
    H32[(s - 13) * n + i] = (float)a;
    const float sj = up ? tile[((1 + di) * S::TY + tj + dj) * S::TX + tk + dk] : 1.f;
    const float sl = lo ? tile[((1 - di) * S::TY + tj - dj) * S::TX + tk - dk] : 1.f;
    const _Float16 h = up ? coeff16(a, si, sj) : (_Float16)0;
    if (up) comp += a - (double)si * (double)sj * (double)h;
    // the lower neighbour's entry is its upper one, rounded as that row rounds it
    if (lo) comp += al - (double)sl * (double)si * (double)coeff16(al, sl, si);
    const unsigned bits = __builtin_bit_cast(unsigned short, h);
    if ((s - 14) & 1)
      ((unsigned *)H16)[((s - 14) >> 1) * n + i] = pair | bits << 16;
    else
      pair = bits;
  }
  ((unsigned *)H16)[6 * n + i] = pair;  // (the last pair is padded)
  const double dd = aii + comp, s1 = (double)si;
  dg[i] = (float)dd;
  eg[i] = (float)(dd / (s1 * s1));
  fg[i] = (float)((scaled_in ? s1 * s1 : s1) / dd);  // y = c f b is the first smoothing step from b' or (finest) b
}

// sum_j h_ij y_j over the 26 neighbours of row i, on plane q of the block's staged tile.  The coefficients are stored as
// pairs of directions per row ([7][n] dwords, directions 14 + 2j and 15 + 2j, the last pair padded): a row reads its 13
// upper ones with 7 dword loads, and each lower one (the upper one of the lower neighbour's row) with one, instead of
// 26 two-byte loads.  A neighbour outside the box has a zero tile entry; its coefficient is read at whatever entry lies
// there: only the first pair reaches back past the start of H, from the box's first row (direction 14, row0) and first
// line (direction 15, line0), which read on instead.
__device__ __forceinline__ float half16_value(unsigned pair, int hi)
{
  return (float)__builtin_bit_cast(_Float16, (unsigned short)(hi ? pair >> 16 : pair & 0xffffu));
}
template <int BY>
__device__ __forceinline__ float half16_row(const Box &bx, const _Float16 *__restrict__ H, const float *tile, int q,
                                            int tj, int tk, long row, unsigned i, bool line0, bool row0)
{
  constexpr int TX = SweepTile<BY, 1>::TX, TY = SweepTile<BY, 1>::TY;
  const long n = bx.n(), sy = bx.nz, sx = (long)bx.ny * bx.nz;
  const unsigned *__restrict__ H2 = (const unsigned *)H;
  const unsigned i14 = row0 ? i + 1 : i, i15 = line0 ? i + (unsigned)bx.nz : i;
  unsigned up[7];
#pragma unroll
  for (int j = 0; j < 7; j++) up[j] = at(H2, j * n + row, i);
  float acc = 0;
#pragma unroll
  for (int s = 14; s < 27; s++) {
    const int di = s / 9 - 1, dj = (s / 3) % 3 - 1, dk = s % 3 - 1, j = (s - 14) >> 1;
    const long off = di * sx + dj * sy + dk;
    const float hu = half16_value(up[j], (s - 14) & 1);
    const float hl = half16_value(at(H2, j * n + row - off, s == 14 ? i14 : s == 15 ? i15 : i), (s - 14) & 1);
    acc += hu * tile[((q + 1 + di) * TY + tj + dj) * TX + tk + dk];
    acc += hl * tile[((q + 1 - di) * TY + tj - dj) * TX + tk - dk];
  }
  return acc;
}

// r = b - A x on the FP16 coefficients, in the caller's (unscaled) variables.
__global__ void __launch_bounds__(256) half16_residual_kernel(Box bx, const _Float16 *__restrict__ H,
                                                              const float *__restrict__ dg, const float *__restrict__ sc,
                                                              const float *__restrict__ b, const float *__restrict__ x,
                                                              float *__restrict__ r)
{
  __shared__ float tile[SweepTile<kBY, 1>::N];
  const int I = blockIdx.z, J0 = blockIdx.y * kBY, K0 = blockIdx.x * kBX;
  stage_tile<kBY, 1>(bx, I, J0, K0, threadIdx.y * kBX + threadIdx.x, tile,
                     [&](long g, unsigned i, int, int, int) { return at(sc, g, i) * at(x, g, i); });
  const int J = J0 + threadIdx.y, K = K0 + threadIdx.x;
  if (K >= bx.nz || J >= bx.ny) return;
  const long row = ((long)I * bx.ny + J0) * bx.nz + K0;
  const unsigned i = threadIdx.y * (unsigned)bx.nz + threadIdx.x;
  const float ax = at(dg, row, i) * at(x, row, i) +
                   at(sc, row, i) * half16_row<kBY>(bx, H, tile, 0, threadIdx.y + 1, threadIdx.x + 1, row, i,
                                                    I == 0 && J == 0, I == 0 && J == 0 && K == 0);
  at(r, row, i) = (b ? at(b, row, i) : 0.f) - ax;
}

// The V-cycle's sweeps on the FP16 coefficients, in the scaled variables; the modes are half_sweep_kernel's.  The
// residuals leave unscaled (the restriction works on them), and so does the last step of a level (unscale: x = y / s).
// On the finest level b is the caller's (raw) in the _FIRST forms, which store b' = b / s in bs for the later sweeps.
// 48 bytes a row instead of 56 and one staged load per neighbour instead of two (s and x): at 239^3 rows a smoothing step
// 215 -> 174 us, and the first step and the pass that wrote it (55 us) are part of the second one.
template <int MODE, int BY, int NR>
__global__ void __launch_bounds__(kBX *BY) half16_sweep_kernel(Box bx, Split sp, const _Float16 *__restrict__ H,
                                                               const float *__restrict__ e, const float *__restrict__ f,
                                                               const float *__restrict__ s, const float *__restrict__ b,
                                                               const float *__restrict__ y, float *__restrict__ out,
                                                               float *__restrict__ d, float *__restrict__ y1,
                                                               float *__restrict__ bs, float a, float c, float c1,
                                                               int keep_d, int raw, int unscale, Box cb,
                                                               const float *__restrict__ xc)
{
  using S = SweepTile<BY, NR>;
  constexpr bool FIRST = MODE == SW_FIRST_CHEB || MODE == SW_FIRST_RESID, PRO = MODE == SW_PRO_CHEB;
  __shared__ float tile[S::N];
  __shared__ float ct[PRO ? CoarseTile<BY, NR>::N : 1];
  const int I0 = blockIdx.z * NR, J0 = sp.j0(blockIdx.x, blockIdx.y, BY), K0 = sp.k0(blockIdx.x);
  const int J1 = sp.j1(blockIdx.x, bx.ny);
  if (J0 >= J1) return;
  if constexpr (PRO) stage_coarse<BY, NR>(cb, xc, I0, J0, K0, threadIdx.y * kBX + threadIdx.x, ct);
  stage_tile<BY, NR>(bx, I0, J0, K0, threadIdx.y * kBX + threadIdx.x, tile, [&](long g, unsigned i, int gi, int gj, int gk) {
    if constexpr (FIRST) return c1 * at(f, g, i) * at(b, g, i);
    else if constexpr (PRO) return at(y, g, i) + at(s, g, i) * coarse_value<BY, NR>(ct, I0, J0, K0, gi, gj, gk);
    else return at(y, g, i);
  });
  const int J = J0 + threadIdx.y, K = K0 + threadIdx.x, tj = threadIdx.y + 1, tk = threadIdx.x + 1;
  if (K >= bx.nz || J >= J1) return;
  const unsigned i = threadIdx.y * (unsigned)bx.nz + threadIdx.x;
#pragma unroll
  for (int q = 0; q < NR; q++) {
    const int I = I0 + q;
    if (NR > 1 && I >= bx.nx) break;
    const long row = ((long)I * bx.ny + J0) * bx.nz + K0;
    const float ay = half16_row<BY>(bx, H, tile, q, tj, tk, row, i, I == 0 && J == 0, I == 0 && J == 0 && K == 0);
    const float yi = tile[((q + 1) * S::TY + tj) * S::TX + tk], ei = at(e, row, i);
    float bi = at(b, row, i);
    if (FIRST && raw) {
      bi /= at(s, row, i);
      at(bs, row, i) = bi;
    }
    const float r = bi - (ei * yi + ay);
    if constexpr (MODE == SW_RESID || MODE == SW_FIRST_RESID) {
      if constexpr (FIRST) at(y1, row, i) = yi;
      at(out, row, i) = at(s, row, i) * r;
    } else {
      const float dn = (MODE == SW_FIRST_CHEB ? a * yi : a != 0.f ? a * at(d, row, i) : 0.f) + c * r / ei;
      if (keep_d) at(d, row, i) = dn;
      at(out, row, i) = unscale ? (yi + dn) / at(s, row, i) : yi + dn;
    }
  }
}

// Two sweeps in one pass over the coefficients.  A sweep reads 112 (FP64) or 28 bytes of coefficients per row for one
// product and runs at the rate of memory, so two of them that follow each other are taken together: a workgroup owns a
// column of the box, lines x columns of its (J, K) face, and marches along I.  On plane i it takes the first sweep,
// y1 = S1 (A v0), and with it finishes the second one, S2 (A y1), on plane i - 1.  Symmetry lets a plane's coefficients be
// read once: the product of row (i, j, k) with its lower neighbours is summed while their plane is at hand, as the part
// that the plane below adds to plane i (p1 for the first product, p2 for the second).
//  - A thread owns one (j, k); the face has two rows and columns more on each side than the workgroup's output (its
//    first product is valid one row inside, its second two).
//  - LDS holds the coefficients of the current plane (written by their owners, read by the neighbours above them), v0 on
//    planes i and i + 1, and y1 on plane i.  The next plane's coefficients and the vectors of the one after it are
//    loaded into registers a plane ahead.
//  - Faces: one workgroup per compute unit.  FP16 coefficients: 1024 threads, 64 columns wide (32: 252 instead of 221 us
//    at 239^3).  FP64: 768 threads, whose 168 registers hold a plane ahead (1024 threads: 128, and 176 bytes spilled; 915
//    us a pair of power iterations at 191^3 against 256), 48 columns (32: 269 us).
// 239^3 rows, FP16: both pre-smoothing steps and the residual 204 us against 353 in two sweeps, both post-smoothing steps
// 235 against 370.  191^3, FP64: two power iterations 256 us against 462, pre-smoothing 264 against 392, post-smoothing
// 295 against 476.
// PAIR_POWER: w = (D^-1 A)^2 (v / ||v||) and its sum of squares.  PAIR_PRE: the first two smoothing steps from zero and
// their residual.  PAIR_POST: prolongation and the last two smoothing steps.
// PAIR_PRE1 and PAIR_POST1 march with one product, for one smoothing step: the first step from zero and its residual, or
// prolongation and the step (FP16 only: the coefficients come in 7 aligned dwords per row instead of 20, 159^3 rows 70 ->
// 50 and 76 -> 53 us; in FP64 the sweeps are at the rate of memory).
enum { PAIR_POWER, PAIR_PRE, PAIR_POST, PAIR_PRE1, PAIR_POST1 };
constexpr bool pair_two(int mode) { return mode <= PAIR_POST; }
constexpr int kPairPad = 80;  // LDS entries around the face: border threads read past it, values that nothing uses
constexpr int kPairSlots = 256;
template <typename T>
constexpr int pair_threads()
{
  return sizeof(T) == 8 ? 768 : 1024;
}
template <typename T>
constexpr int pair_width()
{
  return sizeof(T) == 8 ? 48 : 64;
}
static_assert(kPairPad > pair_width<float>() + 5, "a border thread reads one line and one column away");
struct PairTiles {
  int tk, tj, nk, nj, ni, chunk;  // columns and lines of a face, workgroups along K, J and I, planes of one
  int blocks() const { return nk * nj * ni; }
};
// Levels that take them.  Below, a face's border and the few planes of a chunk cost more than the second read of the
// coefficients, which then comes from the 256 MB cache: V-cycles of 79^3 rows take 153 us with pairs against 151 (FP64) and
// 126 against 116 (FP16), of 89^3 159 against 211 and 126 against 122, of 99^3 132 against 148 (FP16).  One step a level
// (FP16): 99^3 92 against 91 us, 119^3 96 against 100, 159^3 180 against 202.
template <typename T>
inline bool pair_level(const Box &b, int degree)
{
  return degree <= 2 && b.n() >= (sizeof(T) == 8 ? 600000 : degree == 2 ? 800000 : 1200000);
}
// Faces as wide as the box divides into at most 64 columns, and as many chunks along I as fill `slots` workgroups.
template <typename T>
PairTiles pair_tiles(const Box &b, int slots, bool two = true)
{
  PairTiles g;
  const int e = two ? 4 : 2;
  g.nk = (b.nz + pair_width<T>() - 1) / pair_width<T>();
  g.tk = (b.nz + g.nk - 1) / g.nk + e;
  g.tj = std::min(pair_threads<T>() / g.tk, b.ny + e);
  g.nj = (b.ny + g.tj - e - 1) / (g.tj - e);
  const int ni = std::max(1, std::min(slots / (g.nk * g.nj), b.nx / 8));
  g.chunk = (b.nx + ni - 1) / ni;
  g.ni = (b.nx + g.chunk - 1) / g.chunk;
  return g;
}

template <typename T>
struct PairCoeffs;
template <>
struct PairCoeffs<double> {  // h[0]: diagonal
  typedef double E;
  static constexpr int kRegs = 14;
  double h[14];
  __device__ __forceinline__ void load(const void *H, long n, long row, unsigned i)
  {
#pragma unroll
    for (int j = 0; j < 14; j++) h[j] = at((const double *)H, j * n + row, i);
  }
  static constexpr int kPlanes = 22;  // directions 14..17, and 18..26 of two planes in turn
  static __device__ __forceinline__ int plane(int s, int par)
  {
    return (s < 18 ? s - 14 : 4 + 9 * par + s - 18) * pair_threads<double>();
  }
  __device__ __forceinline__ void store(double *hs, int t, int par) const
  {
#pragma unroll
    for (int s = 14; s < 27; s++) hs[plane(s, par) + t] = h[s - 13];
  }
  __device__ __forceinline__ double up(int s) const { return h[s - 13]; }
  static __device__ __forceinline__ double lo(const double *hs, int s, int t, int par) { return hs[plane(s, par) + t]; }
  // the upper coefficients of the plane before stay in LDS (18 registers fewer)
  __device__ __forceinline__ void keep() {}
  __device__ __forceinline__ double kept(const double *hs, int s, int t, int par) const { return hs[plane(s, 1 - par) + t]; }
};
template <>
struct PairCoeffs<float> {
  typedef unsigned E;
  static constexpr int kRegs = 7;
  unsigned h[7];
  __device__ __forceinline__ void load(const void *H, long n, long row, unsigned i)
  {
#pragma unroll
    for (int j = 0; j < 7; j++) h[j] = at((const unsigned *)H, j * n + row, i);
  }
  static constexpr int kPlanes = 7;
  unsigned k[5] = {};
  __device__ __forceinline__ void store(unsigned *hs, int t, int) const
  {
#pragma unroll
    for (int j = 0; j < 7; j++) hs[j * pair_threads<float>() + t] = h[j];
  }
  __device__ __forceinline__ float up(int s) const { return half16_value(h[(s - 14) >> 1], (s - 14) & 1); }
  __device__ __forceinline__ void keep()
  {
#pragma unroll
    for (int j = 0; j < 5; j++) k[j] = h[j + 2];
  }
  __device__ __forceinline__ float kept(const unsigned *, int s, int, int) const
  {
    return half16_value(k[(s - 18) >> 1], (s - 14) & 1);
  }
  static __device__ __forceinline__ float lo(const unsigned *hs, int s, int t, int)
  {
    return half16_value(hs[((s - 14) >> 1) * pair_threads<float>() + t], (s - 14) & 1);
  }
};

template <typename T>
struct PairArgs {
  Box bx, cb;
  PairTiles g;
  const void *H;
  const T *dinv, *s;      // FP64: D^-1, null.  FP16: e, s of half16_sweep_kernel
  const T *b, *x, *xc;
  T *out, *r;
  T c1, a, c;             // first step's factor, the second one's
  int raw, unscale;
  const double *inv;
  double *part;
};
template <typename T>
constexpr int pair_lds()
{
  return pair_threads<T>() * (PairCoeffs<T>::kPlanes * (int)sizeof(typename PairCoeffs<T>::E) + 3 * (int)sizeof(T)) +
         8 * kPairPad * (int)sizeof(T);
}

template <typename T, int MODE>
__device__ __forceinline__ void pair_body(const PairArgs<T> &A, int blk, char *lds)
{
  typedef PairCoeffs<T> C;
  constexpr bool F16 = sizeof(T) == 4, TWO = pair_two(MODE);
  constexpr bool PRE = MODE == PAIR_PRE || MODE == PAIR_PRE1, POST = MODE == PAIR_POST || MODE == PAIR_POST1;
  constexpr int B = TWO ? 2 : 1;  // border of the face
  const PairTiles &g = A.g;
  const Box &bx = A.bx;
  typename C::E *Hs = (typename C::E *)lds + kPairPad;
  T *V = (T *)(Hs + C::kPlanes * pair_threads<T>()) + kPairPad, *Y = V + 2 * pair_threads<T>() + 2 * kPairPad;
  const int t = threadIdx.x, tk = g.tk;
  const int kt = blk % g.nk, rest = blk / g.nk, jt = rest % g.nj, it = rest / g.nj;
  const int ia = it * g.chunk, ib = min(bx.nx, ia + g.chunk);
  const int tj = (int)((t + 0.5f) * (1.f / tk)), J = jt * (g.tj - 2 * B) - B + tj, K = kt * (tk - 2 * B) - B + t - tj * tk;
  const bool live = tj < g.tj && J >= 0 && J < bx.ny && K >= 0 && K < bx.nz;
  const bool mine = live && tj >= B && tj < g.tj - B && t - tj * tk >= B && t - tj * tk < tk - B;
  const unsigned o = live ? (unsigned)J * bx.nz + K : 0u;
  const long n = bx.n(), sx = (long)bx.ny * bx.nz;
  // coarse plane's in-plane sum at (J, K): the first four terms of coarse_value
  const int j1 = J >> 1, k1 = K >> 1, j0 = j1 - 1 + (J & 1), k0 = k1 - 1 + (K & 1);
  const auto plane_sum = [&](int ci) -> T {
    if (!live || ci < 0 || ci >= A.cb.nx) return T(0);
    const T *p = A.xc + (long)ci * A.cb.ny * A.cb.nz;
    const auto v = [&](int j, int k) {
      const bool in = j >= 0 && j < A.cb.ny && k >= 0 && k < A.cb.nz;
      const T y = p[in ? j * A.cb.nz + k : 0];
      return in ? y : T(0);
    };
    return (v(j0, k0) + v(j0, k1)) + (v(j1, k0) + v(j1, k1));
  };
  struct Row {
    T b, d, s, v;  // right-hand side, D^-1 (FP64) or e (FP16), row scale, v0
  };
  // v0 and the vectors on plane i (zero outside the box); planes come in order from ia - 2 on
  T sum0 = 0, sum1 = 0;
  int have = -2;  // (the coarse plane that sum1 holds)
  const T inv = MODE == PAIR_POWER ? (T)*A.inv : T(0);
  const auto load_row = [&](int i, Row &w) {
    const long row = (long)min(max(i, 0), bx.nx - 1) * sx;
    const bool in = live && i >= 0 && i < bx.nx;
    w.d = at(A.dinv, row, o);
    w.s = F16 ? at(A.s, row, o) : T(1);
    T v;
    if constexpr (MODE == PAIR_POWER) {
      w.b = T(0);
      v = inv * at(A.x, row, o);
    } else if constexpr (PRE) {
      w.b = at(A.b, row, o);
      if (F16 && A.raw) w.b /= w.s;
      v = F16 ? A.c1 * w.b / w.d : A.c1 * w.d * w.b;
    } else {
      w.b = at(A.b, row, o);
      if (F16 && A.raw) w.b /= w.s;
      const int hi = i >> 1, lo = hi - 1 + (i & 1);  // parents of plane i
      if (i >= 0 && have != hi) {
        sum0 = have == hi - 1 ? sum1 : plane_sum(hi - 1);
        sum1 = plane_sum(hi);
        have = hi;
      }
      const T pro = T(0.125) * ((lo == hi ? sum1 : sum0) + sum1);
      // (after one step from zero the iterate is c1 b' / e again, neither stored nor read; on the finest level b' from b)
      const T x = MODE == PAIR_POST1 ? A.c1 * w.b / w.d : at(A.x, row, o);
      v = F16 ? x + w.s * pro : x + pro;
    }
    w.v = in ? v : T(0);
  };
  const int i0 = max(ia - B, 0), ilast = TWO ? ib : ib - 1;  // (plane nx has no rows: its y1 is zero)
  C h, hn;
  Row w0, w1, w2;
  load_row(i0, w0);
  load_row(i0 + 1, w1);
  h.load(A.H, n, (long)i0 * sx, o);
  __syncthreads();  // (the last use of LDS by the caller)
  V[(i0 & 1) * pair_threads<T>() + t] = w0.v;
  V[((i0 + 1) & 1) * pair_threads<T>() + t] = w1.v;
  T p1 = 0, p2 = 0, q = 0, pb = 0, pd = 1, ps = 1, py = 0, pstep = 0;
  double sum = 0;
  for (int i = i0; i <= ilast; i++) {
    const bool inside_i = i < bx.nx;
    h.store(Hs, t, i & 1);
    load_row(i + 2, w2);
    if (i + 1 < bx.nx) hn.load(A.H, n, (long)(i + 1) * sx, o);
    __syncthreads();
    const T *V0 = V + (i & 1) * pair_threads<T>() + t, *V1 = V + ((i + 1) & 1) * pair_threads<T>() + t;
    // first sweep on plane i
    T acc = (F16 ? w0.d : h.up(13)) * V0[0] + p1;
    p1 = T(0);
#pragma unroll
    for (int s = 14; s < 27; s++) {
      const int off = ((s / 3) % 3 - 1) * tk + s % 3 - 1;
      const T lo = C::lo(Hs, s, t - off, i & 1) * V0[-off];
      if (s < 18) {
        acc += h.up(s) * V0[off];
        acc += lo;
      } else {
        acc += h.up(s) * V1[off];
        p1 += lo;
      }
    }
    const T y0 = w0.v;
    T y1, step = T(0);
    if constexpr (MODE == PAIR_POWER) {
      y1 = w0.d * acc;
    } else {
      const T res = w0.b - acc;
      const T cc = MODE == PAIR_PRE ? A.c : A.c1;
      step = F16 ? cc * res / w0.d : cc * w0.d * res;
      if (MODE == PAIR_PRE) step = A.a * y0 + step;
      y1 = y0 + step;
      if (!TWO && mine && i >= ia) {
        if (PRE) {
          at(A.r, i * sx, o) = F16 ? w0.s * res : res;
        } else {
          at(A.out, i * sx, o) = F16 && A.unscale ? y1 / w0.s : y1;
        }
      }
    }
    if constexpr (TWO) {
      if (!live || !inside_i) y1 = T(0);
      Y[t] = y1;
      if (MODE == PAIR_PRE && mine && i >= ia && i < ib) at(A.out, i * sx, o) = y1;
      __syncthreads();
      // second sweep: plane i - 1 is complete with y1 on plane i
      T z = q;
      const T *Yt = Y + t;
#pragma unroll
      for (int s = 18; s < 27; s++) z += h.kept(Hs, s, t, i & 1) * Yt[((s / 3) % 3 - 1) * tk + s % 3 - 1];
      if (mine && i > ia && i <= ib) {
        const long row = (i - 1) * sx;
        if constexpr (MODE == PAIR_POWER) {
          const T y2 = pd * z;
          at(A.out, row, o) = y2;
          sum += (double)y2 * (double)y2;
        } else if constexpr (MODE == PAIR_PRE) {
          at(A.r, row, o) = F16 ? ps * (pb - z) : pb - z;
        } else {
          const T dn = A.a * pstep + (F16 ? A.c * (pb - z) / pd : A.c * pd * (pb - z));
          at(A.out, row, o) = F16 && A.unscale ? (py + dn) / ps : py + dn;
        }
      }
      q = (F16 ? w0.d : h.up(13)) * y1 + p2;
      p2 = T(0);
#pragma unroll
      for (int s = 14; s < 27; s++) {
        const int off = ((s / 3) % 3 - 1) * tk + s % 3 - 1;
        const T lo = C::lo(Hs, s, t - off, i & 1) * Yt[-off];
        if (s < 18) {
          q += h.up(s) * Yt[off];
          q += lo;
        } else {
          p2 += lo;
        }
      }
      pb = w0.b;
      pd = w0.d;
      ps = w0.s;
      py = y1;
      pstep = step;
    } else {
      __syncthreads();
    }
    V[(i & 1) * pair_threads<T>() + t] = w2.v;
    h.keep();
#pragma unroll
    for (int j = 0; j < C::kRegs; j++) h.h[j] = hn.h[j];
    w0 = w1;
    w1 = w2;
    __syncthreads();
  }
  if constexpr (MODE == PAIR_POWER) {
    const double tot = block_sum<pair_threads<T>()>(sum, t, (double *)lds);
    if (t == 0) A.part[blk] = tot;
  }
}

// Workgroups of one XCD take consecutive faces (K, then J, then I), whose borders meet in its L2.
template <typename T, int MODE>
__global__ void __launch_bounds__(pair_threads<T>()) pair_kernel(PairArgs<T> A)
{
  extern __shared__ double pair_smem[];
  const int total = A.g.nk * A.g.nj * A.g.ni, per = (total + 7) / 8;
  const int blk = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if (blk >= total) return;
  pair_body<T, MODE>(A, blk, (char *)pair_smem);
}

template <typename T, int MODE>
void pair_sweep(const PairArgs<T> &A, hipStream_t st)
{
  hipLaunchKernelGGL((pair_kernel<T, MODE>), dim3((unsigned)((A.g.blocks() + 7) / 8 * 8)), dim3(pair_threads<T>()),
                     pair_lds<T>(), st, A);
}

// The half stencil alone (the coarsest level, which is solved directly).
__global__ void half_from_full_kernel(long n, const double *__restrict__ A, double *__restrict__ H,
                                      float *__restrict__ H32)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int s = 13; s < 27; s++) {
    if (H) H[(s - 13) * n + i] = A[s * n + i];
    H32[(s - 13) * n + i] = (float)A[s * n + i];
  }
}

// Two neighbouring entries in one load.
template <typename T>
struct __attribute__((packed, aligned(sizeof(T)))) Two {
  T lo, hi;
};

// bc = P^T rf, divided by the coarse level's row scales s (null: not).  Split over the L2 caches as the sweeps are, and two
// of the three fine rows along k in one load: 119^3 coarse rows in FP32 33 -> 26 us, 79^3 15 -> 11.6.
template <typename T>
__global__ void restrict_kernel(Box f, Box c, Split sp, const T *__restrict__ rf, T *__restrict__ bc,
                                const T *__restrict__ s)
{
  const int I = blockIdx.z, J = sp.j0(blockIdx.x, blockIdx.y, kBY) + threadIdx.y, K = sp.k0(blockIdx.x) + threadIdx.x;
  if (J >= sp.j1(blockIdx.x, c.ny) || K >= c.nz) return;
  const long C = ((long)I * c.ny + J) * c.nz + K;
  const long sy = f.nz, sx = (long)f.ny * f.nz;
  const int F0 = 2 * I + 1, F1 = 2 * J + 1, F2 = 2 * K + 1;
  const long base = F0 * sx + F1 * sy + F2;  // (F0, F1, F2) is inside the fine box; its upper neighbours may not be
  const bool ink = F2 + 1 < f.nz;
  T acc = 0;
#pragma unroll
  for (int a = -1; a <= 1; a++)
#pragma unroll
    for (int b = -1; b <= 1; b++) {
      const bool in = F0 + a < f.nx && F1 + b < f.ny;
      const T w = T((a ? 0.5 : 1.0) * (b ? 0.5 : 1.0));
      const T *p = rf + (in ? base + a * sx + b * sy : base);  // unconditional loads, dropped by a select
      const Two<T> q = *(const Two<T> *)(p - 1);
      const T v = p[ink ? 1 : 0];
      acc += in ? T(0.5) * w * q.lo : T(0);
      acc += in ? w * q.hi : T(0);
      acc += in && ink ? T(0.5) * w * v : T(0);
    }
  bc[C] = s ? acc / s[C] : acc;
}
template <typename T>
void restrict_to(const Box &f, const Box &c, const T *rf, T *bc, const T *s, hipStream_t st)
{
  const Split sp = split_of(c, kBY);
  hipLaunchKernelGGL(restrict_kernel<T>, split_grid(c, sp, kBY, 1), box_block(), 0, st, f, c, sp, rf, bc, s);
}

// 1-D prolongation weight of the coarse node at offset t (in -1..1) from coarse node c at the fine node at offset e
// (in -2..2) from c's own fine node 2c+1: 1 if e = 2t, 1/2 if |e - 2t| = 1, else 0.
__host__ __device__ constexpr double pweight(int e, int t)
{
  return e == 2 * t ? 1.0 : (e - 2 * t == 1 || e - 2 * t == -1) ? 0.5 : 0.0;
}

// Ac = P^T Af P (FP64).  Row C gathers over the 27 fine nodes f of its prolongation's support (weight P[f][C]) and
// their 27 stencil entries A[f][g].  The weights factor by direction: with f at offsets (a, b, d) from C's own fine node
// and g = f + (si, sj, sk), P[f][C] P[g][C + t] = X(a, si, ti) Y(b, sj, tj) Z(d, sk, tk).  A workgroup takes 64 rows;
// each of its nine wavefronts takes one x part (a, si): the 81 (b, d, sj, sk) terms have compile-time y and z weights
// and are summed into 3 x 3 partial sums in registers (every load unconditional: a support node outside the fine box
// reads entry 0 with weight 0).  The partial sums meet the x weights through LDS, three of the 27 entries per wavefront.
// With one thread per row the nine parts followed one another, 729 loads at 13 wavefronts per SIMD in all: latency
// bound, 1.90 ms at 95^3 coarse rows and 0.11 ms at 5^3; this takes 0.46 and 0.01 ms (0.71 with a load for each of the
// three fine nodes along k, whose lanes are two rows apart: two of them come in one).  Entries toward coarse nodes outside
// the box are zero, as the assembly leaves them on the finest level.
__global__ void __launch_bounds__(576) rap_kernel(Box f, Box c, int part, const double *__restrict__ Af,
                                                  double *__restrict__ Ac)
{
  __shared__ double psum[9][9][64];  // [x part][3 x 3 sum][row]
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, a = w / 3 - 1, si = w % 3 - 1;
  const long nc = c.n(), nf = f.n();
  // a part's lines of one plane are one run of rows
  const int xcd = blockIdx.x & 7, jp = xcd * part, lines = min(part, c.ny - jp), o0 = (int)(blockIdx.x >> 3) * 64 + lane;
  if (lines <= 0 || (int)(blockIdx.x >> 3) * 64 >= lines * c.nz) return;
  const bool valid = o0 < lines * c.nz;
  const int o = valid ? o0 : 0, I = blockIdx.y, J = jp + o / c.nz, K = o % c.nz;
  const long C = ((long)I * c.ny + J) * c.nz + K;
  const long sy = f.nz, sx = (long)f.ny * f.nz;
  const int fi = 2 * I + 1 + a;  // >= 0
  double T[9];
#pragma unroll
  for (int u = 0; u < 9; u++) T[u] = 0.0;
  const bool ini = fi < f.nx, ink = 2 * K + 2 < f.nz;
#pragma unroll
  for (int b = -1; b <= 1; b++) {
    const int fj = 2 * J + 1 + b;
    const bool in = ini && fj < f.ny;
    const long fr = in ? fi * sx + fj * sy + 2 * K : 0;  // the fine node at d = -1 (inside along k, as that at d = 0)
    double v[3][9];
#pragma unroll
    for (int s = 0; s < 9; s++) {
      const double *p = Af + ((si + 1) * 9 + s) * nf + fr;
      const Two<double> q = *(const Two<double> *)p;
      v[0][s] = q.lo;
      v[1][s] = q.hi;
      v[2][s] = p[ink ? 2 : 0];
    }
#pragma unroll
    for (int d = -1; d <= 1; d++) {
      const double w0 = in && (d < 1 || ink) ? pweight(b, 0) * pweight(d, 0) : 0.0;
#pragma unroll
      for (int sj = -1; sj <= 1; sj++)
#pragma unroll
        for (int sk = -1; sk <= 1; sk++) {
          const double vs = w0 * v[d + 1][(sj + 1) * 3 + sk + 1];
#pragma unroll
          for (int tj = -1; tj <= 1; tj++)
#pragma unroll
            for (int tk = -1; tk <= 1; tk++) {
              const double q = pweight(b + sj, tj) * pweight(d + sk, tk);
              if (q != 0.0) T[(tj + 1) * 3 + (tk + 1)] = fma(vs, q, T[(tj + 1) * 3 + (tk + 1)]);
            }
        }
    }
  }
#pragma unroll
  for (int u = 0; u < 9; u++) psum[w][u][lane] = T[u];
  __syncthreads();
  if (!valid) return;
#pragma unroll
  for (int x = 0; x < 3; x++) {  // entry t = 9 x + w: x offset x - 1
    const int t = 9 * x + w;
    double acc = 0.0;
#pragma unroll
    for (int aa = -1; aa <= 1; aa++)
#pragma unroll
      for (int ss = -1; ss <= 1; ss++)
        acc = fma(pweight(aa, 0) * pweight(aa + ss, x - 1), psum[(aa + 1) * 3 + ss + 1][w][lane], acc);
    Ac[t * nc + C] = inside(c, I + x - 1, J + w / 3 - 1, K + w % 3 - 1) ? acc : 0.0;
  }
}

// Explicit inverse of the (symmetric positive definite) coarsest matrix, in place, by Gauss-Jordan elimination on
// 32 x 32 blocks without pivoting.  A step k takes two launches: the panel kernel inverts the diagonal block (every
// workgroup for itself, in LDS), forms its part of R = D A_k: and copies its part of the block column A_:k; the update
// kernel writes A_ij -= A_ik R_j, R in block row k, -A_ik D in block column k and D itself: 30 -> 18 us a step at 504
// rows since a pivot pair waits at one barrier and no load waits for another.  A hierarchy's whole set-up at 47 x 47 x 47
// rows over 125 coarsest ones 2.1 -> 0.44 ms, at 63^3 over 343 13.4 -> 0.72 ms, at 65^3 over 512 46 -> 0.94 ms: scalar
// host code between two copies did the elimination before.
constexpr int kCB = 32;
constexpr long kMaxCoarse = 4096;
__global__ void dense_fill_kernel(Box b, const double *__restrict__ st, double *__restrict__ A)
{
  const long n = b.n(), t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * n) return;
  const long r = t / n;
  int I, J, K, I2, J2, K2;
  unrank(b, r, I, J, K);
  unrank(b, t - r * n, I2, J2, K2);
  const int di = I2 - I, dj = J2 - J, dk = K2 - K;
  const bool in = di >= -1 && di <= 1 && dj >= -1 && dj <= 1 && dk >= -1 && dk <= 1;
  A[t] = in ? st[((di + 1) * 9 + (dj + 1) * 3 + (dk + 1)) * n + r] : 0.0;
}

__global__ void __launch_bounds__(256) dense_panel_kernel(int n, int k0, const double *__restrict__ A,
                                                          double *__restrict__ R, double *__restrict__ Cc,
                                                          double *__restrict__ D, double *__restrict__ bad)
{
  // the pivots read one copy of the block and write the other (a thread keeps its own entries in registers), and the
  // block row's part that R needs is loaded ahead of the pivots
  __shared__ double d[2][kCB][kCB + 1], ak[kCB][kCB + 1];
  const int t = threadIdx.x, m = min(kCB, n - k0);
  const int c = t % kCB, r0 = t / kCB;  // this thread's column and rows r0, r0 + 8, ...
  const int j0 = blockIdx.x * kCB, j = j0 + c;  // columns (of R) and rows (of the copied panel) of this workgroup
  // (every load unconditional, here and below: behind branches a thread's loads follow one another, 17 instead of 12 us)
  double v[4], w[4];
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const long row = (long)min(k0 + r0 + 8 * u, n - 1) * n;
    v[u] = A[row + min(k0 + c, n - 1)];
    w[u] = A[row + min(j, n - 1)];
  }
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int r = r0 + 8 * u;
    v[u] = r < m && c < m ? v[u] : r == c ? 1.0 : 0.0;
    ak[r][c] = r < m && j < n ? w[u] : 0.0;
    d[0][r][c] = v[u];
  }
  __syncthreads();
  // (two pivots a barrier: the second one's row and column after the first come from the same copy; past m the block is
  // the identity, on which a pivot changes nothing)
  for (int p = 0; p < m; p += 2) {
    const double(&s)[kCB][kCB + 1] = d[(p >> 1) & 1];
    const double a0 = s[p][p], a0q = s[p][p + 1], b1 = s[p + 1][p], b1q = s[p + 1][p + 1], s0 = s[p][c], s1 = s[p + 1][c];
    double cp[4], cq[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      cp[u] = s[r0 + 8 * u][p];
      cq[u] = s[r0 + 8 * u][p + 1];
    }
    const double i0 = 1.0 / a0, row0 = (c == p ? 1.0 : s0) * i0, row0q = a0q * i0;
    const double x1 = (c == p ? 0.0 : s1) - b1 * row0, a1 = b1q - b1 * row0q;
    const double row1 = (c == p + 1 ? 1.0 : x1) * (1.0 / a1);
    if (t == 0 && blockIdx.x == 0 && !(a0 > 0.0 && a1 > 0.0)) *bad = 1.0;
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int r = r0 + 8 * u;
      const double e0 = (c == p ? 0.0 : v[u]) - cp[u] * row0, e = r == p ? row0 : e0;
      const double q0 = cq[u] - cp[u] * row0q, q = r == p ? row0q : q0;
      const double x = (c == p + 1 ? 0.0 : e) - q * row1;
      v[u] = r == p + 1 ? row1 : x;
      d[1 - ((p >> 1) & 1)][r][c] = v[u];
    }
    __syncthreads();
  }
  const double(&f)[kCB][kCB + 1] = d[((m + 1) >> 1) & 1];
  if (blockIdx.x == 0)
#pragma unroll
    for (int u = 0; u < 4; u++) D[(r0 + 8 * u) * kCB + c] = v[u];
  double sum[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 8
  for (int q = 0; q < kCB; q++) {  // (past m the rows of ak are zero)
    const double a = ak[q][c];
#pragma unroll
    for (int u = 0; u < 4; u++) sum[u] += f[r0 + 8 * u][q] * a;
  }
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int r = r0 + 8 * u;
    if (j < n && r < m) R[(long)r * n + j] = sum[u];
    if (j0 + r < n && c < m) Cc[(long)(j0 + r) * kCB + c] = A[(long)(j0 + r) * n + k0 + c];
  }
}

__global__ void __launch_bounds__(256) dense_update_kernel(int n, int k0, double *__restrict__ A,
                                                           const double *__restrict__ R,
                                                           const double *__restrict__ Cc,
                                                           const double *__restrict__ D)
{
  __shared__ double cs[kCB][kCB + 1], rs[kCB][kCB + 1];
  const int t = threadIdx.x, m = min(kCB, n - k0), i0 = blockIdx.y * kCB, j0 = blockIdx.x * kCB, c = t % kCB, r0 = t / kCB;
  const bool row = i0 == k0, col = j0 == k0;
  double vc[4], vr[4], va[4];  // (unconditional loads, as in the panel kernel)
  const int j = min(j0 + c, n - 1);
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int r = r0 + 8 * u, i = min(i0 + r, n - 1);
    vc[u] = Cc[(long)i * kCB + c];
    vr[u] = col ? D[r * kCB + c] : R[(long)min(r, m - 1) * n + j];
    va[u] = A[(long)i * n + j];
  }
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int r = r0 + 8 * u;
    cs[r][c] = i0 + r < n && c < m ? vc[u] : 0.0;
    rs[r][c] = r < m && j0 + c < n ? vr[u] : 0.0;
  }
  __syncthreads();
  double sum[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 8
  for (int q = 0; q < kCB; q++) {  // (past m both are zero)
    const double x = rs[q][c];
#pragma unroll
    for (int u = 0; u < 4; u++) sum[u] += cs[r0 + 8 * u][q] * x;
  }
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int r = r0 + 8 * u;
    if (i0 + r < n && j0 + c < n)
      A[(long)(i0 + r) * n + j0 + c] = row ? rs[r][c] : (col ? 0.0 : va[u]) - sum[u];
  }
}

// x = Ainv b, one wavefront per row (lanes stride the row, then a butterfly reduction).
template <typename T>
__global__ void dense_mv_kernel(int n, const T *__restrict__ Ainv, const T *__restrict__ b, T *__restrict__ x)
{
  const int r = blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64, lane = threadIdx.x & 63;
  if (r >= n) return;  // whole wavefronts exit together
  T acc = 0;
  for (int c = lane; c < n; c += 64) acc += Ainv[(long)r * n + c] * b[c];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
  if (lane == 0) x[r] = acc;
}

__global__ void zero_kernel(long n, double *__restrict__ a)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = 0.0;
}

__global__ void to_f32(long n, const double *__restrict__ a, float *__restrict__ b)
{
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = (float)a[i];
}

// Start vectors of the power iteration: a counter-based hash (splitmix64) of the row, uniform in [0.25, 1.25), with
// the sums of squares of 256 blocks per level (blockIdx.y).
__global__ void __launch_bounds__(256) power_start_kernel(PowerArgs g)
{
  __shared__ double sh[4];
  const PowerLevel &l = g.l[blockIdx.y];
  const long n = l.bx.n();
  double s = 0;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += 256L * gridDim.x) {
    uint64_t z = (uint64_t)i + 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    z ^= z >> 31;
    const double v = (double)(z >> 11) * (1.0 / 9007199254740992.0) + 0.25;
    l.v[0][i] = v;
    s += v * v;
  }
  const double t = block_sum<256>(s, threadIdx.x, sh);
  if (threadIdx.x == 0) l.part[blockIdx.x] = t;
}

// ||v|| and 1 / ||v|| of every level (blockIdx.x) from its block sums, taken in order: the 256 of the start vector, or
// one per block of the level.
__global__ void __launch_bounds__(1024) power_norm_kernel(PowerArgs g, int start, double *__restrict__ norm,
                                                          double *__restrict__ inv)
{
  __shared__ double sh[16];
  const PowerLevel &l = g.l[blockIdx.x];
  const int m = start ? 256 : l.blocks;
  double s = 0;
  for (int k = threadIdx.x; k < m; k += 1024) s += l.part[k];
  const double t = block_sum<1024>(s, threadIdx.x, sh);
  if (threadIdx.x == 0) {
    const double nw = sqrt(t);
    norm[blockIdx.x] = nw;
    inv[blockIdx.x] = 1.0 / nw;
  }
}

inline dim3 grid_of(long n) { return dim3((unsigned)((n + 255) / 256)); }

}  // namespace

dErr dohpMatPrepareStencil_Private(_p_dohpMat *A, dohpFS fs, bool *box, hipStream_t st)
{
  (void)st;
  const long L0 = (long)fs->p * fs->M[0] + 1, L1 = (long)fs->p * fs->M[1] + 1, L2 = (long)fs->p * fs->M[2] + 1;
  const int m = fs->dirichlet_mask;
  Box b{(int)(L0 - ((m & 1) ? 2 : 0)), (int)(L1 - ((m & 1) ? 2 : 0)), (int)(L2 - ((m & 2) ? 1 : 0) - ((m & 4) ? 1 : 0))};
  *box = false;
  if (b.n() != A->nrows || b.nx <= 0 || b.ny <= 0 || b.nz <= 0) return 0;
  A->box[0] = b.nx;
  A->box[1] = b.ny;
  A->box[2] = b.nz;
  if (!A->st64.holds(27 * b.n()) || !A->st32.holds(27 * b.n())) {  // both or neither
    dErr err = A->st64.alloc(27 * b.n());
    if (!err) err = A->st32.alloc(27 * b.n());
    if (err) {
      A->st64.release();
      A->st32.release();
      return err;
    }
  }
  *box = true;
  return 0;
}

dErr dohpMatStencilToCSR_Private(_p_dohpMat *A, hipStream_t st)
{
  const Box b{A->box[0], A->box[1], A->box[2]};
  hipLaunchKernelGGL(stencil_to_csr_kernel, dim3((unsigned)((b.n() + 255) / 256)), dim3(256), 0, st, b, A->rowptr.ptr,
                     A->col.ptr, A->st64.ptr, A->val.ptr, A->val32.ptr, A->st32.ptr);
  DOHP_HIP(hipGetLastError());
  return 0;
}

dErr dohpStencilMult_Private(const _p_dohpMat *A, const double *x, double *y, hipStream_t st)
{
  const Box b{A->box[0], A->box[1], A->box[2]};
  hipLaunchKernelGGL(stencil_mult_kernel<double>, box_grid(b), box_block(), 0, st, b, A->st64.ptr, x, y);
  DOHP_HIP(hipGetLastError());
  return 0;
}

dErr dohpStencilMultF32_Private(const _p_dohpMat *A, const float *x, float *y, hipStream_t st)
{
  const Box b{A->box[0], A->box[1], A->box[2]};
  hipLaunchKernelGGL(stencil_mult_kernel<float>, box_grid(b), box_block(), 0, st, b, A->st32.ptr, x, y);
  DOHP_HIP(hipGetLastError());
  return 0;
}

struct MGLevel {
  Box box{};
  long n = 0;
  const double *A64 = nullptr;  // full 27-point stencil (finest level: the Q1 matrix's own)
  const double *H = nullptr;    // symmetric half stencil [14][n]: H64 on the finest level, part of own64 below
  DevBuf<double> own64, H64, dinv64, b64, x64, r64, d64;
  DevBuf<float> H32, dinv32, b32, x32, r32, d32;
  DevBuf<_Float16> H16;        // FP16 upper off-diagonals, pairs of directions per row [7][n][2] (half16_row)
  DevBuf<float> dg16, sc16;    // their diagonal d and row scales s
  DevBuf<float> e16, f16;      // d / s^2; the first smoothing step's factor (half_setup_kernel)
  DevBuf<float> t32;           // finest level: the scaled right-hand side
  double lmax = 0;
};

struct _p_dohpMG {
  std::vector<MGLevel> L;
  int degree = 2;
  double lo = 0.1, hi = 1.1;
  int ncoarse = 0;
  int coeff16 = 1;  // the FP32 V-cycle reads the FP16 coefficients
  DevBuf<double> cinv64;
  DevBuf<float> cinv32;
  DevBuf<double> part;   // the power iterations' norms and block sums
  DevBuf<double> cwork;  // the coarsest inverse's panels
  // V-cycles replayed as HIP graphs: the coarse levels' kernels run for a few microseconds each, less than their
  // launch costs the host, so the eager V-cycle leaves the GPU waiting; a graph is captured (on a private stream)
  // per precision for the vectors it was applied to and replayed while they stay the same.
  struct Graph {
    const void *r = nullptr;  // the vectors of the captured graph, or of the last eager application
    void *z = nullptr;
    int coeff16 = -1;
    hipGraphExec_t exec = nullptr;
  };
  Graph g64, g32;
  int graphs = 1;
  hipStream_t cap = nullptr;
  void drop_graphs()
  {
    for (Graph *g : {&g64, &g32}) {
      if (g->exec) (void)hipGraphExecDestroy(g->exec);
      *g = Graph{};
    }
  }
  ~_p_dohpMG()
  {
    drop_graphs();
    if (cap) (void)hipStreamDestroy(cap);
  }
};

namespace {

// The sweep's grid of a level in a power iteration, and the block sums that the level's launches write: 256 of the start
// vector, one per workgroup of a sweep, or one per workgroup of a pair.  Neither of the last two bounds the other: on a
// box of two planes the faces of a pair can be more (2 x 800 x 800 rows: 1360 workgroups against 1352).
dim3 power_grid(const Box &b) { return split_grid(b, split_of(b, 8), 8, sweep_big(b) ? 2 : 1); }
long power_sums(const Box &b)
{
  const dim3 g = power_grid(b);
  const long single = (long)g.x * g.y * g.z;
  const long pair = pair_level<double>(b, 2) ? pair_tiles<double>(b, kPairSlots).blocks() : 0;
  return std::max({256L, single, pair});
}

// lmax of D^-1 A on every smoothed level by power iteration, in the levels' work vectors (free outside a V-cycle).  The
// iterations stay on the device and leave the last norms at the start of mg->part.
dErr estimate_lmax(_p_dohpMG *mg, hipStream_t st, int its)
{
  const int nl = (int)mg->L.size() - 1;
  if (nl == 0) return 0;
  DOHP_CHECK(nl <= kMaxLevels, dohpERR_ARG, "multigrid: too many levels");
  PowerArgs g{};
  g.nl = nl;
  unsigned blocks = 0;
  int nb = 0;
  unsigned blocks_small = 0;
  size_t parts = 2 * kMaxLevels;  // norms and their inverses, then the levels' block sums
  long sums[kMaxLevels];
  for (int k = 0; k < nl; k++) {
    MGLevel &lv = mg->L[k];
    PowerLevel &l = g.l[k];
    l.bx = lv.box;
    l.H = lv.H;
    l.dinv = lv.dinv64.ptr;
    l.v[0] = lv.r64.ptr;
    l.v[1] = lv.d64.ptr;
    l.big = sweep_big(lv.box);
    l.sp = split_of(lv.box, 8);
    const dim3 grid = power_grid(lv.box);
    l.gx = grid.x;
    l.gy = grid.y;
    l.blocks = (int)(grid.x * grid.y * grid.z);
    l.first = blocks;
    blocks += (l.blocks + 7) / 8 * 8;
    parts += sums[k] = power_sums(lv.box);
    if (pair_level<double>(lv.box, 2)) nb = k + 1;  // (levels shrink: the first ones)
  }
  if (!mg->part.holds(parts)) DOHP_CALL(mg->part.alloc(parts));
  double *norm = mg->part.ptr, *inv = norm + kMaxLevels, *at = inv + kMaxLevels;
  for (int k = 0; k < nl; k++) {
    g.l[k].part = at;
    at += sums[k];
  }
  hipLaunchKernelGGL(power_start_kernel, dim3(256, nl), dim3(256), 0, st, g);
  hipLaunchKernelGGL(power_norm_kernel, dim3(nl), dim3(1024), 0, st, g, 1, norm, inv);
  // The vectors are normalised before the last iteration; until then every iteration scales by the start's 1 / ||v||, which
  // leaves them between 1e-66 and 1e22 times the start after fifteen (a norm a launch: 5 us an iteration, 60 of the 560 us
  // of a Newton step at 25 k rows).  Large levels take two iterations a pass, the others one by one beside them; the last
  // iteration, whose growth is the estimate, is a single one everywhere.
  const int pairs = nb ? (its - 1) / 2 : 0;
  PowerArgs gs = g, gb = g;  // the small levels alone; all levels, the large ones with their pairs' block counts
  if (pairs) {
    gs.nl = nl - nb;
    unsigned first = 0;
    for (int k = nb; k < nl; k++) {
      gs.l[k - nb] = g.l[k];
      gs.l[k - nb].first = first;
      first += (g.l[k].blocks + 7) / 8 * 8;
    }
    blocks_small = first;
  }
  for (int q = 0; q < pairs; q++) {
    for (int k = 0; k < nb; k++) {
      PowerLevel &l = gb.l[k];
      PairArgs<double> pa{};
      pa.bx = l.bx;
      pa.g = pair_tiles<double>(l.bx, kPairSlots);
      pa.H = l.H;
      pa.dinv = l.dinv;
      pa.x = l.v[q & 1];
      pa.out = l.v[1 - (q & 1)];
      pa.inv = inv + k;
      pa.part = l.part;
      l.blocks = pa.g.blocks();
      pair_sweep<double, PAIR_POWER>(pa, st);
    }
    for (int k = 0; k < 2 && gs.nl; k++)
      hipLaunchKernelGGL(power_step_kernel, dim3(blocks_small), dim3(kPowerThreads), 0, st, gs, k, inv + nb);
  }
  const int singles = its - 2 * pairs;
  if (pairs && singles == 1) hipLaunchKernelGGL(power_norm_kernel, dim3(nl), dim3(1024), 0, st, gb, 0, norm, inv);
  if (pairs & 1)
    for (int k = 0; k < nb; k++) std::swap(g.l[k].v[0], g.l[k].v[1]);
  for (int k = 0; k < singles; k++) {
    hipLaunchKernelGGL(power_step_kernel, dim3(blocks), dim3(kPowerThreads), 0, st, g, k & 1, inv);
    if (k >= singles - 2) hipLaunchKernelGGL(power_norm_kernel, dim3(nl), dim3(1024), 0, st, g, 0, norm, inv);
  }
  DOHP_HIP(hipGetLastError());
  return 0;
}

// Inverse of the coarsest matrix, FP64 and FP32, on the device; work[0] is set to 1 if a pivot is not positive.
dErr coarse_inverse(_p_dohpMG *mg, hipStream_t st)
{
  const MGLevel &lv = mg->L.back();
  const int n = (int)lv.n;
  const size_t nn = (size_t)n * n, nw = 1 + kCB * kCB + 2 * (size_t)kCB * n;
  if (!mg->cinv64.holds(nn)) DOHP_CALL(mg->cinv64.alloc(nn));
  if (!mg->cinv32.holds(nn)) DOHP_CALL(mg->cinv32.alloc(nn));
  if (!mg->cwork.holds(nw)) DOHP_CALL(mg->cwork.alloc(nw));
  double *A = mg->cinv64.ptr, *bad = mg->cwork.ptr, *D = bad + 1, *R = D + kCB * kCB, *Cc = R + (size_t)kCB * n;
  const unsigned nb = (unsigned)((n + kCB - 1) / kCB);
  hipLaunchKernelGGL(zero_kernel, dim3(1), dim3(64), 0, st, 1L, bad);
  hipLaunchKernelGGL(dense_fill_kernel, grid_of((long)nn), dim3(256), 0, st, lv.box, lv.A64, A);
  for (int k0 = 0; k0 < n; k0 += kCB) {
    hipLaunchKernelGGL(dense_panel_kernel, dim3(nb), dim3(256), 0, st, n, k0, A, R, Cc, D, bad);
    hipLaunchKernelGGL(dense_update_kernel, dim3(nb, nb), dim3(256), 0, st, n, k0, A, R, Cc, D);
  }
  hipLaunchKernelGGL(to_f32, grid_of((long)nn), dim3(256), 0, st, (long)nn, A, mg->cinv32.ptr);
  DOHP_HIP(hipGetLastError());
  return 0;
}

template <typename T>
struct LvPtr;
template <>
struct LvPtr<double> {
  static const double *A(const MGLevel &l) { return l.H; }
  static const double *dinv(const MGLevel &l) { return l.dinv64.ptr; }
  static double *b(MGLevel &l) { return l.b64.ptr; }
  static double *x(MGLevel &l) { return l.x64.ptr; }
  static double *r(MGLevel &l) { return l.r64.ptr; }
  static double *d(MGLevel &l) { return l.d64.ptr; }
  static const double *cinv(const _p_dohpMG *m) { return m->cinv64.ptr; }
};
template <>
struct LvPtr<float> {
  static const float *A(const MGLevel &l) { return l.H32.ptr; }
  static const float *dinv(const MGLevel &l) { return l.dinv32.ptr; }
  static float *b(MGLevel &l) { return l.b32.ptr; }
  static float *x(MGLevel &l) { return l.x32.ptr; }
  static float *r(MGLevel &l) { return l.r32.ptr; }
  static float *d(MGLevel &l) { return l.d32.ptr; }
  static const float *cinv(const _p_dohpMG *m) { return m->cinv32.ptr; }
};

// Coefficients of the Chebyshev smoother of the given degree on [lo, hi] * lmax: step k (from 0) is
// d = a_k d + c_k D^-1 (b - A x), x += d (a_0 = 0).
struct ChebCoeffs {
  double theta, delta, sigma, rho;
  ChebCoeffs(const _p_dohpMG *mg, const MGLevel &lv)
  {
    const double lmin = mg->lo * lv.lmax, lmax = mg->hi * lv.lmax;
    theta = 0.5 * (lmax + lmin);
    delta = 0.5 * (lmax - lmin);
    sigma = theta / delta;
    rho = 1.0 / sigma;
  }
  void step(int k, double &a, double &c)
  {
    a = 0.0;
    c = 1.0 / theta;
    if (k == 0) return;
    const double rho_new = 1.0 / (2.0 * sigma - rho);
    a = rho_new * rho;
    c = 2.0 * rho_new / delta;
    rho = rho_new;
  }
};

// The V-cycle at level l.  The first two pre-smoothing steps from zero are one sweep (at degree 1 the first step and the
// residual are), and the first post-smoothing step takes the prolongation.  Every later step moves the iterate between x
// and the level's residual vector; it starts where the moves end in x.
template <typename T>
void vcycle(_p_dohpMG *mg, size_t l, const T *b, T *x, hipStream_t st)
{
  using P = LvPtr<T>;
  MGLevel &lv = mg->L[l];
  if (l + 1 == mg->L.size()) {
    hipLaunchKernelGGL(dense_mv_kernel<T>, dim3((unsigned)((lv.n + 3) / 4)), dim3(256), 0, st, (int)lv.n,
                       P::cinv(mg), b, x);
    return;
  }
  MGLevel &cv = mg->L[l + 1];
  const T *H = P::A(lv), *dinv = P::dinv(lv);
  T *d = P::d(lv), *cur = x, *other = P::r(lv);
  if (mg->degree == 1) std::swap(cur, other);
  double a, c, c1;
  ChebCoeffs pre(mg, lv);
  pre.step(0, a, c1);
  const bool pair = sizeof(T) == 8 && mg->degree == 2 && pair_level<double>(lv.box, 2);
  PairArgs<double> pa{};
  if (pair) {
    pre.step(1, a, c);
    pa = PairArgs<double>{lv.box, cv.box, pair_tiles<double>(lv.box, kPairSlots), lv.H, lv.dinv64.ptr, nullptr,
                          (const double *)b, nullptr, cv.x64.ptr, lv.d64.ptr, lv.r64.ptr, c1, a, c};
    pair_sweep<double, PAIR_PRE>(pa, st);
  } else if (mg->degree == 1) {
    sweep<T, SW_FIRST_RESID>(lv.box, H, dinv, b, nullptr, other, nullptr, cur, T(0), T(0), (T)c1, 0, st);
  } else {
    for (int k = 1; k < mg->degree; k++) {
      pre.step(k, a, c);
      const int keep_d = k + 1 < mg->degree;
      if (k == 1) {
        sweep<T, SW_FIRST_CHEB>(lv.box, H, dinv, b, nullptr, cur, d, nullptr, (T)a, (T)c, (T)c1, keep_d, st);
      } else {
        sweep<T, SW_CHEB>(lv.box, H, dinv, b, cur, other, d, nullptr, (T)a, (T)c, T(0), keep_d, st);
        std::swap(cur, other);
      }
    }
    residual<T>(lv.box, H, b, cur, other, st);
  }
  restrict_to<T>(lv.box, cv.box, other, P::b(cv), nullptr, st);
  vcycle<T>(mg, l + 1, P::b(cv), P::x(cv), st);
  ChebCoeffs post(mg, lv);
  if (pair) {
    post.step(0, a, c1);
    post.step(1, a, c);
    pa.x = lv.d64.ptr;
    pa.out = (double *)x;
    pa.c1 = c1;
    pa.a = a;
    pa.c = c;
    pair_sweep<double, PAIR_POST>(pa, st);
    return;
  }
  for (int k = 0; k < mg->degree; k++) {
    post.step(k, a, c);
    const int keep_d = k + 1 < mg->degree;
    if (k == 0)
      sweep<T, SW_PRO_CHEB>(lv.box, H, dinv, b, cur, other, d, nullptr, (T)a, (T)c, T(0), keep_d, st, cv.box, P::x(cv));
    else
      sweep<T, SW_CHEB>(lv.box, H, dinv, b, cur, other, d, nullptr, (T)a, (T)c, T(0), keep_d, st);
    std::swap(cur, other);
  }
}

// The tile of the FP16 sweeps: two planes of 64 x 4 rows from 8 million rows on, where the level's 48 bytes a row
// (384 MB) stream from HBM and the fewer staged loads show (a sweep of 239^3 rows 162 against 166 us, 207^3: 115 against
// 118), one plane below, where the level lives in the 256 MB cache (191^3: 78 against 82 us, 95^3: 15.0 against 15.6).
// Levels of that size come here at smoothing degrees of 3 and more; at 1 and 2 they march (pair_level).
template <int MODE>
void sweep16(const MGLevel &lv, const float *b, const float *y, float *out, float *y1, double a, double c, double c1,
             int keep_d, int raw, int unscale, hipStream_t st, const Box &cb = Box{}, const float *xc = nullptr)
{
  const Box &bx = lv.box;
  const auto launch = [&](auto kernel, int BY, int NR) {
    const Split sp = split_of(bx, BY);
    hipLaunchKernelGGL(kernel, split_grid(bx, sp, BY, NR), dim3(kBX, BY), 0, st, bx, sp, lv.H16.ptr, lv.e16.ptr,
                       lv.f16.ptr, lv.sc16.ptr, b, y, out, lv.d32.ptr, y1, lv.t32.ptr, (float)a, (float)c, (float)c1,
                       keep_d, raw, unscale, cb, xc);
  };
  if (lv.n >= 8000000)
    launch(half16_sweep_kernel<MODE, 4, 2>, 4, 2);
  else
    launch(half16_sweep_kernel<MODE, 4, 1>, 4, 1);
}

// FP32 V-cycle on the FP16 coefficients, in the scaled variables: b is b' on the coarse levels (the restriction scales
// it) and the caller's on the finest; the result x is unscaled on every level.  Steps and buffers as in vcycle.
void vcycle16(_p_dohpMG *mg, size_t l, const float *b, float *x, hipStream_t st)
{
  MGLevel &lv = mg->L[l];
  if (l + 1 == mg->L.size()) {
    hipLaunchKernelGGL(dense_mv_kernel<float>, dim3((unsigned)((lv.n + 3) / 4)), dim3(256), 0, st, (int)lv.n,
                       mg->cinv32.ptr, b, x);
    return;
  }
  MGLevel &cv = mg->L[l + 1];
  const int raw = l == 0;
  const float *bs = raw ? lv.t32.ptr : b;
  float *cur = x, *other = lv.r32.ptr;
  if (mg->degree == 1) std::swap(cur, other);
  double a, c, c1;
  ChebCoeffs pre(mg, lv);
  pre.step(0, a, c1);
  const bool two = mg->degree == 2, pair = pair_level<float>(lv.box, mg->degree);
  PairArgs<float> pa{};
  if (pair) {
    if (two) pre.step(1, a, c);
    else a = c = 0;
    other = lv.r32.ptr;
    pa = PairArgs<float>{lv.box, cv.box, pair_tiles<float>(lv.box, kPairSlots, two), lv.H16.ptr, lv.e16.ptr,
                         lv.sc16.ptr, b, nullptr, cv.x32.ptr, lv.d32.ptr, lv.r32.ptr, (float)c1, (float)a, (float)c,
                         raw, 1};
    if (two) pair_sweep<float, PAIR_PRE>(pa, st);
    else pair_sweep<float, PAIR_PRE1>(pa, st);
  } else if (mg->degree == 1) {
    sweep16<SW_FIRST_RESID>(lv, b, nullptr, other, cur, 0, 0, c1, 0, raw, 0, st);
  } else {
    for (int k = 1; k < mg->degree; k++) {
      pre.step(k, a, c);
      const int keep_d = k + 1 < mg->degree;
      if (k == 1) {
        sweep16<SW_FIRST_CHEB>(lv, b, nullptr, cur, nullptr, a, c, c1, keep_d, raw, 0, st);
      } else {
        sweep16<SW_CHEB>(lv, bs, cur, other, nullptr, a, c, 0, keep_d, 0, 0, st);
        std::swap(cur, other);
      }
    }
    sweep16<SW_RESID>(lv, bs, cur, other, nullptr, 0, 0, 0, 0, 0, 0, st);
  }
  restrict_to<float>(lv.box, cv.box, other, cv.b32.ptr, l + 2 < mg->L.size() ? cv.sc16.ptr : nullptr, st);
  vcycle16(mg, l + 1, cv.b32.ptr, cv.x32.ptr, st);
  ChebCoeffs post(mg, lv);
  if (pair) {
    post.step(0, a, c1);
    if (two) post.step(1, a, c);
    pa.x = lv.d32.ptr;
    pa.out = x;
    pa.c1 = (float)c1;
    pa.a = (float)a;
    pa.c = (float)c;
    if (two) pair_sweep<float, PAIR_POST>(pa, st);
    else pair_sweep<float, PAIR_POST1>(pa, st);
    return;
  }
  for (int k = 0; k < mg->degree; k++) {
    post.step(k, a, c);
    const int last = k + 1 == mg->degree;
    if (k == 0)
      sweep16<SW_PRO_CHEB>(lv, bs, cur, other, nullptr, a, c, 0, !last, 0, last, st, cv.box, cv.x32.ptr);
    else
      sweep16<SW_CHEB>(lv, bs, cur, other, nullptr, a, c, 0, !last, 0, last, st);
    std::swap(cur, other);
  }
}

}  // namespace

namespace {

// The operators of every level from the finest level's stencil (L[0].A64): Galerkin products, half stencils in FP64,
// FP32 and FP16, Jacobi scalings, eigenvalue estimates and the coarsest level's inverse, into the hierarchy's buffers.
dErr mg_fill(_p_dohpMG *mg, hipStream_t st)
{
  mg->drop_graphs();  // their kernels carry this hierarchy's smoothing coefficients
  for (size_t l = 1; l < mg->L.size(); l++) {
    const MGLevel &f = mg->L[l - 1];
    MGLevel &c = mg->L[l];
    const int part = (c.box.ny + 7) / 8;
    hipLaunchKernelGGL(rap_kernel, dim3(8u * (unsigned)(((long)part * c.box.nz + 63) / 64), (unsigned)c.box.nx),
                       dim3(576), 0, st, f.box, c.box, part, f.A64, c.own64.ptr);
  }
  for (size_t l = 0; l < mg->L.size(); l++) {
    MGLevel &lv = mg->L[l];
    const long n = lv.n;
    const bool smoothed = l + 1 < mg->L.size();
    hipLaunchKernelGGL(diag_kernel, grid_of(n), dim3(256), 0, st, n, lv.A64, lv.dinv64.ptr, lv.dinv32.ptr,
                       smoothed ? lv.sc16.ptr : nullptr);
    if (smoothed) {
      const Split sp = split_of(lv.box, kBY);
      hipLaunchKernelGGL(half_setup_kernel, split_grid(lv.box, sp, kBY, 1), box_block(), 0, st, lv.box, sp, lv.A64,
                         lv.H64.ptr, lv.H32.ptr, lv.H16.ptr, lv.dg16.ptr, lv.sc16.ptr, lv.e16.ptr, lv.f16.ptr, l > 0);
    } else {
      hipLaunchKernelGGL(half_from_full_kernel, grid_of(n), dim3(256), 0, st, n, lv.A64, lv.H64.ptr, lv.H32.ptr);
    }
    lv.H = lv.H64.ptr ? lv.H64.ptr : lv.A64 + 13 * n;
  }
  DOHP_CALL(estimate_lmax(mg, st, 15));
  DOHP_CALL(coarse_inverse(mg, st));
  // one read of the eigenvalue estimates and the inverse's flag
  const size_t nl = mg->L.size() - 1;
  double h[kMaxLevels + 1] = {};
  if (nl) DOHP_HIP(hipMemcpyAsync(h, mg->part.ptr, sizeof(double) * nl, hipMemcpyDeviceToHost, st));
  DOHP_HIP(hipMemcpyAsync(h + kMaxLevels, mg->cwork.ptr, sizeof(double), hipMemcpyDeviceToHost, st));
  if (hipStreamSynchronize(st) != hipSuccess) {
    set_error("multigrid setup failed");
    return dohpERR_HIP;
  }
  for (size_t l = 0; l < nl; l++) mg->L[l].lmax = h[l];
  DOHP_CHECK(h[kMaxLevels] == 0.0, dohpERR_GENERIC, "multigrid: coarsest matrix is not positive definite");
  mg->ncoarse = (int)mg->L.back().n;
  return 0;
}

}  // namespace

// The places for block sums that the power iterations keep for a level of nx x ny x nz rows, and the sums that a sweep and
// a pair of sweeps write (0: the level takes no pairs).
extern "C" dErr dohpMGPowerSums_Private(int nx, int ny, int nz, long *places, long *single, long *pair)
{
  const Box b{nx, ny, nz};
  const dim3 g = power_grid(b);
  *places = power_sums(b);
  *single = (long)g.x * g.y * g.z;
  *pair = pair_level<double>(b, 2) ? pair_tiles<double>(b, kPairSlots).blocks() : 0;
  return 0;
}

extern "C" dErr dohpMGCreate(dohpMat q1, int smooth_degree, int max_coarse, dohpMG *out, void *stream)
{
  DOHP_CHECK(q1 && out, dohpERR_ARG, "null argument");
  DOHP_CHECK(q1->st64.ptr, dohpERR_ARG, "multigrid needs the stencil form of a block-space Q1 matrix");
  hipStream_t st = (hipStream_t)stream;
  *out = nullptr;
  _p_dohpMG *mg = new _p_dohpMG;
  mg->degree = smooth_degree > 0 ? smooth_degree : 2;
  const long nmax = max_coarse > 0 ? max_coarse : 512;
  dErr err = 0;
  {
    MGLevel lv;
    lv.box = Box{q1->box[0], q1->box[1], q1->box[2]};
    lv.n = lv.box.n();
    lv.A64 = q1->st64.ptr;
    mg->L.push_back(std::move(lv));
  }
  while (!err) {
    MGLevel &f = mg->L.back();
    if (f.n <= nmax) break;
    const Box cb{f.box.nx / 2, f.box.ny / 2, f.box.nz / 2};
    if (cb.nx < 1 || cb.ny < 1 || cb.nz < 1) break;
    MGLevel c;
    c.box = cb;
    c.n = cb.n();
    err = c.own64.alloc(27 * c.n);
    if (err) break;
    c.A64 = c.own64.ptr;
    mg->L.push_back(std::move(c));
  }
  if (!err && mg->L.back().n > kMaxCoarse) {  // (a plate: refused before anything is launched)
    set_error("multigrid: the coarsest level is too large for a direct solve");
    err = dohpERR_ARG;
  }
  for (size_t l = 0; !err && l < mg->L.size(); l++) {
    MGLevel &lv = mg->L[l];
    const long n = lv.n;
    err = lv.dinv64.alloc(n);
    if (!err) err = lv.dinv32.alloc(n);
    if (!err && l == 0) err = lv.H64.alloc(14 * n);  // (the matrix may be refilled or freed before the hierarchy)
    if (!err) err = lv.H32.alloc(14 * n);
    if (!err) err = lv.r64.alloc(n);
    if (!err) err = lv.d64.alloc(n);
    if (!err) err = lv.r32.alloc(n);
    if (!err) err = lv.d32.alloc(n);
    if (!err && l > 0) err = lv.b64.alloc(n);
    if (!err && l > 0) err = lv.x64.alloc(n);
    if (!err && l > 0) err = lv.b32.alloc(n);
    if (!err && l > 0) err = lv.x32.alloc(n);
    if (!err && l + 1 < mg->L.size()) err = lv.H16.alloc(14 * n);
    if (!err && l + 1 < mg->L.size()) err = lv.dg16.alloc(n);
    if (!err && l + 1 < mg->L.size()) err = lv.sc16.alloc(n);
    if (!err && l + 1 < mg->L.size()) err = lv.e16.alloc(n);
    if (!err && l + 1 < mg->L.size()) err = lv.f16.alloc(n);
    if (!err && l == 0 && mg->L.size() > 1) err = lv.t32.alloc(n);
  }
  if (!err && pair_level<double>(mg->L[0].box, 2)) {
    for (const void *k : {(const void *)pair_kernel<double, PAIR_POWER>, (const void *)pair_kernel<double, PAIR_PRE>,
                          (const void *)pair_kernel<double, PAIR_POST>})
      if (!err && hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, pair_lds<double>()) != hipSuccess) {
        set_error("multigrid: the sweeps' LDS is not available");
        err = dohpERR_HIP;
      }
  }
  if (!err) err = mg_fill(mg, st);
  if (err) {
    delete mg;
    return err;
  }
  *out = mg;
  return 0;
}

extern "C" dErr dohpMGRefresh(dohpMG mg, dohpMat q1, void *stream)
{
  DOHP_CHECK(mg && q1, dohpERR_ARG, "null argument");
  DOHP_CHECK(q1->st64.ptr, dohpERR_ARG, "multigrid needs the stencil form of a block-space Q1 matrix");
  const Box &b = mg->L[0].box;
  DOHP_CHECK(q1->box[0] == b.nx && q1->box[1] == b.ny && q1->box[2] == b.nz, dohpERR_ARG,
             "multigrid refresh needs a matrix on the same box");
  mg->L[0].A64 = q1->st64.ptr;
  return mg_fill(mg, (hipStream_t)stream);
}

extern "C" dErr dohpMGGetInfo(dohpMG mg, int *nlevels, long *ncoarse, double *lmax_fine)
{
  DOHP_CHECK(mg, dohpERR_ARG, "null multigrid");
  if (nlevels) *nlevels = (int)mg->L.size();
  if (ncoarse) *ncoarse = mg->ncoarse;
  if (lmax_fine) *lmax_fine = mg->L[0].lmax;
  return 0;
}

extern "C" dErr dohpMGGetLevel(dohpMG mg, int level, int *box, double *stencil_host)
{
  DOHP_CHECK(mg && level >= 0 && level < (int)mg->L.size(), dohpERR_ARG, "no such multigrid level");
  const MGLevel &lv = mg->L[level];
  if (box) {
    box[0] = lv.box.nx;
    box[1] = lv.box.ny;
    box[2] = lv.box.nz;
  }
  if (stencil_host) {
    DOHP_HIP(hipDeviceSynchronize());
    DOHP_HIP(hipMemcpy(stencil_host, lv.A64, sizeof(double) * 27 * lv.n, hipMemcpyDeviceToHost));
  }
  return 0;
}

namespace {

// Applies the V-cycle `run(stream)` for vectors (r, z): replays the graph captured for them; the second consecutive
// application to the same vectors captures it (a Krylov loop applies its preconditioner to the same work vectors
// every iteration; one-off applications stay eager).  A capture that fails leaves the hierarchy on eager launches.
template <class Run>
dErr vcycle_graph(_p_dohpMG *mg, _p_dohpMG::Graph &g, const void *r, void *z, hipStream_t st, Run run)
{
  const bool same = g.r == r && g.z == z && g.coeff16 == mg->coeff16;
  if (!mg->graphs || !same) {
    if (g.exec) (void)hipGraphExecDestroy(g.exec);
    g = _p_dohpMG::Graph{};
    g.r = r;
    g.z = z;
    g.coeff16 = mg->coeff16;
    run(st);
    DOHP_HIP(hipGetLastError());
    return 0;
  }
  if (!g.exec) {
    if (!mg->cap) DOHP_HIP(hipStreamCreateWithFlags(&mg->cap, hipStreamNonBlocking));
    hipGraph_t graph = nullptr;
    bool ok = hipStreamBeginCapture(mg->cap, hipStreamCaptureModeThreadLocal) == hipSuccess;
    if (ok) {
      run(mg->cap);
      ok = hipStreamEndCapture(mg->cap, &graph) == hipSuccess && graph;
    }
    if (ok) ok = hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0) == hipSuccess;
    if (graph) (void)hipGraphDestroy(graph);
    if (!ok) {  // eager from now on
      (void)hipGetLastError();
      if (g.exec) (void)hipGraphExecDestroy(g.exec);
      g = _p_dohpMG::Graph{};
      mg->graphs = 0;
      run(st);
      DOHP_HIP(hipGetLastError());
      return 0;
    }
  }
  DOHP_HIP(hipGraphLaunch(g.exec, st));
  return 0;
}

}  // namespace

extern "C" dErr dohpMGApply(dohpMG mg, const double *r, double *z, void *stream)
{
  DOHP_CHECK(mg && r && z, dohpERR_ARG, "null argument");
  return vcycle_graph(mg, mg->g64, r, z, (hipStream_t)stream,
                      [&](hipStream_t s) { vcycle<double>(mg, 0, r, z, s); });
}

extern "C" dErr dohpMGSetGraphs(dohpMG mg, int on)
{
  DOHP_CHECK(mg && (on == 0 || on == 1), dohpERR_ARG, "graphs must be 0 (eager launches) or 1");
  mg->drop_graphs();
  mg->graphs = on;
  return 0;
}

extern "C" dErr dohpMGApplyF32(dohpMG mg, const float *r, float *z, void *stream)
{
  DOHP_CHECK(mg && r && z, dohpERR_ARG, "null argument");
  return vcycle_graph(mg, mg->g32, r, z, (hipStream_t)stream, [&](hipStream_t s) {
    if (mg->coeff16 && mg->L.size() > 1)
      vcycle16(mg, 0, r, z, s);
    else
      vcycle<float>(mg, 0, r, z, s);
  });
}

extern "C" dErr dohpMGResidual(dohpMG mg, int level, const double *b, const double *x, double *r, void *stream)
{
  DOHP_CHECK(mg && level >= 0 && level < (int)mg->L.size(), dohpERR_ARG, "no such multigrid level");
  DOHP_CHECK(x && r, dohpERR_ARG, "null argument");
  const MGLevel &lv = mg->L[level];
  residual<double>(lv.box, lv.H, b, x, r, (hipStream_t)stream);
  DOHP_HIP(hipGetLastError());
  return 0;
}

extern "C" dErr dohpMGResidualF32(dohpMG mg, int level, const float *b, const float *x, float *r, void *stream)
{
  DOHP_CHECK(mg && level >= 0 && level < (int)mg->L.size(), dohpERR_ARG, "no such multigrid level");
  DOHP_CHECK(x && r, dohpERR_ARG, "null argument");
  const MGLevel &lv = mg->L[level];
  residual<float>(lv.box, lv.H32.ptr, b, x, r, (hipStream_t)stream);
  DOHP_HIP(hipGetLastError());
  return 0;
}

extern "C" dErr dohpMGResidualF16(dohpMG mg, int level, const float *b, const float *x, float *r, void *stream)
{
  DOHP_CHECK(mg && level >= 0 && level + 1 < (int)mg->L.size(), dohpERR_ARG,
             "no FP16 coefficients on this multigrid level (the coarsest is solved directly)");
  DOHP_CHECK(x && r, dohpERR_ARG, "null argument");
  const MGLevel &lv = mg->L[level];
  hipLaunchKernelGGL(half16_residual_kernel, box_grid(lv.box), box_block(), 0, (hipStream_t)stream, lv.box,
                     lv.H16.ptr, lv.dg16.ptr, lv.sc16.ptr, b, x, r);
  DOHP_HIP(hipGetLastError());
  return 0;
}

extern "C" dErr dohpMGSetCoefficients(dohpMG mg, int fp16)
{
  DOHP_CHECK(mg && (fp16 == 0 || fp16 == 1), dohpERR_ARG, "coefficients must be 0 (FP32) or 1 (FP16)");
  mg->coeff16 = fp16;
  return 0;
}

extern "C" dErr dohpMGDestroy(dohpMG *mg)
{
  if (mg && *mg) {
    delete *mg;
    *mg = nullptr;
  }
  return 0;
}

// FP64 kernels of the pressure solve (reference-semantics path).
//
// Built with -ffp-contract=off: every product and sum is rounded separately, in the order the
// reference writes it, so the GPU path and a scalar CPU evaluation of the same formulas agree
// to the last bit wherever the summation order is the same (stencil rows, transfers, line
// solves, Galerkin products).  Reductions are two-stage and deterministic (fixed partition,
// fixed combination order), but their order differs from a sequential sum.
//
// Index convention (reference ls_stag_uniform_mesh.h:174-185): num = x + N*y + N*M*z.

#include "lsx_kernels.hpp"
#include "lsx_lu.hpp"
#include "lsx_rows.hpp"

#include <algorithm>
#include <cmath>

namespace lsx {

namespace {

constexpr double PLUS_TINY = 1e-16;        // ls_stag_real_constants.h:27
constexpr double EQ_DOUBLE = 1e-5;         // :28
constexpr double EQ_TINY2_DOUBLE = 1e-5;   // :30
constexpr double EQ_TINY_DOUBLE = 1e-12;   // :31
constexpr double EQ_TINY3_DOUBLE = 1e-13;  // :32

inline int div_up(long a, long b) { return (int)((a + b - 1) / b); }

// ---- deterministic block reduction ------------------------------------------------------------
template <int BS>
__device__ double block_sum(double v) {
  __shared__ double lds[BS / 64];
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) lds[wave] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < BS / 64; ++w) s += lds[w];
  __syncthreads();
  return s;  // valid in thread 0
}

template <int BS>
__device__ double block_max(double v) {
  __shared__ double lds[BS / 64];
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_down(v, off, 64));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) lds[wave] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < BS / 64; ++w) s = fmax(s, lds[w]);
  __syncthreads();
  return s;
}

// ---- stencil geometry helpers -------------------------------------------------------------
// One thread per cell for the plain stencil products: 256-thread blocks of 64 x by 4 y cells,
// blocks x fastest, then y, then z (tile_blocks of them).  The cell of this thread, false past the
// grid's edge.  No per-cell division, and each row's loads in flight together (measured 139 us
// against 156 us for 4096-cell chunks walked by 256 threads at 256^3).
__device__ inline bool tile_cell(int N, int M, int* x, int* y, int* z) {
  const int gx = (N + 63) / 64, gy = (M + 3) / 4;
  const int bx = (int)(blockIdx.x % gx), r = (int)(blockIdx.x / gx);
  *x = bx * 64 + (int)(threadIdx.x & 63);
  *y = (r % gy) * 4 + (int)(threadIdx.x >> 6);
  *z = r / gy;
  return *x < N && *y < M;
}

__device__ inline void decode(int i, int N, int M, int* x, int* y, int* z) {
  const int NM = N * M;
  *z = i / NM;
  const int r = i - *z * NM;
  *y = r / N;
  *x = r - *y * N;
}

// The cell of this thread in the one-cell-per-thread kernels: rows of at least 64 cells by tiles
// (tile_cell), shorter ones, which would leave most of a tile's lanes idle, in index order.
__device__ inline bool own_cell(int N, int M, int K, int* x, int* y, int* z) {
  if (N >= 64) return tile_cell(N, M, x, y, z);
  const unsigned i = blockIdx.x * 256u + threadIdx.x;
  if (i >= (unsigned)N * M * K) return false;
  decode((int)i, N, M, x, y, z);
  return true;
}

__host__ __device__ inline int slot_sub(int npts, int dir) {  // coupling to the previous cell of a line
  if (npts == 7) return dir == 0 ? 2 : (dir == 1 ? 1 : 0);
  return dir == 0 ? 12 : (dir == 1 ? 10 : 4);
}
__device__ inline int slot_super(int npts, int dir) {  // coupling to the next cell of a line
  if (npts == 7) return dir == 0 ? 4 : (dir == 1 ? 5 : 6);
  return dir == 0 ? 14 : (dir == 1 ? 16 : 22);
}
__device__ inline int slot_diag(int npts) { return npts == 7 ? 3 : 13; }

// Row i of the operator applied to x, accumulated in ascending column order (the CSR order
// of the reference matrices: [b,s,w,p,e,n,t] on the fine level, sorted columns on Galerkin
// levels).  acc starts at the given value; subtract: terms are subtracted.  Straight-line code: an
// absent neighbour, whose coefficient is stored as 0, reads the cell itself, so that all loads of
// a row are in flight together (a branch per term would wait for each).  ABSENT0: it counts as 0 whatever
// is there, since 0 times an infinite value is NaN.  The smoother's products go without (1 to 2 % of a
// cascade application): the line solves make NaN of an infinite correction in any case.
template <int NPTS, bool ABSENT0 = true>
__device__ inline double row_apply(const double* __restrict__ coef, long n, int i, int x, int y, int z, int N, int M,
                                   int K, const double* __restrict__ xv, double acc, bool subtract) {
  const int ox[3] = {x > 0 ? -1 : 0, 0, x < N - 1 ? 1 : 0};
  const int oy[3] = {y > 0 ? -N : 0, 0, y < M - 1 ? N : 0}, oz[3] = {z > 0 ? -N * M : 0, 0, z < K - 1 ? N * M : 0};
  double a[NPTS], v[NPTS];
#pragma unroll
  for (int q = 0; q < NPTS; ++q) {
    const int p = NPTS == 27 ? q : (const int[7]){4, 10, 12, 13, 14, 16, 22}[q];
    a[q] = coef[q * n + i];
    v[q] = xv[i + ox[p % 3] + oy[p / 3 % 3] + oz[p / 9]];
  }
  if constexpr (ABSENT0) {
    const bool hx[3] = {x > 0, true, x < N - 1}, hy[3] = {y > 0, true, y < M - 1}, hz[3] = {z > 0, true, z < K - 1};
#pragma unroll
    for (int q = 0; q < NPTS; ++q) {
      const int p = NPTS == 27 ? q : (const int[7]){4, 10, 12, 13, 14, 16, 22}[q];
      v[q] = hx[p % 3] && hy[p / 3 % 3] && hz[p / 9] ? v[q] : 0.0;
    }
  }
#pragma unroll
  for (int q = 0; q < NPTS; ++q) acc = subtract ? acc - a[q] * v[q] : acc + a[q] * v[q];
  return acc;
}

// ---- kernels: setup ----------------------------------------------------------------------------
__global__ void k_csr_to_stencil7(const int* __restrict__ rowptr, const int* __restrict__ col,
                                  const double* __restrict__ val, int N, int M, int K, double* __restrict__ coef,
                                  int* err) {
  const long n = (long)N * M * K;
  const int NM = N * M;
  for (long li = blockIdx.x * (long)blockDim.x + threadIdx.x; li < n; li += (long)gridDim.x * blockDim.x) {
    const int i = (int)li;
    int x, y, z;
    decode(i, N, M, &x, &y, &z);
    double a[7] = {0, 0, 0, 0, 0, 0, 0};
    unsigned seen = 0;
    for (int j = rowptr[i]; j < rowptr[i + 1]; ++j) {
      const int off = col[j] - i;
      int q = -1;
      if (off == -NM && z > 0) q = 0;
      else if (off == -N && y > 0) q = 1;
      else if (off == -1 && x > 0) q = 2;
      else if (off == 0) q = 3;
      else if (off == 1 && x < N - 1) q = 4;
      else if (off == N && y < M - 1) q = 5;
      else if (off == NM && z < K - 1) q = 6;
      if (q < 0) {
        atomicOr(err, 1);
      } else if (seen & (1u << q)) {  // a repeated column would drop a term
        atomicOr(err, 2);
      } else {
        seen |= 1u << q;
        a[q] = val[j];
      }
    }
#pragma unroll
    for (int q = 0; q < 7; ++q) coef[q * n + i] = a[q];
  }
}

// Galerkin product A_c = R (A_f P): coarse_grid.h:103-104 with product_sparse_matrix.h:72-104.
// Terms reach each entry in the reference order: V = R A_f accumulates over the 8 children in
// R's column order, then A_c accumulates V's fine columns in ascending order.
__device__ inline void axis_w(int f, int nf, int* c, double* w, int* cnt) {
  const int p = f >> 1;
  if (f == 0 || f == nf - 1) {
    c[0] = p; w[0] = 1.0; *cnt = 1;
  } else if (f & 1) {
    c[0] = p; w[0] = 0.75; c[1] = p + 1; w[1] = 0.25; *cnt = 2;
  } else {
    c[0] = p - 1; w[0] = 0.25; c[1] = p; w[1] = 0.75; *cnt = 2;
  }
}

template <int NPTS>
__global__ void k_galerkin(const double* __restrict__ cf, int Nf, int Mf, int Kf, double* __restrict__ cc, int Nc,
                           int Mc, int Kc) {
  const long nc = (long)Nc * Mc * Kc, nf = (long)Nf * Mf * Kf;
  const int NMf = Nf * Mf;
  for (long li = blockIdx.x * (long)blockDim.x + threadIdx.x; li < nc; li += (long)gridDim.x * blockDim.x) {
    const int I = (int)li;
    int X, Y, Z;
    decode(I, Nc, Mc, &X, &Y, &Z);
    double V[64];
#pragma unroll
    for (int q = 0; q < 64; ++q) V[q] = 0.0;
    for (int ch = 0; ch < 8; ++ch) {
      const int hx = 2 * X + (ch & 1), hy = 2 * Y + ((ch >> 1) & 1), hz = 2 * Z + (ch >> 2);
      const int h = hx + Nf * hy + NMf * hz;
      if (NPTS == 7) {
        const int dxs[7] = {0, 0, -1, 0, 1, 0, 0}, dys[7] = {0, -1, 0, 0, 0, 1, 0}, dzs[7] = {-1, 0, 0, 0, 0, 0, 1};
        for (int q = 0; q < 7; ++q) {
          const int fx = hx + dxs[q], fy = hy + dys[q], fz = hz + dzs[q];
          if (fx < 0 || fx >= Nf || fy < 0 || fy >= Mf || fz < 0 || fz >= Kf) continue;
          const int b = (fx - 2 * X + 1) + 4 * (fy - 2 * Y + 1) + 16 * (fz - 2 * Z + 1);
          V[b] = V[b] + 0.125 * cf[q * nf + h];
        }
      } else {
        for (int q = 0; q < 27; ++q) {
          const int dx = q % 3 - 1, dy = (q / 3) % 3 - 1, dz = q / 9 - 1;
          const int fx = hx + dx, fy = hy + dy, fz = hz + dz;
          if (fx < 0 || fx >= Nf || fy < 0 || fy >= Mf || fz < 0 || fz >= Kf) continue;
          const int b = (fx - 2 * X + 1) + 4 * (fy - 2 * Y + 1) + 16 * (fz - 2 * Z + 1);
          V[b] = V[b] + 0.125 * cf[q * nf + h];
        }
      }
    }
    double A[27];
#pragma unroll
    for (int q = 0; q < 27; ++q) A[q] = 0.0;
    for (int b = 0; b < 64; ++b) {
      const int fx = 2 * X - 1 + (b & 3), fy = 2 * Y - 1 + ((b >> 2) & 3), fz = 2 * Z - 1 + (b >> 4);
      if (fx < 0 || fx >= Nf || fy < 0 || fy >= Mf || fz < 0 || fz >= Kf) continue;
      int cx[2], cy[2], cz[2], nx, ny, nz;
      double wx[2], wy[2], wz[2];
      axis_w(fx, Nf, cx, wx, &nx);
      axis_w(fy, Mf, cy, wy, &ny);
      axis_w(fz, Kf, cz, wz, &nz);
      const double v = V[b];
      for (int c3 = 0; c3 < nz; ++c3)
        for (int c2 = 0; c2 < ny; ++c2)
          for (int c1 = 0; c1 < nx; ++c1) {
            const double w = wx[c1] * wy[c2] * wz[c3];
            const int q = (cx[c1] - X + 1) + 3 * (cy[c2] - Y + 1) + 9 * (cz[c3] - Z + 1);
            A[q] = A[q] + v * w;
          }
    }
#pragma unroll
    for (int q = 0; q < 27; ++q) cc[q * nc + I] = A[q];
  }
}

// ---- odd-odd-odd transfers (transfer_operators_odd_odd_odd.h:44-100, R = P^T by
// transfer_operators_interface.h:572-578 and transposed_sparse_matrix.h:47-68) --------------------
// An odd axis of 2n - 1 fine cells coarsens to n cells centred on the even fine cells: P weights
// 1 on a coincident fine cell, 1/2 on each coarse neighbour of an odd fine cell; a row's entries
// run z, then y, then x, coarse index ascending.  R row C lists fine cells 2C - 1, 2C, 2C + 1 per
// axis (weights 1/2, 1, 1/2, those inside the level) in ascending fine index.
__device__ inline void axis_w_odd(int f, int* c, double* w, int* cnt) {
  if ((f & 1) == 0) {
    c[0] = f >> 1; w[0] = 1.0; *cnt = 1;
  } else {
    c[0] = (f - 1) >> 1; w[0] = 0.5; c[1] = (f + 1) >> 1; w[1] = 0.5; *cnt = 2;
  }
}
__device__ inline int axis_r_odd(int C, int nf, int* f, double* w) {
  int n = 0;
  if (2 * C - 1 >= 0) { f[n] = 2 * C - 1; w[n] = 0.5; ++n; }
  f[n] = 2 * C; w[n] = 1.0; ++n;
  if (2 * C + 1 < nf) { f[n] = 2 * C + 1; w[n] = 0.5; ++n; }
  return n;
}

// Galerkin product A_c = (R A_f) P for odd-odd-odd levels, terms in the order of
// product_sparse_matrix.h:72-104: V = R A_f accumulates over R's fine cells in ascending order,
// each with its A_f row in ascending column order; A_c then accumulates V's fine columns in
// ascending order (V's window: fine cells 2C - 2 .. 2C + 2 per axis).
template <int NPTS>
__global__ void k_galerkin_odd(const double* __restrict__ cf, int Nf, int Mf, int Kf, double* __restrict__ cc,
                               int Nc, int Mc, int Kc) {
  const long nc = (long)Nc * Mc * Kc, nf = (long)Nf * Mf * Kf;
  const int NMf = Nf * Mf;
  for (long li = blockIdx.x * (long)blockDim.x + threadIdx.x; li < nc; li += (long)gridDim.x * blockDim.x) {
    const int I = (int)li;
    int X, Y, Z;
    decode(I, Nc, Mc, &X, &Y, &Z);
    double V[125];
    for (int q = 0; q < 125; ++q) V[q] = 0.0;
    int rx[3], ry[3], rz[3];
    double wx[3], wy[3], wz[3];
    const int nx = axis_r_odd(X, Nf, rx, wx), ny = axis_r_odd(Y, Mf, ry, wy), nz = axis_r_odd(Z, Kf, rz, wz);
    for (int c3 = 0; c3 < nz; ++c3)
      for (int c2 = 0; c2 < ny; ++c2)
        for (int c1 = 0; c1 < nx; ++c1) {
          const double w = wx[c1] * wy[c2] * wz[c3];
          const int hx = rx[c1], hy = ry[c2], hz = rz[c3];
          const int h = hx + Nf * hy + NMf * hz;
          for (int q = 0; q < NPTS; ++q) {
            int dx, dy, dz;
            if (NPTS == 7) {
              const int dxs[7] = {0, 0, -1, 0, 1, 0, 0}, dys[7] = {0, -1, 0, 0, 0, 1, 0}, dzs[7] = {-1, 0, 0, 0, 0, 0, 1};
              dx = dxs[q];
              dy = dys[q];
              dz = dzs[q];
            } else {
              dx = q % 3 - 1;
              dy = (q / 3) % 3 - 1;
              dz = q / 9 - 1;
            }
            const int fx = hx + dx, fy = hy + dy, fz = hz + dz;
            if (fx < 0 || fx >= Nf || fy < 0 || fy >= Mf || fz < 0 || fz >= Kf) continue;
            const int b = (fx - 2 * X + 2) + 5 * (fy - 2 * Y + 2) + 25 * (fz - 2 * Z + 2);
            V[b] = V[b] + w * cf[q * nf + h];
          }
        }
    double A[27];
    for (int q = 0; q < 27; ++q) A[q] = 0.0;
    for (int b = 0; b < 125; ++b) {
      const int fx = 2 * X - 2 + b % 5, fy = 2 * Y - 2 + (b / 5) % 5, fz = 2 * Z - 2 + b / 25;
      if (fx < 0 || fx >= Nf || fy < 0 || fy >= Mf || fz < 0 || fz >= Kf) continue;
      int cx[2], cy[2], cz[2], mx, my, mz;
      double px[2], py[2], pz[2];
      axis_w_odd(fx, cx, px, &mx);
      axis_w_odd(fy, cy, py, &my);
      axis_w_odd(fz, cz, pz, &mz);
      const double v = V[b];
      for (int c3 = 0; c3 < mz; ++c3)
        for (int c2 = 0; c2 < my; ++c2)
          for (int c1 = 0; c1 < mx; ++c1) {
            const double w = px[c1] * py[c2] * pz[c3];
            const int q = (cx[c1] - X + 1) + 3 * (cy[c2] - Y + 1) + 9 * (cz[c3] - Z + 1);
            A[q] = A[q] + v * w;
          }
    }
    for (int q = 0; q < 27; ++q) cc[q * nc + I] = A[q];
  }
}

// One coarse cell of r_c = R r_f and one fine cell of P ch_c; `at` reads a fine (coarse) cell (x, y, z).
// Straight-line code: an absent tap reads a present cell with weight 0, which leaves the sum as it
// is, so that all reads are in flight together.
// Odd-odd-odd levels: R = P^T, fine cells in ascending order.
template <class F>
__device__ inline double restrict_cell_odd(F at, int X, int Y, int Z, int Nf, int Mf, int Kf) {
  auto taps = [](int C, int nf, int (&f)[3], double (&w)[3]) {
    f[0] = C > 0 ? 2 * C - 1 : 2 * C;
    f[1] = 2 * C;
    f[2] = 2 * C + 1 < nf ? 2 * C + 1 : 2 * C;
    w[0] = C > 0 ? 0.5 : 0.0;
    w[1] = 1.0;
    w[2] = 2 * C + 1 < nf ? 0.5 : 0.0;
  };
  int fx[3], fy[3], fz[3];
  double wx[3], wy[3], wz[3], v[27];
  taps(X, Nf, fx, wx);
  taps(Y, Mf, fy, wy);
  taps(Z, Kf, fz, wz);
#pragma unroll
  for (int q = 0; q < 27; ++q) v[q] = at(fx[q % 3], fy[q / 3 % 3], fz[q / 9]);
  double acc = 0.0;
#pragma unroll
  for (int q = 0; q < 27; ++q) acc = acc + wx[q % 3] * wy[q / 3 % 3] * wz[q / 9] * v[q];
  return acc;
}

// sum of the 2 x 2 x 2 taps of a prolongation, z outermost, x innermost
template <class F>
__device__ inline double prolong_taps(F at, const int (&cx)[2], const int (&cy)[2], const int (&cz)[2],
                                      const double (&wx)[2], const double (&wy)[2], const double (&wz)[2]) {
  double v[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) v[q] = at(cx[q & 1], cy[(q >> 1) & 1], cz[q >> 2]);
  double acc = 0.0;
#pragma unroll
  for (int q = 0; q < 8; ++q) acc = acc + wx[q & 1] * wy[(q >> 1) & 1] * wz[q >> 2] * v[q];
  return acc;
}

template <class F>
__device__ inline double prolong_cell_odd(F at, int x, int y, int z) {
  auto taps = [](int f, int (&c)[2], double (&w)[2]) {  // axis_w_odd
    c[0] = f >> 1;
    c[1] = (f + 1) >> 1;
    w[0] = f & 1 ? 0.5 : 1.0;
    w[1] = f & 1 ? 0.5 : 0.0;
  };
  int cx[2], cy[2], cz[2];
  double wx[2], wy[2], wz[2];
  taps(x, cx, wx);
  taps(y, cy, wy);
  taps(z, cz, wz);
  return prolong_taps(at, cx, cy, cz, wx, wy, wz);
}

// even-even-even levels: 1/8 of each child in R's row order a,b,c,d,aa,bb,cc,dd; trilinear P
template <class F>
__device__ inline double restrict_cell(F at, int X, int Y, int Z) {
  double acc = 0.0;
#pragma unroll
  for (int q = 0; q < 8; ++q) acc = acc + 0.125 * at(2 * X + (q & 1), 2 * Y + ((q >> 1) & 1), 2 * Z + (q >> 2));
  return acc;
}

template <class F>
__device__ inline double prolong_cell(F at, int x, int y, int z, int Nf, int Mf, int Kf) {
  auto taps = [](int f, int nf, int (&c)[2], double (&w)[2]) {  // axis_w
    const int p = f >> 1;
    const bool end = f == 0 || f == nf - 1;
    c[0] = end || (f & 1) ? p : p - 1;
    c[1] = end ? p : c[0] + 1;
    w[0] = end ? 1.0 : (f & 1 ? 0.75 : 0.25);
    w[1] = end ? 0.0 : (f & 1 ? 0.25 : 0.75);
  };
  int cx[2], cy[2], cz[2];
  double wx[2], wy[2], wz[2];
  taps(x, Nf, cx, wx);
  taps(y, Mf, cy, wy);
  taps(z, Kf, cz, wz);
  return prolong_taps(at, cx, cy, cz, wx, wy, wz);
}

// r_c = R r_f (ODD: odd-odd-odd level)
template <bool ODD>
__global__ void k_restrict(const double* __restrict__ rf, int Nf, int Mf, int Kf, double* __restrict__ rc, int Nc,
                           int Mc, int Kc) {
  const long nc = (long)Nc * Mc * Kc;
  const int NMf = Nf * Mf;
  auto at = [&](int x, int y, int z) { return rf[x + Nf * y + NMf * z]; };
  for (long li = blockIdx.x * (long)blockDim.x + threadIdx.x; li < nc; li += (long)gridDim.x * blockDim.x) {
    int X, Y, Z;
    decode((int)li, Nc, Mc, &X, &Y, &Z);
    if constexpr (ODD)
      rc[li] = restrict_cell_odd(at, X, Y, Z, Nf, Mf, Kf);
    else
      rc[li] = restrict_cell(at, X, Y, Z);
  }
}

// ch_f = P ch_c, c_f = ch_f (ODD: odd-odd-odd level)
template <bool ODD>
__global__ void k_prolong(const double* __restrict__ chc, int Nc, int Mc, double* __restrict__ chf,
                          double* __restrict__ cf, int Nf, int Mf, int Kf) {
  const long nf = (long)Nf * Mf * Kf;
  const int NMc = Nc * Mc;
  auto at = [&](int x, int y, int z) { return chc[x + Nc * y + NMc * z]; };
  for (long li = blockIdx.x * (long)blockDim.x + threadIdx.x; li < nf; li += (long)gridDim.x * blockDim.x) {
    int x, y, z;
    decode((int)li, Nf, Mf, &x, &y, &z);
    double acc;
    if constexpr (ODD)
      acc = prolong_cell_odd(at, x, y, z);
    else
      acc = prolong_cell(at, x, y, z, Nf, Mf, Kf);
    chf[li] = acc;
    cf[li] = acc;
  }
}

template <int BS>
__global__ void k_diag_absmax_partial(const double* __restrict__ diag, long n, double* partial) {
  long lo, hi;
  chunk_of(n, blockIdx.x, gridDim.x, &lo, &hi);
  double m = 0.0;
  for (long i = lo + threadIdx.x; i < hi; i += BS) m = fmax(m, fabs(diag[i]));
  m = block_max<BS>(m);
  if (threadIdx.x == 0) partial[blockIdx.x] = m;
}

template <int BS>
__global__ void k_max_finalize(const double* partial, int nb, double* out) {
  double m = 0.0;
  for (int i = threadIdx.x; i < nb; i += BS) m = fmax(m, partial[i]);
  m = block_max<BS>(m);
  if (threadIdx.x == 0) out[0] = m;
}

// Line decomposition of direction dir: tridiagonal_matrix.h:45-67 (triLU) applied to the
// lines of smoother_adlj.h:40-86.  One thread per line; the zero-pivot threshold is global
// (max |diag| over the level), pivots below it are set to 0 which decouples the row.
__device__ inline void line_geometry(int t, int dir, int N, int M, int K, int* start, int* stride, int* len) {
  if (dir == 0) {  // lines (y, z)
    *start = t * N;
    *stride = 1;
    *len = N;
  } else if (dir == 1) {  // lines (x, z)
    const int x = t % N, z = t / N;
    *start = x + N * M * z;
    *stride = N;
    *len = M;
  } else {  // lines (x, y)
    *start = t;
    *stride = N * M;
    *len = K;
  }
}

__global__ void k_line_factor(const double* __restrict__ coef, int npts, int N, int M, int K, int dir,
                              const double* absmax, double* __restrict__ dinv, double* __restrict__ eu) {
  const long n = (long)N * M * K;
  const int nlines = dir == 0 ? M * K : (dir == 1 ? N * K : N * M);
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nlines) return;
  double tiny = EQ_TINY2_DOUBLE * absmax[0];
  if (tiny < EQ_TINY_DOUBLE) tiny = EQ_TINY_DOUBLE;
  int start, stride, len;
  line_geometry(t, dir, N, M, K, &start, &stride, &len);
  const double* dg = coef + slot_diag(npts) * n;
  const double* sb = coef + slot_sub(npts, dir) * n;
  const double* sp = coef + slot_super(npts, dir) * n;
  int i = start;
  double aux = dg[i];
  double dprev = (fabs(aux) < tiny) ? 0.0 : (1.0 / aux);
  dinv[i] = dprev;
  for (int k = 1; k < len; ++k) {
    const int ip = i;
    i += stride;
    const double e = sp[ip] * dprev;
    eu[ip] = e;
    aux = dg[i] - sb[i] * e;
    dprev = (fabs(aux) < tiny) ? 0.0 : (1.0 / aux);
    dinv[i] = dprev;
  }
  eu[i] = 0.0;
}

// Dense LU of the coarsest level: lu_decomposition_sparse_matrix.h:60-215 (initScalePerm,
// calcLU).  A single thread: the coarsest level has 8-16 unknowns.
__device__ inline double dense_at(const double* coef, int n, int N, int M, int K, int i, int j) {
  int xi, yi, zi, xj, yj, zj;
  decode(i, N, M, &xi, &yi, &zi);
  decode(j, N, M, &xj, &yj, &zj);
  const int dx = xj - xi, dy = yj - yi, dz = zj - zi;
  if (dx < -1 || dx > 1 || dy < -1 || dy > 1 || dz < -1 || dz > 1) return 0.0;
  return coef[((dx + 1) + 3 * (dy + 1) + 9 * (dz + 1)) * (long)n + i];
}

__global__ void k_lu_factor(const double* __restrict__ coef, int N, int M, int K, double* scale, int* perm, double* L,
                            double* U, double* colv) {
  if (blockIdx.x != 0 || threadIdx.x != 0) return;
  const int n = N * M * K;
  for (int i = 0; i < n; ++i) {
    const double diag = fabs(dense_at(coef, n, N, M, K, i, i));
    scale[i] = (diag > EQ_DOUBLE) ? (1.0 / sqrt(diag)) : 1.0;
    perm[i] = i;
  }
  for (int q = 0; q < n * n; ++q) {
    L[q] = 0.0;
    U[q] = 0.0;
  }
  double maxAbs = 0.0, maxVal = 0.0;
  int pivot = 0;
  double si = scale[0];
  for (int i = 0; i < n; ++i) {
    const double a0 = dense_at(coef, n, N, M, K, i, 0);
    const double absVal = fabs(a0 * scale[i] * si);
    if (absVal > maxVal) {
      maxVal = absVal;
      pivot = i;
    }
    for (int j = 0; j < n; ++j) maxAbs = fmax(maxAbs, fabs(dense_at(coef, n, N, M, K, i, j)));
  }
  const double tiny = EQ_TINY3_DOUBLE * maxAbs;
  if (pivot != 0) {
    const int tmp = perm[0];
    perm[0] = perm[pivot];
    perm[pivot] = tmp;
  }
  int permi = perm[0];
  si = scale[permi];
  for (int j = 0; j < n; ++j) U[j] = dense_at(coef, n, N, M, K, permi, j) * si * scale[j];
  double U00 = U[0];
  if (fabs(U00) < tiny) U00 = (U00 < 0) ? -tiny : tiny;
  U[0] = U00;
  const double invU00 = scale[0] / U00;
  for (int k = 1; k < n; ++k) {
    const int pk = perm[k];
    L[k * n] = dense_at(coef, n, N, M, K, pk, 0) * scale[pk] * invU00;
  }
  L[0] = 1.0;
  for (int i = 1; i < n; ++i) {
    maxVal = 0.0;
    pivot = i;
    si = scale[i];
    for (int k = i; k < n; ++k) {
      double sum = 0.0;
      for (int t = 0; t < i; ++t) sum += L[k * n + t] * U[t * n + i];
      const int pk = perm[k];
      const double val = dense_at(coef, n, N, M, K, pk, i) * scale[pk] * si - sum;
      colv[k] = val;
      if (fabs(val) > maxVal) {
        maxVal = fabs(val);
        pivot = k;
      }
    }
    if (pivot != i) {
      int tmp = perm[i];
      perm[i] = perm[pivot];
      perm[pivot] = tmp;
      for (int t = 0; t < i; ++t) {
        const double d = L[i * n + t];
        L[i * n + t] = L[pivot * n + t];
        L[pivot * n + t] = d;
      }
      const double v = colv[i];
      colv[i] = colv[pivot];
      colv[pivot] = v;
    }
    permi = perm[i];
    si = scale[permi];
    for (int j = i; j < n; ++j) {
      double sum = 0.0;
      for (int t = 0; t < i; ++t) sum += L[i * n + t] * U[t * n + j];
      U[i * n + j] = dense_at(coef, n, N, M, K, permi, j) * si * scale[j] - sum;
    }
    double Uii = U[i * n + i];
    if (fabs(Uii) < tiny) Uii = (Uii < 0) ? -tiny : tiny;
    U[i * n + i] = Uii;
    const double invUii = 1.0 / Uii;
    for (int k = i + 1; k < n; ++k) L[k * n + i] = colv[k] * invUii;
    L[i * n + i] = 1.0;
  }
}

// ---- symmetric storage of the fine operator ----------------------------------------------------
// The reference pressure operator is symmetric except its identity (pinned) rows, whose
// neighbours still couple to them.  A row is an exception when its own off-diagonals are all 0
// while a neighbour's coupling to it is not; each face then takes the coupled side's value.
__device__ inline bool row_decoupled(const double* c7, long n, long i) {
  return c7[0 * n + i] == 0.0 && c7[1 * n + i] == 0.0 && c7[2 * n + i] == 0.0 && c7[4 * n + i] == 0.0 &&
         c7[5 * n + i] == 0.0 && c7[6 * n + i] == 0.0;
}

__global__ void k_sym_check(const double* __restrict__ c7, int N, int M, int K, unsigned char* __restrict__ exc,
                            int* __restrict__ asym) {
  const long n = (long)N * M * K, NM = (long)N * M;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    int x, y, z;
    decode((int)i, N, M, &x, &y, &z);
    unsigned char e = 0;
    const bool di = row_decoupled(c7, n, i);
    // faces towards lower neighbours: (this row's w/s/b) versus (neighbour's e/n/t)
    const long nb[3] = {i - 1, i - N, i - NM};
    const bool has[3] = {x > 0, y > 0, z > 0};
    const int lo_plane[3] = {2, 1, 0}, hi_plane[3] = {4, 5, 6};
    for (int d = 0; d < 3; ++d) {
      if (!has[d]) continue;
      const double mine = c7[lo_plane[d] * n + i], theirs = c7[hi_plane[d] * n + nb[d]];
      if (mine == theirs) continue;
      if (di && mine == 0.0) e = 1;                                   // this row is an identity-like row
      else if (mine != 0.0 && theirs == 0.0 && row_decoupled(c7, n, nb[d])) continue;  // flagged by that row
      else atomicOr(asym, 1);
    }
    const long up[3] = {i + 1, i + N, i + NM};
    const bool hasu[3] = {x < N - 1, y < M - 1, z < K - 1};
    for (int d = 0; d < 3; ++d) {
      if (!hasu[d]) continue;
      const double mine = c7[hi_plane[d] * n + i], theirs = c7[lo_plane[d] * n + up[d]];
      if (mine != theirs && di && mine == 0.0) e = 1;
    }
    exc[i] = e;
  }
}

__global__ void k_sym_build(const double* __restrict__ c7, const unsigned char* __restrict__ exc, int N, int M, int K,
                            double* __restrict__ s4) {
  const long n = (long)N * M * K, NM = (long)N * M;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    int x, y, z;
    decode((int)i, N, M, &x, &y, &z);
    s4[0 * n + i] = c7[3 * n + i];
    s4[1 * n + i] = x < N - 1 ? (exc[i] ? c7[2 * n + i + 1] : c7[4 * n + i]) : 0.0;
    s4[2 * n + i] = y < M - 1 ? (exc[i] ? c7[1 * n + i + N] : c7[5 * n + i]) : 0.0;
    s4[3 * n + i] = z < K - 1 ? (exc[i] ? c7[0 * n + i + NM] : c7[6 * n + i]) : 0.0;
  }
}

// Row i of the symmetric fine operator, terms in the reference CSR order [b,s,w,p,e,n,t]
// (identical values and order to the 7-plane row, hence bit-identical results).  Every load is
// issued unconditionally (absent neighbours read the cell itself) and absent terms leave the sum
// unchanged, so the seven loads of a row are in flight together.
template <class XT>
__device__ inline double row_apply_sym(const double* __restrict__ s4, long n, int i, int x, int y, int z, int N,
                                       int M, int K, const XT* __restrict__ xv, double acc, bool subtract,
                                       const SymExc& ex) {
  const int NM = N * M;
  bool exc_row = false;
#pragma unroll
  for (int q = 0; q < SymExc::CAP; ++q) exc_row |= (q < ex.count) && (ex.row[q] == i);
  const bool hb = !exc_row && z > 0, hs = !exc_row && y > 0, hw = !exc_row && x > 0;
  const bool he = !exc_row && x < N - 1, hn = !exc_row && y < M - 1, ht = !exc_row && z < K - 1;
  const int ib = z > 0 ? i - NM : i, is = y > 0 ? i - N : i, iw = x > 0 ? i - 1 : i;
  const int ie = x < N - 1 ? i + 1 : i, in = y < M - 1 ? i + N : i, it = z < K - 1 ? i + NM : i;
  const double cb = s4[3 * n + ib], cs = s4[2 * n + is], cw = s4[1 * n + iw], cp = s4[i];
  const double ce = s4[1 * n + i], cn = s4[2 * n + i], ct = s4[3 * n + i];
  const double xb = (double)xv[ib], xs = (double)xv[is], xw = (double)xv[iw], xp = (double)xv[i];
  const double xe = (double)xv[ie], xn = (double)xv[in], xt = (double)xv[it];
  auto add = [&](bool h, double c, double xj) {
    const double t = c * xj;
    const double a = subtract ? acc - t : acc + t;
    acc = h ? a : acc;
  };
  add(hb, cb, xb);
  add(hs, cs, xs);
  add(hw, cw, xw);
  add(true, cp, xp);
  add(he, ce, xe);
  add(hn, cn, xn);
  add(ht, ct, xt);
  return acc;
}

// Row i of the transposed operator: A^T(i, j) = A(j, i).  An identity-like row of A becomes a
// full row of A^T (its own faces, which hold the neighbours' couplings to it), and every other
// row drops its couplings to those cells, whose rows in A do not couple back.
__device__ inline bool is_exc(const SymExc& ex, long j) {
  bool e = false;
#pragma unroll
  for (int q = 0; q < SymExc::CAP; ++q) e |= (q < ex.count) && (ex.row[q] == j);
  return e;
}

template <class XT>
__device__ inline double row_apply_sym_t(const double* __restrict__ s4, long n, int i, int x, int y, int z, int N,
                                         int M, int K, const XT* __restrict__ xv, double acc, bool subtract,
                                         const SymExc& ex) {
  const int NM = N * M;
  const bool exc_row = is_exc(ex, i);
  double t;
  auto term = [&](double c, long j) {
    if (!exc_row && is_exc(ex, j)) return;
    t = c * (double)xv[j];
    acc = subtract ? acc - t : acc + t;
  };
  if (z > 0) term(s4[3 * n + i - NM], i - NM);
  if (y > 0) term(s4[2 * n + i - N], i - N);
  if (x > 0) term(s4[1 * n + i - 1], i - 1);
  t = s4[i] * (double)xv[i];
  acc = subtract ? acc - t : acc + t;
  if (x < N - 1) term(s4[1 * n + i], i + 1);
  if (y < M - 1) term(s4[2 * n + i], i + N);
  if (z < K - 1) term(s4[3 * n + i], i + NM);
  return acc;
}

// y = A x or y -= A x (TR: A^T), one thread per cell
template <int MODE, bool TR>
__global__ void __launch_bounds__(256) k_stencil_sym(const double* __restrict__ s4, int N, int M, int K, SymExc ex,
                                                     const double* __restrict__ x, double* __restrict__ y) {
  static_assert(MODE == ST_PROD || MODE == ST_SUBR, "the residual with its norm has a kernel of its own");
  int xx, yy, zz;
  if (!own_cell(N, M, K, &xx, &yy, &zz)) return;
  const long n = (long)N * M * K;
  const int i = xx + N * (yy + M * zz);
  double q;
  if constexpr (TR)
    q = row_apply_sym_t(s4, n, i, xx, yy, zz, N, M, K, x, 0.0, false, ex);
  else
    q = row_apply_sym(s4, n, i, xx, yy, zz, N, M, K, x, 0.0, false, ex);
  y[i] = MODE == ST_PROD ? q : y[i] - q;
}

// y = b - A x (TR: A^T) with the partial sums of y^2 over the reductions' fixed chunks
template <int BS, bool TR>
__global__ void k_stencil_sym_resid(const double* __restrict__ s4, int N, int M, int K, SymExc ex,
                                    const double* __restrict__ x, const double* __restrict__ b, double* __restrict__ y,
                                    double* __restrict__ partial) {
  const long n = (long)N * M * K;
  long lo, hi;
  chunk_of(n, blockIdx.x, gridDim.x, &lo, &hi);
  double ss = 0.0;
  for (long li = lo + threadIdx.x; li < hi; li += BS) {
    const int i = (int)li;
    int xx, yy, zz;
    decode(i, N, M, &xx, &yy, &zz);
    double r;
    if constexpr (TR)
      r = row_apply_sym_t(s4, n, i, xx, yy, zz, N, M, K, x, b[i], true, ex);
    else
      r = row_apply_sym(s4, n, i, xx, yy, zz, N, M, K, x, b[i], true, ex);
    y[i] = r;
    ss += r * r;
  }
  ss = block_sum<BS>(ss);
  if (threadIdx.x == 0) partial[blockIdx.x] = ss;
}

// y = A^T x with an FP32 x
__global__ void k_stencil_sym_t_f32x(const double* __restrict__ s4, int N, int M, int K, SymExc ex,
                                     const float* __restrict__ x, double* __restrict__ y) {
  const long n = (long)N * M * K;
  int xx, yy, zz;
  if (!tile_cell(N, M, &xx, &yy, &zz)) return;
  const int i = xx + N * (yy + M * zz);
  y[i] = row_apply_sym_t(s4, n, i, xx, yy, zz, N, M, K, x, 0.0, false, ex);
}

// y = A x with an FP32 x (mixed-precision Krylov products)
__global__ void k_stencil_sym_f32x(const double* __restrict__ s4, int N, int M, int K, SymExc ex,
                                   const float* __restrict__ x, double* __restrict__ y) {
  const long n = (long)N * M * K;
  int xx, yy, zz;
  if (!tile_cell(N, M, &xx, &yy, &zz)) return;
  const int i = xx + N * (yy + M * zz);
  y[i] = row_apply_sym(s4, n, i, xx, yy, zz, N, M, K, x, 0.0, false, ex);
}

// ---- kernels: solve phase ---------------------------------------------------------------------
// y = A x or y -= A x, one thread per cell: what bounds it is the NPTS + 2 planes moved, and on
// small levels the latency of one row, so no thread takes a second cell (27 points: 4 us at 16^3 and
// 32^3, 36 us at 96^3; up to four cells a thread, their loads behind branches: 17 us averaged over
// the levels of 64^3)
template <int NPTS, int MODE>
__global__ void __launch_bounds__(256) k_stencil(const double* __restrict__ coef, int N, int M, int K,
                                                 const double* __restrict__ x, double* __restrict__ y) {
  static_assert(MODE == ST_PROD || MODE == ST_SUBR, "the residual with its norm has a kernel of its own");
  int xx, yy, zz;
  if (!own_cell(N, M, K, &xx, &yy, &zz)) return;
  const int i = xx + N * (yy + M * zz);
  const double q =
      row_apply<NPTS, MODE == ST_PROD>(coef, (long)N * M * K, i, xx, yy, zz, N, M, K, x, 0.0, false);
  y[i] = MODE == ST_PROD ? q : y[i] - q;
}

// y = b - A x with the partial sums of y^2 over the reductions' fixed chunks
template <int NPTS, int BS>
__global__ void k_stencil_resid(const double* __restrict__ coef, int N, int M, int K, const double* __restrict__ x,
                                const double* __restrict__ b, double* __restrict__ y, double* __restrict__ partial) {
  const long n = (long)N * M * K;
  long lo, hi;
  chunk_of(n, blockIdx.x, gridDim.x, &lo, &hi);
  double ss = 0.0;
  for (long li = lo + threadIdx.x; li < hi; li += BS) {
    const int i = (int)li;
    int xx, yy, zz;
    decode(i, N, M, &xx, &yy, &zz);
    const double r = row_apply<NPTS>(coef, n, i, xx, yy, zz, N, M, K, x, b[i], true);
    y[i] = r;
    ss += r * r;
  }
  ss = block_sum<BS>(ss);
  if (threadIdx.x == 0) partial[blockIdx.x] = ss;
}

// c = omega * T_dir^{-1} r ; ch += c (smoother_adlj_interface.h:73-82 with the TDMA kernels
// smoother_adlj_x.h:38-48, smoother_adlj_y.h:36-50).  One thread per line, the Thomas steps in the
// reference's order.  For z lines the reference reads the first right-hand-side element at index
// y*N*K + x (its z call passes N*K where the y kernel expects N*M); z_head_fix = 0 reproduces
// that read.
//
// A step is three dependent FP64 operations, far shorter than a memory access, so what bounds a line
// is its loads.  A wavefront takes LT lines and moves them in tiles of LT lines x LW cells: 64 lanes
// load a tile of every array (16 loads a lane and array, all in flight, the next tile's under way
// while this one is worked on), post it to LDS, and LT lanes run the Thomas steps on LDS operands.
// Adjacent lanes load adjacent memory for every direction (LW cells of a row for x lines, LT
// adjacent x of a row for y and z lines: whole 128-byte pieces).  The forward result y stays in
// LDS, so r, the factors, the coupling and ch are read once and c and ch written once (56 bytes a
// cell); a line of at most LW cells waits for memory twice in all.  YG: lines too long for that
// pass y through c in memory.  Few lines to a wavefront, so that small levels spread over the
// chip; the LDS accesses of the LT lanes are what a long line then waits for (two values to an
// access; ch stays in registers).  Measured (x / y / z pass): 192^3 90 / 96 / 99 us (4.0-4.4 TB/s),
// 128^3 27 / 29 / 28 us, 64^3 11 us; one thread per line with its loads in the loop: 57 us averaged
// over the levels of 192^3, 111 us over the directions at 127 x 128 x 128.
constexpr int LT = 16, LW = 64, LB = 8;

template <int DIR, bool YG>
__global__ void __launch_bounds__(64) k_line_tile(const double* __restrict__ sb, int N, int M, int K,
                                                  const double* __restrict__ dinv, const double* __restrict__ eu,
                                                  const double* __restrict__ r, double* c,
                                                  double* __restrict__ ch, double omega, int z_head_fix) {
  // tiles of LT rows of LP values: the coupling or eu, dinv, and the r tiles, which y replaces
  // (one for each LW cells of a line; YG: one for all)
  constexpr int LP = LW + 2, TILE = LT * LP, E = LT * LW / 64;
  extern __shared__ __align__(16) double lds_line[];
  double *tb = lds_line, *tc = tb + TILE, *ty = tc + TILE;
  const int nlines = DIR == 0 ? M * K : (DIR == 1 ? N * K : N * M);
  const int len = DIR == 0 ? N : (DIR == 1 ? M : K);
  const int stride = DIR == 0 ? 1 : (DIR == 1 ? N : N * M);
  const int lane = threadIdx.x, line0 = blockIdx.x * LT;
  auto start_of = [&](int t) {
    if (DIR == 0) return t * N;
    if (DIR == 1) return t % N + N * M * (t / N);
    return t;
  };
  // the tile elements of this lane: x lines cell `lane` of line j; y and z lines line lane % LT,
  // cells lane / LT + 4 j
  auto el = [&](int j, int& l, int& k) {
    l = DIR == 0 ? j : lane % LT;
    k = DIR == 0 ? lane : lane / LT + (64 / LT) * j;
  };
  const int own = line0 + lane % LT < nlines ? line0 + lane % LT : nlines - 1;
  const int base = DIR == 0 ? 0 : start_of(own);
  auto index = [&](int l, int k) {  // past the last line or cell: the last one
    const int kk = k < len ? k : len - 1;
    if (DIR == 0) return start_of(line0 + l < nlines ? line0 + l : nlines - 1) + kk;
    return base + stride * kk;
  };
  double a[E], b[E], d[E];
  auto load = [&](int k0, const double* pa, const double* pb, const double* pd) {
#pragma unroll
    for (int j = 0; j < E; ++j) {
      int l, k;
      el(j, l, k);
      const int i = index(l, k0 + k);
      if (pa) a[j] = pa[i];
      b[j] = pb[i];
      d[j] = pd[i];
    }
  };
  // LB consecutive values of this lane's line in a tile, two to an LDS access
  auto take = [&](const double* t, int u0, double (&v)[LB]) {
    const double2* q = reinterpret_cast<const double2*>(t + lane * LP + u0);
#pragma unroll
    for (int u = 0; u < LB / 2; ++u) {
      const double2 w = q[u];
      v[2 * u] = w.x;
      v[2 * u + 1] = w.y;
    }
  };
  auto put = [&](double* t, int u0, const double (&v)[LB]) {
    double2* q = reinterpret_cast<double2*>(t + lane * LP + u0);
#pragma unroll
    for (int u = 0; u < LB / 2; ++u) q[u] = make_double2(v[2 * u], v[2 * u + 1]);
  };
  load(0, r, sb, dinv);
  if (DIR == 2 && !z_head_fix && lane < LT) a[0] = r[own / N * N * K + own % N];
  double yprev = 0.0;
  for (int k0 = 0; k0 < len; k0 += LW) {
    double* yt = YG ? ty : ty + k0 / LW * TILE;
#pragma unroll
    for (int j = 0; j < E; ++j) {
      int l, k;
      el(j, l, k);
      yt[l * LP + k] = a[j];
      tb[l * LP + k] = k0 + k == 0 ? 0.0 : b[j];  // the first cell couples to none: r - 0 y = r
      tc[l * LP + k] = d[j];
    }
    __syncthreads();
    if (k0 + LW < len) load(k0 + LW, r, sb, dinv);
    if (lane < LT) {
      // the operands of the next LB cells are read before the results of these are written, which
      // would hold them back
      const int m = len - k0 < LW ? len - k0 : LW;
      double ra[LB], rb[LB], rd[LB];
      take(yt, 0, ra);
      take(tb, 0, rb);
      take(tc, 0, rd);
      for (int u0 = 0; u0 < m; u0 += LB) {
        double yv[LB];
#pragma unroll
        for (int u = 0; u < LB; ++u) {
          yprev = (ra[u] - rb[u] * yprev) * rd[u];
          yv[u] = yprev;  // past the line's end: unused
        }
        if (u0 + LB < m) {
          take(yt, u0 + LB, ra);
          take(tb, u0 + LB, rb);
          take(tc, u0 + LB, rd);
        }
        put(yt, u0, yv);
      }
    }
    __syncthreads();
    if constexpr (YG) {
#pragma unroll
      for (int j = 0; j < E; ++j) {
        int l, k;
        el(j, l, k);
        if (line0 + l < nlines && k0 + k < len) c[index(l, k0 + k)] = ty[l * LP + k];
      }
      __threadfence_block();  // read back below by other lanes
      __syncthreads();
    }
  }
  // backward: x_k = y_k - e_k x_{k+1}; write omega x and accumulate into ch.  Cells past the line's
  // end have y = e = 0, so that the last cell starts from x = 0 (its own e is 0)
  const int last = (len - 1) / LW * LW;
  const double* yg = YG ? c : nullptr;
  load(last, yg, eu, ch);
  double xnext = 0.0;
  for (int k0 = last; k0 >= 0; k0 -= LW) {
    double* yt = YG ? ty : ty + k0 / LW * TILE;
    double h[E];  // this tile's ch stays with the lanes that loaded it
#pragma unroll
    for (int j = 0; j < E; ++j) {
      int l, k;
      el(j, l, k);
      const bool in = k0 + k < len;
      if (YG || !in) yt[l * LP + k] = YG && in ? a[j] : 0.0;
      tb[l * LP + k] = in ? b[j] : 0.0;
      h[j] = d[j];
    }
    __syncthreads();
    if (k0 >= LW) load(k0 - LW, yg, eu, ch);
    if (lane < LT) {
      const int m = len - k0 < LW ? len - k0 : LW;
      double ra[LB], rb[LB];
      const int top = (m - 1) / LB * LB;
      take(yt, top, ra);
      take(tb, top, rb);
      for (int u0 = top; u0 >= 0; u0 -= LB) {
        double cv[LB];
#pragma unroll
        for (int u = LB - 1; u >= 0; --u) {
          xnext = ra[u] - rb[u] * xnext;
          cv[u] = xnext * omega;
        }
        if (u0 >= LB) {
          take(yt, u0 - LB, ra);
          take(tb, u0 - LB, rb);
        }
        put(yt, u0, cv);
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < E; ++j) {
      int l, k;
      el(j, l, k);
      if (line0 + l < nlines && k0 + k < len) {
        const int i = index(l, k0 + k);
        const double cv = yt[l * LP + k];
        c[i] = cv;
        ch[i] = h[j] + cv;
      }
    }
    __syncthreads();
  }
}

constexpr int LU_SOLVE_THREADS = 256;
__global__ void __launch_bounds__(LU_SOLVE_THREADS) k_lu_solve(const double* scale, const int* perm,
                                                               const double* L, const double* U, int n,
                                                               const double* __restrict__ b, double* __restrict__ x) {
  __shared__ double lds[lu_lds_size(64)];
  const LuLds q = lu_lds(lds, n);
  lu_stage(q, n, scale, perm, L, U);
  for (int k = threadIdx.x; k < n; k += blockDim.x) q.rhs[k] = b[k];
  __syncthreads();
  if (threadIdx.x < 64) lu_substitute(q, n);
  __syncthreads();
  for (int k = threadIdx.x; k < n; k += blockDim.x) x[k] = q.rhs[k];
}

// ---- the cascade's small levels in one workgroup -----------------------------------------------
// A level of a few thousand cells is nothing but latency: its 9 products and 9 line solves per
// application took 18 launches of 3 to 6 us, whatever its size.  One workgroup runs all small levels
// (the last one the LU level): the right-hand sides of every level and the current correction in
// LDS, each thread's part of ch and its one row of a 27-point operator in registers for all sweeps of
// a level, barriers for launches.  Operations and orders are those of the per-level kernels
// (k_stencil, k_line_tile, k_restrict, k_prolong, k_lu_solve).  A 7-point level may have 4096 cells
// and a 27-point level 1024; a 16^3 27-point level would stream 0.9 MB of coefficients through one CU
// for every sweep (5.8 us at 64 bytes a cycle, no less than its two launches) and stays outside.
// Measured: 8^3, 4^3 and the LU 38 us (45 launches: 190 us); with a 16^3 7-point level 104 us (7.3 us
// a sweep, of which the coefficients' and factors' way from L2 takes about half).
constexpr int CS_THREADS = 512, CS_CELLS = 8, CS_LEN = 17;
constexpr int CS_LDS = 18432;  // doubles: 144 KB of the CU's 160

// rows of a level in LDS: x fastest with an odd pitch (x lines: adjacent lanes hold adjacent rows)
struct CsGrid {
  int N, M, K, P;
  __device__ CsGrid(Dims d) : N(d.N), M(d.M), K(d.K), P(d.N | 1) {}
  __device__ int at(int x, int y, int z) const { return x + P * (y + M * z); }
};

// element i of p by a 32-bit byte offset from a uniform base: one address register a load
__device__ inline double ld32(const double* __restrict__ p, unsigned i) {
  return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(p) + i * 8u);
}

// all sweeps of one level of axes of at most ML cells: c holds the prolonged correction (every
// cell), chv each thread's own
template <int NP, int CELLS, int ML>
__device__ inline void cs_sweeps(const CascadeLevel& L, int n_post, double omega, int z_head_fix, double* __restrict__ r,
                                 double* __restrict__ c, double (&chv)[CS_CELLS]) {
  const CsGrid g(L.d);
  const int n = g.N * g.M * g.K, tid = threadIdx.x;
  // a thread's one 27-point row stays in registers for all sweeps; several rows are read again by
  // each sweep, HELD at a time: with the lines' factors they would spill
  constexpr bool KEEP = CELLS == 1;
  constexpr int HELD = NP == 27 ? 1 : 2;
  double a[HELD][NP];
  unsigned shift = 0;
  auto rows = [&](int j0) {
#pragma unroll
    for (int j = 0; j < HELD; ++j)
      if (tid + CS_THREADS * (j0 + j) < n)
#pragma unroll
        for (int q = 0; q < NP; ++q) a[j][q] = ld32(L.coef + q * n, shift + tid + CS_THREADS * (j0 + j));
  };
  if (KEEP) rows(0);
  int own[CELLS];
  unsigned okm[CELLS];  // axis neighbours present: bit 0/1 x -/+, 2/3 y, 4/5 z
#pragma unroll
  for (int j = 0; j < CELLS; ++j) {
    const int i = tid + CS_THREADS * j;
    own[j] = 0;
    okm[j] = 0;
    if (i >= n) continue;
    int x, y, z;
    decode(i, g.N, g.M, &x, &y, &z);
    own[j] = g.at(x, y, z);
    okm[j] = (x > 0) | (x < g.N - 1) << 1 | (y > 0) << 2 | (y < g.M - 1) << 3 | (z > 0) << 4 | (z < g.K - 1) << 5;
  }
  const int sy = g.P, sz = g.P * g.M;
  for (int s = 0; s < n_post; ++s)
#pragma unroll 1
    for (int dir = 2; dir >= 0; --dir) {  // z, y, x
      // one thread per line; its couplings and pivots are on their way while the product runs
      const int len = dir == 0 ? g.N : (dir == 1 ? g.M : g.K);
      const int stg = dir == 0 ? n / len : (dir == 1 ? g.N : g.N * g.M), stl = dir == 0 ? 1 : (dir == 1 ? sy : sz);
      const bool line = tid < n / len;
      const int p = dir == 0 ? 0 : tid % g.N, q = dir == 0 ? tid : tid / g.N;
      const int g0 = dir == 1 ? p + g.N * g.M * q : tid;  // x lines: of the transposed factors
      const int l0 = dir == 0 ? g.P * q : (dir == 1 ? p + sz * q : p + sy * q);
      double fs[ML], fd[ML];
      if (line) {
        const double* sb = dir == 0 ? L.xt : L.coef + slot_sub(NP, dir) * n;
        const double* di = dir == 0 ? L.xt + n : L.dinv[dir];
#pragma unroll
        for (int u = 0; u < ML; ++u) {
          const int k = u < len ? u : len - 1;
          fs[u] = ld32(sb, g0 + stg * k);
          fd[u] = ld32(di, g0 + stg * k);
        }
      }
      // r -= A c.  The empty asm statements hide that a sweep's addresses are the last one's: kept
      // over the sweeps instead of computed again, they spill
      if (!KEEP) asm volatile("" : "+s"(shift));
#pragma unroll
      for (int j = 0; j < CELLS; ++j) {
        if (!KEEP && j % HELD == 0) rows(j);
        if (tid + CS_THREADS * j >= n) continue;
        // straight-line as row_apply: an absent neighbour has coefficient 0 and reads the cell itself
        int o = own[j];
        unsigned m = okm[j];
        asm volatile("" : "+v"(o), "+v"(m));
        const int ox[3] = {m & 1 ? -1 : 0, 0, m & 2 ? 1 : 0}, oy[3] = {m & 4 ? -sy : 0, 0, m & 8 ? sy : 0};
        const int oz[3] = {m & 16 ? -sz : 0, 0, m & 32 ? sz : 0};
        double acc = 0.0, v[NP];
#pragma unroll
        for (int q = 0; q < NP; ++q) {
          const int p = NP == 27 ? q : (const int[7]){4, 10, 12, 13, 14, 16, 22}[q];
          v[q] = c[o + ox[p % 3] + oy[p / 3 % 3] + oz[p / 9]];
        }
#pragma unroll
        for (int q = 0; q < NP; ++q) acc = acc + a[j % HELD][q] * v[q];
        r[o] = r[o] - acc;
      }
      __syncthreads();
      // c = omega T^-1 r
      if (line) {
        const double* eu = dir == 0 ? L.xt + 2 * n : L.eu[dir];
        double fe[ML], v[ML];
#pragma unroll
        for (int u = 0; u < ML; ++u) {
          const int k = u < len ? u : len - 1;
          v[u] = r[l0 + stl * k];
          fe[u] = ld32(eu, g0 + stg * k);
        }
        if (dir == 2 && !z_head_fix) {
          int hx, hy, hz;
          decode(q * g.N * g.K + p, g.N, g.M, &hx, &hy, &hz);
          v[0] = r[g.at(hx, hy, hz)];
        }
        v[0] = v[0] * fd[0];
#pragma unroll
        for (int u = 1; u < ML; ++u)
          if (u < len) v[u] = (v[u] - fs[u] * v[u - 1]) * fd[u];  // uniform branch
        double xnext = 0.0;
#pragma unroll
        for (int u = ML - 1; u >= 0; --u)
          if (u < len) {
            xnext = v[u] - fe[u] * xnext;
            c[l0 + stl * u] = xnext * omega;
          }
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < CELLS; ++j)
        if (tid + CS_THREADS * j < n) chv[j] = chv[j] + c[own[j]];
    }
}

// xt: a level's x couplings, dinv and eu with the line index fastest, so that the threads of
// k_cascade_small, one per x line, load adjacent values (set-up)
__global__ void k_x_factors_t(const double* __restrict__ sb, const double* __restrict__ dinv,
                              const double* __restrict__ eu, int N, int nl, double* __restrict__ xt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, n = N * nl;
  if (i >= n) return;
  const int j = i / nl + N * (i % nl);
  xt[i] = sb[j];
  xt[n + i] = dinv[j];
  xt[2 * n + i] = eu[j];
}

__global__ void __launch_bounds__(CS_THREADS) k_cascade_small(CascadeLevels C, int n_post, double omega, int z_head_fix,
                                                              const double* __restrict__ lu_scale,
                                                              const int* __restrict__ lu_perm,
                                                              const double* __restrict__ Lf,
                                                              const double* __restrict__ Uf,
                                                              const double* __restrict__ r0, double* __restrict__ ch0) {
  __shared__ double lds[CS_LDS];
  const int tid = threadIdx.x, last = C.count - 1;
  // r of every level, then c (the largest level's size), then ch of the level below, then the LU
  double* c = lds + C.off[last + 1];
  double* chl = c + C.c_size;
  const int n_last = (int)C.L[last].d.n();
  const LuLds lu = lu_lds(chl + C.ch_size, n_last);
  lu_stage(lu, n_last, lu_scale, lu_perm, Lf, Uf);
  {
    const CsGrid g(C.L[0].d);
    const int n = g.N * g.M * g.K;
    for (int i = tid; i < n; i += CS_THREADS) {
      int x, y, z;
      decode(i, g.N, g.M, &x, &y, &z);
      lds[g.at(x, y, z)] = r0[i];
    }
  }
  __syncthreads();
  for (int q = 0; q < last; ++q) {
    const CsGrid f(C.L[q].d), g(C.L[q + 1].d);
    const double* rf = lds + C.off[q];
    double* rc = q + 1 == last ? lu.rhs : lds + C.off[q + 1];
    auto at = [&](int x, int y, int z) { return rf[f.at(x, y, z)]; };
    for (int i = tid; i < g.N * g.M * g.K; i += CS_THREADS) {
      int X, Y, Z;
      decode(i, g.N, g.M, &X, &Y, &Z);
      const double v = f.N & 1 ? restrict_cell_odd(at, X, Y, Z, f.N, f.M, f.K) : restrict_cell(at, X, Y, Z);
      rc[q + 1 == last ? i : g.at(X, Y, Z)] = v;
    }
    __syncthreads();
  }
  if (tid < 64) lu_substitute(lu, n_last);
  __syncthreads();
  for (int q = last - 1; q >= 0; --q) {
    const CsGrid f(C.L[q].d), g(C.L[q + 1].d);
    const int n = f.N * f.M * f.K;
    const double* chc = q + 1 == last ? lu.rhs : chl;
    auto at = [&](int x, int y, int z) { return chc[x + g.N * (y + g.M * z)]; };
    double chv[CS_CELLS];
#pragma unroll
    for (int j = 0; j < CS_CELLS; ++j) {
      const int i = tid + CS_THREADS * j;
      chv[j] = 0.0;
      if (i >= n) continue;
      int x, y, z;
      decode(i, f.N, f.M, &x, &y, &z);
      chv[j] = f.N & 1 ? prolong_cell_odd(at, x, y, z) : prolong_cell(at, x, y, z, f.N, f.M, f.K);
      c[f.at(x, y, z)] = chv[j];
    }
    __syncthreads();
    if (C.L[q].npts == 7)
      cs_sweeps<7, CS_CELLS, CS_LEN>(C.L[q], n_post, omega, z_head_fix, lds + C.off[q], c, chv);
    else if (n > CS_THREADS || max(f.N, max(f.M, f.K)) > 9)
      cs_sweeps<27, CS_CELLS / 4, CS_LEN>(C.L[q], n_post, omega, z_head_fix, lds + C.off[q], c, chv);
    else
      cs_sweeps<27, 1, 9>(C.L[q], n_post, omega, z_head_fix, lds + C.off[q], c, chv);
    double* out = q == 0 ? ch0 : chl;
#pragma unroll
    for (int j = 0; j < CS_CELLS; ++j)
      if (tid + CS_THREADS * j < n) out[tid + CS_THREADS * j] = chv[j];
    __syncthreads();
  }
}

// ---- kernels: BLAS-1 ---------------------------------------------------------------------------
__global__ void k_copy(const double* __restrict__ a, double* __restrict__ b, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) b[i] = a[i];
}

__global__ void k_fill_zero(double* __restrict__ b, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) b[i] = 0.0;
}

__global__ void k_scale_copy(const double* __restrict__ w, const double* __restrict__ normw, double* __restrict__ v,
                             long n) {
  const double f = 1.0 / normw[0];
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) v[i] = f * w[i];
}

__global__ void k_scale_copy_f32(const double* __restrict__ w, const double* __restrict__ normw, double* __restrict__ v,
                                 float* __restrict__ vf, long n) {
  const double f = 1.0 / normw[0];
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const double a = f * w[i];
    v[i] = a;
    vf[i] = (float)a;
  }
}

template <int BS>
__global__ void k_dot_partial(const double* __restrict__ a, const double* __restrict__ b, long n, double* partial) {
  long lo, hi;
  chunk_of(n, blockIdx.x, gridDim.x, &lo, &hi);
  double s = 0.0;
  for (long i = lo + threadIdx.x; i < hi; i += BS) s += a[i] * b[i];
  s = block_sum<BS>(s);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// the partial sums of a . b and c . d, gridDim.x each: BiCGStab asks for its dots in pairs, and at 129 x 111
// x 95 a dot alone is 5.1 us of kernel, 2.5 of summing and a round trip to the host
template <int BS>
__global__ void k_dot2_partial(const double* __restrict__ a, const double* __restrict__ b, const double* __restrict__ c,
                               const double* __restrict__ d, long n, double* __restrict__ partial) {
  long lo, hi;
  chunk_of(n, blockIdx.x, gridDim.x, &lo, &hi);
  double s = 0.0, t = 0.0;
  for (long i = lo + threadIdx.x; i < hi; i += BS) {
    s += a[i] * b[i];
    t += c[i] * d[i];
  }
  s = block_sum<BS>(s);
  t = block_sum<BS>(t);
  if (threadIdx.x == 0) {
    partial[blockIdx.x] = s;
    partial[gridDim.x + blockIdx.x] = t;
  }
}

template <int BS>
__global__ void k_finalize(const double* partial, int nb, double* out, int sqrt_flag) {
  double s = 0.0;
  // each thread sums a contiguous run so the combination order is fixed
  const int per = (nb + BS - 1) / BS;
  const int lo = threadIdx.x * per;
  for (int i = lo; i < lo + per && i < nb; ++i) s += partial[i];
  s = block_sum<BS>(s);
  if (threadIdx.x == 0) out[0] = sqrt_flag ? sqrt(s) : s;
}

// One step of modified Gram-Schmidt: h = the dot whose partial sums are `pin`, w -= h v, partial sums of
// the next dot (w . vnext, or w . w) into `pout`.  A step is a chain of two launches' latencies, not of
// bytes: every block sums the partials itself, as k_finalize does and to the same bits, while its
// first rows are on their way, instead of waiting for a launch of one workgroup to do it.  16^3: 7.9
// us a step in two launches, 4.6 in one; 64^3: 6.5 and 3.9
template <int BS>
__global__ void __launch_bounds__(BS) k_axpy_dot(double* __restrict__ w, const double* __restrict__ v,
                                                 const double* __restrict__ pin, double* __restrict__ h,
                                                 const double* __restrict__ vnext, long n, double* __restrict__ pout) {
  constexpr int R = 4;  // rows per step
  __shared__ double hs;
  long lo, hi;
  chunk_of(n, blockIdx.x, gridDim.x, &lo, &hi);
  long i = lo + threadIdx.x;
  double vr[R], wr[R], nr[R];
  auto load = [&] {  // of a thread with a row i
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const long q = row_ahead(i, r * BS, hi);
      vr[r] = v[q];
      wr[r] = w[q];
      nr[r] = vnext ? vnext[q] : 0.0;
    }
  };
  if (i < hi) load();
  double p = 0.0;
  const int nb = gridDim.x, per = (nb + BS - 1) / BS, from = threadIdx.x * per;
  for (int k = from; k < from + per && k < nb; ++k) p += pin[k];
  p = block_sum<BS>(p);
  if (threadIdx.x == 0) {
    hs = p;
    if (blockIdx.x == 0) h[0] = p;
  }
  __syncthreads();
  const double hv = hs;
  double s = 0.0;
  while (i < hi) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (i + r * BS < hi) {
        const double aux = vr[r] * hv;
        const double wn = wr[r] - aux;
        w[i + r * BS] = wn;
        s += vnext ? wn * nr[r] : wn * wn;
      }
    i += R * BS;
    if (i < hi) load();
  }
  s = block_sum<BS>(s);
  if (threadIdx.x == 0) pout[blockIdx.x] = s;
}

// ---- classical Gram-Schmidt passes ------------------------------------------------------------
// V holds cnt <= CGS_MAX basis vectors, vector k at V + k*ldv.  The dot pass runs on a 2D grid
// (row chunks x groups of CGS_GROUP vectors) so each thread keeps only CGS_GROUP accumulators and
// pointers; partial[k * nb + chunk] is summed in a fixed order by k_finalize_multi.  The update
// pass keeps the coefficients in LDS and streams the vectors row by row.
constexpr int CGS_GROUP = 8;

// rows per step of the Gram-Schmidt passes: their loads are in flight together
constexpr int CGS_ROWS = 4;

// acc[k] += sum over the thread's rows i of V_k[i] w[i], rows in increasing order, CGS_ROWS
// rows (i, i + BS, ...) per step so that CGS_ROWS (KC + 1) loads are in flight
template <int BS, int KC, class VT>
__device__ inline void cgs_dot_rows(const VT* __restrict__ Vg, long ldv, const double* __restrict__ w, long lo,
                                    long hi, double (&acc)[CGS_GROUP]) {
  constexpr int R = CGS_ROWS;
  long i = lo + threadIdx.x;
  for (; i + (R - 1) * BS < hi; i += R * BS) {
    double wr[R], v[R][KC];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      wr[r] = w[i + r * BS];
#pragma unroll
      for (int k = 0; k < KC; ++k) v[r][k] = (double)Vg[k * ldv + i + r * BS];
    }
#pragma unroll
    for (int k = 0; k < KC; ++k)
#pragma unroll
      for (int r = 0; r < R; ++r) acc[k] += v[r][k] * wr[r];
  }
  for (; i < hi; i += BS) {
    const double w0 = w[i];
#pragma unroll
    for (int k = 0; k < KC; ++k) acc[k] += (double)Vg[k * ldv + i] * w0;
  }
}

// Block (chunk c, group g) is block c % 8 + 8 (g + ng (c / 8)) of a 1-D grid of 8 ceil(nb / 8) ng
// blocks (those of chunks past nb exit at once): workgroups go to the 8 XCDs round-robin, so the
// ng blocks of one chunk run on one XCD one after the other and read its slice of w from that
// XCD's L2 after the first.
template <int BS, class VT>
__global__ void __launch_bounds__(BS) k_cgs_dot(const VT* __restrict__ V, long ldv, int cnt,
                                                const double* __restrict__ w, long n, int nb, int ng,
                                                double* __restrict__ partial) {
  __shared__ double lds[BS / 64][CGS_GROUP];
  const int b = blockIdx.x, r = b / 8;
  const int chunk = b % 8 + 8 * (r / ng), grp = r % ng;
  if (chunk >= nb) return;  // uniform over the block
  const int k0 = grp * CGS_GROUP;
  const int kc = cnt - k0 < CGS_GROUP ? cnt - k0 : CGS_GROUP;
  long lo, hi;
  chunk_of(n, chunk, nb, &lo, &hi);
  const VT* Vg = V + (long)k0 * ldv;
  double acc[CGS_GROUP];
#pragma unroll
  for (int k = 0; k < CGS_GROUP; ++k) acc[k] = 0.0;
  switch (kc) {  // uniform over the block: every load of a step is issued unconditionally
    case 1: cgs_dot_rows<BS, 1, VT>(Vg, ldv, w, lo, hi, acc); break;
    case 2: cgs_dot_rows<BS, 2, VT>(Vg, ldv, w, lo, hi, acc); break;
    case 3: cgs_dot_rows<BS, 3, VT>(Vg, ldv, w, lo, hi, acc); break;
    case 4: cgs_dot_rows<BS, 4, VT>(Vg, ldv, w, lo, hi, acc); break;
    case 5: cgs_dot_rows<BS, 5, VT>(Vg, ldv, w, lo, hi, acc); break;
    case 6: cgs_dot_rows<BS, 6, VT>(Vg, ldv, w, lo, hi, acc); break;
    case 7: cgs_dot_rows<BS, 7, VT>(Vg, ldv, w, lo, hi, acc); break;
    default: cgs_dot_rows<BS, CGS_GROUP, VT>(Vg, ldv, w, lo, hi, acc); break;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < CGS_GROUP; ++k) {
    double v = acc[k];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if (lane == 0) lds[wave][k] = v;
  }
  __syncthreads();
  if ((int)threadIdx.x < kc) {
    double s = 0.0;
    for (int q = 0; q < BS / 64; ++q) s += lds[q][threadIdx.x];
    partial[(long)(k0 + threadIdx.x) * nb + chunk] = s;
  }
}

// w -= sum_k h_k v_k ; with_norm: partial ||w||^2 per block
template <int BS>
__global__ void __launch_bounds__(BS) k_cgs_update(const double* __restrict__ V, long ldv, int cnt,
                                                   const double* __restrict__ h, double* __restrict__ w, long n,
                                                   int with_norm, double* __restrict__ partial) {
  __shared__ double hk[CGS_MAX];
  if ((int)threadIdx.x < cnt) hk[threadIdx.x] = h[threadIdx.x];
  __syncthreads();
  long lo, hi;
  chunk_of(n, blockIdx.x, gridDim.x, &lo, &hi);
  double ss = 0.0;
  constexpr int R = CGS_ROWS;
  long i = lo + threadIdx.x;
  for (; i + (R - 1) * BS < hi; i += R * BS) {  // R rows per step, each updated in the order k = 0, 1, ...
    double wr[R];
#pragma unroll
    for (int r = 0; r < R; ++r) wr[r] = w[i + r * BS];
    const double* vp = V + i;
#pragma unroll 8
    for (int k = 0; k < cnt; ++k)
#pragma unroll
      for (int r = 0; r < R; ++r) wr[r] -= hk[k] * vp[k * ldv + r * BS];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      w[i + r * BS] = wr[r];
      ss += wr[r] * wr[r];
    }
  }
  for (; i < hi; i += BS) {
    double wn = w[i];
    const double* vp = V + i;
#pragma unroll 8
    for (int k = 0; k < cnt; ++k) wn -= hk[k] * vp[k * ldv];
    w[i] = wn;
    ss += wn * wn;
  }
  if (with_norm) {
    ss = block_sum<BS>(ss);
    if (threadIdx.x == 0) partial[blockIdx.x] = ss;
  }
}

// out = post (w - sum_k (h_k isq_k) v_k) (out may alias w), out32 = (float)out when given;
// with_norm: partial ||out||^2 per block
// R rows per step and the vector loop unrolled U times: R U loads in flight (8 x 4 measured
// 342 against 355 us for 4 x 8 at 256^3 with 21 basis vectors)
template <int BS, int R, int U>
__global__ void __launch_bounds__(BS) k_cgs_update_scaled(const double* __restrict__ V, long ldv, int cnt,
                                                          const double* __restrict__ h, CgsScales sc, double post,
                                                          const double* w, double* out, float* __restrict__ out32,
                                                          long n, int with_norm, double* __restrict__ partial) {
  __shared__ double hk[CGS_MAX];
  if ((int)threadIdx.x < cnt) hk[threadIdx.x] = h[threadIdx.x] * sc.isq[threadIdx.x];
  __syncthreads();
  long lo, hi;
  chunk_of(n, blockIdx.x, gridDim.x, &lo, &hi);
  double ss = 0.0;
  long i = lo + threadIdx.x;
  for (; i + (R - 1) * BS < hi; i += R * BS) {
    double wr[R];
#pragma unroll
    for (int r = 0; r < R; ++r) wr[r] = w[i + r * BS];
    const double* vp = V + i;
#pragma unroll U
    for (int k = 0; k < cnt; ++k)
#pragma unroll
      for (int r = 0; r < R; ++r) wr[r] -= hk[k] * vp[k * ldv + r * BS];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const double o = wr[r] * post;
      out[i + r * BS] = o;
      if (out32) out32[i + r * BS] = (float)o;
      ss += o * o;
    }
  }
  for (; i < hi; i += BS) {
    double wn = w[i];
    const double* vp = V + i;
#pragma unroll 8
    for (int k = 0; k < cnt; ++k) wn -= hk[k] * vp[k * ldv];
    const double o = wn * post;
    out[i] = o;
    if (out32) out32[i] = (float)o;
    ss += o * o;
  }
  if (with_norm) {
    ss = block_sum<BS>(ss);
    if (threadIdx.x == 0) partial[blockIdx.x] = ss;
  }
}

template <int BS>
__global__ void k_finalize_multi(const double* __restrict__ partial, int nb, double* __restrict__ out,
                                 int sqrt_flag) {
  const double* p = partial + (long)blockIdx.x * nb;
  double s = 0.0;
  const int per = (nb + BS - 1) / BS;
  const int lo = threadIdx.x * per;
  for (int i = lo; i < lo + per && i < nb; ++i) s += p[i];
  s = block_sum<BS>(s);
  if (threadIdx.x == 0) out[blockIdx.x] = sqrt_flag ? sqrt(s) : s;
}

// y = A x on the fine 7-point operator with an FP32 input vector (mixed-precision Krylov basis)
__global__ void k_stencil7_prod_f32x(const double* __restrict__ coef, int N, int M, int K,
                                     const float* __restrict__ x, double* __restrict__ y) {
  const long n = (long)N * M * K;
  const int NM = N * M;
  for (long li = blockIdx.x * (long)blockDim.x + threadIdx.x; li < n; li += (long)gridDim.x * blockDim.x) {
    const int i = (int)li;
    int xx, yy, zz;
    decode(i, N, M, &xx, &yy, &zz);
    double acc = 0.0;
    if (zz > 0) acc = acc + coef[0 * n + i] * (double)x[i - NM];
    if (yy > 0) acc = acc + coef[1 * n + i] * (double)x[i - N];
    if (xx > 0) acc = acc + coef[2 * n + i] * (double)x[i - 1];
    acc = acc + coef[3 * n + i] * (double)x[i];
    if (xx < N - 1) acc = acc + coef[4 * n + i] * (double)x[i + 1];
    if (yy < M - 1) acc = acc + coef[5 * n + i] * (double)x[i + N];
    if (zz < K - 1) acc = acc + coef[6 * n + i] * (double)x[i + NM];
    y[i] = acc;
  }
}

struct YCoef {
  double y[64];
};

// x += sum_k y_k z_k, k = count-1 .. 0 in that order for every row; four rows per step (grid
// stride apart) with the vector loop unrolled four times, so that 16 loads are in flight
template <class ZT>
__global__ void k_sol_update_t(double* __restrict__ x, const ZT* __restrict__ Z, long ldz, YCoef yk, int count,
                               long n) {
  constexpr int R = 4;
  const long st = (long)gridDim.x * blockDim.x;
  long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  for (; i + (R - 1) * st < n; i += R * st) {
    double aux[R];
#pragma unroll
    for (int r = 0; r < R; ++r) aux[r] = x[i + r * st];
#pragma unroll 4
    for (int k = count - 1; k >= 0; --k)
#pragma unroll
      for (int r = 0; r < R; ++r) aux[r] = aux[r] + (double)Z[k * ldz + i + r * st] * yk.y[k];
#pragma unroll
    for (int r = 0; r < R; ++r) x[i + r * st] = aux[r];
  }
  for (; i < n; i += st) {
    double aux = x[i];
    for (int k = count - 1; k >= 0; --k) aux = aux + (double)Z[k * ldz + i] * yk.y[k];
    x[i] = aux;
  }
}

__global__ void k_bicg_s(double* __restrict__ nu, const double* __restrict__ r, double* __restrict__ sv, double alpha,
                         long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const double nv = nu[i] * alpha;
    nu[i] = nv;
    sv[i] = r[i] - nv;
  }
}

__global__ void k_bicg_sol(const double* __restrict__ sv, double* __restrict__ y, double* __restrict__ z,
                           double* __restrict__ x, double* __restrict__ t, double* __restrict__ r, double alpha,
                           double w, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const double yi = y[i] * alpha;
    y[i] = yi;
    const double zi = z[i] * w;
    z[i] = zi;
    const double cs = yi + zi;
    x[i] = x[i] + cs;
    const double ti = t[i] * w;
    t[i] = ti;
    r[i] = sv[i] - ti;
  }
}

__global__ void k_bicg_p(double* __restrict__ p, const double* __restrict__ nu, const double* __restrict__ r,
                         double coef, double beta, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const double cv = (p[i] - nu[i] * coef) * beta;
    p[i] = r[i] + cv;
  }
}

__global__ void k_sub(const double* __restrict__ b, const double* __restrict__ z, double* __restrict__ r, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) r[i] = b[i] - z[i];
}

int grid_1d(long n, int bs = 256) {
  long g = (n + bs - 1) / bs;
  if (g > 8192) g = 8192;
  if (g < 1) g = 1;
  return (int)g;
}

}  // namespace

// ================================================================================================
// launchers
// ================================================================================================
// blocks of tile_cell
static unsigned tile_blocks(Dims d) { return (unsigned)((long)((d.N + 63) / 64) * ((d.M + 3) / 4) * d.K); }
// blocks of own_cell
static unsigned cell_blocks(Dims d) { return d.N >= 64 ? tile_blocks(d) : (unsigned)((d.n() + 255) / 256); }

int reduction_blocks(long n) {
  long b = (n + RED_THREADS * 4 - 1) / (RED_THREADS * 4);
  if (b > RED_BLOCKS_MAX) b = RED_BLOCKS_MAX;
  if (b < 1) b = 1;
  return (int)b;
}

void csr_to_stencil7(const int* rowptr, const int* col, const double* val, Dims d, double* coef7, int* err_flag,
                     hipStream_t s) {
  k_csr_to_stencil7<<<grid_1d(d.n()), 256, 0, s>>>(rowptr, col, val, d.N, d.M, d.K, coef7, err_flag);
}

void galerkin(const double* coef_f, int npts_f, Dims df, double* coef27_c, Dims dc, hipStream_t s) {
  if (df.N & 1) {  // odd-odd-odd level (the only odd class the hierarchy admits)
    if (npts_f == 7)
      k_galerkin_odd<7><<<grid_1d(dc.n(), 64), 64, 0, s>>>(coef_f, df.N, df.M, df.K, coef27_c, dc.N, dc.M, dc.K);
    else
      k_galerkin_odd<27><<<grid_1d(dc.n(), 64), 64, 0, s>>>(coef_f, df.N, df.M, df.K, coef27_c, dc.N, dc.M, dc.K);
    return;
  }
  if (npts_f == 7)
    k_galerkin<7><<<grid_1d(dc.n(), 64), 64, 0, s>>>(coef_f, df.N, df.M, df.K, coef27_c, dc.N, dc.M, dc.K);
  else
    k_galerkin<27><<<grid_1d(dc.n(), 64), 64, 0, s>>>(coef_f, df.N, df.M, df.K, coef27_c, dc.N, dc.M, dc.K);
}

void diag_absmax(const double* coef, int npts, Dims d, double* partial, double* out, hipStream_t s) {
  const int nb = reduction_blocks(d.n());
  const double* dg = coef + (long)(npts == 7 ? 3 : 13) * d.n();
  k_diag_absmax_partial<RED_THREADS><<<nb, RED_THREADS, 0, s>>>(dg, d.n(), partial);
  k_max_finalize<RED_THREADS><<<1, RED_THREADS, 0, s>>>(partial, nb, out);
}

void absmax(const double* a, long n, double* partial, double* out, hipStream_t s) {
  const int nb = reduction_blocks(n);
  k_diag_absmax_partial<RED_THREADS><<<nb, RED_THREADS, 0, s>>>(a, n, partial);
  k_max_finalize<RED_THREADS><<<1, RED_THREADS, 0, s>>>(partial, nb, out);
}

void line_factor(const double* coef, int npts, Dims d, int dir, const double* absmax, double* dinv, double* eu,
                 hipStream_t s) {
  const int nlines = dir == 0 ? d.M * d.K : (dir == 1 ? d.N * d.K : d.N * d.M);
  k_line_factor<<<div_up(nlines, 64), 64, 0, s>>>(coef, npts, d.N, d.M, d.K, dir, absmax, dinv, eu);
}

void lu_factor(const double* coef27, Dims d, double* scale, int* perm, double* L, double* U, double* col_scratch,
               hipStream_t s) {
  k_lu_factor<<<1, 1, 0, s>>>(coef27, d.N, d.M, d.K, scale, perm, L, U, col_scratch);
}

void stencil_apply(const double* coef, int npts, Dims d, const double* x, const double* b, double* y, int mode,
                   double* partial, hipStream_t s) {
  const int nb = reduction_blocks(d.n());
#define LSX_ST(NP)                                                                                          \
  do {                                                                                                      \
    if (mode == ST_RESID)                                                                                   \
      k_stencil_resid<NP, RED_THREADS><<<nb, RED_THREADS, 0, s>>>(coef, d.N, d.M, d.K, x, b, y, partial);   \
    else if (mode == ST_PROD)                                                                               \
      k_stencil<NP, ST_PROD><<<cell_blocks(d), 256, 0, s>>>(coef, d.N, d.M, d.K, x, y);                     \
    else                                                                                                    \
      k_stencil<NP, ST_SUBR><<<cell_blocks(d), 256, 0, s>>>(coef, d.N, d.M, d.K, x, y);                     \
  } while (0)
  if (npts == 7)
    LSX_ST(7);
  else
    LSX_ST(27);
#undef LSX_ST
}

template <bool TR>
static void stencil_sym_any(const double* s4, const SymExc& ex, Dims d, const double* x, const double* b, double* y,
                            int mode, double* partial, hipStream_t s) {
  if (mode == ST_RESID)
    k_stencil_sym_resid<RED_THREADS, TR><<<reduction_blocks(d.n()), RED_THREADS, 0, s>>>(s4, d.N, d.M, d.K, ex, x, b,
                                                                                         y, partial);
  else if (mode == ST_PROD)
    k_stencil_sym<ST_PROD, TR><<<cell_blocks(d), 256, 0, s>>>(s4, d.N, d.M, d.K, ex, x, y);
  else
    k_stencil_sym<ST_SUBR, TR><<<cell_blocks(d), 256, 0, s>>>(s4, d.N, d.M, d.K, ex, x, y);
}

void sym_check(const double* coef7, Dims d, unsigned char* exc, int* asym, hipStream_t s) {
  k_sym_check<<<grid_1d(d.n()), 256, 0, s>>>(coef7, d.N, d.M, d.K, exc, asym);
}

void sym_build(const double* coef7, const unsigned char* exc, Dims d, double* s4, hipStream_t s) {
  k_sym_build<<<grid_1d(d.n()), 256, 0, s>>>(coef7, exc, d.N, d.M, d.K, s4);
}

void stencil_apply_sym(const double* s4, const SymExc& ex, Dims d, const double* x, const double* b, double* y,
                       int mode, double* partial, hipStream_t s) {
  stencil_sym_any<false>(s4, ex, d, x, b, y, mode, partial, s);
}

void restrict_full(const double* rf, Dims df, double* rc, Dims dc, hipStream_t s) {
  if (df.N & 1)
    k_restrict<true><<<grid_1d(dc.n()), 256, 0, s>>>(rf, df.N, df.M, df.K, rc, dc.N, dc.M, dc.K);
  else
    k_restrict<false><<<grid_1d(dc.n()), 256, 0, s>>>(rf, df.N, df.M, df.K, rc, dc.N, dc.M, dc.K);
}

void prolong_copy(const double* chc, Dims dc, double* chf, double* cf, Dims df, hipStream_t s) {
  if (df.N & 1)
    k_prolong<true><<<grid_1d(df.n()), 256, 0, s>>>(chc, dc.N, dc.M, chf, cf, df.N, df.M, df.K);
  else
    k_prolong<false><<<grid_1d(df.n()), 256, 0, s>>>(chc, dc.N, dc.M, chf, cf, df.N, df.M, df.K);
}

void line_solve(const double* coef, int npts, Dims d, int dir, const double* dinv, const double* eu, const double* r,
                double* c, double* ch, double omega, int z_head_fix, hipStream_t s) {
  const double* sb = coef + slot_sub(npts, dir) * d.n();
  const int len = dir == 0 ? d.N : (dir == 1 ? d.M : d.K);
  const int blocks = div_up(d.n() / len, LT);
  // y in LDS while two workgroups and more share a CU's (lines of up to 5 LW cells)
  const size_t tile = LT * (LW + 2) * sizeof(double), tiles = 3 * tile, lds = (2 + (len + LW - 1) / LW) * tile;
#define LSX_LINE(DIR)                                                                                              \
  do {                                                                                                             \
    if (lds <= 65536)                                                                                              \
      k_line_tile<DIR, false><<<blocks, 64, lds, s>>>(sb, d.N, d.M, d.K, dinv, eu, r, c, ch, omega, z_head_fix);   \
    else                                                                                                           \
      k_line_tile<DIR, true><<<blocks, 64, tiles, s>>>(sb, d.N, d.M, d.K, dinv, eu, r, c, ch, omega, z_head_fix);  \
  } while (0)
  if (dir == 0)
    LSX_LINE(0);
  else if (dir == 1)
    LSX_LINE(1);
  else
    LSX_LINE(2);
#undef LSX_LINE
}

void lu_solve(const double* scale, const int* perm, const double* L, const double* U, int n, const double* b,
              double* x, hipStream_t s) {
  k_lu_solve<<<1, LU_SOLVE_THREADS, 0, s>>>(scale, perm, L, U, n, b, x);
}

bool cascade_small_fits(CascadeLevels& C) {
  if (C.count < 2 || C.count > CascadeLevels::MAX) return false;
  auto pitched = [](Dims d) { return (d.N | 1) * d.M * d.K; };
  const long n_last = C.L[C.count - 1].d.n();
  C.off[0] = 0;
  C.c_size = 0;
  C.ch_size = 0;
  long total = 0;
  for (int q = 0; q < C.count; ++q) {
    const long n = C.L[q].d.n();
    if (n > (C.L[q].npts == 7 ? CS_CELLS : CS_CELLS / 4) * CS_THREADS) return false;
    if (q + 1 < C.count && std::max(C.L[q].d.N, std::max(C.L[q].d.M, C.L[q].d.K)) > CS_LEN) return false;
    if (q + 1 < C.count) {
      total += pitched(C.L[q].d);
      C.c_size = std::max(C.c_size, pitched(C.L[q].d));
      if (q > 0) C.ch_size = std::max(C.ch_size, (int)n);
    }
    C.off[q + 1] = (int)total;
  }
  return n_last <= 64 && total + C.c_size + C.ch_size + lu_lds_size((int)n_last) <= CS_LDS;
}

void x_factors_t(const double* coef, int npts, Dims d, const double* dinv, const double* eu, double* xt,
                 hipStream_t s) {
  k_x_factors_t<<<div_up(d.n(), 256), 256, 0, s>>>(coef + slot_sub(npts, 0) * d.n(), dinv, eu, d.N, d.M * d.K, xt);
}

void cascade_small(const CascadeLevels& C, int n_post, double omega, int z_head_fix, const double* lu_scale,
                   const int* lu_perm, const double* L, const double* U, const double* r, double* ch, hipStream_t s) {
  k_cascade_small<<<1, CS_THREADS, 0, s>>>(C, n_post, omega, z_head_fix, lu_scale, lu_perm, L, U, r, ch);
}

void copy(const double* a, double* b, long n, hipStream_t s) { k_copy<<<grid_1d(n), 256, 0, s>>>(a, b, n); }

void scale_copy_f32(const double* w, const double* normw, double* v, float* vf, long n, hipStream_t s) {
  k_scale_copy_f32<<<grid_1d(n), 256, 0, s>>>(w, normw, v, vf, n);
}

void fill_zero(double* b, long n, hipStream_t s) { k_fill_zero<<<grid_1d(n), 256, 0, s>>>(b, n); }

void scale_copy(const double* w, const double* normw, double* v, long n, hipStream_t s) {
  k_scale_copy<<<grid_1d(n), 256, 0, s>>>(w, normw, v, n);
}

void dot_partial(const double* a, const double* b, long n, double* partial, hipStream_t s) {
  k_dot_partial<RED_THREADS><<<reduction_blocks(n), RED_THREADS, 0, s>>>(a, b, n, partial);
}

void dot2(const double* a, const double* b, const double* c, const double* d, long n, double* partial, double* out,
          hipStream_t s) {
  const int nb = reduction_blocks(n);
  k_dot2_partial<RED_THREADS><<<nb, RED_THREADS, 0, s>>>(a, b, c, d, n, partial);
  k_finalize_multi<RED_THREADS><<<2, RED_THREADS, 0, s>>>(partial, nb, out, 0);
}

void finalize(const double* partial, int nb, double* out, int sqrt_flag, hipStream_t s) {
  k_finalize<RED_THREADS><<<1, RED_THREADS, 0, s>>>(partial, nb, out, sqrt_flag);
}

void axpy_dot(double* w, const double* v, const double* pin, double* h, const double* vnext, long n, double* pout,
              hipStream_t s) {
  k_axpy_dot<RED_THREADS><<<reduction_blocks(n), RED_THREADS, 0, s>>>(w, v, pin, h, vnext, n, pout);
}

void sol_update(double* x, const double* Z, long ldz, const double* yk, int count, long n, hipStream_t s) {
  // chunks of 64 coefficients, highest k first (the reference order k = last..0)
  int hi = count;
  while (hi > 0) {
    const int lo = hi > 64 ? hi - 64 : 0;
    YCoef c;
    for (int k = lo; k < hi; ++k) c.y[k - lo] = yk[k];
    k_sol_update_t<double><<<grid_1d(n), 256, 0, s>>>(x, Z + (long)lo * ldz, ldz, c, hi - lo, n);
    hi = lo;
  }
}

int cgs_blocks(long n) {
  long b = (n + 1023) / 1024;
  if (b > CGS_BLOCKS_MAX) b = CGS_BLOCKS_MAX;
  if (b < 1) b = 1;
  return (int)b;
}

void cgs_dot(const double* V, long ldv, int cnt, const double* w, long n, double* partial, double* out,
             hipStream_t s) {
  const int nb = cgs_blocks(n), ng = (cnt + CGS_GROUP - 1) / CGS_GROUP;
  k_cgs_dot<RED_THREADS, double><<<(nb + 7) / 8 * 8 * ng, RED_THREADS, 0, s>>>(V, ldv, cnt, w, n, nb, ng, partial);
  k_finalize_multi<RED_THREADS><<<cnt, RED_THREADS, 0, s>>>(partial, nb, out, 0);
}

void cgs_dot_f32(const float* V, long ldv, int cnt, const double* w, long n, double* partial, double* out,
                 hipStream_t s) {
  const int nb = cgs_blocks(n), ng = (cnt + CGS_GROUP - 1) / CGS_GROUP;
  k_cgs_dot<RED_THREADS, float><<<(nb + 7) / 8 * 8 * ng, RED_THREADS, 0, s>>>(V, ldv, cnt, w, n, nb, ng, partial);
  k_finalize_multi<RED_THREADS><<<cnt, RED_THREADS, 0, s>>>(partial, nb, out, 0);
}

void cgs_update(const double* V, long ldv, int cnt, const double* h, double* w, long n, double* partial,
                double* norm_out, hipStream_t s) {
  const int nb = cgs_blocks(n);
  k_cgs_update<RED_THREADS><<<nb, RED_THREADS, 0, s>>>(V, ldv, cnt, h, w, n, norm_out != nullptr, partial);
  if (norm_out) k_finalize_multi<RED_THREADS><<<1, RED_THREADS, 0, s>>>(partial, nb, norm_out, 1);
}

void cgs_update_scaled(const double* V, long ldv, int cnt, const double* h, const CgsScales& sc, double post,
                       const double* w, double* out, float* out32, long n, double* partial, double* norm_out,
                       hipStream_t s) {
  const int nb = cgs_blocks(n);
  k_cgs_update_scaled<RED_THREADS, 8, 4><<<nb, RED_THREADS, 0, s>>>(V, ldv, cnt, h, sc, post, w, out, out32, n,
                                                                    norm_out != nullptr, partial);
  if (norm_out) k_finalize_multi<RED_THREADS><<<1, RED_THREADS, 0, s>>>(partial, nb, norm_out, 1);
}

void stencil_apply_sym_t(const double* s4, const SymExc& ex, Dims d, const double* x, const double* b, double* y,
                         int mode, double* partial, hipStream_t s) {
  stencil_sym_any<true>(s4, ex, d, x, b, y, mode, partial, s);
}

void stencil_prod_sym_t_f32x(const double* s4, const SymExc& ex, Dims d, const float* x, double* y, hipStream_t s) {
  k_stencil_sym_t_f32x<<<tile_blocks(d), 256, 0, s>>>(s4, d.N, d.M, d.K, ex, x, y);
}

void stencil_prod_sym_f32x(const double* s4, const SymExc& ex, Dims d, const float* x, double* y, hipStream_t s) {
  k_stencil_sym_f32x<<<tile_blocks(d), 256, 0, s>>>(s4, d.N, d.M, d.K, ex, x, y);
}

void stencil7_prod_f32x(const double* coef, Dims d, const float* x, double* y, hipStream_t s) {
  k_stencil7_prod_f32x<<<grid_1d(d.n()), 256, 0, s>>>(coef, d.N, d.M, d.K, x, y);
}

void sol_update_f32(double* x, const float* Z, long ldz, const double* yk, int count, long n, hipStream_t s) {
  int hi = count;
  while (hi > 0) {
    const int lo = hi > 64 ? hi - 64 : 0;
    YCoef c;
    for (int k = lo; k < hi; ++k) c.y[k - lo] = yk[k];
    k_sol_update_t<float><<<grid_1d(n), 256, 0, s>>>(x, Z + (long)lo * ldz, ldz, c, hi - lo, n);
    hi = lo;
  }
}

void bicg_s_update(double* nu, const double* r, double* sv, double alpha, long n, hipStream_t s) {
  k_bicg_s<<<grid_1d(n), 256, 0, s>>>(nu, r, sv, alpha, n);
}

void bicg_sol_update(const double* sv, double* y, double* z, double* x, double* t, double* r, double alpha, double w,
                     long n, hipStream_t s) {
  k_bicg_sol<<<grid_1d(n), 256, 0, s>>>(sv, y, z, x, t, r, alpha, w, n);
}

void bicg_p_update(double* p, const double* nu, const double* r, double coef, double beta, long n, hipStream_t s) {
  k_bicg_p<<<grid_1d(n), 256, 0, s>>>(p, nu, r, coef, beta, n);
}

void sub_vec(const double* b, const double* z, double* r, long n, hipStream_t s) {
  k_sub<<<grid_1d(n), 256, 0, s>>>(b, z, r, n);
}

}  // namespace lsx

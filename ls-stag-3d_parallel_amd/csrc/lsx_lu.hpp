// Device code of the coarsest level's LU substitution, shared by the cascade's and the V-cycle's kernels.
#pragma once

#include <hip/hip_runtime.h>

namespace lsx {
namespace {

// lu_decomposition_sparse_matrix.h:216-259 + decomposition_sparse_matrix_interface.h:43-71.
// The factors (n <= 64) and the right-hand side are staged in LDS by the whole workgroup; one
// wavefront then substitutes, a row to a lane.  Every row's operations keep the reference's order:
// forward the finished unknowns are subtracted as they come, backward a row's products are formed
// by all lanes at once and subtracted one after the other.
struct LuLds {
  double *L, *U, *scale, *rhs;
  int* perm;
};
// doubles of LDS that lu_lds takes
__host__ __device__ constexpr int lu_lds_size(int n) { return 2 * n * n + 3 * n; }
__device__ inline LuLds lu_lds(double* p, int n) {
  return LuLds{p, p + n * n, p + 2 * n * n, p + 2 * n * n + n, reinterpret_cast<int*>(p + 2 * n * n + 2 * n)};
}
__device__ inline void lu_stage(const LuLds& q, int n, const double* __restrict__ scale, const int* __restrict__ perm,
                                const double* __restrict__ L, const double* __restrict__ U) {
  for (int k = threadIdx.x; k < n * n; k += blockDim.x) {
    q.L[k] = L[k];
    q.U[k] = U[k];
  }
  for (int k = threadIdx.x; k < n; k += blockDim.x) {
    q.scale[k] = scale[k];
    q.perm[k] = perm[k];
  }
}
// the value of lane j (uniform j)
__device__ inline double lane_value(double v, int j) {
  const unsigned long long u = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)u, j), hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), j);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
// x into q.rhs (the first wavefront of the workgroup).  CAP >= n: every operand is read from LDS before the
// first step (0: read as needed).
template <int CAP>
__device__ inline void lu_substitute_n(const LuLds& q, int n) {
  const int lane = threadIdx.x, row = lane < n ? lane : n - 1;
  double y = q.scale[q.perm[row]] * q.rhs[q.perm[row]], b = 0.0;
  if constexpr (CAP > 0) {
    double l[CAP], u[CAP], d[CAP];
#pragma unroll
    for (int t = 0; t < CAP; ++t) {
      const int k = t < n ? t : n - 1;
      l[t] = q.L[row * n + k];
      u[t] = q.U[k * n + row];
      d[t] = q.U[k * n + k];
    }
#pragma unroll
    for (int t = 0; t < CAP; ++t)
      if (t < n) {  // uniform
        const double s = y - l[t] * lane_value(y, t);
        y = lane > t ? s : y;
      }
#pragma unroll
    for (int i = CAP - 1; i >= 0; --i)
      if (i < n) {
        const double p = u[i] * b;
        double aux = lane_value(y, i);
#pragma unroll
        for (int j = i + 1; j < CAP; ++j)
          if (j < n) aux -= lane_value(p, j);
        aux = aux / d[i];
        b = lane == i ? aux : b;
      }
  } else {
    for (int t = 0; t < n; ++t) {
      const double s = y - q.L[row * n + t] * lane_value(y, t);
      y = lane > t ? s : y;
    }
    for (int i = n - 1; i >= 0; --i) {
      const double p = q.U[i * n + row] * b;
      double aux = lane_value(y, i);
      for (int j = i + 1; j < n; ++j) aux -= lane_value(p, j);
      aux = aux / q.U[i * n + i];
      b = lane == i ? aux : b;
    }
  }
  if (lane < n) q.rhs[lane] = q.scale[lane] * b;
}
__device__ inline void lu_substitute(const LuLds& q, int n) {
  if (n <= 8)
    lu_substitute_n<8>(q, n);
  else if (n <= 16)
    lu_substitute_n<16>(q, n);
  else
    lu_substitute_n<0>(q, n);
}

}  // namespace
}  // namespace lsx

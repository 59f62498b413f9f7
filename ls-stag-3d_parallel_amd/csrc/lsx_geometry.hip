// Cut-cell geometry of the pressure grid and the pressure operator's coefficients, on the GPU.
//
// One thread per node/cell.  The level-set oscillation fix depends on the order nodes are
// visited (reference ls_stag_uniform_mesh.h:2906-2916 inside the serial sweep
// flow_task_description.h:102-137).  A node can only change there if its level set is positive
// and one of its upper neighbours is negative, so a flag pass marks those few nodes and
// repeated parallel passes over them reach the ordered sweep's result (k_osc_iter); every other
// node keeps its value and all later stages read final values only.
//
// Built with -ffp-contract=off: every formula is evaluated with the operation order of the
// reference expressions it restates.

#include <hip/hip_runtime.h>

#include <cmath>
#include <mutex>

#include "lsx_geometry.hpp"

namespace lsx {
namespace geo {

namespace {

constexpr double PLUS_TINY = 1e-16;
constexpr double EQ_DOUBLE = 1e-5;
constexpr double THETA_EQ_ZERO = 0.05;
constexpr double EQ_TINY_DOUBLE = 1e-12;
constexpr double ONE_THIRD = 1.0 / 3.0;
constexpr int FLUID_SIDE = 1111;

__device__ inline void decode(long i, int N, int M, int* x, int* y, int* z) {
  const long NM = (long)N * M;
  *z = (int)(i / NM);
  const long r = i - (long)*z * NM;
  *y = (int)(r / N);
  *x = (int)(r - (long)*y * N);
}

__device__ inline bool in_box(int x, int y, const Box& b) { return x >= b.hs && x < b.hf && y >= b.vs && y < b.vf; }

// ---- six-patch bicubic Bezier body ----------------------------------------------------------------
// Patches on the six cube faces: face f has normal axis BZ_A[f] with sign BZ_S[f], u along BZ_U[f]
// and v along BZ_V[f] (S_u x S_v outwards); control point (i, j) of face f, coordinate c, at
// ctrl[(f * 16 + i * 4 + j) * 3 + c].  phi = +distance inside, -distance outside: per patch 12
// Newton steps from the cube-sphere inverse of the point (a coordinate at its bound with the
// gradient pointing out holds there while the other takes a 1D step; Gauss-Newton where the
// Hessian is not positive definite), smallest distance wins, side from (x - S) . (S_u x S_v).
// BZ_A = {0, 0, 1, 1, 2, 2}, BZ_S = {1, -1, 1, -1, 1, -1}, BZ_U = {1, 2, 2, 0, 0, 1}, BZ_V = {2, 1, 0, 2, 1, 0}
__device__ inline int bz_next_axis(int a, int k) { return a + k < 3 ? a + k : a + k - 3; }
__device__ inline int bz_a(int f) { return f >> 1; }
__device__ inline int bz_u(int f) { return bz_next_axis(f >> 1, 1 + (f & 1)); }
__device__ inline int bz_v(int f) { return bz_next_axis(f >> 1, 2 - (f & 1)); }
__device__ inline double bz_pick(const double* d, int k) { return k == 0 ? d[0] : (k == 1 ? d[1] : d[2]); }

__device__ inline void bz_basis(double t, double* b, double* db, double* ddb) {
  const double s = 1.0 - t;
  b[0] = s * s * s;
  b[1] = 3.0 * t * s * s;
  b[2] = 3.0 * t * t * s;
  b[3] = t * t * t;
  db[0] = -3.0 * s * s;
  db[1] = 3.0 * s * s - 6.0 * t * s;
  db[2] = 6.0 * t * s - 3.0 * t * t;
  db[3] = 3.0 * t * t;
  ddb[0] = 6.0 * s;
  ddb[1] = 18.0 * t - 12.0;
  ddb[2] = 6.0 - 18.0 * t;
  ddb[3] = 6.0 * t;
}

// S, S_u and S_v of patch P at (u, v): each row i of the control net is first reduced along v
// (q_i = sum_j B_j(v) P_ij and its v derivative), then the rows along u
__device__ inline void bz_eval1(const double* __restrict__ P, double u, double v, double* S, double* Su, double* Sv) {
  double bu[4], dbu[4], ddbu[4], bv[4], dbv[4], ddbv[4];
  bz_basis(u, bu, dbu, ddbu);
  bz_basis(v, bv, dbv, ddbv);
  for (int c = 0; c < 3; ++c) S[c] = Su[c] = Sv[c] = 0.0;
  for (int i = 0; i < 4; ++i)
    for (int c = 0; c < 3; ++c) {
      double q = 0.0, dq = 0.0;
      for (int j = 0; j < 4; ++j) {
        const double p = P[(i * 4 + j) * 3 + c];
        q += bv[j] * p;
        dq += dbv[j] * p;
      }
      S[c] += bu[i] * q;
      Su[c] += dbu[i] * q;
      Sv[c] += bu[i] * dq;
    }
}

// r . S_uu, r . S_uv and r . S_vv of patch P at (u, v), through w_ij = P_ij . r
__device__ inline void bz_eval2(const double* __restrict__ P, double u, double v, const double* r, double* ruu,
                                double* ruv, double* rvv) {
  double bu[4], dbu[4], ddbu[4], bv[4], dbv[4], ddbv[4];
  bz_basis(u, bu, dbu, ddbu);
  bz_basis(v, bv, dbv, ddbv);
  double a = 0.0, b = 0.0, c = 0.0;
  for (int i = 0; i < 4; ++i) {
    double q = 0.0, dq = 0.0, ddq = 0.0;
    for (int j = 0; j < 4; ++j) {
      const double* pij = P + (i * 4 + j) * 3;
      const double w = pij[0] * r[0] + pij[1] * r[1] + pij[2] * r[2];
      q += bv[j] * w;
      dq += dbv[j] * w;
      ddq += ddbv[j] * w;
    }
    a += ddbu[i] * q;
    b += dbu[i] * dq;
    c += bu[i] * ddq;
  }
  *ruu = a;
  *ruv = b;
  *rvv = c;
}

__device__ inline double bz_dot(const double* a, const double* b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }
__device__ inline double bz_clamp(double t) { return t < 0.0 ? 0.0 : (t > 1.0 ? 1.0 : t); }

// closest point of the winning patch: phi = sgn * |X - S(u, v)| with r = X - S
struct BzHit {
  int f;
  double u, v, r[3], dist, sgn;
};

// Newton search for the closest point of patch f (control values P) to X (d: X in the body's
// normalised coordinates, for the start); returns |X - S|^2 with (u, v), r = X - S and
// side = r . (S_u x S_v) there.  A step that leaves (u, v) unchanged ends the search: the steps
// after it would repeat it exactly.
__device__ inline double bz_patch(const double* __restrict__ P, int f, const double* X, const double* d, double& u,
                                  double& v, double* r, double& side) {
  const double da = fabs(bz_pick(d, bz_a(f)));
  u = 0.5;
  v = 0.5;
  if (da > 0.0) {
    u = bz_clamp(0.5 * (bz_pick(d, bz_u(f)) / da + 1.0));
    v = bz_clamp(0.5 * (bz_pick(d, bz_v(f)) / da + 1.0));
  }
  double S[3], Su[3], Sv[3];
  for (int it = 0; it < 12; ++it) {
    bz_eval1(P, u, v, S, Su, Sv);
    double q[3];
    for (int c = 0; c < 3; ++c) q[c] = S[c] - X[c];
    const double gu = bz_dot(Su, q), gv = bz_dot(Sv, q);
    const double juu = bz_dot(Su, Su), juv = bz_dot(Su, Sv), jvv = bz_dot(Sv, Sv);
    double ruu, ruv, rvv;
    bz_eval2(P, u, v, q, &ruu, &ruv, &rvv);
    double huu = juu + ruu, huv = juv + ruv, hvv = jvv + rvv;
    double det = huu * hvv - huv * huv;
    if (!(det > 0.0 && huu > 0.0)) {
      huu = juu;
      huv = juv;
      hvv = jvv;
      det = huu * hvv - huv * huv;
    }
    const bool hold_u = (u >= 1.0 && gu < 0.0) || (u <= 0.0 && gu > 0.0);
    const bool hold_v = (v >= 1.0 && gv < 0.0) || (v <= 0.0 && gv > 0.0);
    double du = 0.0, dv = 0.0;
    if (hold_u && hold_v) break;
    if (hold_u) {
      dv = -gv / (hvv > 0.0 ? hvv : jvv);
    } else if (hold_v) {
      du = -gu / (huu > 0.0 ? huu : juu);
    } else {
      if (!(det > 0.0)) break;
      du = -(hvv * gu - huv * gv) / det;
      dv = -(huu * gv - huv * gu) / det;
    }
    const double un = bz_clamp(u + du), vn = bz_clamp(v + dv);
    if (un == u && vn == v) break;
    u = un;
    v = vn;
  }
  bz_eval1(P, u, v, S, Su, Sv);
  for (int c = 0; c < 3; ++c) r[c] = X[c] - S[c];
  const double nrm[3] = {Su[1] * Sv[2] - Su[2] * Sv[1], Su[2] * Sv[0] - Su[0] * Sv[2], Su[0] * Sv[1] - Su[1] * Sv[0]};
  side = bz_dot(r, nrm);
  return bz_dot(r, r);
}

// A workgroup's copy of the control values, a patch BZ_STRIDE apart (lanes on different patches read
// different banks), and the bounding box of each patch's control points (the patch lies in their
// convex hull)
constexpr int BZ_STRIDE = 53;
struct BzBody {
  double P[6 * BZ_STRIDE], lo[18], hi[18];
};
// every thread of the workgroup takes part
__device__ inline void bz_load(const double* __restrict__ ctrl, BzBody& B) {
  for (int k = threadIdx.x; k < 288; k += blockDim.x) B.P[k / 48 * BZ_STRIDE + k % 48] = ctrl[k];
  __syncthreads();
  if (threadIdx.x < 18) {
    const double* P = B.P + threadIdx.x / 3 * BZ_STRIDE + threadIdx.x % 3;
    double lo = P[0], hi = P[0];
    for (int k = 1; k < 16; ++k) {
      lo = fmin(lo, P[3 * k]);
      hi = fmax(hi, P[3 * k]);
    }
    B.lo[threadIdx.x] = lo;
    B.hi[threadIdx.x] = hi;
  }
  __syncthreads();
}
// squared distance from X to the bounding box of patch f
__device__ inline double bz_box_dist2(const BzBody& B, int f, const double* X) {
  double acc = 0.0;
  for (int c = 0; c < 3; ++c) {
    const double lo = B.lo[3 * f + c], hi = B.hi[3 * f + c];
    const double e = X[c] < lo ? lo - X[c] : (X[c] > hi ? X[c] - hi : 0.0);
    acc += e * e;
  }
  return acc;
}

// The patch with the smallest distance wins, the lowest index among equal distances.  Each point
// first searches its home patch (the cube face its normalised direction points to), then, in
// order, every other patch whose control-point box comes within the best distance so far plus a
// margin of 1e-12, far above rounding (a patch further away cannot win or tie).  A search is up to
// 13 evaluations in FP64, so what counts is how many a wavefront makes: the lanes search their
// own patches at the same time, control values from LDS, where going through the patches in turn
// with uniform control values took every patch that any lane of the wavefront needed.
__device__ void bezier_closest(const BzBody& B, const double* c0, const double* a0, double x, double y, double z,
                               BzHit& hit) {
  const double X[3] = {x, y, z};
  double d[3];
  for (int c = 0; c < 3; ++c) d[c] = (X[c] - c0[c]) / a0[c];
  int ax = 0;
  double da = d[0];
  for (int c = 1; c < 3; ++c)
    if (fabs(d[c]) > fabs(da)) {
      ax = c;
      da = d[c];
    }
  const int home = 2 * ax + (da < 0.0 ? 1 : 0);  // faces 2a, 2a + 1: normal axis a, sign + / -
  double best = 0.0, side = 0.0;
  int f = home, next = 0;
  bool first = true;
  for (;;) {
    double u, v, r[3], sd;
    const double dist2 = bz_patch(B.P + f * BZ_STRIDE, f, X, d, u, v, r, sd);
    if (first || dist2 < best || (dist2 == best && f < hit.f)) {
      best = dist2;
      side = sd;
      hit.f = f;
      hit.u = u;
      hit.v = v;
      for (int c = 0; c < 3; ++c) hit.r[c] = r[c];
    }
    first = false;
    for (; next < 6; ++next) {
      if (next == home) continue;
      const double m = sqrt(bz_box_dist2(B, next, X)) - 1e-12;
      if (!(m > 0.0 && m * m > best)) break;
    }
    if (next >= 6) break;
    f = next++;
  }
  const double dist = sqrt(best);
  hit.dist = dist;
  hit.sgn = side > 0.0 ? -1.0 : 1.0;
}

// ---- level set -------------------------------------------------------------------------------
__global__ void k_level_set(const double* __restrict__ cx, const double* __restrict__ cy, const double* __restrict__ cz,
                            int N, int M, int K, Box box, Body body, double* __restrict__ phi) {
  const long n = (long)N * M * K;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    int x, y, z;
    decode(i, N, M, &x, &y, &z);
    double v = 0.0;
    if (in_box(x, y, box)) {
      if (body.kind == BODY_SPHERE) {
        const double qx = cx[x] - body.c[0], qy = cy[y] - body.c[1], qz = cz[z] - body.c[2];
        v = body.a[0] - sqrt(qx * qx + qy * qy + qz * qz);
      } else {
        const double s = fmin(body.a[0], fmin(body.a[1], body.a[2]));
        const double qx = (cx[x] - body.c[0]) / body.a[0], qy = (cy[y] - body.c[1]) / body.a[1],
                     qz = (cz[z] - body.c[2]) / body.a[2];
        v = s * (1.0 - sqrt(qx * qx + qy * qy + qz * qz));
      }
    }
    phi[i] = v;
  }
}

// the level set of a Bezier body, a wavefront to 4 x 4 x 4 nodes (neighbours search the same patches),
// a workgroup to 8 x 8 x 4.  64^3: 480 us with 64 nodes of a row a wavefront and the patches in
// turn, 232 so (the shape gradient's closest points at 72 x 64 x 64: 238 -> 75)
__global__ void __launch_bounds__(256) k_level_set_bezier(const double* __restrict__ cx, const double* __restrict__ cy,
                                                          const double* __restrict__ cz, int N, int M, int K, Box box,
                                                          Body body, double* __restrict__ phi) {
  __shared__ BzBody B;
  bz_load(body.ctrl, B);
  const int gx = (N + 7) / 8, gy = (M + 7) / 8, t = threadIdx.x, w = t >> 6;
  const int x = (int)(blockIdx.x % gx) * 8 + (w & 1) * 4 + (t & 3);
  const int y = (int)(blockIdx.x / gx % gy) * 8 + (w >> 1) * 4 + ((t >> 2) & 3);
  const int z = (int)(blockIdx.x / gx / gy) * 4 + ((t >> 4) & 3);
  if (x >= N || y >= M || z >= K) return;
  double v = 0.0;
  if (in_box(x, y, box)) {
    BzHit hit;
    bezier_closest(B, body.c, body.a, cx[x], cy[y], cz[z], hit);
    v = hit.sgn < 0.0 ? -hit.dist : hit.dist;
  }
  phi[x + (long)N * (y + (long)M * z)] = v;
}

__global__ void k_osc_flags(const double* __restrict__ phi, int N, int M, int K, Box box, unsigned char* __restrict__ flag) {
  const long n = (long)N * M * K, NM = (long)N * M;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    int x, y, z;
    decode(i, N, M, &x, &y, &z);
    unsigned char f = 0;
    if (in_box(x, y, box) && phi[i] > EQ_DOUBLE) {
      const bool mid = z > 0 && z < K - 1;
      f = (phi[i + 1] < 0) || (phi[i + N] < 0) || (mid && phi[i + NM] < 0);
    }
    flag[i] = f;
  }
}

__device__ inline void check_osc(double& f, double lower, double upper) {
  if ((f > EQ_DOUBLE) && (lower < 0) && (upper < 0)) f = 0.5 * (lower + upper);
}

// The reference visits nodes in index order and updates phi in place, so a flagged node reads
// the final values of its lower neighbours (j-1, j-N, j-NM: visited before it) and the original
// values of its upper ones.  One pass recomputes every flagged node from the current lower
// values (`cur`) and the original upper values (`phi0`) into `nxt`; node j depends only on nodes
// below it, so repeating the pass until nothing changes reproduces the ordered sweep exactly.
__global__ void k_osc_iter(const double* __restrict__ phi0, const unsigned char* __restrict__ flag,
                           const double* __restrict__ cur, double* __restrict__ nxt, int N, int M, int K,
                           int* __restrict__ changed) {
  const long n = (long)N * M * K, NM = (long)N * M;
  for (long j = blockIdx.x * (long)blockDim.x + threadIdx.x; j < n; j += (long)gridDim.x * blockDim.x) {
    if (!flag[j]) continue;
    const int z = (int)(j / NM);
    double f = phi0[j];
    check_osc(f, cur[j - 1], phi0[j + 1]);
    check_osc(f, cur[j - N], phi0[j + N]);
    if (z > 0 && z < K - 1) check_osc(f, cur[j - NM], phi0[j + NM]);
    if (f != cur[j]) *changed = 1;
    nxt[j] = f;
  }
}

__device__ inline double edge_fraction(double f, double fo) {
  return (f * fo < 0) ? ((f > 0) ? (fo / (fo - f)) : (f / (f - fo))) : ((f > -fo) ? 0.0 : 1.0);
}

// edge fractions of the edges below node (x, y, z) along x, y and z; phi(dx, dy, dz) reads a node near it
template <class P>
__device__ inline void alpha_of(P phi, int x, int y, int z, int K, const Box& box, double (&a)[3]) {
  a[0] = a[1] = a[2] = 1.0;
  if (in_box(x, y, box)) {
    const double f = phi(0, 0, 0);
    a[0] = edge_fraction(f, phi(-1, 0, 0));
    a[1] = edge_fraction(f, phi(0, -1, 0));
    a[2] = (z == 0 || z == K - 1) ? ((f > 0.0) ? 0.0 : 1.0) : edge_fraction(f, phi(0, 0, -1));
  }
}

__global__ void k_alpha(const double* __restrict__ phi, int N, int M, int K, Box box, double* __restrict__ ax,
                        double* __restrict__ ay, double* __restrict__ az) {
  const long n = (long)N * M * K, NM = (long)N * M;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    int x, y, z;
    decode(i, N, M, &x, &y, &z);
    double a[3];
    alpha_of([&](int dx, int dy, int dz) { return phi[i + dx + (long)N * dy + NM * dz]; }, x, y, z, K, box, a);
    ax[i] = a[0];
    ay[i] = a[1];
    az[i] = a[2];
  }
}

// ---- types -----------------------------------------------------------------------------------
__device__ inline int type_of_side(double phi, double phiW, double phiSW, double phiS) {
  int number = (phiS < EQ_DOUBLE) ? 1 : 0;
  if (phiSW < EQ_DOUBLE) number += 10;
  if (phiW < EQ_DOUBLE) number += 100;
  if (phi < EQ_DOUBLE) number += 1000;
  return number;
}

__device__ inline int border_type(int x, int y, int z, int N, int M, int K) {
  const bool w = x == 0, e = x == N - 1, s = y == 0, nn = y == M - 1, b = z == 0, t = z == K - 1;
  if (b) {
    if (s) return w ? BSW_Corner : (e ? BSE_Corner : BS_Edge);
    if (nn) return w ? BNW_Corner : (e ? BNE_Corner : BN_Edge);
    return w ? BW_Edge : (e ? BE_Edge : B_Border);
  }
  if (t) {
    if (s) return w ? TSW_Corner : (e ? TSE_Corner : TS_Edge);
    if (nn) return w ? TNW_Corner : (e ? TNE_Corner : TN_Edge);
    return w ? TW_Edge : (e ? TE_Edge : T_Border);
  }
  if (s) return w ? SW_Edge : (e ? SE_Edge : S_Border);
  if (nn) return w ? NW_Edge : (e ? NE_Edge : N_Border);
  if (w) return W_Border;
  if (e) return E_Border;
  return FluidCell;
}

// type code of cell (x, y, z) and of its east, north and top faces; p as in alpha_of
template <class P>
__device__ inline int type_of(P p, int x, int y, int z, int N, int M, int K, const Box& box, int (&side)[3]) {
  int t = border_type(x, y, z, N, M, K);
  side[0] = side[1] = side[2] = FLUID_SIDE;
  if (in_box(x, y, box)) {
    const double phi = p(0, 0, 0), phiW = p(-1, 0, 0), phiS = p(0, -1, 0);
    const int tT = type_of_side(phi, phiW, p(-1, -1, 0), phiS);
    if (z == 0 || z == K - 1) {
      side[0] = type_of_side(phi, phiS, phiS, phi);
      side[1] = type_of_side(phi, phiW, phiW, phi);
      side[2] = tT;
      t = (tT == 0) ? SolidCell : (z == 0 ? B_Border : T_Border);
    } else {
      const double phiSB = p(0, -1, -1), phiB = p(0, 0, -1), phiBW = p(-1, 0, -1);
      side[0] = type_of_side(phi, phiS, phiSB, phiB);
      side[1] = type_of_side(phi, phiW, phiBW, phiB);
      side[2] = tT;
      t = tT * 10000 + type_of_side(phiB, phiBW, p(-1, -1, -1), phiSB);
    }
  }
  return t;
}

__global__ void k_types(const double* __restrict__ p, int N, int M, int K, Box box, int* __restrict__ type,
                        int* __restrict__ sx, int* __restrict__ sy, int* __restrict__ sz) {
  const long n = (long)N * M * K, NM = (long)N * M;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    int x, y, z, side[3];
    decode(i, N, M, &x, &y, &z);
    type[i] = type_of([&](int dx, int dy, int dz) { return p[i + dx + (long)N * dy + NM * dz]; }, x, y, z, N, M, K, box,
                      side);
    sx[i] = side[0];
    sy[i] = side[1];
    sz[i] = side[2];
  }
}

// ---- face fractions ---------------------------------------------------------------------------
__device__ inline double face_theta(int side, double P0, double P1, double Q0, double Q1) {
  double t;
  switch (side) {
    case FLUID_SIDE: return 1.0;
    case 0: return 0.0;
    case 11: case 1100: t = 0.5 * (P0 + P1); break;
    case 1001: case 110: t = 0.5 * (Q0 + Q1); break;
    case 1011: t = 1.0 - 0.5 * (1.0 - P1) * (1.0 - Q0); break;
    case 111: t = 1.0 - 0.5 * (1.0 - P0) * (1.0 - Q0); break;
    case 1101: t = 1.0 - 0.5 * (1.0 - P1) * (1.0 - Q1); break;
    case 1110: t = 1.0 - 0.5 * (1.0 - P0) * (1.0 - Q1); break;
    case 1: t = 0.5 * P0 * Q1; break;
    case 10: t = 0.5 * P1 * Q1; break;
    case 1000: t = 0.5 * P0 * Q0; break;
    case 100: t = 0.5 * P1 * Q0; break;
    default: return 1.0;
  }
  return t < THETA_EQ_ZERO ? 0.0 : t;
}

// open fractions of the east, north and top faces of cell (x, y, z); a(c, dx, dy, dz) reads edge
// fraction c near it
template <class A>
__device__ inline void theta_of(A a, const int (&side)[3], int x, int y, int z, int K, const Box& box, double (&t)[3]) {
  t[0] = t[1] = t[2] = 1.0;
  if (in_box(x, y, box)) {
    t[2] = face_theta(side[2], a(1, 0, 0, 0), a(1, -1, 0, 0), a(0, 0, 0, 0), a(0, 0, -1, 0));
    if (z == 0 || z == K - 1) {
      const double ay = a(1, 0, 0, 0), ax = a(0, 0, 0, 0);
      t[0] = ay < THETA_EQ_ZERO ? 0.0 : ay;
      t[1] = ax < THETA_EQ_ZERO ? 0.0 : ax;
    } else {
      t[0] = face_theta(side[0], a(2, 0, 0, 0), a(2, 0, -1, 0), a(1, 0, 0, 0), a(1, 0, 0, -1));
      t[1] = face_theta(side[1], a(2, 0, 0, 0), a(2, -1, 0, 0), a(0, 0, 0, 0), a(0, 0, 0, -1));
    }
  }
}

__global__ void k_theta(const double* __restrict__ ax, const double* __restrict__ ay, const double* __restrict__ az,
                        const int* __restrict__ sx, const int* __restrict__ sy, const int* __restrict__ sz, int N, int M,
                        int K, Box box, double* __restrict__ tx, double* __restrict__ ty, double* __restrict__ tz) {
  const long n = (long)N * M * K, NM = (long)N * M;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    int x, y, z;
    decode(i, N, M, &x, &y, &z);
    const int side[3] = {sx[i], sy[i], sz[i]};
    double t[3];
    theta_of(
        [&](int c, int dx, int dy, int dz) {
          const long j = i + dx + (long)N * dy + NM * dz;
          return c == 0 ? ax[j] : (c == 1 ? ay[j] : az[j]);
        },
        side, x, y, z, K, box, t);
    tx[i] = t[0];
    ty[i] = t[1];
    tz[i] = t[2];
  }
}

// ---- cut volumes --------------------------------------------------------------------------------
// Formula families of the reference volume table; each cut code names a family and the
// alpha/theta entries (component, corner offset) it reads.
enum Fam : unsigned char { F_TET, F_HEP3, F_PRISM, F_HEP5, F_HEX5, F_HEP6 };
struct Ref {
  signed char dx, dy, dz, comp;
};
struct Rule {
  int code;
  unsigned char fam, axis, sel, pad;
  Ref a, b, a2, b2;
};

#define R_(dx, dy, dz, c) Ref{dx, dy, dz, c}
#define NONE R_(0, 0, 0, 0)
// sorted by code for binary search
__constant__ Rule c_rules[] = {
    {1, F_TET, 0, 0, 0, R_(0, -1, -1, 0), R_(0, 0, 0, 0), NONE, NONE},
    {10, F_TET, 0, 0, 0, R_(0, -1, -1, 0), R_(-1, 0, 0, 0), NONE, NONE},
    {11, F_PRISM, 0, 0, 0, NONE, NONE, NONE, NONE},
    {100, F_TET, 0, 0, 0, R_(0, 0, -1, 0), R_(-1, 0, 0, 0), NONE, NONE},
    {110, F_PRISM, 1, 0, 0, NONE, NONE, NONE, NONE},
    {111, F_HEX5, 1, 1, 0, R_(0, 0, -1, 0), R_(0, 0, 0, 1), NONE, NONE},
    {1000, F_TET, 0, 0, 0, R_(0, 0, -1, 0), R_(0, 0, 0, 0), NONE, NONE},
    {1001, F_PRISM, 1, 0, 0, NONE, NONE, NONE, NONE},
    {1011, F_HEX5, 1, 1, 0, R_(0, 0, -1, 0), R_(-1, 0, 0, 1), NONE, NONE},
    {1100, F_PRISM, 0, 0, 0, NONE, NONE, NONE, NONE},
    {1101, F_HEX5, 1, 0, 0, R_(0, -1, -1, 0), R_(-1, 0, 0, 1), NONE, NONE},
    {1110, F_HEX5, 1, 0, 0, R_(0, -1, -1, 0), R_(0, 0, 0, 1), NONE, NONE},
    {1111, F_PRISM, 0, 0, 0, NONE, NONE, NONE, NONE},
    {10000, F_TET, 0, 0, 0, R_(0, -1, 0, 0), R_(0, 0, 0, 0), NONE, NONE},
    {10001, F_PRISM, 2, 0, 0, NONE, NONE, NONE, NONE},
    {10011, F_HEX5, 0, 0, 0, R_(-1, -1, 0, 2), R_(0, -1, 0, 0), NONE, NONE},
    {11001, F_HEX5, 2, 1, 0, R_(0, 0, 0, 1), R_(0, 0, 0, 2), NONE, NONE},
    {11011, F_HEP6, 0, 1, 0, R_(0, 0, 0, 2), R_(0, 0, -1, 0), R_(0, 0, 0, 1), R_(0, -1, 0, 0)},
    {11111, F_HEP5, 1, 0, 0, R_(0, -1, 0, 0), R_(-1, 0, 0, 1), NONE, NONE},
    {100000, F_TET, 0, 0, 0, R_(0, -1, 0, 0), R_(-1, 0, 0, 0), NONE, NONE},
    {100010, F_PRISM, 2, 0, 0, NONE, NONE, NONE, NONE},
    {100011, F_HEX5, 0, 1, 0, R_(0, -1, 0, 2), R_(0, -1, 0, 0), NONE, NONE},
    {100110, F_HEX5, 2, 1, 0, R_(-1, 0, 0, 1), R_(-1, 0, 0, 2), NONE, NONE},
    {100111, F_HEP6, 0, 0, 0, R_(-1, 0, 0, 2), R_(0, 0, -1, 0), R_(-1, 0, 0, 1), R_(0, -1, 0, 0)},
    {101111, F_HEP5, 1, 0, 0, R_(0, -1, 0, 0), R_(0, 0, 0, 1), NONE, NONE},
    {110000, F_PRISM, 0, 0, 0, NONE, NONE, NONE, NONE},
    {110001, F_HEX5, 0, 0, 0, R_(-1, -1, 0, 2), R_(0, -1, -1, 0), NONE, NONE},
    {110010, F_HEX5, 0, 1, 0, R_(0, -1, 0, 2), R_(0, -1, -1, 0), NONE, NONE},
    {110011, F_PRISM, 0, 0, 0, NONE, NONE, NONE, NONE},
    {110111, F_HEP5, 0, 0, 0, R_(-1, 0, 0, 2), R_(0, 0, -1, 0), NONE, NONE},
    {111011, F_HEP5, 0, 1, 0, R_(0, 0, 0, 2), R_(0, 0, -1, 2), NONE, NONE},
    {111111, F_PRISM, 0, 0, 0, NONE, NONE, NONE, NONE},
    {1000000, F_TET, 0, 0, 0, R_(0, 0, 0, 0), R_(-1, 0, 0, 0), NONE, NONE},
    {1000100, F_PRISM, 2, 0, 0, NONE, NONE, NONE, NONE},
    {1000110, F_HEX5, 2, 1, 0, R_(-1, 0, 0, 1), R_(-1, -1, 0, 2), NONE, NONE},
    {1001100, F_HEX5, 0, 1, 0, R_(0, 0, 0, 2), R_(0, 0, 0, 0), NONE, NONE},
    {1001110, F_HEP6, 0, 0, 0, R_(-1, -1, 0, 2), R_(0, -1, -1, 0), R_(-1, 0, 0, 1), R_(0, 0, 0, 0)},
    {1001111, F_HEP5, 1, 1, 0, R_(0, 0, 0, 0), R_(-1, 0, 0, 1), NONE, NONE},
    {1100000, F_PRISM, 1, 0, 0, NONE, NONE, NONE, NONE},
    {1100010, F_HEX5, 2, 0, 0, R_(-1, 0, -1, 1), R_(-1, 0, 0, 2), NONE, NONE},
    {1100100, F_HEX5, 2, 0, 0, R_(-1, 0, -1, 1), R_(-1, -1, 0, 2), NONE, NONE},
    {1100110, F_PRISM, 1, 0, 0, NONE, NONE, NONE, NONE},
    {1100111, F_HEP5, 2, 0, 0, R_(0, 0, -1, 1), R_(0, -1, 0, 2), NONE, NONE},
    {1101110, F_HEP5, 2, 0, 0, R_(0, 0, -1, 1), R_(0, 0, 0, 2), NONE, NONE},
    {1101111, F_PRISM, 1, 0, 0, NONE, NONE, NONE, NONE},
    {1110000, F_HEX5, 1, 1, 0, R_(0, 0, 0, 0), R_(0, 0, 0, 1), NONE, NONE},
    {1110010, F_HEP6, 0, 0, 0, R_(-1, 0, 0, 2), R_(0, 0, 0, 0), R_(-1, 0, -1, 1), R_(0, -1, -1, 0)},
    {1110011, F_HEP5, 0, 0, 0, R_(-1, 0, 0, 2), R_(0, 0, 0, 0), NONE, NONE},
    {1110110, F_HEP5, 2, 1, 0, R_(0, 0, 0, 1), R_(0, -1, 0, 2), NONE, NONE},
    {1110111, F_PRISM, 2, 0, 0, NONE, NONE, NONE, NONE},
    {1111111, F_HEP3, 0, 0, 0, R_(0, 0, 0, 0), R_(0, 0, 0, 0), NONE, NONE},
    {10000000, F_TET, 0, 0, 0, R_(0, 0, 0, 0), R_(0, 0, 0, 0), NONE, NONE},
    {10001000, F_PRISM, 2, 0, 0, NONE, NONE, NONE, NONE},
    {10001001, F_HEX5, 2, 1, 0, R_(0, 0, 0, 1), R_(0, -1, 0, 2), NONE, NONE},
    {10001100, F_HEX5, 0, 0, 0, R_(-1, 0, 0, 2), R_(0, 0, 0, 0), NONE, NONE},
    {10001101, F_HEP6, 0, 1, 0, R_(0, -1, 0, 2), R_(0, -1, -1, 0), R_(0, 0, 0, 1), R_(0, 0, 0, 0)},
    {10001111, F_HEP5, 1, 1, 0, R_(0, 0, 0, 0), R_(0, 0, 0, 1), NONE, NONE},
    {10010000, F_PRISM, 1, 0, 0, NONE, NONE, NONE, NONE},
    {10010001, F_HEX5, 2, 0, 0, R_(0, 0, -1, 1), R_(0, 0, 0, 2), NONE, NONE},
    {10011000, F_HEX5, 2, 0, 0, R_(0, 0, -1, 1), R_(0, -1, 0, 2), NONE, NONE},
    {10011001, F_PRISM, 1, 0, 0, NONE, NONE, NONE, NONE},
    {10011011, F_HEP5, 2, 0, 0, R_(-1, 0, -1, 1), R_(-1, -1, 0, 2), NONE, NONE},
    {10011101, F_HEP5, 2, 0, 0, R_(-1, 0, -1, 1), R_(-1, 0, 0, 2), NONE, NONE},
    {10011111, F_PRISM, 1, 0, 0, NONE, NONE, NONE, NONE},
    {10110000, F_HEX5, 1, 1, 0, R_(0, 0, 0, 0), R_(-1, 0, 0, 1), NONE, NONE},
    {10110001, F_HEP6, 0, 1, 0, R_(0, 0, 0, 2), R_(0, 0, 0, 0), R_(0, 0, -1, 1), R_(0, -1, -1, 0)},
    {10110011, F_HEP5, 0, 1, 0, R_(0, 0, 0, 2), R_(0, 0, 0, 0), NONE, NONE},
    {10111001, F_HEP5, 2, 1, 0, R_(-1, 0, 0, 1), R_(-1, -1, 0, 2), NONE, NONE},
    {10111011, F_PRISM, 2, 0, 0, NONE, NONE, NONE, NONE},
    {10111111, F_HEP3, 0, 0, 0, R_(0, 0, 0, 0), R_(-1, 0, 0, 0), NONE, NONE},
    {11000000, F_PRISM, 0, 0, 0, NONE, NONE, NONE, NONE},
    {11000100, F_HEX5, 0, 1, 0, R_(0, 0, 0, 2), R_(0, 0, -1, 0), NONE, NONE},
    {11001000, F_HEX5, 0, 0, 0, R_(-1, 0, 0, 2), R_(0, 0, -1, 0), NONE, NONE},
    {11001100, F_PRISM, 0, 0, 0, NONE, NONE, NONE, NONE},
    {11001101, F_HEP5, 0, 1, 0, R_(0, -1, 0, 2), R_(0, -1, -1, 0), NONE, NONE},
    {11001110, F_HEP5, 0, 0, 0, R_(-1, -1, 0, 2), R_(0, -1, -1, 0), NONE, NONE},
    {11001111, F_PRISM, 0, 0, 0, NONE, NONE, NONE, NONE},
    {11010000, F_HEX5, 1, 0, 0, R_(0, -1, 0, 0), R_(-1, 0, 0, 1), NONE, NONE},
    {11011000, F_HEP6, 0, 1, 0, R_(0, -1, 0, 2), R_(0, 0, -1, 0), R_(0, 0, -1, 1), R_(0, -1, 0, 0)},
    {11011001, F_HEP5, 2, 1, 0, R_(-1, 0, 0, 1), R_(-1, 0, 0, 2), NONE, NONE},
    {11011100, F_HEP5, 0, 1, 0, R_(0, -1, 0, 2), R_(0, -1, 0, 0), NONE, NONE},
    {11011101, F_PRISM, 2, 0, 0, NONE, NONE, NONE, NONE},
    {11011111, F_HEP3, 0, 0, 0, R_(0, -1, 0, 0), R_(-1, 0, 0, 0), NONE, NONE},
    {11100000, F_HEX5, 1, 0, 0, R_(0, -1, 0, 0), R_(0, 0, 0, 1), NONE, NONE},
    {11100100, F_HEP6, 0, 0, 0, R_(-1, -1, 0, 2), R_(0, -1, 0, 0), R_(-1, 0, -1, 1), R_(0, 0, -1, 0)},
    {11100110, F_HEP5, 2, 1, 0, R_(0, 0, 0, 1), R_(0, 0, 0, 2), NONE, NONE},
    {11101100, F_HEP5, 0, 0, 0, R_(-1, -1, 0, 2), R_(0, -1, 0, 0), NONE, NONE},
    {11101110, F_PRISM, 2, 0, 0, NONE, NONE, NONE, NONE},
    {11101111, F_HEP3, 0, 0, 0, R_(0, -1, 0, 0), R_(0, 0, 0, 0), NONE, NONE},
    {11110000, F_PRISM, 0, 0, 0, NONE, NONE, NONE, NONE},
    {11110001, F_HEP5, 1, 0, 0, R_(0, -1, -1, 0), R_(0, 0, -1, 1), NONE, NONE},
    {11110010, F_HEP5, 1, 0, 0, R_(0, -1, -1, 0), R_(-1, 0, -1, 1), NONE, NONE},
    {11110011, F_PRISM, 0, 0, 0, NONE, NONE, NONE, NONE},
    {11110100, F_HEP5, 1, 1, 0, R_(0, 0, -1, 0), R_(-1, 0, -1, 1), NONE, NONE},
    {11110110, F_PRISM, 1, 0, 0, NONE, NONE, NONE, NONE},
    {11110111, F_HEP3, 0, 0, 0, R_(0, 0, -1, 0), R_(0, 0, 0, 0), NONE, NONE},
    {11111000, F_HEP5, 1, 1, 0, R_(0, 0, -1, 0), R_(0, 0, -1, 1), NONE, NONE},
    {11111001, F_PRISM, 1, 0, 0, NONE, NONE, NONE, NONE},
    {11111011, F_HEP3, 0, 0, 0, R_(0, 0, -1, 0), R_(-1, 0, 0, 0), NONE, NONE},
    {11111100, F_PRISM, 0, 0, 0, NONE, NONE, NONE, NONE},
    {11111101, F_HEP3, 0, 0, 0, R_(0, -1, -1, 0), R_(-1, 0, 0, 0), NONE, NONE},
    {11111110, F_HEP3, 0, 0, 0, R_(0, -1, -1, 0), R_(0, 0, 0, 0), NONE, NONE},
};
#undef NONE
#undef R_
constexpr int N_RULES = sizeof(c_rules) / sizeof(Rule);

__device__ inline int find_rule(int code) {
  int lo = 0, hi = N_RULES - 1;
  while (lo <= hi) {
    const int mid = (lo + hi) >> 1;
    const int c = c_rules[mid].code;
    if (c == code) return mid;
    if (c < code) lo = mid + 1;
    else hi = mid - 1;
  }
  return -1;
}

// cut volume of a cell of type ty and full volume fullV; a(c, dx, dy, dz) and t(c, ...) read edge and
// face fraction c near it
template <class A, class T>
__device__ inline double vof_of(int ty, double fullV, A a, T t) {
  auto at = [](auto f, Ref r) { return f((int)r.comp, (int)r.dx, (int)r.dy, (int)r.dz); };
  double vol = fullV;
  if (ty == B_Border || ty == T_Border) {
    vol *= t(2, 0, 0, 0);
  } else if (ty == SolidCell) {
    vol = 0.0;
  } else if (ty > 0 && ty != FluidCell) {
    const int k = find_rule(ty);
    if (k >= 0) {
      const Rule r = c_rules[k];
      const double tUp = t(r.axis, 0, 0, 0), tLo = t(r.axis, -(r.axis == 0), -(r.axis == 1), -(r.axis == 2));
      switch (r.fam) {
        case F_TET:
          vol = at(a, r.a) * at(t, r.b) * fullV * ONE_THIRD;
          break;
        case F_HEP3:
          vol = (3.0 - (1.0 - at(a, r.a)) * (1.0 - at(t, r.b))) * fullV * ONE_THIRD;
          break;
        case F_PRISM:
          vol = (tUp + tLo) * fullV * 0.5;
          break;
        case F_HEP5: {
          const double tsel = r.sel ? tUp : tLo;
          double ap = at(a, r.a);
          const double denom = 1.0 - ap;
          double term = 0.0;
          if (denom > EQ_DOUBLE) {
            ap /= denom;
            term = (1.0 - tsel) * (3.0 - 2.0 * at(a, r.b)) * ap * ap * ONE_THIRD;
          }
          vol = (tLo + tUp + term) * fullV * 0.5;
          break;
        }
        case F_HEX5: {
          const double denom = at(a, r.a);
          double term2 = r.sel ? tUp : tLo;
          const double other = r.sel ? tLo : tUp;
          if (denom > EQ_DOUBLE) {
            const double coef = (1.0 - denom) / denom;
            term2 *= (1.0 - (1.0 + 2.0 * at(a, r.b)) * coef * coef * ONE_THIRD);
          }
          vol = (other + term2) * fullV * 0.5;
          break;
        }
        default: {  // F_HEP6
          const double tsel = r.sel ? tUp : tLo;
          const double other = r.sel ? tLo : tUp;
          double term = 0.0;
          double al = at(a, r.a);
          double denom = 1.0 - al;
          if (denom > EQ_DOUBLE) {
            al /= denom;
            term = (3.0 - 2.0 * at(a, r.b)) * al * al;
          }
          al = at(a, r.a2);
          denom = 1.0 - al;
          if (denom > EQ_DOUBLE) {
            al /= denom;
            term += (3.0 - 2.0 * at(a, r.b2)) * al * al;
          }
          vol = (other + tsel + (1.0 - tsel) * term * ONE_THIRD) * fullV * 0.5;
        }
      }
    }
  }
  return vol + PLUS_TINY;
}

struct Fields {
  const double* a[3];
  const double* t[3];
  int N, NM;
};

__global__ void k_vof(const int* __restrict__ type, Fields F, const double* __restrict__ dx,
                      const double* __restrict__ dy, const double* __restrict__ dz, int N, int M, int K,
                      double* __restrict__ vof) {
  const long n = (long)N * M * K;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    int x, y, z;
    decode(i, N, M, &x, &y, &z);
    auto rd = [&](const double* const* f) {
      return [&, f](int c, int ex, int ey, int ez) { return f[c][i + ex + (long)F.N * ey + (long)F.NM * ez]; };
    };
    vof[i] = vof_of(type[i], dx[x] * dy[y] * dz[z], rd(F.a), rd(F.t));
  }
}

// ---- masses and operator coefficients -------------------------------------------------------------
__device__ inline double inv_mass(double v) { return (v < EQ_TINY_DOUBLE) ? 0.0 : (1.0 / v); }

__device__ inline bool no_b(int t) { return t == B_Border || t == BN_Edge || t == BS_Edge || t == BE_Edge || t == BW_Edge || t == BNE_Corner || t == BNW_Corner || t == BSE_Corner || t == BSW_Corner; }
__device__ inline bool no_t(int t) { return t == T_Border || t == TN_Edge || t == TS_Edge || t == TE_Edge || t == TW_Edge || t == TNE_Corner || t == TNW_Corner || t == TSE_Corner || t == TSW_Corner; }
__device__ inline bool no_s(int t) { return t == S_Border || t == TS_Edge || t == BS_Edge || t == SE_Edge || t == SW_Edge || t == TSE_Corner || t == TSW_Corner || t == BSE_Corner || t == BSW_Corner; }
__device__ inline bool no_n(int t) { return t == N_Border || t == TN_Edge || t == BN_Edge || t == NE_Edge || t == NW_Edge || t == TNE_Corner || t == TNW_Corner || t == BNE_Corner || t == BNW_Corner; }
__device__ inline bool no_w(int t) { return t == W_Border || t == TW_Edge || t == BW_Edge || t == NW_Edge || t == SW_Edge || t == TNW_Corner || t == TSW_Corner || t == BNW_Corner || t == BSW_Corner; }
__device__ inline bool no_e(int t) { return t == E_Border || t == TE_Edge || t == BE_Edge || t == NE_Edge || t == SE_Edge || t == TNE_Corner || t == TSE_Corner || t == BNE_Corner || t == BSE_Corner; }

// the fields near cell i of a whole grid
struct GridCell {
  const int* __restrict__ ty;
  const double* __restrict__ th[3];
  const double* __restrict__ vo;
  long i;
  int N;
  long NM;
  __device__ int type() const { return ty[i]; }
  __device__ double theta(int c, int dx, int dy, int dz) const { return th[c][i + dx + (long)N * dy + NM * dz]; }
  __device__ double vof(int dx, int dy, int dz) const { return vo[i + dx + (long)N * dy + NM * dz]; }
};

// Pressure operator row of cell i as 7 coefficients c = [b,s,w,p,e,n,t] (absent = 0): the
// values of LaplaceDiscreteOperator::calcLap (laplace_discrete_operator.h:107-686) with the
// staggered masses M = (V_i + V_nb)/2 inlined, and identity rows at the two pinned cells.  g reads
// the cell's type and the face fractions and volumes near it.
template <class G>
__device__ inline void laplace_row(const G& g, long i, int x, int y, int z, const double* __restrict__ dxs,
                                   const double* __restrict__ dys, const double* __restrict__ dzs, int N, int M, int pin,
                                   double* c) {
  const long NM = (long)N * M;
  const int t = g.type();
  double a_b = 0, a_s = 0, a_w = 0, a_p = 0, a_e = 0, a_n = 0, a_t = 0;
  if (t == SolidCell) {
    a_p = PLUS_TINY;
  } else {
    const double v = g.vof(0, 0, 0);
    const double ddx = dxs[x], ddy = dys[y], ddz = dzs[z];
    const bool hb = !no_b(t), hs = !no_s(t), hw = !no_w(t), he = !no_e(t), hn = !no_n(t), ht = !no_t(t);
    // masses of the six faces (only the present ones are read)
    const double imw = hw ? inv_mass(0.5 * (g.vof(-1, 0, 0) + v)) : 0.0;
    const double ime = he ? inv_mass(0.5 * (v + g.vof(1, 0, 0))) : 0.0;
    const double ims = hs ? inv_mass(0.5 * (g.vof(0, -1, 0) + v)) : 0.0;
    const double imn = hn ? inv_mass(0.5 * (v + g.vof(0, 1, 0))) : 0.0;
    const double imb = hb ? inv_mass(0.5 * (g.vof(0, 0, -1) + v)) : 0.0;
    const double imt = ht ? inv_mass(0.5 * (v + g.vof(0, 0, 1))) : 0.0;
    if (t == FluidCell) {
      const double dyz = ddy * ddz, dxz = ddx * ddz, dxy = ddy * ddx;
      double aux = dyz * dyz;
      a_w = aux * imw;
      a_e = aux * ime;
      aux = dxz * dxz;
      a_s = aux * ims;
      a_n = aux * imn;
      aux = dxy * dxy;
      a_b = aux * imb;
      a_t = aux * imt;
      a_p = -a_b - a_s - a_w - a_e - a_n - a_t;
    } else {
      const double dyz = ddy * ddz, dxz = ddx * ddz, dxy = ddx * ddy;
      double aux;
      if (hw) { aux = g.theta(0, -1, 0, 0) * dyz; a_w = aux * aux * imw; }
      if (he) { aux = g.theta(0, 0, 0, 0) * dyz; a_e = aux * aux * ime; }
      if (hs) { aux = g.theta(1, 0, -1, 0) * dxz; a_s = aux * aux * ims; }
      if (hn) { aux = g.theta(1, 0, 0, 0) * dxz; a_n = aux * aux * imn; }
      if (hb) { aux = g.theta(2, 0, 0, -1) * dxy; a_b = aux * aux * imb; }
      if (ht) { aux = g.theta(2, 0, 0, 0) * dxy; a_t = aux * aux * imt; }
      bool first = true;
      if (hb) { a_p = -a_b; first = false; }
      if (hs) { a_p = first ? -a_s : a_p - a_s; first = false; }
      if (hw) { a_p = first ? -a_w : a_p - a_w; first = false; }
      if (he) { a_p = first ? -a_e : a_p - a_e; first = false; }
      if (hn) { a_p = first ? -a_n : a_p - a_n; first = false; }
      if (ht) { a_p = first ? -a_t : a_p - a_t; first = false; }
    }
    if (pin && (i == NM - 1 || i == N - 1)) {
      a_b = a_s = a_w = a_e = a_n = a_t = 0.0;
      a_p = 1.0;
    }
  }
  c[0] = a_b;
  c[1] = a_s;
  c[2] = a_w;
  c[3] = a_p;
  c[4] = a_e;
  c[5] = a_n;
  c[6] = a_t;
}

__global__ void k_laplace7(const int* __restrict__ type, const double* __restrict__ tx, const double* __restrict__ ty,
                           const double* __restrict__ tz, const double* __restrict__ vof,
                           const double* __restrict__ dxs, const double* __restrict__ dys,
                           const double* __restrict__ dzs, int N, int M, int K, int pin, double* __restrict__ coef) {
  const long n = (long)N * M * K;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    int x, y, z;
    decode(i, N, M, &x, &y, &z);
    double c[7];
    laplace_row(GridCell{type, {tx, ty, tz}, vof, i, N, (long)N * M}, i, x, y, z, dxs, dys, dzs, N, M, pin, c);
    for (int q = 0; q < 7; ++q) coef[q * n + i] = c[q];
  }
}

// ---- momentum (Helmholtz) operators on the staggered meshes --------------------------------------
// Rows of HelmholtzDiscreteOperatorX / Y / Z::calcHelm* (helmholtz_discrete_operator_x.h:98-689 and
// the _y, _z files) for a box without cut cells, in stencil form [b, s, w, p, e, n, t]: viscous
// couplings across the cross faces ((area nu) (sum of the two widths) / (sum of the two distances)),
// nu (area)^2 / V along the component's own axis, no-slip wall terms (bottom and top ones dropped
// for flow tasks), diagonal -(coef M) - sum in each boundary type's own order, and the outflow term
// added to the last cell of every x row of a flow task.  Face and edge fractions are 1 in such a
// box and the reference's products by them are exact, so they are left out.  One thread per
// staggered cell; the type of a staggered cell is the smaller of its two base cells' types
// (ls_stag_uniform_mesh.h:108-130), the mass half the sum of their volumes (:2804-2826).
__device__ inline bool hb_(int t) { return t == B_Border || t == BN_Edge || t == BS_Edge || t == BE_Edge || t == BW_Edge || t == BNE_Corner || t == BNW_Corner || t == BSE_Corner || t == BSW_Corner; }
__device__ inline bool ht_(int t) { return t == T_Border || t == TN_Edge || t == TS_Edge || t == TE_Edge || t == TW_Edge || t == TNE_Corner || t == TNW_Corner || t == TSE_Corner || t == TSW_Corner; }
__device__ inline bool hs_(int t) { return t == S_Border || t == TS_Edge || t == BS_Edge || t == SE_Edge || t == SW_Edge || t == TSE_Corner || t == TSW_Corner || t == BSE_Corner || t == BSW_Corner; }
__device__ inline bool hn_(int t) { return t == N_Border || t == TN_Edge || t == BN_Edge || t == NE_Edge || t == NW_Edge || t == TNE_Corner || t == TNW_Corner || t == BNE_Corner || t == BNW_Corner; }
__device__ inline bool hw_(int t) { return t == W_Border || t == TW_Edge || t == BW_Edge || t == NW_Edge || t == SW_Edge || t == TNW_Corner || t == TSW_Corner || t == BNW_Corner || t == BSW_Corner; }
__device__ inline bool he_(int t) { return t == E_Border || t == TE_Edge || t == BE_Edge || t == NE_Edge || t == SE_Edge || t == TNE_Corner || t == TSE_Corner || t == BNE_Corner || t == BSE_Corner; }

__global__ void k_helmholtz7(const int* __restrict__ type, const double* __restrict__ thx,
                             const double* __restrict__ thy, const double* __restrict__ thz,
                             const double* __restrict__ vof, const double* __restrict__ dxs,
                             const double* __restrict__ dys, const double* __restrict__ dzs, int N, int M, int K,
                             int dir, double nu, double cf, int flow, double* __restrict__ out) {
  const int Nd = N - (dir == 0), Md = M - (dir == 1), Kd = K - (dir == 2);
  const long nd = (long)Nd * Md * Kd, NM = (long)N * M;
  const long step = dir == 0 ? 1 : (dir == 1 ? N : NM);
  for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < nd; q += (long)gridDim.x * blockDim.x) {
    const int i = (int)(q % Nd), j = (int)((q / Nd) % Md), k = (int)(q / ((long)Nd * Md));
    const long c = i + N * (j + (long)M * k);
    const int tc = type[c], td = type[c + step];
    const double th = dir == 0 ? thx[c] : (dir == 1 ? thy[c] : thz[c]);
    const int t = th < EQ_DOUBLE ? SolidCell : (td < tc ? td : tc);
    auto iv = [&](long cc) { return vof[cc] < EQ_TINY_DOUBLE ? 0.0 : 1.0 / vof[cc]; };
    const double dx = dxs[i], dy = dys[j], dz = dzs[k];
    const double mass = 0.5 * (vof[c] + vof[c + step]);
    double rb = 0, rs = 0, rw = 0, re = 0, rn = 0, rt = 0, rp = 0;
    if (t == FluidCell) {
      if (dir == 0) {
        const double dxx = nu * (dxs[i + 1] + dx);
        double aux = dz * dxx;
        rs = aux / (dy + dys[j - 1]);
        rn = aux / (dy + dys[j + 1]);
        aux = dy * dxx;
        rb = aux / (dz + dzs[k - 1]);
        rt = aux / (dz + dzs[k + 1]);
        aux = dy * dz;
        const double d2 = nu * aux * aux;
        re = d2 * iv(c + 1);
        rw = d2 * iv(c);
      } else if (dir == 1) {
        const double dyy = nu * (dys[j + 1] + dy);
        double aux = dz * dyy;
        rw = aux / (dx + dxs[i - 1]);
        re = aux / (dx + dxs[i + 1]);
        aux = dx * dyy;
        rb = aux / (dz + dzs[k - 1]);
        rt = aux / (dz + dzs[k + 1]);
        aux = dx * dz;
        const double d2 = nu * aux * aux;
        rn = d2 * iv(c + N);
        rs = d2 * iv(c);
      } else {
        const double dzz = nu * (dzs[k + 1] + dz);
        double aux = dzz * dy;
        rw = aux / (dx + dxs[i - 1]);
        re = aux / (dx + dxs[i + 1]);
        aux = dx * dzz;
        rs = aux / (dy + dys[j - 1]);
        rn = aux / (dy + dys[j + 1]);
        aux = dx * dy;
        const double d2 = nu * aux * aux;
        rt = d2 * iv(c + NM);
        rb = d2 * iv(c);
      }
      rp = -(cf * mass) - rb - rs - rw - re - rn - rt;
    } else if (t != SolidCell) {
      const bool hb = !hb_(t), ht = !ht_(t), hs = !hs_(t), hn = !hn_(t), hw = !hw_(t);
      const bool zw = hb_(t) || ht_(t), yw = hn_(t) || hs_(t);
      double p = -(cf * mass);
      if (dir == 0) {
        const double dxx = dxs[i + 1], sx = dx + dxx;
        const double az = dz * nu, ay = dy * nu;
        if (hs) rs = az * sx / (dy + dys[j - 1]);
        if (hn) rn = az * sx / (dy + dys[j + 1]);
        if (hb) rb = ay * sx / (dz + dzs[k - 1]);
        if (ht) rt = ay * sx / (dz + dzs[k + 1]);
        const double a2 = dy * dz, d2 = nu * a2 * a2;
        const double ke = d2 * iv(c + 1), kw = hw ? d2 * iv(c) : 0.0;
        re = ke;
        rw = kw;
        double wz = 0.0, wy = 0.0;
        if (t == TN_Edge) {  // the reference's TN edge: (dy dz) / dz in place of dy
          const double q2 = a2 / dz;
          wz = flow ? 0.0 : q2 * nu * sx / dz;
          wy = nu * dz * sx / q2;
        } else {
          if (zw) wz = flow ? 0.0 : dy * nu * sx / dz;
          if (yw) wy = nu * dz * sx / dy;
        }
        if (hb) p -= rb;
        if (hs) p -= rs;
        p -= hw ? (kw + ke) : ke;
        if (hn) p -= rn;
        if (ht) p -= rt;
        if (zw) p -= wz;
        if (yw) p -= wy;
      } else if (dir == 1) {
        const double dyy = dys[j + 1], sy = dy + dyy;
        const double az = dz * nu, ax = dx * nu;
        if (hw) rw = az * sy / (dx + dxs[i - 1]);
        const double ke = az * sy / (dx + dxs[(c + 1) % N]);  // east boundary: the next row's first cell
        re = ke;
        if (hb) rb = ax * sy / (dz + dzs[k - 1]);
        if (ht) rt = ax * sy / (dz + dzs[k + 1]);
        const double a2 = dx * dz, d2 = nu * a2 * a2;
        const double ks = d2 * iv(c), kn = d2 * iv(c + N);
        rs = ks;
        rn = kn;
        double wz = 0.0;
        if (zw) {
          const double dxw = (t == B_Border || t == T_Border) ? dx : a2;  // edges and corners: dx dz
          wz = flow ? 0.0 : dxw * nu * sy / dz;
        }
        const double wy = hn_(t) ? kn : (hs_(t) ? ks : 0.0);
        if (hb) p -= rb;
        if (hn_(t)) {
          if (t == N_Border) {
            p -= rw;
            p -= ks;
          } else {
            p -= ks;
            if (hw) p -= rw;
          }
          p -= ke;
        } else if (hs_(t)) {
          if (hw) p -= rw;
          p -= ke;
          p -= kn;
        } else {
          p -= ks + kn;
          if (hw) p -= rw;
          p -= ke;
        }
        if (ht) p -= rt;
        if (zw) p -= wz;
        if (yw) p -= wy;
      } else {
        const double dzz = dzs[k + 1], sz = dz + dzz;
        const double ay = dy * nu, ax = dx * nu;
        if (hw) rw = ay * sz / (dx + dxs[i - 1]);
        const double ke = ay * sz / (dx + dxs[(c + 1) % N]);
        re = ke;
        if (hs) rs = ax * sz / (dy + dys[j - 1]);
        if (hn) rn = ax * sz / (dy + dys[j + 1]);
        const double wy = yw ? ax * sz / dy : 0.0;
        const double a2 = dx * dy, d2 = nu * a2 * a2;
        const double kb = d2 * iv(c), kt = d2 * iv(c + NM);
        rb = kb;
        rt = kt;
        if (hb_(t)) {
          const double wb = flow ? 0.0 : kb;
          if (hs) p -= rs;
          if (hw) p -= rw;
          p -= ke;
          if (hn) p -= rn;
          p -= kt + wb;
        } else if (ht_(t)) {
          const double wt = flow ? 0.0 : kt;
          p -= kb + wt;
          if (hs) p -= rs;
          if (hw) p -= rw;
          p -= ke;
          if (hn) p -= rn;
        } else if (t == N_Border) {
          p -= rs;
          p -= rw;
          p -= kb + kt;
          p -= ke;
        } else {
          p -= kb + kt;
          if (hs) p -= rs;
          if (hw) p -= rw;
          p -= ke;
          if (hn) p -= rn;
        }
        if (yw) p -= wy;
      }
      rp = p;
    } else {
      rp = PLUS_TINY;
    }
    if (flow && t != SolidCell && i == Nd - 1) {  // outflow term (addPlusOutFlow)
      if (dir == 0)
        rp += nu * dys[j] * dzs[k] / dxs[N - 1];
      else if (dir == 1)
        rp += nu * (dys[j] + dys[j + 1]) * dzs[k] / dxs[N - 1];
      else
        rp += nu * (dzs[k] + dzs[k + 1]) * dys[j] / dxs[N - 1];
    }
    const bool fl = t == FluidCell, so = t == SolidCell;
    out[q] = (fl || (!so && !hb_(t))) ? rb : 0.0;
    out[nd + q] = (fl || (!so && !hs_(t))) ? rs : 0.0;
    out[2 * nd + q] = (fl || (!so && !hw_(t))) ? rw : 0.0;
    out[3 * nd + q] = rp;
    out[4 * nd + q] = (fl || (!so && !he_(t))) ? re : 0.0;
    out[5 * nd + q] = (fl || (!so && !hn_(t))) ? rn : 0.0;
    out[6 * nd + q] = (fl || (!so && !ht_(t))) ? rt : 0.0;
  }
}

int grid_1d(long n) {
  long g = (n + 255) / 256;
  if (g > 16384) g = 16384;
  return (int)(g < 1 ? 1 : g);
}

}  // namespace

int rule_count() { return N_RULES; }

void level_set(const double* cx, const double* cy, const double* cz, int N, int M, int K, Box box, Body body,
               double* phi, hipStream_t s) {
  if (body.kind == BODY_BEZIER6)
    k_level_set_bezier<<<(unsigned)((long)((N + 7) / 8) * ((M + 7) / 8) * ((K + 3) / 4)), 256, 0, s>>>(cx, cy, cz, N, M, K,
                                                                                              box, body, phi);
  else
    k_level_set<<<grid_1d((long)N * M * K), 256, 0, s>>>(cx, cy, cz, N, M, K, box, body, phi);
}

int oscillation_fix(const double* phi0, double* phi, double* tmp, unsigned char* flag, int* changed, int N, int M,
                    int K, Box box, hipStream_t s) {
  const long n = (long)N * M * K;
  k_osc_flags<<<grid_1d(n), 256, 0, s>>>(phi0, N, M, K, box, flag);
  if (hipMemcpyAsync(phi, phi0, n * sizeof(double), hipMemcpyDeviceToDevice, s) != hipSuccess) return -1;
  if (hipMemcpyAsync(tmp, phi0, n * sizeof(double), hipMemcpyDeviceToDevice, s) != hipSuccess) return -1;
  double *cur = phi, *nxt = tmp;
  for (int pass = 1;; ++pass) {
    int h = 0;
    if (hipMemsetAsync(changed, 0, sizeof(int), s) != hipSuccess) return -1;
    k_osc_iter<<<grid_1d(n), 256, 0, s>>>(phi0, flag, cur, nxt, N, M, K, changed);
    if (hipMemcpyAsync(&h, changed, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess) return -1;
    if (hipStreamSynchronize(s) != hipSuccess) return -1;
    double* t = cur;
    cur = nxt;
    nxt = t;
    // an unchanged pass leaves both buffers equal: phi holds the result
    if (!h) return pass;
  }
}

void alpha(const double* phi, int N, int M, int K, Box box, double* ax, double* ay, double* az, hipStream_t s) {
  k_alpha<<<grid_1d((long)N * M * K), 256, 0, s>>>(phi, N, M, K, box, ax, ay, az);
}

void types(const double* phi, int N, int M, int K, Box box, int* type, int* sx, int* sy, int* sz, hipStream_t s) {
  k_types<<<grid_1d((long)N * M * K), 256, 0, s>>>(phi, N, M, K, box, type, sx, sy, sz);
}

void theta(const double* ax, const double* ay, const double* az, const int* sx, const int* sy, const int* sz, int N,
           int M, int K, Box box, double* tx, double* ty, double* tz, hipStream_t s) {
  k_theta<<<grid_1d((long)N * M * K), 256, 0, s>>>(ax, ay, az, sx, sy, sz, N, M, K, box, tx, ty, tz);
}

void vof(const int* type, const double* ax, const double* ay, const double* az, const double* tx, const double* ty,
         const double* tz, const double* dx, const double* dy, const double* dz, int N, int M, int K, double* v,
         hipStream_t s) {
  Fields F;
  F.a[0] = ax;
  F.a[1] = ay;
  F.a[2] = az;
  F.t[0] = tx;
  F.t[1] = ty;
  F.t[2] = tz;
  F.N = N;
  F.NM = N * M;
  k_vof<<<grid_1d((long)N * M * K), 256, 0, s>>>(type, F, dx, dy, dz, N, M, K, v);
}

void helmholtz7(const int* type, const double* tx, const double* ty, const double* tz, const double* v,
                const double* dx, const double* dy, const double* dz, int N, int M, int K, int dir, double nu,
                double coef_time, int flow, double* coef, hipStream_t s) {
  const long nd = (long)(N - (dir == 0)) * (M - (dir == 1)) * (K - (dir == 2));
  k_helmholtz7<<<grid_1d(nd), 256, 0, s>>>(type, tx, ty, tz, v, dx, dy, dz, N, M, K, dir, nu, coef_time, flow, coef);
}

void laplace7(const int* type, const double* tx, const double* ty, const double* tz, const double* v, const double* dx,
              const double* dy, const double* dz, int N, int M, int K, int pin, double* coef, hipStream_t s) {
  k_laplace7<<<grid_1d((long)N * M * K), 256, 0, s>>>(type, tx, ty, tz, v, dx, dy, dz, N, M, K, pin, coef);
}

// ---- pressure right-hand side ------------------------------------------------------------------
// b = Dx u* + Dy v* + Dz w* + flux, b = 0 at the pinned cells: PoissonDiscreteEquation::
// recalcRightMember (poisson_discrete_equation.h:145-159) with the divergence rows of calcDx/Dy/Dz
// (divergence_discrete_operator_{x,y,z}.h) summed in their portrait order, and the static-body
// flux of initFlux / addFluxNSp / addFluxTBp / setBaseFlux (laplace_discrete_operator.h:48-83,
// 744-750) applied in that order.  One thread per cell; no FMA contraction.
namespace {

__device__ inline bool x_east(int t) {
  return t == E_Border || t == NE_Edge || t == SE_Edge || t == TE_Edge || t == BE_Edge || t == TNE_Corner ||
         t == TSE_Corner || t == BNE_Corner || t == BSE_Corner;
}
__device__ inline bool x_west(int t) {
  return t == W_Border || t == NW_Edge || t == SW_Edge || t == TW_Edge || t == BW_Edge || t == TNW_Corner ||
         t == TSW_Corner || t == BNW_Corner || t == BSW_Corner;
}
__device__ inline bool y_north(int t) {
  return t == N_Border || t == NE_Edge || t == NW_Edge || t == TN_Edge || t == BN_Edge || t == TNE_Corner ||
         t == TNW_Corner || t == BNE_Corner || t == BNW_Corner;
}
__device__ inline bool y_south(int t) {
  return t == S_Border || t == SE_Edge || t == SW_Edge || t == TS_Edge || t == BS_Edge || t == TSE_Corner ||
         t == TSW_Corner || t == BSE_Corner || t == BSW_Corner;
}
__device__ inline bool z_bottom(int t) {
  return t == B_Border || t == BN_Edge || t == BS_Edge || t == BE_Edge || t == BW_Edge || t == BNE_Corner ||
         t == BNW_Corner || t == BSE_Corner || t == BSW_Corner;
}
__device__ inline bool z_top(int t) {
  return t == T_Border || t == TN_Edge || t == TS_Edge || t == TE_Edge || t == TW_Edge || t == TNE_Corner ||
         t == TNW_Corner || t == TSE_Corner || t == TSW_Corner;
}

struct RhsIn {
  const double *u, *v, *w, *u_west, *u_out;
  FlowBc bc;
};

template <class G>
__device__ inline double rhs_cell(const G& g, long i, int x, int y, int z, const double* __restrict__ dxa,
                                  const double* __restrict__ dya, const double* __restrict__ dza, int N, int M, int K,
                                  const RhsIn& in) {
  const long NM = (long)N * M;
  const double* __restrict__ u = in.u;
  const double* __restrict__ v = in.v;
  const double* __restrict__ w = in.w;
  const FlowBc& bc = in.bc;
  const int t = g.type();
  const double dx = dxa[x], dy = dya[y], dz = dza[z];
  const long row = y + (long)z * M;
  // flux: initFlux, addFluxNSp, addFluxTBp, setBaseFlux (static body: ibFlux = 0)
  double flux = 0.0;
  if (x == 0) flux = -in.u_west[row] * (dy * dz);
  if (x == N - 1) flux = bc.U_E * (dy * dz);
  if (y == 0) flux -= (dx * dz) * bc.V_S;
  if (y == M - 1) flux += (dx * dz) * bc.V_N;
  if (z == 0) flux -= (dy * dx) * g.theta(2, 0, 0, 0) * bc.W_B;
  if (z == K - 1) flux += (dy * dx) * g.theta(2, 0, 0, 0) * bc.W_T;
  if (in.u_out && x == N - 1) flux = in.u_out[row * (N - 1) + N - 2] * dy * dz;
  // Dx u
  double aux = 0.0;
  {
    const long p = row * (N - 1) + x;
    if (t == SolidCell) aux += 0.0 * u[x == 0 ? p : p - 1];
    else if (x_east(t)) aux += (-g.theta(0, -1, 0, 0) * dy * dz) * u[p - 1];
    else if (x_west(t)) aux += (g.theta(0, 0, 0, 0) * dy * dz) * u[p];
    else {
      const double dyz = dy * dz;
      aux += (-g.theta(0, -1, 0, 0) * dyz) * u[p - 1];
      aux += (g.theta(0, 0, 0, 0) * dyz) * u[p];
    }
  }
  // (aux + flux) + Dy v
  double r = aux + flux;
  {
    const long p = (long)z * N * (M - 1) + (long)y * N + x;
    if (t == SolidCell) r += 0.0 * v[y == 0 ? p : p - N];
    else if (y_north(t)) r += (-g.theta(1, 0, -1, 0) * dx * dz) * v[p - N];
    else if (y_south(t)) r += (g.theta(1, 0, 0, 0) * dx * dz) * v[p];
    else {
      const double dxz = dx * dz;
      r += (-g.theta(1, 0, -1, 0) * dxz) * v[p - N];
      r += (g.theta(1, 0, 0, 0) * dxz) * v[p];
    }
  }
  // + Dz w
  double auxz = 0.0;
  {
    if (t == SolidCell) auxz += 0.0 * w[z == 0 ? i : i - NM];
    else if (z_bottom(t)) auxz += (g.theta(2, 0, 0, 0) * dx * dy) * w[i];
    else if (z_top(t)) auxz += (-g.theta(2, 0, 0, -1) * dx * dy) * w[i - NM];
    else {
      const double dxy = dx * dy;
      auxz += (-g.theta(2, 0, 0, -1) * dxy) * w[i - NM];
      auxz += (g.theta(2, 0, 0, 0) * dxy) * w[i];
    }
  }
  r += auxz;
  if (bc.pin && (i == N - 1 || i == NM - 1)) r = 0.0;
  return r;
}

__global__ void k_pressure_rhs(const int* __restrict__ type, const double* __restrict__ tx,
                               const double* __restrict__ ty, const double* __restrict__ tz,
                               const double* __restrict__ dxa, const double* __restrict__ dya,
                               const double* __restrict__ dza, int N, int M, int K, RhsIn in,
                               double* __restrict__ b) {
  const long n = (long)N * M * K, NM = (long)N * M;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const int z = (int)(i / NM);
    const long r2 = i - (long)z * NM;
    const int y = (int)(r2 / N), x = (int)(r2 - (long)y * N);
    b[i] = rhs_cell(GridCell{type, {tx, ty, tz}, nullptr, i, N, NM}, i, x, y, z, dxa, dya, dza, N, M, K, in);
  }
}

// Velocity correction u = (G dp) inv_M + u* (SetSolutions::correction, set_solutions.h:215-237,
// with GradientDiscreteOperatorX/Y/Z::calc and the staggered types of cvu/cvv/cvw,
// ls_stag_uniform_mesh.h:108-130).  One thread per face of the three staggered grids; the
// inverse staggered mass is 1 / (0.5 (V_a + V_b)), 0 below 1e-12 (inverseVOF).
__device__ inline double inv_mass(double va, double vb) {
  const double m = 0.5 * (va + vb);
  return m < EQ_TINY_DOUBLE ? 0.0 : 1.0 / m;
}

__device__ inline bool staggered_solid(double theta, int a, int b) {
  return theta < EQ_DOUBLE || (b < a ? b : a) == SolidCell;
}

__global__ void k_correct(const int* __restrict__ type, const double* __restrict__ tx, const double* __restrict__ ty,
                          const double* __restrict__ tz, const double* __restrict__ vof,
                          const double* __restrict__ dxa, const double* __restrict__ dya,
                          const double* __restrict__ dza, int N, int M, int K, const double* __restrict__ dp,
                          const double* __restrict__ us, const double* __restrict__ vs, const double* __restrict__ ws,
                          double* __restrict__ u, double* __restrict__ v, double* __restrict__ w) {
  const long nu = (long)(N - 1) * M * K, nv = (long)N * (M - 1) * K, nw = (long)N * M * (K - 1);
  const long NM = (long)N * M;
  for (long q = blockIdx.x * (long)blockDim.x + threadIdx.x; q < nu + nv + nw; q += (long)gridDim.x * blockDim.x) {
    if (q < nu) {  // x faces: index x + (N-1)(y + M z)
      const long f = q, row = f / (N - 1);
      const int x = (int)(f - row * (N - 1)), y = (int)(row % M), z = (int)(row / M);
      const long a = x + (long)N * row, b = a + 1;
      double aux = 0.0;
      if (staggered_solid(tx[a], type[a], type[b])) {
        aux += 0.0 * dp[a];
      } else {
        const double cell = tx[a] * dya[y] * dza[z];
        aux += cell * dp[a];
        aux += -cell * dp[b];
      }
      aux *= inv_mass(vof[a], vof[b]);
      u[f] = aux + us[f];
    } else if (q < nu + nv) {  // y faces: index x + N (y + (M-1) z)
      const long f = q - nu, xy = f % ((long)N * (M - 1));
      const int z = (int)(f / ((long)N * (M - 1))), y = (int)(xy / N), x = (int)(xy - (long)y * N);
      const long a = x + (long)N * y + NM * z, b = a + N;
      double aux = 0.0;
      if (staggered_solid(ty[a], type[a], type[b])) {
        aux += 0.0 * dp[a];
      } else {
        const double cell = ty[a] * dxa[x] * dza[z];
        aux += cell * dp[a];
        aux += -cell * dp[b];
      }
      aux *= inv_mass(vof[a], vof[b]);
      v[f] = aux + vs[f];
    } else {  // z faces: index of the lower cell
      const long a = q - nu - nv, b = a + NM;
      const int z = (int)(a / NM);
      const long r2 = a - (long)z * NM;
      const int y = (int)(r2 / N), x = (int)(r2 - (long)y * N);
      double aux = 0.0;
      if (staggered_solid(tz[a], type[a], type[b])) {
        aux += 0.0 * dp[a];
      } else {
        const double cell = tz[a] * dxa[x] * dya[y];
        aux += cell * dp[a];
        aux += -cell * dp[b];
      }
      aux *= inv_mass(vof[a], vof[b]);
      w[a] = aux + ws[a];
    }
  }
}

}  // namespace

namespace {
__global__ void k_pressure_update(double* __restrict__ p, const double* __restrict__ dp, double coef, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    p[i] = p[i] + dp[i] * coef;
}
}  // namespace

void pressure_update(double* p, const double* dp, double coef, long n, hipStream_t s) {
  k_pressure_update<<<grid_1d(n), 256, 0, s>>>(p, dp, coef, n);
}

void correct(const int* type, const double* tx, const double* ty, const double* tz, const double* vof, const double* dx,
             const double* dy, const double* dz, int N, int M, int K, const double* dp, const double* us,
             const double* vs, const double* ws, double* u, double* v, double* w, hipStream_t s) {
  const long total = (long)(N - 1) * M * K + (long)N * (M - 1) * K + (long)N * M * (K - 1);
  k_correct<<<grid_1d(total), 256, 0, s>>>(type, tx, ty, tz, vof, dx, dy, dz, N, M, K, dp, us, vs, ws, u, v, w);
}

void pressure_rhs(const int* type, const double* tx, const double* ty, const double* tz, const double* dx,
                  const double* dy, const double* dz, int N, int M, int K, const double* u, const double* v,
                  const double* w, const double* u_west, const double* u_out, FlowBc bc, double* b, hipStream_t s) {
  const RhsIn in{u, v, w, u_west, u_out, bc};
  k_pressure_rhs<<<grid_1d((long)N * M * K), 256, 0, s>>>(type, tx, ty, tz, dx, dy, dz, N, M, K, in, b);
}

// ---- objective and shape gradient ---------------------------------------------------------------
// Pressure drag J = sum over cut cells of (theta_x west - theta_x east) dy dz p: the pressure term
// of LoadsCalculator::calc (loads_calculator.h:97-116, n_x dS = (theta^u_{i-1} - theta^u_i) dy dz).
//
// Shape gradient.  With A p = b solved and lambda = A^{-T} dJ/dp, the derivative of J along a
// change of the geometry is that of the Lagrangian F = J(theta, p) + lambda . (b - A p) with p and
// lambda held fixed.  F is a sum over cells of terms that read the level set at the corners of
// the cell and of its six neighbours, after an oscillation fix that reads one node further:
// corner c reaches the cells c + [-2, 3]^3, and dF/dphi_c is the central difference of those cells'
// terms with the corner moved by +h and -h.  Differences are taken per coefficient (c+ - c-)
// before they meet p, so the large cancelling products of A p never enter them.  A Bezier body
// then chains dF/dphi to its control values through the closest point: phi = sgn |X - S(u*, v*)|
// gives dphi/dP_ij = -sgn (X - S)/|X - S| B_i(u*) B_j(v*) (the minimiser's own change does not
// enter at a minimum).
//
// A corner whose level set and whose neighbours' along the axes, before and after the fix, lie on one
// side of the surface by more than the step changes no edge fraction and no sign, so its difference
// is exactly 0: only the corners along the surface are worked on (k_active: their list, in index
// order), one workgroup each (k_corner), which rebuilds the geometry around its corner twice in LDS
// and reads the unmoved geometry outside it.  72 x 64 x 64 cells, 3210 corners: 224 us (two rebuilds
// of the whole grid for each of 216 classes of corners: 59 ms).
//
// A fixed node may have read another fixed node; such chains carry a move beyond its corner's
// reach.  There (more than two passes of the fix) the corners of a class, 6 apart in every
// direction with disjoint reach, move together, and what a chain carries further counts with the
// class's corner that reaches it: the fixed nodes' values under each class's two moves come from a
// table (k_chain_table), and the corners whose cells read a chained node are listed too.
namespace {

__device__ inline bool cut_cell(int t) { return t > 0 && t != FluidCell; }

__global__ void k_drag(const int* __restrict__ type, const double* __restrict__ tx, const double* __restrict__ dys,
                       const double* __restrict__ dzs, int N, int M, int K, Box box, const double* __restrict__ p,
                       double* __restrict__ dJdp, double* __restrict__ partial) {
  __shared__ double lds[256];
  const long n = (long)N * M * K;
  const long per = (n + gridDim.x - 1) / gridDim.x;
  const long lo = per * blockIdx.x, hi = lo + per < n ? lo + per : n;
  double acc = 0.0;
  for (long i = lo + threadIdx.x; i < hi; i += blockDim.x) {
    int x, y, z;
    decode(i, N, M, &x, &y, &z);
    double g = 0.0;
    if (in_box(x, y, box) && cut_cell(type[i])) g = (tx[i - 1] - tx[i]) * dys[y] * dzs[z];
    if (dJdp) dJdp[i] = g;
    acc += g * p[i];
  }
  lds[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) lds[threadIdx.x] += lds[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = lds[0];
}

template <class G>
__device__ inline double drag_cell(const G& g, int x, int y, int z, const double* dys, const double* dzs, const Box& box,
                                   double p) {
  if (!in_box(x, y, box) || !cut_cell(g.type())) return 0.0;
  return (g.theta(0, -1, 0, 0) - g.theta(0, 0, 0, 0)) * dys[y] * dzs[z] * p;
}

// Corners 6 apart in every direction move together: their classes (x mod 6, y mod 6, z mod 6).
constexpr int SG_SPACING = 6, SG_CLASSES = SG_SPACING * SG_SPACING * SG_SPACING;

__device__ inline int corner_class(int x, int y, int z) {
  return x % SG_SPACING + SG_SPACING * (y % SG_SPACING) + SG_SPACING * SG_SPACING * (z % SG_SPACING);
}

// (F_i(+) - F_i(-)) / 2h of cell i from its fields in the two moved geometries
struct LagrArgs {
  const double *dxs, *dys, *dzs, *p, *lam;
  int N, M, K, pin, objective, has_rhs;
  Box box;
  RhsIn rin;
  double inv2h;
};
template <class G>
__device__ inline double lagr_diff(const G& gp, const G& gm, long i, int x, int y, int z, const LagrArgs& a) {
  const int N = a.N, M = a.M, K = a.K;
  const long NM = (long)N * M;
  const double* __restrict__ p = a.p;
  double dJ = 0.0;
  if (a.objective == OBJ_DRAG_X && in_box(x, y, a.box)) {
    if (cut_cell(gp.type()) && cut_cell(gm.type())) {
      const double dw = gp.theta(0, -1, 0, 0) - gm.theta(0, -1, 0, 0);
      const double de = gp.theta(0, 0, 0, 0) - gm.theta(0, 0, 0, 0);
      dJ = (dw - de) * a.dys[y] * a.dzs[z] * p[i];
    } else {
      dJ = drag_cell(gp, x, y, z, a.dys, a.dzs, a.box, p[i]) - drag_cell(gm, x, y, z, a.dys, a.dzs, a.box, p[i]);
    }
  }
  double ca[7], cb[7];
  laplace_row(gp, i, x, y, z, a.dxs, a.dys, a.dzs, N, M, a.pin, ca);
  laplace_row(gm, i, x, y, z, a.dxs, a.dys, a.dzs, N, M, a.pin, cb);
  const long nb[7] = {i - NM, i - N, i - 1, i, i + 1, i + N, i + NM};
  const bool has[7] = {z > 0, y > 0, x > 0, true, x < N - 1, y < M - 1, z < K - 1};
  double dAp = 0.0;
  for (int q = 0; q < 7; ++q)
    if (has[q]) dAp += (ca[q] - cb[q]) * p[nb[q]];
  double db = 0.0;
  if (a.has_rhs)
    db = rhs_cell(gp, i, x, y, z, a.dxs, a.dys, a.dzs, N, M, K, a.rin) -
         rhs_cell(gm, i, x, y, z, a.dxs, a.dys, a.dzs, N, M, K, a.rin);
  return (dJ + a.lam[i] * (db - dAp)) * a.inv2h;
}

// whether moving corner i by h can change the geometry: its level set and its neighbours', before
// (raw) and after (phi) the oscillation fix, do not all lie on one side by more than the step
__device__ inline bool corner_active(const double* __restrict__ raw, const double* __restrict__ phi, long i, int N, int M,
                                     int K, const Box& box, double h) {
  int x, y, z;
  decode(i, N, M, &x, &y, &z);
  if (!in_box(x, y, box)) return false;
  const long NM = (long)N * M;
  const double t = 2.0 * (EQ_DOUBLE + h);
  const bool inside = raw[i] > 0.0;
  auto apart = [&](bool there, long j) {
    const long k = there ? j : i;
    const double r = raw[k], f = phi[k];
    return inside ? !(r > t && f > t) : !(r < -t && f < -t);
  };
  return apart(true, i) || apart(x - 1 >= box.hs, i - 1) || apart(x + 1 < box.hf, i + 1) ||
         apart(y - 1 >= box.vs, i - N) || apart(y + 1 < box.vf, i + N) || apart(z > 0, i - NM) ||
         apart(z + 1 < K, i + NM);
}

// Bits of a node's mark: a corner whose cells read a chained node; a node that the oscillation fix can
// change in some moved geometry.
constexpr unsigned char MARK_CORNER = 1, MARK_FIXABLE = 2;

// A node of the box and its neighbours along the axes, for what the fix can do to it once one of them has
// moved by h.  It changes the node in a direction only if it is above the threshold between two nodes
// below 0: the upper one unfixed (between), the lower one by itself (alone) or because the fix brought it
// there.  The first such direction decides (check_osc): one that is so by itself whatever moves
// (decided) leaves nothing for the directions after it to read.  NaN compares false: never fixed.
struct FixNode {
  double r, lo[3], up[3], h;
  __device__ FixNode(const double* __restrict__ raw, long i, int z, int N, long NM, int K, double h_) : h(h_) {
    const bool mid = z > 0 && z < K - 1;
    r = raw[i];
    lo[0] = raw[i - 1];
    up[0] = raw[i + 1];
    lo[1] = raw[i - N];
    up[1] = raw[i + N];
    const double b = raw[mid ? i - NM : i], t = raw[mid ? i + NM : i];
    lo[2] = mid ? b : 1.0;
    up[2] = mid ? t : 1.0 + h;  // never between
  }
  __device__ bool between(int d) const { return r + h > EQ_DOUBLE && up[d] - h < 0; }
  __device__ bool any() const { return between(0) || between(1) || between(2); }
  __device__ bool alone() const {
    return (between(0) && lo[0] - h < 0) || (between(1) && lo[1] - h < 0) || (between(2) && lo[2] - h < 0);
  }
  __device__ bool decided(int d) const { return r - h > EQ_DOUBLE && lo[d] + h < 0 && up[d] + h < 0; }
};
// Fixable nodes' marks by one pass: from the level set (cur null: the nodes fixable by themselves and those
// that read one), or those of a pass before and those that read one of them.  seen: bit 0 there is a
// node that reads one (the fix chains in some moved geometry), bit 1 it was not marked yet.
__device__ inline bool fixable_pass(const double* __restrict__ raw, long i, int N, int M, int K, const Box& box, double h,
                                    const unsigned char* __restrict__ cur, int* seen) {
  if (!(raw[i] + h > EQ_DOUBLE)) return false;  // as between: most nodes
  int x, y, z;
  decode(i, N, M, &x, &y, &z);
  if (!in_box(x, y, box)) return false;
  const long NM = (long)N * M;
  const FixNode f(raw, i, z, N, NM, K, h);
  if (!f.any()) return false;
  const bool was = cur ? cur[i] != 0 : f.alone();
  auto reads = [&](int d) {  // the lower neighbour's mark
    if (!f.between(d)) return false;
    const long j = i - (d == 0 ? 1 : (d == 1 ? N : NM));
    if (cur) return cur[j] != 0;
    return in_box(x - (d == 0), y - (d == 1), box) && FixNode(raw, j, z - (d == 2), N, NM, K, h).alone();
  };
  const bool rd = reads(0) || (!f.decided(0) && (reads(1) || (!f.decided(1) && reads(2))));
  *seen |= (rd ? 1 : 0) | (rd && !was ? 2 : 0);
  return was || rd;
}

// Lists of nodes in index order.  AC_LOOK: the active corners, with a first pass over the fixable nodes;
// AC_FIXABLE: the fixable nodes after another pass (cur null: the first); AC_CORNERS: the active
// corners and those marked in `cur`.  Blocks of AC_NODES consecutive nodes count theirs (list null) and say
// what the pass saw, one workgroup turns the counts into offsets, the total and what all saw
// (k_active_scan), and the blocks write (ranks within a block by ballots; AC_FIXABLE: those marked in `cur`).
constexpr int AC_NODES = 1024;
__global__ void __launch_bounds__(256) k_active(const double* __restrict__ raw, const double* __restrict__ phi,
                                                const unsigned char* __restrict__ cur, unsigned char* __restrict__ nxt,
                                                int mode, int N, int M, int K, Box box, double h,
                                                int* __restrict__ count, int* __restrict__ list) {
  __shared__ int waves[4];
  const long n = (long)N * M * K;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int at = list ? count[blockIdx.x] : 0, seen = 0;
  for (int q = 0; q < AC_NODES / 256; ++q) {
    const long i = (long)blockIdx.x * AC_NODES + q * 256 + threadIdx.x;
    bool on = false;
    if (i < n) {
      bool fixable = false;
      if (mode != AC_CORNERS) {
        if (list) {
          fixable = mode == AC_FIXABLE && cur[i] != 0;
        } else {
          fixable = fixable_pass(raw, i, N, M, K, box, h, mode == AC_LOOK ? nullptr : cur, &seen);
          nxt[i] = fixable ? MARK_FIXABLE : 0;
        }
      }
      on = mode == AC_FIXABLE ? fixable
                              : (mode == AC_CORNERS && cur[i] & MARK_CORNER) || corner_active(raw, phi, i, N, M, K, box, h);
    }
    const unsigned long long m = __ballot(on);
    if (lane == 0) waves[wave] = __popcll(m);
    __syncthreads();
    int before = 0, all = 0;
    for (int w = 0; w < 4; ++w) {
      before += w < wave ? waves[w] : 0;
      all += waves[w];
    }
    if (list && on) list[at + before + __popcll(m & ((1ull << lane) - 1))] = (int)i;
    at += all;
    __syncthreads();
  }
  if (list) return;
  const int any = __syncthreads_or(seen & 1), fresh = __syncthreads_or(seen & 2);
  if (threadIdx.x == 0) {
    count[blockIdx.x] = at;
    count[gridDim.x + 2 + blockIdx.x] = (any ? 1 : 0) | (fresh ? 2 : 0);
  }
}

// count: nb counts (then offsets), total, what all blocks saw, nb blocks' own
__global__ void __launch_bounds__(1024) k_active_scan(int* __restrict__ count, int nb) {
  __shared__ int sum[1024];
  const int per = (nb + 1023) / 1024, lo = threadIdx.x * per, hi = lo + per < nb ? lo + per : nb;
  int mine = 0, seen = 0;
  for (int b = lo; b < hi; ++b) {
    mine += count[b];
    seen |= count[nb + 2 + b];
  }
  const int any = __syncthreads_or(seen & 1), fresh = __syncthreads_or(seen & 2);
  sum[threadIdx.x] = mine;
  __syncthreads();
  for (int st = 1; st < 1024; st <<= 1) {
    const int v = (int)threadIdx.x >= st ? sum[threadIdx.x - st] : 0;
    __syncthreads();
    sum[threadIdx.x] += v;
    __syncthreads();
  }
  int at = sum[threadIdx.x] - mine;
  for (int b = lo; b < hi; ++b) {
    const int c = count[b];
    count[b] = at;
    at += c;
  }
  if (threadIdx.x == 1023) {
    count[nb] = sum[1023];
    count[nb + 1] = (any ? 1 : 0) | (fresh ? 2 : 0);
  }
}

// Index of node j in the sorted list of fixable nodes.
__device__ inline int find_node(const int* __restrict__ list, int count, int j) {
  int lo = 0, hi = count - 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (list[mid] < j)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// The level set with the corners of a class moved by +h (move 0) or -h (move 1), before the fix and,
// from the values `val` of the fixable nodes, after it.
struct MovedLevelSet {
  const double* __restrict__ raw0;
  const unsigned char* __restrict__ mark;
  const int* __restrict__ list;  // fixable nodes
  const double* val;
  int count, cls, move, N, M;
  double h;
  Box box;
  __device__ double raw(long j) const {
    int x, y, z;
    decode(j, N, M, &x, &y, &z);
    const double v = raw0[j];
    const bool on = in_box(x, y, box) && corner_class(x, y, z) == cls;
    return on ? (move == 0 ? v + h : v - h) : v;
  }
  __device__ double fixed(long j) const {
    return mark[j] & MARK_FIXABLE ? val[find_node(list, count, (int)j)] : raw(j);
  }
};

// table[(cls * 2 + move) * count + l] = level set of fixable node l after the fix with the corners of class cls
// moved: one workgroup per class and move repeats k_osc_iter's pass over the list until nothing
// changes (a node depends on lower ones only, so that is the ordered sweep's result whatever the
// order of the updates within a pass)
__global__ void __launch_bounds__(256) k_chain_table(const double* __restrict__ raw0, const double* __restrict__ phi0,
                                                     const unsigned char* __restrict__ mark,
                                                     const int* __restrict__ list, int count, int N, int M, int K,
                                                     Box box, double h, double* table) {
  const long NM = (long)N * M;
  volatile double* val = table + (long)blockIdx.x * count;
  const MovedLevelSet f{raw0, mark, list, table + (long)blockIdx.x * count, count, (int)blockIdx.x / 2,
                        (int)blockIdx.x % 2, N, M, h, box};
  for (int l = threadIdx.x; l < count; l += blockDim.x) val[l] = phi0[list[l]];
  for (;;) {
    __threadfence_block();
    __syncthreads();
    bool changed = false;
    for (int l = threadIdx.x; l < count; l += blockDim.x) {
      const long j = list[l];
      const int z = (int)(j / NM);
      auto lower = [&](long k) {
        return mark[k] & MARK_FIXABLE ? (double)val[find_node(list, count, (int)k)] : f.raw(k);
      };
      double v = f.raw(j);
      check_osc(v, lower(j - 1), f.raw(j + 1));
      check_osc(v, lower(j - N), f.raw(j + N));
      if (z > 0 && z < K - 1) check_osc(v, lower(j - NM), f.raw(j + NM));
      if (v != val[l]) {
        val[l] = v;
        changed = true;
      }
    }
    if (!__syncthreads_or(changed)) break;
  }
}

// mark the corners whose cells read a fixable node next to a lower one: its cells' rows reach the corners
// within 4 of it (every writer of a byte adds the same bit to the same marks)
__global__ void __launch_bounds__(256) k_chain_mark(const int* __restrict__ list, int N, int M, int K, Box box,
                                                    unsigned char* mark) {
  const long NM = (long)N * M, j = list[blockIdx.x];
  int x, y, z;
  decode(j, N, M, &x, &y, &z);
  auto fixable = [&](long k) { return (mark[k] & MARK_FIXABLE) != 0; };
  if (!fixable(j - 1) && !fixable(j - N) && !(z > 0 && fixable(j - NM))) return;
  for (int q = threadIdx.x; q < 729; q += blockDim.x) {
    const int cx = x + q % 9 - 4, cy = y + q / 9 % 9 - 4, cz = z + q / 81 - 4;
    if (cx >= 0 && cx < N && cy >= 0 && cy < M && cz >= 0 && cz < K && in_box(cx, cy, box)) {
      unsigned char* m = mark + cx + (long)N * cy + NM * cz;
      *m = (*m & MARK_FIXABLE) | MARK_CORNER;
    }
  }
}

// One moved geometry around a corner: cells c + [LO, LO + PA - 1]^3.
template <int PA>
struct Patch {
  static constexpr int CELLS = PA * PA * PA;
  double phi[CELLS], a[3][CELLS], t[3][CELLS], vof[CELLS];
  int type[CELLS];
};
// the fields near a cell at (lx, ly, lz) of the patch, grid index i: the patch's inside it, the
// unmoved geometry's outside
template <int PA>
struct PatchCell {
  const Patch<PA>* s;
  const GeoBase& g;
  int lx, ly, lz;
  long i;
  int N;
  long NM;
  __device__ double get(const double* in, const double* __restrict__ out, int dx, int dy, int dz) const {
    const int a = lx + dx, b = ly + dy, c = lz + dz;
    const bool local = (unsigned)a < PA && (unsigned)b < PA && (unsigned)c < PA;
    return local ? in[a + PA * (b + PA * c)] : out[i + dx + (long)N * dy + NM * dz];
  }
  __device__ double phi(int dx, int dy, int dz) const { return get(s->phi, g.phi, dx, dy, dz); }
  __device__ double alpha(int c, int dx, int dy, int dz) const { return get(s->a[c], g.a[c], dx, dy, dz); }
  __device__ double theta(int c, int dx, int dy, int dz) const { return get(s->t[c], g.t[c], dx, dy, dz); }
  __device__ double vof(int dx, int dy, int dz) const { return get(s->vof, g.vof, dx, dy, dz); }
  __device__ int type() const {
    const bool local = (unsigned)lx < PA && (unsigned)ly < PA && (unsigned)lz < PA;
    return local ? s->type[lx + PA * (ly + PA * lz)] : g.type[i];
  }
};

// out[c] = dF/dphi_c of the listed corners, a workgroup at a time.  Every stage is the whole grid's
// (alpha_of, type_of, theta_of, vof_of, laplace_row, rhs_cell), one thread per cell of the patch and
// both moves in turn; the terms of the 216 reached cells are added in index order.  Bound by the
// latency of its dozen stages.  Without chains the corner's move changes nodes and cells c + [-1, 4]^3 at
// most and the fix is repeated in LDS (31 KB: four workgroups share a CU); CHAIN: every cell and edge
// that the rows of the reach read, c + [-4, 4]^3, with the fixable nodes' values from the table.
template <bool CHAIN>
__global__ void __launch_bounds__(CHAIN ? 768 : 256) k_corner(GeoBase g, const int* __restrict__ list, int n_active,
                                                              LagrArgs la, double h,
                                                              const unsigned char* __restrict__ mark,
                                                              const int* __restrict__ fixable, int n_fixable,
                                                              const double* __restrict__ table,
                                                              double* __restrict__ out) {
  constexpr int PA = CHAIN ? 9 : 6, LO = CHAIN ? -4 : -1, CELLS = PA * PA * PA, RA = 6, REACH = RA * RA * RA;
  __shared__ Patch<PA> S[2];
  __shared__ double dF[REACH];
  const int N = la.N, M = la.M, K = la.K;
  const Box& box = la.box;
  const double *__restrict__ dxs = la.dxs, *__restrict__ dys = la.dys, *__restrict__ dzs = la.dzs;
  const long NM = (long)N * M;
  const int tid = threadIdx.x;
  const int lx = tid % PA, ly = tid / PA % PA, lz = tid / (PA * PA);
  for (int w = blockIdx.x; w < n_active; w += gridDim.x) {
    const long c = list[w];
    int cx, cy, cz;
    decode(c, N, M, &cx, &cy, &cz);
    const int x = cx + LO + lx, y = cy + LO + ly, z = cz + LO + lz;
    const long i = x + (long)N * y + NM * z;
    const bool own = tid < CELLS && x >= 0 && x < N && y >= 0 && y < M && z >= 0 && z < K;
    if constexpr (!CHAIN) {
      auto raw = [&](int m, long j) {  // the moved level set before the oscillation fix
        const double v = g.raw[j];
        return j == c ? (m == 0 ? v + h : v - h) : v;
      };
      // oscillation fix (k_osc_flags, k_osc_iter): nodes below the patch hold their unmoved final values
      bool flag[2] = {false, false};
      if (own)
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const double f = raw(m, i);
          S[m].phi[tid] = f;
          if (in_box(x, y, box) && f > EQ_DOUBLE)
            flag[m] = raw(m, i + 1) < 0 || raw(m, i + N) < 0 || (z > 0 && z < K - 1 && raw(m, i + NM) < 0);
        }
      for (;;) {
        __syncthreads();
        double nxt[2];
        bool changed = false;
#pragma unroll
        for (int m = 0; m < 2; ++m)
          if (flag[m]) {
            const PatchCell<PA> q{&S[m], g, lx, ly, lz, i, N, NM};
            double f = raw(m, i);
            check_osc(f, q.phi(-1, 0, 0), raw(m, i + 1));
            check_osc(f, q.phi(0, -1, 0), raw(m, i + N));
            if (z > 0 && z < K - 1) check_osc(f, q.phi(0, 0, -1), raw(m, i + NM));
            changed = changed || f != S[m].phi[tid];
            nxt[m] = f;
          }
        if (!__syncthreads_or(changed)) break;
#pragma unroll
        for (int m = 0; m < 2; ++m)
          if (flag[m]) S[m].phi[tid] = nxt[m];
      }
    }
    int side[2][3];
    if (own)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const PatchCell<PA> q{&S[m], g, lx, ly, lz, i, N, NM};
        const int cls = corner_class(cx, cy, cz);
        const MovedLevelSet f{g.raw, mark, fixable, table + (long)(cls * 2 + m) * n_fixable, n_fixable, cls, m, N, M, h,
                              box};
        auto phi = [&](int dx, int dy, int dz) {
          if constexpr (CHAIN)
            return f.fixed(i + dx + (long)N * dy + NM * dz);
          else
            return q.phi(dx, dy, dz);
        };
        double a[3];
        alpha_of(phi, x, y, z, K, box, a);
        for (int k = 0; k < 3; ++k) S[m].a[k][tid] = a[k];
        S[m].type[tid] = type_of(phi, x, y, z, N, M, K, box, side[m]);
      }
    __syncthreads();
    // (CHAIN: what the patch's first layer of faces and volumes lacks below it, no row of the reach reads)
    if (own)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const PatchCell<PA> q{&S[m], g, lx, ly, lz, i, N, NM};
        double t[3];
        theta_of([&](int k, int dx, int dy, int dz) { return q.alpha(k, dx, dy, dz); }, side[m], x, y, z, K, box, t);
        for (int k = 0; k < 3; ++k) S[m].t[k][tid] = t[k];
      }
    __syncthreads();
    if (own)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const PatchCell<PA> q{&S[m], g, lx, ly, lz, i, N, NM};
        S[m].vof[tid] = vof_of(
            S[m].type[tid], dxs[x] * dys[y] * dzs[z],
            [&](int k, int dx, int dy, int dz) { return q.alpha(k, dx, dy, dz); },
            [&](int k, int dx, int dy, int dz) { return q.theta(k, dx, dy, dz); });
      }
    __syncthreads();
    // the reached cells c + [-2, 3]^3
    if (tid < REACH) {
      const int ex = tid % RA - 2, ey = tid / RA % RA - 2, ez = tid / (RA * RA) - 2;
      const int rx = cx + ex, ry = cy + ey, rz = cz + ez;
      double v = 0.0;
      if (rx >= 0 && rx < N && ry >= 0 && ry < M && rz >= 0 && rz < K) {
        const long r = rx + (long)N * ry + NM * rz;
        const PatchCell<PA> gp{&S[0], g, ex - LO, ey - LO, ez - LO, r, N, NM};
        const PatchCell<PA> gm{&S[1], g, ex - LO, ey - LO, ez - LO, r, N, NM};
        v = lagr_diff(gp, gm, r, rx, ry, rz, la);
      }
      dF[tid] = v;
    }
    __syncthreads();
    if (tid == 0) {
      double acc = 0.0;
#pragma unroll 8
      for (int q = 0; q < REACH; ++q) acc += dF[q];
      out[c] = acc;
    }
    __syncthreads();
  }
}

// per listed corner with g != 0: winning patch, its parameters and w = g dphi/dS (3 values)
__global__ void __launch_bounds__(64) k_bz_hits(const double* __restrict__ g, const int* __restrict__ list, int count,
                          const double* __restrict__ cx, const double* __restrict__ cy, const double* __restrict__ cz,
                          int N, int M, Body body, int* __restrict__ hf, double* __restrict__ huv,
                          double* __restrict__ hw) {
  __shared__ BzBody B;
  bz_load(body.ctrl, B);
  const int l = blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= count) return;
  const long i = list[l];
  int x, y, z;
  decode(i, N, M, &x, &y, &z);
  int f = -1;
  if (g[i] != 0.0) {
    BzHit hit;
    bezier_closest(B, body.c, body.a, cx[x], cy[y], cz[z], hit);
    if (hit.dist > 0.0) {
      f = hit.f;
      huv[2 * l] = hit.u;
      huv[2 * l + 1] = hit.v;
      for (int c = 0; c < 3; ++c) hw[3 * l + c] = g[i] * (-hit.sgn * hit.r[c] / hit.dist);
    }
  }
  hf[l] = f;
}

// one workgroup per control point (f, i, j): out[(f*16 + i*4 + j)*3 + c] = sum over the listed corners
__global__ void k_bz_reduce(const int* __restrict__ hf, const double* __restrict__ huv, const double* __restrict__ hw,
                            int count, double* __restrict__ out) {
  __shared__ double lds[3][256];
  const int cp = blockIdx.x, f = cp / 16, bi = (cp / 4) % 4, bj = cp % 4;
  double acc[3] = {0.0, 0.0, 0.0};
  for (int k = threadIdx.x; k < count; k += blockDim.x) {
    if (hf[k] != f) continue;
    double bu[4], dbu[4], ddbu[4], bv[4], dbv[4], ddbv[4];
    bz_basis(huv[2 * k], bu, dbu, ddbu);
    bz_basis(huv[2 * k + 1], bv, dbv, ddbv);
    const double wgt = bu[bi] * bv[bj];
    for (int c = 0; c < 3; ++c) acc[c] += wgt * hw[3 * k + c];
  }
  for (int c = 0; c < 3; ++c) lds[c][threadIdx.x] = acc[c];
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s)
      for (int c = 0; c < 3; ++c) lds[c][threadIdx.x] += lds[c][threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x < 3) out[cp * 3 + threadIdx.x] = lds[threadIdx.x][0];
}

}  // namespace

constexpr int DRAG_BLOCKS = 256;

// ---- allocation-free drag -------------------------------------------------------------------
// The partial sums of the drag reduction (one per workgroup of the fixed DRAG_BLOCKS-workgroup
// launch, for any grid size) in a device array of the library instead of caller- or
// library-allocated memory: 2 KiB per GPU, held until the process ends.  Each GPU has its own
// copy at its own address; host code uses the address hipGetSymbolAddress returns on that
// device (kept per device below), never the array's name.  Every call on one GPU shares it.
constexpr int DRAG_SCRATCH = 256;
static_assert(DRAG_BLOCKS <= DRAG_SCRATCH, "drag partials exceed the scratch array");
static __device__ __align__(256) double scratch[DRAG_SCRATCH];

namespace {
constexpr int MAX_DEVICES = 64;
double* scratch_dev[MAX_DEVICES] = {};
std::mutex scratch_mu;

// J = sum of the partials in block order, the order of the host sum in drag() (bit-identical)
__global__ void k_drag_sum(const double* __restrict__ partial, double* __restrict__ J) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    double acc = 0.0;
    for (int b = 0; b < DRAG_BLOCKS; ++b) acc += partial[b];
    J[0] = acc;
  }
}
}  // namespace

int drag_scratch(double** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return -1;
  std::lock_guard<std::mutex> lk(scratch_mu);
  if (!scratch_dev[dev]) {
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return -2;
    scratch_dev[dev] = (double*)ptr;
  }
  *out = scratch_dev[dev];
  return 0;
}

void drag_noalloc(const int* type, const double* tx, const double* dy, const double* dz, int N, int M, int K, Box box,
                  const double* p, double* dJdp, double* partial, double* J, hipStream_t s) {
  k_drag<<<DRAG_BLOCKS, 256, 0, s>>>(type, tx, dy, dz, N, M, K, box, p, dJdp, partial);
  k_drag_sum<<<1, 64, 0, s>>>(partial, J);
}

double drag(const int* type, const double* tx, const double* dy, const double* dz, int N, int M, int K, Box box,
            const double* p, double* dJdp, double* partial, hipStream_t s) {
  k_drag<<<DRAG_BLOCKS, 256, 0, s>>>(type, tx, dy, dz, N, M, K, box, p, dJdp, partial);
  double h[DRAG_BLOCKS];
  if (hipMemcpyAsync(h, partial, sizeof(h), hipMemcpyDeviceToHost, s) != hipSuccess) return NAN;
  if (hipStreamSynchronize(s) != hipSuccess) return NAN;
  double J = 0.0;
  for (int b = 0; b < DRAG_BLOCKS; ++b) J += h[b];
  return J;
}

int active_blocks(long n) { return (int)((n + AC_NODES - 1) / AC_NODES); }

void count_nodes(const double* phi_raw, const double* phi, const unsigned char* cur, unsigned char* nxt, int mode, int N,
                 int M, int K, Box box, double h, int* count, hipStream_t s) {
  const int nb = active_blocks((long)N * M * K);
  k_active<<<nb, 256, 0, s>>>(phi_raw, phi, cur, nxt, mode, N, M, K, box, h, count, nullptr);
  k_active_scan<<<1, 1024, 0, s>>>(count, nb);
}

void list_nodes(const double* phi_raw, const double* phi, const unsigned char* cur, int mode, int N, int M, int K, Box box,
                double h, int* count, int* list, hipStream_t s) {
  const int nb = active_blocks((long)N * M * K);
  k_active<<<nb, 256, 0, s>>>(phi_raw, phi, cur, nullptr, mode, N, M, K, box, h, count, list);
}

void chain_tables(const double* phi_raw, const double* phi, const int* fixable, int n_fixable, int N, int M, int K,
                  Box box, double h, double* table, unsigned char* mark, hipStream_t s) {
  if (n_fixable < 1) return;
  k_chain_mark<<<n_fixable, 256, 0, s>>>(fixable, N, M, K, box, mark);
  k_chain_table<<<2 * SG_CLASSES, 256, 0, s>>>(phi_raw, phi, mark, fixable, n_fixable, N, M, K, box, h, table);
}

static LagrArgs lagr_args(const double* dx, const double* dy, const double* dz, int N, int M, int K, Box box, int pin,
                          const double* p, const double* lam, int objective, const RhsArgs* rhs, double h) {
  RhsIn in{nullptr, nullptr, nullptr, nullptr, nullptr, FlowBc{0, 0, 0, 0, 0, 0}};
  if (rhs) in = RhsIn{rhs->u, rhs->v, rhs->w, rhs->u_west, rhs->u_out, rhs->bc};
  return LagrArgs{dx, dy, dz, p, lam, N, M, K, pin, objective, rhs ? 1 : 0, box, in, 0.5 / h};
}

void corner_gradient(const GeoBase& g, const int* list, int count, const unsigned char* mark, const int* fixable,
                     int n_fixable, const double* table, const double* dx, const double* dy, const double* dz, int N,
                     int M, int K, Box box, int pin, const double* p, const double* lam, int objective,
                     const RhsArgs* rhs, double h, double* out, hipStream_t s) {
  if (count < 1) return;
  const LagrArgs la = lagr_args(dx, dy, dz, N, M, K, box, pin, p, lam, objective, rhs, h);
  const int blocks = count < 4096 ? count : 4096;
  if (table)
    k_corner<true><<<blocks, 768, 0, s>>>(g, list, count, la, h, mark, fixable, n_fixable, table, out);
  else
    k_corner<false><<<blocks, 256, 0, s>>>(g, list, count, la, h, nullptr, nullptr, 0, nullptr, out);
}

void bezier_chain(const double* g, const int* list, int count, const double* cx, const double* cy, const double* cz,
                  int N, int M, Body body, int* hf, double* huv, double* hw, double* out, hipStream_t s) {
  if (count > 0) k_bz_hits<<<(count + 63) / 64, 64, 0, s>>>(g, list, count, cx, cy, cz, N, M, body, hf, huv, hw);
  k_bz_reduce<<<96, 256, 0, s>>>(hf, huv, hw, count, out);
}

}  // namespace geo
}  // namespace lsx

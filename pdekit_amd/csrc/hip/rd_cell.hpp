// Fused residual-distribution cell kernel for gfx950.
//
// One thread owns one element and performs, in registers, the work of
//   gather (GeometryCache / SolutionCache push_back_to_buffer,
//           src/interpolation/GeometryCache.hpp:329-400, SolutionCache.hpp:361-388)
//   geometry metric (GeometryMetric.hpp:366-425, 3D 487-560)
//   P+1 flux metric (FluxSpaceMetric.hpp:562-743)
//   element scheme  (PGLDA.hpp:109-311, PGN.hpp:96-290, PGB.hpp:314-498,
//                    PSI limiter LFResidualLimiter.hpp:84-110, and the PSI /
//                    LDA blend by PGB's cell theta, PGB.hpp:437-477)
//   scatter res[v] += Phi_v, lambda[v] += |T| max lambda
//           (PGRDMExplicitCellWorker.hpp:546-567)
// The division by the dual volume is done once per node in the nodal pass.
//
// Algebraic forms used on the device (same mathematics as the reference):
//   * flux divergence at q: sum_f sum_xi dVf[xi][q][f] G_xi(f) with the
//     contravariant flux G_xi(f) = sum_d Jinv[d][xi] F_d(f) (affine cells);
//   * N dissipation  sum_{m!=n} K+_n S^-1 K+_m (U_n - U_m) = K+_n (U_n - S^-1 sum_m K+_m U_m),
//     S = sum_m K+_m, so one extra solve replaces the O(nd^2) pair loop;
//   * S^-1 is never formed: S x = r and S y = sum K+_m U_m are solved in the
//     entropy and acoustic parts of K+ (EulerSum: one reciprocal and a
//     Cholesky-like factor, no pivoting);
//   * the element Jacobians keep the full matrices and eliminate with partial
//     pivoting by predicated row swaps (solve_pp).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <type_traits>

#include "rd_physics.hpp"

namespace pdrd {

struct CellArgs
{
  const double *__restrict__ tab;      // packed FE tables of the block
  const uint32_t *__restrict__ gconn;  // [NG][ne] (structure of arrays)
  const uint32_t *__restrict__ sconn;  // [ND][ne]
  const double *__restrict__ coords;   // [nv][D]
  const double *__restrict__ u;        // [N][M]
  double *__restrict__ acc_res;        // [N][M]
  double *__restrict__ acc_ws;         // [N]
  int *__restrict__ status;
  uint32_t first;  // first element of the launch (block order)
  uint32_t count;  // elements in the launch
  uint32_t ne;     // elements in the block (SoA stride)
  int atomic;      // 1: FP64 atomics, 0: plain read-modify-write (one colour)
  PhysParams pp;
  const double *__restrict__ nodal;  // [N] blending coefficient (B) or artificial viscosity (LDA), or null
  // when non-zero, vertex ids >= nv_check or node ids >= nn_check are not
  // followed: the cell is skipped and bit 2 of *status is set (connectivity
  // the host has not validated)
  uint32_t nv_check, nn_check;
};

template <int D, int NG, int ND, int NF, int NQ>
struct TabOffsets
{
  static constexpr int qp = 0;
  static constexpr int w = qp + NQ * D;
  static constexpr int Vg = w + NQ;
  static constexpr int dVg = Vg + NQ * NG;
  static constexpr int V = dVg + D * NQ * NG;
  static constexpr int dV = V + NQ * ND;
  static constexpr int Vf = dV + D * NQ * ND;
  static constexpr int dVf = Vf + NQ * NF;
  static constexpr int Vgf = dVf + D * NQ * NF;
  static constexpr int Vsf = Vgf + NF * NG;
  static constexpr int sol_nodes = Vsf + NF * ND;
  static constexpr int flux_nodes = sol_nodes + ND * D;
  static constexpr int size = flux_nodes + NF * D;
  // Device-only copies appended by the host, laid out so that the values one
  // iteration of a rolled loop needs are contiguous (one scalar load each):
  static constexpr int dVfT = size;                  // [NF][D][NQ]
  static constexpr int dVT = dVfT + NF * D * NQ;     // [NQ][D][ND]
  static constexpr int dVgT = dVT + NQ * D * ND;     // [NQ][D][NG]
  static constexpr int dev_size = dVgT + NQ * D * NG;
};

// Workgroups are dealt round-robin to the 8 XCDs; give each XCD one
// contiguous range of workgroups so neighbouring cells (which share nodes)
// meet in the same L2.
__device__ __forceinline__ uint32_t xcd_block_index(uint32_t bid, uint32_t nb)
{
  const uint32_t x = bid & 7u, k = bid >> 3, q8 = nb >> 3, r8 = nb & 7u;
  return x * q8 + (x < r8 ? x : r8) + k;
}

__device__ __forceinline__ uint32_t xcd_block_index() { return xcd_block_index(blockIdx.x, gridDim.x); }

// Barrier of a workgroup that exchanges data through LDS only: waits for the
// wave's LDS operations, not for its global loads in flight (as __syncthreads
// does), so that data loaded ahead may cross it.
__device__ __forceinline__ void lds_barrier()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int D>
__device__ __forceinline__ double det_inv(const double J[D][D], double Ji[D][D])
{
  if constexpr (D == 2) {
    const double det = J[0][0] * J[1][1] - J[0][1] * J[1][0];
    const double id = recip(det);
    Ji[0][0] = id * J[1][1];
    Ji[1][1] = id * J[0][0];
    Ji[0][1] = -id * J[0][1];
    Ji[1][0] = -id * J[1][0];
    return det;
  } else {
    const double c00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
    const double c01 = J[1][2] * J[2][0] - J[1][0] * J[2][2];
    const double c02 = J[1][0] * J[2][1] - J[1][1] * J[2][0];
    const double det = J[0][0] * c00 + J[0][1] * c01 + J[0][2] * c02;
    const double id = recip(det);
    Ji[0][0] = c00 * id;
    Ji[1][0] = c01 * id;
    Ji[2][0] = c02 * id;
    Ji[0][1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) * id;
    Ji[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * id;
    Ji[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * id;
    Ji[0][2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) * id;
    Ji[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * id;
    Ji[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * id;
    return det;
  }
}

// Solve A X = B (M x M, R right-hand sides) in place; partial pivoting by
// predicated swaps so that every index stays a compile-time constant.
template <int M, int R>
__device__ __forceinline__ void solve_pp(double A[M][M], double B[M][R])
{
  double ipv[M];
#pragma unroll
  for (int c = 0; c < M; ++c) {
#pragma unroll
    for (int r = c + 1; r < M; ++r) {
      const bool sw = fabs(A[r][c]) > fabs(A[c][c]);
#pragma unroll
      for (int j = c; j < M; ++j) {
        const double t = A[c][j];
        A[c][j] = sw ? A[r][j] : t;
        A[r][j] = sw ? t : A[r][j];
      }
#pragma unroll
      for (int j = 0; j < R; ++j) {
        const double t = B[c][j];
        B[c][j] = sw ? B[r][j] : t;
        B[r][j] = sw ? t : B[r][j];
      }
    }
    const double ip = recip(A[c][c]);
    ipv[c] = ip;
#pragma unroll
    for (int r = c + 1; r < M; ++r) {
      const double f = A[r][c] * ip;
#pragma unroll
      for (int j = c + 1; j < M; ++j) A[r][j] -= f * A[c][j];
#pragma unroll
      for (int j = 0; j < R; ++j) B[r][j] -= f * B[c][j];
    }
  }
#pragma unroll
  for (int c = M - 1; c >= 0; --c) {
    const double ip = ipv[c];
#pragma unroll
    for (int j = 0; j < R; ++j) {
      double s = B[c][j];
#pragma unroll
      for (int k = c + 1; k < M; ++k) s -= A[c][k] * B[k][j];
      B[c][j] = s * ip;
    }
  }
}

// Nodal states as the quadrature loop reads them: from the thread's
// registers, or from the patch's LDS copy (which frees the registers of the
// state after the flux-node loop).
template <int ND, int M>
struct URegs
{
  const double (&U)[ND][M];
  __device__ __forceinline__ double operator()(int n, int k) const { return U[n][k]; }
};

template <int ND, int M>
struct ULds
{
  const double *ul;   // [local node][M]
  const int (&row)[ND];  // local node of each cell node
  __device__ __forceinline__ double operator()(int n, int k) const { return ul[row[n] * M + k]; }
};

// A nodal scalar input of the cell (external blending coefficient of the B
// scheme, artificial viscosity of the LDA scheme): none, from the patch's
// LDS rows, or from global memory by node id.
struct NodalNone
{
  __device__ __forceinline__ double operator()(int) const { return 0.0; }
};

// The nodal source field of the reaction residuals (PREC 3) from the
// patch's LDS rows: source(n, k) of the cell's node n.
template <int ND, int M>
struct SourceLds
{
  const double *s;       // [local node][M]
  const int (&row)[ND];  // local node of each cell node
  __device__ __forceinline__ double operator()(int n, int k) const { return s[row[n] * M + k]; }
};

// PREC 5 (the B scheme with a source field and an external blending
// coefficient): source(n, k) as SourceLds, theta(n) from a second LDS column.
template <int ND, int M>
struct SourceThetaLds
{
  const double *s;       // [local node][M]
  const double *th;      // [local node]
  const int (&row)[ND];
  __device__ __forceinline__ double operator()(int n, int k) const { return s[row[n] * M + k]; }
  __device__ __forceinline__ double operator()(int n) const { return th[row[n]]; }
};

template <int ND>
struct NodalLds
{
  const double *v;       // [local node]
  const int (&row)[ND];
  __device__ __forceinline__ double operator()(int n) const { return v[row[n]]; }
};

template <int ND>
struct NodalGlobal
{
  const double *__restrict__ v;  // [N]
  const uint32_t (&nid)[ND];
  __device__ __forceinline__ double operator()(int n) const { return v[nid[n]]; }
};

// K+ of the Euler cells in the variables that block-diagonalise it. At a point
// with velocity V, total enthalpy H and sound speed a, a vector x has the parts
//   p = (gm1 / a) (|V|^2/2 x_0 - V . x_m + x_E),  Q = x_m - V x_0,  s = x_0 - p / a,
//   x = s (1, V, |V|^2/2) + (p / a) (1, V, H) + (0, Q, V . Q),
// and the upwind matrix of a node with unit gradient n acts on them as
//   s -> l0 s,  p -> l0 p + al,  Q -> l0 Q + be n,
//   al = hs p + hd (n . Q),  be = hs (n . Q) + hd p,
// l0, lp, lm the positive parts of |g| (V.n), |g| (V.n + a), |g| (V.n - a),
// hs = (lp + lm) / 2 - l0, hd = (lp - lm) / 2; in conservative variables
//   K+_n x = l0 x + (al / a) (1, V, H) + be (0, n, V . n).
// So S = sum_n K+_n is sum l0 on s and, on (p, Q), the symmetric positive
// definite (D + 1) x (D + 1) matrix
//   [ sum l0 + sum hs, w^T; w, sum l0 I + T ],  w = sum hd n, T = sum hs n n^T,
// whose solve needs no pivoting: one reciprocal and a Cholesky-like
// elimination of 3 (2D) or 4 (3D) unknowns instead of the elimination with row
// swaps of a 4 x 4 or 5 x 5 matrix, whose selects alone were a hundred (2D) to
// 240 (3D) instructions of a quadrature point. These cells are bound by FP64
// issue and latency, so a sweep follows the count: 786 432 P2 / Q2 cells (LDA)
// 368 -> 301 us, 5.3 M P1 tetrahedra (PSI / LDA blend) 1.86 -> 1.44 ms, 0.66 M
// P2 tetrahedra (LDA) 605 -> 516 us, with 40 to 150 registers less.
template <int D>
struct EulerNodeK
{
  double l0, hs, hd, un, nh[D], emax;
};

// The geometric part of a node's K+ parameters: nh = g / |g| and |g| for the
// physical gradient g of the node's basis function; normk: |g|, or 0 where
// |g| is negligible (and nh = 0 then).
template <int D>
struct EulerNodeG
{
  double nh[D], norm, normk;
};

// Jq: the inverse Jacobian at the point, dvk: the reference gradients of the
// ND basis functions there ([D][ND]).
template <int D, int ND>
__device__ __forceinline__ EulerNodeG<D> euler_node_g(const double (&Jq)[D][D], const double *dvk, int n)
{
  EulerNodeG<D> ge;
  double g[D];
#pragma unroll
  for (int x = 0; x < D; ++x) {
    double t = 0.0;
#pragma unroll
    for (int xi = 0; xi < D; ++xi) t += Jq[x][xi] * dvk[xi * ND + n];
    g[x] = t;
  }
  double nn = 0.0;
#pragma unroll
  for (int x = 0; x < D; ++x) nn += g[x] * g[x];
  double norm, inorm;
  sqrt_rsqrt(nn, norm, inorm);
  norm = (nn > 0.0) ? norm : 0.0;  // sqrt_rsqrt(0) is NaN
  const bool tiny = (D == 2) ? (norm < 1.e-9) : (norm == 0.0);
  inorm = tiny ? 0.0 : inorm;
#pragma unroll
  for (int x = 0; x < D; ++x) ge.nh[x] = g[x] * inorm;
  ge.norm = norm;
  ge.normk = (D == 2) ? (tiny ? 0.0 : norm) : norm;
  return ge;
}

// The K+ parameters from the geometric part and the point's velocity V and
// sound speed a; un = V . nh, emax the largest |eigenvalue| |g| (un, un +- a).
template <int D>
__device__ __forceinline__ EulerNodeK<D> euler_node_k(const EulerNodeG<D> &ge, const double (&V)[D], double a)
{
  EulerNodeK<D> k;
  double un = 0.0;
#pragma unroll
  for (int x = 0; x < D; ++x) {
    k.nh[x] = ge.nh[x];
    un += V[x] * ge.nh[x];
  }
  k.un = un;
  const double e0 = ge.norm * un, c = ge.normk * a;
  k.emax = fabs(e0) + ((D == 2) ? ge.norm * a : c);
  k.l0 = fmax(0.0, e0);
  const double lp = fmax(0.0, e0 + c), lm = fmax(0.0, e0 - c);
  k.hs = 0.5 * (lp + lm) - k.l0;
  k.hd = 0.5 * (lp - lm);
  return k;
}

template <int D, int ND>
__device__ __forceinline__ EulerNodeK<D> euler_node_k(const double (&Jq)[D][D], const double *dvk, int n,
                                                      const double (&V)[D], double a)
{
  return euler_node_k<D>(euler_node_g<D, ND>(Jq, dvk, n), V, a);
}

// A point's quantities in those variables (hv = |V|^2 / 2, ga = gm1 / a).
template <int D>
struct EulerPoint
{
  double V[D], H, a, ia, hv, ga;
  __device__ __forceinline__ double p_of(const double (&x)[D + 2]) const
  {
    double t = x[D + 1] + hv * x[0];
#pragma unroll
    for (int d = 0; d < D; ++d) t -= V[d] * x[1 + d];
    return ga * t;
  }
  // K+ of a node from (p, n . Q) of a vector: al / a and be
  __device__ __forceinline__ void acoustic(const EulerNodeK<D> &k, double p, double t, double &al, double &be) const
  {
    al = (k.hs * p + k.hd * t) * ia;
    be = k.hs * t + k.hd * p;
  }
  // out += l0 x + al (1, V, H) + be (0, n, V . n)
  __device__ __forceinline__ void add(const EulerNodeK<D> &k, const double (&x)[D + 2], double al, double be,
                                      double (&out)[D + 2]) const
  {
    out[0] += k.l0 * x[0] + al;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      double t = out[1 + d] + k.l0 * x[1 + d];
      t += al * V[d];
      out[1 + d] = t + be * k.nh[d];
    }
    double t = out[D + 1] + k.l0 * x[D + 1];
    t += al * H;
    out[D + 1] = t + be * k.un;
  }
  // out += K+ x with (p, Q) of x at hand, or from x itself
  __device__ __forceinline__ void apply(const EulerNodeK<D> &k, const double (&x)[D + 2], double p,
                                        const double (&Q)[D], double (&out)[D + 2]) const
  {
    double t = 0.0, al, be;
#pragma unroll
    for (int d = 0; d < D; ++d) t += k.nh[d] * Q[d];
    acoustic(k, p, t, al, be);
    add(k, x, al, be, out);
  }
  __device__ __forceinline__ void apply(const EulerNodeK<D> &k, const double (&x)[D + 2], double (&out)[D + 2]) const
  {
    double t = -k.un * x[0], al, be;
#pragma unroll
    for (int d = 0; d < D; ++d) t += k.nh[d] * x[1 + d];
    acoustic(k, p_of(x), t, al, be);
    add(k, x, al, be, out);
  }
};

// S = sum_n K+_n: the sums over the nodes, then the factors of its solve.
template <int D>
struct EulerSum
{
  double l0, hs, w[D], T[D][D];
  double il0, ip[D + 1], L[D + 1][D + 1];
  __device__ __forceinline__ void clear()
  {
    l0 = hs = 0.0;
#pragma unroll
    for (int x = 0; x < D; ++x) {
      w[x] = 0.0;
#pragma unroll
      for (int y = x; y < D; ++y) T[x][y] = 0.0;
    }
  }
  __device__ __forceinline__ void add(const EulerNodeK<D> &k)
  {
    l0 += k.l0;
    hs += k.hs;
#pragma unroll
    for (int x = 0; x < D; ++x) {
      w[x] += k.hd * k.nh[x];
      const double t = k.hs * k.nh[x];
#pragma unroll
      for (int y = x; y < D; ++y) T[x][y] += t * k.nh[y];
    }
  }
  // L D L^T of the (p, Q) block
  __device__ __forceinline__ void factor()
  {
    constexpr int K = D + 1;
    double A[K][K];
    A[0][0] = l0 + hs;
#pragma unroll
    for (int x = 0; x < D; ++x) {
      A[0][1 + x] = w[x];
#pragma unroll
      for (int y = x; y < D; ++y) A[1 + x][1 + y] = T[x][y] + ((x == y) ? l0 : 0.0);
    }
    il0 = recip(l0);
#pragma unroll
    for (int c = 0; c < K; ++c) {
      ip[c] = recip(A[c][c]);
#pragma unroll
      for (int r = c + 1; r < K; ++r) {
        const double f = A[c][r] * ip[c];
        L[r][c] = f;
#pragma unroll
        for (int j = r; j < K; ++j) A[r][j] -= f * A[c][j];
      }
    }
  }
  // x = S^-1 b in conservative variables, with its (p, Q)
  __device__ __forceinline__ void solve(const EulerPoint<D> &pt, const double (&b)[D + 2], double (&x)[D + 2],
                                        double &p, double (&Q)[D]) const
  {
    constexpr int K = D + 1;
    double y[K];
    y[0] = pt.p_of(b);
    const double s = (b[0] - y[0] * pt.ia) * il0;
#pragma unroll
    for (int d = 0; d < D; ++d) y[1 + d] = b[1 + d] - pt.V[d] * b[0];
#pragma unroll
    for (int r = 1; r < K; ++r)
#pragma unroll
      for (int c = 0; c < r; ++c) y[r] -= L[r][c] * y[c];
#pragma unroll
    for (int r = K - 1; r >= 0; --r) {
      double t = y[r] * ip[r];
#pragma unroll
      for (int c = r + 1; c < K; ++c) t -= L[c][r] * y[c];
      y[r] = t;
    }
    p = y[0];
    const double pa = p * pt.ia;
    x[0] = s + pa;
    double e = s * pt.hv + pa * pt.H;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      Q[d] = y[1 + d];
      x[1 + d] = pt.V[d] * x[0] + Q[d];
      e += pt.V[d] * Q[d];
    }
    x[D + 1] = e;
  }
};

template <int D>
__device__ __forceinline__ EulerPoint<D> euler_point(const EulerState<double, D> &st, double gm1)
{
  EulerPoint<D> pt;
#pragma unroll
  for (int d = 0; d < D; ++d) pt.V[d] = st.V[d];
  pt.H = st.H;
  pt.a = st.a;
  pt.ia = st.inv_a;
  pt.hv = 0.5 * st.v2;
  pt.ga = gm1 * st.inv_a;
  return pt;
}

// sum_n K+_n U_n over the nodes of a point, gathered in parts: sum l0 U, sum
// al / a, sum be n and sum be (V . n).
template <int D>
struct EulerKU
{
  double lu[D + 2], al, be[D], bu;
  __device__ __forceinline__ void clear()
  {
#pragma unroll
    for (int k = 0; k < D + 2; ++k) lu[k] = 0.0;
    al = bu = 0.0;
#pragma unroll
    for (int d = 0; d < D; ++d) be[d] = 0.0;
  }
  __device__ __forceinline__ void add(const EulerPoint<D> &pt, const EulerNodeK<D> &k, const double (&x)[D + 2])
  {
    double t = -k.un * x[0];
#pragma unroll
    for (int d = 0; d < D; ++d) t += k.nh[d] * x[1 + d];
    const double p = pt.p_of(x);
    al += k.hs * p + k.hd * t;
    const double b = k.hs * t + k.hd * p;
#pragma unroll
    for (int d = 0; d < D; ++d) be[d] += b * k.nh[d];
    bu += b * k.un;
#pragma unroll
    for (int c = 0; c < D + 2; ++c) lu[c] += k.l0 * x[c];
  }
  __device__ __forceinline__ void total(const EulerPoint<D> &pt, double (&out)[D + 2]) const
  {
    const double ai = al * pt.ia;
    out[0] = lu[0] + ai;
#pragma unroll
    for (int d = 0; d < D; ++d) out[1 + d] = lu[1 + d] + ai * pt.V[d] + be[d];
    out[D + 1] = lu[D + 1] + ai * pt.H + bu;
  }
};

// Waves per SIMD the register allocation of a patch kernel must leave room
// for: 5 for the scalar affine P1 / P2 cells (at most 96 VGPRs, measured
// faster than 4 waves); 2 for the Euler cells of up to 4 nodes, which need at
// most 256 registers but for the tetrahedra's blends (28 bytes of scratch per
// lane): 1.57 M P1 tetrahedra per sweep at 1 and 2 waves: N 289 -> 223 us, PSI
// / LDA blend 412 -> 336 us, 233 us since the last node's residual comes from
// the cell's (the second wave covers the first's waits, a third of its life);
// 2 for the schemes with one residual sum per node (LDA, N, PSI)
// on P2 triangles and for the LDA of P2 tetrahedra with the 4-point rule, which
// need 256 registers or a few more, their pair sums in phases (PatchWork) so
// that 8 waves fit the LDS too: 131 072 P2 triangles LDA 42.0 -> 33.9 us, N 45.5
// -> 38.6 us, 0.20 M P2 tetrahedra LDA 146 -> 125 us a sweep. The others keep
// the compiler's choice, 1 wave: at 2 the B scheme of P2 triangles takes 220
// bytes of scratch (54 -> 60 us), Q2 quadrilaterals 312 (65 536 cells LDA 44 ->
// 55 us), the P2 tetrahedra's N 172 (137 -> 151 us). Forms with inputs that take
// some scratch at these waves are still faster there: the P2 tetrahedra's LDA with
// an artificial viscosity, 184 bytes at 2 waves, 144 us against 161 at 1 wave and no
// scratch (196 608 cells), 79 against 88 us (82 944). The linear sweeps (PREC 4,
// J delta per cell) are bound by the Jacobians' bandwidth and keep 4 waves (2
// for blocks of more than 24 unknowns).
template <int M, int ND, int NQ, bool AFFINE, int SC, int PREC>
struct PatchMinWaves
{
  static constexpr bool one_sum = SC == SC_LDA || SC == SC_N || SC == SC_PSI;
  static constexpr bool two_p2 =
      AFFINE && ((M == 4 && ND == 6 && one_sum) || (M == 5 && ND == 10 && NQ == 4 && SC == SC_LDA));
  static constexpr int value = (PREC == 4)                        ? (ND * M <= 24 ? 4 : 2)
                               : (M == 1 && ND <= 6 && AFFINE)    ? 5
                               : (M > 1 && (ND <= 4 || two_p2)) ? 2
                                                                  : 1;
};

// Doubles of LDS that carry a cell's flux divergence from the flux nodes to the
// quadrature points (none where the scheme's own parameters give it).
template <int D, int ND, int NQ, bool AFFINE, int PH>
struct CellColumn
{
  static constexpr bool linear_flux = ScalarFlux<PH, AFFINE ? D + 1 : (1 << D), ND>::exact;
  static constexpr int value = linear_flux ? 0 : NQ * PhysTraits<PH>::M;
};

// Use of a patch workgroup's LDS work region, in doubles per cell. `column`:
// what the cell computation keeps in its own column, the flux divergence at
// the quadrature points or, with `two` passes over them (the dissipative
// schemes of the 3D P2 cells, see cell_residual), also the `rhs` solutions of
// every point. Afterwards the region carries the (cell, node) pair sums, `comps`
// of the M + 1 components at a time: all of them at once, or as many as the
// column holds where the region would otherwise grow for the pairs and the LDS,
// not the registers, would then limit the waves: the kernels of 2 waves on more
// than 4 nodes, and the two-pass ones (0.20 M P2 tetrahedra N 143 -> 137 us). On
// the others the phases' barriers cost more than they give (P2 triangles at 1
// wave 42 -> 46 us, Q2 44 -> 48 us).
template <int D, int ND, int NQ, bool AFFINE, int PH, int SC, int PREC>
struct PatchWork
{
  static constexpr int M = PhysTraits<PH>::M;
  static constexpr int rhs = (SC == SC_B || SC == SC_BPSI) ? 2 : 1;
  static constexpr bool two =
      D == 3 && SC != SC_LDA && AFFINE && M == D + 2 && PREC != 4 && NQ * (1 + rhs) * M <= ND * (M + 1);
  static constexpr int column = (PREC == 4) ? 0 : (two ? NQ * (1 + rhs) * M : CellColumn<D, ND, NQ, AFFINE, PH>::value);
  static constexpr bool phased = M > 1 && PREC != 4 && ND > 4 && ND * (M + 1) > column &&
                                 (two || PatchMinWaves<M, ND, NQ, AFFINE, SC, PREC>::value == 2);
  static constexpr int comps = phased ? (column >= ND ? column / ND : 1) : M + 1;
  static constexpr int per_cell =
      column > comps * ND ? (column > M + 1 ? column : M + 1) : (comps * ND > M + 1 ? comps * ND : M + 1);
};

// Residuals phi[ND][M] and wave speed of one element from its vertex
// coordinates X and nodal state U. lds_div: this thread's slice of CellColumn
// doubles of LDS (stride `stride` between entries) that carries the flux
// divergence from the flux-node loop to the quadrature loop.
//
// PREC 0: everything in FP64. PREC 2: FP64 with the
// nodal input `nodal` -- for the B scheme the external blending coefficient
// (set_blending_coeff, PGB.hpp:141-148, 467-477), for the LDA scheme the
// artificial viscosity of the shock-capturing term (PGLDA.hpp:245-256).
// PREC 3: FP64 with a nodal source field (`nodal` gives source(n, k)): the
// reaction residuals compute_adv_reaction_residuals, whose residual at a
// quadrature point is div F - s_q, s_q = V . source (PGLDA.hpp:553-741,
// PGN.hpp:470-660, PGB.hpp:825-1050).
// DLDS: the caller's LDS column at lds_div extends past the NQ M divergence
// slices to ND (M + 1) entries (the patch kernel's work region). The
// dissipative schemes of the 3D P2 cells then run the quadrature in two
// passes that carry the per-point results in that column (see TWO below).
template <int D, int NG, int ND, int NF, int NQ, bool AFFINE, int PH, int SC, int PREC, bool DLDS = false, class UA,
          class NA = NodalNone>
__device__ __forceinline__ void cell_residual(const double *__restrict__ tab, const double (&X)[NG][D],
                                              const double (&U)[ND][PhysTraits<PH>::M], const UA &Uq,
                                              const PhysParams &pp, double (&phi)[ND][PhysTraits<PH>::M],
                                              double &wave, bool &bad, double *lds_div, int stride,
                                              const NA &nodal = NA{})
{
  constexpr int M = PhysTraits<PH>::M;
  static_assert(PhysTraits<PH>::DIM == D, "physics / element dimension mismatch");
  using O = TabOffsets<D, NG, ND, NF, NQ>;
  // ---- geometry ----------------------------------------------------------
  constexpr int NJ = AFFINE ? 1 : NQ;
  double Jinv[NJ][D][D];
  double detJ[NJ];
#pragma unroll
  for (int q = 0; q < NJ; ++q) {
    double J[D][D];
#pragma unroll
    for (int xi = 0; xi < D; ++xi)
#pragma unroll
      for (int x = 0; x < D; ++x) {
        double s = 0.0;
#pragma unroll
        for (int g = 0; g < NG; ++g) s += tab[O::dVgT + (q * D + xi) * NG + g] * X[g][x];
        J[xi][x] = s;
      }
    detJ[q] = det_inv<D>(J, Jinv[q]);
  }

  // ---- P+1 flux element: divergence of the interpolated flux at q ---------
  // Scalar fluxes that the P+1 element interpolates exactly need none: linear
  // advection (a u and, rotating, a(x) u with a linear and divergence-free are
  // of order P + 1) and the Burgers flux (u^2 / 2, u) of first-order elements;
  // div F at q is then a . grad u = sum_n k_n U_n, from the upwind parameters
  // that the scheme forms anyway. The loop below would take two thirds of a P3
  // cell's instructions (101 250 cells N 26.3 -> 20.9 us a sweep without it).
  constexpr bool LINF = CellColumn<D, ND, NQ, AFFINE, PH>::linear_flux;
  if constexpr (!LINF) {
  double divr[NQ][M];
  // P1 simplices of the Euler equations: their P2 flux element has the
  // vertices and the edge midpoints as nodes, so with b_i the gradients of the
  // vertex functions l_i,
  //   div F = sum_i l_i E_i,  E_i = 4 (F_i . b_i + sum_{j != i} F_ij . b_j) - sum_k F_k . b_k;
  // the state at a vertex is the vertex's, at a midpoint half the sum of two,
  // and F(x / 2) = F(x) / 2. 10 (3D) or 6 (2D) point fluxes are contracted
  // with 16 (9) vectors and D + 1 vectors E_i interpolated, where the general
  // form below takes the fluxes of every node to every quadrature point: 470
  // instead of 1 700 instructions of a P1 tetrahedron's 5 500 (PSI / LDA
  // blend, 5.3 M cells: with the cap of PatchMinWaves 1.44 -> 1.15 ms).
  constexpr bool P1S = (M > 1) && AFFINE && (ND == D + 1);
  if constexpr (P1S) {
    double b[ND][D], A[ND][M], C[M];
#pragma unroll
    for (int n = 0; n < ND; ++n) {
#pragma unroll
      for (int x = 0; x < D; ++x) {
        double t = 0.0;
#pragma unroll
        for (int xi = 0; xi < D; ++xi) t += Jinv[0][x][xi] * tab[O::dVT + xi * ND + n];
        b[n][x] = t;
      }
    }
#pragma unroll
    for (int k = 0; k < M; ++k) C[k] = 0.0;
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      const EulerState<double, D> st = euler_state<double, D>(U[i], double(pp.p0));
      bad = bad || st.bad;
      double c[M];
#pragma unroll
      for (int k = 0; k < M; ++k) c[k] = 0.0;
      euler_flux_add<D>(U[i], st, b[i], c);
#pragma unroll
      for (int k = 0; k < M; ++k) {
        C[k] += c[k];
        A[i][k] = 2.0 * c[k];
      }
    }
#pragma unroll
    for (int i = 0; i < ND; ++i)
#pragma unroll
      for (int j = i + 1; j < ND; ++j) {
        double s[M];
#pragma unroll
        for (int k = 0; k < M; ++k) s[k] = U[i][k] + U[j][k];
        const EulerState<double, D> st = euler_state<double, D>(s, double(pp.p0));
        bad = bad || st.bad;
        euler_flux_add<D>(s, st, b[j], A[i]);
        euler_flux_add<D>(s, st, b[i], A[j]);
      }
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int k = 0; k < M; ++k) {
        double t = 0.0;
#pragma unroll
        for (int n = 0; n < ND; ++n) t += tab[O::V + q * ND + n] * A[n][k];
        divr[q][k] = 2.0 * t - C[k];
      }
  } else {
  // The flux-node loop stays rolled: each trip reads one row of Vsf and one
  // [D][NQ] slab of dVf with scalar loads, so the table never has to be held
  // in (and spilled from) scalar registers as a whole.
#pragma unroll
  for (int q = 0; q < NQ; ++q)
#pragma unroll
    for (int k = 0; k < M; ++k) divr[q][k] = 0.0;
  // two trips at a time for the Euler cells of more than 4 nodes: their table
  // loads wait once per two trips (the scalar registers do not hold both
  // trips' rows at once otherwise; measured 5 % off that loop on P2 triangles)
#pragma unroll((M > 1 && ND > 4) ? 2 : 1)
  for (int f = 0; f < NF; ++f) {
    const double *vs = tab + O::Vsf + f * ND;
    const double *dvf = tab + O::dVfT + f * D * NQ;
    double s[M];
#pragma unroll
    for (int k = 0; k < M; ++k) {
      double t = 0.0;
#pragma unroll
      for (int n = 0; n < ND; ++n) t += vs[n] * U[n][k];
      s[k] = t;
    }
    double F[D][M];
    double G[AFFINE ? D : 1][M];
    if constexpr (M > 1 && AFFINE) {
      // the contravariant fluxes straight from the state
      const EulerState<double, D> st = euler_state<double, D>(s, double(pp.p0));
      bad = bad || st.bad;
#pragma unroll
      for (int xi = 0; xi < D; ++xi) {
        double b[D];
#pragma unroll
        for (int d = 0; d < D; ++d) b[d] = Jinv[0][d][xi];
#pragma unroll
        for (int k = 0; k < M; ++k) G[xi][k] = 0.0;
        euler_flux_add<D>(s, st, b, G[xi]);
      }
    } else {
    PhysParams ppf = pp;
    if constexpr (PH == PH_ROTATION2D) {
      // the velocity (y, -x) at the flux node's coordinates Vgf X
      double xf[2] = {0.0, 0.0};
#pragma unroll
      for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int d = 0; d < 2; ++d) xf[d] += tab[O::Vgf + f * NG + g] * X[g][d];
      ppf.p0 = xf[1];
      ppf.p1 = -xf[0];
    }
    point_flux<PH, double>(s, ppf, F, bad);
    if constexpr (AFFINE) {
#pragma unroll
      for (int xi = 0; xi < D; ++xi)
#pragma unroll
        for (int k = 0; k < M; ++k) {
          double t = 0.0;
#pragma unroll
          for (int d = 0; d < D; ++d) t += Jinv[0][d][xi] * F[d][k];
          G[xi][k] = t;
        }
    }
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      if constexpr (AFFINE) {
#pragma unroll
        for (int k = 0; k < M; ++k) {
          double t = divr[q][k];
#pragma unroll
          for (int xi = 0; xi < D; ++xi) t += dvf[xi * NQ + q] * G[xi][k];
          divr[q][k] = t;
        }
      } else {
        double b[D];
#pragma unroll
        for (int d = 0; d < D; ++d) {
          double t = 0.0;
#pragma unroll
          for (int xi = 0; xi < D; ++xi) t += Jinv[q][d][xi] * dvf[xi * NQ + q];
          b[d] = t;
        }
#pragma unroll
        for (int k = 0; k < M; ++k) {
          double t = divr[q][k];
#pragma unroll
          for (int d = 0; d < D; ++d) t += b[d] * F[d][k];
          divr[q][k] = t;
        }
      }
    }
  }
  }
  if constexpr (PREC == 3 || PREC == 5) {
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int k = 0; k < M; ++k) {
        double sq = 0.0;
#pragma unroll
        for (int n = 0; n < ND; ++n) sq += tab[O::V + q * ND + n] * nodal(n, k);
        divr[q][k] -= sq;
      }
  }
#pragma unroll
  for (int q = 0; q < NQ; ++q)
#pragma unroll
    for (int k = 0; k < M; ++k) lds_div[(q * M + k) * stride] = divr[q][k];
  }

  // ---- element scheme ------------------------------------------------------
  // NDIS: the scheme has the N dissipation. B and the PSI / LDA blend need it
  // apart from the LDA part (DIS2); N and PSI only their sum, which one K+
  // product per node and point gives: K+_n (w U_n + y), S y = w (r - sum K+ U).
  constexpr bool NDIS = (SC != SC_LDA);
  constexpr bool DIS2 = (SC == SC_B || SC == SC_BPSI);
  double lda[ND][M];  // (N and PSI: the N residual)
  double dis[DIS2 ? ND : 1][M];
  // max over nodes and quadrature points of |eigenvalue|; the floor 1e-6 of
  // every (node, point) term is applied once at the end (max(1e-6, max x) =
  // max over x of max(1e-6, x))
  double lmax = 0.0;
  double fint[M];
#pragma unroll
  for (int n = 0; n < ND; ++n) {
#pragma unroll
    for (int k = 0; k < M; ++k) lda[n][k] = 0.0;
  }
#pragma unroll
  for (int n = 0; n < (DIS2 ? ND : 1); ++n)
#pragma unroll
    for (int k = 0; k < M; ++k) dis[n][k] = 0.0;
#pragma unroll
  for (int k = 0; k < M; ++k) fint[k] = 0.0;
  double vol = 0.0;

  // TWO: the dissipative schemes of the 3D P2 cells (affine, R right-hand
  // sides) in two passes over the quadrature points,
  // so that neither holds the K+ parameters of all nodes beside the residual
  // sums:
  //   1. per point q: S_q = sum_n K+_n (one evaluation of each node's
  //      parameters, which also gives sum_n K+_n U_n) and its solves; the
  //      point's (V, a, H) replace its divergence slice in the LDS column and
  //      the R solutions follow the slices;
  //   2. per point q again, every node: its K+ products added to its sums (a
  //      second evaluation of the parameters).
  constexpr int R = DIS2 ? 2 : 1;
  constexpr bool TWO = DLDS && PatchWork<D, ND, NQ, AFFINE, PH, SC, PREC>::two;

  // LAST: the last node's residual from the cell's: the K+ products of a
  // point's nodes add up to its weighted residual (LDA part) and to zero
  // (dissipation), so the last node needs neither the products nor sums to
  // carry through the points. The P1 tetrahedra's blends then fit 256 registers
  // (28 instead of 160 bytes of scratch: 1.57 M cells PSI / LDA 307 -> 233 us a
  // sweep), other cells gain 0 to 4 %; P2 triangles with one sum per node keep
  // all products (N 91.6 against 92.8 us on the 196 608-cell channel). The errors
  // against a 64-bit reference are those of the products.
  constexpr bool LAST = M > 1 && !TWO && (DIS2 || ND != 6);

  // P1 simplices of the Euler physics (affine, D + 1 nodes): the basis
  // gradients, and with them the geometric part of every node's K+
  // parameters, are the same at every quadrature point; formed once per cell
  constexpr bool CG = (M > 1) && AFFINE && (ND == D + 1);
  EulerNodeG<D> cg[CG ? ND : 1];
  if constexpr (CG) {
#pragma unroll
    for (int n = 0; n < ND; ++n) cg[n] = euler_node_g<D, ND>(Jinv[0], tab + O::dVT, n);
  }

  auto quad_point = [&](const int q, double (&r)[M], const double (&Jq)[D][D], const double detq) {
    const double wj = tab[O::w + q] * detq;
    vol += wj;
    if constexpr (!LINF) {
#pragma unroll
      for (int k = 0; k < M; ++k) fint[k] += wj * r[k];
    }
    // reference gradients [D][ND] at q (P1 simplices: the same at every point, so
    // that what depends on them alone is formed once per cell: 524 288 P1
    // triangles of advection 15.3 -> 13.4 us)
    const double *dvq = tab + O::dVT + (AFFINE && ND == D + 1 ? 0 : q) * D * ND;

    if constexpr (PREC == 2 && SC == SC_LDA) {
      // shock capturing: w |J| nu_q grad(phi_n) . grad(u_k), nu interpolated
      // from the nodes like the state, added before the LDA share of q
      double nuq = 0.0;
#pragma unroll
      for (int n = 0; n < ND; ++n) nuq += tab[O::V + q * ND + n] * nodal(n);
      if (nuq != 0.0) {
        double gu[D][M];
#pragma unroll
        for (int x = 0; x < D; ++x)
#pragma unroll
          for (int k = 0; k < M; ++k) gu[x][k] = 0.0;
#pragma unroll
        for (int n = 0; n < ND; ++n) {
#pragma unroll
          for (int x = 0; x < D; ++x) {
            double gx = 0.0;
#pragma unroll
            for (int xi = 0; xi < D; ++xi) gx += Jq[x][xi] * dvq[xi * ND + n];
#pragma unroll
            for (int k = 0; k < M; ++k) gu[x][k] += gx * Uq(n, k);
          }
        }
#pragma unroll
        for (int n = 0; n < ND; ++n) {
#pragma unroll
          for (int x = 0; x < D; ++x) {
            double gx = 0.0;
#pragma unroll
            for (int xi = 0; xi < D; ++xi) gx += Jq[x][xi] * dvq[xi * ND + n];
            const double cx = wj * nuq * gx;
#pragma unroll
            for (int k = 0; k < M; ++k) lda[n][k] += cx * gu[x][k];
          }
        }
      }
    }

    if constexpr (M == 1) {
      double vel0, vel1;
      if constexpr (PH == PH_ADVECTION2D) {
        vel0 = double(pp.p0);
        vel1 = double(pp.p1);
      } else if constexpr (PH == PH_ROTATION2D) {
        // the velocity (y, -x) at the quadrature point's coordinates Vg X
        double xq[2] = {0.0, 0.0};
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
          for (int d = 0; d < 2; ++d) xq[d] += tab[O::Vg + q * NG + g] * X[g][d];
        vel0 = double(xq[1]);
        vel1 = double(-xq[0]);
      } else {
        double uq = 0.0;
#pragma unroll
        for (int n = 0; n < ND; ++n) uq += tab[O::V + q * ND + n] * Uq(n, 0);
        vel0 = uq;
        vel1 = 1.0;
      }
      // k_n = a . grad(phi_n) = sum_xi c_xi dphi_n/dxi with c_xi = sum_x a_x dxi/dx
      const double *dvk = dvq;
      double c[D];
#pragma unroll
      for (int xi = 0; xi < D; ++xi) c[xi] = vel0 * double(Jq[0][xi]) + vel1 * double(Jq[1][xi]);
      double kp[ND];
      double S = 0.0, SU = 0.0, kU = 0.0;
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        double knt = double(0);
#pragma unroll
        for (int xi = 0; xi < D; ++xi) knt += c[xi] * dvk[xi * ND + n];
        const double kn = knt;
        kp[n] = fmax(kn, 0.0);
        lmax = fmax(lmax, fabs(kn));
        S += kp[n];
        if constexpr (NDIS) SU += kp[n] * Uq(n, 0);
        if constexpr (LINF) kU += kn * Uq(n, 0);
      }
      if constexpr (LINF) {
        r[0] = kU;
        if constexpr (PREC == 3 || PREC == 5) {
#pragma unroll
          for (int n = 0; n < ND; ++n) r[0] -= tab[O::V + q * ND + n] * nodal(n, 0);
        }
        fint[0] += wj * r[0];
      }
      const double inv = recip(S);
      const double ub = NDIS ? SU * inv : 0.0;
      const double wr = wj * inv * r[0];
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        if constexpr (DIS2 || !NDIS) lda[n][0] += kp[n] * wr;
        if constexpr (DIS2) dis[n][0] += wj * (kp[n] * (Uq(n, 0) - ub));
        if constexpr (NDIS && !DIS2) lda[n][0] += kp[n] * (wr + wj * (Uq(n, 0) - ub));
      }
    } else {
      double uq[M];
#pragma unroll
      for (int k = 0; k < M; ++k) {
        double t = 0.0;
#pragma unroll
        for (int n = 0; n < ND; ++n) t += tab[O::V + q * ND + n] * Uq(n, k);
        uq[k] = t;
      }
      const EulerState<double, D> st = euler_state<double, D>(uq, double(pp.p0));
      bad = bad || st.bad;
      const EulerPoint<D> pt = euler_point<D>(st, pp.p0 - 1.0);
      const double *dvk = dvq;
      using NodeK = EulerNodeK<D>;
      // the K+ parameters of node n (recomputed where keeping them for all
      // nodes costs spills)
      auto node_k = [&](const int n) {
        if constexpr (CG)
          return euler_node_k<D>(cg[n], pt.V, pt.a);
        else
          return euler_node_k<D, ND>(Jq, dvk, n, pt.V, pt.a);
      };
      // 3D P2: recompute in the application instead of keeping ND sets
      constexpr bool KEEP = (D == 2) || CG;
      NodeK nk[KEEP ? ND : 1];
      EulerSum<D> S;
      S.clear();
      EulerKU<D> ku;
      if constexpr (NDIS) ku.clear();
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        const NodeK k = node_k(n);
        if constexpr (KEEP) nk[n] = k;
        lmax = fmax(lmax, k.emax);
        S.add(k);
        if constexpr (NDIS) {
          double un[M];
#pragma unroll
          for (int c = 0; c < M; ++c) un[c] = Uq(n, c);
          ku.add(pt, k, un);
        }
      }
      auto node_at = [&](const int n) -> NodeK {
        if constexpr (KEEP) {
          return nk[n];
        } else if constexpr (SC == SC_LDA) {
          // an opaque copy of the index: the parameters are recomputed here,
          // not kept alive from the loop over S (which common-subexpression
          // elimination would otherwise do); measured faster for LDA (no
          // scratch) and slower for the dissipative schemes, whose second
          // application per node reuses the parameters
          int nn = n;
          asm volatile("" : "+s"(nn));
          return node_k(nn);
        } else {
          return node_k(n);
        }
      };
      S.factor();
      // the right-hand sides: w r (LDA part) and w sum K+ U, or their
      // difference where only the N residual is needed
      double b[M], x[M], p, Q[D], kun[M], ub[M], pu, Qu[D];
      if constexpr (NDIS) ku.total(pt, kun);
#pragma unroll
      for (int k = 0; k < M; ++k) b[k] = wj * ((NDIS && !DIS2) ? r[k] - kun[k] : r[k]);
      S.solve(pt, b, x, p, Q);
      if constexpr (DIS2) S.solve(pt, kun, ub, pu, Qu);
#pragma unroll
      for (int n = 0; n < (LAST ? ND - 1 : ND); ++n) {
        const NodeK kn = node_at(n);
        if constexpr (DIS2 || !NDIS) pt.apply(kn, x, p, Q, lda[n]);
        if constexpr (NDIS) {
          double du[M];
#pragma unroll
          for (int k = 0; k < M; ++k) du[k] = DIS2 ? wj * (Uq(n, k) - ub[k]) : wj * Uq(n, k) + x[k];
          pt.apply(kn, du, DIS2 ? dis[n] : lda[n]);
        }
      }
    }
  };

  if constexpr (TWO) {
    const double gm1 = pp.p0 - 1.0;
    const double(&Jq)[D][D] = Jinv[0];
    // LDS column: [q M, q M + M) the divergence of q, then (V, a, H) of q;
    // [NQ M + R M q, + R M) its solutions
    double *const qx = lds_div + static_cast<size_t>(NQ) * M * stride;
#pragma unroll 1
    for (int q = 0; q < NQ; ++q) {
      double r[M];
#pragma unroll
      for (int k = 0; k < M; ++k) r[k] = lds_div[(q * M + k) * stride];
      const double wj = tab[O::w + q] * detJ[0];
      vol += wj;
#pragma unroll
      for (int k = 0; k < M; ++k) fint[k] += wj * r[k];
      const double *dvk = tab + O::dVT + q * D * ND;
      double uq[M];
#pragma unroll
      for (int k = 0; k < M; ++k) {
        double t = 0.0;
#pragma unroll
        for (int n = 0; n < ND; ++n) t += tab[O::V + q * ND + n] * Uq(n, k);
        uq[k] = t;
      }
      const EulerState<double, D> st = euler_state<double, D>(uq, double(pp.p0));
      bad = bad || st.bad;
      const EulerPoint<D> pt = euler_point<D>(st, gm1);
      EulerSum<D> S;
      EulerKU<D> ku;
      S.clear();
      ku.clear();
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        const EulerNodeK<D> k = euler_node_k<D, ND>(Jq, dvk, n, pt.V, pt.a);
        lmax = fmax(lmax, k.emax);
        S.add(k);
        double un[M];
#pragma unroll
        for (int c = 0; c < M; ++c) un[c] = Uq(n, c);
        ku.add(pt, k, un);
      }
      S.factor();
      double b[M], kun[M], x[M], p, Q[D];
      ku.total(pt, kun);
#pragma unroll
      for (int k = 0; k < M; ++k) b[k] = wj * (DIS2 ? r[k] : r[k] - kun[k]);
      S.solve(pt, b, x, p, Q);
#pragma unroll
      for (int k = 0; k < M; ++k) qx[(R * M * q + k) * stride] = x[k];
      if constexpr (DIS2) {
        S.solve(pt, kun, x, p, Q);
#pragma unroll
        for (int k = 0; k < M; ++k) qx[(R * M * q + M + k) * stride] = x[k];
      }
#pragma unroll
      for (int d = 0; d < D; ++d) lds_div[(q * M + d) * stride] = pt.V[d];
      lds_div[(q * M + D) * stride] = pt.a;
      lds_div[(q * M + D + 1) * stride] = pt.H;
    }
#pragma unroll 1
    for (int q = 0; q < NQ; ++q) {
      EulerPoint<D> pt;
      double x[M], ub[M], Q[D];
      double v2 = 0.0;
#pragma unroll
      for (int d = 0; d < D; ++d) {
        pt.V[d] = lds_div[(q * M + d) * stride];
        v2 += pt.V[d] * pt.V[d];
      }
      pt.a = lds_div[(q * M + D) * stride];
      pt.H = lds_div[(q * M + D + 1) * stride];
      pt.ia = recip(pt.a);
      pt.hv = 0.5 * v2;
      pt.ga = gm1 * pt.ia;
#pragma unroll
      for (int k = 0; k < M; ++k) x[k] = qx[(R * M * q + k) * stride];
      if constexpr (DIS2) {
#pragma unroll
        for (int k = 0; k < M; ++k) ub[k] = qx[(R * M * q + M + k) * stride];
      }
#pragma unroll
      for (int d = 0; d < D; ++d) Q[d] = x[1 + d] - pt.V[d] * x[0];
      const double p = pt.p_of(x);
      const double wj = tab[O::w + q] * detJ[0];
      const double *dvk = tab + O::dVT + q * D * ND;
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        const EulerNodeK<D> k = euler_node_k<D, ND>(Jq, dvk, n, pt.V, pt.a);
        double du[M];
#pragma unroll
        for (int c = 0; c < M; ++c) du[c] = DIS2 ? wj * (Uq(n, c) - ub[c]) : wj * Uq(n, c) + x[c];
        if constexpr (DIS2) pt.apply(k, x, p, Q, lda[n]);
        pt.apply(k, du, DIS2 ? dis[n] : lda[n]);
      }
    }
  } else {
#pragma unroll 1
  for (int q = 0; q < NQ; ++q) {
    double r[M];
    if constexpr (!LINF) {
#pragma unroll
      for (int k = 0; k < M; ++k) r[k] = lds_div[(q * M + k) * stride];
    }
    if constexpr (AFFINE) {
      quad_point(q, r, Jinv[0], detJ[0]);
    } else {
      // recompute the Jacobian at q instead of indexing a per-q array
      double J[D][D], Ji[D][D];
#pragma unroll
      for (int xi = 0; xi < D; ++xi)
#pragma unroll
        for (int x = 0; x < D; ++x) {
          double t = 0.0;
#pragma unroll
          for (int g = 0; g < NG; ++g) t += tab[O::dVgT + (q * D + xi) * NG + g] * X[g][x];
          J[xi][x] = t;
        }
      const double dq = det_inv<D>(J, Ji);
      quad_point(q, r, Ji, dq);
    }
  }
  }

  if constexpr (LAST) {
#pragma unroll
    for (int k = 0; k < M; ++k) {
      double s = fint[k], d = 0.0;
#pragma unroll
      for (int n = 0; n < ND - 1; ++n) {
        s -= lda[n][k];
        if constexpr (DIS2) d -= dis[n][k];
      }
      lda[ND - 1][k] = s;
      if constexpr (DIS2) dis[DIS2 ? ND - 1 : 0][k] = d;
    }
  }

  // ---- blend / limit -------------------------------------------------------
  if constexpr (SC == SC_LDA || SC == SC_N) {
#pragma unroll
    for (int n = 0; n < ND; ++n)
#pragma unroll
      for (int k = 0; k < M; ++k) phi[n][k] = lda[n][k];
  } else if constexpr (SC == SC_B && (PREC == 2 || PREC == 5)) {
    // external nodal coefficient; below 1e-6 at every node the cell keeps
    // its LDA residuals
    double th[ND];
    double tmax = 0.0;
#pragma unroll
    for (int n = 0; n < ND; ++n) {
      th[n] = nodal(n);
      tmax = fmax(tmax, th[n]);
    }
    const bool skip = tmax < 1.e-6;
#pragma unroll
    for (int n = 0; n < ND; ++n)
#pragma unroll
      for (int k = 0; k < M; ++k) phi[n][k] = skip ? lda[n][k] : lda[n][k] + th[n] * dis[n][k];
  } else if constexpr (SC == SC_B) {
    double an = 0.0;
#pragma unroll
    for (int n = 0; n < ND; ++n) an += fabs(lda[n][0] + dis[n][0]);
    const double theta = fabs(fint[0]) / (an + 1.e-6);
#pragma unroll
    for (int n = 0; n < ND; ++n)
#pragma unroll
      for (int k = 0; k < M; ++k) phi[n][k] = lda[n][k] + theta * dis[n][k];
  } else {
    // PSI: the x+ limiter of the N residuals, per equation; the PSI / LDA
    // blend then takes (1 - theta) LDA + theta PSI with PGB's cell theta
    double theta = 1.0;
    if constexpr (SC == SC_BPSI) {
      double an = 0.0;
#pragma unroll
      for (int n = 0; n < ND; ++n) an += fabs(lda[n][0] + dis[n][0]);
      theta = fabs(fint[0]) / (an + 1.e-6);
    }
#pragma unroll
    for (int k = 0; k < M; ++k) {
      const double tot = fint[k];
      const bool lim = fabs(tot) > 1.e-14;
      const double itot = lim ? 1.0 / tot : 0.0;
      double xs[ND];
      double sx = 0.0;
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        xs[n] = fmax((DIS2 ? lda[n][k] + dis[n][k] : lda[n][k]) * itot, 0.0) + 1.e-12;
        sx += xs[n];
      }
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        const double psi = lim ? xs[n] / sx * tot : (DIS2 ? lda[n][k] + dis[n][k] : lda[n][k]);
        phi[n][k] = (SC == SC_BPSI) ? (1.0 - theta) * lda[n][k] + theta * psi : psi;
      }
    }
  }

  wave = vol * fmax(lmax, 1.e-6);
}

template <int D, int NG, int NQ, int M>
__device__ __forceinline__ void gather_coords(const CellArgs &a, uint32_t e, double (&X)[NG][D])
{
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const size_t v = a.gconn[static_cast<size_t>(g) * a.ne + e];
#pragma unroll
    for (int d = 0; d < D; ++d) X[g][d] = a.coords[v * D + d];
  }
}

// Table of a workgroup's nodes in LDS (FP64 atomics): SLOTS entries of a node id
// and its M + 1 sums, the entry of a node being its id modulo SLOTS. A power of
// two, at least half the number of the workgroup's (cell, node) pairs, which is
// above the number of nodes of cells in any sensible order, but for two elements
// where that would take more than 48 KiB: 256 P2 tetrahedra of the Euler equations
// have 512 entries for about 770 nodes, 256 of their Q2 quadrilaterals 1 024 for
// about 1 090, so that some of their nodes always go to global memory directly.
template <int ND, int M>
struct NodeTable
{
  static constexpr size_t entry = sizeof(uint32_t) + (M + 1) * sizeof(double);
  __host__ __device__ static constexpr int slots(int block)
  {
    int n = 64;
    while (2 * n < block * ND) n *= 2;
    while (n * entry > 49152) n /= 2;
    return n;
  }
  __host__ __device__ static constexpr size_t bytes(int block) { return slots(block) * entry; }
};

// Waves per SIMD that the registers of a cell kernel must leave room for: 2 for the
// LDA of P2 triangles (Euler), which would take 259 registers and has 20 bytes of
// scratch at 256: 786 432 P2 / Q2 cells by colours 479 -> 420 us, 250 000 triangles
// with atomics 288 -> 275 us. The compiler's choice for the others (rotating P3 LDA
// and the Q1 B scheme with a blending coefficient, 130 and 258 registers: no change).
template <int M, int ND, int SC, int PREC>
struct CellMinWaves
{
  static constexpr int value = (M == 4 && ND == 6 && SC == SC_LDA && PREC == 0) ? 2 : 1;
};

// Element-per-thread cell loop with a global scatter: FP64 atomics or, one
// colour per launch, plain read-modify-write.
// With atomics the workgroup first adds its cells' parts in LDS: a node's entry
// is claimed by the first cell that finds it free, cells whose node finds its
// entry taken by another one add to global memory directly, and each claimed
// entry then goes to global memory once. Cells next to each other in the
// caller's order share most of their nodes, and the global atomics are what
// bounds this kernel (its arithmetic is 5 us of it): 262 144 P2 Burgers cells 86
// us with every part in global memory, 54 us with entries for a third of the
// pairs, 44 us for two thirds.
// The cells of a method are sorted by colour here and those of one colour share no
// node; there the entries only put the atomics in the order of the nodes, still
// worth 20 % (131 072 P1 cells 21 us directly, 17 us). It does not pay where few
// workgroups hold cells in no order at all (32 768 shuffled P2 Euler triangles LDA
// 64 us directly, 73 us).
template <int D, int NG, int ND, int NF, int NQ, bool AFFINE, int PH, int SC, int PREC = 0>
__global__ __launch_bounds__(256, (CellMinWaves<PhysTraits<PH>::M, ND, SC, PREC>::value)) void rd_cell_kernel(CellArgs a)
{
  constexpr int M = PhysTraits<PH>::M;
  extern __shared__ double lds[];
  const uint32_t local = xcd_block_index() * blockDim.x + threadIdx.x;
  bool active = local < a.count;
  const uint32_t e = a.first + (active ? local : 0);
  bool bad = false, outside = false;
  uint32_t nid[ND];
#pragma unroll
  for (int n = 0; n < ND; ++n) nid[n] = a.sconn[static_cast<size_t>(n) * a.ne + e];
  if (a.nn_check) {
    bool out = false;
#pragma unroll
    for (int g = 0; g < NG; ++g) out = out || a.gconn[static_cast<size_t>(g) * a.ne + e] >= a.nv_check;
#pragma unroll
    for (int n = 0; n < ND; ++n) out = out || nid[n] >= a.nn_check;
    outside = active && out;
    active = active && !out;
  }
  double phi[ND][M];
  double wave = 0.0;
  if (active) {
    double X[NG][D];
    gather_coords<D, NG, NQ, M>(a, e, X);
    double U[ND][M];
#pragma unroll
    for (int n = 0; n < ND; ++n)
#pragma unroll
      for (int k = 0; k < M; ++k) U[n][k] = a.u[static_cast<size_t>(nid[n]) * M + k];
    if constexpr (PREC == 2)
      cell_residual<D, NG, ND, NF, NQ, AFFINE, PH, SC, 2>(a.tab, X, U, URegs<ND, M>{U}, a.pp, phi, wave, bad,
                                                       lds + threadIdx.x, static_cast<int>(blockDim.x),
                                                       NodalGlobal<ND>{a.nodal, nid});
    else
      cell_residual<D, NG, ND, NF, NQ, AFFINE, PH, SC, 0>(a.tab, X, U, URegs<ND, M>{U}, a.pp, phi, wave, bad,
                                                       lds + threadIdx.x, static_cast<int>(blockDim.x));
  }
  if (a.atomic) {
    const int slots = NodeTable<ND, M>::slots(blockDim.x);
    double *const sum = lds;  // [M + 1][slots]
    uint32_t *const key = reinterpret_cast<uint32_t *>(lds + static_cast<size_t>(M + 1) * slots);
    constexpr uint32_t FREE = 0xffffffffu;
    lds_barrier();  // the columns' region becomes the table
    for (int i = threadIdx.x; i < slots; i += blockDim.x) {
      key[i] = FREE;
#pragma unroll
      for (int k = 0; k <= M; ++k) sum[k * slots + i] = 0.0;
    }
    lds_barrier();
    if (active) {
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        const uint32_t i = nid[n] & (slots - 1);
        const uint32_t was = atomicCAS(key + i, FREE, nid[n]);
        if (was == FREE || was == nid[n]) {
#pragma unroll
          for (int k = 0; k < M; ++k) unsafeAtomicAdd(sum + k * slots + i, phi[n][k]);
          unsafeAtomicAdd(sum + M * slots + i, wave);
        } else {
#pragma unroll
          for (int k = 0; k < M; ++k) unsafeAtomicAdd(a.acc_res + static_cast<size_t>(nid[n]) * M + k, phi[n][k]);
          unsafeAtomicAdd(a.acc_ws + nid[n], wave);
        }
      }
    }
    lds_barrier();
    for (int i = threadIdx.x; i < slots; i += blockDim.x) {
      const uint32_t g = key[i];
      if (g == FREE) continue;
#pragma unroll
      for (int k = 0; k < M; ++k) unsafeAtomicAdd(a.acc_res + static_cast<size_t>(g) * M + k, sum[k * slots + i]);
      unsafeAtomicAdd(a.acc_ws + g, sum[M * slots + i]);
    }
  } else if (active) {
#pragma unroll
    for (int n = 0; n < ND; ++n) {
      const size_t b = static_cast<size_t>(nid[n]);
#pragma unroll
      for (int k = 0; k < M; ++k) a.acc_res[b * M + k] += phi[n][k];
      a.acc_ws[b] += wave;
    }
  }
  // (behind the cell work: a store ahead of it turns the table loads from scalar
  // into vector loads; without them 262 144 P2 Burgers cells of a caller's arrays
  // take 41.8 instead of 54.1 us a residual, 32 768 P3 ones of a method 30.2
  // instead of 43.1 us)
  if (outside) atomicOr(a.status, 2);
  if (bad) atomicOr(a.status, 1);
}

// ---------------------------------------------------------------------------
// Patch assembly: one workgroup owns one patch of up to PATCH cells (a
// spatially compact run of the Morton-ordered cells). The states of the
// patch's nodes are gathered once into LDS; every cell writes its residuals
// and wave speed to the LDS slot of each of its (cell, node) pairs, the pairs
// being grouped by node (the rank of a pair within its node comes with the
// connectivity), so each node then sums a contiguous run of slots in a fixed
// order -- no atomics and the same result on every run. Then
//   * nodes held by this patch only are finished here: residual / V, wave
//     speed, and -- in iteration mode -- dt = CFL V / sum lambda,
//     u -= dt res (after the strong Dirichlet value),
//   * nodes shared with other patches write their partial sums to their slot;
//     patch_fixup_kernel sums the slots of every shared node in a fixed order.
// Between two iterations the fix-up can be left out: the next sweep's
// patches then finish their shared nodes themselves while gathering them
// (prev_acc: the previous sweep's rows; base_in: the shared nodes' states at
// its start), each holder summing the same rows in the same order, so all
// holders agree bit for bit with each other and with the fix-up. The holder
// owning the node's first row (its lowest-numbered patch) stores the new
// state to u and, when the sweep after this one is deferred too, to
// base_out. The rows and the states alternate between two buffers, since
// other patches of a sweep still read the previous sweep's.
// ---------------------------------------------------------------------------
constexpr int LC_BITS = 10;  // local node index bits of a patch connectivity entry
constexpr int LC_MASK = (1 << LC_BITS) - 1;

struct PatchArgs
{
  const double *__restrict__ tab;
  const uint32_t *__restrict__ gconn;       // [NG][ne] global vertex ids
  const uint16_t *__restrict__ lconn;       // [ND][ne] local node | rank << LC_BITS
  const uint32_t *__restrict__ pnode_off;   // [np + 1] first slot of each patch
  const uint32_t *__restrict__ pnodes;      // [slots] global node id of each slot
  const uint32_t *__restrict__ pn_inner;    // [np] number of patch-only nodes (listed first)
  const uint16_t *__restrict__ pn_coff;     // [slots] first (cell, node) pair of the slot's node
  const double *__restrict__ coords;
  double *__restrict__ u;                   // [N][M] (updated in place in iteration mode)
  const double *__restrict__ vol;           // [N]
  const int *__restrict__ dir_index;        // [N] row in dir_vals or -1
  const double *__restrict__ dir_vals;      // [ndir][M]
  // linear sweeps of the mixed-precision form (PREC 4): the element
  // Jacobians of the block in FP32, [ND M][ND M][ne] (entry-major, patch
  // order), and the linearisation point: its state u_ref [N][M], its FP64
  // residual lin_res [N][M] and time step lin_dt [N]
  const float *__restrict__ jlin;
  const double *__restrict__ u_ref;
  const double *__restrict__ lin_res;
  const double *__restrict__ lin_dt;
  double *__restrict__ res;                 // [N][M]
  double *__restrict__ dt;                  // [N]
  double *__restrict__ ws;                  // [N]
  double *__restrict__ slot_acc;            // [shared slots][M + 1] partial sums, grouped by node
  const uint32_t *__restrict__ slot_pos;    // [slots] row of a shared slot in slot_acc
  const uint32_t *__restrict__ pn_sid;      // [slots] shared-node index of a shared slot
  const uint2 *__restrict__ pn_rows;        // [slots] rows [x, y) of a shared slot's node
  const double *__restrict__ prev_acc;      // rows of the previous sweep, not yet summed, or null
  const double *__restrict__ base_in;       // [n_shared][M] states at the start of the previous sweep
  double *__restrict__ base_out;            // [n_shared][M] states at the start of this sweep, or null
  double *__restrict__ norm_partial;        // [np][M + 1]
  const double *__restrict__ nodal;         // [N] blending coefficient (B) / artificial viscosity (LDA), PREC 2;
                                            // [N][M] source field, PREC 3 and 5
  const double *__restrict__ theta;         // [N] PREC 5: the B scheme's external blending coefficient
  int *__restrict__ status;
  uint32_t ne, np, first_patch;             // first_patch: offset of this block's patches
  int maxl;                                 // LDS rows of node state
  int update;                               // 0: assemble (res, ws), 1: iterate, 2: assemble with dt
  int outputs;                              // iterate: also store res, dt, ws and norm partials
  int excl;                                 // norm without Dirichlet rows
  double cfl;
  PhysParams pp;
};

// Largest (and default) number of cells per patch (= threads per
// workgroup): 256 for scalar physics on elements of up to 6 nodes, 128 for
// the Euler systems (larger per-thread state) and for P3 / Q2 elements (more
// nodes per patch), 64 for the 3D Euler equations on P2 tetrahedra (whose
// (cell, node) pair sums of 128 cells alone would fill 60 KB of LDS). A block
// may use 64 or 128 instead (PDRD_OPT_PATCH_CELLS).
template <int M, int ND>
struct PatchSize
{
  static constexpr int value = (M == 1 && ND <= 6) ? 256 : ((M == 5 && ND > 4) ? 64 : 128);
};

// Nodes of a thread that a patch kernel gathers together: the nodes of a full
// patch of a structured mesh over its threads, rounded up (a patch of C cells
// has about C / 2 + sqrt(2 C) P1, 2 C P2 and 4.5 C P3 nodes of triangles, C Q1
// and 4 C Q2 nodes of quadrilaterals, C / 2 P1 and 3 C P2 nodes of
// tetrahedra). None for the P2 tetrahedra at 2 waves, whose 256 registers it
// would spill.
template <int M, int ND, int NQ, bool AFFINE, int SC, int PREC>
struct PatchNodes
{
  static constexpr bool full = M == 5 && ND > 4 && PatchMinWaves<M, ND, NQ, AFFINE, SC, PREC>::value == 2;
  static constexpr int value = (PREC == 4 || full) ? 0
                               : (ND == 3)         ? 1
                               : (ND == 4)         ? (M == 5 ? 1 : 2)
                               : (ND == 6)         ? 3
                               : (M == 5)          ? 3
                                                   : 5;
};

// Dynamic LDS of one patch workgroup of P cells, in doubles: node state
// [maxl][M], the pair offsets of the nodes [maxl] (u16), then a work region of
// PatchWork::per_cell doubles a cell, shared in turn by the cells' columns, the
// (cell, node) pair sums and the norm reduction. With a nodal input (PREC 2)
// its values follow the work region, one per local node; with a source field
// (PREC 3), M per local node, and with both (PREC 5) M + 1. In a linear sweep
// (PREC 4) the state differences delta of the patch's nodes follow, [maxl][M]
// floats.
__host__ __device__ constexpr size_t patch_coff_doubles(int maxl) { return (static_cast<size_t>(maxl) + 3) / 4; }

template <class PW, int PREC>
__host__ __device__ constexpr size_t patch_lds_doubles(int maxl, int P)
{
  constexpr int M = PW::M;
  const size_t n = static_cast<size_t>(maxl);
  return n * M + patch_coff_doubles(maxl) + static_cast<size_t>(P) * PW::per_cell +
         (PREC == 2 ? n : (PREC == 3 ? n * M : (PREC == 4 ? (n * M + 1) / 2 : (PREC == 5 ? n * (M + 1) : 0))));
}

// Finishes node g from its sums acc[M + 1] (residual sum, wave-speed sum);
// u_old is the node's state at the start of the sweep.
// Sum of the partial-sum rows [r0, r1) of one shared node, in row order;
// the loads of four rows are issued before their additions.
template <int M>
__device__ __forceinline__ void sum_rows(const double *__restrict__ rows, uint32_t r0, uint32_t r1, double (&acc)[M + 1])
{
  constexpr int RB = 4;
#pragma unroll
  for (int k = 0; k <= M; ++k) acc[k] = 0.0;
  for (uint32_t s = r0; s < r1; s += RB) {
    double v[RB][M + 1];
#pragma unroll
    for (int j = 0; j < RB; ++j)
      if (s + j < r1)
#pragma unroll
        for (int k = 0; k <= M; ++k) v[j][k] = rows[static_cast<size_t>(s + j) * (M + 1) + k];
#pragma unroll
    for (int j = 0; j < RB; ++j)
      if (s + j < r1)
#pragma unroll
        for (int k = 0; k <= M; ++k) acc[k] += v[j][k];
  }
}

// The pseudo-time step of node g: residual r = sum / V, dt = CFL V / sum
// lambda, new state = (strong Dirichlet value or u_old) - dt r. In a linear
// sweep (lin_res set) the sums are those of J delta and r = lin_res + sum / V,
// dt = lin_dt: the residual linearised about u_ref with the time step there.
// Both the in-kernel finish and the deferred one use it, so they round alike.
// (The time step is a quotient rounded once: a product with the reciprocal is up to
// 1.5 ulp off. 50 sweeps of 32 768 P1 cells: product 296.4, this 298.4, IEEE division
// 302.6 us.)
// v = vol[g] and di = dir_index[g] come from the caller (loaded ahead).
template <int M>
__device__ __forceinline__ void node_step(const PatchArgs &a, uint32_t g, const double *acc, const double *u_old,
                                          double v, int di, double (&r)[M], double (&un)[M], double &d)
{
  const double iv = recip(v);
  d = a.lin_res ? a.lin_dt[g] : quotient(a.cfl * v, acc[M]);
#pragma unroll
  for (int k = 0; k < M; ++k) {
    const size_t j = static_cast<size_t>(g) * M + k;
    r[k] = a.lin_res ? acc[k] * iv + a.lin_res[j] : acc[k] * iv;
    const double u0 = (di >= 0) ? a.dir_vals[static_cast<size_t>(di) * M + k] : u_old[k];
    un[k] = u0 - d * r[k];
  }
}

template <int M>
__device__ __forceinline__ void finish_node(const PatchArgs &a, uint32_t g, const double *acc, const double *u_old,
                                            double v, int di, double (&sq)[M + 1])
{
  if (a.update == 1) {
    double r[M], un[M], d;
    node_step<M>(a, g, acc, u_old, v, di, r, un, d);
    const bool count = a.outputs && !(a.excl && di >= 0);
#pragma unroll
    for (int k = 0; k < M; ++k) {
      const size_t j = static_cast<size_t>(g) * M + k;
      a.u[j] = un[k];
      if (a.outputs) a.res[j] = r[k];
      if (count) sq[k] += r[k] * r[k];
    }
    if (count) sq[M] += 1.0;
    if (a.outputs) {
      a.dt[g] = d;
      a.ws[g] = acc[M];
    }
  } else {
    const double iv = recip(v);
#pragma unroll
    for (int k = 0; k < M; ++k) a.res[static_cast<size_t>(g) * M + k] = acc[k] * iv;
    a.ws[g] = acc[M];
    if (a.update == 2) a.dt[g] = quotient(a.cfl * v, acc[M]);
    // the strong Dirichlet value (nobody reads a node's state any more once it
    // is finished)
    if (di >= 0) {
#pragma unroll
      for (int k = 0; k < M; ++k) a.u[static_cast<size_t>(g) * M + k] = a.dir_vals[static_cast<size_t>(di) * M + k];
    }
  }
}

template <int M>
__device__ __forceinline__ void block_sum_store(double (&sq)[M + 1], double *red, double *out)
{
  // red: blockDim * (M + 1) doubles of LDS
  __syncthreads();
#pragma unroll
  for (int k = 0; k <= M; ++k) red[k * blockDim.x + threadIdx.x] = sq[k];
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) {
#pragma unroll
      for (int k = 0; k <= M; ++k) red[k * blockDim.x + threadIdx.x] += red[k * blockDim.x + threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k <= M; ++k) out[k] = red[k * blockDim.x];
  }
}

// One patch (local index pl of the block described by a) on one workgroup. BATCH: a
// lies in device memory (the batch kernels).
template <int D, int NG, int ND, int NF, int NQ, bool AFFINE, int PH, int SC, int PREC, bool BATCH = false>
__device__ __forceinline__ void patch_body(const PatchArgs &a, uint32_t pl, double *lds)
{
  constexpr int M = PhysTraits<PH>::M;
  const int PATCH = blockDim.x;     // cells per patch of this block (a multiple of 64, <= PatchSize)
  const int NPAIR = PATCH * ND;      // stride of one component in the pair sums
  double *ul = lds;
  uint16_t *coff = reinterpret_cast<uint16_t *>(lds + static_cast<size_t>(a.maxl) * M);
  double *work = lds + static_cast<size_t>(a.maxl) * M + patch_coff_doubles(a.maxl);

  const uint32_t p = a.first_patch + pl;
  const uint32_t s0 = a.pnode_off[p];
  const int nl = static_cast<int>(a.pnode_off[p + 1] - s0);
  const int tid = threadIdx.x;
  const uint32_t e0 = pl * PATCH;
  const int ecount = static_cast<int>(min(static_cast<uint32_t>(PATCH), a.ne - e0));
  const bool active = tid < ecount;

  // the cell's vertices and local nodes do not depend on LDS: issue their
  // loads before the gather
  double X[NG][D];
  uint16_t lc[ND];
  if (active) {
    const uint32_t e = e0 + tid;
    if constexpr (PREC != 4) {
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const size_t v = a.gconn[static_cast<size_t>(g) * a.ne + e];
#pragma unroll
        for (int d = 0; d < D; ++d) X[g][d] = a.coords[v * D + d];
      }
    }
#pragma unroll
    for (int n = 0; n < ND; ++n) lc[n] = a.lconn[static_cast<size_t>(n) * a.ne + e];
  }
  using PW = PatchWork<D, ND, NQ, AFFINE, PH, SC, PREC>;
  double *nodal_l = work + static_cast<size_t>(PATCH) * PW::per_cell;  // PREC 2, 3 and 5 only
  float *delta_l = reinterpret_cast<float *>(nodal_l);                 // PREC 4 only
  // (no global store before the cell work: the table loads stay scalar)
  const int ninner = static_cast<int>(a.pn_inner[p]);
  // The first GN nodes of a thread (nearly always all of them) are gathered
  // together: all their ids, then all their states, so that a thread waits for
  // two rounds of memory and not for two per node. What the node finish needs
  // of them (id, volume, Dirichlet index, slot) is loaded here too where the
  // registers are free (EARLY) and arrives during the cell work, or else
  // behind the cell work, ahead of the pair sums, again all nodes together.
  // The timed sweeps are 1 to 4 % shorter for it, those of the small scalar
  // meshes 4 to 11 % (101 250 P3 triangles N 22.6 -> 20.2 us). It costs registers:
  // the scalar P3 cells run 3 waves per SIMD with it (B and the blend 2) and could
  // run 4 (3) without, and are up to 11 % faster with it at every size (7 200 to 500
  // 000 cells, LDA 13.5 against 14.1 us and 62.5 against 64.0). The Q2 Burgers
  // cells, which also hold the flux loop's sums, fall from 3 waves to 2: the finish
  // is loaded late there (LATE; not with a source field and the blending coefficient,
  // which have 2 waves either way: 46 against 51 us). 160 000 cells, LDA, which 3
  // waves hold at once: 42.6 -> 27.6 us (33.6 with the nodes one by one), 25 600
  // cells 18.6 -> 17.7; with a nodal input or a source field 44.1 -> 33.3 us, and
  // 18.3 -> 19.8 (21.5). Batches, whose arguments lie in memory, load it early: one
  // method of 25 600 cells 26.3 against 30.3 us, four of 160 000 cells 168 us (198
  // with the nodes one by one); only where 3 waves hold the batch and 2 don't, the
  // late loads win (160 000 cells in all 59.3 against 50.7, 54.6 one by one).
  constexpr int GN = PatchNodes<M, ND, NQ, AFFINE, SC, PREC>::value;
  constexpr int GNS = GN > 0 ? GN : 1;
  constexpr bool LATE = !BATCH && M == 1 && ND == 9 && PREC != 5 && !CellColumn<D, ND, NQ, AFFINE, PH>::linear_flux;
  constexpr bool EARLY = M == 1 ? ND != 6 && !LATE : PatchMinWaves<M, ND, NQ, AFFINE, SC, PREC>::value == 1;
  // The scalar kernels read of every node only what its kind needs (volume and
  // Dirichlet index of the patch's own nodes; slot, rows and start state of the
  // shared ones): 1.05 M P2 Burgers cells fetch 105 MB a chained sweep, without
  // these branches 147 MB, 58.3 against 59.5 us; on the Euler kernels the branches
  // cost 1 to 5 %.
  constexpr bool SPLIT = M == 1;
  uint32_t pg[GNS], psp[GNS];
  double pv[GNS];
  int pdi[GNS];
  auto load_finish = [&]() {
    int t = tid;
    if constexpr (!EARLY) {
      // (an opaque copy: the gather's addresses are not kept for this)
      asm volatile("" : "+v"(t));
#pragma unroll
      for (int j = 0; j < GN; ++j) pg[j] = a.pnodes[s0 + min(t + j * PATCH, nl - 1)];
    }
#pragma unroll
    for (int j = 0; j < GN; ++j) {
      const int l = min(t + j * PATCH, nl - 1);
      if constexpr (SPLIT) {
        double v = 1.0;
        int di = -1;
        uint32_t sp = 0;
        if (l < ninner) {
          v = a.vol[pg[j]];
          di = a.dir_index[pg[j]];
        } else {
          sp = a.slot_pos[s0 + l];
        }
        pv[j] = v;
        pdi[j] = di;
        psp[j] = sp;
      } else {
        pv[j] = a.vol[pg[j]];
        pdi[j] = a.dir_index[pg[j]];
        psp[j] = a.slot_pos[s0 + l];
      }
    }
  };
  // state un of node l (id g) and its other inputs to LDS
  auto put_node = [&](const int l, const uint32_t g, const double (&un)[M]) {
#pragma unroll
    for (int k = 0; k < M; ++k) ul[l * M + k] = un[k];
    if constexpr (PREC == 4)
#pragma unroll
      for (int k = 0; k < M; ++k)
        delta_l[l * M + k] = static_cast<float>(un[k] - a.u_ref[static_cast<size_t>(g) * M + k]);
    if constexpr (PREC == 2) nodal_l[l] = a.nodal[g];
    if constexpr (PREC == 3 || PREC == 5)
#pragma unroll
      for (int k = 0; k < M; ++k) nodal_l[l * M + k] = a.nodal[static_cast<size_t>(g) * M + k];
    if constexpr (PREC == 5) nodal_l[static_cast<size_t>(a.maxl) * M + l] = a.theta[g];
  };
  // a node on its own
  auto gather_node = [&](const int l, const uint32_t g) {
    double un[M];
    if (a.prev_acc && l >= ninner) {
      // shared node whose previous sweep is summed here
      const uint32_t i = a.pn_sid[s0 + l];
      const uint2 rr = a.pn_rows[s0 + l];
      double acc[M + 1], uo[M], r[M], d;
#pragma unroll
      for (int k = 0; k < M; ++k) uo[k] = a.base_in[static_cast<size_t>(i) * M + k];
      sum_rows<M>(a.prev_acc, rr.x, rr.y, acc);
      node_step<M>(a, g, acc, uo, a.vol[g], a.dir_index[g], r, un, d);
    } else {
#pragma unroll
      for (int k = 0; k < M; ++k) un[k] = a.u[static_cast<size_t>(g) * M + k];
    }
    put_node(l, g, un);
    coff[l] = a.pn_coff[s0 + l];
  };
  if constexpr (GN > 0) {
    uint16_t pc[GNS];
#pragma unroll
    for (int j = 0; j < GN; ++j) {
      const int l = min(tid + j * PATCH, nl - 1);
      pg[j] = a.pnodes[s0 + l];
      pc[j] = a.pn_coff[s0 + l];
    }
    if (a.prev_acc) {
      if constexpr (M == 1) {
        // chained: the shared nodes' rows (mostly two) and start states with
        // the other nodes' states
        uint32_t sid[GNS];
        uint2 rr[GNS];
#pragma unroll
        for (int j = 0; j < GN; ++j) {
          const int l = min(tid + j * PATCH, nl - 1);
          sid[j] = 0;
          rr[j] = uint2{0, 0};
          if (l >= ninner) {
            sid[j] = a.pn_sid[s0 + l];
            rr[j] = a.pn_rows[s0 + l];
          }
        }
        double uo[GNS], row[GNS][2][M + 1], v[GNS];
        int di[GNS];
#pragma unroll
        for (int j = 0; j < GN; ++j) {
          const int l = min(tid + j * PATCH, nl - 1);
          uo[j] = *(l >= ninner ? a.base_in + sid[j] : a.u + pg[j]);
          v[j] = 1.0;
          di[j] = -1;
          if (EARLY || l >= ninner) {
            v[j] = a.vol[pg[j]];
            di[j] = a.dir_index[pg[j]];
          }
#pragma unroll
          for (int t = 0; t < 2; ++t) {
#pragma unroll
            for (int k = 0; k <= M; ++k) row[j][t][k] = 0.0;
            if (rr[j].x + t < rr[j].y)
#pragma unroll
              for (int k = 0; k <= M; ++k) row[j][t][k] = a.prev_acc[static_cast<size_t>(rr[j].x + t) * (M + 1) + k];
          }
        }
#pragma unroll
        for (int j = 0; j < GN; ++j) {
          const int l = tid + j * PATCH;
          if constexpr (EARLY) {
            pv[j] = v[j];
            pdi[j] = di[j];
            psp[j] = l >= ninner ? a.slot_pos[s0 + min(l, nl - 1)] : 0;
          }
          if (l < nl) {
            double un[M] = {uo[j]};
            if (l >= ninner) {
              double acc[M + 1], r[M], d;
#pragma unroll
              for (int k = 0; k <= M; ++k) acc[k] = (0.0 + row[j][0][k]) + row[j][1][k];
              for (uint32_t s = rr[j].x + 2; s < rr[j].y; ++s)
#pragma unroll
                for (int k = 0; k <= M; ++k) acc[k] += a.prev_acc[static_cast<size_t>(s) * (M + 1) + k];
              const double us[M] = {uo[j]};
              node_step<M>(a, pg[j], acc, us, v[j], di[j], r, un, d);
            }
            put_node(l, pg[j], un);
            coff[l] = pc[j];
          }
        }
      } else {
#pragma unroll
        for (int j = 0; j < GN; ++j)
          if (tid + j * PATCH < nl) gather_node(tid + j * PATCH, pg[j]);
        if constexpr (EARLY) load_finish();
      }
    } else {
      double un[GNS][M];
#pragma unroll
      for (int j = 0; j < GN; ++j)
#pragma unroll
        for (int k = 0; k < M; ++k) un[j][k] = a.u[static_cast<size_t>(pg[j]) * M + k];
      if constexpr (EARLY) load_finish();
#pragma unroll
      for (int j = 0; j < GN; ++j) {
        const int l = tid + j * PATCH;
        if (l < nl) {
          put_node(l, pg[j], un[j]);
          coff[l] = pc[j];
        }
      }
    }
  }
  for (int l = tid + GN * PATCH; l < nl; l += PATCH) gather_node(l, a.pnodes[s0 + l]);
  lds_barrier();

  bool bad = false;
  double phi[ND][M];
  double wave = 0.0;
  if constexpr (PREC == 4) {
    // linear sweep: J delta with the cell's FP32 Jacobian (entry-major over
    // the block's cells, so that every load is coalesced), written straight
    // to the (cell, node) pair slots (no divergence slices share the work
    // region here); the node loop stays rolled, one block row per trip
    if (active) {
      constexpr int NDM = ND * M;
      const int NPAIR_ = blockDim.x * ND;
      float dv[NDM];
#pragma unroll
      for (int n = 0; n < ND; ++n)
#pragma unroll
        for (int k = 0; k < M; ++k) dv[n * M + k] = delta_l[(lc[n] & LC_MASK) * M + k];
      const float *__restrict__ jc = a.jlin + (e0 + tid);
      const size_t stride = a.ne;
#pragma unroll 1
      for (int n = 0; n < ND; ++n) {
        const uint16_t l = a.lconn[static_cast<size_t>(n) * a.ne + e0 + tid];
        const int slot = coff[l & LC_MASK] + (l >> LC_BITS);
#pragma unroll
        for (int k = 0; k < M; ++k) {
          const float *__restrict__ row = jc + static_cast<size_t>((n * M + k) * NDM) * stride;
          float y = 0.0f;
#pragma unroll
          for (int j = 0; j < NDM; ++j) y += row[static_cast<size_t>(j) * stride] * dv[j];
          work[k * NPAIR_ + slot] = static_cast<double>(y);
        }
        work[M * NPAIR_ + slot] = 0.0;
      }
    }
  } else if (active) {
    double U[ND][M];
    int row[ND];
#pragma unroll
    for (int n = 0; n < ND; ++n) {
      row[n] = lc[n] & LC_MASK;
#pragma unroll
      for (int k = 0; k < M; ++k) U[n][k] = ul[row[n] * M + k];
    }
    if constexpr (PREC == 5 && M == 1)
      cell_residual<D, NG, ND, NF, NQ, AFFINE, PH, SC, PREC, true>(
          a.tab, X, U, URegs<ND, M>{U}, a.pp, phi, wave, bad, work + tid, PATCH,
          SourceThetaLds<ND, M>{nodal_l, nodal_l + static_cast<size_t>(a.maxl) * M, row});
    else if constexpr (PREC == 5)
      cell_residual<D, NG, ND, NF, NQ, AFFINE, PH, SC, PREC, true>(
          a.tab, X, U, ULds<ND, M>{ul, row}, a.pp, phi, wave, bad, work + tid, PATCH,
          SourceThetaLds<ND, M>{nodal_l, nodal_l + static_cast<size_t>(a.maxl) * M, row});
    else if constexpr (PREC == 3 && M == 1)
      cell_residual<D, NG, ND, NF, NQ, AFFINE, PH, SC, PREC, true>(a.tab, X, U, URegs<ND, M>{U}, a.pp, phi, wave, bad, work + tid,
                                                       PATCH, SourceLds<ND, M>{nodal_l, row});
    else if constexpr (PREC == 3)
      cell_residual<D, NG, ND, NF, NQ, AFFINE, PH, SC, PREC, true>(a.tab, X, U, ULds<ND, M>{ul, row}, a.pp, phi, wave, bad,
                                                       work + tid, PATCH, SourceLds<ND, M>{nodal_l, row});
    else if constexpr (PREC == 2 && M == 1)
      cell_residual<D, NG, ND, NF, NQ, AFFINE, PH, SC, PREC, true>(a.tab, X, U, URegs<ND, M>{U}, a.pp, phi, wave, bad, work + tid,
                                                       PATCH, NodalLds<ND>{nodal_l, row});
    else if constexpr (PREC == 2)
      cell_residual<D, NG, ND, NF, NQ, AFFINE, PH, SC, PREC, true>(a.tab, X, U, ULds<ND, M>{ul, row}, a.pp, phi, wave, bad,
                                                       work + tid, PATCH, NodalLds<ND>{nodal_l, row});
    else if constexpr (M == 1)
      cell_residual<D, NG, ND, NF, NQ, AFFINE, PH, SC, PREC, true>(a.tab, X, U, URegs<ND, M>{U}, a.pp, phi, wave, bad, work + tid,
                                                       PATCH);
    else
      cell_residual<D, NG, ND, NF, NQ, AFFINE, PH, SC, PREC, true>(a.tab, X, U, ULds<ND, M>{ul, row}, a.pp, phi, wave, bad,
                                                       work + tid, PATCH);
  }
  if constexpr (GN > 0 && !EARLY) load_finish();
  const int npair = ecount * ND;
  double sq[M + 1];
#pragma unroll
  for (int k = 0; k <= M; ++k) sq[k] = 0.0;
  // components [c0, c0 + n) of the cell's residuals and wave speed to its pairs
  auto put_pairs = [&](const int c0, const int n) {
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      const int slot = coff[lc[i] & LC_MASK] + (lc[i] >> LC_BITS);
#pragma unroll
      for (int k = 0; k <= M; ++k)
        if (k >= c0 && k < c0 + n) work[(k - c0) * NPAIR + slot] = (k < M) ? phi[i][k < M ? k : 0] : wave;
    }
  };
  // their sums over the pairs of node l
  auto sum_pairs = [&](const int l, const int c0, const int n, double (&acc)[M + 1]) {
    const int b = coff[l];
    const int e = (l + 1 < nl) ? static_cast<int>(coff[l + 1]) : npair;
#pragma unroll
    for (int k = 0; k <= M; ++k)
      if (k >= c0 && k < c0 + n) acc[k] = 0.0;
    for (int i = b; i < e; ++i)
#pragma unroll
      for (int k = 0; k <= M; ++k)
        if (k >= c0 && k < c0 + n) acc[k] += work[(k - c0) * NPAIR + i];
  };
  // node l of the patch from its sums; pre: its node id, slot, volume and
  // Dirichlet index were loaded ahead (pgv, pspv, pvv, pdiv)
  auto finish_l = [&](const int l, const double (&acc)[M + 1], const bool pre, const uint32_t pgv, const uint32_t pspv,
                      const double pvv, const int pdiv) {
    if (l < ninner) {
      const uint32_t g = pre ? pgv : a.pnodes[s0 + l];
      finish_node<M>(a, g, acc, ul + l * M, pre ? pvv : a.vol[g], pre ? pdiv : a.dir_index[g], sq);
    } else {
      const uint32_t sp = pre ? pspv : a.slot_pos[s0 + l];
      double *slot = a.slot_acc + static_cast<size_t>(sp) * (M + 1);
#pragma unroll
      for (int k = 0; k <= M; ++k) slot[k] = acc[k];
      if (a.prev_acc || a.base_out) {
        // the holder of the node's first row stores its start state
        const uint32_t i = a.pn_sid[s0 + l];
        if (sp == a.pn_rows[s0 + l].x) {
#pragma unroll
          for (int k = 0; k < M; ++k) {
            const double v = ul[l * M + k];
            if (a.prev_acc) a.u[static_cast<size_t>(a.pnodes[s0 + l]) * M + k] = v;
            if (a.base_out) a.base_out[static_cast<size_t>(i) * M + k] = v;
          }
        }
      }
    }
  };
  if constexpr (PW::phased) {
    // a few components at a time, the sums of a thread's NPT nodes in
    // registers; patches of more nodes take another round of all phases
    constexpr int NPT = 4;
    for (int l0 = 0; l0 < nl; l0 += NPT * PATCH) {
      double acc[NPT][M + 1];
#pragma unroll
      for (int c0 = 0; c0 <= M; c0 += PW::comps) {
        lds_barrier();
        if (active) put_pairs(c0, PW::comps);
        lds_barrier();
#pragma unroll
        for (int j = 0; j < NPT; ++j) {
          const int l = l0 + tid + j * PATCH;
          if (l < nl) sum_pairs(l, c0, PW::comps, acc[j]);
        }
      }
#pragma unroll
      for (int j = 0; j < NPT; ++j) {
        const int l = l0 + tid + j * PATCH;
        if (l < nl) {
          if (j < GN && l0 == 0)
            finish_l(l, acc[j], true, pg[j % GNS], psp[j % GNS], pv[j % GNS], pdi[j % GNS]);
          else
            finish_l(l, acc[j], false, 0u, 0u, 0.0, 0);
        }
      }
    }
  } else {
    lds_barrier();  // the work region changes from the cells' columns to pair sums
    if (active && PREC != 4) put_pairs(0, M + 1);
    lds_barrier();
    double acc[M + 1];
    if constexpr (GN > 0) {
#pragma unroll
      for (int j = 0; j < GN; ++j) {
        const int l = tid + j * PATCH;
        if (l < nl) {
          sum_pairs(l, 0, M + 1, acc);
          finish_l(l, acc, true, pg[j], psp[j], pv[j], pdi[j]);
        }
      }
    }
    for (int l = tid + GN * PATCH; l < nl; l += PATCH) {
      sum_pairs(l, 0, M + 1, acc);
      finish_l(l, acc, false, 0u, 0u, 0.0, 0);
    }
  }
  if (bad) atomicOr(a.status, 1);
  if (a.update == 1 && a.outputs) block_sum_store<M>(sq, work, a.norm_partial + static_cast<size_t>(p) * (M + 1));
}

template <int D, int NG, int ND, int NF, int NQ, bool AFFINE, int PH, int SC, int PREC>
__global__ __launch_bounds__((PatchSize<PhysTraits<PH>::M, ND>::value),
                             (PatchMinWaves<PhysTraits<PH>::M, ND, NQ, AFFINE, SC, PREC>::value)) void rd_patch_kernel(PatchArgs a)
{
  extern __shared__ double lds[];
  const uint32_t pl = xcd_block_index();
  if (pl >= a.np) return;
  patch_body<D, NG, ND, NF, NQ, AFFINE, PH, SC, PREC>(a, pl, lds);
}

// Patches of several blocks (of several methods) of one element type /
// physics / scheme in one launch: workgroup g runs patch g - first[i] of
// args[i], first[i] <= g < first[i + 1]. The dynamic LDS is the largest of
// the entries'.
template <int D, int NG, int ND, int NF, int NQ, bool AFFINE, int PH, int SC, int PREC>
__global__ __launch_bounds__((PatchSize<PhysTraits<PH>::M, ND>::value),
                             (PatchMinWaves<PhysTraits<PH>::M, ND, NQ, AFFINE, SC, PREC>::value)) void
rd_patch_batch_kernel(const PatchArgs *__restrict__ args, const uint32_t *__restrict__ first, int count)
{
  extern __shared__ double lds[];
  const uint32_t g = xcd_block_index();
  if (g >= first[count]) return;
  int i = 0;
  while (i + 1 < count && first[i + 1] <= g) ++i;
  patch_body<D, NG, ND, NF, NQ, AFFINE, PH, SC, PREC, true>(args[i], g - first[i], lds);
}

struct FixupArgs
{
  const uint32_t *__restrict__ nodes;     // [nb] shared nodes
  const uint32_t *__restrict__ slot_off;  // [nb + 1]
  const double *__restrict__ slot_acc;    // rows of node i: [slot_off[i], slot_off[i + 1])
  PatchArgs pa;                           // node outputs as in the patch kernel
  uint32_t nb;
  double *__restrict__ norm_partial;      // [gridDim.x][M + 1]
};

// Sums of the shared nodes of one method: local block lb of nblk blocks
// (grid-stride over the nodes), norm partial of the block at lb.
template <int M>
__device__ __forceinline__ void fixup_body(const FixupArgs &f, uint32_t lb, uint32_t nblk, double *red)
{
  double sq[M + 1];
#pragma unroll
  for (int k = 0; k <= M; ++k) sq[k] = 0.0;
  for (uint32_t i = lb * blockDim.x + threadIdx.x; i < f.nb; i += nblk * blockDim.x) {
    double acc[M + 1];
    sum_rows<M>(f.slot_acc, f.slot_off[i], f.slot_off[i + 1], acc);
    const uint32_t g = f.nodes[i];
    double u_old[M];
#pragma unroll
    for (int k = 0; k < M; ++k) u_old[k] = f.pa.u[static_cast<size_t>(g) * M + k];
    finish_node<M>(f.pa, g, acc, u_old, f.pa.vol[g], f.pa.dir_index[g], sq);
  }
  if (f.pa.update == 1 && f.pa.outputs) block_sum_store<M>(sq, red, f.norm_partial + static_cast<size_t>(lb) * (M + 1));
}

template <int M>
__global__ __launch_bounds__(256) void patch_fixup_kernel(FixupArgs f)
{
  __shared__ double red[256 * (M + 1)];
  fixup_body<M>(f, blockIdx.x, gridDim.x, red);
}

// Shared-node sums of several methods in one launch: block g serves
// args[i] as its block g - first[i] of first[i + 1] - first[i].
template <int M>
__global__ __launch_bounds__(256) void patch_fixup_batch_kernel(const FixupArgs *__restrict__ args,
                                                                const uint32_t *__restrict__ first, int count)
{
  __shared__ double red[256 * (M + 1)];
  const uint32_t g = blockIdx.x;
  if (g >= first[count]) return;
  int i = 0;
  while (i + 1 < count && first[i + 1] <= g) ++i;
  fixup_body<M>(args[i], g - first[i], first[i + 1] - first[i], red);
}

}  // namespace pdrd

// Registry of the compiled cell-kernel instantiations.
#pragma once

#include <hip/hip_runtime.h>

#include "rd_cell.hpp"
#include "rd_jacobian.hpp"
#include "rd_weakbc.hpp"

namespace pdrd {

using CellLauncher = hipError_t (*)(const CellArgs &, unsigned grid, unsigned block, hipStream_t);
using PatchLauncher = hipError_t (*)(const PatchArgs &, unsigned grid, int cells, hipStream_t);
using PatchBatchLauncher = hipError_t (*)(const PatchArgs *args, const uint32_t *first, int count, unsigned grid,
                                          int cells, size_t lds_bytes, hipStream_t);
// quad, tri: the two blocks; weak: the facets of the method's weak boundary
// conditions (groups of 64; weak_groups 0: none)
using PatchMixedLauncher = hipError_t (*)(const PatchArgs &quad, const PatchArgs &tri, const WeakRange &weak,
                                          unsigned weak_groups, int cells, hipStream_t);
// The same over `count` methods: args [2][count] (quadrilaterals, triangles) and
// the prefix sums of their patches first [2][count + 1], grids nq and nt.
using PatchMixedBatchLauncher = hipError_t (*)(const PatchArgs *args, const uint32_t *first, int count, unsigned nq,
                                               unsigned nt, const WeakRange &weak, unsigned weak_groups, int cells,
                                               size_t lds, hipStream_t);
using JacobianLauncher = hipError_t (*)(const JacArgs &, unsigned grid, hipStream_t);

struct CellKey
{
  int shape, sol_order, nq, physics, scheme;
};

// Everything the host needs to launch one instantiation.
struct KernelSet
{
  CellLauncher cell = nullptr;    // element per thread, global scatter
  PatchLauncher patch = nullptr;  // patch assembly
  PatchBatchLauncher patch_batch = nullptr;  // patch assembly of several blocks / methods
  // the same with a nodal input (LDA / B) or a source field
  PatchBatchLauncher patch_nodal_batch = nullptr;
  PatchBatchLauncher patch_src_batch = nullptr;
  PatchLauncher patch_lin = nullptr;  // linear sweep of the mixed-precision form: J delta per cell
  // quadrilaterals of the 2D Euler equations: with the triangles of the same
  // mesh and the weak facets in one launch
  PatchMixedLauncher patch_mixed = nullptr;
  PatchMixedBatchLauncher patch_mixed_batch = nullptr;
  // with the nodal input of the scheme (LDA: artificial viscosity, B:
  // external blending coefficient); null for N and PSI, which take none
  CellLauncher cell_nodal = nullptr;
  PatchLauncher patch_nodal = nullptr;
  // FP64 patch assembly with a nodal source field (reaction residuals), and
  // for the B scheme with an external blending coefficient beside it
  PatchLauncher patch_src = nullptr;
  PatchLauncher patch_src_theta = nullptr;
  PatchBatchLauncher patch_src_theta_batch = nullptr;
  // element residuals and Jacobians of the implicit form (null for PSI)
  JacobianLauncher jacobian = nullptr;
  int patch_size = 0;             // largest (default) cells per patch workgroup
  size_t (*patch_lds_bytes)(int maxl, int cells) = nullptr;
  size_t (*patch_src_lds_bytes)(int maxl, int cells) = nullptr;
  size_t (*patch_nodal_lds_bytes)(int maxl, int cells) = nullptr;
  size_t (*patch_src_theta_lds_bytes)(int maxl, int cells) = nullptr;
  size_t (*patch_lin_lds_bytes)(int maxl, int cells) = nullptr;
  explicit operator bool() const { return cell != nullptr; }
};

// Element types built: (shape, P, dim, ng, nd, nf, quadrature points, affine)
//   triangle P1 / P4 rule (6 points), P2 / P4 rule, P3 / P6 rule (12 points),
//   quadrilateral Q1 and Q2 / P4 rule (8 points), tetrahedron P1 / P2 rule
//   (4 points), tetrahedron P2 / P2 rule and P4 rule (11 points)
#define PDRD_ELEMENT_TYPES(X)                      \
  X(0, 1, 2, 3, 3, 6, 6, true)                     \
  X(0, 2, 2, 3, 6, 10, 6, true)                    \
  X(0, 3, 2, 3, 10, 15, 12, true)                  \
  X(1, 1, 2, 4, 4, 9, 8, false)                    \
  X(1, 2, 2, 4, 9, 16, 8, false)                   \
  X(2, 1, 3, 4, 4, 10, 4, true)                    \
  X(2, 2, 3, 4, 10, 20, 4, true)                   \
  X(2, 2, 3, 4, 10, 20, 11, true)

template <int D, int NG, int ND, int NF, int NQ, bool AFF, int PH, int SC, int PREC = 0>
hipError_t launch_cell(const CellArgs &a, unsigned grid, unsigned block, hipStream_t s)
{
  const size_t column = static_cast<size_t>(CellColumn<D, ND, NQ, AFF, PH>::value) * block * sizeof(double);
  const size_t table = a.atomic ? NodeTable<ND, PhysTraits<PH>::M>::bytes(block) : 0;
  const size_t lds = column > table ? column : table;
  hipLaunchKernelGGL((rd_cell_kernel<D, NG, ND, NF, NQ, AFF, PH, SC, PREC>), dim3(grid), dim3(block), lds, s, a);
  return hipGetLastError();
}

template <int D, int NG, int ND, int NF, int NQ, bool AFF, int PH, int SC, int PREC>
hipError_t launch_patch(const PatchArgs &a, unsigned grid, int cells, hipStream_t s)
{
  using PW = PatchWork<D, ND, NQ, AFF, PH, SC, PREC>;
  const size_t lds = patch_lds_doubles<PW, PREC>(a.maxl, cells) * sizeof(double);
  hipLaunchKernelGGL((rd_patch_kernel<D, NG, ND, NF, NQ, AFF, PH, SC, PREC>), dim3(grid), dim3(cells), lds, s, a);
  return hipGetLastError();
}

// A sweep of a mixed mesh of quadrilaterals and triangles of order P of the 2D
// Euler equations in one launch: workgroups [0, quad.np) take the
// quadrilaterals' patches, the next tri.np the triangles', the rest the weak
// facets (64 to a wave), all of which only read the state of shared nodes. One
// after the other, each kind fills the chip for a round or two and then drains
// it: 65 536 + 131 072 first-order cells LDA 30.6 + 16.8 us, and 5 us of facets,
// 39 us together. Of second order only small meshes go together, whose waves
// have a SIMD to themselves anyway (see the patch sizes in pdrd_initialize): in
// one kernel the triangles run at the quadrilaterals' 1 wave per SIMD.
template <int P, int SC>
struct MixedPatch
{
  static constexpr int waves = P == 1 ? 2 : 1;
  static constexpr int NDQ = (P + 1) * (P + 1), NFQ = (P + 2) * (P + 2), NDT = (P + 1) * (P + 2) / 2,
                       NFT = (P + 2) * (P + 3) / 2;
  static __device__ __forceinline__ void quad(const PatchArgs &a, uint32_t pl, double *lds)
  {
    patch_body<2, 4, NDQ, NFQ, 8, false, PH_EULER2D, SC, 0>(a, pl, lds);
  }
  static __device__ __forceinline__ void tri(const PatchArgs &a, uint32_t pl, double *lds)
  {
    patch_body<2, 3, NDT, NFT, 6, true, PH_EULER2D, SC, 0>(a, pl, lds);
  }
  // facets of workgroup g (counted behind the patches) of the launch
  static __device__ __forceinline__ void facets(const WeakRange &weak, uint32_t weak_groups, uint32_t g)
  {
    const uint32_t w = g * (blockDim.x / WEAK_THREADS) + threadIdx.x / WEAK_THREADS;
    if (w < weak_groups) weak_group<PH_EULER2D, P + 1>(weak, w, threadIdx.x % WEAK_THREADS);
  }
  static unsigned facet_blocks(unsigned weak_groups, int cells)
  {
    const unsigned n = cells / WEAK_THREADS;
    return (weak_groups + n - 1) / n;
  }
};

template <int P, int SC>
__global__ __launch_bounds__(128, (MixedPatch<P, SC>::waves)) void rd_patch_mixed_kernel(PatchArgs quad, PatchArgs tri,
                                                                                         WeakRange weak,
                                                                                         uint32_t weak_groups)
{
  extern __shared__ double lds[];
  const uint32_t g = blockIdx.x;
  if (g < quad.np)
    MixedPatch<P, SC>::quad(quad, xcd_block_index(g, quad.np), lds);
  else if (g < quad.np + tri.np)
    MixedPatch<P, SC>::tri(tri, xcd_block_index(g - quad.np, tri.np), lds);
  else
    MixedPatch<P, SC>::facets(weak, weak_groups, g - quad.np - tri.np);
}

template <int P, int SC>
__global__ __launch_bounds__(128, (MixedPatch<P, SC>::waves)) void rd_patch_mixed_batch_kernel(
    const PatchArgs *__restrict__ args, const uint32_t *__restrict__ first, int count, uint32_t nq, uint32_t nt,
    WeakRange weak, uint32_t weak_groups)
{
  extern __shared__ double lds[];
  uint32_t g = blockIdx.x;
  if (g >= nq + nt) {
    MixedPatch<P, SC>::facets(weak, weak_groups, g - nq - nt);
    return;
  }
  const bool is_tri = g >= nq;
  g = is_tri ? xcd_block_index(g - nq, nt) : xcd_block_index(g, nq);
  if (is_tri) {
    first += count + 1;
    args += count;
  }
  int i = 0;
  while (i + 1 < count && first[i + 1] <= g) ++i;
  if (is_tri)
    MixedPatch<P, SC>::tri(args[i], g - first[i], lds);
  else
    MixedPatch<P, SC>::quad(args[i], g - first[i], lds);
}

template <int P, int SC>
hipError_t launch_patch_mixed_batch(const PatchArgs *args, const uint32_t *first, int count, unsigned nq, unsigned nt,
                                    const WeakRange &weak, unsigned weak_groups, int cells, size_t lds, hipStream_t s)
{
  const unsigned grid = nq + nt + MixedPatch<P, SC>::facet_blocks(weak_groups, cells);
  hipLaunchKernelGGL((rd_patch_mixed_batch_kernel<P, SC>), dim3(grid), dim3(cells), lds, s, args, first, count, nq, nt,
                     weak, weak_groups);
  return hipGetLastError();
}

template <int P, int SC>
hipError_t launch_patch_mixed(const PatchArgs &quad, const PatchArgs &tri, const WeakRange &weak, unsigned weak_groups,
                              int cells, hipStream_t s)
{
  using MP = MixedPatch<P, SC>;
  const size_t lq = patch_lds_doubles<PatchWork<2, MP::NDQ, 8, false, PH_EULER2D, SC, 0>, 0>(quad.maxl, cells);
  const size_t lt = patch_lds_doubles<PatchWork<2, MP::NDT, 6, true, PH_EULER2D, SC, 0>, 0>(tri.maxl, cells);
  const unsigned grid = quad.np + tri.np + MP::facet_blocks(weak_groups, cells);
  hipLaunchKernelGGL((rd_patch_mixed_kernel<P, SC>), dim3(grid), dim3(cells), (lq > lt ? lq : lt) * sizeof(double), s,
                     quad, tri, weak, weak_groups);
  return hipGetLastError();
}

template <int D, int NG, int ND, int NF, int NQ, bool AFF, int PH, int SC, int PREC>
hipError_t launch_patch_batch(const PatchArgs *args, const uint32_t *first, int count, unsigned grid, int cells,
                              size_t lds, hipStream_t s)
{
  hipLaunchKernelGGL((rd_patch_batch_kernel<D, NG, ND, NF, NQ, AFF, PH, SC, PREC>), dim3(grid), dim3(cells), lds, s,
                     args, first, count);
  return hipGetLastError();
}

template <int D, int NG, int ND, int NF, int NQ, bool AFF, int PH, int SC>
hipError_t launch_jacobian(const JacArgs &a, unsigned grid, hipStream_t s)
{
  if constexpr (PhysTraits<PH>::M > 1) {
    // the Euler cells: LPC lanes per cell, one wave per workgroup, a slab of
    // QpRows rows (grid from the cell count: `grid` counts workgroups of 64
    // cells)
    constexpr int CPB = 64 / QpLanes<NQ>::value;
    constexpr size_t lds = static_cast<size_t>(QP_XS) * QpRows<PhysTraits<PH>::M, ND>::value * sizeof(double);
    (void)grid;
    hipLaunchKernelGGL((rd_jacobian_qp_kernel<D, NG, ND, NF, NQ, AFF, PH, SC>), dim3((a.ne + CPB - 1) / CPB), dim3(64),
                       lds, s, a);
  }
  else
    hipLaunchKernelGGL((rd_jacobian_kernel<D, NG, ND, NF, NQ, AFF, PH, SC>), dim3(grid), dim3(64), 0, s, a);
  return hipGetLastError();
}

template <int D, int ND, int NQ, bool AFF, int PH, int SC, int PREC>
size_t patch_lds_bytes(int maxl, int cells)
{
  return patch_lds_doubles<PatchWork<D, ND, NQ, AFF, PH, SC, PREC>, PREC>(maxl, cells) * sizeof(double);
}

template <int D, int NG, int ND, int NF, int NQ, bool AFF, int PH, int SC>
KernelSet kernel_set()
{
  KernelSet k;
  k.cell = &launch_cell<D, NG, ND, NF, NQ, AFF, PH, SC>;
  k.patch = &launch_patch<D, NG, ND, NF, NQ, AFF, PH, SC, 0>;
  k.patch_batch = &launch_patch_batch<D, NG, ND, NF, NQ, AFF, PH, SC, 0>;
  // the linear sweep depends on the block size only: one instantiation per
  // element type and equation count (that of the advection physics for the
  // scalar ones)
  if constexpr ((PH == PH_ADVECTION2D || PH == PH_EULER2D || PH == PH_EULER3D) && SC == SC_LDA) {
    k.patch_lin = &launch_patch<D, NG, ND, NF, NQ, AFF, PH, SC, 4>;
    k.patch_lin_lds_bytes = &patch_lds_bytes<D, ND, NQ, AFF, PH, SC, 4>;
  }
  if constexpr (PH == PH_EULER2D && !AFF && NQ == 8) {
    constexpr int P = ND == 4 ? 1 : 2;
    k.patch_mixed = &launch_patch_mixed<P, SC>;
    k.patch_mixed_batch = &launch_patch_mixed_batch<P, SC>;
  }
  if constexpr (SC == SC_LDA || SC == SC_B) {
    k.cell_nodal = &launch_cell<D, NG, ND, NF, NQ, AFF, PH, SC, 2>;
    k.patch_nodal = &launch_patch<D, NG, ND, NF, NQ, AFF, PH, SC, 2>;
    k.patch_nodal_batch = &launch_patch_batch<D, NG, ND, NF, NQ, AFF, PH, SC, 2>;
    k.patch_nodal_lds_bytes = &patch_lds_bytes<D, ND, NQ, AFF, PH, SC, 2>;
  }
  k.patch_src = &launch_patch<D, NG, ND, NF, NQ, AFF, PH, SC, 3>;
  k.patch_src_batch = &launch_patch_batch<D, NG, ND, NF, NQ, AFF, PH, SC, 3>;
  if constexpr (SC == SC_B) {
    k.patch_src_theta = &launch_patch<D, NG, ND, NF, NQ, AFF, PH, SC, 5>;
    k.patch_src_theta_batch = &launch_patch_batch<D, NG, ND, NF, NQ, AFF, PH, SC, 5>;
    k.patch_src_theta_lds_bytes = &patch_lds_bytes<D, ND, NQ, AFF, PH, SC, 5>;
  }
  if constexpr (SC != SC_PSI && SC != SC_BPSI) k.jacobian = &launch_jacobian<D, NG, ND, NF, NQ, AFF, PH, SC>;
  k.patch_size = PatchSize<PhysTraits<PH>::M, ND>::value;
  k.patch_lds_bytes = &patch_lds_bytes<D, ND, NQ, AFF, PH, SC, 0>;
  k.patch_src_lds_bytes = &patch_lds_bytes<D, ND, NQ, AFF, PH, SC, 3>;
  return k;
}

// Lookup functions, one per compilation unit of instantiations.
KernelSet find_cell_scalar_adv(const CellKey &k);
KernelSet find_cell_scalar_burgers(const CellKey &k);
KernelSet find_cell_scalar_rot(const CellKey &k);
KernelSet find_cell_euler2d(const CellKey &k);
KernelSet find_cell_euler3d(const CellKey &k);

inline KernelSet find_cell(const CellKey &k)
{
  switch (k.physics) {
    case PH_ADVECTION2D: return find_cell_scalar_adv(k);
    case PH_BURGERS2D: return find_cell_scalar_burgers(k);
    case PH_ROTATION2D: return find_cell_scalar_rot(k);
    case PH_EULER2D: return find_cell_euler2d(k);
    case PH_EULER3D: return find_cell_euler3d(k);
  }
  return KernelSet{};
}

template <int SH, int P, int D, int NG, int ND, int NF, int NQ, bool AFF, int PH>
KernelSet pick_cell(const CellKey &k)
{
  if constexpr (D != PhysTraits<PH>::DIM) {
    (void)k;
    return KernelSet{};
  } else {
    if (k.shape == SH && k.sol_order == P && k.nq == NQ) {
      switch (k.scheme) {
        case SC_LDA: return kernel_set<D, NG, ND, NF, NQ, AFF, PH, SC_LDA>();
        case SC_N: return kernel_set<D, NG, ND, NF, NQ, AFF, PH, SC_N>();
        case SC_B: return kernel_set<D, NG, ND, NF, NQ, AFF, PH, SC_B>();
        case SC_PSI: return kernel_set<D, NG, ND, NF, NQ, AFF, PH, SC_PSI>();
        case SC_BPSI: return kernel_set<D, NG, ND, NF, NQ, AFF, PH, SC_BPSI>();
      }
    }
    return KernelSet{};
  }
}

}  // namespace pdrd

// Body of a lookup function for one physics (PHYS_): every element type of
// matching dimension and every scheme.
#define PDRD_CELL_CASE(SH, P, D, NG, ND, NF, NQ, AFF) \
  if (KernelSet f = pick_cell<SH, P, D, NG, ND, NF, NQ, AFF, PHYS_>(k)) return f;

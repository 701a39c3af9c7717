"""Pair sums of the Euler P2 cells in phases: patches with more nodes than one
round of the sums holds (4 per thread). Every cell of a mesh gets its own copy of
its nodes and vertices, so that a patch of 64 cells has 384 (triangles) or 640
(tetrahedra) nodes: two or three rounds, the last one ragged, against one round
on the connected mesh. Both against the oracle, 1e-12 normwise as in the parity
tests; the exploded mesh's cells do not share nodes, so no sums are reordered."""
import numpy as np
import pytest

from pdekit_amd import _lib as L
from pdekit_amd.mesh import CellBlock, Mesh
from pdekit_amd.rdm import PGRDMethodExplicit
from tests.helpers import CASES, euler_state, oracle_problem, quad_orders, rel_err

pytestmark = pytest.mark.gpu


def exploded(mesh):
    coords, node_coords, blocks, nv, nn = [], [], [], 0, 0
    for b in mesh.blocks:
        ne, ng = b.geo_conn.shape
        nd = b.sol_conn.shape[1]
        coords.append(mesh.coords[b.geo_conn].reshape(-1, mesh.dim))
        node_coords.append(mesh.node_coords[b.sol_conn].reshape(-1, mesh.dim))
        blocks.append(CellBlock(b.shape, b.cells, np.arange(nv, nv + ne * ng, dtype=np.uint32).reshape(ne, ng),
                                np.arange(nn, nn + ne * nd, dtype=np.uint32).reshape(ne, nd)))
        nv += ne * ng
        nn += ne * nd
    return Mesh(mesh.dim, np.concatenate(coords), mesh.cell_shape, mesh.order, nn, np.concatenate(node_coords), blocks)


@pytest.mark.parametrize("scheme", [L.LDA, L.N, L.B, L.PSI, L.BPSI])
@pytest.mark.parametrize("cells", [64, 128])
@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("case", ["euler2d_p2", "euler2d_q2_mixed", "euler3d_p2"])
def test_phased_pair_sums(case, split, cells, scheme):
    build, physics, params, _ = CASES[case]
    mesh = exploded(build()) if split else build()
    u = euler_state(mesh, dim=mesh.dim)
    m = PGRDMethodExplicit(physics, scheme, params=params).configure_mesh_data(mesh)
    m.initialize_work_data(quad_order=quad_orders(mesh), patch_cells=cells)
    m.set_vec_function("solution", u)
    m.assemble_rhs()
    res, ws = m.vec_function("residuals"), m.vec_function("wave_speed")
    m.assemble_rhs()
    assert np.array_equal(res, m.vec_function("residuals"))
    # the node finish of an iteration takes the same sums
    m.iterate(0.5, 1)
    assert np.array_equal(res, m.vec_function("residuals"))
    v, dt = m.vec_function("dual_volume"), m.vec_function("time_step")
    assert rel_err(m.vec_function("solution"), u - dt[:, None] * res) <= 1e-15
    assert rel_err(dt, 0.5 * v / ws) <= 1e-15
    m.destroy()
    ref, ref_ws, rc = oracle_problem(mesh, physics, scheme, params).assemble_rhs(u)
    assert rc == 0
    assert rel_err(res, ref) <= 1e-12
    assert rel_err(ws, ref_ws) <= 1e-12

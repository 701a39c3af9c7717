"""The atomic assembly's table of nodes per workgroup: cells in mesh order (most
nodes of a workgroup share entries) and in a random one (more nodes than entries,
so that most parts go to global memory directly), every workgroup size, element
types from the smallest to the largest table, a ragged last workgroup and single
cells. Against the oracle, 1e-12 normwise as the parity tests: atomics only
reorder a node's few additions."""
import dataclasses

import numpy as np
import pytest

from pdekit_amd import _lib as L
from pdekit_amd.mesh import CellBlock, box_tetra, rectangle
from pdekit_amd.rdm import PGRDMethodExplicit
from tests.helpers import advection_state, burgers_state, euler_state, oracle_problem, quad_orders, rel_err

pytestmark = pytest.mark.gpu

CASES = {
    "one_cell_pair": (lambda: rectangle(1, 1, split=2, order=1), L.ADVECTION2D, (0.8, 0.6), advection_state),
    "p1": (lambda: rectangle(61, 47, split=2, order=1), L.ADVECTION2D, (0.8, 0.6), advection_state),
    "p2": (lambda: rectangle(33, 41, split=4, order=2, jitter=0.1, seed=2), L.BURGERS2D, (), burgers_state),
    "p3": (lambda: rectangle(29, 31, split=2, order=3), L.ADVECTION2D, (0.8, 0.6), advection_state),
    "euler_q2p2": (lambda: rectangle(30, 22, extent=(-0.5, 1.5, 0.0, 1.0), split=2, quad_rows=11, order=2,
                                     bump=(1.0, 0.1, 25.0, 0.5)), L.EULER2D, (1.4, 287.05), euler_state),
    "tetra_p2": (lambda: box_tetra(6, 5, 5, extent=(1.0, 1.0, 0.5), order=2, jitter=0.1, seed=4), L.EULER3D,
                 (1.4, 287.05), lambda m: euler_state(m, dim=3)),
}


@pytest.mark.parametrize("shuffle", [False, True])
@pytest.mark.parametrize("block", [64, 192, 256])
@pytest.mark.parametrize("name", list(CASES))
def test_atomic_table(name, block, shuffle):
    build, physics, params, state = CASES[name]
    mesh = build()
    u = state(mesh)
    ref, ref_ws, rc = oracle_problem(mesh, physics, L.N, params).assemble_rhs(u)
    assert rc == 0
    if shuffle:
        rng = np.random.default_rng(1)
        blocks = []
        for b in mesh.blocks:
            o = rng.permutation(b.cells.size)
            blocks.append(CellBlock(b.shape, b.cells[o], np.ascontiguousarray(b.geo_conn[o]),
                                    np.ascontiguousarray(b.sol_conn[o])))
        mesh = dataclasses.replace(mesh, blocks=blocks)
    m = PGRDMethodExplicit(physics, L.N, params=params or None).configure_mesh_data(mesh)
    m.initialize_work_data(quad_order=quad_orders(mesh), scatter=0)
    m.set_option(L.OPT_BLOCK, block)
    m.set_vec_function("solution", u)
    for _ in range(2):  # (the accumulators are left clear)
        m.assemble_rhs()
        assert rel_err(m.vec_function("residuals"), ref) <= 1e-12
        assert rel_err(m.vec_function("wave_speed"), ref_ws) <= 1e-12
    m.destroy()

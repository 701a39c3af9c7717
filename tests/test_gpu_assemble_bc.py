"""Strong Dirichlet values written by the assembly's node finish, and the norm of
one workgroup, on both sides of its largest node count: boundary nodes of one
patch and of several, with and without a time step.

The values are copied, so they must be equal. The norm sums squares only, at most
a few hundred one after the other: 1e-13 (300 x 1.1e-16, half of it in the root)."""
import numpy as np
import pytest

from pdekit_amd import _lib as L
from pdekit_amd.mesh import unit_quad_triag
from pdekit_amd.rdm import PGRDMethodExplicit
from tests.helpers import advection_state, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("step", [False, True])
@pytest.mark.parametrize("n", [4, 64, 65])
def test_assembly_applies_boundary_values(n, step):
    mesh = unit_quad_triag(n)
    nodes = np.unique(np.concatenate([mesh.boundaries["Edge0"], mesh.boundaries["Edge1"]]))
    values = np.linspace(2.0, 3.0, len(nodes)).reshape(-1, 1)
    got = {}
    for scatter in (2, 1):
        m = PGRDMethodExplicit(L.ADVECTION2D, L.N, params=(0.8, 0.6)).configure_mesh_data(mesh)
        m.initialize_work_data(quad_order={b.shape: 4 for b in mesh.blocks}, scatter=scatter)
        m.set_vec_function("solution", advection_state(mesh))
        m.add_boundary_condition("StrongDirichlet", "in", nodes, values)
        m.assemble_lhs_and_rhs(0.4) if step else m.assemble_rhs()
        u, res = m.vec_function("solution"), m.vec_function("residuals")
        assert np.array_equal(u[nodes], values)
        inner = np.setdiff1d(np.arange(mesh.nb_nodes), nodes)
        assert np.array_equal(u[inner], advection_state(mesh)[inner])
        r = np.delete(res, nodes, axis=0)
        assert rel_err(m.residual_norm_L2(True), np.sqrt((r ** 2).mean(0))) <= 1e-13
        got[scatter] = res
        m.destroy()
    assert rel_err(got[2], got[1]) <= 1e-12

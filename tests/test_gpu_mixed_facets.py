"""Joint launches of a mixed mesh with weak facets, in every form the facets take: one
or two groups of 64 facets a workgroup (64 and 128 cells a patch), an odd and an even
number of groups (the last workgroup then half empty), every scheme, alone and in a
batch. Against chained sweeps, whose facets have a launch of their own: the same
bits; the first-order residuals against the oracle, 1e-12 normwise as in the weak
boundary tests."""
import numpy as np
import pytest

from pdekit_amd import _lib as L
from pdekit_amd.mesh import rectangle
from pdekit_amd.rdm import Batch, PGRDMethodExplicit
from tests.helpers import add_oracle_weak, euler_state, oracle_problem, rel_err

pytestmark = pytest.mark.gpu

PARAMS = (1.4, 287.05)


def _method(mesh, u, scheme, cells, half, chain):
    top = mesh.boundaries["ymax"]
    m = PGRDMethodExplicit(L.EULER2D, scheme, params=PARAMS).configure_mesh_data(mesh)
    m.initialize_work_data(quad_order=4, patch_cells=cells)
    if half:
        m.add_boundary_condition("WeakWall", "half", _half(mesh))
    m.add_boundary_condition("WeakFarfield", "top", top, values=u[0])
    m.set_vec_function("solution", u)
    m.set_option(L.OPT_CHAIN, chain)
    return m


def _half(mesh):
    top = mesh.boundaries["ymax"]
    return top[mesh.node_coords[top, 0] <= mesh.node_coords[top, 0].mean()]


# facets of the two conditions: 18 + 37 (two groups), 50 + 100 (three)
@pytest.mark.parametrize("nx", [37, 100])
@pytest.mark.parametrize("scheme", [L.LDA, L.N, L.B, L.PSI, L.BPSI])
@pytest.mark.parametrize("order,cells", [(1, 64), (1, 128), (2, None)])
def test_joint_launch(order, cells, scheme, nx):
    mesh = rectangle(nx, 12, extent=(-0.5, 1.5, 0.0, 1.0), split=2, quad_rows=5, order=order, bump=(1.0, 0.1, 25.0, 0.5))
    u = euler_state(mesh)
    one, chained = (_method(mesh, u, scheme, cells, True, c) for c in (0, 1))
    # in a batch with a method of one condition less (groups of both: an odd number)
    few, few_chained = (_method(mesh, u, scheme, cells, False, c) for c in (0, 1))
    batched, few_batched = _method(mesh, u, scheme, cells, True, 0), _method(mesh, u, scheme, cells, False, 0)
    if order == 1:
        one.assemble_rhs()
        P = oracle_problem(mesh, L.EULER2D, scheme, PARAMS)
        add_oracle_weak(P, mesh, "WeakWall", _half(mesh))
        add_oracle_weak(P, mesh, "WeakFarfield", mesh.boundaries["ymax"], tuple(u[0]))
        ref, ref_ws, rc = P.assemble_rhs(u)
        assert rc == 0
        assert rel_err(one.vec_function("residuals"), ref) <= 1e-12
        assert rel_err(one.vec_function("wave_speed"), ref_ws) <= 1e-12
    n = [m.iterate(0.3, 3) for m in (one, chained, few, few_chained)]
    nb = Batch().iterate([batched, few_batched], 0.3, 3)
    assert np.array_equal(n[0], n[1]) and np.array_equal(n[2], n[3])
    assert np.array_equal(n[0], nb[0]) and np.array_equal(n[2], nb[1])
    for a, b in ((one, chained), (one, batched), (few, few_chained), (few, few_batched)):
        for f in ("solution", "residuals", "time_step"):
            assert np.array_equal(a.vec_function(f), b.vec_function(f))
    for m in (one, chained, few, few_chained, batched, few_batched):
        m.destroy()

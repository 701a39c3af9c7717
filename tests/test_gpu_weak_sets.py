"""All weak boundary conditions of a method in one launch: many conditions with
few facets each (ends of the workgroup ranges, conditions of one facet, an empty
one) against one condition over the same boundary, alone and in a batch, and
point states set and removed between sweeps.

A facet's part does not depend on the condition it belongs to; a node's sum may
take its (at most two) facet rows in another order: 1e-14."""
import numpy as np
import pytest

from pdekit_amd import _lib as L
from pdekit_amd.mesh import rectangle
from pdekit_amd.rdm import Batch, PGRDMethodExplicit
from tests.helpers import advection_state, euler_state, rel_err

pytestmark = pytest.mark.gpu


def _method(mesh, u, parts, order=4):
    m = PGRDMethodExplicit(L.EULER2D, L.LDA, params=(1.4, 287.05)).configure_mesh_data(mesh)
    m.initialize_work_data(quad_order=order)
    for k, nodes in enumerate(parts):
        m.add_boundary_condition("WeakWall", f"wall{k}", nodes)
    m.set_vec_function("solution", u)
    return m


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("nparts", [1, 2, 9, 20])
def test_split_wall(order, nparts):
    mesh = rectangle(160, 6, extent=(-0.5, 1.5, 0.0, 1.0), split=2, order=order, bump=(1.0, 0.1, 25.0, 0.5))
    u = euler_state(mesh)
    x = mesh.node_coords[:, 0]
    wall = mesh.boundaries["ymin"]
    wall = wall[np.argsort(x[wall], kind="stable")]
    # cuts at vertices (every order-th node); 1 facet, some, the rest, and none
    cuts = np.concatenate([[0], np.sort(np.random.default_rng(nparts).choice(np.arange(1, 159), nparts - 1, False)), [160]])
    parts = [wall[order * a:order * b + 1] for a, b in zip(cuts[:-1], cuts[1:])] + [wall[:1]]
    one, many = _method(mesh, u, [wall]), _method(mesh, u, parts)
    one.iterate(0.5, 3)
    many.iterate(0.5, 3)
    for f in ("solution", "residuals", "wave_speed"):
        assert rel_err(many.vec_function(f), one.vec_function(f)) <= 1e-14
    # the same bits in a batch of both
    a, b = _method(mesh, u, [wall]), _method(mesh, u, parts)
    Batch().iterate([a, b], 0.5, 3)
    assert np.array_equal(a.vec_function("solution"), one.vec_function("solution"))
    assert np.array_equal(b.vec_function("solution"), many.vec_function("solution"))
    for m in (one, many, a, b):
        m.destroy()


def test_point_states_between_sweeps():
    mesh = rectangle(40, 30, split=2, order=1, jitter=0.1, seed=3)
    u = advection_state(mesh)
    b = mesh.boundaries

    def method(vals):
        m = PGRDMethodExplicit(L.ADVECTION2D, L.N, params=(0.8, 0.6)).configure_mesh_data(mesh)
        m.initialize_work_data(quad_order=4)
        for name, v in zip(("xmin", "ymin"), vals):
            m.add_boundary_condition("WeakDirichlet", name, b[name], values=[v])
        m.set_vec_function("solution", u)
        return m

    m, ref = method((0.3, 0.7)), method((0.9, 0.7))

    def residual(x):
        x.assemble_rhs()
        return x.vec_function("residuals")

    base = residual(m)
    info = m.weak_bc_info(0)
    m.set_weak_bc_state(0, np.full((info["facets"], info["quadrature_points"], 1), 0.9))
    assert np.array_equal(residual(m), residual(ref))  # the point state of condition 0 alone
    m.set_weak_bc_state(0, None)
    m.set_weak_bc_state(0, None)
    assert np.array_equal(residual(m), base)
    m.destroy()
    ref.destroy()


@pytest.mark.parametrize("scheme", [L.LDA, L.B])
@pytest.mark.parametrize("order", [1, 2])
def test_mixed_mesh_launches(order, scheme):
    """Quadrilaterals, triangles and weak facets of a mixed mesh in one launch
    (alone and in a batch) against chained sweeps, whose facets have a launch of
    their own: the same bits. Ragged last patches of both element types; walls on
    the triangles' side only (second order has no facets on quadrilaterals)."""
    mesh = rectangle(37, 22, extent=(-0.5, 1.5, 0.0, 1.0), split=2, quad_rows=9, order=order, bump=(1.0, 0.1, 25.0, 0.5))
    u = euler_state(mesh)
    top = mesh.boundaries["ymax"]
    half = top[mesh.node_coords[top, 0] <= mesh.node_coords[top, 0].mean()]

    def method(chain):
        m = PGRDMethodExplicit(L.EULER2D, scheme, params=(1.4, 287.05)).configure_mesh_data(mesh)
        m.initialize_work_data(quad_order=4)
        m.add_boundary_condition("WeakWall", "half", half)
        m.add_boundary_condition("WeakFarfield", "top", top, values=u[0])
        m.set_vec_function("solution", u)
        m.set_option(L.OPT_CHAIN, chain)
        return m

    one, chained, batched, other = method(0), method(1), method(0), method(1)
    n = [m.iterate(0.4, 4) for m in (one, chained)]
    nb = Batch().iterate([batched, other], 0.4, 4)
    assert np.array_equal(n[0], n[1]) and np.array_equal(n[0], nb[0]) and np.array_equal(n[0], nb[1])
    for m in (chained, batched, other):
        for f in ("solution", "residuals", "time_step"):
            assert np.array_equal(m.vec_function(f), one.vec_function(f))
    for m in (one, chained, batched, other):
        m.destroy()

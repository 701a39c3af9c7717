"""Scalar cells without a flux element (constant and rotating advection, Burgers
on first-order elements), whose residual is a . grad u: against the oracle, which
interpolates the flux at the P+1 nodes, where the two could differ -- strongly
distorted bilinear quadrilaterals (the flux element must still be exact there),
every order, with and without a source field, both assemblies. 1e-12 normwise,
as the parity tests."""
import numpy as np
import pytest

from pdekit_amd import _lib as L
from pdekit_amd.fe import element_tables
from pdekit_amd.mesh import rectangle
from pdekit_amd.rdm import PGRDMethodExplicit
from oracle.pyoracle import Problem
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu

MESHES = {
    "p1": dict(split=2, order=1), "p2": dict(split=2, order=2), "p3": dict(split=2, order=3),
    "q1": dict(split=1, quad_rows=7, order=1), "q2": dict(split=1, quad_rows=7, order=2),
    "q1p1": dict(split=2, quad_rows=4, order=1), "q2p2": dict(split=2, quad_rows=3, order=2),
}
PHYSICS = {"advection": (L.ADVECTION2D, (0.8, -0.6)), "rotation": (L.ROTATION2D, ()), "burgers": (L.BURGERS2D, ())}


@pytest.mark.parametrize("source", [False, True])
@pytest.mark.parametrize("scheme", [L.LDA, L.N, L.B, L.PSI, L.BPSI])
@pytest.mark.parametrize("mesh_name", list(MESHES))
@pytest.mark.parametrize("phys", list(PHYSICS))
def test_linear_flux(phys, mesh_name, scheme, source):
    physics, params = PHYSICS[phys]
    mesh = rectangle(9, 7, extent=(0.3, 1.7, 0.2, 1.1), jitter=0.3, seed=8, **MESHES[mesh_name])
    q = 6 if mesh.order == 3 else 4
    rng = np.random.default_rng(3)
    u = rng.uniform(0.2, 1.0, (mesh.nb_nodes, 1))
    src = rng.uniform(-1.0, 1.0, (mesh.nb_nodes, 1)) if source else None
    tables = {b.shape: element_tables(b.shape, mesh.order, q) for b in mesh.blocks}
    vol = {b.shape: element_tables(b.shape, mesh.order, mesh.order) for b in mesh.blocks}
    problem = Problem(mesh, tables, vol, physics, scheme, params)
    problem.set_sources(src)
    ref, ref_ws, rc = problem.assemble_rhs(u)
    assert rc == 0
    for scatter in ([2] if source else [2, 0]):
        m = PGRDMethodExplicit(physics, scheme, params=params or None).configure_mesh_data(mesh)
        m.initialize_work_data(quad_order=q, scatter=scatter)
        m.set_vec_function("solution", u)
        if source:
            m.set_sources(src)
        m.assemble_rhs()
        assert rel_err(m.vec_function("residuals"), ref) <= 1e-12
        assert rel_err(m.vec_function("wave_speed"), ref_ws) <= 1e-12
        m.destroy()

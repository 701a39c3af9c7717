"""The norms' reduction on the device against numpy on the residual field: fewer
norm partials than one pass of the reduction's threads, one more than that, and
many; 1, 4 and 5 equations; the driver loop's time step and norm; every assembly.

Tolerance: all terms are squares, and no sum is longer than a few hundred
additions one after the other (a thread's nodes or rows, then trees): 300 x
1.1e-16, half of it in the root: 1e-13 leaves a factor of six."""
import numpy as np
import pytest

from pdekit_amd import _lib as L
from pdekit_amd.mesh import box_tetra, rectangle, unit_quad_triag
from pdekit_amd.rdm import Batch, PGRDMethodExplicit
from tests.helpers import advection_state, euler_state, rel_err

pytestmark = pytest.mark.gpu

CASES = {
    "one_patch": (lambda: unit_quad_triag(5), L.ADVECTION2D, (0.8, 0.6)),
    "advection_513": (lambda: unit_quad_triag(182), L.ADVECTION2D, (0.8, 0.6)),
    "channel": (lambda: rectangle(96, 48, extent=(-0.5, 1.5, 0.0, 1.0), split=2, quad_rows=24), L.EULER2D, (1.4, 287.05)),
    "channel_many": (lambda: rectangle(512, 256, extent=(-0.5, 1.5, 0.0, 1.0), split=2), L.EULER2D, (1.4, 287.05)),
    "box": (lambda: box_tetra(20, 18, 16, extent=(1.0, 1.0, 0.5)), L.EULER3D, (1.4, 287.05)),
}


def _method(name, scatter=None):
    build, physics, params = CASES[name]
    mesh = build()
    m = PGRDMethodExplicit(physics, L.N, params=params).configure_mesh_data(mesh)
    m.initialize_work_data(quad_order={b.shape: 2 if b.shape == L.TETRA else 4 for b in mesh.blocks}, scatter=scatter)
    m.set_vec_function("solution", advection_state(mesh) if m.neq == 1 else euler_state(mesh, dim=mesh.dim))
    b = mesh.boundaries
    nodes = b["Edge0"] if "Edge0" in b else b["xmin"]
    m.add_boundary_condition("StrongDirichlet", "in", nodes, m.vec_function("solution")[nodes])
    return m, nodes


def _norm(res, nodes, excl):
    r = np.delete(res, nodes, axis=0) if excl else res
    return np.sqrt((r ** 2).mean(0))


@pytest.mark.parametrize("scatter", [2, 1])
@pytest.mark.parametrize("excl", [False, True])
@pytest.mark.parametrize("name", list(CASES))
def test_norms(name, excl, scatter):
    m, nodes = _method(name, scatter)
    for n in (1, 3):
        assert rel_err(m.iterate(0.4, n, exclude_dirichlet=excl), _norm(m.vec_function("residuals"), nodes, excl)) <= 1e-13
    assert rel_err(m.residual_norm_L2(excl), _norm(m.vec_function("residuals"), nodes, excl)) <= 1e-13
    m.assemble_lhs_and_rhs(0.4)
    dt, res = m.vec_function("time_step"), m.vec_function("residuals")
    assert rel_err(dt, 0.4 * m.vec_function("dual_volume") / m.vec_function("wave_speed")) <= 1e-15
    u = m.vec_function("solution")
    m.solve()
    assert rel_err(m.vec_function("solution"), u - dt[:, None] * res) <= 1e-15
    assert rel_err(m.compute_residual_norm(), _norm(res * dt[:, None], nodes, False)) <= 1e-13
    m.destroy()


def test_batch_norms():
    ms = [_method(name)[0] for name in CASES]
    norms = Batch().iterate(ms, 0.4, 2, exclude_dirichlet=True)
    for name, m, n in zip(CASES, ms, norms):
        alone, _ = _method(name)
        assert np.array_equal(alone.iterate(0.4, 2, exclude_dirichlet=True), n)
        alone.destroy()
        m.destroy()

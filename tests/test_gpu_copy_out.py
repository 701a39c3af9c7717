"""Copies of results to the host through the pinned ring: sizes below one piece (1
MiB), at its edge, several pieces, one full ring (16 MiB) and just beyond, into
fresh and reused memory, and several threads at once (one of them takes the ring,
the others copy directly). Every byte against the same data computed another way:
the exact values set, and the Jacobian of cell k against that of a smaller mesh's
run with the same cells."""
import threading

import numpy as np
import pytest

from pdekit_amd import _lib as L
from pdekit_amd.mesh import rectangle, unit_quad_triag
from pdekit_amd.rdm import PGRDMethodExplicit
from tests.helpers import euler_state, oracle_problem, rel_err

pytestmark = pytest.mark.gpu


def _method(n):
    mesh = unit_quad_triag(n)
    m = PGRDMethodExplicit(L.ADVECTION2D, L.N, params=(0.8, 0.6)).configure_mesh_data(mesh)
    m.initialize_work_data(quad_order=4)
    return m, mesh.nb_nodes


# nodes (n x n): 8 n^2 bytes around 1 MiB (362^2 x 8 = 1 048 352, 363^2), several
# pieces, 16 MiB (1448^2 x 8 = 16 773 632, 1449^2)
@pytest.mark.parametrize("n", [2, 362, 363, 700, 1448, 1449])
def test_field_copies(n):
    m, nn = _method(n)
    u = np.random.default_rng(n).uniform(-1.0, 1.0, (nn, 1))
    m.set_vec_function("solution", u)
    for _ in range(3):
        assert np.array_equal(m.vec_function("solution"), u)
    m.destroy()


def test_threads_copy_at_once():
    ms = [_method(n)[0] for n in (500, 700, 363, 30)]
    us = [np.random.default_rng(k).uniform(-1.0, 1.0, (m.mesh.nb_nodes, 1)) for k, m in enumerate(ms)]
    bad = []

    def run(m, u):
        m.set_vec_function("solution", u)
        for _ in range(20):
            if not np.array_equal(m.vec_function("solution"), u):
                bad.append(m)

    threads = [threading.Thread(target=run, args=a) for a in zip(ms, us)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for m in ms:
        m.destroy()


@pytest.mark.parametrize("scheme", [L.LDA, L.N, L.B])
@pytest.mark.parametrize("nx", [1, 12, 90, 130])
def test_jacobian_copies(nx, scheme):
    """Jacobians of 0.6 KB to 19 MB in pieces against the oracle's (12 x 12 doubles
    a cell); twice, as the second call reuses the permutation on the device."""
    mesh = rectangle(nx, max(1, nx // 2), extent=(-0.5, 1.5, 0.0, 1.0), split=2, order=1)
    u = euler_state(mesh)
    m = PGRDMethodExplicit(L.EULER2D, scheme, params=(1.4, 287.05)).configure_mesh_data(mesh)
    m.initialize_work_data(quad_order=4)
    m.set_vec_function("solution", u)
    first = m.element_jacobians(0)
    for a, b in zip(first, m.element_jacobians(0)):
        assert np.array_equal(a, b)
    ref = oracle_problem(mesh, L.EULER2D, scheme, (1.4, 287.05)).cell_jacobians(0, u)
    for a, b in zip(first, ref):
        assert rel_err(a, b) <= 1e-12
    m.destroy()

"""Results into pinned memory of the caller, which take the runtime's direct copy: every
byte as in pageable memory, below one piece (1 MiB) and above, at the start of the
allocation and inside it."""
import ctypes as C

import numpy as np
import pytest
import torch

from pdekit_amd import _lib as L
from pdekit_amd.mesh import rectangle, unit_quad_triag
from pdekit_amd.rdm import PGRDMethodExplicit
from tests.helpers import euler_state

pytestmark = pytest.mark.gpu


def _pinned(n, shift):
    t = torch.full((n + shift,), -1.0, dtype=torch.float64).pin_memory()[shift:]
    return t, C.cast(t.data_ptr(), C.POINTER(C.c_double))


@pytest.mark.parametrize("shift", [0, 3])
@pytest.mark.parametrize("n", [2, 300, 700])
def test_field(n, shift):
    mesh = unit_quad_triag(n)
    m = PGRDMethodExplicit(L.ADVECTION2D, L.N, params=(0.8, 0.6)).configure_mesh_data(mesh)
    m.initialize_work_data(quad_order=4)
    u = np.random.default_rng(n).uniform(-1.0, 1.0, (mesh.nb_nodes, 1))
    m.set_vec_function("solution", u)
    t, p = _pinned(u.size, shift)
    L.check(L.lib().pdrd_get_field(m._h, L.SOLUTION, p), "pdrd_get_field")
    assert np.array_equal(t.numpy(), u.ravel())
    m.destroy()


@pytest.mark.parametrize("nx", [3, 60])
def test_jacobians(nx):
    mesh = rectangle(nx, max(1, nx // 2), extent=(-0.5, 1.5, 0.0, 1.0), split=2, order=1)
    m = PGRDMethodExplicit(L.EULER2D, L.N, params=(1.4, 287.05)).configure_mesh_data(mesh)
    m.initialize_work_data(quad_order=4)
    m.set_vec_function("solution", euler_state(mesh))
    ref = m.element_jacobians(0)
    out = [_pinned(a.size, 0) for a in ref]
    L.check(L.lib().pdrd_element_jacobians(m._h, 0, out[0][1], out[1][1], out[2][1]), "pdrd_element_jacobians")
    for (t, _), a in zip(out, ref):
        assert np.array_equal(t.numpy(), a.ravel())
    m.destroy()

"""The local time step CFL V / sum lambda is one division of what the method itself
reports: the same bits as numpy's quotient (a product with a reciprocal rounds twice
and is off in the last bit at every third node). From the assembly's node finish and
the fix-up, from iterations (chained and not, whose other patches take the step of a
shared node over: their states would differ) and from the other assemblies."""
import numpy as np
import pytest

from pdekit_amd import _lib as L
from pdekit_amd.rdm import Batch, PGRDMethodExplicit
from tests.helpers import CASES, quad_orders

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scatter", [0, 1, 2])
@pytest.mark.parametrize("name", ["adv_p1", "adv_p3", "burgers_p2", "euler2d_mixed", "euler2d_p2", "euler3d_p1"])
def test_time_step_is_the_quotient(name, scatter):
    build, physics, params, state = CASES[name]
    mesh = build()
    u, cfl = state(mesh), 0.37
    m = PGRDMethodExplicit(physics, L.N, params=params or None).configure_mesh_data(mesh)
    m.initialize_work_data(quad_order=quad_orders(mesh), scatter=scatter)
    m.set_vec_function("solution", u)

    def check():
        v, ws = m.vec_function("dual_volume"), m.vec_function("wave_speed")
        assert np.array_equal(m.vec_function("time_step"), cfl * v / ws)

    m.assemble_lhs_and_rhs(cfl)
    check()
    for chain in (0, 1) if scatter == 2 else (0,):
        m.set_option(L.OPT_CHAIN, chain)
        for n in (1, 3):
            m.iterate(cfl, n)
            check()
    if scatter == 2:
        Batch().iterate([m], cfl, 3)
        check()
    m.destroy()

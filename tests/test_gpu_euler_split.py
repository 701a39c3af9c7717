"""The split solve of the Euler cells (entropy part by one reciprocal, acoustic
block by its symmetric elimination) against the oracle's explicit inverse, over
the range of Mach numbers that changes the conditioning of S = sum K+: nearly
stagnant (sum l0 small beside the acoustic part), subsonic, transonic and
supersonic (some nodes without any K+).

Tolerance: both sides solve with S, whose condition number is at most about
2 (1 + M) / M on these near-uniform states; with 30 roundings of 1.1e-16 in a
solve and its products that is 7e-13 at M = 0.01 and less above: 1e-12."""
import numpy as np
import pytest

from pdekit_amd import _lib as L
from pdekit_amd.rdm import PGRDMethodExplicit
from tests.helpers import CASES, euler_state, oracle_problem, quad_orders, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", [L.LDA, L.N, L.B, L.PSI, L.BPSI])
@pytest.mark.parametrize("mach", [0.01, 0.98, 3.0])
@pytest.mark.parametrize("case", ["euler2d_mixed", "euler2d_q2_mixed", "euler3d_p1", "euler3d_p2"])
def test_split_solve_over_mach(case, mach, scheme):
    build, physics, params, _ = CASES[case]
    mesh = build()
    dim = 3 if physics == L.EULER3D else 2
    u = euler_state(mesh, mach=mach, dim=dim)
    # a cross flow, so that no velocity component is zero to rounding
    u[:, 2] += 0.3 * u[:, 1]
    u[:, -1] += 0.5 * u[:, 2] ** 2 / u[:, 0]
    m = PGRDMethodExplicit(physics, scheme, params=params).configure_mesh_data(mesh)
    m.initialize_work_data(quad_order=quad_orders(mesh))
    m.set_vec_function("solution", u)
    m.assemble_rhs()
    m.check_status()
    res, ws = m.vec_function("residuals"), m.vec_function("wave_speed")
    m.destroy()
    ref, ref_ws, rc = oracle_problem(mesh, physics, scheme, params).assemble_rhs(u)
    assert rc == 0
    assert np.isfinite(res).all()
    assert rel_err(res, ref) <= 1e-12
    assert rel_err(ws, ref_ws) <= 1e-12

"""Default cells per patch of the Euler equations on second-order triangles: 64 for the
schemes at 2 waves per SIMD while a wave per SIMD holds the mesh, 128 for the others
and beyond. A size the caller sets is kept. Both sizes against the oracle where it is
quick, 1e-12 normwise as in the parity tests."""
import pytest

from pdekit_amd import _lib as L
from pdekit_amd.mesh import rectangle
from pdekit_amd.rdm import PGRDMethodExplicit
from tests.helpers import euler_state, oracle_problem, rel_err

pytestmark = pytest.mark.gpu

PARAMS = (1.4, 287.05)


@pytest.mark.parametrize("scheme,nx,want", [(L.LDA, 128, 64), (L.N, 20, 64), (L.PSI, 128, 64), (L.LDA, 129, 128),
                                            (L.B, 128, 128), (L.BPSI, 20, 128)])
def test_second_order_triangles(scheme, nx, want):
    mesh = rectangle(2 * nx, nx, extent=(-0.5, 1.5, 0.0, 1.0), split=2, order=2)
    for cells in (None, 64, 128):
        m = PGRDMethodExplicit(L.EULER2D, scheme, params=PARAMS).configure_mesh_data(mesh)
        m.initialize_work_data(quad_order=4, patch_cells=cells)
        assert m.get_option(L.OPT_PATCH_CELLS) == (cells or want)
        if nx == 20:
            u = euler_state(mesh)
            m.set_vec_function("solution", u)
            m.assemble_rhs()
            ref, _, rc = oracle_problem(mesh, L.EULER2D, scheme, PARAMS).assemble_rhs(u)
            assert rc == 0 and rel_err(m.vec_function("residuals"), ref) <= 1e-12
        m.destroy()

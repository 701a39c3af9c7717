"""LF_Blend on first-order quadrilaterals and triangles of one mesh whose state changes
sign (the case where |u| + |avg| of a cell gets small), against its two passes in
numpy. The operations are the kernel's own in its order, so the values differ by what
a last bit of the average moves the quotient: per addition half an ulp of the largest
partial sum, 2 nd 2^-53 max|u| / min(|u| + |avg|), and an ulp of the quotient."""
import numpy as np
import pytest

from pdekit_amd import _lib as L
from pdekit_amd.rdm import PGRDMethodExplicit
from tests.helpers import CASES, quad_orders

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [None, 64, 128])
def test_lf_blend_first_order_mixed(cells):
    build, physics, params, state = CASES["burgers_q1"]
    mesh = build()
    u = state(mesh)
    m = PGRDMethodExplicit(physics, L.B, params=params or None).configure_mesh_data(mesh)
    m.initialize_work_data(quad_order=quad_orders(mesh), patch_cells=cells)
    m.set_vec_function("solution", u)
    theta = m.compute_blending_coeff("LF_Blend")
    assert np.array_equal(theta, m.compute_blending_coeff("LF_Blend"))
    m.destroy()
    top, out, least = np.zeros(mesh.nb_nodes), np.zeros(mesh.nb_nodes), np.inf
    for b in mesh.blocks:
        c = b.sol_conn.astype(np.int64)
        un, avg = u[c, 0], np.zeros(len(c))
        for n in range(c.shape[1]):
            avg += un[:, n]
        avg /= c.shape[1]
        denominator = np.abs(un) + np.abs(avg)[:, None] + 1e-12
        least = min(least, denominator.min())
        np.maximum.at(top, c, (np.abs(un - avg[:, None]) / denominator).max(1)[:, None])
    for b in mesh.blocks:
        c = b.sol_conn.astype(np.int64)
        np.maximum.at(out, c, (1.0 - top[c].max(1))[:, None])
    assert np.abs(theta - out).max() <= 2 * 4 * 2.0 ** -53 * np.abs(u).max() / least + 2.0 ** -52

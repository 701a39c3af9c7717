"""LF_Blend over the patches against its two passes in numpy, at the vertices (the
other nodes interpolate them), on every element type, with ragged last patches and
64 to 256 cells a
patch."""
import numpy as np
import pytest

from pdekit_amd import _lib as L
from pdekit_amd.rdm import PGRDMethodExplicit
from tests.helpers import CASES, oracle_problem, quad_orders, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [None, 64, 128])
@pytest.mark.parametrize("name", [n for n in CASES if n not in ("burgers_q1",)])
def test_lf_blend_by_patches(name, cells):
    build, physics, params, state = CASES[name]
    mesh = build()
    u = state(mesh)
    m = PGRDMethodExplicit(physics, L.B, params=params or None).configure_mesh_data(mesh)
    m.initialize_work_data(quad_order=quad_orders(mesh), patch_cells=cells)
    m.set_vec_function("solution", u)
    theta = m.compute_blending_coeff("LF_Blend")
    again = m.compute_blending_coeff("LF_Blend")
    assert np.array_equal(theta, again)
    m.destroy()
    # the two passes in numpy, the divisions and maxima in the kernels' order
    top = np.zeros(mesh.nb_nodes)
    out = np.zeros(mesh.nb_nodes)
    for b in mesh.blocks:
        c = b.sol_conn.astype(np.int64)
        un = u[c, 0]
        avg = np.zeros(len(c))
        for n in range(c.shape[1]):
            avg += un[:, n]
        avg /= c.shape[1]
        ksi = (np.abs(un - avg[:, None]) / (np.abs(un) + np.abs(avg)[:, None] + 1e-12)).max(1)
        np.maximum.at(top, c, ksi[:, None])
    for b in mesh.blocks:
        c = b.sol_conn.astype(np.int64)
        nv = b.geo_conn.shape[1]
        np.maximum.at(out, c[:, :nv], (1.0 - top[c].max(1))[:, None])
    verts = np.unique(np.concatenate([b.sol_conn[:, :b.geo_conn.shape[1]].ravel() for b in mesh.blocks]))
    # a rounding of the average and of the quotient apart (contracted on the device)
    assert rel_err(theta[verts], out[verts]) <= 4e-16

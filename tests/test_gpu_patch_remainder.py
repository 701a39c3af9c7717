"""Nodes of a patch beyond those that a thread of the scalar kernels gathers together: a
patch of C cells has about C / 2 (P1) to 4.5 C (P3) nodes, for which the threads'
batches are sized, so that a connected mesh never reaches the loop behind them.
Here it does: every cell with nodes of its own ("split"), or every cell in one of
three layers that share no node ("layers": about three times the nodes, many of them
shared between patches, so that chained sweeps finish shared nodes in that loop).
Against the oracle, 1e-12 normwise as the parity tests; chained and plain sweeps,
alone and in a batch, the same bits."""
import numpy as np
import pytest

from pdekit_amd import _lib as L
from pdekit_amd.mesh import CellBlock, Mesh, rectangle
from pdekit_amd.rdm import Batch, PGRDMethodExplicit
from tests.helpers import advection_state, burgers_state, oracle_problem, quad_orders, rel_err

pytestmark = pytest.mark.gpu


def layered(mesh, layers):
    """Cell c of a block in layer c % layers (layers 0: each in its own) of the nodes."""
    nn, node_coords, blocks, seen = 0, [], [], {}
    for b in mesh.blocks:
        conn = np.empty_like(b.sol_conn)
        for c, cell in enumerate(b.sol_conn):
            layer = c % layers if layers else (b.shape, c)
            for k, v in enumerate(cell):
                key = (layer, int(v))
                if key not in seen:
                    seen[key] = nn
                    node_coords.append(mesh.node_coords[v])
                    nn += 1
                conn[c, k] = seen[key]
        blocks.append(CellBlock(b.shape, b.cells, b.geo_conn, conn))
    return Mesh(mesh.dim, mesh.coords, mesh.cell_shape, mesh.order, nn, np.array(node_coords), blocks)


MESHES = {"p1": lambda: rectangle(23, 19, split=2, order=1, jitter=0.1, seed=2),
          "p2": lambda: rectangle(17, 13, split=2, order=2, jitter=0.1, seed=2),
          "p3": lambda: rectangle(13, 11, split=2, order=3, jitter=0.1, seed=2),
          "q1": lambda: rectangle(23, 19, split=1, order=1, jitter=0.1, seed=2),
          "q2": lambda: rectangle(17, 13, split=1, order=2, jitter=0.1, seed=2)}


@pytest.mark.parametrize("scheme", [L.LDA, L.B])
@pytest.mark.parametrize("physics", [L.ADVECTION2D, L.BURGERS2D])
@pytest.mark.parametrize("layers", [0, 3])
@pytest.mark.parametrize("name", list(MESHES))
def test_more_nodes_than_a_batch(name, layers, physics, scheme):
    mesh = layered(MESHES[name](), layers)
    params = (0.8, 0.6) if physics == L.ADVECTION2D else ()
    u = advection_state(mesh) if physics == L.ADVECTION2D else burgers_state(mesh)
    extra = np.random.default_rng(3).uniform(0.0, 0.1, mesh.nb_nodes)
    dirichlet = np.arange(0, mesh.nb_nodes, 7)

    def method(form, chain):
        m = PGRDMethodExplicit(physics, scheme, params=params or None).configure_mesh_data(mesh)
        m.initialize_work_data(quad_order=quad_orders(mesh), patch_cells=64)
        m.set_vec_function("solution", u)
        m.set_option(L.OPT_CHAIN, chain)
        if form == "nodal":
            m.set_artificial_viscosity(extra) if scheme == L.LDA else m.set_blending_coeff(extra)
        if form == "sources":
            m.set_sources(extra[:, None])
        return m

    for form in ("plain", "nodal", "sources"):
        ms = [method(form, chain) for chain in (0, 1, 0, 1)]
        assert ms[0].get_option(L.OPT_SCATTER) == 2
        if form == "plain":
            ms[0].assemble_rhs()
            ref, ref_ws, rc = oracle_problem(mesh, physics, scheme, params).assemble_rhs(u)
            assert rc == 0
            assert rel_err(ms[0].vec_function("residuals"), ref) <= 1e-12
            assert rel_err(ms[0].vec_function("wave_speed"), ref_ws) <= 1e-12
        for m in ms:
            m.add_boundary_condition("StrongDirichlet", "some", dirichlet, np.full((dirichlet.size, 1), 0.5))
        norms = [m.iterate(0.2, 4) for m in ms[:2]] + Batch().iterate(ms[2:], 0.2, 4)
        for m, n in zip(ms[1:], norms[1:]):
            assert np.array_equal(n, norms[0])
            for f in ("solution", "residuals", "time_step"):
                assert np.array_equal(m.vec_function(f), ms[0].vec_function(f))
        for m in ms:
            m.destroy()

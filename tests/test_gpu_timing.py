"""The intervals that a timed iterate reports: weak boundary facets belong to the nodal
pass, in every form of a sweep (chained and not, and the joint launch of a mixed
mesh, whose results stay the same bits). A strip with a facet on every second cell:
what the conditions add has to show in the nodal interval and not in the cells'."""
import numpy as np
import pytest

from pdekit_amd import _lib as L
from pdekit_amd.mesh import rectangle
from pdekit_amd.rdm import PGRDMethodExplicit
from tests.helpers import advection_state, euler_state

pytestmark = pytest.mark.gpu


def _mean(m, u):
    m.set_vec_function("solution", u)
    m.set_option(L.OPT_TIMING, 1)
    m.iterate(1e-6, 5)
    t = []
    for _ in range(5):
        m.iterate(1e-6, 20)
        t.append(m.last_timing())
    return np.median(np.array(t), axis=0) * 1e3


@pytest.mark.parametrize("name", ["chained", "plain", "mixed"])
def test_facets_in_the_nodal_interval(name):
    mesh = rectangle(40000, 2, extent=(0.0, 20000.0, 0.0, 1.0), split=2, quad_rows=1 if name == "mixed" else 0)
    euler = name == "mixed"
    u = euler_state(mesh) if euler else advection_state(mesh)
    ms = []
    for weak in (False, True):
        m = PGRDMethodExplicit(L.EULER2D if euler else L.ADVECTION2D, L.LDA, params=(1.4, 287.05) if euler else (0.8, 0.6))
        m.configure_mesh_data(mesh).initialize_work_data(quad_order=4)
        for side in ("ymin", "ymax") if weak else ():
            m.add_boundary_condition("WeakWall" if euler else "WeakDirichlet", side, mesh.boundaries[side],
                                     values=None if euler else [0.5])
        m.set_option(L.OPT_CHAIN, int(name == "chained"))
        ms.append(m)
    (cell0, node0), (cell1, node1) = (_mean(m, u) for m in ms)
    print(f"{name}: cells {cell0:.1f} -> {cell1:.1f} us, nodes {node0:.1f} -> {node1:.1f} us", flush=True)
    assert node1 - node0 > cell1 - cell0
    # timed and not: the same bits
    weak = ms[1]
    out = []
    for timing in (0, 1):
        weak.set_option(L.OPT_TIMING, timing)
        weak.set_vec_function("solution", u)
        weak.iterate(0.3, 4)
        out.append([weak.vec_function(f) for f in ("solution", "residuals", "time_step", "wave_speed")])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    for m in ms:
        m.destroy()

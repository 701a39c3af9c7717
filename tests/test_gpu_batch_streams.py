"""Batches on several streams: groups of methods that share no launch run side by
side. Every method must advance as on its own (the same bits): more groups than
streams, methods that join groups (a mixed mesh between a triangle and a
quadrilateral one), and two batches in two threads."""
import threading

import numpy as np
import pytest

from pdekit_amd import _lib as L
from pdekit_amd.rdm import Batch, PGRDMethodExplicit
from pdekit_amd.mesh import rectangle
from tests.helpers import CASES, euler_state, quad_orders

pytestmark = pytest.mark.gpu

# (case, scheme): eight kernels in seven groups (the mixed mesh joins the
# triangle and the quadrilateral one), some with two methods
MIX = [("adv_p1", L.N), ("adv_p2", L.N), ("adv_p3", L.N), ("burgers_p2", L.B), ("burgers_p1", L.N),
       ("euler2d_p1", L.LDA), ("euler2d_mixed", L.LDA), ("euler2d_q1", L.LDA), ("euler3d_p1", L.BPSI), ("adv_p1", L.N),
       ("euler2d_mixed", L.LDA), ("adv_p2", L.LDA)]


def _case(name):
    if name == "euler2d_q1":
        return (lambda: rectangle(10, 9, extent=(-0.5, 1.5, 0.0, 1.0), split=1, quad_rows=9, order=1,
                                  bump=(1.0, 0.1, 25.0, 0.5)), L.EULER2D, (1.4, 287.05), euler_state)
    return CASES[name]


def _method(name, scheme, weak):
    build, physics, params, state = _case(name)
    mesh = build()
    m = PGRDMethodExplicit(physics, scheme, params=params or None).configure_mesh_data(mesh)
    m.initialize_work_data(quad_order=quad_orders(mesh))
    if weak and physics == L.EULER2D:
        m.add_boundary_condition("WeakWall", "wall", mesh.boundaries["ymin"])
    m.set_vec_function("solution", state(mesh))
    return m


def _run(mix, n_iter, weak, out, key):
    batch, ms = Batch(), [_method(c, s, weak) for c, s in mix]
    norms = batch.iterate(ms, 0.4, n_iter, exclude_dirichlet=True)
    norms = batch.iterate(ms, 0.4, n_iter, exclude_dirichlet=True)
    out[key] = [(m.vec_function("solution"), m.vec_function("residuals"), n) for m, n in zip(ms, norms)]
    for m in ms:
        m.destroy()


def _alone(mix, n_iter, weak):
    out = []
    for c, s in mix:
        m = _method(c, s, weak)
        m.iterate(0.4, n_iter, exclude_dirichlet=True)
        n = m.iterate(0.4, n_iter, exclude_dirichlet=True)
        out.append((m.vec_function("solution"), m.vec_function("residuals"), n))
        m.destroy()
    return out


def _same(a, b):
    return all(np.array_equal(x, y) for p, q in zip(a, b) for x, y in zip(p, q))


@pytest.mark.parametrize("weak", [False, True])
@pytest.mark.parametrize("n_iter", [1, 2, 7])
@pytest.mark.parametrize("count", [1, 2, 5, len(MIX)])
def test_groups_on_streams(count, n_iter, weak):
    out = {}
    _run(MIX[-count:], n_iter, weak, out, 0)
    assert _same(out[0], _alone(MIX[-count:], n_iter, weak))


def test_two_batches_in_two_threads():
    out = {}
    mixes = [MIX, MIX[::-1]]
    threads = [threading.Thread(target=_run, args=(mix, 9, True, out, k)) for k, mix in enumerate(mixes)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k, mix in enumerate(mixes):
        assert _same(out[k], _alone(mix, 9, True))

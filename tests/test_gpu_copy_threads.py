"""Copies of several threads at once: every thread has to end all of its copies (one
that fails in a thread would otherwise go unseen), large ones and small ones, on
methods made and destroyed meanwhile, so that the pinned pieces come and go."""
import threading

import numpy as np
import pytest

from pdekit_amd import _lib as L
from pdekit_amd.mesh import unit_quad_triag
from pdekit_amd.rdm import PGRDMethodExplicit

pytestmark = pytest.mark.gpu

ROUNDS, COPIES = 4, 8


def test_every_copy_of_every_thread():
    meshes = [unit_quad_triag(n) for n in (500, 700, 363, 30)]
    done, errors = [0] * len(meshes), []

    def run(k):
        try:
            u = np.random.default_rng(k).uniform(-1.0, 1.0, (meshes[k].nb_nodes, 1))
            for _ in range(ROUNDS):
                m = PGRDMethodExplicit(L.ADVECTION2D, L.N, params=(0.8, 0.6)).configure_mesh_data(meshes[k])
                m.initialize_work_data(quad_order=4)
                m.set_vec_function("solution", u)
                for _ in range(COPIES):
                    assert np.array_equal(m.vec_function("solution"), u)
                    done[k] += 1
                m.destroy()
        except BaseException as e:
            errors.append(e)

    threads = [threading.Thread(target=run, args=(k,)) for k in range(len(meshes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    assert done == [ROUNDS * COPIES] * len(meshes)

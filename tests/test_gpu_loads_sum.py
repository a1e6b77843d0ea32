"""The surface loads' sums over face counts at the edges of the kernel's chunks
(256 terms, two a face; 16 terms read at once), on one handle in turn, so that
its scratch grows and shrinks.  Bitwise against the oracle."""
import numpy as np
import pytest

from pfem2_amd import FP64, ParticleStage
from pfem2_amd import mesh as M
from oracle_binding import Oracle
from parity_util import bitwise_equal
from test_gpu_fem import _oracle_loads

pytestmark = pytest.mark.gpu


def test_face_counts():
    m = M.cylinder_channel(0.2, seed=67)
    V = M.cylinder_flow(m, 1.0, eps=0.02, seed=68)
    P = 0.3 * np.random.default_rng(69).normal(size=m.n_dofs) + 1.0
    patch = M.boundary_faces(m, "cylinder")
    g = ParticleStage(m, 0.01, 2, 3, [2, 2], FP64)
    o = Oracle(m, 0.01, 2, 3, [2, 2])
    args = (0.001, 1.0, 0.2, 0.1, 3, 17)
    for n in (1, 7, 8, 9, 127, 128, 129, 300, 1000, 2):
        faces = np.ascontiguousarray(patch[np.arange(n) % len(patch)])
        a = g.calculate_loads(P, faces, *args, V=V)
        assert bitwise_equal(a, _oracle_loads(o, V, P, faces, *args)), n
        g.reinterpolate_fields(np.zeros((m.n_vertices, 2)), P)   # another user of the scratch in between
    g.close()


def test_kept_scratch_is_counted():
    """memory_bytes includes the scratch that the nodal routines keep: the
    displacements, the new velocities, and each extra field twice; a smaller
    call afterwards takes no more."""
    m = M.cylinder_channel(0.2, seed=67)
    g = ParticleStage(m, 0.01, 2, 3, [2, 2], FP64)
    g.upload_fields(np.zeros((2, m.n_dofs)), np.zeros((2, m.n_dofs)))
    own = g.memory_bytes()
    P = np.zeros(m.n_dofs)
    g.reinterpolate_fields(np.zeros((m.n_vertices, 2)), P)
    kept = 8 * (2 * m.n_vertices + 2 * m.n_dofs + 2 * m.n_dofs)
    assert g.memory_bytes() == own + kept
    g.reinterpolate_fields(np.zeros((m.n_vertices, 2)))
    assert g.memory_bytes() == own + kept
    g.close()

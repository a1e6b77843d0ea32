"""The output offsets of a regroup from the census's sums over groups of
cells: mesh sizes at the edges of a write workgroup's cells (16) and of a tile
(256), and on both sides of the size from which the offsets are scanned instead
(32,768 cells), with empty parts reseeded and a mesh move between steps; bitwise
against the oracle."""
import numpy as np
import pytest

from pfem2_amd import FP64, ParticleStage
from pfem2_amd import mesh as M
from oracle_binding import Oracle
from parity_util import assert_particles_match, bitwise_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(5, 3), (17, 1), (51, 5), (16, 16), (257, 1), (31, 33), (145, 113), (128, 256), (331, 99)])
def test_offsets(nx, ny):
    m = M.quad_2d(nx, ny, (0.0, 0.0), (0.1 * nx, 0.1 * ny), jitter=0.1, seed=4)
    rng = np.random.default_rng(6)
    V = np.array([[0.9], [0.2]]) + rng.uniform(-0.3, 0.3, size=(2, m.n_dofs))
    g = ParticleStage(m, 0.06, 3, 2, [2, 2], FP64, keep_velocity_ext=True)
    o = Oracle(m, 0.06, 3, 2, [2, 2])
    X0 = m.vertices.copy()
    bump = np.sin(np.pi * X0[:, 0] / X0[:, 0].max())
    for s in (g, o):
        s.upload_fields(V, V)
        s.seed_particles()
    for step in range(3):
        Vg, Vo = g.step(download=True), o.step()
        assert bitwise_equal(Vg, Vo), step
        X = X0.copy()
        X[:, 1] += 0.012 * (step + 1) * bump
        g.move_mesh(X)
        o.update_vertices(X)
        o.sort_particles_into_subdomains_and_cells()
        o.check_empty_cells()
    assert g.particle_counter() == o.particle_counter()
    assert np.array_equal(g.cell_counts(), o.cell_counts())
    assert_particles_match(g.particles(), o.particles(), 0.0, f"{nx}x{ny}", bitwise=True)
    g.close()

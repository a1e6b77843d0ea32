"""Cells that the census lists for k_cell_big: candidate counts at the edges of
its rows (64, 128) and beyond, on lattices of at most 16 parts and of more,
with arrivals from crowded neighbours; a few cells (a block each) and more than
its blocks (16-lane groups first).  Bitwise against the oracle."""
import numpy as np
import pytest

from pfem2_amd import FP64, ParticleStage
from pfem2_amd import mesh as M
from oracle_binding import Oracle
from parity_util import assert_particles_match, bitwise_equal

pytestmark = pytest.mark.gpu

FEW = [1, 63, 64, 65, 66, 127, 128, 129, 130, 300, 1100]
MANY = [65, 66, 127, 128, 129, 130, 20]


def _run(nx, ny, counts, q, max_per_part, speed, steps):
    m = M.quad_2d(nx, ny, (0.0, 0.0), (0.1 * nx, 0.1 * ny), jitter=0.1, seed=8)
    rng = np.random.default_rng(9)
    V = speed * (np.array([[1.0], [0.1]]) + rng.uniform(-0.2, 0.2, size=(2, m.n_dofs)))
    per = np.array([2 if counts is FEW and c % 2 else counts[c % len(counts)] for c in range(m.n_cells)])
    cell = np.repeat(np.arange(m.n_cells, dtype=np.int32), per)
    xi = rng.uniform(0.02, 0.98, size=(len(cell), 2))
    g = ParticleStage(m, 0.05, 3, max_per_part, q, FP64, capacity=3 * len(cell) + 64 * m.n_cells)
    o = Oracle(m, 0.05, 3, max_per_part, q)
    for s in (g, o):
        s.upload_fields(V, V)
        s.insert_particles(cell, xi)
    for step in range(steps):
        Vg, Vo = g.step(download=True), o.step()
        assert bitwise_equal(Vg, Vo), step
    assert np.array_equal(g.cell_counts(), o.cell_counts())
    assert g.particle_counter() == o.particle_counter() and g.stats()["deleted"] == o.stats()["deleted"]
    assert_particles_match(g.particles(), o.particles(), 0.0, str(q), bitwise=True)
    g.close()


@pytest.mark.parametrize("q,max_per_part", [([3, 3], 2), ([4, 4], 40), ([5, 5], 2), ([8, 8], 3)])
@pytest.mark.parametrize("speed", [0.0, 0.6])
def test_few(q, max_per_part, speed):
    _run(3 * len(FEW), 3, FEW, q, max_per_part, speed, 2)


@pytest.mark.parametrize("q,max_per_part", [([4, 4], 20), ([5, 5], 2)])
def test_many(q, max_per_part):
    _run(300, 8, MANY, q, max_per_part, 0.6, 2)

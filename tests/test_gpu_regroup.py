"""The regroup write with the projection sums (k_cell_write): mesh sizes around
its cells per workgroup, cells whose segments span several of its passes,
empty cells, and cells whose survivors outnumber the slot row (their sources
go through the position map).  FP64 bitwise against the oracle; FP32-mixed
bitwise against the three separate calls (whose sums come from
k_cell_partials32)."""
import numpy as np
import pytest

from pfem2_amd import FP32_MIXED, FP64, ParticleStage
from pfem2_amd import mesh as M
from oracle_binding import Oracle
from parity_util import assert_particles_match, bitwise_equal

pytestmark = pytest.mark.gpu

CASES = {   # cells, lattice, MAX, particles per lattice point, dim, degree
    "1 cell": ((1, 1), [3, 3], 2, 1, 2, 1),
    "15 cells": ((5, 3), [2, 2], 1, 1, 2, 1),
    "16 cells": ((4, 4), [3, 2], 2, 2, 2, 1),
    "17 cells": ((17, 1), [4, 4], 3, 2, 2, 1),
    "33 cells, past the slots": ((11, 3), [8, 8], 3, 4, 2, 1),
    "33 cells q2": ((11, 3), [4, 3], 2, 2, 2, 2),
    "31 hexes": ((31, 1, 1), [2, 2, 2], 2, 2, 3, 1),
    "36 hexes, past the slots": ((4, 3, 3), [4, 4, 4], 3, 4, 3, 1),
    "18 hexes q2": ((3, 3, 2), [2, 2, 2], 2, 1, 3, 2),
}


def _setup(case):
    n, q, mx, per, dim, deg = CASES[case]
    ext = [0.2 * k for k in n]
    m = M.quad_2d(*n, (0.0, 0.0), tuple(ext), jitter=0.1, seed=3) if dim == 2 else \
        M.box_3d(*n, (0.0, 0.0, 0.0), tuple(ext), jitter=0.1, seed=3)
    if deg == 2:
        m = M.q2(m)
    rng = np.random.default_rng(9)
    V = np.array([0.8, 0.3, 0.2])[:dim, None] + rng.uniform(-0.3, 0.3, size=(dim, m.n_dofs))
    cell, xi = M.jittered_lattice(m, q, 0.0, 1)
    cell, xi = np.repeat(cell, per), np.repeat(xi, per, axis=0)
    xi = np.clip(xi + rng.uniform(-0.2, 0.2, size=xi.shape) / np.array(q), 0.0, 1.0)
    keep = cell != m.n_cells // 2 if m.n_cells > 4 else np.ones(len(cell), bool)   # one cell starts empty
    return m, V, q, mx, cell[keep], xi[keep]


@pytest.mark.parametrize("case", list(CASES))
def test_fp64_bitwise(case):
    m, V, q, mx, cell, xi = _setup(case)
    g = ParticleStage(m, 0.05, 4, mx, q, FP64, capacity=20000)
    o = Oracle(m, 0.05, 4, mx, q)
    for s in (g, o):
        s.upload_fields(V, V)
        s.insert_particles(cell, xi)
    for step in range(3):
        assert bitwise_equal(g.step(download=True), o.step()), step
    assert_particles_match(g.particles(), o.particles(), 0.0, case, bitwise=True)
    assert np.array_equal(g.cell_counts(), o.cell_counts())
    g.close()


@pytest.mark.parametrize("case", list(CASES))
def test_fp32_fused_equals_separate(case):
    m, V, q, mx, cell, xi = _setup(case)
    a, b = (ParticleStage(m, 0.05, 4, mx, q, FP32_MIXED, capacity=20000) for _ in range(2))
    for s in (a, b):
        s.upload_fields(V, V)
        s.insert_particles(cell, xi)
    for step in range(3):
        Va = a.step(download=True)
        b.correct_particles_velocities()
        b.move_particles()
        assert bitwise_equal(Va, b.distribute_particle_velocities_to_grid()), step
    assert_particles_match(a.particles(), b.particles(), 0.0, case, bitwise=True)
    assert a.stats() == b.stats()
    a.close()
    b.close()

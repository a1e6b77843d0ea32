"""The own-cell test's closed form (closed_form in pf2_geom.hpp) on the cell
shapes that take each of its branches, bitwise against the oracle: general
quads, rectangles (|b| = sqrt(disc)), parallelograms (a near 0), cells whose
local x axis runs along global y (the divisor of xi_0 from the y
coordinates), coordinates far from the origin, and lengths at which the
discriminant leaves the middle exponent range (the general path decides)."""
import numpy as np
import pytest

from pfem2_amd import FP64, ParticleStage
from pfem2_amd import mesh as M
from oracle_binding import Oracle
from parity_util import assert_particles_match, bitwise_equal

pytestmark = pytest.mark.gpu


def _mesh(shape):
    m = M.quad_2d(9, 7, (0.0, 0.0), (1.8, 1.4), jitter=0.2 if shape == "general" else 0.0, seed=5)
    X = m.vertices.copy()
    size = 1.0
    if shape == "parallelogram":
        c, s = np.cos(0.5), np.sin(0.5)
        X = np.stack([c * X[:, 0] - s * X[:, 1] + 0.3 * X[:, 1], s * X[:, 0] + c * X[:, 1]], axis=1)
    elif shape == "turned":
        X = np.stack([-X[:, 1], X[:, 0]], axis=1)
    elif shape == "far":
        X = X + np.array([1.0e7, -3.0e6])
    elif shape in ("tiny", "tinier", "huge"):
        size = {"tiny": 1e-40, "tinier": 1e-47, "huge": 1e47}[shape]
        X = X * size
    m.vertices = np.ascontiguousarray(X)
    return m, size


@pytest.mark.parametrize("shape", ["general", "rectangle", "parallelogram", "turned", "far", "tiny", "tinier", "huge"])
def test_cell_shapes_bitwise(shape):
    m, size = _mesh(shape)
    rng = np.random.default_rng(11)
    V = size * (np.array([[0.9], [0.4]]) + rng.uniform(-0.5, 0.5, size=(2, m.n_dofs)))
    if shape == "rectangle":
        V[1, ::3] = 0.0   # some particles stay on one coordinate line
    g = ParticleStage(m, 0.1, 6, 2, [3, 3], FP64)
    o = Oracle(m, 0.1, 6, 2, [3, 3])
    cell, xi = M.jittered_lattice(m, [3, 3], 0.1, 7)
    # corners and edges of the unit square: zero and extreme quotients
    edge = np.array([[0.0, 0.0], [1.0, 1.0], [0.0, 0.5], [0.5, 0.0], [1.0, 0.25]])
    cell = np.concatenate([cell, np.repeat(np.arange(5, dtype=np.int32) * 3, len(edge))])
    xi = np.concatenate([xi, np.tile(edge, (5, 1))])
    for s in (g, o):
        s.upload_fields(V, V)
        s.insert_particles(cell, xi)
    for step in range(3):
        Vg, Vo = g.step(download=True), o.step()
        assert bitwise_equal(Vg, Vo), step
    assert_particles_match(g.particles(), o.particles(), 0.0, shape, bitwise=True)
    sg, so = g.stats(), o.stats()
    assert sg["searches"] == so["searches"] and sg["lost"] == so["lost"] and sg["deleted"] == so["deleted"]
    g.close()


@pytest.mark.parametrize("degree", [1, 2])
@pytest.mark.parametrize("shape", ["general", "box", "sheared", "far", "tiny", "large"])
def test_hexahedron_shapes_bitwise(shape, degree):
    """The tabulated inverse map of hexahedra (hex_map): affine cells that end
    at its early out, general ones through its Newton iteration, residuals
    near the rounding of far coordinates, small and large lengths."""
    m = M.box_3d(5, 4, 3, (0.0, 0.0, 0.0), (1.0, 0.8, 0.6), jitter=0.0 if shape in ("box", "sheared") else 0.2, seed=4)
    X, size = m.vertices.copy(), {"tiny": 1e-60, "large": 1e60}.get(shape, 1.0)
    if shape == "sheared":
        X[:, 0] += 0.3 * X[:, 1] - 0.2 * X[:, 2]
    if shape == "far":
        X += np.array([2.0e5, -1.0e5, 3.0e4])
    m.vertices = np.ascontiguousarray(size * X)
    if degree == 2:
        m = M.q2(m)
    rng = np.random.default_rng(12)
    V = size * (np.array([[0.7], [0.3], [-0.2]]) + rng.uniform(-0.4, 0.4, size=(3, m.n_dofs)))
    g = ParticleStage(m, 0.1, 5, 2, [2, 2, 2], FP64)
    o = Oracle(m, 0.1, 5, 2, [2, 2, 2])
    cell, xi = M.jittered_lattice(m, [2, 2, 2], 0.1, 7)
    edge = np.array([[0.0, 0.0, 0.0], [1.0, 1.0, 1.0], [0.0, 0.5, 1.0]])
    cell = np.concatenate([cell, np.repeat(np.arange(5, dtype=np.int32) * 3, len(edge))])
    xi = np.concatenate([xi, np.tile(edge, (5, 1))])
    for s in (g, o):
        s.upload_fields(V, V)
        s.insert_particles(cell, xi)
    for step in range(3):
        assert bitwise_equal(g.step(download=True), o.step()), step
    assert_particles_match(g.particles(), o.particles(), 0.0, shape, bitwise=True)
    assert g.stats()["searches"] == o.stats()["searches"] and g.stats()["lost"] == o.stats()["lost"]
    g.close()

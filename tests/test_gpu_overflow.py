"""A regroup that needs more particles than the capacity on meshes of many
write workgroups (RegroupShape::CB = 16 cells, 32 degree-1 hexahedra): the
range is cut in the middle of a workgroup, the workgroups behind it start past
the capacity, and some start after the flag is raised.  Likewise cells past the
census limit among many that k_cell_big counts.  Every wavefront of a
workgroup has to take the same decision on the flag that its launch raises.  The
capacity error is reported, and the particles and fields of another handle, of
another member of the same batch, stay those of a run without the overflow."""
import numpy as np
import pytest

from parity_util import bitwise_equal
from pfem2_amd import FP32_MIXED, FP64, Batch, ParticleStage, Pf2Error
from pfem2_amd import mesh as M

pytestmark = pytest.mark.gpu


def _one_cell(m, q, n=64):
    """n particles in cell 0: the reseed fills all other cells."""
    rng = np.random.default_rng(41)
    return np.zeros(n, dtype=np.int32), rng.uniform(0.05, 0.95, size=(n, m.dim))


def _every_third(m, q):
    """Every third cell crowded past its slot row, the others empty."""
    cell, xi = M.jittered_lattice(m, q, 0.0, 1)
    keep = cell % 3 == 0
    return np.repeat(cell[keep], 4), np.repeat(xi[keep], 4, axis=0)


CASES = {   # mesh, lattice, MAX, inserted particles, capacity as a share of the lattice points
    "800 quads": (lambda: M.quad_2d(40, 20, (0.0, 0.0), (2.0, 1.0), jitter=0.1, seed=3), [2, 2], 3, _one_cell, 0.53),
    "34,000 quads": (lambda: M.quad_2d(200, 170, (0.0, 0.0), (2.0, 1.7)), [2, 2], 3, _one_cell, 0.53),
    "99 quads past the slots": (lambda: M.quad_2d(11, 9, (0.0, 0.0), (1.1, 0.9)), [8, 8], 3, _every_third, 1.34),
    "800 quads q2": (lambda: M.q2(M.quad_2d(40, 20, (0.0, 0.0), (2.0, 1.0))), [2, 2], 3, _one_cell, 0.47),
    "768 hexes": (lambda: M.box_3d(12, 8, 8, (0.0, 0.0, 0.0), (1.2, 0.8, 0.8), jitter=0.1, seed=3), [2, 2, 2], 3,
                  _one_cell, 0.53),
    "768 hexes q2": (lambda: M.q2(M.box_3d(12, 8, 8, (0.0, 0.0, 0.0), (1.2, 0.8, 0.8))), [2, 2, 2], 3, _one_cell, 0.47),
}


def _overflowing(case, precision):
    """A handle whose first step overflows, and its field."""
    mesh, q, mx, insert, share = CASES[case]
    m = mesh()
    points = m.n_cells * int(np.prod(q))
    cap = int(share * points)
    cell, xi = insert(m, q)
    # what the census leaves: up to MAX of each occupied part, one in every other
    part = cell.astype(np.int64) * np.prod(q) + np.minimum((xi * q).astype(int), np.array(q) - 1) @ \
        np.cumprod([1] + list(q))[:m.dim]
    n = np.bincount(part, minlength=points)
    assert len(cell) <= cap < np.minimum(np.maximum(n, 1), mx).sum()
    V = M.uniform_field(m, [0.0] * m.dim)
    g = ParticleStage(m, 0.01, 2, mx, q, precision, capacity=cap)
    g.upload_fields(V, V)
    g.insert_particles(cell, xi)
    return g, V


def _bystander(dim, precision, seed):
    m = M.quad_2d(30, 12, (0.0, 0.0), (1.5, 0.6), jitter=0.1, seed=seed) if dim == 2 else \
        M.box_3d(8, 6, 6, (0.0, 0.0, 0.0), (0.8, 0.6, 0.6), jitter=0.1, seed=seed)
    V = M.uniform_field(m, [0.4, 0.2, 0.1][:dim])
    s = ParticleStage(m, 0.02, 4, 2, [3, 3, 2][:dim], precision)
    s.upload_fields(V, V)
    s.seed_particles()
    return s, V


def _assert_same(a, b):
    pa, pb = a.particles(), b.particles()
    for key in ("cell", "id", "x", "xi", "v"):
        assert np.array_equal(pa[key], pb[key]), key
    assert bitwise_equal(a.download_field(), b.download_field())
    assert a.stats() == b.stats()


@pytest.mark.parametrize("separate", [False, True])
@pytest.mark.parametrize("precision", [FP64, FP32_MIXED])
@pytest.mark.parametrize("case", list(CASES))
def test_overflow_over_many_workgroups(case, precision, separate):
    dim = 3 if "hex" in case else 2
    a, _ = _bystander(dim, precision, 5)
    b, _ = _bystander(dim, precision, 5)
    g, _ = _overflowing(case, precision)
    a.step()
    for _ in range(3):   # the later ones start in a dead state
        if separate:
            g.correct_particles_velocities()
            g.move_particles()
            g.distribute_particle_velocities_to_grid(download=False)
        else:
            g.step()
    a.step()
    for call in (g.n_global_particles, g.cell_counts, g.particles, lambda: g.step(download=True)):
        with pytest.raises(Pf2Error, match="capacity"):
            call()
    g.close()
    b.step()
    b.step()
    _assert_same(a, b)
    a.close()
    b.close()


@pytest.mark.parametrize("precision", [FP64, FP32_MIXED])
@pytest.mark.parametrize("case", ["800 quads", "34,000 quads", "768 hexes"])
def test_overflow_of_a_batch_member(case, precision):
    import torch
    dim = 3 if "hex" in case else 2
    solo, bat = ([_bystander(dim, precision, 5 + k) for k in range(2)] for _ in range(2))
    g, Vg = _overflowing(case, precision)
    members = [bat[0][0], g, bat[1][0]]
    fields = [torch.from_numpy(np.ascontiguousarray(V)).to("cuda") for V in (bat[0][1], Vg, bat[1][1])]
    torch.cuda.synchronize()
    b = Batch(3)
    for _ in range(3):
        b.step(members, [f.data_ptr() for f in fields])
        for (s, _), f in zip(solo, (fields[0], fields[2])):
            s.step_with_field(f.data_ptr())
    with pytest.raises(Pf2Error, match="capacity"):
        g.n_global_particles()
    for (s, _), (t, _) in zip(solo, bat):
        _assert_same(s, t)
    b.close()
    g.close()


def _crowded(shape, precision):
    """Cells of more than 2048 particles among cells that the census lists for
    k_cell_big: fewer of them than its workgroups, or more."""
    nx, ny = {"few": (33, 3), "many": (300, 8)}[shape]
    m = M.quad_2d(nx, ny, (0.0, 0.0), (0.1 * nx, 0.1 * ny), jitter=0.1, seed=8)
    rng = np.random.default_rng(43)
    per = np.array([66, 100, 130, 300, 128, 20])[np.arange(m.n_cells) % 6]
    per[[5, m.n_cells // 2, m.n_cells - 3]] = 2100
    cell = np.repeat(np.arange(m.n_cells, dtype=np.int32), per)
    V = M.uniform_field(m, [0.6, 0.1])
    g = ParticleStage(m, 0.05, 3, 20, [4, 4], precision, capacity=2 * len(cell))
    g.upload_fields(V, V)
    g.insert_particles(cell, rng.uniform(0.02, 0.98, size=(len(cell), 2)))
    return g, V


@pytest.mark.parametrize("batch", [False, True])
@pytest.mark.parametrize("precision", [FP64, FP32_MIXED])
@pytest.mark.parametrize("shape", ["few", "many"])
def test_crowded_cells_among_listed_ones(shape, precision, batch):
    import torch
    a, V = _bystander(2, precision, 5)
    b, _ = _bystander(2, precision, 5)
    g, Vg = _crowded(shape, precision)
    fields = [torch.from_numpy(np.ascontiguousarray(f)).to("cuda") for f in (Vg, V)]
    torch.cuda.synchronize()
    bt = Batch(2)
    for _ in range(3):
        if batch:
            bt.step([g, a], [f.data_ptr() for f in fields])
        else:
            g.step_with_field(fields[0].data_ptr())
            a.step_with_field(fields[1].data_ptr())
        b.step_with_field(fields[1].data_ptr())
    with pytest.raises(Pf2Error, match="2048"):
        g.n_global_particles()
    _assert_same(a, b)
    bt.close()
    for s in (a, b, g):
        s.close()


@pytest.mark.parametrize("precision", [FP64, FP32_MIXED])
@pytest.mark.parametrize("case", ["800 quads", "34,000 quads", "768 hexes"])
def test_overflow_of_a_pending_layout(case, precision):
    """The new particles of a mesh move exceed the capacity: the host's estimate
    (the 64 inserted) leaves room for a full reseed, but the step before has
    reseeded the whole mesh, and the stretched mesh needs more at its rim."""
    mesh, q, mx, insert, _ = CASES[case]
    m = mesh()
    cell, xi = insert(m, q)
    V = M.uniform_field(m, [0.02, 0.01, 0.01][:m.dim])
    mid = 0.5 * (m.vertices.min(axis=0) + m.vertices.max(axis=0))
    X = mid + (m.vertices - mid) * (1.0 + 0.6 / max(round(m.n_cells ** (1.0 / m.dim)), 12))
    cap = len(cell) + m.n_cells * int(np.prod(q))
    a, _ = _bystander(m.dim, precision, 5)
    b, _ = _bystander(m.dim, precision, 5)
    full, g = (ParticleStage(m, 0.01, 2, mx, q, precision, keep_velocity_ext=True, capacity=c) for c in (4 * cap, cap))
    for s in (full, g):
        s.upload_fields(V, V)
        s.insert_particles(cell, xi)
        s.set_profiling()
        s.step()
        s.move_mesh(X)
        assert s.kernel_times()["k_cell_pend"][1] == 1
    assert full.n_global_particles() > cap
    a.step()
    g.step()
    g.move_mesh(m.vertices)
    g.step()
    with pytest.raises(Pf2Error, match="capacity"):
        g.n_global_particles()
    b.step()
    _assert_same(a, b)
    for s in (a, b, full, g):
        s.close()

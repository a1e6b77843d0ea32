"""The search's refilling lanes over queues from a few entries to several
chunks per segment, with particles that cross many cells in a step: FP64
bitwise against the oracle, and a batched FP32-mixed step (its own grid and
segments) bitwise against the step of each handle alone."""
import numpy as np
import pytest

from pfem2_amd import FP32_MIXED, FP64, Batch, ParticleStage
from pfem2_amd import mesh as M
from oracle_binding import Oracle
from parity_util import assert_particles_match, bitwise_equal

pytestmark = pytest.mark.gpu

# cells, particles per direction: a queue below one wavefront; near one chunk a
# segment; more chunks than segments; more entries than the grid has lanes
SIZES = [(3, 2, 2), (40, 10, 3), (120, 60, 4), (300, 100, 4)]


def _sim(nx, ny, q, precision, seed=3):
    m = M.quad_2d(nx, ny, (0.0, 0.0), (1.0 * nx, 1.0 * ny), jitter=0.15, seed=seed)
    rng = np.random.default_rng(seed)
    V = np.array([[1.0], [0.3]]) + rng.uniform(-0.4, 0.4, size=(2, m.n_dofs))
    st = ParticleStage(m, 4.0, 7, 3, [q, q], precision)   # several cells a step
    st.upload_fields(V, V)
    st.seed_particles()
    return m, V, st


@pytest.mark.parametrize("nx,ny,q", SIZES)
def test_fp64_bitwise(nx, ny, q):
    m, V, g = _sim(nx, ny, q, FP64)
    o = Oracle(m, 4.0, 7, 3, [q, q])
    o.upload_fields(V, V)
    o.seed_particles()
    for step in range(2):
        Vg, Vo = g.step(download=True), o.step()
        assert bitwise_equal(Vg, Vo), step
    assert_particles_match(g.particles(), o.particles(), 0.0, f"{nx}x{ny}", bitwise=True)
    assert g.stats()["searches"] == o.stats()["searches"]
    g.close()


def test_fp32_batch_equals_single():
    import torch

    alone = [_sim(*s, FP32_MIXED) for s in SIZES]
    group = [_sim(*s, FP32_MIXED) for s in SIZES]
    fields = [torch.from_numpy(np.ascontiguousarray(V)).to("cuda") for _, V, _ in alone]
    torch.cuda.synchronize()
    b = Batch(len(group))
    for step in range(2):
        b.step([st for _, _, st in group], [f.data_ptr() for f in fields])
        for (_, _, st), f in zip(alone, fields):
            st.step_with_field(f.data_ptr())
    for (_, _, s), (_, _, t) in zip(alone, group):
        ps, pt = s.particles(), t.particles()
        for k in ("cell", "id", "xi", "v"):
            assert np.array_equal(ps[k], pt[k]), k
        assert np.array_equal(s.download_field(), t.download_field())
        i, j = s.step_info(), t.step_info()
        assert i == j and i["queued"][0] >= i["queued"][1] > 0
        s.close()
        t.close()

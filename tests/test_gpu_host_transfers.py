"""Fields through the pinned staging blocks: sizes up to a block (1 MiB), one
that only the upload fits in, and one past it (the pageable copy); more threads
than blocks; handles that come and go."""
import threading

import numpy as np
import pytest

from pfem2_amd import FP32_MIXED, FP64, ParticleStage, Pf2Error, _mesh_struct
from pfem2_amd import mesh as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(3, 2), (255, 255), (256, 256)])
@pytest.mark.parametrize("precision", [FP64, FP32_MIXED])
def test_round_trip(nx, ny, precision):
    m = M.quad_2d(nx, ny, (0.0, 0.0), (1.0, 1.0))
    st = ParticleStage(m, 0.001, 2, 1, [1, 1], precision)
    for seed in range(3):
        V = np.random.default_rng(seed).normal(size=(2, m.n_dofs))
        st.upload_fields(V, V)
        assert np.array_equal(st.download_field(), V)
    st.close()


def test_three_dimensional():
    m = M.box_3d(7, 5, 4, (0, 0, 0), (1.0, 1.0, 1.0))
    st = ParticleStage(m, 0.001, 2, 1, [1, 1, 1], FP64)
    V = np.random.default_rng(1).normal(size=(3, m.n_dofs))
    st.upload_fields(V, V)
    assert np.array_equal(st.download_field(), V)
    st.close()


def test_threads():
    wrong = []

    def work(k):
        m = M.quad_2d(20 + 9 * k, 30, (0.0, 0.0), (1.0, 1.0))
        st = ParticleStage(m, 0.001, 2, 1, [2, 2], FP64)
        st.upload_fields(np.zeros((2, m.n_dofs)), np.zeros((2, m.n_dofs)))
        st.seed_particles()
        for i in range(20):
            V = np.random.default_rng(100 * k + i).normal(size=(2, m.n_dofs))
            st.upload_fields(V, None)
            if not np.array_equal(st.download_field(), V) or st.n_global_particles() != 4 * m.n_cells:
                wrong.append((k, i))
        st.close()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(12)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.parametrize("upload", [False, True])
def test_block_is_kept_while_a_kernel_uses_it(upload):
    """A call that reports an error left by an earlier HIP call of the thread
    has launched its transfer all the same: it returns (and gives its block to
    other threads) only when that is done."""
    import ctypes

    import torch
    m = M.quad_2d(200, 200, (0.0, 0.0), (1.0, 1.0))
    stream = torch.cuda.Stream()
    st = ParticleStage(m, 0.001, 2, 1, [1, 1], FP64)
    lib, own = st._lib, st._h
    ms, h = _mesh_struct(m, st._arrays), ctypes.c_void_p()
    assert lib.pf2_create_in(ctypes.byref(ms), ctypes.byref(st._params), 0, None, 0, stream.cuda_stream,
                             ctypes.byref(h)) == 0
    st._h = h   # the same stage on a stream that can be asked
    lib.pf2_destroy(own)
    V = np.random.default_rng(5).normal(size=(2, m.n_dofs))
    st.upload_fields(V, V)
    st.synchronize()
    with torch.cuda.stream(stream):   # about 0.1 s of work ahead of the transfer
        a = torch.randn(4096, 4096, device="cuda")
        for _ in range(60):
            a = (a @ a).clamp(-1.0, 1.0)
    assert lib.hipSetDevice(ctypes.c_int(9999)) != 0
    try:
        st.upload_fields(V, None) if upload else st.download_field()
    except Pf2Error:
        assert stream.query()
    assert np.array_equal(st.download_field(), V)
    st.close()

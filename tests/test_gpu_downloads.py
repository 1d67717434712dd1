"""Downloads of device buffers to host arrays at sizes around the pinned ring's
chunks (256 KB to 2 MB, four of them): every element, after the ring has grown
and with a destination that is pinned itself."""
import sys

import numpy as np
import pytest

import miniafqmc_amd as m
from miniafqmc_amd import _native as nat

pytestmark = pytest.mark.gpu


def test_download_sizes(require_gpu):
    # bytes of W: 32 M N nw; M = 64, N = 32 gives 64 KB a walker
    for nw in (1, 2, 4, 15, 16, 17, 31, 32, 33, 64, 65, 255, 256, 257, 300, 700):
        print("download", nw, flush=True)
        sys.stdout.flush()
        s = m.make_system(64, 32, 2, density=1.0, sigma_L=0.01, sigma_h=1.0, dt=0.005, seed=1)
        g = m.AfqmcSys(s, nw, "fp64_dense", dense_exchange=False)
        n = nw * 2 * 64 * 32
        W = (np.arange(n) + 1j * np.arange(n, 0, -1)).reshape(nw, 2, 64, 32) + 0.25
        g.set(nat.BUF_W, W)
        for _ in range(2):
            assert np.array_equal(g.W, W)
        G = g.calculate_mixed_density_matrix()  # a transposed download
        assert np.array_equal(G, g.get(nat.BUF_G))
        wd = g.W_data
        assert wd.shape == (nw, 8)
        g.close()


def test_download_to_pinned_memory(require_gpu):
    import torch
    s = m.make_system(64, 32, 2, density=1.0, sigma_L=0.01, sigma_h=1.0, dt=0.005, seed=1)
    nw = 40
    g = m.AfqmcSys(s, nw, "fp64_dense", dense_exchange=False)
    W = np.random.default_rng(3).standard_normal((nw, 2, 64, 32)) + 0j
    g.set(nat.BUF_W, W)
    out = torch.empty(nw, 2, 64, 32, dtype=torch.complex128, pin_memory=True).numpy()
    nat.check(nat.lib.afqmc_copy(g.ctx, nat.BUF_W, 0, out.ctypes.data_as(nat.C.POINTER(nat.C.c_double))))
    assert np.array_equal(out, W)
    g.close()


def test_downloads_from_several_threads(require_gpu):
    """Contexts of their own in four threads download at the same time, twice,
    with the last context of each round giving the shared rings back."""
    import threading
    bad = []

    def one(seed):
        try:
            nw = 200 + seed
            s = m.make_system(64, 32, 2, density=1.0, sigma_L=0.01, sigma_h=1.0, dt=0.005, seed=1)
            g = m.AfqmcSys(s, nw, "fp64_dense", dense_exchange=False)
            W = np.random.default_rng(seed).standard_normal((nw, 2, 64, 32)) + 1j
            g.set(nat.BUF_W, W)
            for _ in range(5):
                if not np.array_equal(g.W, W):
                    bad.append(seed)
            g.close()
        except Exception as e:  # reported by the main thread
            bad.append(e)

    for _ in range(2):
        th = [threading.Thread(target=one, args=(k,)) for k in range(4)]
        for t in th:
            t.start()
        for t in th:
            t.join()
    assert not bad, bad

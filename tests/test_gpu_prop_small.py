"""The one-kernel propagator of small systems against the chain of products
(forced by a GEMM tile): the same walkers bit for bit in FP32 and split-BF16,
1e-13 relative in FP64 (other summation groups), at one row tile and less, at
wave counts and their remainders, odd M (unaligned rows), column blocks that
end inside a spin or past the last column, few and many walkers."""
import sys

import numpy as np
import pytest

import miniafqmc_amd as m
from miniafqmc_amd import _native as nat

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("mode", ["fp64_dense", "fp64_csr", "mixed_fp32", "mixed_bf16"])
@pytest.mark.parametrize("M,N,nw", [(5, 2, 1), (31, 7, 40), (32, 16, 300), (33, 9, 3), (64, 33, 130), (95, 24, 17),
                                    (100, 31, 5), (128, 8, 257), (150, 37, 2), (176, 20, 9), (192, 48, 33)])
def test_small_propagator_matches_chain(require_gpu, mode, M, N, nw):
    if mode.startswith("fp64") and M > 128:
        pytest.skip("the FP64 kernel ends at 128 orbitals")
    say("small propagator", mode, M, N, nw)
    s = m.make_system(M, N, 6, density=1.0, sigma_L=0.3 / M ** 0.5, sigma_h=1.0, dt=0.005, seed=M)
    r = np.random.default_rng(nw)
    V = 0.3 * (r.standard_normal((M * M, nw)) + 1j * r.standard_normal((M * M, nw))) / M ** 0.5
    W = r.standard_normal((nw, 2, M, N)) + 1j * r.standard_normal((nw, 2, M, N))
    out = []
    for tile in (0, 1):
        g = m.AfqmcSys(s, nw, mode, energy_precision=0, dense_exchange=False)
        g.set_tile(tile)
        g.set(nat.BUF_W, W)
        g.set(nat.BUF_VHS, V)
        g.profile(True)
        g.propagate()
        st = g.kernel_stats()
        assert ("prop_fused" in st) == (tile == 0) and ("prop_taylor" in st) == (tile == 1)
        out.append(g.W)
        g.close()
    if mode.startswith("fp64"):
        assert np.abs(out[0] - out[1]).max() <= 1e-13 * np.abs(out[1]).max()
    else:
        assert np.array_equal(out[0], out[1]), np.abs(out[0] - out[1]).max()


@pytest.mark.parametrize("M,N,nw", [(208, 13, 3), (224, 56, 40), (256, 1, 5), (272, 70, 2)])
def test_ring_propagator_walkers_as_columns(require_gpu, M, N, nw):
    """Above the one-kernel sizes, split-BF16: the products that take walkers
    and spins as columns (folded output columns, tiles that end inside a
    spin) against the register-staged products per walker and spin, and every
    ring tile, bit for bit."""
    say("ring propagator", M, N, nw)
    s = m.make_system(M, N, 6, density=1.0, sigma_L=0.3 / M ** 0.5, sigma_h=1.0, dt=0.005, seed=M)
    r = np.random.default_rng(nw)
    V = 0.3 * (r.standard_normal((M * M, nw)) + 1j * r.standard_normal((M * M, nw))) / M ** 0.5
    W = r.standard_normal((nw, 2, M, N)) + 1j * r.standard_normal((nw, 2, M, N))
    out = []
    for level, tile in ((0, 0), (2, 0), (2, 1), (2, 2), (2, 3), (2, 4), (2, 5)):
        g = m.AfqmcSys(s, nw, "mixed_bf16", energy_precision=0, dense_exchange=False)
        g.set_direct_lds(level)
        g.set_tile(tile)
        g.set(nat.BUF_W, W)
        g.set(nat.BUF_VHS, V)
        g.propagate()
        out.append(g.W)
        g.close()
    for o in out[1:]:
        assert np.array_equal(o, out[0]), np.abs(o - out[0]).max()

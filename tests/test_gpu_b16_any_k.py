"""Split-BF16 products whose sums end inside a k-tile of 16, on rows padded to
pairs (staged-ring kernel) against the register-staged products on the same
padded rows: X, the HS potential and the walkers bit for bit, the potential
also after a round trip through the host, and the energies against FP64.
Sizes: one k-tile and less, remainders 1, 2, 9 and 15 of M and K, odd and even
N*M (odd stays on the register path)."""
import sys

import numpy as np
import pytest

import miniafqmc_amd as m
from miniafqmc_amd import _native as nat

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("M,N,K,nw", [(6, 2, 9, 3), (45, 12, 99, 70), (94, 23, 161, 33), (193, 8, 65, 130), (194, 31, 143, 5),
                                      (201, 37, 90, 20), (223, 56, 402, 9), (250, 61, 111, 64)])
def test_ring_products_of_any_length(require_gpu, M, N, K, nw):
    s = m.make_system(M, N, K, density=0.5, sigma_L=0.02 * (64.0 * 256 / (M * K)) ** 0.5, seed=M)
    x = m.fields_block(M, K, nw, 0, 3)
    out = []
    for direct, tile in ((0, 0), (2, 0), (2, 6)):  # tile 6: 32 x 32, four stages
        say("any k", M, N, K, nw, "level", direct, "tile", tile)
        g = m.AfqmcSys(s, nw, "mixed_bf16", energy_precision=1)
        g.set_direct_lds(direct)
        g.set_tile(tile)
        g.init_walkers()
        g.stage_fields(x)
        g.run(1, 2, 5, s.dt, energy=False)
        r = [g.get(nat.BUF_X), g.get(nat.BUF_VHS), g.W]
        g.set(nat.BUF_VHS, r[1])
        g.set(nat.BUF_X, r[0])
        assert np.array_equal(g.get(nat.BUF_VHS), r[1]) and np.array_equal(g.get(nat.BUF_X), r[0])
        g.propagate()
        r.append(g.W)
        g.calculate_energy()
        e = g.W_data[:, 0]
        g.set(nat.BUF_W, r[2])
        g.calculate_mixed_density_matrix()
        g.calculate_energy()
        out.append((r, e, g.W_data[:, 0]))
        g.close()
    for o in out[1:]:
        for q, (a, b) in enumerate(zip(out[0][0], o[0])):
            assert np.array_equal(a, b), f"output {q}: max diff {np.abs(a - b).max():.3e}"
    ref = m.AfqmcSys(s, nw, "fp64_dense")
    ref.set(nat.BUF_W, out[0][0][2])
    ref.calculate_mixed_density_matrix()
    ref.calculate_energy()
    e64 = ref.W_data[:, 0]
    ref.close()
    for o in out:
        # operands of 16 bits and FP32 sums in the exchange, a part of E
        assert np.abs(o[2] - e64).max() <= 2.0 ** -15 * np.abs(e64).max()

"""The CSR products (csrmm semantics) on the GPU against dense numpy products,
over the row kernel's widths (16, 32 and 64 walkers per wave, a partial last
chunk), its waves per row (1, 4, 16 by the rows' length; rows without entries)
and the windowed kernel (sorted rows against an operand beyond the L2).
Tolerance: n-term FP64 sums, 1e-12 of the largest result."""
import sys

import numpy as np
import pytest

import miniafqmc_amd as m
from miniafqmc_amd import _native as nat

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def cn(r, shape):
    return r.standard_normal(shape) + 1j * r.standard_normal(shape)


def close(a, b):
    assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max()


@pytest.mark.parametrize("nw", [5, 16, 17, 64, 70])
@pytest.mark.parametrize("M,K,density", [(9, 1500, 0.9), (9, 500, 0.8), (12, 40, 0.1), (33, 70, 0.4)])
def test_csr_vhs_vs_dense(require_gpu, M, K, density, nw):
    say("csr vHS", M, K, density, nw)
    s = m.make_system(M, 2, K, density=density, sigma_L=0.03, sigma_h=1.0, dt=0.005, seed=M + K)
    X = cn(np.random.default_rng(nw), (K, nw))
    g = m.AfqmcSys(s, nw, "fp64_csr")
    g.set(nat.BUF_X, X)
    V = g.get_vHS()
    g.close()
    close(V, s.spvn.dense() @ X)


@pytest.mark.parametrize("M,N,K,nw,density", [(96, 4, 1024, 256, 0.2), (40, 4, 30, 20, 0.9), (13, 3, 100, 130, 0.5)])
def test_csr_full_bias_vs_dense(require_gpu, M, N, K, nw, density):
    """T(Spvn) times the full density matrix; the first shape takes the
    windowed kernel (1024 rows, 9216 columns x 256 walkers)."""
    say("csr full bias", M, N, K, nw, density)
    s = m.make_system(M, N, K, density=density, sigma_L=0.03, sigma_h=1.0, dt=0.005, seed=M + K)
    g = m.AfqmcSys(s, nw, "fp64_csr", transposed=False)
    g.init_walkers()
    g.calculate_mixed_density_matrix_full()
    G = cn(np.random.default_rng(nw), (2 * M * M, nw))
    g.set(nat.BUF_GFULL, G)
    vb = g.get_vbias_full()
    g.close()
    close(vb, s.spvn.dense().T @ (G[:M * M] + G[M * M:]))

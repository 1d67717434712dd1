"""The FP64 products' folded operands, split sums and operand staging at sizes
where they can go wrong: row and column tiles that end inside a walker, a
last chunk of a split sum shorter than the others, k shorter than one k-tile,
operands aligned to 8 bytes only."""
import sys

import numpy as np
import pytest

import miniafqmc_amd as m
import oracle_lib as orc
from miniafqmc_amd import _native as nat
from test_zz_no_alloc import Hip, walkers

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("mode", ["fp64_dense", "fp64_csr"])
@pytest.mark.parametrize("M,N,K,nw", [(37, 19, 45, 7), (65, 33, 130, 65), (130, 5, 257, 3), (9, 3, 11, 33)])
def test_f64_ragged_step_vs_oracle(require_gpu, mode, M, N, K, nw):
    """Two substeps with an orthogonalisation and an energy against the oracle
    at the FP64 bound of the whole steps (1e-9 relative)."""
    say("f64 ragged", mode, M, N, K, nw)
    s = m.make_system(M, N, K, density=0.6, sigma_L=0.03, sigma_h=1.0, dt=0.005, seed=M + K)
    x = m.fields_block(5, K, nw, 0, 2)
    cutoff = 1e-6 if mode == "fp64_csr" else -1.0
    g = m.AfqmcSys(s, nw, mode, cutoff=cutoff)
    g.init_walkers()
    g.stage_fields(x)
    eav = g.run(1, 2, 1, s.dt)
    W, Wd = g.W, g.W_data
    g.close()
    eo, Wo, Wdo, _, _, info = orc.run(s, nw, 1, 2, 1, x, cutoff=cutoff)
    assert info == 0
    assert abs(eav[0] - eo[1]) <= 1e-9 * abs(eo[1])
    assert np.abs(W - Wo).max() <= 1e-9 * np.abs(Wo).max()
    assert np.abs(Wd[:, :5] - Wdo[:, :5]).max() <= 1e-9 * np.abs(Wdo[:, :5]).max()


@pytest.mark.parametrize("M,N,nw", [(40, 9, 5), (96, 24, 33)])
def test_noalloc_pointers_aligned_to_eight_bytes(require_gpu, M, N, nw):
    """Device pointers that are aligned to 8 bytes only give the aligned call's
    G and overlaps bit for bit."""
    say("no-alloc, 8-byte aligned", M, N, nw)
    s = m.make_system(M, N, 8, density=1.0, sigma_L=0.01, sigma_h=1.0, dt=0.005, seed=M)
    trial = np.stack([s.trial_alpha, s.trial_beta])
    W = walkers(s, nw, seed=M + N)
    hip = Hip()
    try:
        got = []
        for shift in (0, 8):
            ptr = []
            for a in (trial, W):
                p = hip.alloc(a.nbytes + 16) + shift
                a = np.ascontiguousarray(a)
                assert hip.lib.hipMemcpy(p, a.ctypes.data, a.nbytes, 1) == 0
                ptr.append(p)
            d_G, d_ov = hip.alloc(2 * N * M * nw * 16 + 16) + shift, hip.alloc(2 * nw * 16 + 16) + shift
            nat.check(nat.lib.afqmc_mixed_density_matrix_noalloc(M, N, nw, ptr[0], ptr[1], d_G, d_ov, None))
            assert hip.lib.hipDeviceSynchronize() == 0
            got.append((hip.download(d_G, (2 * N * M, nw)), hip.download(d_ov, (nw, 2))))
        assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
    finally:
        hip.free_all()

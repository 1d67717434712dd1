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


@pytest.mark.parametrize("mode,level,tol", [("fp64_dense", 1, 1e-11), ("mixed_bf16", 1, 5e-5), ("mixed_bf16", 2, 2e-6)])
@pytest.mark.parametrize("M,N,nw", [(16, 4, 3), (40, 8, 129), (64, 36, 65), (48, 45, 20)])
def test_exchange_in_one_launch_vs_cholesky_form(require_gpu, mode, level, tol, M, N, nw):
    """The exchange energy's work items (chunk, row tile, walker tile, spin)
    against the Cholesky form in FP64, per walker and relative to the largest
    exchange energy: N*M below one tile, one chunk, and a second chunk that
    is partial (2304, 2160 with chunks of 2048), at tile remainders of
    walkers.  Tolerances: FP64 sums; two-piece (16-bit) and three-piece
    (24-bit) operands of terms of one sign or another, a few times their
    rounding."""
    say("exchange", mode, level, M, N, nw)
    s = m.make_system(M, N, 32, density=0.7, sigma_L=0.05, sigma_h=1.0, dt=0.005, seed=M * N)
    W = walkers(s, nw, seed=nw)
    Wd = np.zeros((nw, 8), complex)
    Wd[:, 1] = 1.0
    ex = []
    for md, lv, dense in ((mode, level, True), ("fp64_dense", 1, False)):
        g = m.AfqmcSys(s, nw, md, energy_precision=lv, dense_exchange=dense, cutoff=-1.0)
        for tile in (0, 1, 2, 3, 5) if dense else (0,):
            g.set_tile(tile)
            g.set(nat.BUF_W, W)
            g.set(nat.BUF_WDATA, Wd)
            g.calculate_mixed_density_matrix()
            g.calculate_energy()
            ex.append(g.energy_terms()[:, 2])
        g.close()
    ref = ex.pop()
    for e in ex:
        assert np.abs(e - ref).max() <= tol * np.abs(ref).max()


@pytest.mark.parametrize("M,N,nw", [(9, 3, 5), (24, 6, 64), (37, 19, 67)])
def test_vakbl_dense_vs_csr(require_gpu, M, N, nw):
    """Vakbl kept dense gives the CSR product's energy terms; one whose entries
    repeat (each stored as two halves) keeps the CSR product, which adds them."""
    say("Vakbl dense", M, N, nw)
    s = m.make_system(M, N, 32, density=0.7, sigma_L=0.05, sigma_h=1.0, dt=0.005, seed=M * N, with_vakbl=True)
    full = s.vakbl
    twice = m.Csr(full.nrows, full.ncols, (2 * full.rowptr).astype(full.rowptr.dtype), np.repeat(full.col, 2),
                  np.repeat(full.val, 2) / 2)
    assert 2 * full.nnz >= full.nrows**2
    W = walkers(s, nw, seed=nw)
    Wd = np.zeros((nw, 8), complex)
    Wd[:, 1] = 1.0
    got = []
    for v, dense in ((full, False), (full, True), (twice, True)):
        s.vakbl = v
        g = m.AfqmcSys(s, nw, "fp64_csr", csr_dense=dense)
        g.set(nat.BUF_W, W)
        g.set(nat.BUF_WDATA, Wd)
        g.calculate_mixed_density_matrix()
        g.profile(True)
        g.calculate_energy()
        names = set(g.kernel_stats())
        g.profile(False)
        got.append(np.concatenate([g.energy_terms(), g.W_data[:, :1]], axis=1))
        g.close()
        assert ("csrmm_vakbl" in names) == (not dense or v is twice), sorted(names)
    for e in got[1:]:
        assert np.abs(e - got[0]).max() <= 1e-12 * np.abs(got[0]).max()


@pytest.mark.parametrize("N", [1, 2, 4, 5, 15, 16, 17, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 160, 256])
def test_batched_inverse_pivots(require_gpu, N):
    """Overlap matrices with prescribed pivot choices (the trial is the first N
    unit vectors, so a walker's top block is its overlap matrix): Gaussian
    entries, rows in reverse order (an interchange at every step), entries of
    exactly equal size (LAPACK takes the first), sizes 1e-200 and 1e200; inverse
    and determinant against numpy."""
    say("batched inverse", N)
    M = N + 3
    r = np.random.default_rng(N)

    def cn(*shape):
        return r.standard_normal(shape) + 1j * r.standard_normal(shape)

    T = [cn(N, N), cn(N, N)[::-1] + 8 * np.eye(N)[::-1], 1e-200 * cn(N, N), 1e200 * cn(N, N)]
    h = np.array([[1.0]])
    while h.shape[0] < N:
        h = np.block([[h, h], [h, -h]])
    T.append((h[:N, :N] + 1j * np.tril(h[:N, :N])) if N > 1 else np.array([[1 + 1j]]))
    s = m.make_system(M, N, 2, density=1.0, sigma_L=0.01, sigma_h=1.0, dt=0.005, seed=N)
    s.trial_alpha[:] = np.eye(M, N)
    s.trial_beta[:] = np.eye(M, N)
    nw = len(T)
    W = np.zeros((nw, 2, M, N), complex)
    for w in range(nw):
        W[w, 0, :N] = T[w].T  # T1[a][b] = W[b][a]
        W[w, 1, :N] = cn(N, N) + 3 * np.eye(N)
    W[:, :, N:] = 0.1
    g = m.AfqmcSys(s, nw, "fp64_dense", dense_exchange=False)
    g.set(nat.BUF_W, W)
    g.set(nat.BUF_WDATA, np.zeros((nw, 8), complex))
    G = g.calculate_mixed_density_matrix().reshape(2, N, M, nw)
    ov = g.W_data[:, 2:4]
    g.close()
    for w in range(nw):
        for sp in range(2):
            A = W[w, sp, :N].T
            sign, logd = np.linalg.slogdet(A / np.abs(A).max())
            logd += N * np.log(np.abs(A).max())
            inv = np.linalg.inv(A / np.abs(A).max()) / np.abs(A).max()
            cond = np.linalg.cond(A / np.abs(A).max())
            ref = inv @ W[w, sp].T
            assert np.abs(G[sp, :, :, w] - ref).max() <= 1e-14 * N * cond * np.abs(ref).max()
            if abs(logd) < 600:
                det = sign * np.exp(logd)
                assert abs(ov[w, sp] - det) <= 1e-13 * N * cond * abs(det)


@pytest.mark.parametrize("M,N,K,nw", [(8, 2, 4, 1), (50, 7, 62, 5), (51, 6, 62, 5), (64, 16, 100, 33),
                                      (90, 30, 150, 128), (200, 40, 134, 70)])
def test_f32_ring_matches_register_staged(require_gpu, M, N, K, nw):
    """FP32 products by direct LDS loads (every tile) against the kernel that
    stages through registers: the walkers are the same bits after two substeps
    (k that is no multiple of a k-tile, odd M), the energy terms, whose
    exchange is summed in another order, agree to FP64 rounding."""
    say("f32 ring", M, N, K, nw)
    s = m.make_system(M, N, K, density=0.5, sigma_L=0.03, sigma_h=1.0, dt=0.005, seed=7)
    x = m.fields_block(5, K, nw, 0, 2)
    got = []
    for direct, tile in ((0, 0), (2, 0), (2, 1), (2, 2), (2, 3)):
        g = m.AfqmcSys(s, nw, "mixed_fp32")
        nat.check(nat.lib.afqmc_set_option(g.ctx, nat.OPT_DIRECT_LDS, float(direct)))
        g.set_tile(tile)
        g.init_walkers()
        g.stage_fields(x)
        g.run(1, 2, 1, s.dt)
        got.append((g.W, g.energy_terms()))
        g.close()
    for W, e in got[1:]:
        assert np.array_equal(W, got[0][0])
        assert np.abs(e - got[0][1]).max() <= 1e-14 * np.abs(got[0][1]).max()


@pytest.mark.parametrize("N", [1, 3, 16, 17, 32, 33, 64, 65, 96, 97, 128, 129, 160, 256])
def test_batched_inverse_mixed_modes(require_gpu, N):
    """The mixed modes' inverse (pivot rows scaled as they are chosen):
    determinants in FP64, and G within the FP32 rounding of its operands and
    of a sum of N products; with interchanges at random and at every step."""
    say("batched inverse, mixed", N)
    M, nw = N + 3, 3
    r = np.random.default_rng(100 + N)
    s = m.make_system(M, N, 2, density=1.0, sigma_L=0.01, sigma_h=1.0, dt=0.005, seed=N)
    s.trial_alpha[:] = np.eye(M, N)
    s.trial_beta[:] = np.eye(M, N)
    W = 0.1 * (r.standard_normal((nw, 2, M, N)) + 1j * r.standard_normal((nw, 2, M, N)))
    W[:, 0, :N] += np.eye(N)
    W[:, 1, :N] += np.eye(N)[::-1]
    g = m.AfqmcSys(s, nw, "mixed_fp32", dense_exchange=False)
    g.set(nat.BUF_W, W)
    g.set(nat.BUF_WDATA, np.zeros((nw, 8), complex))
    G = g.calculate_mixed_density_matrix().reshape(2, N, M, nw)
    ov = g.W_data[:, 2:4]
    g.close()
    for w in range(nw):
        for sp in range(2):
            A = W[w, sp, :N].T
            inv, cond = np.linalg.inv(A), np.linalg.cond(A)
            bound = 2 * (2 * N + 4) * 2.0**-24 * (np.abs(inv) @ np.abs(W[w, sp].T))
            ref = inv @ W[w, sp].T
            assert np.all(np.abs(G[sp, :, :, w] - ref) <= bound + 1e-14 * N * cond * np.abs(ref).max())
            det = np.linalg.det(A)
            assert abs(ov[w, sp] - det) <= 1e-13 * N * cond * abs(det)

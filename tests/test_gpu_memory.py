"""Device memory that a context holds, by what hipMemGetInfo reports free.  The
runtime takes and returns memory of its own at times (scratch), so each figure
is the median of several contexts'."""
import gc
import sys

import numpy as np
import pytest

import miniafqmc_amd as m
from hip_rt import free_bytes

pytestmark = pytest.mark.gpu
MB = 1 << 20


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def median(run):
    """Of five runs, after one that loads the kernels."""
    run()
    gc.collect()
    d = [run() for _ in range(5)]
    say(d)
    return np.median(np.array(d), axis=0)


def test_dense_vakbl_allocates_at_upload_only(require_gpu):
    """With Vakbl kept dense the energy's workspace is there after the upload
    (two partial products, 101 MB here) and the CSR form's Y (50 MB) is not;
    the first energy allocates nothing."""
    M, N, K, nw = 64, 16, 64, 1536
    s = m.make_system(M, N, K, density=0.3, sigma_L=0.02, sigma_h=1.0, dt=0.005, seed=4, with_vakbl=True)

    def run(dense):
        f0 = free_bytes()
        g = m.AfqmcSys(s, nw, "fp64_csr", csr_dense=dense)
        g.init_walkers()
        f1 = free_bytes()
        g.calculate_mixed_density_matrix()
        f2 = free_bytes()
        g.calculate_energy()
        g.calculate_energy()
        d = f0 - f1, f2 - free_bytes()
        g.close()
        return d

    say("dense Vakbl")
    dense = median(lambda: run(True))
    say("CSR Vakbl")
    csr = median(lambda: run(False))
    assert abs(dense[1]) < 4 * MB and abs(csr[1]) < 4 * MB
    v = (2 * N * M) ** 2
    d = 16 * v + 2 * 16 * nw * 2 * N * M + 16 * K * 2 * N * M  # Vakbl, workspace, SpvnT
    c = 20 * s.vakbl.nnz + 16 * nw * 2 * N * M                 # Vakbl, Y
    assert abs(dense[0] - csr[0] - (d - c)) < 12 * MB, (dense, csr, d, c)


@pytest.mark.parametrize("mode,zs", [("fp64_dense", 16), ("mixed_fp32", 8), ("mixed_bf16", 8)])
def test_dense_exchange_holds_its_block_only(require_gpu, mode, zs):
    """The dense exchange block costs its own size at the upload, not the
    product's [walkers][N M] output beside it (33 or 17 MB here), which only
    the form in chunks writes: that one allocates it when it runs."""
    M, N, K, nw = 256, 4, 4, 2048
    s = m.make_system(M, N, K, density=1.0, sigma_L=0.02, sigma_h=1.0, dt=0.005, seed=4)

    def run(block):
        f0 = free_bytes()
        g = m.AfqmcSys(s, nw, mode, dense_exchange=block)
        d = f0 - free_bytes()
        g.close()
        return d

    say("dense exchange", mode)
    used = median(lambda: run(True)) - median(lambda: run(False))
    assert abs(used - 2 * zs * (N * M) ** 2) < 6 * MB, used
    if mode == "fp64_dense":
        return
    g = m.AfqmcSys(s, nw, mode)
    g.init_walkers()
    g.calculate_mixed_density_matrix()
    e = []
    for level in (2, 0):  # one launch, in chunks
        g.set_direct_lds(level)
        e.append(g.calculate_energy())
    g.close()
    assert abs(e[1] - e[0]) <= 1e-4 * abs(e[0])


@pytest.mark.parametrize("mode", ["fp64_dense", "fp64_csr", "mixed_bf16"])
@pytest.mark.parametrize("block", [True, False])
def test_energy_after_capture_allocates_nothing(require_gpu, mode, block):
    """The workspace of captured substeps (34 MB here) holds the energy's
    partial sums too: one energy after another, none takes memory."""
    M, N, K, nw = 96, 24, 128, 512
    s = m.make_system(M, N, K, density=0.3, sigma_L=0.02, sigma_h=1.0, dt=0.005, seed=4)
    x = m.fields_block(4, K, nw, 0, 4)

    def run():
        g = m.AfqmcSys(s, nw, mode, dense_exchange=block)
        g.init_walkers()
        g.stage_fields(x)
        g.use_graphs(True)
        for t in range(2):
            g.substep(t, False, s.dt)
        g.calculate_mixed_density_matrix()
        f0 = free_bytes()
        g.calculate_energy()
        g.substep(2, False, s.dt)
        g.calculate_mixed_density_matrix()
        g.calculate_energy()
        d = f0 - free_bytes()
        g.close()
        return d

    say("energy after capture", mode, block)
    # split-BF16's block has its two-piece G (19 MB) from the first energy on
    extra = 8 * 2 * N * M * nw if block and mode == "mixed_bf16" else 0
    assert abs(median(run) - extra) < 4 * MB

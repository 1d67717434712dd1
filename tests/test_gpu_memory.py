"""Device memory that a context holds, by what hipMemGetInfo reports free."""
import sys

import pytest

import miniafqmc_amd as m
from hip_rt import free_bytes

pytestmark = pytest.mark.gpu
MB = 1 << 20


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def test_dense_vakbl_allocates_at_upload_only(require_gpu):
    """With Vakbl kept dense the energy's workspace is there after the upload
    (two partial products, 101 MB here) and the CSR form's Y (50 MB) is not;
    the first energy allocates nothing."""
    M, N, K, nw = 64, 16, 64, 1536
    s = m.make_system(M, N, K, density=0.3, sigma_L=0.02, sigma_h=1.0, dt=0.005, seed=4, with_vakbl=True)
    used = {}
    for dense in (True, False, True):  # the first one loads the kernels
        say("vakbl dense", dense)
        f0 = free_bytes()
        g = m.AfqmcSys(s, nw, "fp64_csr", csr_dense=dense)
        g.init_walkers()
        f1 = free_bytes()
        g.calculate_mixed_density_matrix()
        f2 = free_bytes()
        g.calculate_energy()
        g.calculate_energy()
        used[dense] = f0 - f1, f1 - f2, f2 - free_bytes()
        g.close()
    say(used)
    assert used[True][2] == 0 and used[False][2] == 0, used
    v = (2 * N * M) ** 2
    dense = 16 * v + 2 * 16 * nw * 2 * N * M + 16 * K * 2 * N * M  # Vakbl, workspace, SpvnT
    csr = 20 * s.vakbl.nnz + 16 * nw * 2 * N * M                   # Vakbl, Y
    assert abs(used[True][0] - used[False][0] - (dense - csr)) < 12 * MB, (used, dense, csr)

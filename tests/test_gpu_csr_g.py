"""G of the FP64 CSR mode in and out (the reference's walker-last layout),
held walker-first on the device when only dense products read it."""
import sys

import numpy as np
import pytest

import miniafqmc_amd as m
from miniafqmc_amd import _native as nat

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def draw(M, N, nw, seed):
    r = np.random.default_rng(seed)
    return r.standard_normal((2 * N, M, nw)) + 1j * r.standard_normal((2 * N, M, nw))


@pytest.mark.parametrize("vakbl", [False, True])
@pytest.mark.parametrize("M,N,nw", [(24, 5, 1), (31, 7, 33), (40, 8, 64), (64, 16, 100)])
def test_g_round_trip_is_turned_on_the_device(require_gpu, M, N, nw, vakbl):
    say("G round trip", M, N, nw, vakbl)
    s = m.make_system(M, N, 30, density=0.5, sigma_L=0.03, sigma_h=1.0, dt=0.005, seed=M, with_vakbl=vakbl)
    G = draw(M, N, nw, nw).reshape(2 * N * M, nw)
    out = {}
    for dense in (True, False):  # walker-first, walker-last on the device
        g = m.AfqmcSys(s, nw, "fp64_csr", csr_dense=dense)
        g.profile(True)
        g.set(nat.BUF_G, G)
        assert np.array_equal(np.asarray(g.get(nat.BUF_G)).reshape(G.shape), G)
        n = g.kernel_stats().get("g_transpose", (0, 0.0))[0]
        assert n == (2 if dense else 0)
        g.profile(False)
        out[dense] = np.asarray(g.get_vbias())
        if vakbl:
            g.calculate_energy()  # the turned copy and the energy share a workspace
            assert np.array_equal(np.asarray(g.get(nat.BUF_G)).reshape(G.shape), G)
        g.close()
    d = np.abs(out[True] - out[False]).max()
    assert d <= 1e-12 * np.abs(out[False]).max()


@pytest.mark.parametrize("dense", [True, False])
def test_g_written_before_the_upload(require_gpu, dense):
    """Through the C entries: a G copied in before the system is the G that
    the bias product reads after it, whichever layout the upload settles on."""
    M, N, nw = 31, 7, 33
    s = m.make_system(M, N, 30, density=0.5, sigma_L=0.03, sigma_h=1.0, dt=0.005, seed=M)
    G = np.ascontiguousarray(draw(M, N, nw, 9).reshape(2 * N * M, nw))
    say("early G, dense", dense)
    want = m.AfqmcSys(s, nw, "fp64_csr", csr_dense=dense)
    want.set(nat.BUF_G, G)
    vb = np.asarray(want.get_vbias())
    want.close()
    arg = [np.ascontiguousarray(a) for a in (s.trial_alpha, s.trial_beta, s.propg1, s.haj)]
    ptr = [a.ctypes.data_as(nat.C.POINTER(nat.C.c_double)) for a in arg]
    h = nat.C.c_void_p()
    nat.check(nat.lib.afqmc_ctx_create(M, N, s.nchol, nw, nat.MODES["fp64_csr"], nat.C.byref(h)))
    nat.check(nat.lib.afqmc_set_option(h, nat.OPT_CSR_DENSE, 1.0 if dense else 0.0), h)
    dbl = nat.C.POINTER(nat.C.c_double)
    nat.check(nat.lib.afqmc_copy(h, nat.BUF_G, 1, G.ctypes.data_as(dbl)), h)
    back = np.empty_like(G)
    nat.check(nat.lib.afqmc_copy(h, nat.BUF_G, 0, back.ctypes.data_as(dbl)), h)
    assert np.array_equal(back, G)
    sp = s.spvn.view()
    nat.check(nat.lib.afqmc_upload_system(h, *ptr, nat.C.byref(sp), None, 1e-6, s.dt), h)
    nat.check(nat.lib.afqmc_copy(h, nat.BUF_G, 0, back.ctypes.data_as(dbl)), h)
    assert np.array_equal(back, G)
    nat.check(nat.lib.afqmc_vbias(h), h)
    got = np.empty_like(vb)
    nat.check(nat.lib.afqmc_copy(h, nat.BUF_VBIAS, 0, got.ctypes.data_as(dbl)), h)
    nat.lib.afqmc_ctx_destroy(h)
    assert np.array_equal(got, vb)

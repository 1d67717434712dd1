"""Which propagator runs (call sites of afqmc_kernel_stats) and that all give
the same walkers bit for bit in split-BF16: the option's kernel wherever it is
asked for and fits, the small systems' kernel, the products."""
import sys

import numpy as np
import pytest

import miniafqmc_amd as m
from miniafqmc_amd import _native as nat

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def walk(M, N, nw, mode="mixed_bf16", fused=False, tile=0):
    """One propagation of random walkers with a random HS potential."""
    s = m.make_system(M, N, 6, density=1.0, sigma_L=0.3 / M ** 0.5, sigma_h=1.0, dt=0.005, seed=M)
    r = np.random.default_rng(nw)
    V = 0.3 * (r.standard_normal((M * M, nw)) + 1j * r.standard_normal((M * M, nw))) / M ** 0.5
    W = r.standard_normal((nw, 2, M, N)) + 1j * r.standard_normal((nw, 2, M, N))
    g = m.AfqmcSys(s, nw, mode, energy_precision=0, dense_exchange=False)
    if fused:
        g.set_fused_propagator(True)
    g.set_tile(tile)
    g.set(nat.BUF_W, W)
    g.set(nat.BUF_VHS, V)
    g.profile(True)
    g.propagate()
    st = {k: v for k, v in g.kernel_stats().items() if k.startswith("prop_")}
    out = g.W
    g.close()
    say(f"M={M} N={N} nw={nw} {mode} fused={fused} tile={tile}: {st}")
    return out, st


@pytest.mark.parametrize("M,N,nw", [(64, 16, 5), (64, 48, 70), (128, 32, 9), (192, 64, 3), (256, 64, 4), (448, 16, 2)])
def test_fused_option_selects_its_kernel(require_gpu, M, N, nw):
    chain, sc = walk(M, N, nw, tile=1)
    assert "prop_taylor" in sc and not {"prop_fused", "prop_fused_cols"} & set(sc)
    for fused, tile in ((True, 0), (True, 1), (False, 0)):
        out, st = walk(M, N, nw, fused=fused, tile=tile)
        if fused:
            assert set(st) == {"prop_fused_cols"}
        else:
            assert set(st) == {"prop_fused"} if M <= 192 else "prop_taylor" in st
        assert np.array_equal(out, chain), np.abs(out - chain).max()


@pytest.mark.parametrize("M,N,mode", [(96, 32, "mixed_bf16"), (64, 12, "mixed_bf16"), (64, 16, "fp64_dense")])
def test_fused_option_leaves_other_shapes(require_gpu, M, N, mode):
    """M no multiple of 64, N none of 16, FP64: as without the option."""
    a, sa = walk(M, N, 6, mode, fused=True)
    b, sb = walk(M, N, 6, mode)
    assert set(sa) == set(sb) == {"prop_fused"} and np.array_equal(a, b)


@pytest.mark.parametrize("mode", ["fp64_dense", "mixed_fp32", "mixed_bf16"])
def test_statistics_count_launches(require_gpu, mode):
    """One kernel is one launch in the statistics, whatever it runs; the
    timers count its eight products."""
    _, st = walk(64, 16, 6, mode)
    assert st["prop_fused"][0] == 1
    calls, ms = m.reference_timers(st)["Propagation"]
    assert calls == 8 and ms == st["prop_fused"][1]

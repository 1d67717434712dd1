"""The staging levels (AFQMC_OPT_DIRECT_LDS) above the sizes that one kernel
propagates, so that the propagator's products take them: partial row tiles,
and sums that are a multiple of 16 (208), of 8 (200) and of neither (201,
whose rows are padded).  The same walkers, overlaps and energies bit for bit
in split-BF16; FP32 the same walkers, its exchange summed in another order."""
import sys

import numpy as np
import pytest

import miniafqmc_amd as m

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def run(s, x, nw, mode, level, **kw):
    g = m.AfqmcSys(s, nw, mode, **kw)
    g.set_direct_lds(level)
    g.init_walkers()
    g.stage_fields(x)
    g.calculate_mixed_density_matrix()
    e = g.calculate_energy()
    g.profile(True)
    g.run(1, 4, 2, s.dt)
    names = set(g.kernel_stats())
    assert {"prop_pw", "prop_taylor", "prop_ps"} <= names and "prop_fused" not in names
    out = g.W, g.W_data, e
    g.close()
    return out


@pytest.mark.parametrize("mode", ["mixed_bf16", "mixed_fp32"])
@pytest.mark.parametrize("M,N,K,block", [(208, 12, 96, False), (200, 8, 64, True), (201, 9, 65, True)])
def test_levels_above_the_one_kernel_sizes(require_gpu, mode, M, N, K, block):
    s = m.make_system(M, N, K, density=0.5, sigma_L=0.02, seed=9)
    nw = 16
    x = m.fields_block(9, K, nw, 0, 4)
    out = []
    for level in (0, 1, 2):
        say("staging", mode, M, N, K, "level", level)
        out.append(run(s, x, nw, mode, level, dense_exchange=block))
    for lv in (1, 2):
        assert np.array_equal(out[0][0], out[lv][0]), f"level {lv}: walkers"
        if mode == "mixed_bf16" and not block:
            assert np.array_equal(out[0][1], out[lv][1]), f"level {lv}: W_data"
        else:  # the block's exchange: other FP64 groups of the same products
            assert np.array_equal(out[0][1][:, 1:], out[lv][1][:, 1:]), f"level {lv}: W_data"
            assert np.abs(out[0][1][:, 0] - out[lv][1][:, 0]).max() <= 1e-6 * np.abs(out[0][1][:, 0]).max()

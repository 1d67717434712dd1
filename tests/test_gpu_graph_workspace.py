"""Energies between replays of captured substeps (one context, a group): the
substep's workspace keeps its address whatever the energy needs, so the
replays equal eager substeps and write no memory that others were given
meanwhile.  Vakbl kept dense (FP64 CSR) has the energy that needs most."""
import sys

import numpy as np
import pytest

import miniafqmc_amd as m
import hip_rt

pytestmark = pytest.mark.gpu

NSUB = 7


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def system(M, N, K, nw, mode, seed):
    s = m.make_system(M, N, K, density=0.3, sigma_L=0.02 * (64.0 / M) ** 0.5, sigma_h=1.0, dt=0.005, seed=seed,
                      with_vakbl=(mode == "fp64_csr"))
    return s, m.fields_block(seed, K, nw, 0, NSUB), nw, mode


def start(s, x, nw, mode, graphs=False):
    g = m.AfqmcSys(s, nw, mode)
    g.init_walkers()
    g.stage_fields(x)
    g.use_graphs(graphs)
    g.calculate_mixed_density_matrix()
    return g


def energy(g):
    g.calculate_mixed_density_matrix()
    g.calculate_energy()


class Neighbours:
    """Allocations of the sizes a freed workspace leaves, made after the first
    energy and never written again."""

    def __init__(self, s, nw):
        n = 32 * nw * s.nchol * 2
        r = np.random.default_rng(nw)
        self.t = [hip_rt.Buffer(r.standard_normal(n // k)) for k in (1, 2, 4, 16) for _ in range(8)]
        self.g = m.AfqmcSys(s, nw, "fp64_csr" if s.vakbl is not None else "fp64_dense")
        self.g.init_walkers()
        energy(self.g)

    def check(self):
        assert all(t.unchanged() for t in self.t), "another allocation was written"
        for t in self.t:
            t.free()
        self.g.close()


def same(a, b, what):
    assert np.array_equal(a.W, b.W), f"{what}: walkers differ"
    assert np.array_equal(a.W_data, b.W_data), f"{what}: W_data differ"


@pytest.mark.parametrize("mode,M,N,K,nw", [("fp64_csr", 64, 16, 256, 16), ("fp64_csr", 40, 7, 53, 5),
                                           ("fp64_dense", 96, 24, 200, 12), ("mixed_bf16", 96, 24, 384, 16)])
def test_energies_between_replays(require_gpu, mode, M, N, K, nw):
    s, x, nw, mode = system(M, N, K, nw, mode, M)
    eager, replay = start(s, x, nw, mode), start(s, x, nw, mode, graphs=True)
    others = None
    for t in range(NSUB):
        say("substep", mode, M, t)
        for g in (eager, replay):
            g.substep(t, t in (2, 5), s.dt)
        same(eager, replay, f"substep {t}")
        for g in (eager, replay):
            energy(g)
        if others is None:
            others = Neighbours(s, nw)
        same(eager, replay, f"energy after substep {t}")
    others.check()
    eager.close()
    replay.close()


def test_member_energies_between_group_replays(require_gpu):
    specs = [system(64, 16, 256, 16, "fp64_csr", 5), system(96, 24, 200, 12, "mixed_bf16", 6)]
    alone = [start(*sp) for sp in specs]
    members = [start(*sp) for sp in specs]
    grp = m.AfqmcGroup(members)
    others = []
    for t in range(NSUB):
        say("group substep", t)
        grp.substep(t, t in (2, 5), 0.005)
        for g in alone:
            g.substep(t, t in (2, 5), 0.005)
        for g in alone + members:
            energy(g)
        if not others:
            others = [Neighbours(sp[0], sp[2]) for sp in specs]
        for i, (a, b) in enumerate(zip(alone, members)):
            same(a, b, f"member {i} after substep {t}")
    for o in others:
        o.check()
    grp.close()
    for g in alone + members:
        g.close()

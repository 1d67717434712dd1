"""Timed cases of the walker step: what a user's program has this library do.

A case is a short walk (the reference driver's step loop from walkers at the
trial), the phases of one substep called one by one, the allocation-free
density matrix on device tensors, or several systems advanced by one graph.
Systems are synthetic (random Hermitian Cholesky vectors under a magnitude
threshold, a one-body Hamiltonian with a semicircle spectrum, the lowest
orbitals as trial), with sizes from this repository's presets, its uneven
multi-system batch and its tests, or generic ones.
"""
import math

import numpy as np
import torch

import miniafqmc_amd as m
from miniafqmc_amd import _native as nat

DT = 0.005
# M * K * E|L|^2 of the 64-orbital preset (256 vectors at 30 % density,
# sigma 0.02), which sets the size of the HS potential; every system here is
# scaled to it
VHS_SCALE = 64 * 256 * 2 * 0.02 ** 2 * 0.3 * (1 - math.log(0.3))


def listed():
    walk = dict(kind="walk", steps=1, substeps=10, northo=5, energy=True, level=1, dense_exchange=True, three=0,
                steps3=255, one=0, graphs=False, vakbl=False, walkers_out=False)

    # a block of substeps ends with what the program reads: the step energies,
    # W_data and, where it keeps the walkers (small populations, restarts), W;
    # gigabytes of walkers stay on the GPU
    def w(name, mode, M, N, K, walkers, density, **over):
        return dict(walk, name=name, mode=mode, M=M, N=N, K=K, walkers=walkers, density=density, **over)

    return [
        # the reference's own small example: 64 orbitals, 16 walkers, CSR
        # throughout, two-body energy from Vakbl after every substep; launches
        # and their gaps are all it costs
        w("csr_64orb_16w", "fp64_csr", 64, 16, 256, 16, 0.3, steps=6, substeps=1, vakbl=True, walkers_out=True),
        # a serving loop's density matrix on tensors that the caller keeps on
        # the GPU, the smallest call there is
        dict(name="noalloc_96orb_64w", kind="noalloc", M=96, N=24, walkers=64),
        # the reference's driver patched call by call: the phases of one
        # substep with the non-transposed bias (-t no), fields from the host
        dict(name="phases_96orb_64w", kind="phases", M=96, N=24, K=384, walkers=64, density=0.15),
        # a production walk of a small system: split-BF16, captured graphs
        w("bf16_128orb_96w", "mixed_bf16", 128, 32, 512, 96, 0.2, graphs=True, walkers_out=True),
        # the FP32 mode on a middle-sized system
        w("fp32_192orb_128w", "mixed_fp32", 192, 48, 768, 128, 0.25, graphs=True, walkers_out=True),
        # sizes as a molecule gives them, no multiple of anything, FP64 on
        # dense vectors
        w("dense_250orb_200w", "fp64_dense", 250, 61, 999, 200, 0.3, walkers_out=True),
        # the 256-orbital preset with the reference's algorithm in FP64
        w("csr_256orb_256w", "fp64_csr", 256, 64, 1024, 256, 0.2, walkers_out=True),
        # energies after every second substep (level 2: the exchange in
        # three-piece split-BF16), propagator precision of the benchmark
        w("bf16_256orb_energy", "mixed_bf16", 256, 64, 1024, 256, 0.2, steps=4, substeps=2, level=2, three=4,
          steps3=0x81, one=0x06, graphs=True),
        # split-BF16 in two pieces throughout, a member of the uneven batch
        w("bf16_384orb_256w", "mixed_bf16", 384, 96, 1536, 256, 0.4, graphs=True),
        # the benchmark's system and settings (10 substeps, one
        # orthogonalisation, as its cadence has it; the energy's exchange
        # block leaves no room for several of these on one card, so none is
        # evaluated); the vectors are dense on the device whatever their
        # density in the input
        w("bf16_512orb_1024w", "mixed_bf16", 512, 128, 2048, 1024, 0.2, northo=6, energy=False, three=4, steps3=0x81,
          one=0x06, graphs=True),
        # more than 128 electrons per spin (the uneven batch's largest member
        # has 160): half filling, FP64
        w("dense_320orb_160el", "fp64_dense", 320, 160, 640, 64, 0.3, substeps=4, northo=2, dense_exchange=False,
          walkers_out=True),
        # three uneven systems side by side, one graph launch per substep
        dict(name="group_96_128_192", kind="group", mode="mixed_bf16", M0=96, M1=128, M2=192, walkers0=64, walkers1=96,
             walkers2=128, density=0.2, substeps=10, northo=5),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["walk"] * 7 + ["noalloc", "phases", "group"])
    if kind == "noalloc":
        M = _log(rng, 32, 256)
        N = max(4, min(100, int(M * rng.uniform(0.15, 0.5))))
        return dict(kind=kind, M=M, N=N, walkers=max(4, min(_log(rng, 8, 512), (3 << 20) // (2 * N * N))))
    if kind == "phases":
        M = _log(rng, 32, 160)
        return dict(kind=kind, M=M, N=max(4, int(M * rng.uniform(0.15, 0.5))), K=int(M * rng.uniform(2, 4)),
                    walkers=_log(rng, 8, 128), density=round(rng.uniform(0.1, 0.4), 3))
    if kind == "group":
        Ms = [16 * rng.randint(3, 14) for _ in range(3)]
        ws = [_log(rng, 16, 160) for _ in range(3)]
        return dict(kind=kind, mode=rng.choice(["fp64_dense", "mixed_bf16", "mixed_bf16"]), M0=Ms[0], M1=Ms[1], M2=Ms[2],
                    walkers0=ws[0], walkers1=ws[1], walkers2=ws[2], density=round(rng.uniform(0.15, 0.4), 3),
                    substeps=rng.randint(3, 10), northo=rng.randint(2, 5))
    mode = rng.choice(["fp64_csr", "fp64_csr", "fp64_dense", "fp64_dense", "mixed_fp32", "mixed_bf16", "mixed_bf16",
                       "mixed_bf16"])
    M = _log(rng, 40, 384)
    even = mode == "mixed_bf16" and rng.random() < 0.6
    if even:
        M = 16 * max(3, M // 16)
    N = max(6, min(176, int(M * rng.choice([0.25, 0.25, rng.uniform(0.15, 0.5)]))))
    K = int(M * rng.uniform(2, 4))
    if even:
        K = 16 * (K // 16)
    walkers = _log(rng, 12, 512)
    # no dearer than the largest listed case, on the mode's own terms
    top = 4e13 if mode.startswith("mixed_bf16") else 8e12
    substeps = rng.randint(2, 10)
    case = dict(kind="walk", mode=mode, M=M, N=N, K=K, walkers=walkers, density=round(rng.uniform(0.15, 0.4), 3), steps=1,
                substeps=substeps, northo=rng.randint(2, 5), energy=rng.random() < 0.7, level=rng.choice([1, 1, 2]),
                dense_exchange=N * M <= 16384, three=rng.choice([0, 4]) if even else 0, steps3=0x81, one=0x06,
                graphs=rng.random() < 0.6, vakbl=False, walkers_out=M * N * walkers < 1 << 20)
    while walkers > 12 and work(case)["flops"] > top:
        walkers = case["walkers"] = max(12, walkers // 2)
    while case["substeps"] > 2 and work(case)["flops"] > top:
        case["substeps"] -= 1
    return case


# -- inputs ---------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _cn(shape, g):
    return torch.complex(torch.randn(shape, generator=g, device="cuda", dtype=torch.float64),
                         torch.randn(shape, generator=g, device="cuda", dtype=torch.float64))


def _orbitals(M, N, g):
    """One-body Hamiltonian U diag(lam) U^H, exp(-dt/2 h) and the trial's two spins (conjugated)."""
    U = torch.from_numpy(np.linalg.qr(_cn((M, M), g).cpu().numpy())[0]).cuda()
    V = torch.from_numpy(np.linalg.qr(_cn((N, N), g).cpu().numpy())[0]).cuda()
    x = np.linspace(-1, 1, 4001)  # quantiles of the semicircle law of radius sqrt(2M)
    F = 0.5 + (x * np.sqrt(1 - x * x) + np.arcsin(x)) / math.pi
    lam = torch.from_numpy(np.interp((np.arange(M) + 0.5) / M, F, x) * math.sqrt(2.0 * M)).cuda()
    h = (U * lam) @ U.conj().T
    P = (U * torch.exp(-0.5 * DT * lam)) @ U.conj().T
    trial = torch.stack([U[:, :N].conj(), (U[:, :N] @ V).conj()])
    return trial, h, P


def _vectors(M, K, density, g):
    """Hermitian Cholesky vectors under the magnitude threshold, times sqrt(dt): [M*M][K]."""
    tau = math.sqrt(-2.0 * math.log(density))
    sigma = math.sqrt(VHS_SCALE / (M * K * 2 * density * (1 - math.log(density))))
    L = _cn((M, M, K), g)
    i = torch.arange(M, device="cuda")
    for a in range(M):  # row a below the diagonal is the conjugate of column a above it
        L[a, :a] = L[:a, a].conj()
    L[i, i] = torch.complex(L[i, i].real, torch.zeros_like(L[i, i].real))
    L = L.view(M * M, K)
    L *= L.abs() > tau
    L *= sigma * math.sqrt(DT)
    return L


def _csr(D):
    mask = D != 0
    rp = torch.zeros(D.shape[0] + 1, dtype=torch.int32, device="cuda")
    rp[1:] = mask.sum(1).cumsum(0)
    col = torch.arange(D.shape[1], dtype=torch.int32, device="cuda").expand(D.shape)[mask]
    return m.Csr(D.shape[0], D.shape[1], rp.cpu().numpy(), col.cpu().numpy(), D[mask].cpu().numpy())


def _rotated(trial, L):
    """Half-rotated vectors [2][K][N][M] from dense [M*M][K]."""
    M, K = trial.shape[1], L.shape[1]
    A = L.view(M, M * K)
    return torch.stack([(t.T.contiguous() @ A).view(-1, M, K).permute(2, 0, 1).contiguous() for t in trial])


def _vakbl(Lt):
    K, N, M = Lt.shape[1:]
    A = Lt.permute(1, 0, 2, 3).reshape(K, -1) / math.sqrt(DT)
    V = A.T @ A
    for s in range(2):
        B = Lt[s] / math.sqrt(DT)
        X = torch.einsum("nal,nbk->akbl", B, B).reshape(N * M, N * M)
        V[s * N * M:(s + 1) * N * M, s * N * M:(s + 1) * N * M] -= X
    return V


def _dense_system(case, seed):
    g = _gen(seed)
    trial, h, P = _orbitals(case["M"], case["N"], g)
    return trial, h, P, _vectors(case["M"], case["K"], case["density"], g)


def _fields(case, seed, n):
    g = _gen(seed + 7919)
    return torch.randn((n, case["K"], case["walkers"]), generator=g, device="cuda", dtype=torch.float64)


def _system(case, seed):
    trial, h, P, L = _dense_system(case, seed)
    haj = (trial.transpose(1, 2) @ h).reshape(-1, case["M"])
    vak = _csr(_vakbl(_rotated(trial, L))) if case.get("vakbl") else None
    host = [np.ascontiguousarray(t.cpu().numpy()) for t in (trial[0], trial[1], haj, P, h)]
    spvn = _csr(L)
    del L
    torch.cuda.empty_cache()
    return m.System(case["M"], case["N"], case["K"], DT, seed, *host, spvn, vak)


def _context(case, seed, **over):
    bf16 = case["mode"] == "mixed_bf16"
    g = m.AfqmcSys(_system(case, seed), case["walkers"], case["mode"], energy_precision=case.get("level", 1),
                   dense_exchange=case.get("dense_exchange", True), three_piece=case.get("three", 0) if bf16 else 0, **over)
    if bf16 and case.get("three", 0) & 4:
        g.set_three_piece_steps(case["steps3"])
        g.set_one_piece_steps(case["one"])
    return g


def _members(case):
    return [dict(kind="walk", mode=case["mode"], M=case["M%d" % i], N=case["M%d" % i] // 4, K=4 * case["M%d" % i],
                 walkers=case["walkers%d" % i], density=case["density"], steps=1, substeps=case["substeps"],
                 northo=case["northo"], energy=False, dense_exchange=False) for i in range(3)]


def _walkers(case, seed):
    """Walkers some way from the trial, as a walk leaves them: [nw][2][M][N]."""
    g = _gen(seed)
    trial, _, _ = _orbitals(case["M"], case["N"], g)
    W = trial.conj()[None].repeat(case["walkers"], 1, 1, 1)
    return trial, W + 0.05 / math.sqrt(case["M"]) * _cn(W.shape, g)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "noalloc":
        trial, W = _walkers(case, seed)
        nw, M, N = case["walkers"], case["M"], case["N"]
        return dict(case=case, trial=trial.contiguous(), W=W.contiguous(),
                    G=torch.empty((2 * N * M, nw), dtype=torch.complex128, device="cuda"),
                    ovlp=torch.empty((nw, 2), dtype=torch.complex128, device="cuda"))
    if kind == "group":
        cs = _members(case)
        gs = [_context(c, seed + i) for i, c in enumerate(cs)]
        for i, (c, g) in enumerate(zip(cs, gs)):
            g.stage_fields(_fields(c, seed + i, c["substeps"]).cpu().numpy())
        return dict(case=case, members=gs, group=m.AfqmcGroup(gs))
    if kind == "phases":
        g = _context(dict(case, mode="fp64_csr"), seed, transposed=False)
        return dict(case=case, g=g, x=np.ascontiguousarray(_fields(case, seed, 1)[0].cpu().numpy()))
    g = _context(case, seed)
    g.stage_fields(_fields(case, seed, case["steps"] * case["substeps"]).cpu().numpy())
    if case["graphs"]:
        g.use_graphs(True)
    return dict(case=case, g=g)


# -- one pass ---------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "noalloc":
        nat.check(m.lib.afqmc_mixed_density_matrix_noalloc(
            case["M"], case["N"], case["walkers"], state["trial"].data_ptr(), state["W"].data_ptr(), state["G"].data_ptr(),
            state["ovlp"].data_ptr(), torch.cuda.current_stream().cuda_stream))
        return {"G": state["G"], "overlaps": state["ovlp"]}
    if kind == "group":
        for g in state["members"]:
            g.init_walkers()
            g.set_eshift(0.0)
        for s in range(case["substeps"]):
            state["group"].substep(s, s > 0 and s % case["northo"] == 0, DT)
        state["group"].sync()
        return [g.W_data for g in state["members"]]
    g = state["g"]
    g.init_walkers()
    if kind == "phases":
        lib, c = m.lib, g.ctx
        nat.check(lib.afqmc_mixed_density_matrix_full(c), c)
        nat.check(lib.afqmc_vbias_full(c), c)
        g.fields(state["x"])
        nat.check(lib.afqmc_vhs(c), c)
        g.propagate()
        g.save_overlaps()
        g.calculate_overlaps()
        eshift = g.weights(DT, 0.0)
        g.orthogonalize()
        return {"walkers": g.W, "walker_data": g.W_data, "vbias": g.get(nat.BUF_VBIAS), "eshift": eshift}
    g.set_eshift(0.0)
    eav = g.run(case["steps"], case["substeps"], case["northo"], DT, energy=case["energy"])
    out = {"walker_data": g.W_data, "eshift": g.eshift()}
    if case["energy"]:
        out["eav"] = eav
    if case["walkers_out"]:
        out["walkers"] = g.W
    return out


# -- what a pass cannot do without ---------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "group":
        ws = [work(c) for c in _members(case)]
        return {k: sum(w[k] for w in ws) for k in ("bytes", "flops")}
    M, N, nw = case["M"], case["N"], case["walkers"]
    dens = nw * 8.0 * (2 * N * N * M + 2 * N ** 3 + 2 * N * N * M)  # overlaps, inverse, G (complex multiply-adds, 8 flops)
    if kind == "noalloc":
        return {"flops": dens, "bytes": 16.0 * (2 * M * N + 2 * nw * 2 * M * N + 2 * nw)}
    K = case["K"]
    mode = case.get("mode", "fp64_csr")
    csr = mode == "fp64_csr"
    nsub = case["steps"] * case["substeps"] if kind == "walk" else 1
    north = sum(1 for t in range(1, nsub) if t % case["northo"] == 0) if kind == "walk" else 1
    zs = 8.0 if mode.startswith("mixed") else 16.0
    vhs = M * M * K * (case["density"] if csr else 1.0)
    bias = 2 * vhs if kind == "phases" else 2 * N * M * K
    step = dens + nw * 8.0 * (bias + vhs + 16.0 * M * M * N)
    flops = nsub * step + north * nw * 8.0 * 4 * N * N * M
    ham = vhs * (20.0 if csr else zs) + (0 if kind == "phases" else 2 * N * M * K * zs) + 16.0 * (M * M + 4 * M * N)
    bytes_ = ham + 16.0 * nw * (2 * M * N + 8) + 8.0 * nsub * K * nw + (16.0 * nw * (2 * M * N + K) if kind == "phases" else 0)
    if kind == "walk" and case["energy"]:
        NM = float(N * M)
        if case["vakbl"]:
            two = (2 * NM) ** 2
            bytes_ += 20.0 * two
        elif case["dense_exchange"]:
            two = 2 * NM * K + NM * NM  # Coulomb, and the exchange block's triangle for two spins
            bytes_ += zs * NM * NM
        else:
            two = 2 * NM * K + 2 * NM * N * K
        flops += case["steps"] * nw * 8.0 * two
    return {"flops": flops, "bytes": bytes_}


# -- the same in 64 bits with torch alone ----------------------------------------------
def _inverse(T):
    """Inverse and determinant of [b][N][N] by Gauss-Jordan elimination with row pivoting."""
    b, N = T.shape[:2]
    X = torch.cat([T, torch.eye(N, dtype=T.dtype, device=T.device).expand(b, N, N)], 2)
    at, det = torch.arange(b, device=T.device), torch.ones(b, dtype=T.dtype, device=T.device)
    for k in range(N):
        p = X[:, k:, k].abs().argmax(1) + k
        row = X[at, p]
        X[at, p] = X[:, k]
        det = det * torch.where(p == k, row[:, k], -row[:, k])
        row = row / row[:, k:k + 1]
        f = X[:, :, k].clone()
        f[:, k] = 0
        X -= f[:, :, None] * row[:, None, :]
        X[:, k] = row
    return X[:, :, N:], det


def _qr(W):
    """The unitary factor of every conj(W) [b][M][N] by Householder reflectors (beta = -sign(Re alpha) |x|), conjugated."""
    A = W.conj().resolve_conj().clone()
    b, M, N = A.shape
    Q = torch.eye(M, N, dtype=A.dtype, device=A.device).repeat(b, 1, 1)
    refl = []
    for k in range(N):
        v = A[:, k:, k].clone()
        alpha = v[:, 0].clone()
        beta = -torch.copysign(torch.linalg.vector_norm(v, dim=1), alpha.real)
        tau = (beta - alpha) / beta
        v = v / (alpha - beta)[:, None]
        v[:, 0] = 1
        A[:, k:, k:] -= (tau.conj()[:, None] * v)[:, :, None] * (v.conj()[:, None, :] @ A[:, k:, k:])
        refl.append((tau, v))
    for k in reversed(range(N)):
        tau, v = refl[k]
        Q[:, k:, k:] -= (tau[:, None] * v)[:, :, None] * (v.conj()[:, None, :] @ Q[:, k:, k:])
    return Q.conj().resolve_conj()


class _Walk:
    def __init__(self, case, seed):
        self.M, self.N, self.K, self.nw = case["M"], case["N"], case["K"], case["walkers"]
        self.trial, h, self.P, self.L = _dense_system(case, seed)
        self.haj = self.trial.transpose(1, 2) @ h
        self.Lt = _rotated(self.trial, self.L)
        self.case = case
        self.Lb = self.Lt
        if case.get("mode") == "fp64_csr":  # the half rotation's cutoff
            self.Lb = self.Lt * (self.Lt.abs() > 1e-6)
        self.W = self.trial.conj()[None].repeat(self.nw, 1, 1, 1)
        self.d = torch.zeros((self.nw, 8), dtype=torch.complex128, device="cuda")
        self.d[:, 1] = 1
        self.eshift = 0.0

    def density(self):
        T = (self.W.transpose(2, 3) @ self.trial[None]).reshape(-1, self.N, self.N)
        Ti, det = _inverse(T)
        self.d[:, 2:4] = det.view(self.nw, 2)
        return Ti.view(self.nw, 2, self.N, self.N) @ self.W.transpose(2, 3)

    def substep(self, x, ortho):
        G = self.density()
        vb = G[:, 0].reshape(self.nw, -1) @ self.Lb[0].reshape(self.K, -1).T
        vb = vb + G[:, 1].reshape(self.nw, -1) @ self.Lb[1].reshape(self.K, -1).T
        del G
        x = x.T.to(torch.complex128)
        hyb = -(1j * vb * (x + 0.5j * vb)).sum(1)
        self.vb = vb
        V = ((x + 1j * vb) @ self.L.T).view(self.nw, self.M, self.M)
        # the spins' columns side by side: [nw][M][2N]
        S = (self.P @ self.W).permute(0, 2, 1, 3).reshape(self.nw, self.M, -1)
        T = S.clone()
        for n in range(1, 7):
            T = (1j / n) * (V @ T)
            S += T
        del V, T
        self.W = (self.P @ S).view(self.nw, self.M, 2, self.N).permute(0, 2, 1, 3).contiguous()
        d = self.d
        d[:, 5] = d[:, 4]
        d[:, 6:8] = d[:, 2:4]
        self.density()
        lr = torch.log(d[:, 2]) + torch.log(d[:, 3]) - torch.log(d[:, 6]) - torch.log(d[:, 7])
        ang = torch.remainder(lr.imag + math.pi, 2 * math.pi) - math.pi
        d[:, 4] = -(hyb + torch.complex(lr.real, ang)) / DT
        f = torch.clamp(torch.cos(ang), min=0) * torch.exp(-DT * (0.5 * (d[:, 4] + d[:, 5]).real - self.eshift))
        d[:, 1] *= f
        self.eshift = float(d[:, 4].real.mean())
        if ortho:
            self.W = _qr(self.W.view(-1, self.M, self.N)).view(self.W.shape)
            if self.case["kind"] != "phases":
                self.density()

    def energy(self):
        G = self.density()
        e = (G * self.haj[None]).sum((1, 2, 3))
        if self.case.get("vakbl"):
            g = G.reshape(self.nw, -1)
            e = e + 0.5 * ((g @ _vakbl(self.Lt).T) * g).sum(1)
        else:
            v = sum(G[:, s].reshape(self.nw, -1) @ self.Lt[s].reshape(self.K, -1).T for s in range(2))
            two = (v * v).sum(1)
            for s in range(2):
                g = G[:, s].reshape(-1, self.M).T  # [M][nw*N]
                n1 = max(1, int(6e7 / (self.N * self.N * self.nw)))
                for n0 in range(0, self.K, n1):
                    Y = (self.Lt[s, n0:n0 + n1].reshape(-1, self.M) @ g).view(-1, self.N, self.nw, self.N)
                    two = two - (Y * Y.transpose(1, 3)).sum((0, 1, 3))
            e = e + 0.5 * two / DT
        self.d[:, 0] = e
        return float((e.real * self.d[:, 1].real).sum() / self.d[:, 1].real.sum())


def exact(case, seed):
    kind = case["kind"]
    if kind == "noalloc":
        trial, W = _walkers(case, seed)
        Ti, det = _inverse((W.transpose(2, 3) @ trial[None]).reshape(-1, case["N"], case["N"]))
        G = Ti.view(case["walkers"], 2, case["N"], case["N"]) @ W.transpose(2, 3)
        return {"G": G.reshape(case["walkers"], -1).T.contiguous(), "overlaps": det.view(-1, 2)}
    if kind == "group":
        out = []
        for i, c in enumerate(_members(case)):
            w, x = _Walk(c, seed + i), _fields(c, seed + i, c["substeps"])
            for s in range(c["substeps"]):
                w.substep(x[s], s > 0 and s % c["northo"] == 0)
            out.append(w.d.cpu().numpy())
        return out
    if kind == "phases":
        w = _Walk(case, seed)
        w.substep(_fields(case, seed, 1)[0], True)
        return {"walkers": w.W.cpu().numpy(), "walker_data": w.d.cpu().numpy(), "vbias": w.vb.T.contiguous().cpu().numpy(),
                "eshift": w.eshift}
    if work(case)["flops"] > 3e14:
        return None
    w, x, t, eav = _Walk(case, seed), _fields(case, seed, case["steps"] * case["substeps"]), 0, []
    for _ in range(case["steps"]):
        for _ in range(case["substeps"]):
            w.substep(x[t], t > 0 and t % case["northo"] == 0)
            t += 1
        if case["energy"]:
            eav.append(w.energy())
    out = {"walker_data": w.d.cpu().numpy(), "eshift": w.eshift}
    if case["energy"]:
        out["eav"] = np.array(eav)
    if case["walkers_out"]:
        out["walkers"] = w.W.cpu().numpy()
    return out

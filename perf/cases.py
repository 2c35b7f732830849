"""The work that users of this package have it do, as cases of stated sizes.

A case is one call, or one captured run of calls, of the phaseless-AFQMC path: walker steps
(hybrid and local-energy form, FP64 and INT8_SPLIT), the energy estimator, re-orthogonalisation,
back-propagation, and the energy and force bias of a particle-hole multi-determinant trial.
`listed()` holds the fixed cases, `draw(rng)` gives another one of the same ranges: 16 to 128
orbitals, 3 to 32 electrons per spin, 3 to 6 Cholesky vectors per orbital, 24 to 1024 walkers, real
and complex trial orbitals.

Inputs are made from the seed alone: a Hamiltonian with a random symmetric one-body part and random
symmetric Cholesky vectors whose sizes decay as exp(-10 n / K) (the decay of the package's largest
synthetic workload) with a leading spectral norm near 1, a trial of orthonormal orbitals, and
walkers around the trial with weights in [0.5, 1.5], as in a run between population controls.

`exact` restates each path in 64-bit torch, without the package.
"""
from __future__ import annotations

import math

import numpy as np
import torch

DT = 0.005
WEIGHT, PHASE, PSEUDO_ELOC, E1, EXX, EJ, OVLP, IS_UNITARY, THETA, COUNT = 0, 1, 2, 3, 4, 5, 6, 9, 10, 11


def listed():
    return [
        # One step of a small molecule's run on few walkers (the BH test system's sizes): latency.
        {"name": "step_hybrid_19_3_w50", "op": "step", "M": 19, "N": 3, "K": 78, "W": 50,
         "form": "fp64", "hybrid": True, "complex": False, "steps": 1, "graph": False},
        # A block between re-orthogonalisations, captured once and replayed, as a run of a small
        # system does it: five local-energy steps and the QR.
        {"name": "block_24_6_w64", "op": "step", "M": 24, "N": 6, "K": 96, "W": 64,
         "form": "fp64", "hybrid": False, "complex": False, "steps": 5, "graph": True},
        # The default propagation (hybrid energy) of a mid-sized system in the plain form.
        {"name": "step_hybrid_64_16_w512", "op": "step", "M": 64, "N": 16, "K": 320, "W": 512,
         "form": "fp64", "hybrid": True, "complex": False, "steps": 1, "graph": False},
        # The same system in the mixed form with local energies.
        {"name": "step_int8_64_16_w512", "op": "step", "M": 64, "N": 16, "K": 320, "W": 512,
         "form": "int8", "hybrid": False, "complex": False, "steps": 1, "graph": False},
        # The benchmark's largest system, mixed form.
        {"name": "step_int8_128_32_w1024", "op": "step", "M": 128, "N": 32, "K": 640, "W": 1024,
         "form": "int8", "hybrid": False, "complex": False, "steps": 1, "graph": False},
        # The same in the plain form: what a user runs who wants every contraction in 64 bits.
        {"name": "step_fp64_128_32_w1024", "op": "step", "M": 128, "N": 32, "K": 640, "W": 1024,
         "form": "fp64", "hybrid": False, "complex": False, "steps": 1, "graph": False},
        # Sizes that no tile divides and complex trial orbitals (twisted boundaries, spin-orbit).
        {"name": "step_fp64_77_19_w201", "op": "step", "M": 77, "N": 19, "K": 385, "W": 201,
         "form": "fp64", "hybrid": False, "complex": True, "steps": 1, "graph": False},
        # The energy estimator of one system of an uneven batch, mixed form.
        {"name": "energy_int8_88_22_w137", "op": "energy", "M": 88, "N": 22, "K": 440, "W": 137,
         "form": "int8", "complex": False},
        # Re-orthogonalisation of the largest walkers, with the new overlaps.
        {"name": "orthogonalize_128_32_w1024", "op": "orthogonalize", "M": 128, "N": 32, "K": 384,
         "W": 1024, "complex": False},
        # Back-propagation of one reference through ten stored steps.
        {"name": "back_propagate_48_12_w256", "op": "back_propagate", "M": 48, "N": 12, "K": 240,
         "W": 256, "complex": False, "nback": 10, "nstab": 5},
        # The local energy of a thousand-determinant trial (the default algorithm).
        {"name": "phmsd_energy_64_10_w256", "op": "phmsd_energy", "M": 64, "N": 10, "K": 320,
         "W": 256, "ndet": 1000, "algorithm": "woodbury", "complex": False},
        # The force bias that every step of such a trial needs.
        {"name": "phmsd_vbias_64_10_w256", "op": "phmsd_vbias", "M": 64, "N": 10, "K": 320,
         "W": 256, "ndet": 1000, "complex": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["step"] * 10 + ["energy"] * 2 + ["orthogonalize", "back_propagate"] * 2 +
                    ["phmsd_energy"] * 2 + ["phmsd_vbias"])
    complex_ = rng.random() < 0.25
    if op.startswith("phmsd"):
        M = rng.randint(16, 64)
        case = {"op": op, "M": M, "N": rng.randint(3, min(10, M // 2)),
                "K": rng.randint(3 * M, 5 * M), "W": _log_int(rng, 16, 192),
                "ndet": _log_int(rng, 50, 900), "complex": complex_}
        if op == "phmsd_energy":
            case["algorithm"] = rng.choice(["woodbury", "reference"])
        return case
    M = _log_int(rng, 16, 128)
    case = {"op": op, "M": M, "N": rng.randint(3, min(32, M // 2)),
            "K": rng.randint(3 * M, min(6 * M, 640)), "W": _log_int(rng, 24, 1024),
            "complex": complex_}
    if op == "step":
        case["form"] = rng.choice(["fp64", "int8"])
        case["hybrid"] = rng.random() < 0.5
        case["graph"] = rng.random() < 0.3
        case["steps"] = rng.randint(2, 5) if case["graph"] and M <= 48 else 1
    elif op == "energy":
        case["form"] = rng.choice(["fp64", "int8"])
    elif op == "back_propagate":
        case["W"] = min(case["W"], 400)
        case["nback"] = rng.randint(2, 12)
        case["nstab"] = rng.randint(2, 6)
    return case


# ---------------------------------------------------------------------------------- inputs
def _system(rng, M, K):
    """One-body part [M][M] and Cholesky vectors [M][M][K], real symmetric."""
    a = rng.standard_normal((M, M))
    h = 0.1 * (a + a.T) / math.sqrt(2.0)
    h[np.diag_indices(M)] = np.linspace(-2.0, 0.0, M)
    size = 0.5 / math.sqrt(M) * np.exp(-10.0 * np.arange(K) / K)
    b = rng.standard_normal((M, M, K))
    b *= size
    b += b.transpose(1, 0, 2).copy()   # exactly symmetric, as the integrals of real orbitals
    b *= math.sqrt(0.5)
    return h, b


def _orbitals(rng, M, complex_):
    """An M x M orthonormal set, the trial's orbitals in its columns."""
    a = rng.standard_normal((M, M))
    if complex_:
        a = a + 1j * rng.standard_normal((M, M))
    return np.linalg.qr(a)[0].astype(np.complex128)


def _cloud(rng, phi0, W):
    """W Slater matrices around phi0 [M][N]."""
    M, N = phi0.shape
    z = rng.standard_normal((W, M, N)) + 1j * rng.standard_normal((W, M, N))
    return phi0 + (0.4 / math.sqrt(M)) * z


def _expansion(rng, M, N, ndet):
    """A CI expansion over the reference: excitations of total rank 1 to 4, unique, with
    coefficients that fall off with the rank. occs [ndet][2 N], ci [ndet]."""
    occs, ranks = [tuple(range(N)) + tuple(range(M, M + N))], [0]
    seen = set(occs)
    while len(occs) < ndet:
        r = int(rng.integers(1, 5))
        up = int(rng.integers(max(0, r - N), min(r, N) + 1))
        conf = ()
        for nex, base in ((up, 0), (r - up, M)):
            occ = list(range(base, base + N))
            holes = rng.permutation(N)[:nex]
            parts = rng.permutation(M - N)[:nex]
            for i, p in zip(holes, parts):
                occ[i] = base + N + int(p)
            conf += tuple(sorted(occ))
        if conf not in seen:
            seen.add(conf)
            occs.append(conf)
            ranks.append(r)
    c = rng.standard_normal(ndet) * np.exp(-np.array(ranks, float))
    c[1:] *= math.sqrt(0.19) / np.linalg.norm(c[1:])
    c[0] = 0.9
    return np.array(occs, np.int32), c.astype(np.complex128)


def _inputs(case, seed):
    rng = np.random.default_rng([int(seed) % (1 << 63), 17])
    M, N, K, W = case["M"], case["N"], case["K"], case["W"]
    x = {}
    x["h"], x["L"] = _system(rng, M, K)
    q = _orbitals(rng, M, case["complex"])
    x["PsiT"] = np.ascontiguousarray(q[:, :N].conj().T)
    if case["op"].startswith("phmsd"):
        x["orbitals"] = np.ascontiguousarray(q.conj().T)
        x["occs"], x["ci"] = _expansion(rng, M, N, case["ndet"])
        x["up"], x["dn"] = _cloud(rng, q[:, :N], W), _cloud(rng, q[:, :N], W)
        return x
    x["phi"] = _cloud(rng, q[:, :N], W)
    x["weight"] = rng.uniform(0.5, 1.5, W)
    if case["op"] == "step":
        x["xi"] = rng.standard_normal((case["steps"], W, K))
    elif case["op"] == "back_propagate":
        n = case["nback"]
        x["fields"] = (rng.standard_normal((W, n, K)) +
                       0.2 * (rng.standard_normal((W, n, K)) + 1j * rng.standard_normal((W, n, K))))
    return x


def _walker_buffer(case, x):
    M, N, W = case["M"], case["N"], case["W"]
    buf = np.zeros((W, M * N + COUNT), np.complex128)
    buf[:, :M * N] = x["phi"].reshape(W, -1)
    buf[:, M * N + WEIGHT] = x["weight"]
    buf[:, M * N + PHASE] = 1.0
    buf[:, M * N + IS_UNITARY] = 1.0
    return buf


# ---------------------------------------------------------------------------------- the calls
def prepare(case, seed):
    from safire_amd import afqmc as A
    x = _inputs(case, seed)
    M, N, K, W = case["M"], case["N"], case["K"], case["W"]
    s = {"op": case["op"], "A": A, "MN": M * N}
    if case["op"].startswith("phmsd"):
        s["ph"] = A.PHMSD(x["occs"], x["ci"], x["orbitals"], x["h"], x["L"])
        wbuf = np.concatenate([x["up"].reshape(W, -1), x["dn"].reshape(W, -1)], axis=1)
        s["wbuf"] = A.to_device(wbuf)
        if case["op"] == "phmsd_energy":
            s["ph"].set_energy_algorithm(case["algorithm"])
        return s
    ham = A.HamiltonianOperations(x["h"], x["L"], x["PsiT"], 0.0, DT)
    s["ham"], s["prop"] = ham, A.Propagator(ham)
    ham.set_precision(A.INT8_SPLIT if case.get("form") == "int8" else A.FP64)
    wset = A.WalkerSet(ham, W, _walker_buffer(case, x))
    s["wset"] = wset
    if case["op"] == "energy":
        s["E"] = torch.empty((W, 3), dtype=torch.complex128, device="cuda")
        s["ov"] = torch.empty(W, dtype=torch.complex128, device="cuda")
        return s
    if case["op"] == "back_propagate":
        n = case["nback"]
        wset.set_back_propagation(n)
        wset.getFields().copy_(A.to_device(x["fields"]))
        s["nback"], s["nstab"] = n, case["nstab"]
        s["refs0"] = A.to_device(np.repeat(x["PsiT"].conj().T[None, None], W, axis=0))
        s["refs"] = torch.empty_like(s["refs0"])
        s["logdet"] = torch.empty((W, 1), dtype=torch.complex128, device="cuda")
        return s
    ham.set_params(hybrid=int(case.get("hybrid", True)))
    s["prop"].seed(wset)
    s["start"] = wset.buf.clone()
    if case["op"] == "step":
        sums = s["prop"].weighted_sums(wset).cpu().numpy()
        s["Eshift"] = float((sums[0] / sums[1]).real)
        s["xi"], s["steps"] = A.to_device(x["xi"]), case["steps"]
        if case["graph"]:
            _steps(s)   # the first calls of a handle run eagerly
            torch.cuda.synchronize()
            s["replay"] = A.capture(lambda: _steps(s))
    return s


def _steps(s):
    for t in range(s["steps"]):
        s["prop"].Propagate(s["wset"], s["xi"][t], s["Eshift"])
    if s["steps"] > 1:
        s["prop"].Orthogonalize(s["wset"])


def run(state):
    s = state
    op, A = s["op"], s["A"]
    if op == "phmsd_energy":
        E, ov = s["ph"].energy(s["wbuf"])
        return {"E": E, "log_overlap": ov}
    if op == "phmsd_vbias":
        return {"vbias": s["ph"].vbias(s["wbuf"], DT)}
    wset, prop = s["wset"], s["prop"]
    if op == "energy":
        A.check(A.lib().afq_wfn_energy(s["ham"].handle, wset.W, A.ptr(wset.buf), wset.ldw,
                                       A.ptr(s["E"]), A.ptr(s["ov"]), A.stream_ptr()))
        return {"E": s["E"], "log_overlap": s["ov"]}
    if op == "back_propagate":
        s["refs"].copy_(s["refs0"])
        prop.BackPropagate(s["nback"], s["nstab"], wset, s["refs"], s["logdet"])
        return {"refs": s["refs"], "logdet": s["logdet"]}
    wset.buf.copy_(s["start"])   # every pass starts from the same walkers
    if op == "orthogonalize":
        prop.Orthogonalize(wset)
    elif "replay" in s:
        s["replay"].replay()
    else:
        _steps(s)
    return {"slater": wset.buf[:, :s["MN"]], "properties": wset.buf[:, s["MN"]:]}


# ---------------------------------------------------------------------------------- work
def work(case):
    """Bytes: every operand of the call read once and every result written once. Operations: a
    complex multiply-add counts 8, a real by complex one 4; with real trial orbitals the
    half-rotated Cholesky vectors are real, and the Cholesky vectors are symmetric."""
    M, N, K, W = case["M"], case["N"], case["K"], case["W"]
    mac = 8.0 if case["complex"] else 4.0
    green = 2 * mac * M * N * N + 16.0 * N ** 3
    energy = mac * N * N * M * K + 8.0 * N * N * K / 2
    lnak = mac / 4 * 8 * N * M * K
    walkers = 16.0 * W * M * N
    if case["op"] == "step":
        f = (green + mac * N * M * K + 2.0 * M * (M + 1) * K      # G, vbias, vHS
             + 2 * 4.0 * M * M * N + 6 * 8.0 * M * M * N)         # P1 twice, the Taylor series
        f += mac * M * N * N + 8.0 * N ** 3 if case["hybrid"] else green + energy
        b = 2 * walkers + lnak + 4.0 * M * (M + 1) * K + 8.0 * W * K
        qr = 16.0 * M * N * N if case["steps"] > 1 else 0.0
        return {"bytes": case["steps"] * b, "flops": W * (case["steps"] * f + qr)}
    if case["op"] == "energy":
        return {"bytes": walkers + lnak + 64.0 * W, "flops": W * (green + energy)}
    if case["op"] == "orthogonalize":
        return {"bytes": 2 * walkers, "flops": W * (16.0 * M * N * N + mac * M * N * N)}
    if case["op"] == "back_propagate":
        n = case["nback"]
        f = n * (2.0 * M * (M + 1) * K + 2 * 4.0 * M * M * N + 6 * 8.0 * M * M * N)
        return {"bytes": 2 * walkers + 16.0 * W * n * K + 4.0 * M * (M + 1) * K,
                "flops": W * (f + 16.0 * M * N * N)}
    # multi-determinant: the walker products with the rotated vectors (needed once per spin), then
    # per unique excited configuration its N x N blocks of every Cholesky vector (energy) or its
    # share of the density matrix (force bias); about 0.6 ndet unique configurations per spin
    products = 2 * mac * N * M * M * K
    per_conf = 8.0 * N * N * 2.5 * K if case["op"] == "phmsd_energy" else 8.0 * N * N
    f = 2 * 0.6 * case["ndet"] * per_conf
    f += products if case["op"] == "phmsd_energy" else 2 * 8.0 * N * M * M + 2 * mac * M * M * K
    out = 64.0 if case["op"] == "phmsd_energy" else 16.0 * K
    return {"bytes": 2 * walkers + 8.0 * M * M * K + out * W, "flops": W * f}


# ---------------------------------------------------------------------------------- 64 bits
def _t(a):
    t = torch.from_numpy(np.ascontiguousarray(a))
    return t.cuda() if torch.cuda.is_available() else t


def _c(a):
    return _t(a).to(torch.complex128)


def _wrap(a):
    return torch.remainder(a + math.pi, 2 * math.pi) - math.pi


def _logdet(T):
    sign, logabs = torch.linalg.slogdet(T)
    return torch.complex(logabs, torch.angle(sign))


def _green(PsiT, phi):
    """(G [W][N][M], log det T) of T = PsiT phi."""
    T = torch.matmul(PsiT, phi)
    return torch.linalg.solve(T.transpose(1, 2).contiguous(), phi.transpose(1, 2).contiguous()), _logdet(T)


class _Setup:
    def __init__(self, x):
        self.h, self.L, self.PsiT = _c(x["h"]), _t(x["L"]), _c(x["PsiT"])
        M, K, N = self.L.shape[0], self.L.shape[2], self.PsiT.shape[0]
        self.M, self.N, self.K = M, N, K
        self.haj = self.PsiT @ self.h
        flat = self.L.reshape(M, M * K).to(torch.complex128)
        self.Lnak = (self.PsiT @ flat).reshape(N, M, K).permute(2, 0, 1).contiguous()
        self.Lij = self.L.reshape(M * M, K).to(torch.complex128)

    def propagator(self):
        phi0 = self.PsiT.conj().T.contiguous()[None]
        self.vmf = self.vbias(_green(self.PsiT, phi0)[0])[0].real
        v0 = -0.5 * torch.matmul(self.L.reshape(self.M, -1), self.L.reshape(self.M, -1).T)
        h1 = DT * (self.h.real + v0) + math.sqrt(DT) * (self.L @ self.vmf)
        h1 = 0.5 * (h1 + h1.T)
        e, u = torch.linalg.eigh(h1)
        p1 = (u * torch.exp(-0.5 * e)) @ u.T
        self.P1 = torch.where(p1.abs() > 1e-8, p1, torch.zeros_like(p1)).to(torch.complex128)

    def vbias(self, G):
        return 2 * math.sqrt(DT) * (G.reshape(len(G), -1) @ self.Lnak.reshape(self.K, -1).T)

    def vhs(self, X):
        return math.sqrt(DT) * (X @ self.Lij.T).reshape(len(X), self.M, self.M)

    def energy(self, G):
        W = len(G)
        e1 = 2 * (G * self.haj).sum((1, 2))
        exx, ej = torch.zeros_like(e1), torch.zeros_like(e1)
        rows = G.reshape(W * self.N, self.M)
        step = max(1, (1 << 27) // max(1, W * self.N * self.N))
        for n in range(0, self.K, step):
            L = self.Lnak[n:n + step]
            T = (rows @ L.reshape(-1, self.M).T).reshape(W, self.N, len(L), self.N).permute(0, 2, 1, 3)
            exx -= (T * T.transpose(2, 3)).sum((1, 2, 3))
            ej += 2 * (torch.diagonal(T, dim1=2, dim2=3).sum(2) ** 2).sum(1)
        return torch.stack([e1, exx, ej], 1)

    def overlap(self, phi):
        return 2 * _logdet(torch.matmul(self.PsiT, phi))


def _propagate(phi, P1, V, adjoint=False):
    P = P1.conj().T if adjoint else P1
    s = P @ phi
    t = s
    A = -1j * V.conj().transpose(1, 2) if adjoint else 1j * V
    for k in range(1, 7):
        t = torch.matmul(A, t) / k
        s = s + t
    return P @ s


def _qr(phi):
    q, r = torch.linalg.qr(phi)
    d = torch.diagonal(r, dim1=1, dim2=2)
    phase = d / d.abs()
    return q * phase[:, None, :], torch.log(d.abs()).sum(1).to(torch.complex128)


def _bounded(z, bound=50.0):
    a = z.abs()
    return torch.where(a > bound, z * (bound / a), z)


def _exact_steps(case, x):
    S = _Setup(x)
    S.propagator()
    phi, W = _c(x["phi"]), case["W"]
    weight, phase = _c(x["weight"]), torch.ones(W, dtype=torch.complex128, device=_t(x["h"]).device)
    theta = torch.zeros_like(weight)
    G, logdet = _green(S.PsiT, phi)
    ov, E = 2 * logdet, S.energy(G)
    pseudo = E.sum(1)
    hybrid = case.get("hybrid", True)
    shift = float(((weight * E.sum(1)).sum() / weight.sum()).real)
    lo, hi = shift - math.sqrt(2 / DT), shift + 10 * math.sqrt(2 / DT)
    for t in range(case.get("steps", 0)):
        vb = _bounded(S.vbias(_green(S.PsiT, phi)[0]))
        vm = _bounded(S.vmf.to(torch.complex128))
        vdiff = 1j * (vb - vm)
        X = _t(x["xi"][t]) + vdiff
        hw = -(vdiff * (X - 0.5 * vdiff)).sum(1)
        xv = X @ S.vmf.to(torch.complex128)
        mf = torch.complex(-0.5 * (S.vmf ** 2).sum() - xv.imag, xv.real)
        phi = _propagate(phi, S.P1, S.vhs(X))
        G, logdet = _green(S.PsiT, phi)
        new = 2 * logdet
        dtheta = new.imag - ov.imag - mf.imag
        scale = torch.clamp(torch.cos(dtheta), min=0.0)
        if hybrid:
            eloc = (mf - hw - (new - ov)) / DT
        else:
            E = S.energy(G)
            eloc = E.sum(1)
        eloc = torch.complex(eloc.real.clamp(lo, hi), eloc.imag)
        eff = eloc if hybrid else 0.5 * (eloc + pseudo)
        weight = weight * scale * torch.exp(-DT * (eff.real - shift))
        cap = max(100.0, 0.1 * W)
        weight = torch.where(weight.abs() > cap, weight * (cap / weight.abs()), weight)
        phase = phase * torch.exp(-1j * DT * eff.imag)
        theta, pseudo, ov = dtheta.to(torch.complex128), eloc, new
    if case["op"] == "orthogonalize" or case["steps"] > 1:
        phi = _qr(phi)[0]
        ov = S.overlap(phi)
    p = torch.zeros((W, COUNT), dtype=torch.complex128, device=phi.device)
    for k, v in ((WEIGHT, weight), (PHASE, phase), (PSEUDO_ELOC, pseudo), (OVLP, ov),
                 (IS_UNITARY, 1.0), (THETA, theta)):
        p[:, k] = v
    p[:, E1:EJ + 1] = E
    return {"slater": phi.reshape(W, -1), "properties": p}


def _exact_back_propagate(case, x):
    S = _Setup(x)
    S.propagator()
    W, n = case["W"], case["nback"]
    fields = _c(x["fields"])
    refs = S.PsiT.conj().T.contiguous().expand(W, S.M, S.N)
    logdet = torch.zeros(W, dtype=torch.complex128, device=refs.device)
    for ni in range(n - 1, -1, -1):     # the ring was just filled: its last slot is the newest
        refs = _propagate(refs, S.P1, S.vhs(fields[:, ni].contiguous()), adjoint=True)
        if ni == 0 or ni % case["nstab"] == 0:
            refs, ld = _qr(refs)
            logdet = logdet + ld
    return {"refs": refs[:, None], "logdet": logdet[:, None]}


def _exact_phmsd(case, x):
    """Every determinant explicitly: per spin and unique occupation its overlap, one-body and
    exchange energy and Cholesky traces, then the CI-weighted sums."""
    A, L, ci = _c(x["orbitals"]), _t(x["L"]), _c(x["ci"]).conj()
    M, K = L.shape[0], L.shape[2]
    N, W = case["N"], case["W"]
    energy = case["op"] == "phmsd_energy"
    Lna = (A @ L.reshape(M, M * K).to(torch.complex128)).reshape(M, M, K).permute(2, 0, 1).contiguous()
    haj = A @ _c(x["h"])
    index, ratio, e1, exx, ke = [], [], [], [], []
    ref_phase, ref_log = 0.0, 0.0
    for s, key in enumerate(("up", "dn")):
        phi = _c(x[key])
        occ = x["occs"][:, s * N:(s + 1) * N] - s * M
        unique, inverse = np.unique(occ, axis=0, return_inverse=True)
        inverse = inverse.reshape(-1)
        index.append(inverse)
        rows = torch.matmul(A, phi)                                   # [W][M][N]: A phi
        hrow = torch.matmul(haj, phi)
        P = torch.matmul(Lna.reshape(K * M, M), phi).reshape(W, K, M, N)
        lds = []
        part = ([], [], [])
        for conf in unique:
            c = torch.from_numpy(conf.astype(np.int64)).to(phi.device)
            T = rows[:, c].contiguous()
            lds.append(_logdet(T))
            Ti = torch.linalg.inv(T)
            part[0].append(torch.einsum("wab,wba->w", hrow[:, c], Ti))
            Y = torch.matmul(P[:, :, c].reshape(W, K * N, N), Ti).reshape(W, K, N, N)
            part[2].append(torch.diagonal(Y, dim1=2, dim2=3).sum(2))
            if energy:
                part[1].append(-0.5 * (Y * Y.transpose(2, 3)).sum((1, 2, 3)))
        ref = lds[int(inverse[0])]
        ref_log = ref_log + ref.real
        ref_phase = _wrap(ref_phase + ref.imag)
        ratio.append(torch.exp(torch.stack(lds) - ref))
        e1.append(torch.stack(part[0]))
        exx.append(torch.stack(part[1]) if energy else None)
        ke.append(torch.stack(part[2]))
    total = torch.zeros(W, dtype=torch.complex128, device=A.device)
    acc = torch.zeros((W, 3), dtype=torch.complex128, device=A.device)
    trace = torch.zeros((W, K), dtype=torch.complex128, device=A.device)
    for k in range(len(ci)):
        u, d = int(index[0][k]), int(index[1][k])
        o = ci[k] * ratio[0][u] * ratio[1][d]
        total = total + o
        kk = ke[0][u] + ke[1][d]
        if energy:
            acc[:, 0] += o * (e1[0][u] + e1[1][d])
            acc[:, 1] += o * (exx[0][u] + exx[1][d])
            acc[:, 2] += o * 0.5 * (kk * kk).sum(1)
        else:
            trace += o[:, None] * kk
    if not energy:
        return {"vbias": math.sqrt(DT) * trace / total[:, None]}
    log = torch.log(total)
    return {"E": acc / total[:, None], "log_overlap": log + torch.complex(ref_log, ref_phase)}


def exact(case, seed):
    x = _inputs(case, seed)
    if case["op"].startswith("phmsd"):
        return _exact_phmsd(case, x)
    if case["op"] == "back_propagate":
        return _exact_back_propagate(case, x)
    if case["op"] == "energy":
        S = _Setup(x)
        G, logdet = _green(S.PsiT, _c(x["phi"]))
        return {"E": S.energy(G), "log_overlap": 2 * logdet}
    return _exact_steps(case, x)

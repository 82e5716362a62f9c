"""The performance cases of mcpi_amd: what its users run, over the range of
sizes, types of Hamiltonian and storage modes that they run it at.

The framework's work is exact diagonalization in the Fock space of N bosons in
M orbitals: H.v on device vectors, Lanczos ground states (one at a time, or
many at once), and the density matrices with the energy's gradient.  Two kinds
of Hamiltonian occur: Lieb-Liniger (diagonal Ho, contact interaction that
conserves momentum: few non-zero couplings) and dense (random Hermitian Ho and
bosonic Hint, as variational orbitals give).  Vectors are complex128.

Device vectors are torch tensors handed to the library by address.  A program
builds the tables of its basis once and keeps them: the states prepared one
after another for the same basis share it.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import mcpi_amd
import mcpi_amd.reference

# ------------------------------------------------------------------ cases --


def listed():
    return [
        # H.v at the smallest size that the batched ground states use: a
        # program that iterates on its own, where the call itself counts
        {"name": "hv_small", "kind": "hv", "ham": "ll", "N": 6, "M": 9, "maps": "full", "skip": True, "g": 2.0},
        # H.v of the ordinary Lieb-Liniger size, every map on the device
        {"name": "hv_ll", "kind": "hv", "ham": "ll", "N": 12, "M": 12, "maps": "full", "skip": True, "g": 10.0},
        # H.v of the largest size: 13 million configurations, single-jump map
        {"name": "hv_ll_large", "kind": "hv", "ham": "ll", "N": 16, "M": 12, "maps": "single", "skip": True,
         "g": 50.0},
        # H.v with all couplings present (a dense Hamiltonian)
        {"name": "hv_dense", "kind": "hv", "ham": "dense", "N": 10, "M": 12, "maps": "full", "skip": True, "g": 0.0},
        # H.v that evaluates every term from the stored maps, as the
        # reference does (zero-skipping off)
        {"name": "hv_every_term", "kind": "hv", "ham": "ll", "N": 12, "M": 12, "maps": "full", "skip": False,
         "g": 10.0},
        # the reference's own call on host tables and host vectors, as a
        # program written against its headers makes it inside its loop
        {"name": "hv_host", "kind": "host", "ham": "ll", "N": 8, "M": 11, "g": 5.0},
        # Lieb-Liniger ground state of five particles in 21 orbitals (the
        # reference's published table): odd sizes, many steps of a short vector
        {"name": "ground_m21", "kind": "ground", "ham": "ll", "N": 5, "M": 21, "maps": "full", "g": 30.0, "lm": 400},
        # ground state of the largest basis: long vectors, few steps
        {"name": "ground_large", "kind": "ground", "ham": "ll", "N": 16, "M": 12, "maps": "single", "g": 50.0,
         "lm": 60},
        # energy and its gradient over Ho and Hint for a dense Hamiltonian:
        # the forward solve and the adjoint
        {"name": "adjoint_dense", "kind": "adjoint", "ham": "dense", "N": 10, "M": 12, "maps": "full", "g": 0.0,
         "lm": 300},
        # a scan over 64 couplings and three bases in one call
        {"name": "batched", "kind": "batched", "ham": "ll", "count": 64, "shapes": "6,9 8,11 10,13", "lm": 120,
         "pick": 64120},
        # one- and two-body density matrices (the gradient) of a given state
        {"name": "vjp", "kind": "vjp", "N": 12, "M": 12},
        # the same at the largest basis
        {"name": "vjp_large", "kind": "vjp", "N": 16, "M": 12},
    ]


def _nc(N, M):
    return math.comb(N + M - 1, N)


def _full_bytes(N, M):
    """Bytes of the jump maps of a basis with all of them stored."""
    nu2 = _nc(N - 2, M)
    return 4 * M * M * (_nc(N, M) + (M + M * (M - 1) // 2) * nu2)


def _size(rng, orbitals, lo, hi):
    """(N, M): M of the given range, the number of configurations spread over
    lo .. hi evenly in its logarithm."""
    while True:
        M = rng.randint(*orbitals)
        want = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        N = 2
        while _nc(N, M) < want and N < 100:
            N += 1
        if lo <= _nc(N, M) <= hi:
            return N, M


def _coupling(rng):
    return round(10 ** rng.uniform(-1, 2), 3)


def draw(rng):
    kind = rng.choice(["hv", "hv", "hv", "ground", "ground", "adjoint", "batched", "vjp", "host"])
    if kind == "hv":
        ham = rng.choice(["ll", "ll", "dense"])
        # no specialised kernel covers a dense Hamiltonian beyond 13 orbitals
        N, M = _size(rng, (3, 24), 300, 13_037_895) if ham == "ll" else _size(rng, (4, 13), 300, 1_352_078)
        modes = ["single", "none"] + (["full", "full"] if _nc(N, M) <= 2_000_000 and _full_bytes(N, M) < 2e10 else [])
        if ham == "ll" and M <= 13:
            modes.append("sectors")
        return {"kind": kind, "ham": ham, "N": N, "M": M, "maps": rng.choice(modes), "skip": True,
                "g": _coupling(rng) if ham == "ll" else 0.0}
    if kind == "host":
        N, M = _size(rng, (4, 13), 300, 50_000)
        return {"kind": kind, "ham": rng.choice(["ll", "dense"]), "N": N, "M": M, "g": _coupling(rng)}
    if kind == "batched":
        shapes = [_size(rng, (5, 13), 300, 200_000) for _ in range(rng.randint(1, 3))]
        return {"kind": kind, "ham": "ll", "count": rng.randint(4, 40),
                "shapes": " ".join("%d,%d" % s for s in shapes), "lm": rng.randint(20, 120),
                "pick": rng.randrange(1 << 30)}
    if kind == "vjp":
        N, M = _size(rng, (3, 24), 300, 2_000_000)
        return {"kind": kind, "N": N, "M": M}
    ham = "dense" if kind == "adjoint" else rng.choice(["ll", "ll", "dense"])
    N, M = _size(rng, (4, 12), 300, 400_000) if ham == "dense" else _size(rng, (4, 24), 300, 1_400_000)
    return {"kind": kind, "ham": ham, "N": N, "M": M,
            "maps": "full" if _full_bytes(N, M) < 2e10 else "single",
            "g": _coupling(rng) if ham == "ll" else 0.0, "lm": rng.randint(20, 200)}


# ----------------------------------------------------------------- inputs --


class TorchVector(mcpi_amd.DeviceArray):
    """A torch tensor's memory as the library's device vector (torch owns it)."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.n = tensor.numel()
        self.dtype = np.dtype(np.complex128)
        self.nbytes = self.n * self.dtype.itemsize
        self.ptr = tensor.data_ptr()

    def free(self):
        self.ptr = None

    close = free


_kept = {}   # the bases of the program that runs now


def _keep(key, make, wanted):
    """The table set `key`, made once and kept while cases of the same bases
    (`wanted`) follow."""
    for old in [k for k in _kept if k not in wanted]:
        del _kept[old]
    if key not in _kept:
        _kept[key] = make()
    return _kept[key]


def _basis(N, M, maps, wanted=None):
    key = (N, M, maps)

    def make():
        if maps == "sectors":   # rows sorted by total momentum
            return mcpi_amd.Basis(N, M, "single", charge=np.arange(M))
        return mcpi_amd.Basis(N, M, maps)

    return _keep(key, make, wanted or [key])


def _vector(nc, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    v = torch.randn(nc, dtype=torch.complex128, device="cuda", generator=gen)
    return v / torch.linalg.vector_norm(v)


def _hamiltonian(case, seed):
    """Ho, Hint: Lieb-Liniger on a ring of length 1, or random Hermitian Ho and
    random Hint with the bosonic symmetries (entries of size 0.1)."""
    M = case["M"]
    if case["ham"] == "ll":
        return mcpi_amd.ll_ho(M), mcpi_amd.ll_hint(M, case["g"])
    rng = np.random.default_rng(seed)
    A = 0.1 * (rng.standard_normal((M, M)) + 1j * rng.standard_normal((M, M)))
    B = 0.1 * (rng.standard_normal((M,) * 4) + 1j * rng.standard_normal((M,) * 4))
    B = 0.5 * (B + B.transpose(1, 0, 2, 3))
    B = 0.5 * (B + B.transpose(0, 1, 3, 2))
    return 0.5 * (A + A.conj().T), 0.5 * (B + np.conj(B.transpose(2, 3, 0, 1)))


def _instances(case):
    """[(N, M, g)] of a batched case: shapes and couplings of its scan."""
    shapes = [tuple(int(x) for x in s.split(",")) for s in case["shapes"].split()]
    rng = np.random.default_rng(case["pick"])
    picks = rng.integers(0, len(shapes), case["count"])
    gs = 10 ** rng.uniform(-1, 2, case["count"])
    return [(*shapes[int(p)], float(g)) for p, g in zip(picks, gs)]


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "batched":
        inst = _instances(case)
        wanted = [(N, M, "full") for N, M, _ in inst]
        s["lm"] = case["lm"]
        s["hams"] = [mcpi_amd.Hamiltonian(_basis(N, M, "full", wanted), mcpi_amd.ll_ho(M), mcpi_amd.ll_hint(M, g))
                     for N, M, g in inst]
        size = [_nc(N, M) for N, M, _ in inst]
        s["starts"] = [TorchVector(_vector(n, 1000 * seed + x)) for x, n in enumerate(size)]
        s["vectors"] = torch.empty(sum(size), dtype=torch.complex128, device="cuda")
        s["outs"] = [TorchVector(v) for v in s["vectors"].split(size)]
        return s
    N, M = case["N"], case["M"]
    if kind == "host":
        key = (N, M, "host")
        s["tables"] = _keep(key, lambda: mcpi_amd.reference.RefBasis(N, M), [key])
        s["C"] = _vector(_nc(N, M), seed).cpu().numpy()
        s["Ho"], s["Hint"] = _hamiltonian(case, seed)
        return s
    basis = _basis(N, M, "single" if kind == "vjp" else case["maps"])
    s["basis"] = basis
    s["C"] = TorchVector(_vector(basis.nc, seed))
    if kind == "vjp":
        return s
    s["H"] = mcpi_amd.Hamiltonian(basis, *_hamiltonian(case, seed), skip_zero=case.get("skip", True))
    s["lm"] = case.get("lm", 0)
    s["out"] = TorchVector(torch.empty(basis.nc, dtype=torch.complex128, device="cuda"))
    return s


# -------------------------------------------------------------------- run --


def run(s):
    kind = s["kind"]
    if kind == "hv":
        s["H"].apply(s["C"], s["out"])
        return s["out"].tensor
    if kind == "host":
        return s["tables"].applyHconf_omp(s["C"], s["Ho"], s["Hint"])
    if kind == "vjp":
        return list(s["basis"].vjp(s["C"]))
    if kind == "batched":
        E0, steps = mcpi_amd.lanczos_batched(s["hams"], s["starts"], s["lm"], s["outs"])
        return {"E0": E0, "steps": steps, "vectors": s["vectors"]}
    E0, vec, steps = s["H"].ground(s["lm"], s["C"], out=s["out"])
    got = {"E0": E0, "steps": steps, "vector": vec.tensor}
    if kind == "adjoint":
        got["dHo"], got["dHint"] = s["basis"].vjp(vec)
    return got


# ------------------------------------------------------------------- work --


def _hv_work(ham, N, M, skip=True):
    """Bytes and real operations of one H.v: both vectors once, and (every
    term from stored maps) the target of each rule term once; the pair
    amplitudes, their sums or products, and the way back."""
    nc, nu2, NP = _nc(N, M), _nc(N - 2, M), M * (M + 1) // 2
    b, f = 32 * nc, 8 * NP * nu2
    if not skip:
        pairs1, pairs2 = M * (M - 1) // 2, (M - 1) * (M - 2) // 2
        b += 4 * (M * (M - 1) * _nc(N - 1, M) + (M * pairs1 + M * (M - 1) // 2 * pairs2) * nu2)
        f = 4 * (M * pairs1 + M * (M - 1) // 2 * pairs2) * nu2
    elif ham == "dense":
        f += 6 * NP * NP * nu2
    return b, f


def _lanczos_work(ham, N, M, lm):
    """lm steps: an H.v each, and every earlier vector read for the dots and
    once more for the update (8 real operations a complex pair)."""
    b, f = _hv_work(ham, N, M)
    nc, pairs = _nc(N, M), lm * (lm + 1) // 2 - 1
    return lm * b + 32 * nc * pairs + 16 * nc * lm, lm * f + 16 * nc * pairs + 4 * nc * lm


def _vjp_work(N, M):
    NP = M * (M + 1) // 2
    return 16 * (_nc(N, M) + M ** 2 + M ** 4), 4 * NP * (NP + 1) * _nc(N - 2, M) + 4 * M * (M + 1) * _nc(N - 1, M)


def work(case):
    kind = case["kind"]
    if kind == "batched":
        parts = [_lanczos_work("ll", N, M, case["lm"]) for N, M, _ in _instances(case)]
    elif kind == "vjp":
        parts = [_vjp_work(case["N"], case["M"])]
    elif kind in ("hv", "host"):
        parts = [_hv_work(case["ham"], case["N"], case["M"], case.get("skip", True))]
    else:
        parts = [_lanczos_work(case["ham"], case["N"], case["M"], case["lm"])]
        if kind == "adjoint":
            parts.append(_vjp_work(case["N"], case["M"]))
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


# ------------------------------------------------------------------ exact --


class _Fock:
    """The basis of N bosons in M orbitals in plain torch: occupations of the
    states in the reference's order, and their ranks."""

    def __init__(self, N, M):
        self.N, self.M, self.nc = N, M, _nc(N, M)
        # C(p + j - 1, j) for p particles below orbital j
        self.B = torch.tensor([[math.comb(p + j - 1, j) if j else 0 for p in range(N + 1)] for j in range(M)],
                              device="cuda")

    def states(self):
        left = self.nc - 1 - torch.arange(self.nc, device="cuda")
        above = torch.full((self.nc,), self.N, device="cuda")
        v = torch.empty((self.M, self.nc), dtype=torch.int64, device="cuda")
        for j in range(self.M - 1, 0, -1):
            below = torch.searchsorted(self.B[j], left, right=True) - 1
            v[j] = above - below
            left = left - self.B[j][below]
            above = below
        v[0] = above
        return v

    def rank(self, v):
        total, below = torch.zeros_like(v[0]), torch.zeros_like(v[0])
        for j in range(1, self.M):
            below = below + v[j - 1]
            total = total + self.B[j][below]
        return self.nc - 1 - total


class _PairSpace:
    """<u|a_q a_l|C> over the states u of N - 2 particles and pairs q <= l."""

    def __init__(self, N, M):
        self.N, self.M = N, M
        big, small = _Fock(N, M), _Fock(N - 2, M)
        u = small.states()
        self.nc = big.nc
        self.pairs = [(q, l) for l in range(M) for q in range(l + 1)]
        self.at = torch.empty((len(self.pairs), small.nc), dtype=torch.int64, device="cuda")
        self.f = torch.empty((len(self.pairs), small.nc), dtype=torch.float64, device="cuda")
        for x, (q, l) in enumerate(self.pairs):
            self.f[x] = torch.sqrt(((u[q] + 1) * (u[l] + 1 + (q == l))).double())
            w = u.clone()
            w[q] += 1
            w[l] += 1
            self.at[x] = big.rank(w)

    def amplitudes(self, C):
        return C[self.at] * self.f

    def back(self, Y):
        """sum over pairs of (a*_q a*_l Y_ql)"""
        out = torch.zeros(self.nc, dtype=torch.complex128, device="cuda")
        return out.index_add_(0, self.at.reshape(-1), (Y * self.f).reshape(-1))


def _operator(P, Ho, Hint):
    """H.v of sum Ho a*a + 1/2 sum Hint a*a*aa through the pair space P (the
    one-body part by a*_k a_l = sum_s a*_k a*_s a_s a_l / (N - 1))."""
    N, M = P.N, P.M
    T = 0.5 * Hint.transpose(0, 1, 3, 2) + np.einsum("kl,st->kslt", Ho, np.eye(M)) / (N - 1)
    W = np.zeros((len(P.pairs),) * 2, np.complex128)
    index = {}
    for x, (q, l) in enumerate(P.pairs):
        index[q, l] = index[l, q] = x
    at = np.array([[index[k, s] for s in range(M)] for k in range(M)]).reshape(-1)
    np.add.at(W, (at[:, None], at[None, :]), T.reshape(M * M, M * M))
    W = torch.from_numpy(W).cuda()
    return lambda C: P.back(W @ P.amplitudes(C))


def _lowest(apply, C, lm):
    """Ritz value and vector of lm Lanczos steps from C."""
    V, alpha, beta = torch.empty((lm, C.numel()), dtype=torch.complex128, device="cuda"), [], []
    V[0] = C
    for i in range(lm):
        w = apply(V[i])
        alpha.append(float(torch.vdot(V[i], w).real))
        if i + 1 == lm:
            break
        for _ in range(2):
            w = w - V[:i + 1].T @ (V[:i + 1].conj() @ w)
        beta.append(float(torch.linalg.vector_norm(w)))
        V[i + 1] = w / beta[-1]
    E, z = np.linalg.eigh(np.diag(alpha) + np.diag(beta, 1) + np.diag(beta, -1))
    return float(E[0]), V.T @ torch.from_numpy(z[:, 0]).cuda().to(V.dtype)


def _densities(N, M, C, scale):
    """rho1, and scale times rho2, of the vector C."""
    f = _Fock(N, M)
    u = _Fock(N - 1, M).states()
    rows = []
    for k in range(M):
        w = u.clone()
        w[k] += 1
        rows.append(C[f.rank(w)] * torch.sqrt((u[k] + 1).double()))
    A = torch.stack(rows)
    P = _PairSpace(N, M)
    X = P.amplitudes(C)
    G1, G2 = A.conj() @ A.T, X.conj() @ X.T
    at = torch.tensor([[max(a, b) * (max(a, b) + 1) // 2 + min(a, b) for b in range(M)] for a in range(M)])
    return G1.cpu().numpy(), scale * G2.cpu().numpy()[at[:, :, None, None], at[None, None, :, :]]


def exact(case, seed):
    """What run() returns, in plain torch in 64 bits.  An eigenvector's sign
    is arbitrary: no value for it."""
    kind = case["kind"]
    if kind == "batched":
        inst, E, P = _instances(case), [], {}
        for x, (N, M, g) in enumerate(inst):
            if (N, M) not in P:
                P[N, M] = _PairSpace(N, M)
            apply = _operator(P[N, M], mcpi_amd.ll_ho(M), mcpi_amd.ll_hint(M, g))
            E.append(_lowest(apply, _vector(_nc(N, M), 1000 * seed + x), case["lm"])[0])
        return {"E0": np.array(E), "steps": None, "vectors": None}
    N, M = case["N"], case["M"]
    C = _vector(_nc(N, M), seed)
    if kind == "vjp":
        return list(_densities(N, M, C, 0.5))
    apply = _operator(_PairSpace(N, M), *_hamiltonian(case, seed))
    if kind == "hv":
        return apply(C)
    if kind == "host":
        return apply(C).cpu().numpy()
    E, v = _lowest(apply, C, case["lm"])
    got = {"E0": E, "steps": None, "vector": None}
    if kind == "adjoint":
        got["dHo"], got["dHint"] = _densities(N, M, v, 0.5)
    return got

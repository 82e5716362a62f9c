"""Lanczos chains whose sums are formed inside other kernels: segment and group
edges, breakdowns, many instances, against the oracle."""
import numpy as np
import pytest

import mcpi_amd
import oracle
from tests.gpu_util import note

pytestmark = pytest.mark.gpu


def _unit(n, seed):
    rng = np.random.default_rng(seed)
    v = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    return v / np.linalg.norm(v)


# rows: 15, 210 (below one segment of 512 or 1024), 1,287, 3,003 and 6,188
# (several); steps: 2, one group of 32 vectors less and more one, several
@pytest.mark.parametrize("N,M,lm", [(2, 5, 14), (4, 7, 2), (4, 7, 31), (5, 9, 33), (5, 9, 66), (6, 9, 40), (12, 6, 45)])
def test_ground_state_short(oracle_lib, N, M, lm):
    note(f"short chain N={N} M={M} lm={lm}")
    o = oracle.Basis(N, M)
    _, Ho, Hint = oracle.random_inputs(N, M, seed=N + M)
    v = _unit(o.nc, 3 * lm)
    b = mcpi_amd.Basis(N, M, "single")
    H = mcpi_amd.Hamiltonian(b, Ho, Hint)
    E, psi, steps = H.ground(lm, v)
    E_o, psi_o, steps_o = o.ground(lm, v, Ho, Hint)
    scale = max(1.0, abs(E_o))
    assert steps == steps_o
    assert abs(E - E_o) <= 1e-10 * scale
    assert abs(abs(np.vdot(psi.numpy(), psi_o)) - 1) < 1e-8


def test_lanczos_basis_orthonormal():
    """The Krylov basis that mcpi_hip_lanczos returns: V V^H = 1 and V H V^H =
    T to rounding (chains with and without sums of their own)."""
    for N, M, lm in ((5, 9, 50), (8, 12, 40)):
        note(f"krylov basis N={N} M={M} lm={lm}")
        b = mcpi_amd.Basis(N, M, "single")
        H = mcpi_amd.Hamiltonian(b, mcpi_amd.ll_ho(M), mcpi_amd.ll_hint(M, 2.0))
        C0 = mcpi_amd.DeviceArray.from_numpy(_unit(b.nc, 9))
        lvec = mcpi_amd.DeviceArray(b.nc * lm)
        steps, diag, off = H.lanczos(lm, C0, lvec)
        V = lvec.numpy().reshape(lm, b.nc)
        assert steps == lm
        # one pass of classical Gram-Schmidt a step (at most 50): a few hundred ulps
        assert np.abs(V.conj() @ V.T - np.eye(lm)).max() < 1e-12
        HV = np.array([H(V[t]) for t in range(lm)])
        T = np.diag(diag.real) + np.diag(off.real[:-1], 1) + np.diag(off.real[:-1], -1)
        assert np.abs(V.conj() @ HV.T - T).max() < 1e-11 * np.abs(T).max()


def test_mixed_chains_and_breakdown(oracle_lib):
    """Short and long vectors in one call (no sums inside), and all short ones
    with an instance that breaks down (a two-state basis) beside others."""
    for spec, lm in (([(5, 9), (9, 13), (4, 6)], 20), ([(1, 2), (5, 9), (4, 6)], 40)):
        note(f"mixed chains {spec}")
        bases = [mcpi_amd.Basis(N, M, "single") for N, M in spec]
        mats = [oracle.random_inputs(N, M, seed=N)[1:] for N, M in spec]
        hams = [mcpi_amd.Hamiltonian(b, *m) for b, m in zip(bases, mats)]
        vs = [_unit(b.nc, 5) for b in bases]
        starts = [mcpi_amd.DeviceArray.from_numpy(v) for v in vs]
        E, steps = mcpi_amd.lanczos_batched(hams, starts, lm)
        for x, (N, M) in enumerate(spec):
            if (N, M) == (9, 13):
                E1, _, st = hams[x].ground(lm, starts[x])
                assert steps[x] == st and abs(E[x] - E1) <= 1e-10 * max(1.0, abs(E1))
                continue
            E_o, _, st = oracle.Basis(N, M).ground(lm, vs[x], *mats[x])
            assert steps[x] == st and abs(E[x] - E_o) <= 1e-10 * max(1.0, abs(E_o)), (x, E[x], E_o)

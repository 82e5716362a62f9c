"""Lanczos steps of one instance whose pair-space H.v subtracts beta v_i and
leaves the partials of alpha: the Lanczos relation V^H H V = T, with H applied
on its own, by terms, through the two passes (whole rows, rows shared by
wavefronts, three words of occupations) and through the pair product; a
schedule that does not do it (the last) beside them."""
import numpy as np
import pytest

import mcpi_amd
import oracle
from tests.gpu_util import note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,M,kind,schedule", [(2, 3, "ll", 7), (6, 9, "ll", 7), (7, 10, "ll", 7), (9, 11, "ll", 7),
                                               (10, 12, "ll", 7), (3, 21, "ll", 7), (2, 5, "dense", 6),
                                               (5, 8, "dense", 6), (9, 11, "dense", 6), (1, 4, "dense", 6),
                                               (7, 10, "ll", 2)])
def test_lanczos_relation(oracle_lib, N, M, kind, schedule):
    note(f"step epilogue N={N} M={M} {kind} schedule={schedule}")
    b = mcpi_amd.Basis(N, M, "single")
    Ho, Hint = (oracle.ll_ho(M), oracle.ll_hint(M, 2.0)) if kind == "ll" else oracle.random_inputs(N, M, seed=N)[1:]
    H = mcpi_amd.Hamiltonian(b, Ho, Hint, schedule=schedule)
    rng = np.random.default_rng(M)
    v = rng.standard_normal(b.nc) + 1j * rng.standard_normal(b.nc)
    lm = min(9, b.nc - 1)
    lvec = mcpi_amd.DeviceArray(b.nc * lm)
    steps, diag, off = H.lanczos(lm, mcpi_amd.DeviceArray.from_numpy(v / np.linalg.norm(v)), lvec)
    # (a start in few sectors may end early)
    V = lvec.numpy().reshape(lm, b.nc)[:steps]
    HV = np.array([H(x) for x in V])
    T = np.diag(diag.real[:steps]) + np.diag(off.real[:steps - 1], 1) + np.diag(off.real[:steps - 1], -1)
    # one pass of Gram-Schmidt a step over nine steps: tens of ulps of |H|
    assert np.abs(V.conj() @ V.T - np.eye(steps)).max() < 1e-12
    assert np.abs(V.conj() @ HV.T - T).max() < 1e-12 * max(1.0, np.abs(T).max()) * lm

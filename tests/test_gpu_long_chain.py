"""Lanczos chains of one mid-size instance at the length where the short-vector
kernels give way to the separate ones (basis vectors of 512 MB in all)."""
import numpy as np
import pytest

import mcpi_amd
from tests.gpu_util import note

pytestmark = pytest.mark.gpu


# 167,960 rows: 16 n lm = 2^29 lies between 199 and 200 steps
@pytest.mark.parametrize("lm", [199, 200])
def test_krylov_basis(lm):
    N, M = 9, 12
    note(f"Krylov basis N={N} M={M} lm={lm}")
    b = mcpi_amd.Basis(N, M, "single")
    H = mcpi_amd.Hamiltonian(b, mcpi_amd.ll_ho(M), mcpi_amd.ll_hint(M, 20.0))
    rng = np.random.default_rng(lm)
    v = rng.standard_normal(b.nc) + 1j * rng.standard_normal(b.nc)
    C0 = mcpi_amd.DeviceArray.from_numpy(v / np.linalg.norm(v))
    lvec = mcpi_amd.DeviceArray(b.nc * lm)
    steps, diag, off = H.lanczos(lm, C0, lvec)
    V = lvec.numpy().reshape(lm, b.nc)
    assert steps == lm
    # one pass of classical Gram-Schmidt a step, 200 at most
    assert np.abs(V.conj() @ V.T - np.eye(lm)).max() < 1e-12
    # H v_t = beta_{t-1} v_{t-1} + alpha_t v_t + beta_t v_{t+1}, relative to |H|
    scale = np.abs(diag).max() + 2 * np.abs(off).max()
    for t in (0, 1, 2, 31, 32, 33, 97, lm - 2):
        r = H(V[t]) - diag[t] * V[t] - off[t] * V[t + 1] - (off[t - 1] * V[t - 1] if t else 0)
        assert np.linalg.norm(r) < 1e-12 * scale, t

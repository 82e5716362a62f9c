"""Batched Lanczos over Hamiltonians of one basis whose pair matrices differ in
form (factorized with more or fewer blocks, or not), so that their coefficient
blocks differ past the tables that the number of orbitals alone gives."""
import numpy as np
import pytest

import mcpi_amd
import oracle
from tests.gpu_util import note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [0, 1, 2, 3])
@pytest.mark.parametrize("M,drops", [(8, (0, 1, 2, 3)), (8, (1, 2, 1)), (5, (2, 3, 2, 0)), (6, (0, 0, 1, 1, -1))])
def test_members_of_different_form(oracle_lib, M, drops, kind):
    N, lm = 5, 40
    note(f"batched forms M={M} drops={drops} kind={kind}")
    a = np.arange(M)
    K = a[:, None] + a[None, :]
    o = oracle.Basis(N, M)
    b = mcpi_amd.Basis(N, M, "full")
    rng = np.random.default_rng(M)
    hams, starts, refs = [], [], []
    for d in drops:
        Ho, Hint = mcpi_amd.ll_ho(M), mcpi_amd.ll_hint(M, 3.0)
        Hint = np.where(K[:, :, None, None] >= abs(d), Hint, 0)   # without the lowest total momenta
        if d < 0:
            Hint = Hint * (1 + 0.1 * np.add.outer(np.multiply.outer(a, a), np.multiply.outer(a, a)))   # blocks of rank two
        v = rng.standard_normal(b.nc) + 1j * rng.standard_normal(b.nc)
        v /= np.linalg.norm(v)
        hams.append(mcpi_amd.Hamiltonian(b, Ho, Hint))
        starts.append(mcpi_amd.DeviceArray.from_numpy(v))
        refs.append(o.ground(lm, v, Ho, Hint))
    mcpi_amd.set_batched_kernel(kind)
    try:
        E, steps = mcpi_amd.lanczos_batched(hams, starts, lm)
    finally:
        mcpi_amd.set_batched_kernel(0)
    for x, (E_o, _, steps_o) in enumerate(refs):
        assert steps[x] == steps_o and abs(E[x] - E_o) <= 1e-10 * max(1.0, abs(E_o)), (x, E[x], E_o)

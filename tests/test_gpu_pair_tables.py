"""Schedule 6 of a Hamiltonian in the factorized pair form, whose tables of the
pair product are laid out when the schedule first runs."""
import numpy as np
import pytest

import mcpi_amd
import oracle
from tests.gpu_util import assert_close, note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,M", [(1, 4), (2, 3), (5, 6), (6, 9), (3, 12), (9, 11)])
def test_product_on_a_factorized_hamiltonian(oracle_lib, N, M):
    note(f"pair product, factorized Hamiltonian N={N} M={M}")
    C, _, _ = oracle.random_inputs(N, M, seed=N + M)
    Ho, Hint = mcpi_amd.ll_ho(M), mcpi_amd.ll_hint(M, 4.0)
    ref = oracle.Basis(N, M).acth(C, Ho, Hint)
    b = mcpi_amd.Basis(N, M, "single")
    H = mcpi_amd.Hamiltonian(b, Ho, Hint)
    other = mcpi_amd.Hamiltonian(b, Ho, Hint, schedule=7)
    for schedule in (7, 6, 0, 6, 2):
        H.set_schedule(schedule)
        assert_close(H(C), ref, 1e-13, f"schedule {schedule}")
    assert_close(other(C), ref, 1e-13, "another Hamiltonian")


def test_members_of_which_one_has_run_the_product(oracle_lib):
    """Batched groups take Hamiltonians that have run the pair product beside
    others."""
    N, M, lm = 6, 8, 30
    note("batched after the pair product")
    o = oracle.Basis(N, M)
    b = mcpi_amd.Basis(N, M, "full")
    mats = [(mcpi_amd.ll_ho(M), mcpi_amd.ll_hint(M, g)) for g in (1.0, 5.0, 20.0)]
    hams = [mcpi_amd.Hamiltonian(b, *m) for m in mats]
    rng = np.random.default_rng(1)
    v = rng.standard_normal(b.nc) + 1j * rng.standard_normal(b.nc)
    v /= np.linalg.norm(v)
    hams[1].set_schedule(6)
    hams[1](v)
    for schedule in (0, 6):
        for H in hams:
            H.set_schedule(schedule)
        E, steps = mcpi_amd.lanczos_batched(hams, [mcpi_amd.DeviceArray.from_numpy(v)] * 3, lm)
        for x, m in enumerate(mats):
            E_o, _, st = o.ground(lm, v, *m)
            assert steps[x] == st and abs(E[x] - E_o) < 1e-10 * max(1.0, abs(E_o))

"""The pair product of the dense pair-space H.v (schedule 6) at the edges of its
row blocks, steps and pair groups, against the oracle."""
import pytest

import mcpi_amd
import oracle
from tests.gpu_util import assert_close, note

pytestmark = pytest.mark.gpu


# states of N - 2 particles: 1, 15, 20, 21 (two 16-row blocks), 126 (eight
# blocks: one an XCD), 136, 495, 792, 4,368; pairs 6 and 15 (one group of 16),
# 21 (two), 36 (three), 55 (four), 66 and 78 (five; 78 is no multiple of four)
@pytest.mark.parametrize("N,M", [(2, 3), (6, 3), (17, 3), (5, 4), (7, 6), (4, 6), (7, 5), (6, 9), (4, 10), (5, 11), (3, 12),
                                 (7, 12), (1, 5)])
def test_pair_product_edges(oracle_lib, N, M):
    note(f"pair product N={N} M={M}")
    o = oracle.Basis(N, M)
    C, Ho, Hint = oracle.random_inputs(N, M, seed=900 + 7 * N + M)
    b = mcpi_amd.Basis(N, M, "none")
    H = mcpi_amd.Hamiltonian(b, Ho, Hint, schedule=6)
    assert_close(H(C), o.acth(C, Ho, Hint), 1e-12, "schedule 6")
    # a second product in the same workspace
    C2 = C[::-1].copy()
    assert_close(H(C2), o.acth(C2, Ho, Hint), 1e-12, "again")

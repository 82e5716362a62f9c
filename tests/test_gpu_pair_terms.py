"""The factorized H.v term by term on bases of few rows, against the oracle and
against the two passes through the pair space (the Hamiltonian's term list
dropped), at the edges of its words of packed occupations, of its lists and of
the rule on the number of rows."""
import numpy as np
import pytest

import mcpi_amd
import oracle
from tests.gpu_util import assert_close, note
from tests.test_gpu_pairz import disguised

pytestmark = pytest.mark.gpu


def drop_terms(H):
    f = mcpi_amd.lib().mcpi_hip_ham_drop_terms
    f.argtypes = [mcpi_amd._vp]
    assert f(H.handle) == 0


# one row and three more a block; M at 8, 9, 16, 17 (words); few and many
# particles; 14 orbitals (511 terms) and 15 (more than are kept); 8,008 rows and
# 8,568 and 12,376 past the rule
@pytest.mark.parametrize("N,M", [(2, 3), (2, 4), (100, 3), (13, 5), (5, 8), (6, 9), (3, 14), (3, 15), (2, 24), (6, 11),
                                 (5, 14), (6, 12)])
@pytest.mark.parametrize("phases", [False, True])
def test_terms_and_passes(oracle_lib, N, M, phases):
    note(f"pair terms N={N} M={M} phases={phases}")
    o = oracle.Basis(N, M)
    C, _, _ = oracle.random_inputs(N, M, seed=N + M)
    Ho, Hint = disguised(M, 2.0, N + M, phases)
    H = mcpi_amd.Hamiltonian(mcpi_amd.Basis(N, M, "single"), Ho, Hint, schedule=7)
    ref = o.acth(C, Ho, Hint)
    # the sums have the same terms: rounding of a few tens of them
    assert_close(H(C), ref, 1e-13, "by terms")
    drop_terms(H)
    assert_close(H(C), ref, 1e-13, "two passes")


@pytest.mark.parametrize("phases", [False, True])
def test_infinite_entry(phases):
    """The entries of the result that an infinite entry of C reaches are the
    same ones by terms and through the two passes."""
    N, M = 5, 8
    note(f"pair terms infinite entry phases={phases}")
    b = mcpi_amd.Basis(N, M, "none")
    H = mcpi_amd.Hamiltonian(b, *disguised(M, 2.0, 3, phases), schedule=7)
    rng = np.random.default_rng(2)
    for j in (0, b.nc // 3, b.nc - 1):
        C = rng.standard_normal(b.nc) + 1j * rng.standard_normal(b.nc)
        C[j] = complex(np.inf, 1.0)
        H2 = mcpi_amd.Hamiltonian(b, *disguised(M, 2.0, 3, phases), schedule=7)
        drop_terms(H2)
        x, y = H(C), H2(C)
        assert np.array_equal(np.isfinite(x.real), np.isfinite(y.real))
        assert np.array_equal(np.isfinite(x.imag), np.isfinite(y.imag))
        assert 0 < np.count_nonzero(~np.isfinite(x.real)) < b.nc


# two words with terms in the second, three words: one larger block of pairs
@pytest.mark.parametrize("M", [10, 16, 17, 24])
def test_one_block_of_pairs(oracle_lib, M):
    N = 3
    note(f"pair terms one block M={M}")
    rng = np.random.default_rng(M)
    pairs = [(0, 0), (0, M - 1), (M - 1, M - 1), (M // 2, M - 2), (7, 8), (M - 2, M - 2), (1, 9)]
    a = rng.standard_normal(len(pairs)) + 1j * rng.standard_normal(len(pairs))
    Hint = np.zeros((M,) * 4, complex)
    for x, (k, s) in enumerate(pairs):
        for y, (q, l) in enumerate(pairs):
            for kk, ss in {(k, s), (s, k)}:
                for qq, ll in {(q, l), (l, q)}:
                    Hint[kk, ss, qq, ll] = a[x] * np.conj(a[y])
    Ho = np.diag(rng.standard_normal(M)).astype(complex)
    o = oracle.Basis(N, M)
    C, _, _ = oracle.random_inputs(N, M, seed=1)
    H = mcpi_amd.Hamiltonian(mcpi_amd.Basis(N, M, "none"), Ho, Hint, schedule=7)
    ref = o.acth(C, Ho, Hint)
    assert_close(H(C), ref, 1e-13, "by terms")
    drop_terms(H)
    assert_close(H(C), ref, 1e-13, "two passes")

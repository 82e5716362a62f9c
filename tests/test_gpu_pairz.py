"""The factorized pair-space H.v on contact interactions in other guises than
the plane-wave order: orbitals permuted (blocks of pairs in any order) and
given phases (complex factors), at the edges of its tiles and runs."""
import numpy as np
import pytest

import mcpi_amd
import oracle
from tests.gpu_util import assert_close, note

pytestmark = pytest.mark.gpu


def disguised(M, g, seed, phases=True):
    """Lieb-Liniger Ho and Hint with the orbitals permuted and a_k -> e^{i p_k}
    a_k: the same spectrum, pair blocks scattered over the pairs, and with
    phases complex factors."""
    rng = np.random.default_rng(seed)
    perm = rng.permutation(M)
    ph = np.exp(1j * rng.uniform(0, 2 * np.pi, M)) if phases else np.ones(M)
    Ho = oracle.ll_ho(M)[np.ix_(perm, perm)]
    Hint = oracle.ll_hint(M, g)[np.ix_(perm, perm, perm, perm)]
    Hint = np.einsum("ksql,k,s,q,l->ksql", Hint, ph.conj(), ph.conj(), ph, ph)
    return Ho, Hint


# rows of N - 2 particles: 1, below and above one 64-row tile, several tiles
# with several runs of pairs each, more than eight tiles; 32-byte rows (M > 16)
@pytest.mark.parametrize("N,M", [(2, 3), (2, 24), (4, 4), (9, 4), (8, 5), (3, 12), (7, 8), (6, 11), (5, 13), (4, 17),
                                 (30, 3)])
@pytest.mark.parametrize("phases", [False, True])
def test_disguised_contact_interaction(oracle_lib, N, M, phases):
    note(f"pairz disguised N={N} M={M} phases={phases}")
    o = oracle.Basis(N, M)
    C, _, _ = oracle.random_inputs(N, M, seed=700 + N + M)
    Ho, Hint = disguised(M, 3.0, 10 * N + M, phases)
    b = mcpi_amd.Basis(N, M, "none")
    H = mcpi_amd.Hamiltonian(b, Ho, Hint, schedule=7)
    assert_close(H(C), o.acth(C, Ho, Hint), 1e-12, "schedule 7")
    # without the occupation table the schedule does not apply (2 or 1 runs)
    drop = mcpi_amd.lib().mcpi_hip_basis_drop_occ2
    drop.argtypes = [mcpi_amd._vp]
    assert drop(b.handle) == 0
    assert_close(H(C), o.acth(C, Ho, Hint), 1e-12, "without the table")


@pytest.mark.parametrize("N,M", [(4, 6), (6, 12)])
def test_disguised_members(oracle_lib, N, M):
    """Seven members with one set of blocks and complex factors: four, two and
    one at a time."""
    note(f"pairz disguised members N={N} M={M}")
    b = mcpi_amd.Basis(N, M, "single")
    o = oracle.Basis(N, M)
    C, _, _ = oracle.random_inputs(N, M, seed=5)
    C = C / np.linalg.norm(C)
    mats = [disguised(M, g, 77) for g in np.logspace(-1, 1, 7)]
    hams = [mcpi_amd.Hamiltonian(b, *m) for m in mats]
    starts = [mcpi_amd.DeviceArray.from_numpy(C) for _ in hams]
    lm = 12
    mcpi_amd.set_batched_kernel(3)
    try:
        E, _ = mcpi_amd.lanczos_batched(hams, starts, lm)
    finally:
        mcpi_amd.set_batched_kernel(0)
    for x, (Ho, Hint) in enumerate(mats):
        E_o = o.ground(lm, C, Ho, Hint)[0]
        # twelve steps of a start in every sector: rounding of 1e-16 grows with
        # the norm of H (about 1e4) only
        assert abs(E[x] - E_o) <= 1e-11 * max(1.0, np.abs(Ho).max() * N), (x, E[x], E_o)


@pytest.mark.parametrize("sizes", [(1,), (1, 2), (1, 1, 1, 3), (1, 9), (1, 1, 6, 1)])
@pytest.mark.parametrize("N,M", [(2, 3), (5, 5), (3, 11), (4, 18)])
def test_single_pair_blocks(oracle_lib, N, M, sizes):
    """Blocks of one pair beside larger ones, only blocks of one pair, and
    pairs in no block: Hermitian rank-one blocks over a random order of the
    pairs, zero on the rest."""
    note(f"pairz single pairs N={N} M={M} sizes={sizes}")
    rng = np.random.default_rng(100 * N + M + len(sizes))
    pairs = [(q, l) for l in range(M) for q in range(l + 1)]
    order = list(rng.permutation(len(pairs)))
    Hint = np.zeros((M,) * 4, complex)
    while order:
        for s in sizes:
            blk, order = [pairs[x] for x in order[:s]], order[s:]
            if rng.random() < 0.2:
                continue
            a = rng.standard_normal(len(blk)) + 1j * rng.standard_normal(len(blk))
            w = rng.choice([-1.0, 1.0])
            for x, (k, s2) in enumerate(blk):
                for y, (q, l) in enumerate(blk):
                    for kk, ss in {(k, s2), (s2, k)}:
                        for qq, ll in {(q, l), (l, q)}:
                            Hint[kk, ss, qq, ll] = w * a[x] * np.conj(a[y])
    Ho = np.diag(rng.standard_normal(M)).astype(complex)
    o = oracle.Basis(N, M)
    C, _, _ = oracle.random_inputs(N, M, seed=3)
    b = mcpi_amd.Basis(N, M, "single")
    H = mcpi_amd.Hamiltonian(b, Ho, Hint, schedule=7)
    assert_close(H(C), o.acth(C, Ho, Hint), 1e-12, "schedule 7")

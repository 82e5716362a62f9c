"""Batched Lanczos over many mid-size instances, at the sizes where a chain
goes from two rows a thread to four in its vector passes (1024 blocks of four
rows in all), and where it stops to form its sums inside other kernels: every
row of every vector takes part in every pass."""
import numpy as np
import pytest

import mcpi_amd
import oracle
from tests.gpu_util import note

pytestmark = pytest.mark.gpu

LM = 120


def _start(nc, seed):
    rng = np.random.default_rng(seed)
    v = rng.standard_normal(nc) + 1j * rng.standard_normal(nc)
    return v / np.linalg.norm(v)


def _low_orbital(M, seed):
    """Ho, Hint with the last orbital far below the others: the ground state
    sits in a vector's last rows, is found after some 40 steps, and what
    rounding leaves of it in the later vectors grows where it is not taken
    out again."""
    rng = np.random.default_rng(seed)
    A = 0.01 * (rng.standard_normal((M, M)) + 1j * rng.standard_normal((M, M)))
    B = 0.01 * (rng.standard_normal((M,) * 4) + 1j * rng.standard_normal((M,) * 4))
    B = 0.5 * (B + B.transpose(1, 0, 2, 3))
    B = 0.5 * (B + B.transpose(0, 1, 3, 2))
    A = 0.5 * (A + A.conj().T)
    A[-1, -1] -= 3.0
    return A, 0.5 * (B + np.conj(B.transpose(2, 3, 0, 1)))


# blocks of four rows (1,024 entries): (8,11) 43, (10,11) 181, (6,9) 3, (9,13) 288
@pytest.mark.parametrize(
    "spec",
    [
        [(8, 11)] * 23,                       # 989 blocks: two rows a thread
        [(8, 11)] * 24,                       # 1,032: four
        [(8, 11)] * 24 + [(6, 9), (4, 6)],    # short ones beside
        [(10, 11)] * 6,                       # 1,086 blocks of few instances
        [(10, 11)] * 33,                      # 33 181^2 partials: sums in kernels of their own
        [(8, 11)] * 21 + [(9, 13)],           # a vector too long for the split update
    ],
    ids=["23", "24", "24+short", "6-long", "33-long", "mixed"],
)
def test_batched_mid_size(oracle_lib, spec):
    note(f"batched {len(spec)} instances, first {spec[0]}, last {spec[-1]}")
    bases = {nm: mcpi_amd.Basis(*nm, "single") for nm in set(spec)}
    mats = [_low_orbital(nm[1], x) for x, nm in enumerate(spec)]
    hams = [mcpi_amd.Hamiltonian(bases[nm], *m) for nm, m in zip(spec, mats)]
    starts = [mcpi_amd.DeviceArray.from_numpy(_start(bases[nm].nc, x)) for x, nm in enumerate(spec)]
    outs = [mcpi_amd.DeviceArray(bases[nm].nc) for nm in spec]
    E, steps = mcpi_amd.lanczos_batched(hams, starts, LM, outs)
    for x in range(len(spec)):
        E1, v1, s1 = hams[x].ground(LM, starts[x])
        v = outs[x].numpy()
        assert steps[x] == s1 == LM
        assert abs(E[x] - E1) <= 1e-10 * max(1.0, abs(E1)), (x, E[x], E1)
        # an orthonormal Krylov basis (rounding of at most 120 one-pass steps)
        assert abs(np.linalg.norm(v) - 1) < 1e-10, (x, np.linalg.norm(v))
        assert abs(abs(np.vdot(v, v1.numpy())) - 1) < 1e-8, x
    if (6, 9) in spec:
        x = spec.index((6, 9))
        E_o, psi_o, _ = oracle.Basis(6, 9).ground(LM, _start(bases[6, 9].nc, x), *mats[x])
        assert abs(E[x] - E_o) < 1e-10 * abs(E_o) and abs(abs(np.vdot(psi_o, outs[x].numpy())) - 1) < 1e-8

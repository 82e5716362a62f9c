"""The hooks that take a table away for tests leave the handle's account and
tuning in order."""
import ctypes as ct
import math

import numpy as np
import pytest

import mcpi_amd
import oracle
from tests.gpu_util import assert_close, note

pytestmark = pytest.mark.gpu


def _hook(name, handle):
    f = getattr(mcpi_amd.lib(), name)
    f.restype, f.argtypes = ct.c_int, [ct.c_void_p]
    assert f(handle) == 0


def _bytes(b):
    info = mcpi_amd._BasisInfo()
    mcpi_amd._check(mcpi_amd.lib().mcpi_hip_basis_info(b.handle, ct.byref(info)))
    return int(info.device_bytes)


@pytest.mark.parametrize("N,M", [(1, 5), (5, 8), (3, 17)])
def test_account_of_the_occupation_table(N, M):
    note(f"drop occupation table N={N} M={M}")
    b = mcpi_amd.Basis(N, M, "single")
    before = _bytes(b)
    rows = math.comb(N + M - 3, N - 2) if N >= 2 else 0
    for _ in range(2):
        _hook("mcpi_hip_basis_drop_occ2", b.handle)
        assert before - _bytes(b) == rows * (16 if M <= 16 else 32)


def test_tuning_without_the_terms(oracle_lib):
    N, M = 6, 9
    note("drop terms after tuning")
    Ho, Hint = mcpi_amd.ll_ho(M), mcpi_amd.ll_hint(M, 2.0)
    C, _, _ = oracle.random_inputs(N, M, seed=1)
    ref = oracle.Basis(N, M).acth(C, Ho, Hint)
    H = mcpi_amd.Hamiltonian(mcpi_amd.Basis(N, M, "single"), Ho, Hint)
    assert_close(H(C), ref, 1e-13, "tuned")
    assert H.schedule != 0
    _hook("mcpi_hip_ham_drop_terms", H.handle)
    assert H.schedule == 0
    assert_close(H(C), ref, 1e-13, "tuned again")
    assert H.schedule != 0

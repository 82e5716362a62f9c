"""The reference-shaped entry points on several sets of tables in turn: the
device state kept from the last call belongs to one set, and a call with
another one (other sizes, or equal ones at other addresses) does not see it."""
import pytest

import mcpi_amd.reference as R
import oracle
from tests.gpu_util import assert_close, note

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("turn", [[0, 1, 0], [0, 2, 2, 0], [1, 3, 0, 1]])
def test_tables_in_turn(oracle_lib, turn):
    note(f"reference tables in turn {turn}")
    spec = [(5, 6), (6, 5), (5, 6), (2, 4)]
    tabs = [R.RefBasis(*s) for s in spec]
    for x in turn:
        N, M = spec[x]
        o = oracle.Basis(N, M)
        C, Ho, Hint = oracle.random_inputs(N, M, seed=40 + x)
        ref = o.acth(C, Ho, Hint)
        for _ in range(2):
            assert_close(tabs[x].applyHconf_omp(C, Ho, Hint), ref, 1e-12, "omp")
        assert_close(tabs[x].applyHconf(C, Ho, Hint), ref, 1e-12, "no maps")
        assert_close(tabs[x].applyHconf_omp(C, Ho, Hint), ref, 1e-12, "omp again")
    R.release_cached()

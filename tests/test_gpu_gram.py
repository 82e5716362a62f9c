"""The Gram product of the densities at the edges of its tiles, with and without
the occupation table, against the oracle."""
import ctypes as ct

import pytest

import mcpi_amd
import oracle
from tests.gpu_util import assert_close, note

pytestmark = pytest.mark.gpu

# pair columns M(M+1)/2: 6 and 15 (one 16-column group), 21 (two), 36 (three),
# 55 (four), 66 and 78 (five), 91 and 105 (two tiles), 153 (32-byte rows);
# rows of N-2 particles: 1, below and above one 32-row tile, many tiles
SHAPES = [(1, 4), (2, 3), (4, 5), (7, 6), (6, 8), (5, 10), (4, 11), (5, 12), (4, 13), (3, 14), (4, 17), (25, 3)]


@pytest.mark.parametrize("table", [True, False])
@pytest.mark.parametrize("N,M", SHAPES)
def test_densities_at_tile_edges(oracle_lib, N, M, table):
    """rho1 alone (its own product), rho2 alone, and both in one call (rho1 as
    the contraction of rho2; N = 1: rho2 is zero and rho1 its own product)."""
    note(f"gram N={N} M={M} table={table}")
    o = oracle.Basis(N, M)
    C, _, _ = oracle.random_inputs(N, M, seed=300 + 10 * M + N)
    b = mcpi_amd.Basis(N, M, "none")
    if not table:
        drop = mcpi_amd.lib().mcpi_hip_basis_drop_occ2
        drop.restype, drop.argtypes = ct.c_int, [ct.c_void_p]
        assert drop(b.handle) == 0
    dC = mcpi_amd.DeviceArray.from_numpy(C)
    r1, r2 = o.rho1(C), o.rho2(C)
    g1, g2 = b.vjp(dC)
    assert_close(g1, r1, 1e-12, "dE/dHo")
    assert_close(b.rho1(dC), r1, 1e-12, "rho1")
    if N == 1:
        assert not g2.any() and not b.rho2(dC).any()
    else:
        assert_close(g2, 0.5 * r2, 1e-12, "dE/dHint")
        assert_close(b.rho2(dC), r2, 1e-12, "rho2")

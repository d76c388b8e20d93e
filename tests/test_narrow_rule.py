"""Which products with one or two columns are formed directly: shapes at which one of the two routes was measured
at least a tenth faster (one MI355X), on the sides of limb count, rows, batch and rounding."""
import pytest

from sdpvibe_amd import batched as Bm

DIRECT, RESIDUES = True, False


@pytest.mark.parametrize("rounded,L,nb,M,N,K,route", [
    (True, 24, 60, 162, 1, 3000, DIRECT), (True, 24, 60, 162, 2, 1500, DIRECT), (True, 35, 1, 1500, 2, 1500, DIRECT),
    (True, 40, 20, 160, 2, 1000, DIRECT), (True, 40, 3000, 1, 1, 42, DIRECT), (True, 40, 1, 200, 2, 200, DIRECT),
    (True, 8, 500, 2, 2, 200, DIRECT), (True, 24, 3000, 2, 2, 42, DIRECT), (True, 48, 1, 500, 1, 500, DIRECT),
    (True, 24, 1, 1, 1, 100000, DIRECT), (True, 35, 100, 2, 2, 42, DIRECT), (True, 48, 2000, 8, 1, 8, DIRECT),
    (True, 63, 2000, 8, 1, 8, DIRECT), (True, 16, 500, 2, 2, 200, RESIDUES), (True, 24, 500, 2, 2, 1000, RESIDUES), (True, 35, 500, 8, 2, 1000, RESIDUES),
    (True, 35, 3000, 2, 2, 42, RESIDUES), (True, 48, 20, 160, 2, 1000, RESIDUES), (True, 48, 2000, 1, 1, 42, RESIDUES),
    (True, 44, 1, 1500, 1, 1500, RESIDUES), (True, 63, 60, 162, 1, 1500, RESIDUES), (True, 63, 1, 2000, 2, 2000, RESIDUES),
    (False, 24, 60, 162, 1, 3000, DIRECT), (False, 40, 20, 160, 2, 1000, DIRECT), (False, 48, 1, 1500, 1, 1500, DIRECT),
    (False, 63, 1, 500, 1, 500, DIRECT), (False, 63, 60, 96, 1, 96, DIRECT), (False, 63, 3000, 1, 1, 42, DIRECT),
    (False, 48, 1, 1500, 2, 1500, RESIDUES), (False, 63, 1, 1500, 2, 1500, RESIDUES), (False, 63, 60, 96, 2, 96, RESIDUES),
    (False, 48, 500, 2, 2, 1000, RESIDUES), (False, 64, 1, 32, 1, 32, RESIDUES), (False, 24, 1, 32, 3, 32, RESIDUES),
])
def test_route(rounded, L, nb, M, N, K, route):
    assert Bm._narrow(M, N, K, L, nb, rounded) is route

"""The factored tile with its inverse rounded in the same call against the wide inverse rounded by the separate
passes: views as input, tile sizes and limb counts at the edges, ill conditioned tiles and tiles that are
not positive definite (inverses that fill the wide words)."""
import pytest
import torch

from sdpvibe_amd.basecase import LI, tile_factor, tile_factor_inverse
from sdpvibe_amd.limbops import bitlen_words, shift_round
from sdpvibe_amd.mpmat import headroom_bits
from tests.intutil import spd_tile, to_planes

pytestmark = pytest.mark.gpu


def parity(tiles, L, BT):
    nb = len(tiles)
    flat = [v for t in tiles for row in t for v in row]
    A = torch.from_numpy(to_planes(flat, L).reshape(L, nb, BT, BT)).cuda()
    room = torch.full((L, nb + 1, BT + 5, BT + 3), -1, dtype=torch.int32, device="cuda")
    view = room[:, 1:, 2:2 + BT, 1:1 + BT]
    view.copy_(A)
    Lout, Xw, _ = tile_factor(A, BT)
    top = bitlen_words(Xw.reshape(L + LI, -1)).view(nb, BT * BT).amax(1)
    s = (top - headroom_bits(L)).repeat_interleave(BT * BT)
    X = shift_round(Xw.reshape(L + LI, -1), s, L).view(L, nb, BT, BT)
    for x in (A, view):
        got = tile_factor_inverse(x, BT, headroom_bits(L))
        assert torch.equal(got[0], Lout) and torch.equal(got[1], X)
        assert torch.equal(got[2], (top - headroom_bits(L) - 32 * L)[:, None].expand(nb, BT))


@pytest.mark.parametrize("L,BT,logc", [(2, 1, 3), (2, 32, 10), (3, 5, 9), (8, 33, 100), (12, 64, 60), (24, 32, 20), (24, 31, 600),
                                       (41, 12, 300), (44, 6, 40)])
def test_against_separate_passes(L, BT, logc):
    parity([spd_tile(BT, logc, 3 * L + b, 32 * L - 40) for b in range(3)], L, BT)


def test_indefinite_tiles():
    L, BT = 12, 9
    t = spd_tile(BT, 4, 7, 32 * L - 40)
    t[2][2], t[5][5] = 0, 1
    parity([t, [[-v for v in row] for row in t], [[0] * BT for _ in range(BT)]], L, BT)

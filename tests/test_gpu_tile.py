"""The tile factorisation and inverse (sdpv_tile_chol) against the oracle's restatement, bit for bit, at the
limb counts where the kernel's operand size class changes, with well and ill conditioned tiles (pivot
reciprocals far above one) and with tiles that are not positive definite (factors above one, pivots that
are not positive)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.intutil import int_to_words, rnd_half_up, spd_tile, to_planes, words_to_int, wrap

cu = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()


def tile_parity(tiles, L, BT):
    from sdpvibe_amd.basecase import tile_factor
    WL, nb = L + 24, len(tiles)
    flat = [tiles[b][i][j] for b in range(nb) for i in range(BT) for j in range(BT)]
    A = to_planes(flat, L).reshape(L, nb, BT, BT)
    W = np.array([int_to_words(v << 40, WL) for v in flat], np.uint32).reshape(nb, BT, BT, WL)
    Lw, _, X = O.tile_chol(W, L)
    Lo, Xw, _ = tile_factor(cu(A), BT)
    want = to_planes([wrap(rnd_half_up(words_to_int(w), 40), L) for w in Lw.reshape(-1, WL)], L).reshape(L, nb, BT, BT)
    assert np.array_equal(Lo.cpu().numpy(), want), "factor"
    assert np.array_equal(Xw.cpu().numpy(), np.ascontiguousarray(X.transpose(3, 0, 1, 2)).view(np.int32)), "inverse"


@pytest.mark.gpu
@pytest.mark.parametrize("L", [1, 8, 9, 16, 17, 24, 25, 28, 29, 32, 33, 36, 37, 40, 41])
def test_tile_size_classes(L):
    tile_parity([spd_tile(32, min(20, 8 * L), L, 32 * L - 40)] if L > 1 else [[[1 << 0]]], L, 32 if L > 1 else 1)


@pytest.mark.gpu
@pytest.mark.parametrize("L,BT,logc", [(24, 32, 300), (24, 32, 600), (35, 20, 900), (8, 32, 150), (12, 17, 60)])
def test_ill_conditioned_tiles(L, BT, logc):
    tile_parity([spd_tile(BT, logc, 3 * L + b, 32 * L - 40) for b in range(2)], L, BT)


@pytest.mark.gpu
@pytest.mark.parametrize("L", [4, 24])
def test_indefinite_tiles(L):
    BT, one = 12, 1 << (32 * L - 40)
    t = spd_tile(BT, 4, 7, 32 * L - 40)
    for p, r in ((0, 20), (3, 0), (5, 900)):             # small, zero and tiny pivots beside large entries
        t[p][p] = one >> r if r else 0
    tile_parity([t, [[-v for v in row] for row in t]], L, BT)

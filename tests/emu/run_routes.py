"""Emulated comparison of the routes that small calls take with the general ones: bgemm_nt's fused addition and
strided output, mpf.gemm's single native call, the blocks of a stack, the rounded tile inverse."""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__)))))
from tests.emu import harness  # noqa: E402

harness.install()
import torch  # noqa: E402

from sdpvibe_amd import batched as Bm  # noqa: E402
from sdpvibe_amd import mpf as F  # noqa: E402
from sdpvibe_amd.basecase import LI, tile_factor, tile_factor_inverse  # noqa: E402
from sdpvibe_amd.limbops import bitlen_words, shift_round  # noqa: E402
from sdpvibe_amd.mpmat import headroom_bits  # noqa: E402
from tests.intutil import spd_tile, to_planes  # noqa: E402

G = torch.Generator().manual_seed(3)
EZ = -(1 << 40)


def rnd(*s):
    return torch.randint(-2 ** 31, 2 ** 31, s, generator=G, dtype=torch.int64).to(torch.int32)


def fused():
    for L, nb, M, K, N, rowexp, sgn in ((2, 2, 5, 9, 3, True, -1), (3, 1, 40, 33, 37, False, 1)):
        A, Bt, e = Bm.BMP(rnd(L, nb, M, K) >> 1, -32 * L), Bm.BMP(rnd(L, nb, N, K) >> 1, -30 * L), -31 * L - 5 + 32 * (L // 2)
        re = torch.randint(-31 * L, -30 * L, (nb, N), generator=G) if rowexp else None
        big = rnd(L, nb, M + 3, N + 5)
        X = Bm.BMP(big[:, :, 1:1 + M, 2:2 + N], e)
        ref = Bm.badd(X, Bm.bgemm_nt(A, Bt, out_exp=e, bt_rowexp=re), sgn, out_exp=e).limbs
        Bm.bgemm_nt(A, Bt, out_exp=e, bt_rowexp=re, plus=X, sgn=sgn, dest=X.limbs)
        assert torch.equal(X.limbs, ref)


def native():
    for L, nb, M, K, N, tA, tB in ((1, 1, 3, 1, 3, False, False), (3, 2, 33, 20, 9, True, False), (2, 1, 5, 97, 40, False, True)):
        mk = lambda r, c: F.MPF(rnd(L, nb, r, c) >> 1, torch.randint(-60, 60, (nb, r, c), generator=G))
        A, B = mk(*((K, M) if tA else (M, K))), mk(*((N, K) if tB else (K, N)))
        one, F.SMALL_GEMM = F.gemm(A, B, tA, tB), 0
        apart, F.SMALL_GEMM = F.gemm(A, B, tA, tB), 1 << 26
        assert torch.equal(one.m, apart.m) and torch.equal(one.e, apart.e)


def blocks():
    L, rows, cols, count = 9, 7, 5, 34
    places = [(rnd(L, cols, r).transpose(1, 2)[:, :, :c], rnd(r, c).long())
              for r, c in ((rows - j % (rows + 1), cols - j % 3) for j in range(count))]
    M, E = rnd(L, count, rows, cols), rnd(count, rows, cols).long()
    F._copy_blocks(places, M, E, True)
    rm, re = torch.zeros_like(M), torch.full_like(E, EZ)
    for j, (m, e) in enumerate(places):
        rm[:, j, :e.shape[0], :e.shape[1]], re[j, :e.shape[0], :e.shape[1]] = m, e
    assert torch.equal(M, rm) and torch.equal(E, re)
    back = [(torch.zeros_like(m), torch.zeros_like(e)) for m, e in places]
    F._copy_blocks(back, M, E, False)
    assert all(torch.equal(a, b) for p, q in zip(places, back) for a, b in zip(p, q))


def tile():
    for L, BT in ((2, 1), (4, 9)):
        t = [v for b in range(2) for row in spd_tile(BT, 5, b, 32 * L - 40) for v in row]
        room = torch.full((L, 3, BT + 2, BT + 1), -1, dtype=torch.int32)
        A = room[:, 1:, 1:1 + BT, :BT]
        A.copy_(torch.from_numpy(to_planes(t, L).reshape(L, 2, BT, BT)))
        Lo, Xw, _ = tile_factor(A, BT)
        top = bitlen_words(Xw.reshape(L + LI, -1)).view(2, BT * BT).amax(1)
        s = top - headroom_bits(L)
        X = shift_round(Xw.reshape(L + LI, -1), s.repeat_interleave(BT * BT), L).view(L, 2, BT, BT)
        got = tile_factor_inverse(A, BT, headroom_bits(L))
        assert torch.equal(got[0], Lo) and torch.equal(got[1], X) and torch.equal(got[2][:, 0], s - 32 * L)


if __name__ == "__main__":
    {"fused": fused, "native": native, "blocks": blocks, "tile": tile}[sys.argv[1]]()
    print("ok")

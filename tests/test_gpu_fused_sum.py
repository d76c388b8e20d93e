"""Reconstructions of small launches (four waves per 64 entries) against those of large ones, and bgemm_nt's
fused exact addition and strided output against the separate product, addition and copy."""
import numpy as np
import pytest
import torch

from sdpvibe_amd import batched as Bm
from sdpvibe_amd import mpmat

pytestmark = pytest.mark.gpu
GEN = lambda: torch.Generator("cpu").manual_seed(7)


def limbs(g, *shape):
    return torch.randint(-2 ** 31, 2 ** 31, shape, generator=g, dtype=torch.int64).to(torch.int32).cuda() >> 1


@pytest.mark.parametrize("L", [1, 2, 8, 9, 17, 24, 25, 40, 63])
def test_small_reconstruction_against_large(L):
    R = mpmat.ctx(L)
    few, many, N = 13, 1 << 11, 35                       # 8 and 1120 groups of 64 entries
    rng = np.random.default_rng(L)
    half = np.array(R.mods, np.int64)[:, None, None] // 2
    acc = torch.from_numpy((rng.integers(-8128, 8129, (R.n, many, N)) % (2 * half) - half).astype(np.int16)).cuda()
    acc[:, 0] = 0
    small = acc[:, :few].contiguous()
    W, bl, _ = R.crt_block(acc, N, 0, N, many, True)
    w, b, _ = R.crt_block(small, N, 0, N, few, True)
    assert torch.equal(w, W[:, :few * N]) and torch.equal(b, bl[:few * N])
    ecol = torch.arange(N, device="cuda")
    for mode in (1, 2):
        got = []
        for a, rows in ((acc, many), (small, few)):
            out = torch.zeros((L, rows, N), dtype=torch.int32, device="cuda")
            e = torch.zeros((rows, N), dtype=torch.int64, device="cuda")
            R.crt(a, rows, N, 0, N, mode, outm=out, oute=e, L=L, plane=rows * N, ldo=N, Mb=rows, ecol=ecol,
                  scol=ecol * (8 * L) + 1, scaled=True)
            got.append((out[:, :few].clone(), e[:few].clone()))
        assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]), mode


@pytest.mark.parametrize("L,nb,M,K,N", [(2, 3, 1, 5, 3), (5, 1, 33, 40, 65), (24, 2, 70, 32, 32), (24, 1, 300, 64, 260),
                                        (4, 2, 9, 20, 2)])
@pytest.mark.parametrize("rowexp", [False, True])
@pytest.mark.parametrize("sgn", [1, -1])
def test_fused_sum(L, nb, M, K, N, rowexp, sgn, monkeypatch):
    g = GEN()
    A = Bm.BMP(limbs(g, L, nb, M, K), -32 * L)
    Bt = Bm.BMP(limbs(g, L, nb, N, K), -30 * L)
    e = -31 * L - 5 + 32 * (L // 2)
    re = torch.randint(-40 * L, -39 * L, (nb, N), generator=g).cuda() + 9 * L if rowexp else None
    big = limbs(g, L, nb, M + 7, N + 11)
    X = Bm.BMP(big[:, :, 3:3 + M, 5:5 + N], e)
    for budget in (None, 2 * mpmat.ctx(L).n * nb * M * 64):
        if budget:
            monkeypatch.setattr(mpmat, "ACC_BUDGET", budget)
        ref = Bm.badd(X, Bm.bgemm_nt(A, Bt, out_exp=e, bt_rowexp=re), sgn, out_exp=e).limbs
        assert torch.equal(Bm.bgemm_nt(A, Bt, out_exp=e, bt_rowexp=re, plus=X, sgn=sgn).limbs, ref)
        wide = torch.full((L, nb, M + 2, N + 6), 17, dtype=torch.int32, device="cuda")
        dest = wide[:, :, 1:1 + M, 4:4 + N]
        got = Bm.bgemm_nt(A, Bt, out_exp=e, bt_rowexp=re, plus=X, sgn=sgn, dest=dest)
        assert got.limbs.data_ptr() == dest.data_ptr() and torch.equal(dest, ref)
        edge = wide.clone()
        edge[:, :, 1:1 + M, 4:4 + N] = 17
        assert bool((edge == 17).all())
        inplace = big.clone()[:, :, 3:3 + M, 5:5 + N]    # the addend's own place
        Bm.bgemm_nt(A, Bt, out_exp=e, bt_rowexp=re, plus=Bm.BMP(inplace, e), sgn=sgn, dest=inplace)
        assert torch.equal(inplace, ref)
    with pytest.raises(ValueError):
        Bm.bgemm_nt(A, Bt, out_exp=e, bt_rowexp=re, plus=Bm.BMP(X.limbs, e + 1))

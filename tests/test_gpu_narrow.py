"""Direct products with one or two columns (sdpv_narrow) against the oracle, bit for bit: mpf.gemm in every
orientation with exponents far apart, zero and unnormalised entries and extreme mantissas, at sizes around
the kernel's tiles (32 rows, slices of 128 k, steps of 16 or 8 k) and limb counts around its 8-limb
chunks; the fused subtraction of the triangular solves and the joined halves against their parts."""
import random

import numpy as np
import pytest
import torch

from oracle import oracle as O
from sdpvibe_amd import batched as Bm
from sdpvibe_amd import mpf as F
from tests.intutil import EZ, to_planes

pytestmark = pytest.mark.gpu

cu = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()


def entries(rng, shape, L, spread, raw=0.1):
    """mantissas and exponents: normalised ones of either sign, some zero, a share `raw` unnormalised, some
    powers of two (exact ties and single bits)"""
    NB, n = 32 * L - 2, int(np.prod(shape))
    m, e = [], []
    for _ in range(n):
        kind = rng.random()
        v = rng.randrange(1 << (NB - 1), 1 << NB)
        if kind < 0.1:
            v = 0
        elif kind < 0.1 + raw:
            v = rng.randrange(1, 1 << rng.randrange(1, NB))
        elif kind < 0.3:
            v = (1 << NB) - 1 if rng.random() < 0.5 else 1 << (NB - 1)
        m.append(-v if rng.random() < 0.5 else v)
        e.append(EZ if v == 0 else rng.randrange(-spread, spread + 1))
    return to_planes(m, L).reshape((L,) + shape), np.array(e, np.int64).reshape(shape)


def gemm_parity(L, nb, M, K, N, tA, tB, spread, seed):
    rng = random.Random(seed)
    Am, Ae = entries(rng, (nb, K, M) if tA else (nb, M, K), L, spread)
    Bmm, Be = entries(rng, (nb, N, K) if tB else (nb, K, N), L, spread)
    C = F.gemm(F.MPF(cu(Am), cu(Ae)), F.MPF(cu(Bmm), cu(Be)), tA, tB)
    rm, re_ = O.mpf_gemm(Am, Ae, Bmm, Be, tA, tB)
    assert np.array_equal(C.m.cpu().numpy(), rm) and np.array_equal(C.e.cpu().numpy(), re_), (L, nb, M, K, N, tA, tB)


SHAPES = [(1, 1, 1, 1), (2, 31, 5, 1), (1, 32, 16, 2), (2, 33, 17, 1), (1, 65, 128, 1), (1, 40, 129, 2), (1, 3, 700, 1),
          (3, 1, 90, 37), (1, 2, 40, 50)]


@pytest.mark.parametrize("nb,M,K,N", SHAPES)
@pytest.mark.parametrize("L", [1, 8, 9, 24])
@pytest.mark.parametrize("tA,tB", [(False, False), (True, False), (False, True)])
def test_gemm_few_columns(L, nb, M, K, N, tA, tB):
    gemm_parity(L, nb, M, K, N, tA, tB, 40, 7 * L + M + K)


@pytest.mark.parametrize("L", [3, 16, 17, 25, 32, 33, 40, 41, 48, 49, 57, 63])
def test_gemm_limb_counts_and_spread(L):
    for spread in (4, 150, 32 * L + 90, 5000):
        gemm_parity(L, 1, 34, 21, 1, False, False, spread, L + spread)


def minus_product_parity(L, nb, M, K, N, trans, seed):
    """X - A P with the columns of P and X at their own exponents, views on both sides"""
    rng = random.Random(seed)
    word = lambda shape: cu(to_planes([rng.randrange(-(1 << (32 * L - 33)), 1 << (32 * L - 33))
                                       for _ in range(int(np.prod(shape)))], L).reshape((L,) + shape))
    e = lambda c: cu(np.array([[rng.randrange(-90, 90) for _ in range(c)] for _ in range(nb)], np.int64))
    big = word((nb, K + 3, M + 2) if trans else (nb, M + 2, K + 3))
    A = big[:, :, 1:1 + K, 2:2 + M].transpose(2, 3) if trans else big[:, :, 2:2 + M, 1:1 + K]
    X, P = Bm.BMP(word((nb, M + 5, N)), e(N)), Bm.BMP(word((nb, K, N)), e(N))
    A = Bm.BMP(A, -(32 * L - 40))
    got = Bm._minus_product(Bm._rows(X, 3, 3 + M), A, P)
    prod = Bm.bgemm_nt(A, Bm._as_rows(P), out_exp="col", bt_rowexp=P.expt())
    want = Bm.badd(Bm._rows(X, 3, 3 + M), prod, -1, out_exp="align")
    assert torch.equal(got.limbs, want.limbs) and torch.equal(got.exp, want.exp)
    ref, rexp = O.bgemm_nt(A.limbs.cpu().numpy().copy(), P.limbs.transpose(2, 3).cpu().numpy().copy(),
                           P.exp.cpu().numpy() - (32 * L - 40), 1)
    assert np.array_equal(prod.limbs.cpu().numpy(), ref) and np.array_equal(prod.exp.cpu().numpy(), rexp)
    top = Bm.BMP(word((nb, 5, N)), e(N))
    st = Bm._stack_common(top, got)
    ee = torch.maximum(top.exp, got.exp)
    assert torch.equal(st.exp, ee) and torch.equal(st.limbs, torch.cat([Bm.brescale(top, ee).limbs,
                                                                        Bm.brescale(got, ee).limbs], 2))


@pytest.mark.parametrize("L", [2, 24, 35])
@pytest.mark.parametrize("nb,M,K,N,trans", [(1, 32, 32, 1, False), (2, 20, 64, 1, True), (1, 96, 32, 2, False),
                                            (1, 70, 200, 1, True), (1, 130, 300, 1, False)])
def test_fused_subtraction_and_joined_halves(L, nb, M, K, N, trans):
    minus_product_parity(L, nb, M, K, N, trans, L + M + K)

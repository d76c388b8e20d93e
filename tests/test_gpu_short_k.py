"""Products with a short inner dimension, padded to a multiple of 32 only: every product tile that takes such
a padding against numpy, and mpf.gemm and bgemm_nt against the oracle at inner dimensions on both sides
of each padding step."""
import random

import numpy as np
import pytest
import torch

from oracle import oracle as O
from sdpvibe_amd import batched as Bm
from sdpvibe_amd import mpf as F
from sdpvibe_amd import mpmat
from tests.intutil import EZ, rand_mpf_ints, to_planes

pytestmark = pytest.mark.gpu

cu = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()


def product_parity(cfg, kp, M, N, L, nb=2):
    from sdpvibe_amd.rns import chunk_major
    R = mpmat.ctx(L)
    rng = np.random.default_rng(kp + M)
    m = np.array(R.mods, np.int64)[:, None, None, None]
    ra, rb = (np.clip(rng.integers(-8128, 8129, (R.n, nb, r, kp)), -(m // 2), m // 2) for r in (M, N))
    sp = lambda r: (((r + 64) & 127) - 64, (r - (((r + 64) & 127) - 64)) >> 7)
    (la, ha), (lb, hb) = sp(ra.reshape(R.n, nb * M, kp)), sp(rb.reshape(R.n, nb * N, kp))
    put = lambda x: chunk_major(cu(x.astype(np.int8)))
    acc = cu(np.zeros((R.n, nb * M, N), np.int16))
    R.product(put(ha), put(la), put(hb), put(lb), acc, nb, M, N, nb * M * N, config=cfg)
    ref = np.matmul(ra, rb.transpose(0, 1, 3, 2)) % m
    assert np.array_equal(acc.cpu().numpy().astype(np.int64).reshape(ref.shape), ref), (cfg, kp, M, N)


@pytest.mark.parametrize("cfg", [-1, 2, 3, 12, 13])
@pytest.mark.parametrize("kp", [32, 96])
def test_product_tiles(cfg, kp):
    for M, N in ((5, 40), (70, 136), (130, 33)):
        product_parity(cfg, kp, M, N, 3)


def test_other_tiles_refuse_odd_multiples_of_32():
    from sdpvibe_amd._lib import HipLibraryError
    with pytest.raises(HipLibraryError):
        product_parity(6, 32, 5, 5, 2)


def gemm_parity(L, nb, M, K, N, seed):
    rng = random.Random(seed)
    out = []
    for shape in ((nb, M, K), (nb, K, N)):
        v, e = rand_mpf_ints(rng, int(np.prod(shape)), L, 60)
        e = np.where(np.array(v, object) == 0, EZ, np.array(e, object)).astype(np.int64).reshape(shape)
        out.append((to_planes(v, L).reshape((L,) + shape), e))
    (Am, Ae), (Bmm, Be) = out
    C = F.gemm(F.MPF(cu(Am), cu(Ae)), F.MPF(cu(Bmm), cu(Be)))
    rm, re_ = O.mpf_gemm(Am, Ae, Bmm, Be)
    assert np.array_equal(C.m.cpu().numpy(), rm) and np.array_equal(C.e.cpu().numpy(), re_), (L, nb, M, K, N)
    A, Bt = Am, Bmm.transpose(0, 1, 3, 2).copy()
    D = Bm.bgemm_nt(Bm.BMP(cu(A), -7), Bm.BMP(cu(Bt), -9))
    ref, rexp = O.bgemm_nt(A, Bt, np.full((nb, N), -16, np.int64), 1)
    assert np.array_equal(D.limbs.cpu().numpy(), ref) and np.array_equal(D.exp.cpu().numpy(), rexp), (L, nb, M, K, N)


@pytest.mark.parametrize("K", [1, 31, 32, 33, 64, 65, 96, 97])
@pytest.mark.parametrize("L", [2, 24])
def test_inner_dimensions(K, L):
    gemm_parity(L, 2, 37, K, 9, K + L)

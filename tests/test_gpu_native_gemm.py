"""mpf.gemm's single call against its launches issued one by one, bit for bit: sizes at the edges of tiles and of the
padding, every transposition, zero rows and columns, and the shapes that keep the other route."""
import ctypes

import pytest
import torch

from sdpvibe_amd import mpf as F
from sdpvibe_amd import mpmat
from sdpvibe_amd._lib import HipLibraryError, call, ptr, stream

pytestmark = pytest.mark.gpu
EZ = -(1 << 40)


def rnd(g, L, *shape):
    m = torch.randint(-2 ** 31, 2 ** 31, (L, *shape), generator=g, dtype=torch.int64).to(torch.int32)
    m[-1] >>= 1
    e = torch.randint(-90, 90, shape, generator=g, dtype=torch.int64)
    zero = torch.rand(shape, generator=g) < 0.1
    zero[0, :1] = True                                    # a row of zeros
    m[:, zero], e[zero] = 0, EZ
    return F.MPF(m.cuda(), e.cuda())


@pytest.mark.parametrize("L,nb,M,K,N", [(1, 1, 3, 1, 3), (3, 2, 33, 32, 31), (14, 5, 27, 14, 27), (24, 3, 64, 97, 65),
                                        (24, 1, 130, 63, 129), (40, 2, 9, 64, 20)])
@pytest.mark.parametrize("tA", [False, True])
@pytest.mark.parametrize("tB", [False, True])
def test_single_call(L, nb, M, K, N, tA, tB, monkeypatch):
    g = torch.Generator("cpu").manual_seed(M + K)
    A, B = rnd(g, L, nb, *((K, M) if tA else (M, K))), rnd(g, L, nb, *((N, K) if tB else (K, N)))
    one = F.gemm(A, B, tA, tB)
    R = mpmat.ctx(L)
    monkeypatch.setattr(mpmat, "ACC_BUDGET", R.n * nb * M * 2 * 64)
    assert mpmat.panelled(R.n, nb, M, N, K) == (N > 64)
    panels = F.gemm(A, B, tA, tB)
    monkeypatch.setattr(F, "SMALL_GEMM", 0)
    apart = F.gemm(A, B, tA, tB)
    for other in (panels, apart):
        assert torch.equal(one.m, other.m) and torch.equal(one.e, other.e)


def test_refusals():
    g = torch.Generator("cpu").manual_seed(1)
    A, B, R = rnd(g, 2, 1, 4, 5), rnd(g, 2, 1, 5, 6), mpmat.ctx(2)
    m, e = torch.empty((2, 1, 4, 6), dtype=torch.int32, device="cuda"), torch.empty((1, 4, 6), dtype=torch.int64, device="cuda")
    work = torch.empty((1024,), dtype=torch.uint8, device="cuda")
    with pytest.raises(HipLibraryError):                  # scratch too small: refused before any launch
        call("sdpv_rns_mpf_gemm", ctypes.byref(R.tables), ptr(A.m), ptr(A.e), 20, 20, 5, 1, ptr(B.m), ptr(B.e), 30, 30, 1,
             6, 2, 1, 4, 6, 5, 32, -1, ptr(m), ptr(e), ptr(work), 1024, stream())
    with pytest.raises(ValueError):
        F.gemm(F.MPF(A.m[:, :, :3], A.e), B)

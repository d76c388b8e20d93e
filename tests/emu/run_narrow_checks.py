"""Operands of the direct products that do not fit each other, or only by broadcasting or by their limb count: refused, or
the result of the fitted operands; never read past their end (AddressSanitizer)."""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__)))))
from tests.emu import harness  # noqa: E402

harness.install()
import pytest  # noqa: E402
import torch  # noqa: E402

from sdpvibe_amd import batched as Bm  # noqa: E402
from sdpvibe_amd import mpf as F  # noqa: E402

G = torch.Generator().manual_seed(5)
REFUSED = (ValueError, AssertionError, IndexError, RuntimeError)


def rnd(*s):
    return torch.randint(-2 ** 31, 2 ** 31, s, generator=G, dtype=torch.int64).to(torch.int32)


def same(a, b):
    assert torch.equal(a.limbs, b.limbs) and torch.equal(torch.as_tensor(a.exp), torch.as_tensor(b.exp))


def exponents(nb, M, K, N, L):
    """exponents that broadcast to a block's columns, or of another integer type"""
    a, b = rnd(L, nb, M, K), rnd(L, nb, N, K)
    ea, eb = torch.arange(nb)[:, None] - 70, torch.arange(nb * N).view(nb, N) % 5 - 60
    for A1, e1, A2, e2 in (
            (-70, torch.arange(N)[None] - 60, -70, (torch.arange(N)[None] - 60).expand(nb, N).contiguous()),
            (-70, ea, -70, ea.expand(nb, N).contiguous()),
            (-70, eb.to(torch.int32), -70, eb),
            (torch.full((1, 3), -70), eb, torch.full((nb, K), -70), eb),
            (ea.to(torch.int32).expand(nb, 2), eb, ea, eb)):
        for mode in ("col", -20):
            same(Bm.bgemm_nt(Bm.BMP(a, A1), Bm.BMP(b, 0), out_exp=mode, bt_rowexp=e1),
                 Bm.bgemm_nt(Bm.BMP(a, A2), Bm.BMP(b, 0), out_exp=mode, bt_rowexp=e2))


def halves(nb, C, L):
    """joined halves whose exponents broadcast to every block"""
    a, b = rnd(L, nb, 2, C) >> 9, rnd(L, nb, 3, C) >> 9
    ea, eb = torch.arange(C)[None] - 9, torch.arange(nb)[:, None] - 7
    wide = lambda e: e.expand(nb, C).contiguous()
    same(Bm._stack_common(Bm.BMP(a, ea), Bm.BMP(b, eb)), Bm._stack_common(Bm.BMP(a, wide(ea)), Bm.BMP(b, wide(eb))))
    for other in (rnd(L, nb, 3, C - 1), rnd(L, nb - 1, 3, C), rnd(L - 1, nb, 3, C)):
        with pytest.raises(REFUSED):
            Bm._stack_common(Bm.BMP(a, -5), Bm.BMP(other, -5))


def limb_counts():
    """a right operand of fewer limbs multiplies as its sign extension does"""
    a, b = rnd(4, 2, 9, 7), rnd(2, 2, 1, 7)
    wide = torch.cat([b, (b[-1:] >> 31).expand(2, -1, -1, -1)], 0)
    for mode in ("col", -20):
        same(Bm.bgemm_nt(Bm.BMP(a, -70), Bm.BMP(b, -50), out_exp=mode), Bm.bgemm_nt(Bm.BMP(a, -70), Bm.BMP(wide, -50), out_exp=mode))


def refused():
    L, nb, M, K = 3, 2, 9, 7
    A, P, X = Bm.BMP(rnd(L, nb, M, K), -70), Bm.BMP(rnd(L, nb, K, 1), -50), Bm.BMP(rnd(L, nb, M, 1), -50)
    Bm._minus_product(X, A, P)
    for bad in (lambda: Bm._minus_product(X, A, Bm._rows(P, 0, K - 2)), lambda: Bm._minus_product(Bm._rows(X, 0, M - 3), A, P),
                lambda: Bm._minus_product(X, A, Bm.BMP(P.limbs[:, :1].contiguous(), -50)),
                lambda: Bm._minus_product(Bm.BMP(X.limbs[:2].contiguous(), -50), A, P),
                lambda: Bm.bgemm_nt(A, Bm.BMP(rnd(L, nb, 1, K - 1), 0)), lambda: Bm.bgemm_nt(A, Bm.BMP(rnd(L, nb + 1, 1, K), 0)),
                lambda: Bm.bgemm_nt(A, Bm.BMP(rnd(L, nb, 1, K), 0), bt_rowexp=torch.zeros((nb + 1, 1), dtype=torch.int64)),
                lambda: Bm.bgemm_nt(Bm.BMP(A.limbs, torch.zeros((nb + 1, K), dtype=torch.int64)), Bm.BMP(rnd(L, nb, 1, K), 0)),
                lambda: Bm.bgemm_nt(Bm.BMP(rnd(L, nb, 0, K), 0), Bm.BMP(rnd(L, nb, 1, K), 0))):
        with pytest.raises(REFUSED):
            bad()
    e = torch.zeros((1, M, K), dtype=torch.int64)
    v = F.MPF(rnd(L, 1, K, 1), torch.zeros((1, K, 1), dtype=torch.int64))
    with pytest.raises(REFUSED):
        F.gemm(F.MPF(rnd(L, 1, M - 2, K), e), v)
    acc = F.KSum(torch.zeros(K, dtype=torch.int64), torch.zeros(1, dtype=torch.int64), L)
    assert acc.direct
    with pytest.raises(REFUSED):
        acc.add(F.MPF(rnd(L, M - 2, K), e[0]), F.MPF(rnd(L, M, 1), torch.zeros((M, 1), dtype=torch.int64)))


if __name__ == "__main__":
    {"exponents": lambda: exponents(3, 5, 9, 2, 2), "few": lambda: exponents(1024, 1, 2, 1, 9), "limbs": limb_counts,
     "halves": lambda: halves(3, 4, 2),
     "refused": refused}[sys.argv[1]]()
    print("ok")

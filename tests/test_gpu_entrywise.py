"""Entrywise products and sums against the oracle, bit for bit, at the limb counts where the kernels' register
arrays change size (and above them, where the operands go through LDS): extreme and unnormalised mantissas,
zeros, exponents from equal to far apart, exact and near cancellation, a broadcast factor, entry counts
around a wave."""
import random

import numpy as np
import pytest
import torch

from oracle import oracle as O
from sdpvibe_amd import mpf as F
from tests.intutil import EZ, to_planes

pytestmark = pytest.mark.gpu

cu = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()


def pick(rng, L):
    """a mantissa of at most 32 L - 1 bits: mostly normalised"""
    NB = 32 * L - 2
    kind = rng.randrange(10)
    if kind == 0:
        return 0
    if kind == 1:
        return rng.choice([1 << NB, (1 << NB) - 1, 1 << (NB - 1), (1 << (NB - 1)) + 1, (1 << (NB + 1)) - 1])
    if kind == 2:
        return rng.randrange(1, 1 << rng.randrange(1, NB + 1))
    return rng.randrange(1 << (NB - 1), 1 << NB)


def operands(rng, n, L):
    a, b, ea, eb = [], [], [], []
    for _ in range(n):
        x, y = pick(rng, L), pick(rng, L)
        d = rng.choice([0, 0, 1, -1, 31, 32, 33, -32, 64, rng.randrange(-32 * L - 70, 32 * L + 70), 10 ** 6])
        if rng.random() < 0.3:                                # near cancellation
            y, d = x + rng.choice([0, 1, -1, 1 << rng.randrange(32 * L - 2)]) if x else 0, 0
            y = max(0, min(y, (1 << (32 * L - 1)) - 1))
        e = rng.randrange(-300, 300)
        a.append(x if rng.random() < 0.5 else -x)
        b.append(y if rng.random() < 0.5 else -y)
        ea.append(EZ if x == 0 else e + d)
        eb.append(EZ if y == 0 else e)
    P = lambda v: to_planes(v, L)
    return P(a), np.array(ea, np.int64), P(b), np.array(eb, np.int64)


def entrywise_parity(L, n, seed):
    rng = random.Random(seed)
    a, ea, b, eb = operands(rng, n, L)
    A, B = F.MPF(cu(a), cu(ea)), F.MPF(cu(b), cu(eb))
    for what, got, ref in (("mul", F.mul(A, B), O.mpf_mul(a, ea, b, eb)), ("add", F.add(A, B), O.mpf_add(a, ea, b, eb, 1)),
                           ("sub", F.add(A, B, -1), O.mpf_add(a, ea, b, eb, -1))):
        m, e = got.m.cpu().numpy(), got.e.cpu().numpy()
        bad = [i for i in range(n) if e[i] != ref[1][i] or not np.array_equal(m[:, i], ref[0][:, i])]
        assert not bad, (what, L, n, bad[:5])
    one = F.MPF(A.m[:, :1].contiguous(), A.e[:1].contiguous())
    s = F.mul(B, one)
    ref = O.mpf_mul(b, eb, np.repeat(a[:, :1], n, 1), np.repeat(ea[:1], n))
    assert np.array_equal(s.m.cpu().numpy(), ref[0]) and np.array_equal(s.e.cpu().numpy(), ref[1]), ("broadcast", L, n)


@pytest.mark.parametrize("L", [1, 2, 7, 8, 9, 16, 17, 24, 25, 28, 29, 32, 33, 36, 37, 40, 41])
@pytest.mark.parametrize("n", [1, 64, 65, 700])
def test_products_and_sums(L, n):
    entrywise_parity(L, n, 31 * L + n)

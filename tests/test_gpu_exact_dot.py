"""The C entry point sdpv_exact_dot (exact words and bit lengths of products with a few columns) against Python
integers: limb counts around a word per lane, one slice of k and several, one or two rows in a large batch,
strided operands, extreme limb values, the shortest and the longest result."""
import random

import numpy as np
import pytest
import torch

from sdpvibe_amd import _lib
from tests.intutil import to_planes, words_to_int

pytestmark = pytest.mark.gpu


def exact_dot_parity(put, L, nb, M, N, K, NW, ldk, stream):
    rng = random.Random(L + nb + M + K)
    top = 1 << (32 * L - 1)
    vals = lambda n: [rng.choice([rng.randrange(-top, top), rng.randrange(-9, 9), top - 1, -top, 0]) for _ in range(n)]
    a, b = vals(nb * M * K), vals(nb * N * K)
    A, B = (to_planes(v, L).reshape(L, nb, r, K) for v, r in ((a, M), (b, N)))
    room = np.full((L, nb, M, K, ldk), 77, np.int32)     # entries ldk words apart along k
    room[..., 0] = A
    A, B = put(torch.from_numpy(room)), put(torch.from_numpy(np.ascontiguousarray(B)))
    E = nb * M * N
    W, bl = put(torch.zeros((NW, E), dtype=torch.int32)), put(torch.zeros(E, dtype=torch.int64))
    nwork = int(_lib.lib().sdpv_exact_dot_work(L, nb, M, N, K))
    work = put(torch.zeros(max(nwork, 1), dtype=torch.int64))
    _lib.call("sdpv_exact_dot", _lib.ptr(A), nb * M * K * ldk, M * K * ldk, K * ldk, ldk, _lib.ptr(B), nb * N * K, N * K, K, 1,
              L, nb, M, N, K, _lib.ptr(W), NW, _lib.ptr(bl), _lib.ptr(work), nwork, stream())
    W, bl = W.cpu().numpy().view(np.uint32), bl.cpu().numpy()
    for e in range(E):
        q, j = divmod(e, N)
        s = sum(x * y for x, y in zip(a[q * K:(q + 1) * K], b[(q // M * N + j) * K:(q // M * N + j + 1) * K]))
        assert words_to_int(W[:, e]) == s and bl[e] == (~s if s < 0 else s).bit_length(), (L, nb, M, N, K, e)


@pytest.mark.parametrize("L,nb,M,N,K,NW,ldk", [
    (1, 1, 1, 1, 1, 4, 1), (2, 1, 40, 2, 5, 128, 3), (8, 2, 3, 1, 200, 18, 1), (24, 1, 33, 1, 20, 50, 2), (25, 1, 5, 2, 300, 52, 1),
    (31, 1, 3, 3, 17, 64, 1), (33, 1, 2, 1, 64, 68, 1), (63, 1, 3, 1, 40, 128, 1), (49, 256, 1, 1, 3, 100, 1), (24, 512, 1, 2, 70, 50, 1),
    (3, 1, 2, 1, 0, 8, 1)])
def test_exact_dot(L, nb, M, N, K, NW, ldk):
    exact_dot_parity(lambda t: t.cuda(), L, nb, M, N, K, NW, ldk, _lib.stream)

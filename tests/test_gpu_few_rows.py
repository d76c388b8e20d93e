"""Products of one or two rows with one or two columns in large batches (a wave per column, or per slice of its k)
against the residue path, bit for bit: limb counts around a word per lane and around the limb classes of the
rule, k around the chunks of 64 and the slices, views as operands, extreme limb values, every rounding, the
fused subtraction, and batches on both sides of the rule."""
import random

import numpy as np
import pytest
import torch

from sdpvibe_amd import batched as Bm
from tests.intutil import to_planes

pytestmark = pytest.mark.gpu


def limbs(rng, L, *shape):
    """random two's complement limbs, one entry in six an extreme one"""
    n, top = int(np.prod(shape)), 1 << (32 * L - 1)
    edge = to_planes([top - 1, -top, 0, -1, 1, -top + 1], L)
    m = np.random.default_rng(rng.randrange(1 << 30)).integers(-2 ** 31, 2 ** 31, (L, n), dtype=np.int64).astype(np.int32)
    at = np.random.default_rng(rng.randrange(1 << 30)).integers(0, 36, n)
    for q in range(6):
        m[:, at == q] = edge[:, q:q + 1]
    return torch.from_numpy(m.reshape((L,) + shape))


def few_rows_parity(put, L, nb, M, N, K, monkeypatch, seed=0):
    rng = random.Random(L + nb + M + N + K + seed)
    big = put(limbs(rng, L, nb, K + 3, M + 1))
    A = Bm.BMP(big[:, :, 2:2 + K, 1:].transpose(2, 3), -(32 * L - 8))       # read through its strides
    B = Bm.BMP(put(limbs(rng, L, nb, N, K)), 0)
    re = put(torch.tensor([[rng.randrange(-70, 70) - 32 * L for _ in range(N)] for _ in range(nb)]))
    X = Bm.BMP(put(limbs(rng, L, nb, M, N)) >> 1, put(torch.tensor([[rng.randrange(-70, 70) for _ in range(N)]
                                                                    for _ in range(nb)])))
    fixed = -(32 * L - 8) - 32 * L + 32 * L + 120
    got, want = [], []
    for direct, out in ((True, got), (False, want)):
        monkeypatch.setattr(Bm, "_narrow", lambda *a, **k: direct)
        for mode in ("col", "mat", fixed):
            C = Bm.bgemm_nt(A, B, out_exp=mode, bt_rowexp=re)
            out += [C.limbs] + ([] if mode == fixed else [C.exp])
        C = Bm._minus_product(X, A, Bm.BMP(B.limbs.transpose(2, 3), re))
        out += [C.limbs, C.exp]
    for q, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(a, b), (L, nb, M, N, K, q)


@pytest.mark.parametrize("L,nb,M,N,K", [
    (3, 2600, 1, 1, 5), (8, 2560, 1, 1, 64), (8, 2559, 1, 1, 65), (8, 1300, 2, 2, 130), (24, 1024, 1, 1, 42), (24, 1023, 1, 1, 1),
    (24, 1100, 2, 2, 64), (24, 520, 1, 2, 129), (25, 1030, 1, 1, 63), (31, 512, 1, 2, 9), (32, 600, 1, 1, 300), (35, 512, 1, 1, 200),
    (35, 128, 2, 2, 1000), (40, 300, 2, 2, 257), (48, 256, 1, 1, 42), (48, 64, 1, 1, 3000), (49, 256, 1, 1, 1), (63, 130, 2, 2, 127),
    (63, 64, 1, 2, 500), (63, 2, 2, 1, 20000), (33, 256, 2, 2, 66), (33, 260, 3, 2, 66)])
def test_few_rows_equal_the_residue_path(L, nb, M, N, K, monkeypatch):
    few_rows_parity(lambda t: t.cuda(), L, nb, M, N, K, monkeypatch)

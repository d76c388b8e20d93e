"""KSum against the oracle's product over the stacked segments, bit for bit: few columns (exact words per entry) with
one and two words per lane and residues, segments of far different magnitudes, empty ones among them."""
import random

import numpy as np
import pytest
import torch

from oracle import oracle as O
from sdpvibe_amd import batched as Bm
from sdpvibe_amd import mpf as F
from tests.test_gpu_narrow import entries

pytestmark = pytest.mark.gpu


def ksum_parity(put, L, M, N, sizes):
    rng = random.Random(10 * L + M + N)
    segs = []
    for k in sizes:
        far = rng.randrange(-200, 200)
        (am, ae), (bm, be) = entries(rng, (k, M), L, 60), entries(rng, (k, N), L, 60)
        ae = np.where(ae == F.EZ, ae, ae + far)
        if M > 1:                                        # a column of zeros over all segments
            am[:, :, 1], ae[:, 1] = 0, F.EZ
        segs.append((am, ae, bm, be))
    stack = [np.ascontiguousarray(np.concatenate([s[q] for s in segs], 1 - q % 2)) for q in range(4)]
    rm, re_ = O.mpf_gemm(stack[0][:, None], stack[1][None], stack[2][:, None], stack[3][None], True, False)
    mpfs = [(F.MPF(put(torch.from_numpy(am)), put(torch.from_numpy(ae))), F.MPF(put(torch.from_numpy(bm)), put(torch.from_numpy(be))))
            for am, ae, bm, be in segs]
    EA = torch.stack([F.col_exps(a) for a, _ in mpfs]).amax(0)
    EB = torch.stack([F.col_exps(b) for _, b in mpfs]).amax(0)
    acc = F.KSum(EA, EB, L)
    for a, b in mpfs:
        acc.add(a, b)
    got = acc.result()
    assert np.array_equal(got.m.cpu().numpy(), rm[:, 0]) and np.array_equal(got.e.cpu().numpy(), re_[0]), (L, M, N, sizes)


@pytest.mark.parametrize("direct", [True, False])        # whichever the rule picks
@pytest.mark.parametrize("N", [1, 2])
@pytest.mark.parametrize("L", [1, 8, 24, 26, 33, 41, 63])
def test_ksum_against_the_oracle(L, N, direct, monkeypatch):
    monkeypatch.setattr(Bm, "_narrow", lambda *a, **k: direct)
    for M, sizes in ((37, [7, 0, 40, 1]), (70, [130, 33]), (3, [1, 300, 16])):
        ksum_parity(lambda t: t.cuda(), L, M, N, sizes)

"""The residue split of small launches (prime blocks shared out over the grid, limbs rounded in registers)
against the form of large launches on the same rows: every limb count of a table width and its neighbours, views
as operands, right and left shifts, zero entries, fewer limbs in than out, ranges of primes."""
import numpy as np
import pytest
import torch

from sdpvibe_amd import mpmat

pytestmark = pytest.mark.gpu
EZ = -(1 << 40)


@pytest.mark.parametrize("L", [1, 2, 7, 8, 9, 16, 17, 24, 25, 31, 32])
@pytest.mark.parametrize("shifted", [False, True])
def test_small_split_against_large(L, shifted):
    R = mpmat.ctx(L)
    rng = np.random.default_rng(10 * L + shifted)
    few, many, K = 21, 16 * 150, 55                      # 2 x 4 tiles against 150 x 4
    for Lin in sorted({L, max(L - 1, 1)}):
        X = rng.integers(-2 ** 31, 2 ** 31, (Lin, K, many), dtype=np.int64).astype(np.int32)
        X[-1] >>= 8                                      # room for the left shifts
        e = Erow = None
        if shifted:
            e = rng.integers(-70 * L, 4, (K, many)).astype(np.int64)
            e[rng.random((K, many)) < 0.1] = EZ
            Erow = torch.full((many,), 0, dtype=torch.int64, device="cuda")
            e = torch.from_numpy(e).cuda()
        X = torch.from_numpy(X).cuda()
        for k0, kc, kp, g0, G in ((0, K, 64, 0, R.n), (3, 31, 32, 5, min(40, R.n - 5))):
            def split(rows):
                Rh = torch.empty((G, kp // 16, rows, 16), dtype=torch.int8, device="cuda")
                Rl = torch.empty_like(Rh)
                R.split(X, e, Erow, Lin, K * many, 1, rows, 0, 1, many, k0, kc, kp, Rh, Rl, g0, G)
                return Rh, Rl
            for a, b in zip(split(few), split(many)):
                assert torch.equal(a, b[:, :, :few]), (L, Lin, shifted, k0)

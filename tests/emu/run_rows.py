"""Emulated products of one or two rows in large batches, and sums over segments with one or two columns, against
the oracle; sdpv_exact_dot against integers. Usage: run_rows.py few L nb M N K | ksum L M N |
exact_dot L nb M N K NW ldk"""
import os
import random
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__)))))
from tests.emu import harness  # noqa: E402

harness.install()
import numpy as np  # noqa: E402
import torch  # noqa: E402

from oracle import oracle as O  # noqa: E402
from sdpvibe_amd import batched as Bm  # noqa: E402


def few(L, nb, M, N, K):
    from tests.test_gpu_few_rows import limbs
    rng = random.Random(L + nb)
    A, B = limbs(rng, L, nb, M, K), limbs(rng, L, nb, N, K)
    eA = -(32 * L - 8)
    eB = np.array([[rng.randrange(-40, 40) - 32 * L for _ in range(N)] for _ in range(nb)], np.int64)
    for mode, om in (("col", 1), (17, 0)):
        C = Bm.bgemm_nt(Bm.BMP(A, eA), Bm.BMP(B, 0), out_exp=mode, bt_rowexp=torch.from_numpy(eB))
        ref, rexp = O.bgemm_nt(A.numpy(), B.numpy(), eA + eB, om, np.full((nb, N), 17, np.int64) if om == 0 else None)
        assert np.array_equal(C.limbs.numpy(), ref) and (om == 0 or np.array_equal(C.exp.numpy(), rexp)), mode


def ksum(L, M, N):
    from tests.test_gpu_ksum_oracle import ksum_parity
    Bm._narrow = lambda *a, **k: True
    ksum_parity(lambda t: t, L, M, N, [5, 0, 18])


def exact_dot(*case):
    from tests.test_gpu_exact_dot import exact_dot_parity
    exact_dot_parity(lambda t: t, *case, lambda: None)


if __name__ == "__main__":
    {"few": few, "ksum": ksum, "exact_dot": exact_dot}[sys.argv[1]](*(int(a) for a in sys.argv[2:]))
    print("ok")

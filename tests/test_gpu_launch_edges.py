"""The residue split and the reconstruction on both sides of the launch sizes where they change their form: the
small split against the general one (also on part of the primes and a short, padded inner dimension), and
reconstructions just below and above the sizes at which four waves share an entry group."""
import numpy as np
import pytest
import torch

from sdpvibe_amd import mpmat

pytestmark = pytest.mark.gpu
EZ = -(1 << 40)
SMALL = 512                                              # 16 x 16 tiles up to which a split takes the small form


@pytest.mark.parametrize("L", [1, 8, 9, 16, 24, 25, 32])
@pytest.mark.parametrize("shifted", [False, True])
def test_split_forms_agree(L, shifted):
    R = mpmat.ctx(L)
    rng = np.random.default_rng(100 + 2 * L + shifted)
    K, many = 45, 16 * 300 + 5
    X = rng.integers(-2 ** 31, 2 ** 31, (L, K, many), dtype=np.int64).astype(np.int32)
    X[-1] >>= 8                                          # room for the left shifts
    e = Erow = None
    if shifted:
        e = rng.integers(-70 * L, 4, (K, many)).astype(np.int64)
        e[rng.random((K, many)) < 0.1] = EZ
        e, Erow = torch.from_numpy(e).cuda(), torch.zeros((many,), dtype=torch.int64, device="cuda")
    X = torch.from_numpy(X).cuda()
    tiles = lambda rows, kp: -(-rows // 16) * (kp // 16)
    # whole and partial prime ranges, an offset into k, both paddings; row counts that share the prime blocks out
    # over many workgroups, some, and none
    for k0, kc, kp, g0, G in ((0, K, 64, 0, R.n), (3, 31, 32, 5, min(40, R.n - 5)), (40, 5, 32, R.n - 1, 1)):
        def split(rows):
            Rh = torch.full((G, kp // 16, rows, 16), 99, dtype=torch.int8, device="cuda")
            Rl = Rh.clone()
            R.split(X, e, Erow, L, K * many, 1, rows, 0, 1, many, k0, kc, kp, Rh, Rl, g0, G)
            return Rh, Rl
        assert tiles(many, kp) > SMALL
        general = split(many)
        for rows in (21, 16 * 12, 16 * 80, 16 * (SMALL // (kp // 16))):
            assert tiles(rows, kp) <= SMALL
            for a, b in zip(split(rows), general):
                assert torch.equal(a, b[:, :, :rows]), (L, shifted, kp, rows)


@pytest.mark.parametrize("L", [8, 24, 25, 36])
def test_reconstructions_around_the_form_changes(L):
    R = mpmat.ctx(L)
    rng = np.random.default_rng(L)
    rows = 64 * 1100
    half = np.array(R.mods, np.int64)[:, None, None] // 2
    part = rng.integers(-8128, 8129, (R.n, 512, 1)) % (2 * half) - half
    part[:, 0] = 0
    full = torch.from_numpy(np.tile(part, (1, rows // 512 + 1, 1))[:, :rows].astype(np.int16)).cuda()
    ecol = torch.zeros(1, dtype=torch.int64, device="cuda")
    X0 = torch.arange(L * rows, device="cuda", dtype=torch.int32).view(L, 1, rows, 1) * 77777

    def run(n):
        acc = full[:, :n].contiguous()
        W, bl, _ = R.crt_block(acc, 1, 0, 1, n, True)
        out = torch.empty((L, n, 1), dtype=torch.int32, device="cuda")
        e = torch.empty((n, 1), dtype=torch.int64, device="cuda")
        R.crt(acc, n, 1, 0, 1, 1, outm=out, oute=e, L=L, plane=n, ldo=1, Mb=n, ecol=ecol, scaled=True)
        X = X0[:, :, :n].clone(memory_format=torch.contiguous_format)
        R.crt_fixed(acc, 1, n, 1, X, 0, 32 * L + 3, None, X, -1)
        return W, bl, out[..., 0], e[:, 0], X[:, 0, :, 0]

    want = run(rows)                                     # single waves
    for groups in (7, 512, 513, 640, 768, 769, 1024, 1025):
        n = 64 * groups - 5
        for name, a, b in zip(("words", "bits", "limbs", "exponents", "sum"), run(n), want):
            assert torch.equal(a, b[..., :n]), (L, groups, name)

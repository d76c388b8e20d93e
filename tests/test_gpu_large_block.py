"""Blocks to and from a stack of more than 2^30 places per limb."""
import pytest
import torch

from sdpvibe_amd import mpf as F

pytestmark = pytest.mark.gpu


def test_stack_of_more_than_two_to_the_thirty_places():
    n, L = 32800, 1                                      # 1.08e9 places: 4.3 GB of limbs, 8.6 GB of exponents
    m = torch.full((L, 1, n, n), 7, dtype=torch.int32, device="cuda")
    e = torch.full((1, n, n), 7, dtype=torch.int64, device="cuda")
    bm = torch.randint(-2 ** 31, 2 ** 31, (L, n, 3), dtype=torch.int32, device="cuda")
    be = torch.randint(-99, 99, (n, 3), device="cuda")
    F._copy_blocks([(bm, be)], m, e, True)
    assert torch.equal(m[:, 0, :, :3], bm) and torch.equal(e[0, :, :3], be)
    assert not m[:, 0, :, 3:].any() and bool((e[0, :, 3:] == F.EZ).all())
    m[0, 0, n - 1, 2], e[0, n - 1, 2] = 11, 12
    gm, ge = torch.zeros_like(bm), torch.zeros_like(be)
    F._copy_blocks([(gm, ge)], m, e, False)
    assert torch.equal(gm, m[:, 0, :, :3]) and torch.equal(ge, e[0, :, :3]) and int(gm[0, n - 1, 2]) == 11

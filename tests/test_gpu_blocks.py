"""Blocks copied to and from a stack in one launch against slice assignment: more blocks than one launch takes,
full, ragged and empty blocks, views with any strides, limb counts that are not a multiple of a group."""
import pytest
import torch

from sdpvibe_amd import mpf as F

pytestmark = pytest.mark.gpu
EZ = -(1 << 40)


@pytest.mark.parametrize("L,rows,cols,count", [(1, 1, 1, 1), (7, 32, 5, 3), (8, 33, 64, 32), (24, 64, 64, 33), (9, 17, 1, 70)])
def test_copy_blocks(L, rows, cols, count):
    g = torch.Generator("cpu").manual_seed(L + count)
    rnd = lambda *s: torch.randint(-2 ** 31, 2 ** 31, s, generator=g, dtype=torch.int64)
    places = []
    for j in range(count):
        r, c = (rows, cols) if j % 3 == 0 else (rows - j % (rows + 1), max(cols - j % 7, 0))
        m, e = rnd(L, r + 2, c + 1).to(torch.int32).cuda()[:, 1:1 + r, :c], rnd(r, c).cuda()
        if j % 2:
            m, e = (rnd(L, c, r).to(torch.int32).cuda().transpose(1, 2), rnd(c, r).cuda().t())
        places.append((m, e))
    M = torch.full((L, count, rows, cols), 7, dtype=torch.int32, device="cuda")
    E = torch.full((count, rows, cols), 7, dtype=torch.int64, device="cuda")
    F._copy_blocks(places, M, E, True)
    rm, re = torch.zeros_like(M), torch.full_like(E, EZ)
    for j, (m, e) in enumerate(places):
        rm[:, j, :e.shape[0], :e.shape[1]], re[j, :e.shape[0], :e.shape[1]] = m, e
    assert torch.equal(M, rm) and torch.equal(E, re)
    back = [(torch.zeros_like(m), torch.zeros_like(e)) for m, e in places]
    F._copy_blocks(back, M, E, False)
    for (m, e), (bm, be) in zip(places, back):
        assert torch.equal(m, bm) and torch.equal(e, be)
    assert torch.equal(M, rm) and torch.equal(E, re)


def test_blocks_that_do_not_fit_are_refused():
    M, E = torch.zeros((2, 1, 4, 4), dtype=torch.int32, device="cuda"), torch.zeros((1, 4, 4), dtype=torch.int64, device="cuda")
    for r, c, L in ((5, 4, 2), (4, 5, 2), (4, 4, 1)):
        with pytest.raises(ValueError):
            F._copy_blocks([(torch.zeros((L, r, c), dtype=torch.int32, device="cuda"),
                             torch.zeros((r, c), dtype=torch.int64, device="cuda"))], M, E, True)

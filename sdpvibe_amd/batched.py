"""Batched multiprecision linear algebra: nb independent blocks of one shape per launch (the
reference's sdpvibe/batched.py interface).

A BMP is a stack of nb fixed-point matrices: limbs (L, nb, R, C) and an exponent that is either one
Python int for the whole stack or one per (block, column), an (nb, C) int64 tensor.

Recursive Cholesky and triangular solves walk a split tree of the dimension (halved at multiples of
the tile size bt, leaves are bt x bt diagonal tiles), so the split points, and with them every
rounding, are those of the reference's recursion; the factor is written in place into one output
array instead of being concatenated level by level.
"""
import torch

from ._lib import call, lib, ptr, ptr_view, stream
from .limbops import _errbuf, add_same, shift_round
from .mpmat import ctx, headroom_bits, residue_gemm
from .rns import dev


class BMP:
    """stack of nb fixed-point matrices (see the module docstring)"""
    __slots__ = ("limbs", "exp")

    def __init__(self, limbs, exp):
        self.limbs, self.exp = limbs, exp

    @property
    def L(self):
        return self.limbs.shape[0]

    @property
    def shape(self):
        return tuple(self.limbs.shape[1:])

    def expt(self):
        """(nb, C) exponents, materialised when uniform"""
        if isinstance(self.exp, int):
            nb, _, C = self.shape
            return torch.full((nb, C), self.exp, dtype=torch.int64, device=self.limbs.device)
        return self.exp

    def __getitem__(self, idx):
        rows, cols = idx
        e = self.exp if isinstance(self.exp, int) else self.exp[:, cols].contiguous()
        return BMP(self.limbs[:, :, rows, cols].contiguous(), e)

    def t(self):
        """per-block transpose (uniform exponent only)"""
        if not isinstance(self.exp, int):
            raise ValueError("transpose needs a uniform exponent")
        return BMP(self.limbs.transpose(2, 3).contiguous(), self.exp)

    def flat(self):
        return self.limbs.reshape(self.L, -1)


def brescale(A, new_exp, Lout=None, share_exp=False):
    """A re-rounded to new_exp (int, or (nb, C) per block and column), into Lout limbs; the result
    holds a copy of a tensor new_exp, or new_exp itself with share_exp"""
    nb, R, C = A.shape
    Lo = Lout or A.L
    if isinstance(new_exp, int) and isinstance(A.exp, int):
        shift = torch.full((nb * R * C,), new_exp - A.exp, dtype=torch.int64, device=A.limbs.device)
        return BMP(shift_round(A.flat(), shift, Lo).view(Lo, nb, R, C), new_exp)
    if not torch.is_tensor(new_exp):
        new_exp = torch.full((nb, C), int(new_exp), dtype=torch.int64, device=A.limbs.device)
    shift = (new_exp - A.expt()).unsqueeze(1).expand(nb, R, C).reshape(-1)
    return BMP(shift_round(A.flat(), shift, Lo).view(Lo, nb, R, C), new_exp if share_exp else new_exp.clone())


def badd(A, B, alpha=1, out_exp=None):
    """A + alpha B: an exact limb addition when both operands sit at the int exponent out_exp; with
    out_exp 'align', both rounded to one more than the larger exponent of each (block, column) and
    added (one fused kernel)"""
    nb, R, C = A.shape
    L = A.L
    if isinstance(out_exp, int):
        if A.exp != out_exp or B.exp != out_exp:
            raise ValueError("exact addition needs both operands at the output exponent")
        return BMP(add_same(A.flat(), B.flat(), alpha).view(L, nb, R, C), out_exp)
    if out_exp != "align":
        raise ValueError("out_exp must be an int or 'align'")
    out = torch.empty((L, nb, R, C), dtype=torch.int32, device=A.limbs.device)
    e = torch.empty((nb, C), dtype=torch.int64, device=A.limbs.device)
    Al, Bl = A.flat().contiguous(), B.flat().contiguous()
    Ae, Be = A.expt().contiguous(), B.expt().contiguous()
    call("sdpv_badd_align", ptr(Al), ptr(Bl), ptr(Ae), ptr(Be), ptr(out), ptr(e), L, nb, R, C, int(alpha), stream())
    return BMP(out, e)


def _residue_desc(R, X, nb, rows, K):
    """residues of a fixed-point (L, nb, rows, K) limb tensor, all primes; panels of rows j0..j0+jw.
    X may be any view with non-negative strides (a transpose, a row or column slice): the split
    reads it in place through its strides."""
    L = X.shape[0]
    if X.is_contiguous():
        base, plane, ldb, ldr, ldk = X, nb * rows * K, rows * K, K, 1
    else:
        plane, ldb, ldr, ldk = X.stride()
        if min(plane, ldb, ldr, ldk) < 0:
            X = X.contiguous()
            base, plane, ldb, ldr, ldk = X, nb * rows * K, rows * K, K, 1
        else:                                # the storage from X's first entry to its last, flat
            extent = (L - 1) * plane + (nb - 1) * ldb + (rows - 1) * ldr + (K - 1) * ldk + 1
            base = torch.as_strided(X, (extent,), (1,))

    def f(k0, kc, kp, j0, jw):
        r0, rn = (0, rows) if j0 is None else (j0, jw)
        Rh = torch.empty((R.n, kp // 16, nb * rn, 16), dtype=torch.int8, device=X.device)
        Rl = torch.empty_like(Rh)
        # a panel is read in place: rows r0.. of every block, offset r0*ldr into each limb plane
        R.split(base, None, None, L, plane, nb, rn, ldb, ldr, ldk, k0, kc, kp, Rh, Rl, off=r0 * ldr)
        return Rh, Rl
    return f


def _rows(B, r0, r1=None):
    """rows r0..r1 of every block as a view (the exponents are per column, shared)"""
    return BMP(B.limbs[:, :, r0:r1, :], B.exp)


def bgemm_nt(A, Bt, out_exp="col", kc=4096, bt_rowexp=None, bt_cache=None, plus=None, sgn=1, dest=None):
    """C[b] = A[b] @ Bt[b]^T for all b (exact, then rounded). A: uniform exponent per block (int or
    (nb, C) tensor read at column 0). Bt: int exponent or per-row exponents bt_rowexp (nb, N).
    out_exp: 'col' (dynamic per (block, column)), 'mat' (dynamic per block), or int (fixed).
    bt_cache: a dict that keeps Bt's residues between calls with the same Bt (its limbs must not
    change while the dict is in use); the residues depend on the limbs only (batched.py:165-197).
    With an int out_exp: plus, a BMP at out_exp (possibly a view), gives badd(plus, C, sgn, out_exp); dest, a
    limb view (L, nb, M, N) that overlaps neither A nor Bt (plus may be its BMP), receives the result."""
    nb, M, K = A.shape
    nb2, N, K2 = Bt.shape
    assert nb == nb2 and K == K2
    L = A.L
    R = ctx(L)
    eB = Bt.exp if bt_rowexp is None else bt_rowexp
    if Bt.L == L and _narrow(M, N, K, L, nb):
        C = _narrow_product(A, Bt, eB, out_exp if isinstance(out_exp, int) else "col")
        if plus is not None:
            C = badd(plus, C, sgn, out_exp=out_exp)
        if dest is not None:
            dest.copy_(C.limbs)
            C = BMP(dest, C.exp)
        if out_exp == "mat":
            C = brescale(C, C.exp.amax(1, keepdim=True).expand(nb, N).contiguous())
        return C
    eA = A.exp if isinstance(A.exp, int) else A.exp[:, 0]
    cache = {}
    Al, Bl = A.limbs, Bt.limbs                      # views are read through their strides
    same = Al.data_ptr() == Bl.data_ptr() and Al.stride() == Bl.stride() and Al.shape == Bl.shape
    fa = _residue_desc(R, Al, nb, M, K)
    fb = _residue_desc(R, Bl, nb, N, K)

    def fa0(k0, kc_, kp, j0, jw):
        cache["a"] = fa(k0, kc_, kp, None, None)
        return cache["a"]

    def fb0(k0, kc_, kp, j0, jw):
        if same and (j0, jw) == (0, N):
            return cache["a"]
        if bt_cache is None:
            return fb(k0, kc_, kp, j0, jw)
        key = (L, k0, kc_, kp, j0, jw)
        if key not in bt_cache:
            bt_cache[key] = fb(k0, kc_, kp, j0, jw)
        return bt_cache[key]

    if isinstance(out_exp, int):
        # a fixed output exponent: the reconstruction rounds by per-(block, column) shifts alone, adds `plus`
        # and writes to `dest` in the same pass (chol(Q) at N = 3000, L = 24: 8368 launches, now 6147, and
        # 116 ms, now 100)
        out = torch.empty((L, nb, M, N), dtype=torch.int32, device=dev) if dest is None else dest
        s0, s = 0, None
        if isinstance(eA, int) and isinstance(eB, int):
            s0 = out_exp - (eA + eB)
        else:
            s = _fixed_shift(eA, eB, out_exp, nb, N, bt_cache)
        X = None
        if plus is not None:
            if plus.exp != out_exp:
                raise ValueError("exact addition needs both operands at the output exponent")
            X = plus.limbs if plus.limbs.stride(3) == 1 else plus.limbs.contiguous()
        for j0, jw, acc in residue_gemm(R, fa0, fb0, nb, M, N, K):
            R.crt_fixed(acc, nb, M, jw, out, j0, s0, s, X, sgn, _errbuf())
        return BMP(out, out_exp)
    out = torch.empty((L, nb, M, N), dtype=torch.int32, device=dev)
    if isinstance(eA, int) and isinstance(eB, int):
        e_in = eA + eB
    else:
        eA_t = eA if torch.is_tensor(eA) else torch.full((nb,), eA, dtype=torch.int64, device=dev)
        eB_t = eB if torch.is_tensor(eB) else torch.full((nb, N), eB, dtype=torch.int64, device=dev)
        if eB_t.dim() == 1:
            eB_t = eB_t[:, None].expand(nb, N)
        e_in = (eA_t[:, None] + eB_t).contiguous()
    exps = torch.empty((nb, N), dtype=torch.int64, device=dev)
    for j0, jw, acc in residue_gemm(R, fa0, fb0, nb, M, N, K):
        _bcrt_round_panel(R, acc, nb, M, N, j0, jw, e_in, out_exp, L, out, exps)
    C = BMP(out, exps)
    if out_exp == "mat":
        C = brescale(C, exps.amax(1, keepdim=True).expand(nb, N).contiguous())
    return C


# Products with at most NARROW right-hand-side columns may be formed directly (sdpv_narrow): the matrix is read
# once and multiplied as bytes, where the residue path reduces each of its entries modulo every prime, whatever
# the columns. NARROW_MK bounds rows times inner length of a block, so that its workgroups stay inside a launch's
# grid; NARROW_K the inner dimension of one direct product.
NARROW = 2
NARROW_MK = 1 << 40
NARROW_K = 1 << 17


def _narrow(M, N, K, L, nb=1, rounded=False):
    """whether nb products of (M, K) with (K, N) are formed directly. rounded: the operands carry exponents and are
    rounded on the way in (mpf.gemm); else their limbs are multiplied as they are.

    The direct kernel starts a workgroup per 32 rows, column and 128 k, and from 41 limbs on no longer holds its
    operands in registers; the residue path's time is that of splitting M + N rows (and of one product tile per
    32 rows). Residues over direct, time on one MI355X, full rows, one / two columns (60 x 162 x 1500, 20 x 160 x 1000):
    rounded L = 24 3.5 / 2.1, L = 40 2.1 / 1.3, L = 48 0.98 / 0.57, L = 63 0.73 / 0.41; as they are L = 40 2.8 / 2.0, L = 48 1.4 / 0.89,
    L = 63 0.96 / 0.55; a 200 x 200 block, where launches count: rounded L = 40 2.0 / 1.9, L = 48 1.3 / 1.1, L = 63
    1.0 / 1.0; as they are 1.6 to 4 at every limb count. Few rows in large batches, rounded, two columns (500 x 2 x
    1000): L = 8 0.92, L = 24 0.63, L = 40 0.39; (3000 x 2 x 42): L = 8 1.7, L = 24 1.3, L = 40 0.85."""
    if N > NARROW or L > 63 or K > NARROW_K or M * K > NARROW_MK:
        return False
    if L <= 40 and not rounded:
        return True
    ks, tiles = -(-L // 8), -(-M // 32)
    cols = nb * N * tiles
    if cols <= 16 and (ks <= 6 or not rounded):              # too few product tiles to fill the device
        return True
    work = cols * K // 128                                   # slices of 32 rows and 128 k
    if not rounded:
        if (M <= 2 and M * N * K <= 200) or (ks == 6 and N == 1):
            return True
        return work <= 256 if ks == 6 else N * work <= 200
    if ks <= 5:
        few = cols * -(-K // 128) <= 256
    else:
        few = N * work <= 128 if ks == 6 else N == 1 and 24 <= work <= 64
    if few:                                                  # both routes wait for launches: fewer of them
        return True
    # per block, in times of a k of a split row: splits and a tile of the product against k of a slice
    per_k = (4.5, 6.8, 6.8, 10, 11, 36, 54, 47)[ks - 1]
    if ks <= 5:
        return (M + N + 3 * tiles) * K + 900 * tiles >= N * tiles * (K + 20) * per_k
    return (M + N + 3 * tiles) * K + 470 * tiles >= N * tiles * K * per_k


def narrow_work(L, nb, M, N, K, device):
    """scratch of sdpv_narrow for this shape: (tensor, int64 entries)"""
    n = int(lib().sdpv_exact_dot_work(L, nb, M, N, K))
    return torch.empty((max(n, 1),), dtype=torch.int64, device=device), n


def _exponents(e, nb, C):
    """exponents that broadcast to (nb, C) as a contiguous int64 tensor of that shape"""
    if e.shape != (nb, C):
        e = e.expand(nb, C)
    return (e if e.dtype == torch.int64 else e.to(torch.int64)).contiguous()


def _narrow_product(A, Bt, eB, out_exp, plus=None, sgn=1):
    """A Bt^T with few rows of Bt as one direct product, rounded to the int out_exp or per (block,
    column) ('col'); plus: a BMP X (possibly a view), the result is then badd(X, A Bt^T, sgn, 'align')"""
    Al, Bl = A.limbs, Bt.limbs
    L, nb, M, K = Al.shape
    N = Bl.shape[2]
    fixed = isinstance(out_exp, int)
    if Bl.shape != (L, nb, N, K):              # the kernel trusts these sizes
        raise ValueError(f"product of {tuple(Al.shape)} and {tuple(Bl.shape)} limbs")
    if M == 0 and not fixed:
        raise IndexError("no rows to take the columns' exponents from")
    out = torch.empty((L, nb, M, N), dtype=torch.int32, device=Al.device)
    e0, ea, lea, eb = 0, None, 0, None
    if isinstance(A.exp, int):
        e0 += A.exp
    else:
        ea = _exponents(A.exp[:, :1], nb, 1)   # (nb, C), read at column 0
        lea = 1
    if isinstance(eB, int):
        e0 += eB
    else:
        eb = _exponents(eB[:, None] if eB.dim() == 1 else eB, nb, N)
    exps = None if fixed else torch.empty((nb, N), dtype=torch.int64, device=Al.device)
    X, sx, eX = None, (0, 0, 0, 0), None
    if plus is not None:
        Xl = plus.limbs
        if Xl.shape != out.shape:
            raise ValueError(f"sum of {tuple(Xl.shape)} and {tuple(out.shape)} limbs")
        X, sx, eX = ptr_view(Xl), Xl.stride(), _exponents(plus.expt(), nb, N)
    work, nwork = narrow_work(L, nb, M, N, K, Al.device)
    call("sdpv_narrow", ptr_view(Al), None, None, *Al.stride(), ptr_view(Bl), None, None, *Bl.stride(), L, nb, M, N, K,
         2 if fixed else 3, ptr(out), nb * M * N, M * N, N, 1, ptr(exps), e0, ptr(ea), lea, ptr(eb),
         out_exp if fixed else 0, X, *sx, ptr(eX), sgn, ptr(_errbuf()), ptr(work), nwork, stream())
    return BMP(out, out_exp if fixed else exps)


def _fixed_shift(eA, eB, out_exp, nb, N, cache=None):
    """out_exp - (eA + eB) per (block, column), (nb * N,) int64: the rounding shifts of a product
    with a fixed output exponent. eA: int or (nb,); eB: int, (nb,) or (nb, N), not both ints. Kept in `cache`
    when eA is an int (the cache of a Bt whose exponents do not change)"""
    key = ("shift", eA, out_exp) if cache is not None and isinstance(eA, int) else None
    if key is not None and key in cache:
        return cache[key]
    eA_t = eA if torch.is_tensor(eA) else torch.full((nb,), eA, dtype=torch.int64, device=dev)
    eB_t = eB if torch.is_tensor(eB) else torch.full((nb, N), eB, dtype=torch.int64, device=dev)
    if eB_t.dim() == 1:
        eB_t = eB_t[:, None].expand(nb, N)
    s = (out_exp - (eA_t[:, None] + eB_t)).reshape(-1).contiguous()
    if key is not None:
        cache[key] = s
    return s


def _bcrt_round_panel(R, acc, nb, M, N, j0, jw, e_in, out_exp, L, out, exps):
    """_bcrt_round (batched.py:200-231) of one column panel with dynamic output exponents: exact
    products -> L limbs (a fixed output exponent is rounded in bgemm_nt's reconstruction)"""
    rows = nb * M
    Wd, bl, Bq = R.crt_block(acc, jw, 0, jw, rows, True)               # entries (b*M + i)*jw + jj
    ein = e_in if torch.is_tensor(e_in) else torch.full((nb, N), e_in, dtype=torch.int64, device=dev)
    sj = bl.view(nb, M, jw).amax(1) - headroom_bits(L)             # (nb, jw)
    ej = ein[:, j0:j0 + jw] + sj
    s = sj[:, None, :].expand(nb, M, jw).reshape(-1)
    exps[:, j0:j0 + jw] = ej
    if (j0, jw) == (0, N):                                          # the whole width: rounded in place
        shift_round(Wd, s, L, out=out.view(L, nb * M * N))
    else:
        out[:, :, :, j0:j0 + jw] = shift_round(Wd, s, L).view(L, nb, M, jw)


# ------------------------------------------------------------------ batched Cholesky / TRSM
class BTile:
    """a factored diagonal tile: Lmp, the factor (fixed point), and X, its explicit inverse (one
    exponent per block); res: residues of X and Lmp as right operands, kept while the factorisation
    that made the tile reuses them (None otherwise)"""
    __slots__ = ("X", "Lmp", "res")


def bchol_tile(A, LI=24, threads=256):
    """factor and invert the bt x bt tiles A (nb, bt, bt) (fixed point at -(32L - 40)) on the GPU:
    (L as a BMP, BTile) with X rounded to headroom_bits(L) below its largest entry, per block. LI and threads are the
    reference's; the kernels have their own (24 words more, and as many threads as the tile takes)"""
    from .basecase import tile_factor_inverse
    nb, b, _ = A.shape
    L = A.L
    if A.exp != -(32 * L - 40):
        raise ValueError("tiles enter at the fixed-point exponent")
    Lw, X, Xe = tile_factor_inverse(A.limbs, b, headroom_bits(L))
    tile = BTile()
    tile.res = None
    tile.Lmp, tile.X = BMP(Lw, A.exp), BMP(X, Xe)
    return tile.Lmp, tile


class _Node:
    """a diagonal range [lo, lo + n) of the split tree; `head`/`tail` its two halves (None for a
    leaf tile); `first` the index of its first leaf tile, `count` its number of tiles"""
    __slots__ = ("lo", "n", "head", "tail", "first", "count")

    def __init__(self, lo, n, bt, first):
        self.lo, self.n, self.first = lo, n, first
        if n <= bt:
            self.head = self.tail = None
            self.count = 1
            return
        k = (n // 2 + bt - 1) // bt * bt                      # leading part: half, up to a tile multiple
        self.head = _Node(lo, k, bt, first)
        self.tail = _Node(lo + k, n - k, bt, first + self.head.count)
        self.count = self.head.count + self.tail.count

    @property
    def k(self):
        return self.head.n


def _tree(n, bt):
    return _Node(0, n, bt, 0)


# a factorisation keeps the residues of its tiles' X and factor, which the panel solves below them
# use at every level of the split tree (331 leaf solves over 94 tiles at n = 3008), when they take
# at most this many bytes
TILE_RES_BUDGET = 1 << 29


def bchol(A, bt=32, refine=1):
    """Cholesky factors of nb SPD equilibrated fixed-point blocks (nb, n, n), n a multiple of bt:
    (L, list of factored diagonal tiles in tree order). Each internal node factors its head, solves
    for the panel below it (btrsm_right), subtracts the panel's Gram matrix exactly and factors
    the tail; the factor is written into one array as it is produced."""
    nb, n, _ = A.shape
    e = A.exp
    out = torch.zeros((A.L, nb, n, n), dtype=torch.int32, device=A.limbs.device)
    tiles = []
    R = ctx(A.L)
    keep_res = nb * (n // bt) * 2 * 2 * R.n * R.kp(bt) * bt <= TILE_RES_BUDGET

    def factor(node, M):
        lo = node.lo
        if node.head is None:
            if node.n != bt:
                raise ValueError("the dimension must be a multiple of the tile size")
            Lt, t = bchol_tile(M)
            if keep_res:
                t.res = {"X": {}, "L": {}}
            tiles.append(t)
            out[:, :, lo:lo + bt, lo:lo + bt] = Lt.limbs
            return
        k, hi = node.k, lo + node.n
        head, tail = slice(None, k), slice(k, None)
        factor(node.head, _view(M, head, head))
        L11 = _view(BMP(out, e), slice(lo, lo + k), slice(lo, lo + k))
        panel = _right_solve(node.head, _view(M, tail, head), L11, tiles, refine, lo, out[:, :, lo + k:hi, lo:lo + k])
        factor(node.tail, bgemm_nt(panel, panel, out_exp=e, plus=_view(M, tail, tail), sgn=-1))

    factor(_tree(n, bt), A)
    for t in tiles:
        t.res = None
    return BMP(out, e), tiles


def _right_solve(node, B, Lf, tiles, refine, base, dest):
    """X with X Lf^T = B for the node's diagonal block Lf (node offsets relative to `base`), written to the
    limb view `dest`, which overlaps neither B nor Lf"""
    e = Lf.exp
    if node.head is None:
        t = tiles[node.first]
        cx, cl = (None, None) if t.res is None else (t.res["X"], t.res["L"])
        X = bgemm_nt(B, t.X, out_exp=e, bt_rowexp=t.X.exp, bt_cache=cx, dest=dest)
        for _ in range(refine):                              # one residual correction per step
            resid = bgemm_nt(X, t.Lmp, out_exp=e, bt_cache=cl, plus=B, sgn=-1)
            bgemm_nt(resid, t.X, out_exp=e, bt_rowexp=t.X.exp, bt_cache=cx, plus=X, dest=dest)
        return X
    k = node.k
    head, tail, every = slice(None, k), slice(k, None), slice(None)
    X1 = _right_solve(node.head, _view(B, every, head), _view(Lf, head, head), tiles, refine, base, dest[..., :k])
    rest = bgemm_nt(X1, _view(Lf, tail, head), out_exp=e, plus=_view(B, every, tail), sgn=-1)
    _right_solve(node.tail, rest, _view(Lf, tail, tail), tiles, refine, base, dest[..., k:])
    return BMP(dest, e)


def btrsm_right(B, Lf, tiles, bt=32, refine=1):
    """X with X L^T = B, batched, fixed point (B (nb, m, n), L from bchol)"""
    return _right_solve(_tree(B.shape[2], bt), B, Lf, tiles, refine, 0,
                        torch.empty(B.limbs.shape, dtype=torch.int32, device=B.limbs.device))


def _as_rows(B):
    """B^T per block as the row-exponent operand of bgemm_nt (its column exponents go separately): a
    transposed view, which the residue split reads through its strides"""
    return BMP(B.limbs.transpose(2, 3), 0)


def _apply_tile(X, Lm, B, refine):
    """Lm^-1 B through the explicit tile inverse X, then `refine` residual corrections, with
    per-(block, column) exponents"""
    P = bgemm_nt(X, _as_rows(B), out_exp="col", bt_rowexp=B.expt())
    for _ in range(refine):
        resid = badd(B, bgemm_nt(Lm, _as_rows(P), out_exp="col", bt_rowexp=P.expt()), -1, out_exp="align")
        P = badd(P, bgemm_nt(X, _as_rows(resid), out_exp="col", bt_rowexp=resid.expt()), 1, out_exp="align")
    return P


def _stack_common(P1, P2):
    """[P1; P2] with one exponent per (block, column): both parts re-rounded to the larger"""
    m1, m2 = P1.limbs.contiguous(), P2.limbs.contiguous()
    L, nb, R1, C = m1.shape
    R2 = m2.shape[2]
    if m2.shape != (L, nb, R2, C):             # the kernel trusts these sizes
        raise ValueError(f"halves of {tuple(m1.shape)} and {tuple(m2.shape)} limbs")
    out = torch.empty((L, nb, R1 + R2, C), dtype=torch.int32, device=m1.device)
    ee = torch.empty((nb, C), dtype=torch.int64, device=m1.device)
    e1, e2 = _exponents(P1.expt(), nb, C), _exponents(P2.expt(), nb, C)
    call("sdpv_stack_common", ptr(m1), ptr(e1), ptr(m2), ptr(e2), ptr(out), ptr(ee), L, nb, R1, R2, C, ptr(_errbuf()),
         stream())
    return BMP(out, ee)


def _minus_product(X, A, P):
    """badd(X, A P, -1, 'align'): rows X of a right-hand side less a block of the factor times the part
    already solved; one direct product with few columns"""
    nb, M, K = A.shape
    if P.L == A.L and _narrow(M, P.shape[2], K, A.L, nb):
        return _narrow_product(A, _as_rows(P), P.expt(), "col", plus=X, sgn=-1)
    return badd(X, bgemm_nt(A, _as_rows(P), out_exp="col", bt_rowexp=P.expt()), -1, out_exp="align")


def _view(A, rows, cols, transpose=False):
    """a sub-block of a uniform-exponent BMP as a view (no copy): bgemm_nt reads views through their
    strides, badd and the tile factorisation copy what they need contiguous"""
    limbs = A.limbs[:, :, rows, cols]
    return BMP(limbs.transpose(2, 3) if transpose else limbs, A.exp)


def _left_solve(node, Lf, B, tiles, refine, upper):
    """L^-1 B (upper=False, forward: head first) or L^-T B (upper=True, backward: tail first)"""
    if node.head is None:
        t = tiles[node.first]
        if upper:
            XT = BMP(t.X.limbs.transpose(2, 3).contiguous(), t.X.exp)
            return _apply_tile(XT, t.Lmp.t(), B, refine)
        return _apply_tile(t.X, t.Lmp, B, refine)
    k = node.k
    head, tail = slice(None, k), slice(k, None)
    if not upper:
        P1 = _left_solve(node.head, _view(Lf, head, head), _rows(B, 0, k), tiles, refine, upper)
        P2 = _left_solve(node.tail, _view(Lf, tail, tail), _minus_product(_rows(B, k), _view(Lf, tail, head), P1), tiles,
                         refine, upper)
    else:
        P2 = _left_solve(node.tail, _view(Lf, tail, tail), _rows(B, k), tiles, refine, upper)
        P1 = _left_solve(node.head, _view(Lf, head, head),
                         _minus_product(_rows(B, 0, k), _view(Lf, tail, head, transpose=True), P2), tiles, refine, upper)
    return _stack_common(P1, P2)


def btrsm_left(Lf, B, tiles, bt=32, refine=0):
    """P = L^-1 B batched; B (nb, n, m) with per-(block, column) exponents, and so is P"""
    return _left_solve(_tree(B.shape[1], bt), Lf, B, tiles, refine, False)


def btrsm_left_T(Lf, B, tiles, bt=32, refine=1):
    """P = L^-T B batched (L lower, fixed point from bchol)"""
    return _left_solve(_tree(B.shape[1], bt), Lf, B, tiles, refine, True)

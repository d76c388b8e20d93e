"""The work that a user of this package has it do, as cases with seeded inputs, timed and compared
by outside tools: listed() and draw() name cases, prepare() makes what a program has in hand before
the call, run() makes one call (or one iteration) through the public entry points.

Every matrix is multiprecision (L 32-bit limbs and an exponent per entry), so outputs are whole
numbers: limbs and exponents. Sizes are those of semidefinite programs: Schur complements of 500 to
3000 variables, batches of blocks of dimension 8 to 192, 256 to 1120 bits (L = 8 to 35; the command
line's default of 400 bits is L = 14, the benchmark runs 768 bits, L = 24).
"""
import math

import numpy as np
import torch

from sdpvibe_amd import mpf as F
from sdpvibe_amd.blockops import mirror_lower
from sdpvibe_amd.ipm import Solver
from sdpvibe_amd.sdp import SDP
from sdpvibe_amd.steplen import min_eig
from sdpvibe_amd.synthetic import powers_of_ten

DEV = "cuda"


def listed():
    return [
        # the products of one small program's blocks at the command line's default precision
        # (bilinear bases against X): short calls, where launches and latency count
        dict(name="gemm small blocks", kind="gemm", L=14, nb=20, M=27, K=14, N=27, transA=True, transB=False),
        # X Y of the dimension-3 blocks of the benchmark's program, both parities (60 blocks)
        dict(name="gemm blocks", kind="gemm", L=24, nb=120, M=42, K=42, N=42, transA=False, transB=False),
        # the plain exact product of the benchmark's GEMM configuration
        dict(name="gemm 512", kind="gemm", L=24, nb=1, M=512, K=512, N=512, transA=False, transB=False),
        # P dy of an iteration: tall blocks against one vector each
        dict(name="gemm vector", kind="gemm", L=24, nb=60, M=162, K=3000, N=1, transA=False, transB=False),
        # entrywise products summed in pairs: the terms of the Schur complement's assembly
        dict(name="entrywise", kind="entry", L=24, nb=120, M=81, N=81),
        # chol(Q) of one iteration at N = 3000
        dict(name="chol 3000", kind="chol", L=24, nb=1, n=3000),
        # the Newton step's solve with Q's factor, one right-hand side
        dict(name="solve vector", kind="solve", L=24, nb=1, n=1000, m=1),
        # P = L_S^-1 B of the dimension-3 blocks: a batch of factors against wide panels
        dict(name="solve panel", kind="lower", L=24, nb=60, n=162, m=3000),
        # Q = sum P^T P over two groups of blocks
        dict(name="gram 3000", kind="gram", L=24, N=3000, rows=8100, chunks=2),
        # factors and solves of 400 blocks of uneven dimension, condition up to 1e80
        dict(name="uneven blocks", kind="uneven", L=24, blocks=400, dmin=8, dmax=96, m=4),
        # the smallest eigenvalue of L^-1 dM L^-T over the dimension-3 blocks: the step length
        dict(name="step length", kind="step", L=24, nb=120, n=42),
        # one whole iteration of the interior-point method, a third of the benchmark's program
        dict(name="iteration", kind="ipm", L=24, n1=100, n3=20, N=1000),
    ]


def _size(rng, lo, hi):
    """a whole number in [lo, hi], uniform in its logarithm"""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """a case of the same ranges: any of the kinds, sizes spread over their logarithm"""
    L = rng.choice((8, 11, 14, 18, 24, 24, 26, 32, 35))
    kind = rng.choice(("gemm", "gemm", "gemm", "entry", "chol", "solve", "lower", "gram", "uneven", "step", "ipm"))
    if kind == "gemm":
        form = rng.choice(("blocks", "plain", "vector"))
        tA, tB = rng.random() < 0.3, rng.random() < 0.3
        if form == "blocks":
            return dict(kind=kind, L=L, nb=_size(rng, 2, 300), M=_size(rng, 8, 100), K=_size(rng, 8, 100),
                        N=_size(rng, 8, 100), transA=tA, transB=tB)
        if form == "plain":
            return dict(kind=kind, L=L, nb=1, M=_size(rng, 32, 800), K=_size(rng, 32, 800), N=_size(rng, 32, 800),
                        transA=tA, transB=tB)
        return dict(kind=kind, L=L, nb=_size(rng, 1, 60), M=_size(rng, 20, 160), K=_size(rng, 100, 2500),
                    N=rng.choice((1, 2, 4)), transA=tA, transB=tB)
    if kind == "entry":
        return dict(kind=kind, L=L, nb=_size(rng, 1, 120), M=_size(rng, 5, 100), N=_size(rng, 5, 100))
    if kind == "chol":
        if rng.random() < 0.5:
            return dict(kind=kind, L=L, nb=1, n=_size(rng, 200, 1600))
        return dict(kind=kind, L=L, nb=_size(rng, 2, 300), n=_size(rng, 8, 180))
    if kind == "solve":
        return dict(kind=kind, L=L, nb=1, n=_size(rng, 200, 1600), m=rng.choice((1, 1, 2, 5)))
    if kind == "lower":
        return dict(kind=kind, L=L, nb=_size(rng, 2, 60), n=_size(rng, 20, 180), m=_size(rng, 40, 1500))
    if kind == "gram":
        return dict(kind=kind, L=L, N=_size(rng, 200, 2000), rows=_size(rng, 100, 4000), chunks=rng.choice((1, 2, 3)))
    if kind == "uneven":
        return dict(kind=kind, L=L, blocks=_size(rng, 10, 200), dmin=8, dmax=rng.choice((40, 64, 96)),
                    m=rng.choice((1, 2, 4)))
    if kind == "step":
        return dict(kind=kind, L=L, nb=_size(rng, 2, 200), n=_size(rng, 6, 60))
    return dict(kind="ipm", L=rng.choice((14, 24, 26)), n1=_size(rng, 8, 60), n3=_size(rng, 2, 12), N=_size(rng, 100, 600))


# ------------------------------------------------------------------ inputs
def _rand(shape, L, gen, espread=16):
    """normalised entries of either sign: uniform mantissas of 32 L - 2 bits, magnitudes spread over
    2 espread binades"""
    m = torch.randint(-2 ** 31, 2 ** 31, (L, *shape), dtype=torch.int32, device=DEV, generator=gen)
    top = torch.randint(2 ** 29, 2 ** 30, shape, dtype=torch.int32, device=DEV, generator=gen)
    neg = torch.rand(shape, device=DEV, generator=gen) < 0.5
    m[-1] = torch.where(neg, ~top, top)
    e = torch.randint(-espread, espread + 1, shape, device=DEV, generator=gen) - F.NBITS(L)
    return F.MPF(m, e)


def _spd(nb, n, L, gen):
    """G G^T per block, the columns of G scaled down to 2^-2L: condition numbers of about 2^4L, as
    Schur complements have them some iterations before the optimum"""
    G = _rand((nb, n, n), L, gen, espread=1)
    down = -(2 * L * torch.arange(n, device=DEV)) // max(n, 1)
    G = G.shift(down[None, None, :])
    return F.gemm(G, G, transB=True)


def _pair(X):
    return [X.m, X.e]


def prepare(case, seed):
    kind, L = case["kind"], case["L"]
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    if kind == "gemm":
        nb, M, K, N = case["nb"], case["M"], case["K"], case["N"]
        A = _rand((nb, K, M) if case["transA"] else (nb, M, K), L, gen)
        B = _rand((nb, N, K) if case["transB"] else (nb, K, N), L, gen)
        return dict(case, A=A, B=B)
    if kind == "entry":
        shape = (case["nb"], case["M"], case["N"])
        return dict(case, A=[_rand(shape, L, gen) for _ in range(4)])
    if kind == "chol":
        A = _spd(case["nb"], case["n"], L, gen)
        return dict(case, A=A.reshape(case["n"], case["n"]) if case["nb"] == 1 else A)
    if kind in ("solve", "lower"):
        nb, n, m = case["nb"], case["n"], case["m"]
        B = _rand((nb, n, m), L, gen)
        return dict(case, C=F.Chol(_spd(nb, n, L, gen)), B=B)
    if kind == "gram":
        return dict(case, P=[_rand((case["rows"], case["N"]), L, gen) for _ in range(case["chunks"])])
    if kind == "uneven":
        # the dimensions are the program's structure: the same for every seed
        dims = np.random.default_rng(case["blocks"]).integers(case["dmin"], case["dmax"] + 1, case["blocks"]).tolist()
        rng = np.random.default_rng(seed)
        p10 = powers_of_ten(-40, 40, L)
        one = F.eye(case["dmax"], L)
        blocks, rhs = [], []
        for n in dims:                                  # D (G G^T + I) D, D = diag(10^u)
            G = _rand((n, n), L, gen, espread=1)
            A = F.add(F.gemm(G, G, transB=True), one[:n, :n])
            u = torch.from_numpy(rng.integers(-20, 21, n)).to(DEV)
            at = u[:, None] + u[None, :] + 40
            blocks.append(F.mul(A, F.MPF(p10.m[:, at].contiguous(), p10.e[at].contiguous())))
            rhs.append(_rand((n, case["m"]), L, gen))
        return dict(case, blocks=blocks, rhs=rhs)
    if kind == "step":
        nb, n = case["nb"], case["n"]
        G = _rand((nb, n, n), L, gen, espread=1)
        X = F.add(F.gemm(G, G, transB=True), F.MPF(*(t.contiguous() for t in _batch_eye(nb, n, L))))
        return dict(case, C=F.Chol(X), dM=F.symmetrize(_rand((nb, n, n), L, gen, espread=2)))
    # a solver two iterations after its start: its launch graphs are captured by then
    sdp = SDP.polynomial(n1=case["n1"], n3=case["n3"], degree=26, N=case["N"], L=L, seed=seed)
    solver = Solver(sdp, L)
    steps = solver.iterate(max_iter=500)
    next(steps)
    next(steps)
    return dict(case, solver=solver, steps=steps)


def _batch_eye(nb, n, L):
    one = F.eye(n, L)
    return one.m[:, None].expand(-1, nb, -1, -1), one.e[None].expand(nb, -1, -1)


# ------------------------------------------------------------------ one pass
def run(state):
    kind = state["kind"]
    if kind == "gemm":
        return _pair(F.gemm(state["A"], state["B"], transA=state["transA"], transB=state["transB"]))
    if kind == "entry":
        a, b, c, d = state["A"]
        return _pair(F.add(F.mul(a, b), F.mul(c, d)))
    if kind == "chol":
        C = F.Chol(state["A"])
        return [C.Lt.limbs, C.k]
    if kind == "solve":
        return _pair(state["C"].solve(state["B"]))
    if kind == "lower":
        return _pair(state["C"].solve_lower(state["B"]))
    if kind == "gram":
        G = F.GramAcc(state["N"], state["L"])
        for P in state["P"]:
            G.add(P)
        return _pair(mirror_lower(G.result()))
    if kind == "uneven":
        C = F.BucketedChol(state["blocks"])
        X = C.solve(state["rhs"])
        factors = [t for _, ch in C.groups for t in (ch.Lt.limbs, ch.k)]
        return factors + [torch.cat([x.m.flatten(1) for x in X], 1), torch.cat([x.e.flatten() for x in X])]
    if kind == "step":
        return float(min_eig([state["C"]], [state["dM"]]))
    solver = state["solver"]
    next(state["steps"])                                # the iterate, its factors and the new y
    out = _pair(solver.y)
    for st in solver.state:
        out += _pair(st.x) + _pair(st.X) + _pair(st.Y)
    f = solver.final_factors
    for C in f["X"] + f["Y"] + f["S"] + [f["Q"]]:
        out += [C.Lt.limbs, C.k]
    return out


# ------------------------------------------------------------------ what a pass cannot do without
def _mac(L):
    """operations of one exact L-limb multiply-add on 8-bit matrix units: the product's 64 L + 18 bits
    in residues of 14 bits, three byte products each"""
    return 2 * 3 * math.ceil((64 * L + 18) / 14)


def work(case):
    """each input read once and each output written once (4 L + 8 bytes an entry), and the exact
    multiply-adds of the mathematical definition"""
    kind, L = case["kind"], case["L"]
    ent = 4 * L + 8
    if kind == "gemm":
        nb, M, K, N = case["nb"], case["M"], case["K"], case["N"]
        return dict(bytes=nb * (M * K + K * N + M * N) * ent, flops=nb * M * K * N * _mac(L))
    if kind == "entry":
        n = case["nb"] * case["M"] * case["N"]
        return dict(bytes=5 * n * ent, flops=2 * n * 2 * L * L)
    if kind == "chol":
        nb, n = case["nb"], case["n"]
        return dict(bytes=nb * n * (n + 1) // 2 * (ent + 4 * L), flops=nb * n ** 3 / 6 * _mac(L))
    if kind in ("solve", "lower"):
        nb, n, m = case["nb"], case["n"], case["m"]
        sweeps = 2 if kind == "solve" else 1
        return dict(bytes=nb * (n * (n + 1) // 2 * 4 * L + 2 * n * m * ent), flops=sweeps * nb * n * n / 2 * m * _mac(L))
    if kind == "gram":
        N, rows = case["N"], case["rows"] * case["chunks"]
        return dict(bytes=(rows * N + N * N) * ent, flops=rows * N * (N + 1) / 2 * _mac(L + 1))
    if kind == "uneven":
        ns = range(case["dmin"], case["dmax"] + 1)
        n2, n3 = sum(n * n for n in ns) / len(ns), sum(n ** 3 for n in ns) / len(ns)
        return dict(bytes=case["blocks"] * n2 * (ent + 4 * L / 2), flops=case["blocks"] * (n3 / 6 + n2 * case["m"]) * _mac(L))
    if kind == "step":
        nb, n = case["nb"], case["n"]
        return dict(bytes=nb * n * n * 2 * ent, flops=nb * n ** 3 * _mac(L))
    N, rows = case["N"], 27 * case["n1"] + 162 * case["n3"]
    tri = (27 ** 2 * case["n1"] + 162 ** 2 * case["n3"]) * N / 2
    return dict(bytes=rows * N * ent + N * N * ent, flops=(rows * N * N / 2 + tri + N ** 3 / 6) * _mac(L))


def exact(case, seed):
    """limbs and exponents are whole numbers without a 64-bit counterpart; the step length's eigenvalue is
    that of the generalised problem dM v = lambda X v in float64"""
    if case["kind"] != "step":
        return None
    state = prepare(case, seed)
    nb, n, L = case["nb"], case["n"], case["L"]
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    G = torch.from_numpy(_rand((nb, n, n), L, gen, espread=1).to_float())
    X = G @ G.transpose(1, 2).contiguous() + torch.eye(n, dtype=torch.float64)
    M = torch.from_numpy(state["dM"].to_float())
    Li = torch.linalg.inv(torch.linalg.cholesky(X))
    W = Li @ M @ Li.transpose(1, 2).contiguous()
    return float(torch.linalg.eigvalsh((W + W.transpose(1, 2)) / 2).min())

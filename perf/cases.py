"""What the speed of this package is measured on: its public routines as a user's program calls them.

Every case is a dict of plain values: the operation `op` and its sizes (n diagonal blocks of order b, an arrowhead
of a rows, r right-hand sides).  prepare() makes what the program has in hand before the call, run() is one pass and
exact() gives run()'s outputs in plain torch, in float64, without this package.

Operations
  evaluate  one step of a Laplace-approximation loop: pobtaf, log-determinant, both pobtas sweeps, pobtasi; the
            matrix is kept, so the blocks are copied first.  a = 0 calls the arrowless pobtf / pobts / pobtsi
  factor    pobtaf on a copy of the kept matrix
  selinv    pobtasi on a copy of the kept factor
  solve     pobtas "N" then "C" with the kept factor on a copy of the right-hand sides
  gradient  pobta_logdet_quad, forward and backward, to the blocks and the data vector
  batched   a BatchedBTA plan over systems of uneven sizes: factor, log-determinant, solve, selected inverse
  refine    pobtaf_mixed on a copy, then pobtas_refine: a solve to FP64 accuracy through the mixed FP32/FP64 factor
  general   ddbtasc and ddbtasci on a copy of a diagonally dominant matrix without symmetry
"""

import math
import random

import torch

import serinv_amd.algs as algs
from serinv_amd.autograd import pobta_logdet_quad
from serinv_amd.batched import BatchedBTA
from serinv_amd.logdet import pobta_logdet
from serinv_amd.mixed import pobtaf_mixed, pobtas_refine

# Factor of the diagonal shift 3b + a (tip: n*b + a) of the SPD matrices, whose entries are uniform in [0, 1): 1 makes
# every row dominant, about 1/6 is where the matrix stops being positive definite.
GAMMA = 0.2


def _case(name, op, n, b, a, r):
    return {"name": name, "op": op, "n": n, "b": b, "a": a, "r": r}


def listed():
    return [
        # the smallest call: a small model, where launches and host work count
        _case("evaluate-n8-b96-a12", "evaluate", 8, 96, 12, 2),
        # the reference's small CPU configuration
        _case("evaluate-n32-b64-a16", "evaluate", 32, 64, 16, 1),
        # odd block size and an arrowhead wider than one 64-wide tile
        _case("evaluate-n24-b200-a70", "evaluate", 24, 200, 70, 4),
        # a purely temporal model: no arrowhead, block size not a multiple of any tile
        _case("evaluate-n100-b130-a0", "evaluate", 100, 130, 0, 3),
        # a hyperparameter gradient at the differentiable configuration's size
        _case("gradient-n128-b256-a8", "gradient", 128, 256, 8, 1),
        # a sweep over 64 hyperparameter settings of uneven sizes, one plan
        {"name": "batched-64", "op": "batched", "systems": 64, "sizes": 63, "r": 4},
        # the large spatio-temporal configuration, call by call
        _case("factor-n256-b1024-a32", "factor", 256, 1024, 32, 0),
        _case("selinv-n256-b1024-a32", "selinv", 256, 1024, 32, 0),
        _case("solve-n256-b1024-a32-r1", "solve", 256, 1024, 32, 1),
        _case("solve-n256-b1024-a32-r64", "solve", 256, 1024, 32, 64),
        # the mixed-precision solve on one partition of it
        _case("refine-n64-b1024-a32-r16", "refine", 64, 1024, 32, 16),
        # the family without symmetry, medium size
        _case("general-n32-b512-a16", "general", 32, 512, 16, 0),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng):
    """One more case: sizes over the listed cases' range (by their logarithm), odd ones among them."""
    op = rng.choice(["evaluate", "evaluate", "evaluate", "gradient", "batched", "factor", "selinv", "solve", "solve",
                     "refine", "general"])
    if op == "batched":
        return {"op": op, "systems": _log_int(rng, 6, 64), "sizes": rng.randrange(1 << 20), "r": _log_int(rng, 1, 16)}
    most = max(work(c)["flops"] for c in listed())
    while True:
        b = _log_int(rng, 24, 1024)
        if rng.random() < 0.5:  # block sizes that are tiles of 64, 16 or 8 are as usual as odd ones
            b = max(24, b // 8 * 8) if b < 128 else (b // 64 * 64 if rng.random() < 0.5 else b // 16 * 16)
        a = 0 if op == "evaluate" and rng.random() < 0.25 else _log_int(rng, 1, 100)
        r = {"evaluate": _log_int(rng, 1, 16), "gradient": _log_int(rng, 1, 4), "solve": _log_int(rng, 1, 64),
             "refine": _log_int(rng, 1, 32)}.get(op, 0)
        case = {"op": op, "n": _log_int(rng, 4, 256), "b": b, "a": a, "r": r}
        if work(case)["flops"] <= most / 2 and case["n"] * b >= 256:
            return case


# ------------------------------------------------------------------ inputs
def _systems(case):
    """Sizes (n, b, a) of a batch: n uniform in [16, 256], b of three block sizes, a uniform in [4, 32]."""
    rng = random.Random(case["sizes"])
    return [(rng.randint(16, 256), rng.choice((64, 128, 256)), rng.randint(4, 32)) for _ in range(case["systems"])]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _uniform(gen, *shape):
    return torch.rand(shape, dtype=torch.float64, device="cuda", generator=gen)


def _spd(n, b, a, gen):
    """A symmetric positive definite BTA matrix: (D, L, R, T)."""
    D = _uniform(gen, n, b, b)
    for i in range(0, n, 64):  # symmetrized in chunks: the largest case holds gigabytes
        D[i:i + 64] = (D[i:i + 64] + D[i:i + 64].mT) * 0.5
    D.diagonal(dim1=1, dim2=2).add_(GAMMA * (3 * b + a))
    L, R, T = _uniform(gen, n - 1, b, b), _uniform(gen, n, a, b), _uniform(gen, a, a)
    T = (T + T.mT) * 0.5
    T.diagonal().add_(GAMMA * (n * b + a))
    return [D, L, R, T]


def _rhs(n, b, a, r, gen):
    return 2.0 * _uniform(gen, n * b + a, r) - 1.0


def _dominant(n, b, a, gen):
    """A diagonally dominant BTA matrix without symmetry: (D, Lo, Up, Rl, Ru, T)."""
    D = _uniform(gen, n, b, b)
    D.diagonal(dim1=1, dim2=2).add_(3 * b + a)
    T = _uniform(gen, a, a)
    T.diagonal().add_(n * b + a)
    return [D, _uniform(gen, n - 1, b, b), _uniform(gen, n - 1, b, b), _uniform(gen, n, a, b), _uniform(gen, n, b, a), T]


def _batch_inputs(case, seed):
    """Each kind of block of all systems in one array, and the systems' views of it."""
    gen = _generator(seed)
    sizes = _systems(case)
    shapes = [[(n, b, b), (n - 1, b, b), (n, a, b), (a, a), (n * b + a, case["r"])] for n, b, a in sizes]
    flat = [torch.empty(sum(math.prod(s[k]) for s in shapes), dtype=torch.float64, device="cuda") for k in range(5)]
    for (n, b, a), views in zip(sizes, _views(flat, shapes)):
        for view, x in zip(views, _spd(n, b, a, gen) + [_rhs(n, b, a, case["r"], gen)]):
            view.copy_(x)
    return flat, shapes


def _views(flat, shapes):
    at, systems = [0] * len(flat), []
    for s in shapes:
        views = []
        for k, shape in enumerate(s):
            size = math.prod(shape)
            views.append(flat[k][at[k]:at[k] + size].view(shape))
            at[k] += size
        systems.append(views)
    return systems


def prepare(case, seed):
    op = case["op"]
    if op == "batched":
        flat, shapes = _batch_inputs(case, seed)
        mine = [torch.empty_like(x) for x in flat]
        views = _views(mine, shapes)
        for x, y in zip(mine, flat):
            x.copy_(y)
        return {"op": op, "A": flat, "F": mine, "plan": BatchedBTA([v[:4] for v in views], rhs=[v[4] for v in views])}
    n, b, a, r = (case[k] for k in "nbar")
    gen = _generator(seed)
    A = _dominant(n, b, a, gen) if op == "general" else _spd(n, b, a, gen)
    state = {"op": op, "a": a, "A": A}
    if r:
        state["B"] = _rhs(n, b, a, r, gen)
        state["X"] = torch.empty_like(state["B"])
    if op == "gradient":
        for x in A + [state["B"]]:
            x.requires_grad_(True)
    elif op == "solve":
        algs.pobtaf(*A)  # the factor is what such a program has
    else:
        state["F"] = [torch.empty_like(x) for x in A]
        if op == "selinv":
            algs.pobtaf(*A)
    return state


# ------------------------------------------------------------------ one pass
def _copied(state):
    for x, y in zip(state["F"], state["A"]):
        x.copy_(y)
    return state["F"]


def run(state):
    op = state["op"]
    if op == "evaluate":
        D, L, R, T = _copied(state)
        X = state["X"].copy_(state["B"])
        if state["a"]:
            algs.pobtaf(D, L, R, T)
            logdet = pobta_logdet(D, T)
            algs.pobtas(D, L, R, T, X, trans="N")
            algs.pobtas(D, L, R, T, X, trans="C")
            algs.pobtasi(D, L, R, T)
            return {"D": D, "L": L, "R": R, "T": T, "X": X, "logdet": logdet}
        algs.pobtf(D, L)
        logdet = pobta_logdet(D)
        algs.pobts(D, L, X, trans="N")
        algs.pobts(D, L, X, trans="C")
        algs.pobtsi(D, L)
        return {"D": D, "L": L, "X": X, "logdet": logdet}
    if op == "factor":
        D, L, R, T = _copied(state)
        algs.pobtaf(D, L, R, T)
        return {"D": D, "L": L, "R": R, "T": T}
    if op == "selinv":
        D, L, R, T = _copied(state)
        algs.pobtasi(D, L, R, T)
        return {"D": D, "L": L, "R": R, "T": T}
    if op == "solve":
        D, L, R, T = state["A"]
        X = state["X"].copy_(state["B"])
        algs.pobtas(D, L, R, T, X, trans="N")
        algs.pobtas(D, L, R, T, X, trans="C")
        return {"X": X}
    if op == "gradient":
        blocks = state["A"] + [state["B"]]
        logdet, quad = pobta_logdet_quad(*blocks)
        grads = torch.autograd.grad(logdet - quad, blocks)
        return {"logdet": logdet.detach(), "quad": quad.detach(), **dict(zip("DLRTy", grads))}
    if op == "batched":
        for x, y in zip(state["F"], state["A"]):
            x.copy_(y)
        state["plan"].run()
        info, logdet, status = state["plan"].results()
        return {"info": info, "logdet": logdet, "status": status, **dict(zip("DLRTX", state["F"]))}
    if op == "refine":
        D, L, R, T = _copied(state)
        X = state["X"].copy_(state["B"])
        pobtaf_mixed(D, L, R, T)
        pobtas_refine(state["A"], (D, L, R, T), X)
        return {"X": X}
    D, Lo, Up, Rl, Ru, T = _copied(state)
    algs.ddbtasc(D, Lo, Up, Rl, Ru, T)
    algs.ddbtasci(D, Lo, Up, Rl, Ru, T)
    return {"D": D, "Lo": Lo, "Up": Up, "Rl": Rl, "Ru": Ru, "T": T}


# ------------------------------------------------------------------ the work it cannot do without
def _blocks(n, b, a):
    return n * b * b + (n - 1) * b * b + n * a * b + a * a


def _factor_flops(n, b, a):
    return ((n - 1) * (7 / 3 * b**3 + 3 * a * b**2 + a * a * b) + b**3 / 3 + a * b**2 + a * a * b + a**3 / 3)


def _selinv_flops(n, b, a):
    return ((n - 1) * (19 / 3 * b**3 + 7 * a * b**2 + 2 * a * a * b) + 4 / 3 * b**3 + 3 * a * b**2 + 2 * a * a * b
            + 2 / 3 * a**3)


def _solve_flops(n, b, a, r):
    """Both sweeps."""
    return 2 * r * (n * b * b + 2 * (n - 1) * b * b + 2 * n * a * b + a * a)


def work(case):
    op = case["op"]
    if op == "batched":
        total = {"bytes": 0, "flops": 0}
        for n, b, a in _systems(case):
            w = work({"op": "evaluate", "n": n, "b": b, "a": a, "r": case["r"]})
            total = {k: total[k] + w[k] for k in total}
        return total
    n, b, a, r = (case[k] for k in "nbar")
    blocks, rows = _blocks(n, b, a), (n * b + a) * r
    factor, selinv, solve = _factor_flops(n, b, a), _selinv_flops(n, b, a), _solve_flops(n, b, a, r)
    if op in ("evaluate", "gradient"):
        return {"bytes": 8 * (2 * blocks + 2 * rows), "flops": factor + selinv + solve}
    if op == "factor":
        return {"bytes": 16 * blocks, "flops": factor}
    if op == "selinv":
        return {"bytes": 16 * blocks, "flops": selinv}
    if op == "solve":
        return {"bytes": 8 * (blocks + 2 * rows), "flops": solve}
    if op == "refine":  # one correction: two solves and a residual
        return {"bytes": 8 * (2 * blocks + 2 * rows), "flops": factor + 3 * solve}
    # general: per block an inverse, two products of the sweep and six of the inversion, and the arrow's share
    return {"bytes": 16 * (n * b * b + 2 * (n - 1) * b * b + 2 * n * a * b + a * a), "flops": n * (18 * b**3 + 26 * a * b * b)}


# ------------------------------------------------------------------ the same in plain torch, float64
def _exact_factor(D, L, R, T):
    D, L, R, T = (x.clone() for x in (D, L, R, T))
    n = D.shape[0]
    for i in range(n):
        D[i] = torch.linalg.cholesky(D[i])
        up = D[i].mT
        R[i] = torch.linalg.solve_triangular(up, R[i], upper=True, left=False)
        T -= R[i] @ R[i].mT
        if i + 1 < n:
            L[i] = torch.linalg.solve_triangular(up, L[i], upper=True, left=False)
            D[i + 1] -= L[i] @ L[i].mT
            R[i + 1] -= R[i] @ L[i].mT
    if T.shape[0]:
        T = torch.linalg.cholesky(T)
    return D, L, R, T


def _lower_inverse(x):
    return torch.linalg.solve_triangular(x, torch.eye(x.shape[0], dtype=x.dtype, device=x.device), upper=False)


def _exact_selinv(D, L, R, T):
    D, L, R = D.clone(), L.clone(), R.clone()
    n = D.shape[0]
    Ti = _lower_inverse(T) if T.shape[0] else T
    T = Ti.mT @ Ti
    for i in range(n - 1, -1, -1):
        inv = _lower_inverse(D[i])
        G, H = (L[i] @ inv if i + 1 < n else None), R[i] @ inv
        D[i] = inv.mT @ inv
        R[i] = -T @ H
        if G is not None:
            L[i] = -(D[i + 1] @ G) - R[i + 1].mT @ H
            R[i] -= R[i + 1] @ G
            D[i] -= L[i].mT @ G
        D[i] -= R[i].mT @ H
    return D, L, R, T


def _exact_solve(D, L, R, T, B):
    n, b = D.shape[:2]
    X = B.clone()
    x, tip = X[:n * b].view(n, b, -1), X[n * b:]
    for i in range(n):
        if i:
            x[i] -= L[i - 1] @ x[i - 1]
        x[i] = torch.linalg.solve_triangular(D[i], x[i], upper=False)
        tip -= R[i] @ x[i]
    if T.shape[0]:
        tip.copy_(torch.linalg.solve_triangular(T, tip, upper=False))
        tip.copy_(torch.linalg.solve_triangular(T.mT, tip, upper=True))
    for i in range(n - 1, -1, -1):
        if i + 1 < n:
            x[i] -= L[i].mT @ x[i + 1]
        x[i] -= R[i].mT @ tip
        x[i] = torch.linalg.solve_triangular(D[i].mT, x[i], upper=True)
    return X


def _exact_logdet(D, T):
    return 2.0 * (D.diagonal(dim1=1, dim2=2).log().sum() + T.diagonal().log().sum())


def _stored_gradient(G):
    """Gradient to a symmetric block of which only the lower triangle is read."""
    return G.tril() + G.tril(-1)


def exact(case, seed):
    op = case["op"]
    if op == "batched":
        flat, shapes = _batch_inputs(case, seed)
        logdet = []
        for D, L, R, T, B in _views(flat, shapes):
            F = _exact_factor(D, L, R, T)
            logdet.append(_exact_logdet(F[0], F[3]))
            B.copy_(_exact_solve(*F, B))
            for x, y in zip((D, L, R, T), _exact_selinv(*F)):
                x.copy_(y)
        return {"info": None, "logdet": torch.stack(logdet), "status": None, **dict(zip("DLRTX", flat))}
    n, b, a, r = (case[k] for k in "nbar")
    gen = _generator(seed)
    if op == "general":
        D, Lo, Up, Rl, Ru, T = _dominant(n, b, a, gen)
        for i in range(n):
            D[i] = torch.linalg.inv(D[i])
            W, V = (D[i] @ Up[i] if i + 1 < n else None), D[i] @ Ru[i]
            if W is not None:
                D[i + 1] -= Lo[i] @ W
                Rl[i + 1] -= Rl[i] @ W
                Ru[i + 1] -= Lo[i] @ V
            T -= Rl[i] @ V
        T = torch.linalg.inv(T)
        for i in range(n - 1, -1, -1):
            S, lo, rl = D[i].clone(), (Lo[i] @ D[i] if i + 1 < n else None), Rl[i] @ D[i]
            if lo is not None:
                up, ru = S @ Up[i], S @ Ru[i]
                Lo[i] = -(D[i + 1] @ lo) - Ru[i + 1] @ rl
                Rl[i] = -(Rl[i + 1] @ lo) - T @ rl
                Up[i] = -(up @ D[i + 1]) - ru @ Rl[i + 1]
                Ru[i] = -(up @ Ru[i + 1]) - ru @ T
                D[i] = S - Up[i] @ lo - Ru[i] @ rl
            else:
                Ru[i] = -(S @ Ru[i]) @ T
                Rl[i] = -T @ rl
                D[i] = S - Ru[i] @ rl
        return {"D": D, "Lo": Lo, "Up": Up, "Rl": Rl, "Ru": Ru, "T": T}
    A = _spd(n, b, a, gen)
    B = _rhs(n, b, a, r, gen) if r else None
    F = _exact_factor(*A)
    if op == "factor":
        return dict(zip("DLRT", F))
    if op == "selinv":
        return dict(zip("DLRT", _exact_selinv(*F)))
    X = _exact_solve(*F, B)
    if op in ("solve", "refine"):
        return {"X": X}
    logdet = _exact_logdet(F[0], F[3])
    D, L, R, T = _exact_selinv(*F)
    if op == "evaluate":
        return {"D": D, "L": L, **({"R": R, "T": T} if a else {}), "X": X, "logdet": logdet}
    x, tip = X[:n * b].view(n, b, r), X[n * b:]
    return {"logdet": logdet, "quad": (B * X).sum(),
            "D": _stored_gradient(D + x @ x.mT), "L": 2.0 * (L + x[1:] @ x[:-1].mT),
            "R": 2.0 * (R + tip @ x.mT), "T": _stored_gradient(T + tip @ tip.mT), "y": -2.0 * X}

"""Performance cases: what programs have this library do, over its real range.

listed() holds the named cases, draw(rng) one more of the same ranges.
prepare() makes what a program holds before the call (the hierarchy with its
operators, or the batch, and the host arrays), run() is one pass through the
public entry points, with the solution read back as a program reads it, and
work() is the least a pass moves and computes.  exact() gives the outputs in
64-bit arithmetic from torch alone: the problem families are written again
here from their definition, and a solve's exact answer is the solution of the
linear system.

Kinds of case:
  solve     a resident operator is solved to a tolerance from x = 0 and the
            solution is copied to the host (precision, smoother, bottom
            solver, family and grid vary)
  ingest    a host program hands over its own 27-point operator and source,
            has the hierarchy built, solves and reads the solution
  smooth    one level's smoother and residual on a given x, as a program that
            builds its own cycle or preconditioner calls them
  batch     independent problems admitted together and advanced to the end
  serve     a burst of requests through the request loop
"""
import math

import numpy as np
import torch

import pgmg_amd as P

FAMILIES = {"face7": P.FAM_FACE7_UNIFORM, "face7log": P.FAM_FACE7_LOGUNI, "q1": P.FAM_Q1_ANISO}
PRECISIONS = {"fp64": P.PREC_FP64, "mixed": P.PREC_MIXED}
SMOOTHERS = {"colour8": P.SMOOTH_COLOUR8, "exact": P.SMOOTH_EXACT}
BOTTOMS = {"gs24": P.BOTTOM_GS24, "lu": P.BOTTOM_LU}
MAX_CYCLES = 400


def _solve(name, m, n, o, family="face7", precision="mixed", smoother="colour8", bottom="gs24", tol=1e-10):
    return {"name": name, "kind": "solve", "m": m, "n": n, "o": o, "family": family, "precision": precision,
            "smoother": smoother, "bottom": bottom, "tol": tol}


def listed():
    return [
        # a small system inside a time step or an outer iteration: latency
        _solve("solve_small", 33, 33, 33),
        # a small ragged system with a direct bottom solve
        _solve("solve_small_ragged_lu", 40, 23, 30, family="q1", precision="fp64", bottom="lu"),
        # an ordinary finite-element system in double precision
        _solve("solve_q1", 65, 65, 65, family="q1", precision="fp64"),
        # an ordinary ragged grid whose rows fill no power of two
        _solve("solve_ragged", 150, 97, 122, family="q1"),
        # the reference's sweep order, for answers that match it bit for bit
        _solve("solve_exact_order", 65, 72, 57, precision="fp64", smoother="exact"),
        # the headline workload, 257^3 to 1e-10, in both precisions
        _solve("solve_large_mixed", 257, 257, 257),
        _solve("solve_large_fp64", 257, 257, 257, precision="fp64"),
        # the largest: rows longer than one wavefront, a dense 27-point operator
        _solve("solve_largest", 385, 257, 321, family="q1"),
        # an implicit step on a periodic box, operator and source from the host
        {"name": "ingest_periodic", "kind": "ingest", "m": 96, "n": 80, "o": 112, "prd": 7, "points": 7,
         "precision": "fp64", "tol": 1e-10},
        # level operations of a program with its own cycle, symmetric sweeps
        {"name": "smooth_symmetric", "kind": "smooth", "m": 161, "n": 130, "o": 147, "points": 27, "mode": 1,
         "sweeps": 2},
        # independent problems of three sizes and strong contrast, solved together
        {"name": "batch", "kind": "batch", "count": 16, "mix": 1, "axes": "33 65 129", "family": "face7log",
         "precision": "mixed", "tol": 1e-8},
        # a burst of requests, axes log-uniform between the smallest and largest served
        {"name": "serve", "kind": "serve", "count": 24, "mix": 1, "low": 17, "high": 129,
         "family": "q1", "precision": "mixed", "tol": 1e-8},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "solve", "ingest", "smooth", "batch", "serve"])
    precision = rng.choice(["fp64", "mixed"])
    if kind == "solve":
        smoother = rng.choice(["colour8", "colour8", "colour8", "exact"])
        base = _log_int(rng, 17, 96 if smoother == "exact" else 257)
        m, n, o = (max(9, int(base * rng.uniform(0.7, 1.0))) for _ in range(3))
        if rng.random() < 0.4:  # the sizes that coarsen evenly
            m, n, o = (1 + 8 * max(1, a // 8) for a in (m, n, o))
        family = rng.choice(["face7", "face7log", "q1"])
        tol = 1e-10
        if family == "face7log":  # hundreds of cycles
            tol, (m, n, o) = 1e-8, (min(a, 97) for a in (m, n, o))
        case = _solve("", m, n, o, family, precision, smoother, rng.choice(["gs24", "gs24", "lu"]), tol)
        del case["name"]
        return case
    if kind == "ingest":
        return {"kind": kind, "m": _log_int(rng, 24, 112), "n": _log_int(rng, 24, 112), "o": _log_int(rng, 24, 112),
                "prd": rng.choice([0, 1, 4, 7]), "points": rng.choice([7, 27]), "precision": precision, "tol": 1e-10}
    if kind == "smooth":
        return {"kind": kind, "m": _log_int(rng, 30, 180), "n": _log_int(rng, 30, 160), "o": _log_int(rng, 30, 160),
                "points": rng.choice([7, 27]), "mode": rng.choice([0, 1]), "sweeps": rng.choice([1, 2, 3])}
    if kind == "batch":
        return {"kind": kind, "count": rng.choice([4, 8, 16]), "mix": rng.randrange(1000), "axes": rng.choice(["33 65 129", "30 48 80"]),
                "family": rng.choice(["face7", "face7log", "q1"]), "precision": precision, "tol": 1e-8}
    return {"kind": kind, "count": rng.choice([6, 12, 24]), "mix": rng.randrange(1000), "low": 17,
            "high": rng.choice([65, 129]), "family": rng.choice(["face7", "q1"]), "precision": precision, "tol": 1e-8}


# ------------------------------------------------------------------ inputs

def _offset(e):
    """(dk, dj, di) of stencil entry e."""
    return e // 9 - 1, e // 3 % 3 - 1, e % 3 - 1


def _host_operator(case, seed):
    """A symmetric diffusion-like operator with random edge weights and a mass
    term (an implicit step), 7 or 27 points, and its source, as host arrays."""
    g = torch.Generator().manual_seed(seed)
    shape = (case["o"], case["n"], case["m"])
    prd = case.get("prd", 0)
    A = torch.zeros(shape + (27,), dtype=torch.float64)
    diag = torch.full(shape, 0.05, dtype=torch.float64)
    for e in range(14, 27):
        d = _offset(e)
        if case["points"] == 7 and sum(map(abs, d)) != 1:
            continue
        w = (1.0 + 9.0 * torch.rand(shape, generator=g, dtype=torch.float64)) / sum(map(abs, d)) ** 2
        back = torch.roll(w, d, dims=(0, 1, 2))  # the same edge, from its other end
        diag += w + back
        A[..., e] = -w
        A[..., 26 - e] = -back
        for axis, step in enumerate(d):  # an edge that leaves the grid is a boundary term
            if step and not (prd >> (2 - axis)) & 1:
                A.select(axis, shape[axis] - 1 if step > 0 else 0)[..., e] = 0.0
                A.select(axis, 0 if step > 0 else shape[axis] - 1)[..., 26 - e] = 0.0
    A[..., 13] = diag
    b = 2.0 * torch.rand(shape, generator=g, dtype=torch.float64) - 1.0
    x = 2.0 * torch.rand(shape, generator=g, dtype=torch.float64) - 1.0
    return A.numpy(), b.numpy(), x.numpy()


def _problems(case, seed):
    """(m, n, o, problem seed) of each problem of a batch or request burst; the
    case's mix fixes the grids, the seed the operators and sources."""
    rng = np.random.default_rng(case["mix"])
    out = []
    for q in range(case["count"]):
        if case["kind"] == "batch":
            m, n, o = (int(a) for a in rng.choice(case["axes"].split(), size=3))
        else:
            lo, hi = math.log(case["low"]), math.log(case["high"])
            m, n, o = (int(round(math.exp(rng.uniform(lo, hi)))) for _ in range(3))
        out.append((m, n, o, 1000 * seed + q))
    return out


def prepare(case, seed):
    state = {"case": case}
    kind = case["kind"]
    dims = [case.get(a) for a in ("m", "n", "o")]
    if kind == "solve":
        h = P.Hierarchy(*dims, precision=PRECISIONS[case["precision"]], smoother=SMOOTHERS[case["smoother"]],
                        bottom=BOTTOMS[case["bottom"]])
        h.generate_problem(FAMILIES[case["family"]], seed)
        h.compute_rats()
        state["h"] = h
    elif kind == "ingest":
        state["A"], state["b"], _ = _host_operator(case, seed)
        state["h"] = P.Hierarchy(*dims, precision=PRECISIONS[case["precision"]], prd=case["prd"])
    elif kind == "smooth":
        A, b, state["x"] = _host_operator(case, seed)
        h = P.Hierarchy(*dims)
        h.set_operator27(A)
        h.set_rhs(b)
        state["h"] = h
    else:
        problems = _problems(case, seed)
        prec = PRECISIONS[case["precision"]]
        need = sum(P.footprint(m, n, o, precision=prec) for m, n, o, _ in problems)
        state["b"] = P.Batch(int(1.05 * need) + (64 << 20), max_slots=case["count"], precision=prec)
        state["problems"] = problems
    return state


# -------------------------------------------------------------------- runs

def _solve_from_zero(h, tol):
    """A solve and its outputs, the history padded to its longest."""
    h.clear_x()
    cycles, hist = h.solve(tol, MAX_CYCLES, check=False)
    history = np.zeros(MAX_CYCLES + 1)
    history[:cycles + 1] = hist
    return {"x": h.get_x(), "cycles": cycles, "history": history}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "solve":
        return _solve_from_zero(state["h"], case["tol"])
    if kind == "ingest":
        h = state["h"]
        h.set_operator27(state["A"])
        h.set_rhs(state["b"])
        h.compute_rats()
        return _solve_from_zero(h, case["tol"])
    if kind == "smooth":
        h = state["h"]
        h.set_x(state["x"])
        h.gauss_seidel(case["mode"], 0, case["sweeps"])
        return {"x": h.get_x(), "residual": h.residual()}
    b, family = state["b"], FAMILIES[case["family"]]
    if kind == "batch":
        slots = [b.admit(m, n, o, family, s, case["tol"], MAX_CYCLES) for m, n, o, s in state["problems"]]
        b.run()
        out = {"x": [b.get_x(s) for s in slots]}
        status = [b.status(s) for s in slots]
        for s in slots:
            b.release(s)
    else:
        res, _ = b.serve([dict(arrival_s=0.0, m=m, n=n, o=o, family=family, seed=s, tol=case["tol"],
                               max_cycles=MAX_CYCLES) for m, n, o, s in state["problems"]])
        out = {"x": [r["x"] for r in res]}
        status = [(r["status"], r["cycles"], r["rel_residual"]) for r in res]
    for key, values in zip(("status", "cycles", "rel_residual"), zip(*status)):
        out[key] = np.array(values)
    return out


def work(case):
    """Least bytes (operator entries, source and solution once each, in the
    host's or the level's doubles) and operations (two per entry and point for
    every sweep and residual: about ten V(2,2) cycles for a solve, with the
    coarser levels' 1/7 on top)."""
    kind = case["kind"]
    if kind in ("batch", "serve"):
        points = sum(m * n * o for m, n, o, _ in _problems(case, 1))
    else:
        points = case["m"] * case["n"] * case["o"]
    entries = case.get("points") or (27 if case.get("family") == "q1" else 7)
    passes = case["sweeps"] * (1 + case["mode"]) + 1 if kind == "smooth" else 10 * 6 * 8 / 7
    words = entries + (4 if kind == "smooth" else 2)
    return {"bytes": 8 * words * points, "flops": 2 * entries * points * passes}


# ------------------------------------------------------- the exact answers

def _u01(seed, stream, idx):
    """Uniform doubles keyed by (seed, stream, index): the splitmix64 finaliser
    of the problem families, in wrapping 64-bit integers."""
    def signed(v):
        v &= (1 << 64) - 1
        return v - (1 << 64) if v >> 63 else v

    def shift(z, q):
        return (z >> q) & ((1 << (64 - q)) - 1)

    def mix(z):
        z = z + signed(0x9e3779b97f4a7c15)
        z = (z ^ shift(z, 30)) * signed(0xbf58476d1ce4e5b9)
        z = (z ^ shift(z, 27)) * signed(0x94d049bb133111eb)
        return z ^ shift(z, 31)

    key = torch.tensor(signed(seed ^ (stream << 56) ^ (stream * 0x632be59bd9b4e019)), device=idx.device)
    return shift(mix(mix(key) + idx), 11).double() * 2.0 ** -53


def _index(dims, device):
    m, n, o = dims
    return torch.arange(m * n * o, device=device).view(o, n, m)


def _face7(family, seed, m, n, o, device):
    """{entry: coefficients} of -div(a grad u) with random face coefficients."""
    def faces(axis):
        size = [m, n, o]
        size[axis] += 1
        u = _u01(seed, axis + 1, _index(size, device))
        return 10.0 ** (4.0 * u - 2.0) if family == "face7log" else 1.0 + 9.0 * u

    A, diag = {}, 0.0
    for axis, (e_low, e_high) in enumerate([(12, 14), (10, 16), (4, 22)]):
        a, dim = faces(axis), 2 - axis
        size = a.shape[dim] - 1
        low, high = a.narrow(dim, 0, size).clone(), a.narrow(dim, 1, size).clone()
        diag = diag + low + high
        low.select(dim, 0).zero_()
        high.select(dim, size - 1).zero_()
        A[e_low], A[e_high] = -low, -high
    A[13] = diag
    return A


def _q1(seed, m, n, o, device):
    """{entry: coefficients} of trilinear elements with a random conductivity
    tensor R diag(1, 10^u1, 10^u2) R^T in every cell."""
    cells = _index((m + 1, n + 1, o + 1), device)
    lam = [torch.ones_like(cells, dtype=torch.float64)]
    lam += [10.0 ** (-2.0 * _u01(seed, stream, cells)) for stream in (5, 6)]
    q = torch.zeros(cells.shape + (4,), dtype=torch.float64, device=device)
    todo = torch.ones_like(cells, dtype=torch.bool)
    for t in range(64):  # a quaternion by rejection
        idx = cells[todo] * 256 + 4 * t
        if not idx.numel():
            break
        cand = torch.stack([2.0 * _u01(seed, 8, idx + c) - 1.0 for c in range(4)], dim=-1)
        s = (cand * cand).sum(-1)
        ok = (s > 1e-6) & (s <= 1.0)
        where = todo.nonzero()[ok]
        q[tuple(where.T)] = cand[ok]
        todo[tuple(where.T)] = False
    a, b, c, d = q.unbind(-1)
    s = a * a + b * b + c * c + d * d
    R = [[a * a + b * b - c * c - d * d, 2 * (b * c - a * d), 2 * (b * d + a * c)],
         [2 * (b * c + a * d), a * a - b * b + c * c - d * d, 2 * (c * d - a * b)],
         [2 * (b * d - a * c), 2 * (c * d + a * b), a * a - b * b - c * c + d * d]]
    K = [[sum(R[p][r] * lam[r] * R[t][r] for r in range(3)) / (s * s) for t in range(3)] for p in range(3)]

    def factor(axis, p, t, la, lb):  # one axis' part of the integral of d_p phi_a d_t phi_b
        ba, bb = (la >> axis) & 1, (lb >> axis) & 1
        if axis == p and axis == t:
            return 1.0 if ba == bb else -1.0
        if axis == p:
            return ba - 0.5
        if axis == t:
            return bb - 0.5
        return 1.0 / 3.0 if ba == bb else 1.0 / 6.0

    A = {e: torch.zeros((o, n, m), dtype=torch.float64, device=device) for e in range(27)}
    for la in range(8):
        own = [1 - ((la >> axis) & 1) for axis in range(3)]  # the point is local node la of this cell
        for lb in range(8):
            step = [((lb >> axis) & 1) - ((la >> axis) & 1) for axis in range(3)]
            entry = (step[2] + 1) * 9 + (step[1] + 1) * 3 + step[0] + 1
            v = sum(K[p][t] * math.prod(factor(axis, p, t, la, lb) for axis in range(3))
                    for p in range(3) for t in range(3))
            A[entry] += v[own[2]:own[2] + o, own[1]:own[1] + n, own[0]:own[0] + m]
    for e, coef in A.items():
        for axis, stepped in enumerate(_offset(e)):
            if stepped:
                coef.select(axis, coef.shape[axis] - 1 if stepped > 0 else 0).zero_()
    return A


def _family(family, seed, m, n, o, device):
    A = _q1(seed, m, n, o, device) if family == "q1" else _face7(family, seed, m, n, o, device)
    return A, 2.0 * _u01(seed, 4, _index((m, n, o), device)) - 1.0


def _neighbour(x, e, prd):
    """x at each point's neighbour of entry e, zero outside the grid."""
    y = x
    for axis, step in enumerate(_offset(e)):
        if step:
            y = torch.roll(y, -step, dims=axis)
            if not (prd >> (2 - axis)) & 1:
                y.select(axis, y.shape[axis] - 1 if step > 0 else 0).zero_()
    return y


def _apply(A, x, prd=0):
    out = A[13] * x
    for e, coef in A.items():
        if e != 13:
            out += coef * _neighbour(x, e, prd)
    return out


def _solution(A, b, prd=0):
    """Conjugate gradients with the diagonal as preconditioner, restarted from
    the true residual until that stops falling."""
    x, best = torch.zeros_like(b), None
    for _ in range(4):
        r = b - _apply(A, x, prd)
        norm = float(r.norm() / b.norm())
        if norm < 2e-15 or (best is not None and norm > 0.5 * best):
            break
        best = norm
        z = r / A[13]
        p, rz, goal = z, (r * z).sum(), 1e-14 * float(b.norm()) if norm == 1.0 else 1e-3 * float(r.norm())
        for it in range(20000):
            q = _apply(A, p, prd)
            alpha = rz / (p * q).sum()
            x = x + alpha * p
            r = r - alpha * q
            if it % 32 == 31 and float(r.norm()) < goal:
                break
            z = r / A[13]
            new = (r * z).sum()
            p, rz = z + (new / rz) * p, new
    return x.cpu().numpy()


def _sweeps(A, b, x, mode, sweeps):
    """Eight-colour Gauss-Seidel: forward sweeps, or forward and backward."""
    colour = torch.zeros(b.shape, dtype=torch.int64, device=b.device)
    for axis, weight in ((0, 4), (1, 2), (2, 1)):
        view = [1, 1, 1]
        view[axis] = -1
        colour += weight * (torch.arange(b.shape[axis], device=b.device) % 2).view(view)
    for _ in range(sweeps):
        for c in list(range(8)) + (list(range(7, -1, -1)) if mode else []):
            new = (b - (_apply(A, x) - A[13] * x)) / A[13]
            x = torch.where(colour == c, new, x)
    return x


def exact(case, seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    kind = case["kind"]
    if kind == "solve":
        if case["m"] * case["n"] * case["o"] > 40_000_000:  # longer than is worth it
            return None
        A, b = _family(case["family"], seed, case["m"], case["n"], case["o"], device)
        return {"x": _solution(A, b), "cycles": None, "history": None}
    if kind in ("ingest", "smooth"):
        A27, b, x = (torch.from_numpy(a).to(device) for a in _host_operator(case, seed))
        A = {e: A27[..., e].contiguous() for e in range(27) if case["points"] == 27 or
             sum(map(abs, _offset(e))) < 2}
        if kind == "ingest":
            return {"x": _solution(A, b, case["prd"]), "cycles": None, "history": None}
        x = _sweeps(A, b, x, case["mode"], case["sweeps"])
        return {"x": x.cpu().numpy(), "residual": (b - _apply(A, x)).cpu().numpy()}
    xs = []
    for m, n, o, s in _problems(case, seed):
        small = m * n * o <= 300_000 or case["count"] <= 8
        xs.append(_solution(*_family(case["family"], s, m, n, o, device)) if small else None)
    return {"x": xs, "status": None, "cycles": None, "rel_residual": None}

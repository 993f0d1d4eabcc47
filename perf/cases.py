"""Work that programs have this framework do, as measurable cases.

A program holds a multiparametric QP (host arrays, as the C ABI takes them)
and calls the library: mpqp() through MpqpLib.run() in one of the precisions
and batchings that the options offer, mpqp_noalloc(), mpqp_many(), the
critical regions of the final sets, the redundancy test of the preprocessing,
or the whole per-problem pipeline of the POP driver.  Problems are drawn by
the package's own generators (Q = G'G + I, unit-norm constraint rows,
b ~ U(1, 2), theta in a box; or their ill-conditioned variant).

A case is a dict of plain values: "op" names the entry point; "n", "m", "p"
are the variables, constraints and parameters, "k" the largest cardinality
that is enumerated.  Results whose count depends on the data go into tables
of a fixed size that the program keeps (-1 or 0 past the last result).
"""
from __future__ import annotations

import itertools
import math

import numpy as np

from mpqpcudasolver_amd import assemble_lps, load_library, precision_stress_mpqp, synthetic_mpqp
from mpqpcudasolver_amd.host import RECORD_DTYPE
from mpqpcudasolver_amd.pop import solve_pop_problem

MIXED, FP64 = 1, 0
PERSISTENT, PLAIN = 1, 0

# outputs of a regions call, in the order that run() and exact() return them
REGION_FIELDS = ("status", "n_rows", "iters", "radius", "center", "parameter_A", "parameter_b", "lagrange_A",
                 "lagrange_b", "cr_A", "cr_b")


def _solve(name, n, m, p, k, mixed, persistent, records=False, stress=False):
    return {"name": name, "op": "solve", "n": n, "m": m, "p": p, "k": k, "mixed": mixed, "persistent": persistent,
            "records": records, "stress": stress}


def listed():
    return [
        # the smallest call: the smoke test's problem with the default options
        # (FP64, one launch per level); launches and synchronisations count
        _solve("tiny_fp64", 10, 20, 2, 2, False, False),
        # the same kind of call from a program that must not allocate
        {"name": "noalloc_small", "op": "noalloc", "n": 20, "m": 40, "p": 4, "k": 2},
        # one problem of the POP driver: preprocessing, full enumeration,
        # second preprocessing, regions
        {"name": "pop_pipeline", "op": "pipeline", "n": 4, "m": 24, "p": 3},
        # full enumeration (k = n) of a small problem, as the POP driver runs
        # it: many candidates, small LPs, FP64 with persistent launches
        _solve("pop_full_fp64", 6, 28, 4, 6, False, True),
        # the mid-size benchmark problem, mixed precision
        _solve("mid_mixed", 30, 62, 8, 4, True, True),
        # the same in the default FP64, with the per-candidate records that a
        # program reads the verdicts from
        _solve("mid_fp64_records", 30, 62, 8, 3, False, False, records=True),
        # ill-conditioned, nearly degenerate data: mixed precision asks for
        # FP32 pivots, the probe sends the call back to FP64
        _solve("stress_mixed", 30, 62, 8, 3, True, True, stress=True),
        # the largest problem, mixed precision: the headline workload
        _solve("large_mixed", 60, 120, 12, 3, True, True),
        # the same problem in FP64, one level less
        _solve("large_fp64", 60, 120, 12, 2, False, True),
        # independent problems of uneven sizes in one call
        {"name": "many_uneven", "op": "many", "count": 16, "shapes": 2, "k": 2},
        # critical regions of final sets of the largest problem
        {"name": "regions_large", "op": "regions", "n": 60, "m": 120, "p": 12, "k": 2, "sets": 3000},
        # redundancy test of a polyhedron in preprocessing
        {"name": "redundant_rows", "op": "redundant", "m": 120, "nz": 16},
    ]


def _candidates(m, k):
    return sum(math.comb(m, i) for i in range(k + 1))


def _pivot_entries(n, m, p):
    """Entries (rows + cost row, columns + rhs) of the feasibility and the
    optimality tableau."""
    feas = (m + 2 * p + 1) * (n + p + 2)
    opt = (2 * m + 2 + 2 * p + n) * (n + p + m + 3)
    return feas, opt


def draw(rng):
    op = rng.choices(["solve", "noalloc", "pipeline", "many", "regions", "redundant"], [8, 1, 1, 1, 2, 1])[0]
    if op == "pipeline":
        n = rng.randint(2, 5)
        return {"op": op, "n": n, "m": rng.randint(3 * n, 24), "p": rng.randint(1, 5)}
    if op == "many":
        return {"op": op, "count": rng.randint(3, 16), "shapes": rng.randint(0, 10 ** 6), "k": 2}
    if op == "redundant":
        nz = rng.randint(3, 20)
        return {"op": op, "m": rng.randint(2 * nz, 120), "nz": nz}
    if op == "noalloc":
        n = rng.randint(5, 24)
        return {"op": op, "n": n, "m": rng.randint(2 * n, 2 * n + 10), "p": rng.randint(1, 6), "k": 2}
    n = round(math.exp(rng.uniform(math.log(5), math.log(60))))
    m = rng.randint(2 * n, min(2 * n + 40, 120))
    p = rng.randint(2, 12)
    if op == "regions":
        return {"op": op, "n": n, "m": m, "p": p, "k": 2, "sets": rng.randint(1, 3000)}
    mixed = rng.random() < 0.5
    persistent = mixed or rng.random() < 0.5
    # the deepest enumeration within a budget of tableau entries, FP64 and
    # ill-conditioned problems at half of the largest listed case's
    stress = n >= 20 and rng.random() < 0.15
    budget = _candidates(120, 3) * _pivot_entries(60, 120, 12)[1] * (0.75 if mixed and not stress else 0.4)
    budget *= math.exp(-rng.uniform(0.0, 3.0))
    k = 1
    while k < min(n, 6) and _candidates(m, k + 1) * _pivot_entries(n, m, p)[1] <= budget:
        k += 1
    return {"op": "solve", "n": n, "m": m, "p": p, "k": k, "mixed": mixed, "persistent": persistent,
            "records": rng.random() < 0.2 and _candidates(m, k) < 100000, "stress": stress}


def _problem(case, seed):
    if case.get("stress"):
        return precision_stress_mpqp(case["n"], case["m"], case["p"], seed, n_dup=min(10, case["m"] // 4))
    return synthetic_mpqp(case["n"], case["m"], case["p"], seed)


def _uneven_shapes(case):
    """Sizes of the problems of a "many" case: n in 5..40, m in 2n..2n+40
    (at most 120), p in 2..10."""
    rng = np.random.default_rng(case["shapes"])
    out = []
    for _ in range(case["count"]):
        n = int(rng.integers(5, 41))
        out.append((n, min(int(rng.integers(2 * n, 2 * n + 41)), 120), int(rng.integers(2, 11))))
    return out


def _library():
    lib = load_library()
    if lib.warm_up() != 0:
        raise RuntimeError(lib.last_error())
    return lib


def _options(case):
    op = case["op"]
    if op == "solve":
        return {"precision": MIXED if case["mixed"] else FP64,
                "batching": PERSISTENT if case["persistent"] else PLAIN, "record": 1 if case["records"] else 0}
    if op == "many":
        return {"precision": MIXED, "batching": PERSISTENT}
    if op == "pipeline":
        return {"batching": PERSISTENT}
    return {}


class _Table:
    """A results table of fixed size: rows past the last result hold `fill`."""

    def __init__(self, shape, dtype, fill):
        self.a, self.fill, self.used = np.full(shape, fill, dtype=dtype), fill, 0

    def put(self, rows):
        n = len(rows)
        if n < self.used:
            self.a[n:self.used] = self.fill
        at = (slice(0, n),) + tuple(slice(0, w) for w in rows.shape[1:])
        if rows.shape[1:] != self.a.shape[1:]:
            self.a[:n] = self.fill
        self.a[at] = rows
        self.used = n
        return self.a

    def put_lists(self, sets):
        n = len(sets)
        size = np.fromiter(map(len, sets), dtype=np.intp, count=n)
        rows = np.full((n, self.a.shape[1]), -1, dtype=self.a.dtype)
        rows[np.arange(self.a.shape[1]) < size[:, None]] = np.fromiter(
            itertools.chain.from_iterable(sets), dtype=self.a.dtype, count=int(size.sum()))
        return self.put(rows)


def prepare(case, seed):
    """Host arrays of the problem, the loaded library, the program's tables
    for the results, and for the regions final sets that a solve has
    returned (repeated if it returned fewer)."""
    op = case["op"]
    st = {"case": case, "lib": _library(), "options": _options(case)}
    if op in ("solve", "noalloc"):
        st["lp"] = assemble_lps(_problem(case, seed))
        cand = _candidates(case["m"], case["k"])
        st["rows"] = _Table((cand, case["k"]), np.intc, -1)
        if case.get("records"):
            st["sets"] = _Table((cand, case["k"]), np.intc, -1)
            st["records"] = {f: _Table((cand,), RECORD_DTYPE[f], 0) for f in RECORD_DTYPE.names}
    elif op == "many":
        st["lps"] = [assemble_lps(synthetic_mpqp(n, m, p, 1000 * seed + i))
                     for i, (n, m, p) in enumerate(_uneven_shapes(case))]
        st["rows"] = _Table((sum(_candidates(m, case["k"]) for _, m, _ in _uneven_shapes(case)), case["k"]), np.intc, -1)
    elif op == "regions":
        st["prog"] = _problem(case, seed)
        lib = st["lib"]
        lib.set_options(batching=PERSISTENT)
        rows = lib.run(assemble_lps(st["prog"]), k_max=case["k"], decode=False).active_rows
        if len(rows) == 0:
            rows = np.full((1, case["n"]), -1, dtype=np.intc)
        st["sets"] = np.resize(rows, (case["sets"], case["n"]))
    elif op == "redundant":
        # unit-norm rows around the origin, right-hand sides spread so that
        # a part of the rows is implied by the others
        rng = np.random.default_rng(seed)
        nz = case["nz"]
        box = np.vstack([np.eye(nz), -np.eye(nz)])
        G = rng.standard_normal((case["m"], nz))
        G[:2 * nz] = box[:case["m"]]
        G /= np.linalg.norm(G, axis=1, keepdims=True)
        h = rng.uniform(0.5, 3.0, case["m"])
        st["G"], st["h"] = G, h
    else:
        pr = synthetic_mpqp(case["n"], case["m"], case["p"], seed)
        st["problem"] = {"A": pr.A, "b": pr.b, "c": pr.c, "F": pr.F, "Q": pr.Q, "Ht": pr.H, "CRA": pr.A_t,
                         "CRb": pr.b_t}
        n, p, m0, most = case["n"], case["p"], case["m"] + 2 * case["p"], 2048
        shapes = {"center": (p,), "parameter_A": (n, p), "parameter_b": (n,), "lagrange_A": (n, p), "lagrange_b": (n,),
                  "cr_A": (m0, p), "cr_b": (m0,)}
        st["regions"] = {f: _Table((most,) + shapes.get(f, ()),
                                   np.int32 if f in ("status", "n_rows", "iters") else np.float64, 0)
                         for f in REGION_FIELDS}
        st["sets"] = _Table((most, n), np.intc, -1)
    return st


def run(st):
    case, lib = st["case"], st["lib"]
    op = case["op"]
    lib.set_options(**st["options"])
    if op == "solve":
        r = lib.run(st["lp"], k_max=case["k"], records=case["records"], decode=False)
        # a set has at most k members, the rest of its row is padding
        out = {"rows": st["rows"].put(r.active_rows[:, :case["k"]]), "n_feasible": r.n_feasible_lps,
               "n_final": r.n_final_lps}
        if case["records"]:
            out["sets"] = st["sets"].put(r.sets)
            for f, table in st["records"].items():
                out[f] = table.put(r.records[f])
        return out
    if op == "noalloc":
        r = lib.run_noalloc(st["lp"], k_max=case["k"], max_sets=_candidates(case["m"], case["k"]))
        return {"rows": st["rows"].put_lists(r.active_sets), "n_feasible": r.n_feasible_lps, "n_final": r.n_final_lps}
    if op == "many":
        runs, _ = lib.run_batch(st["lps"], k_max=case["k"])
        return {"rows": st["rows"].put_lists([s for r in runs for s in r.active_sets]),
                "n_feasible": np.array([r.n_feasible_lps for r in runs]),
                "n_final": np.array([r.n_final_lps for r in runs])}
    if op == "regions":
        b = lib.regions(st["prog"], st["sets"])
        return {f: getattr(b, f) for f in REGION_FIELDS}
    if op == "redundant":
        return {"keep": lib.redundant_rows(st["G"], st["h"])}
    r = solve_pop_problem(st["problem"], lib)
    out = {"n_regions": r.n_regions, "n_final": r.n_final, "sets": st["sets"].put(r.batch.sets)}
    for f, table in st["regions"].items():
        out[f] = table.put(getattr(r.batch, f))
    return out


def work(case):
    """Each candidate's two tableaus differ from its parent's by one pivot at
    least (2 flops an entry); the problem is read and the sets are written.
    Regions: the maps (|S| terms an entry) and the outputs' bytes."""
    op = case["op"]
    if op == "redundant":
        m, nz = case["m"], case["nz"]
        return {"bytes": 8 * m * (nz + 1) + 4 * m, "flops": m * 2 * (m + 1) * (2 * nz + 2)}
    if op == "many":
        tot = {"bytes": 0, "flops": 0}
        for n, m, p in _uneven_shapes(case):
            w = work({"op": "solve", "n": n, "m": m, "p": p, "k": case["k"]})
            tot = {q: tot[q] + w[q] for q in tot}
        return tot
    n, m, p = case["n"], case["m"], case["p"]
    k = case.get("k", n)
    feas, opt = _pivot_entries(n, m, p)
    inputs = 8 * (m * n + (m + 2 * p) * (n + p + 2) + (2 * m + 1 + 2 * p + n) * (n + p + m + 3))
    if op == "regions":
        sets = case["sets"]
        per = n * (p + 1) + n * (p + 1) + (m + 2 * p) * (p + 1) + p
        return {"bytes": 8 * (m * n + n * n + m * (p + 1)) + sets * (8 * per + 4 * n + 24),
                "flops": sets * 2 * k * (p + 1) * (n + m)}
    cand = min(_candidates(m, k), 200000) if op == "pipeline" else _candidates(m, k)
    return {"bytes": inputs + cand * 4 * n // 2, "flops": 2 * cand * (feas + opt)}


def exact(case, seed):
    """The affine maps of the critical regions in plain numpy; verdicts,
    counts and the linear programs' results have no closed form."""
    if case["op"] != "regions":
        return None
    st = prepare(case, seed)
    pr, sets = st["prog"], st["sets"]
    n_s, width = sets.shape
    n, p, m = case["n"], case["p"], case["m"]
    b, c = pr.b.ravel(), pr.c.ravel()
    iQ = np.linalg.inv(pr.Q)
    out = {f: None for f in REGION_FIELDS}
    pA, pb = np.zeros((n_s, n, p)), np.zeros((n_s, n))
    lA, lb = np.zeros((n_s, width, p)), np.zeros((n_s, width))
    Gm, AH, Ac = pr.A @ iQ @ pr.A.T, pr.A @ iQ @ pr.H, pr.A @ iQ @ c
    YA, YH, Yc = iQ @ pr.A.T, iQ @ pr.H, iQ @ c
    size = (sets >= 0).sum(axis=1)
    for k in np.unique(size):
        at = np.flatnonzero(size == k)
        S = sets[at, :k]
        rhs = np.concatenate([AH[S] + pr.F[S], (b[S] + Ac[S])[:, :, None]], axis=2)
        sol = -np.linalg.solve(Gm[S[:, :, None], S[:, None, :]], rhs) if k else rhs
        x = -np.einsum("ijs,sjt->sit", YA[:, S].transpose(0, 2, 1), sol) if k else np.zeros((len(at), n, p + 1))
        lA[at, :k], lb[at, :k] = sol[:, :, :p], sol[:, :, p]
        pA[at], pb[at] = x[:, :, :p] - YH, x[:, :, p] - Yc
    out["parameter_A"], out["parameter_b"], out["lagrange_A"], out["lagrange_b"] = pA, pb, lA, lb
    return out
